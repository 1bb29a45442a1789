"""GPU parity of the gated-delta backward pass (``lampa_gdr_bwd`` behind ``chunk_gated_delta_rule``'s autograd) against
the gradient oracle (``oracle.gated_delta_bwd.backward_manual``, float64 on the same, already rounded, inputs).

Tolerances: the token-serial kernels (``lampa_gdr_bwd``) compute in fp32 from the inputs as given, so fp32 inputs must
agree to 1e-4 (max-abs relative to the largest entry of the gradient; 1e-5 mean-relative); with bf16 / fp16 inputs dq,
dk and dv are rounded to that type on output (mean-relative 5e-3, the forward's bound), dg, dbeta and d(initial state)
stay fp32 (1e-4). The chunked form (``lampa_gdr_chunk_fwd_train`` and ``lampa_gdr_bwd_saved``: 16-bit inputs, heads up to
64 x 64) rounds every MFMA operand to the input type, as the reference's backward kernels do: all six gradients then carry that
type's rounding through a chain of five to six rounded intermediates (max-abs 2e-2 of the largest entry; mean-relative
8e-3; measured 3e-3 to 5.2e-3 for bf16, 5e-4 for fp16).
"""
import pytest
import torch

from lampa_amd import gated_delta as gd
from oracle import gated_delta as og
from oracle import gated_delta_bwd as ob

pytestmark = pytest.mark.gpu

NAMES = ("dq", "dk", "dv", "dg", "dbeta", "dh0")


def _inputs(B, T, H, HV, K, V, dtype, seed, unit, g_scale=1.0):
    gen = torch.Generator().manual_seed(seed)
    q, k = torch.randn(B, T, H, K, generator=gen), torch.randn(B, T, H, K, generator=gen)
    if unit:
        q, k = q / q.norm(dim=-1, keepdim=True), k / k.norm(dim=-1, keepdim=True)
    v = torch.randn(B, T, HV, V, generator=gen)
    g = -g_scale * torch.nn.functional.softplus(torch.randn(B, T, HV, generator=gen))
    beta = torch.sigmoid(torch.randn(B, T, HV, generator=gen))
    do = torch.randn(B, T, HV, V, generator=gen)
    return [x.to(dtype) for x in (q, k, v)] + [g, beta, do.to(dtype)], gen


def _gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, l2, scale=None):
    args = [x.to(device).requires_grad_(True) for x in (q, k, v, g, beta)]
    h0d = None if h0 is None else h0.to(device).requires_grad_(True)
    o, ht = gd.chunk_gated_delta_rule(*args, scale=scale, initial_state=h0d, output_final_state=dht is not None,
                                      cu_seqlens=None if cu is None else cu.to(device), use_qk_l2norm_in_kernel=l2,
                                      allow_fp32=True)
    loss = (o.float() * do.to(device).float()).sum()
    if dht is not None:
        loss = loss + (ht * dht.to(device)).sum()
    loss.backward()
    return [a.grad for a in args] + [None if h0d is None else h0d.grad]


def _check(got, want, dtype, chunked=None):
    """chunked: the gradients came from the chunked form (default: every 16-bit case while ``gd.CHUNKED_BACKWARD``)."""
    if chunked is None:
        chunked = dtype != torch.float32 and gd.CHUNKED_BACKWARD
    for name, a, b in zip(NAMES, got, want):
        if b is None:
            assert a is None, name
            continue
        a = a.double().cpu()
        assert a.shape == b.shape, name
        diff = (a - b).abs()
        rel_max = diff.max().item() / b.abs().max().clamp_min(1e-30).item()
        rel_mean = (diff.mean() / b.abs().mean().clamp_min(1e-30)).item()
        rounded = dtype != torch.float32 and (chunked or name in ("dq", "dk", "dv"))
        mean_bound = (8e-3 if chunked else 5e-3) if rounded else 1e-5
        assert rel_max <= (2e-2 if rounded else 1e-4) and rel_mean <= mean_bound, \
            f"{name}: max {rel_max:.3e} mean {rel_mean:.3e}"


@pytest.mark.parametrize("K,V,H,HV", [(16, 32, 2, 4), (64, 64, 2, 2), (128, 128, 1, 2), (32, 48, 1, 1), (24, 40, 2, 2),
                                      (10, 6, 1, 3), (128, 20, 1, 1)])
@pytest.mark.parametrize("l2", [False, True])
def test_gradients_fp32_match_oracle(device, K, V, H, HV, l2):
    """Equal-length batches with an initial state and a gradient into the final state; T = 75 leaves a partial block of
    8 tokens and a partial segment; head sizes on and off the kernels' shapes (10 x 6 is zero-padded to 12 x 8)."""
    (q, k, v, g, beta, do), gen = _inputs(2, 75, H, HV, K, V, torch.float32, K + V, unit=not l2)
    h0 = 0.5 * torch.randn(2, HV, K, V, generator=gen)
    dht = torch.randn(2, HV, K, V, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, 0.37, h0, None, og.L2_CHUNK if l2 else og.L2_NONE)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, None, l2, scale=0.37), want, torch.float32)


@pytest.mark.parametrize("dtype,chunked", [(torch.float32, False), (torch.bfloat16, False), (torch.float16, False),
                                           (torch.bfloat16, True), (torch.float16, True)])
def test_gradients_varlen_segments(device, dtype, chunked, monkeypatch):
    """Packed sequences (an empty one, one shorter than a block, lengths off the block and segment sizes), cut into
    segments of 64 tokens so that the reverse maps and the reverse scan carry the state gradient over many segments.
    16-bit inputs through both forms: token-serial, and chunked with the 32 x 32 heads zero-padded to 64 x 64 and the
    two value heads of a group sharing their q / k head."""
    monkeypatch.setattr(gd, "BACKWARD_UNITS", 1 << 20)
    monkeypatch.setattr(gd, "CHUNKED_BACKWARD", chunked)
    lens = [0, 5, 333, 64, 1, 500, 97]
    T = sum(lens)
    (q, k, v, g, beta, do), gen = _inputs(1, T, 2, 4, 32, 32, dtype, 7, unit=False)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.long)
    h0 = 0.5 * torch.randn(len(lens), 4, 32, 32, generator=gen)
    dht = torch.randn(len(lens), 4, 32, 32, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, cu, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, True), want, dtype)


def test_gradients_many_short_sequences_more_units_than_workgroups(device):
    """700 packed sequences of 1 .. 20 tokens: 700 segments x 4 heads x 2 slabs = 5 600 units for the segment kernel's
    4 096 workgroups, so some workgroups take a second unit (and reuse their spill area and LDS for it)."""
    gen = torch.Generator().manual_seed(13)
    lens = torch.randint(1, 21, (700,), generator=gen).tolist()
    T = sum(lens)
    (q, k, v, g, beta, do), gen = _inputs(1, T, 2, 4, 16, 32, torch.float32, 17, unit=False)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.long)
    h0 = 0.5 * torch.randn(700, 4, 16, 32, generator=gen)
    dht = torch.randn(700, 4, 16, 32, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, cu, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, True), want, torch.float32)


def test_gradients_scans_in_groups_unbalanced_sequences(device, monkeypatch):
    """Three sequences (one empty, one of a single short segment) cut into 64-token segments, 75 of them: both scans of
    the backward pass (forward, and reversed with one extra row per sequence) run in their three-launch form over groups
    of segments."""
    monkeypatch.setattr(gd, "BACKWARD_UNITS", 1 << 20)
    lens = [0, 4700, 30]
    T = sum(lens)
    (q, k, v, g, beta, do), gen = _inputs(1, T, 1, 2, 16, 16, torch.float32, 23, unit=False, g_scale=0.05)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.long)
    h0 = 0.5 * torch.randn(3, 2, 16, 16, generator=gen)
    dht = torch.randn(3, 2, 16, 16, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, cu, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, True), want, torch.float32)


def test_gradients_without_states_and_with_unused_output(device):
    """No initial state (no d h0), no final state; and a loss that uses the final state only (d o is zero)."""
    (q, k, v, g, beta, do), gen = _inputs(1, 200, 1, 2, 64, 64, torch.float32, 3, unit=True)
    want = ob.backward_manual(q, k, v, g, beta, do, None, None, None, None, og.L2_NONE)
    _check(_gpu_grads(device, q, k, v, g, beta, do, None, None, None, False), want, torch.float32)
    dht = torch.randn(1, 2, 64, 64, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, torch.zeros_like(do), dht, None, None, None, og.L2_NONE)
    args = [x.to(device).requires_grad_(True) for x in (q, k, v, g, beta)]
    _, ht = gd.chunk_gated_delta_rule(*args, output_final_state=True, allow_fp32=True)
    (ht * dht.to(device)).sum().backward()
    _check([a.grad for a in args] + [None], want, torch.float32)


def test_gradients_long_sequence_weak_decay(device):
    """4 096 tokens with g of the order of -0.003 per token: the state and its gradient carry over hundreds of tokens
    and through every segment (token-serial form; the chunked form has its own case below)."""
    gd_chunked = gd.CHUNKED_BACKWARD
    gd.CHUNKED_BACKWARD = False
    try:
        _weak_decay_case(device)
    finally:
        gd.CHUNKED_BACKWARD = gd_chunked


def _weak_decay_case(device):
    (q, k, v, g, beta, do), gen = _inputs(1, 4096, 1, 2, 64, 64, torch.bfloat16, 11, unit=False, g_scale=0.003)
    h0 = 0.5 * torch.randn(1, 2, 64, 64, generator=gen)
    dht = torch.randn(1, 2, 64, 64, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, None, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, None, True), want, torch.bfloat16)


def test_gradients_do_not_depend_on_the_segmentation_at_full_size(device, monkeypatch):
    """Config-2 shape (60 032 tokens, 8 heads, K = V = 64, bf16), too long for the float64 loop, on the token-serial
    form: the same gradients from 63 segments per head and from 8 (fp32 rounding apart), and linear in (d o, d final
    state)."""
    monkeypatch.setattr(gd, "CHUNKED_BACKWARD", False)
    (q, k, v, g, beta, do), gen = _inputs(1, 60032, 8, 8, 64, 64, torch.bfloat16, 5, unit=False)
    dht = torch.randn(1, 8, 64, 64, generator=gen)
    a = _gpu_grads(device, q, k, v, g, beta, do, None, dht, None, True)
    monkeypatch.setattr(gd, "BACKWARD_UNITS", 256)
    b = _gpu_grads(device, q, k, v, g, beta, do, None, dht, None, True)
    for name, x, y in zip(NAMES[:5], a, b):
        x, y = x.float(), y.float()
        assert torch.isfinite(x).all(), name
        rounded = name in ("dq", "dk", "dv")  # bf16 outputs: one rounding step apart at most
        assert (x - y).abs().max().item() <= (1e-2 if rounded else 2e-4) * y.abs().max().item(), name
    c = _gpu_grads(device, q, k, v, g, beta, (2 * do.float()).to(do.dtype), None, 2 * dht, None, True)
    for name, x, y in zip(NAMES[3:5], b[3:5], c[3:5]):  # the fp32 outputs: exactly twice (a power of two)
        assert torch.equal(2 * x, y), name


def test_fused_recurrent_backward_raises_like_the_reference(device):
    (q, k, v, g, beta, do), _ = _inputs(1, 16, 1, 1, 16, 16, torch.float32, 0, unit=True)
    args = [x.to(device).requires_grad_(True) for x in (q, k, v, g, beta)]
    o, _ = gd.fused_recurrent_gated_delta_rule(*args)
    with pytest.raises(NotImplementedError):
        o.sum().backward()


def test_backward_refuses_positive_log_decay(device):
    # for g > 0 the chunk forward masks decay ratios with positive exponents (safe_exp) while the backward pass
    # differentiates the unmasked recurrence: the two would belong to different functions, so backward raises
    (q, k, v, g, beta, do), _ = _inputs(1, 130, 2, 2, 64, 64, torch.bfloat16, 0, True)
    g = g.clone()
    g[0, 70, 1] = 0.25
    args = [x.to(device).requires_grad_(True) for x in (q, k, v, g, beta)]
    o, _ = gd.chunk_gated_delta_rule(*args)          # the forward itself accepts it, as the reference's does
    with pytest.raises(ValueError, match="g <= 0"):
        o.float().sum().backward()


# ------------------------------------------------------------------------------------- chunked form on the MFMA
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("T", [1, 64, 75, 1000])
def test_chunked_gradients_match_oracle(device, dtype, l2, T):
    """K = V = 64, 16-bit inputs take the chunked form: batches with an initial state and a gradient into the final state; one
    token, one chunk, a partial second chunk, 16 chunks in four segments."""
    assert gd._backward_chunk_supported(torch.empty(1, 1, 2, 64, dtype=dtype), torch.empty(1, 1, 2, 64, dtype=dtype))
    (q, k, v, g, beta, do), gen = _inputs(2, T, 2, 2, 64, 64, dtype, T, unit=not l2)
    h0 = 0.5 * torch.randn(2, 2, 64, 64, generator=gen)
    dht = torch.randn(2, 2, 64, 64, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, 0.2, h0, None, og.L2_CHUNK if l2 else og.L2_NONE)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, None, l2, scale=0.2), want, dtype, chunked=True)


def test_chunked_gradients_varlen_and_without_states(device):
    """Packed sequences (an empty one, one token, lengths off the chunk size, one of 80 chunks in 20
    segments) with states; then no initial state and no gradient into the final state; then a loss on the final state only."""
    lens = [0, 5, 333, 64, 1, 5100, 97]
    T = sum(lens)
    (q, k, v, g, beta, do), gen = _inputs(1, T, 3, 3, 64, 64, torch.bfloat16, 7, unit=False, g_scale=0.3)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.long)
    h0 = 0.5 * torch.randn(len(lens), 3, 64, 64, generator=gen)
    dht = torch.randn(len(lens), 3, 64, 64, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, cu, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, True), want, torch.bfloat16, chunked=True)
    want = ob.backward_manual(q, k, v, g, beta, do, None, None, None, cu, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, None, None, cu, True), want, torch.bfloat16, chunked=True)
    want = ob.backward_manual(q, k, v, g, beta, torch.zeros_like(do), dht, None, None, cu, og.L2_CHUNK)
    args = [x.to(device).requires_grad_(True) for x in (q, k, v, g, beta)]
    _, ht = gd.chunk_gated_delta_rule(*args, output_final_state=True, cu_seqlens=cu.to(device),
                                      use_qk_l2norm_in_kernel=True)
    (ht * dht.to(device)).sum().backward()
    _check([a.grad for a in args] + [None], want, torch.bfloat16, chunked=True)


def test_chunked_gradients_long_sequence_weak_decay_against_oracle(device):
    """16 448 tokens (257 chunks in 65 segments: groups of 8 and a remainder of one) with g of the order of
    -0.003 per token, so that states and their gradients carry over thousands of tokens, against the float64 loop."""
    (q, k, v, g, beta, do), gen = _inputs(1, 16448, 2, 2, 64, 64, torch.bfloat16, 11, unit=True, g_scale=0.003)
    h0 = 0.5 * torch.randn(1, 2, 64, 64, generator=gen)
    dht = torch.randn(1, 2, 64, 64, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, None, og.L2_NONE)
    got = _gpu_grads(device, q, k, v, g, beta, do, h0, dht, None, False)
    for name, a, b in zip(NAMES, got, want):
        d = (a.double().cpu() - b).abs()
        print(f"chunked backward T=16448 weak decay {name}: max-rel {d.max().item() / b.abs().max().item():.2e} "
              f"mean-rel {(d.mean() / b.abs().mean()).item():.2e}")
    _check(got, want, torch.bfloat16, chunked=True)


@pytest.mark.parametrize("T,K,V", [(64 * 23, 64, 64), (64 * 24, 64, 64), (64 * 26 + 1, 64, 64), (63, 48, 64), (65, 64, 40)])
def test_chunked_gradients_one_chunk_per_segment(device, T, K, V, monkeypatch):
    """Segments of one chunk, so that a sequence has 23 (the walk passes all of them one by one), 24 (groups of 8, no
    remainder) and 27 segments (groups and a remainder); one partial chunk, and a second chunk of one token; grouped value
    heads, heads below 64 x 64. The gradients are taken twice from one graph: the kept buffer is only read."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 1)
    (q, k, v, g, beta, do), gen = _inputs(1, T, 1, 2, K, V, torch.bfloat16, T + K, unit=False, g_scale=0.02)
    h0 = 0.5 * torch.randn(1, 2, K, V, generator=gen)
    dht = torch.randn(1, 2, K, V, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, None, og.L2_CHUNK)
    leaves = [x.to(device).requires_grad_(True) for x in (q, k, v, g, beta, h0)]
    o, ht = gd.chunk_gated_delta_rule(*leaves[:5], initial_state=leaves[5], output_final_state=True,
                                      use_qk_l2norm_in_kernel=True)
    for _ in range(2):
        got = torch.autograd.grad((o, ht), leaves, (do.to(device), dht.to(device)), retain_graph=True)
        _check(got, want, torch.bfloat16, chunked=True)


def test_chunked_gradients_of_a_long_sequence_beside_a_short_one(device, monkeypatch):
    """40 segments beside 3: more groups of 8 than the workspace has slots for when every sequence gets as many as the longest,
    so that the walk passes all 39 segments behind the first one by one."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 1)
    cu = torch.tensor([0, 64 * 40, 64 * 43])
    (q, k, v, g, beta, do), gen = _inputs(1, 64 * 43, 2, 2, 64, 64, torch.bfloat16, 43, unit=False, g_scale=0.02)
    h0, dht = (torch.randn(2, 2, 64, 64, generator=gen) for _ in range(2))
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, cu, og.L2_CHUNK)
    _check(_gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, True), want, torch.bfloat16, chunked=True)


@pytest.mark.parametrize("cps", [2, 3])
@pytest.mark.parametrize("l2norm", [False, True])
def test_chunked_gradients_tile_sets(device, cps, l2norm, monkeypatch):
    """Segments of two and three chunks (the walks alternate between two sets of tiles and write a chunk's rows of dq and dk a
    chunk later), a sequence ending in a partial chunk, an empty one and one of a single token, two value heads per head."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", cps)
    cu = torch.tensor([0, 64 * 7 + 33, 64 * 7 + 33, 64 * 7 + 34])
    (q, k, v, g, beta, do), gen = _inputs(1, int(cu[-1]), 1, 2, 64, 64, torch.bfloat16, 17 + cps, unit=not l2norm, g_scale=0.05)
    h0 = 0.5 * torch.randn(3, 2, 64, 64, generator=gen)
    dht = torch.randn(3, 2, 64, 64, generator=gen)
    want = ob.backward_manual(q, k, v, g, beta, do, dht, None, h0, cu, og.L2_CHUNK if l2norm else og.L2_NONE)
    got = _gpu_grads(device, q, k, v, g, beta, do, h0, dht, cu, l2norm)
    _check(got, want, torch.bfloat16, chunked=True)


def test_chunked_gradients_at_full_size_against_the_token_serial_form(device, monkeypatch):
    """Config-2 shape (60 000 tokens, 8 heads, K = V = 64, bf16), too long for the float64 loop: the chunked form on the
    MFMA against the fp32 token-serial form, two implementations that share no kernel of the backward pass."""
    (q, k, v, g, beta, do), gen = _inputs(1, 60000, 8, 8, 64, 64, torch.bfloat16, 5, unit=False)
    dht = torch.randn(1, 8, 64, 64, generator=gen)
    h0 = 0.5 * torch.randn(1, 8, 64, 64, generator=gen)
    a = _gpu_grads(device, q, k, v, g, beta, do, h0, dht, None, True)
    monkeypatch.setattr(gd, "CHUNKED_BACKWARD", False)
    b = _gpu_grads(device, q, k, v, g, beta, do, h0, dht, None, True)
    _check(a, [x.double().cpu() for x in b], torch.bfloat16, chunked=True)


@pytest.mark.parametrize("rows,widths,offset", [(1, ((16, 64),), 0), (1023, ((16, 64), (64, 24), (32, 64)), 0),
                                                (2049, ((10, 32), (6, 64), (128, 5), (64, 1)), 0),
                                                (777, ((16, 64), (64, 16)), 1), (64, ((256, 8), (8, 256)), 0),
                                                (1000, ((100, 128), (20, 64)), 0), (515, ((66, 128), (128, 30)), 0),
                                                (4097, ((127, 128), (65, 256), (256, 255), (3, 1)), 0), (999, ((2, 3), (64, 2)), 2)])
def test_resized_heads_are_padded_and_cut_copies(device, rows, widths, offset):
    """Bit for bit what torch's pad and slice give: last blocks of rows, odd widths and odd addresses (one element per
    thread), widths that do not divide a workgroup."""
    src = [torch.arange(rows * w + offset, device=device).to(torch.int16).view(torch.bfloat16)[offset:].view(1, rows, w)
           for w, _ in widths]
    for x, y, (w, n) in zip(src, gd._resize_heads(src, [n for _, n in widths]), widths):
        want = torch.nn.functional.pad(x.view(torch.int16), (0, n - w))  # (a negative pad cuts)
        assert y.is_contiguous() and torch.equal(y.view(torch.int16), want)


def test_resized_heads_of_more_rows_than_one_turn_of_the_grid(device):
    """Rows of 129 elements, one at a time: 31 rows to a workgroup, and 2^20 workgroups."""
    rows = 31 * 2 ** 20 + 9
    src = torch.arange(rows, device=device).to(torch.int16).view(torch.bfloat16).view(1, rows, 1)
    dst = gd._resize_heads((src,), (129,))[0].view(torch.int16)
    assert torch.equal(dst[..., :1], src.view(torch.int16))
    for a in range(0, rows, 2 ** 22):
        assert not bool(dst[:, a:a + 2 ** 22, 1:].any())


@pytest.mark.parametrize("K,V,H,HV", [(8, 8, 2, 2), (16, 32, 3, 3), (48, 56, 1, 2), (64, 24, 2, 2), (20, 64, 2, 2), (40, 30, 1, 1)])
def test_small_heads_are_written_in_their_own_width(device, K, V, H, HV):
    """Output, final state and gradients of heads below 64 x 64 (in sizes the kernels write themselves and in sizes that are
    cut afterwards) against the same call with the heads zero-padded by hand: the same bits. Ragged last chunk, several
    segments, packed sequences."""
    cu = torch.tensor([0, 700, 700, 1501], device=device)
    (q, k, v, g, beta, do), gen = _inputs(1, 1501, H, HV, K, V, torch.float16, K + V, unit=False)
    pad = torch.nn.functional.pad
    wide = [pad(q, (0, 64 - K)), pad(k, (0, 64 - K)), pad(v, (0, 64 - V)), g, beta]

    def run(args, do):
        leaves = [x.to(device).requires_grad_(True) for x in args]
        o, ht = gd.chunk_gated_delta_rule(*leaves, scale=0.25, output_final_state=True, cu_seqlens=cu,
                                          use_qk_l2norm_in_kernel=True)
        return o, ht, *torch.autograd.grad(o, leaves, do.to(device))

    got, want = run((q, k, v, g, beta), do), run(wide, pad(do, (0, 64 - V)))
    cut = (want[0][..., :V], want[1][..., :K, :V], want[2][..., :K], want[3][..., :K], want[4][..., :V], *want[5:])
    for a, b in zip(got, cut):
        assert a.is_contiguous() and torch.equal(a, b)


def test_forward_of_a_training_call_in_a_captured_graph(device):
    """A forward captured into a graph, replayed on other inputs and with eager work in between, then differentiated: the bits
    of the eager call; the check of g looks at the values of the last replay, and a positive entry of an earlier one is
    forgotten."""
    make = lambda seed: [x.to(device) for x in _inputs(1, 1000, 2, 2, 64, 64, torch.bfloat16, seed, unit=False)[0]]
    static = [x.requires_grad_(True) for x in make(1)[:5]]
    call = lambda args: gd.chunk_gated_delta_rule(*args, use_qk_l2norm_in_kernel=True)[0]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = call(static)
    for seed in (2, 3):
        *new, do = make(seed)
        for x, y in zip(static, new):
            x.data.copy_(y)
        graph.replay()
        leaves = [x.requires_grad_(True) for x in new]
        want = call(leaves)
        assert torch.equal(o, want)
        for a, b in zip(torch.autograd.grad(o, static, do, retain_graph=True), torch.autograd.grad(want, leaves, do)):
            assert torch.equal(a, b)
    static[3].data[0, 5, 1] = 0.25
    graph.replay()
    with pytest.raises(ValueError, match="g <= 0"):
        torch.autograd.grad(o, static, do, retain_graph=True)
    static[3].data[0, 5, 1] = -0.25
    graph.replay()
    torch.autograd.grad(o, static, do)


def test_positive_g_of_a_dropped_graph_does_not_reach_the_next_call(device):
    """Forwards that accept a positive g and are never differentiated, each followed at once by a training step on valid values,
    with small pinned buffers made in between: the steps are not refused and the buffers stay as they are."""
    make = lambda seed: [x.to(device) for x in _inputs(1, 20000, 2, 2, 64, 64, torch.bfloat16, seed, unit=False)[0]]
    *bad, do = make(1)
    bad[3] = bad[3].clone()
    bad[3][0, -1, 1] = 0.25
    bad = [x.requires_grad_(True) for x in bad]
    good = [x.requires_grad_(True) for x in make(2)[:5]]
    buffers = []
    for _ in range(20):
        gd.chunk_gated_delta_rule(*bad)
        buffers.append(torch.zeros(1, dtype=torch.int32, pin_memory=True))
        o, _ = gd.chunk_gated_delta_rule(*good)
        torch.autograd.grad(o, good, do)
    torch.cuda.synchronize()
    assert not any(int(b) for b in buffers)


@pytest.mark.parametrize("lens", [[64 * 40 + 7, 0, 1, 64 * 16, 700], [33]])
def test_c_entry_from_the_inputs_alone(device, lens, monkeypatch):
    """``lampa_gdr_bwd_chunk`` with its own plan (segments of 16 chunks) and exactly the workspace it asks for: the bits of the
    operator's gradients on the same segments, nothing written behind the workspace; with and without states."""
    import ctypes

    from lampa_amd import _capi

    lib, ptr = _capi.lib(), _capi.ptr
    T, n = sum(lens), len(lens)
    (q, k, v, g, beta, do), gen = _inputs(1, T, 3, 3, 64, 64, torch.bfloat16, n, unit=False, g_scale=0.05)
    q, k, v, g, beta, do, h0, dht = (x.to(device) for x in (q, k, v, g, beta, do, 0.5 * torch.randn(n, 3, 64, 64, generator=gen),
                                                            torch.randn(n, 3, 64, 64, generator=gen)))
    bounds = [0] + torch.tensor(lens).cumsum(0).tolist()
    cu = (ctypes.c_int64 * (n + 1))(*bounds)
    plan = torch.zeros(_capi.check(lib.lampa_gdr_bwd_chunk_plan_size(cu, n), "plan_size"), dtype=torch.int32)
    host = ctypes.c_void_p(plan.data_ptr())
    _capi.check(lib.lampa_gdr_bwd_chunk_plan_fill(cu, n, host), "plan_fill")
    plan_dev = plan.to(device)
    n_bytes = _capi.check(lib.lampa_gdr_bwd_chunk_workspace_bytes(host, 3), "workspace_bytes")
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 16)
    for states in (True, False):
        ws = torch.full((n_bytes + 65536,), 0xA5, dtype=torch.uint8, device=device)
        s0, ds = (h0, dht) if states else (None, None)
        got = [torch.empty_like(x) for x in (q, k, v, g, beta)] + [torch.empty_like(h0) if states else None]
        _capi.check(lib.lampa_gdr_bwd_chunk(*(ptr(x) for x in (q, k, v, g, beta, s0, do, ds, *got)), host, ptr(plan_dev), 3, 3,
                                            64, 64, 0, 0.2, gd.L2_CHUNK, ptr(ws), n_bytes, _capi.stream_of(q)), "bwd_chunk")
        assert bool((ws[n_bytes:] == 0xA5).all())
        leaves = [x.detach().clone().requires_grad_(True) for x in (q, k, v, g, beta)] + ([h0.clone().requires_grad_(True)] * states)
        o, ht = gd.chunk_gated_delta_rule(*leaves[:5], scale=0.2, initial_state=leaves[5] if states else None,
                                          output_final_state=states, cu_seqlens=torch.tensor(bounds, device=device),
                                          use_qk_l2norm_in_kernel=True)
        want = torch.autograd.grad((o, ht), leaves, (do, dht)) if states else torch.autograd.grad(o, leaves, do)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    short = ptr(ws), n_bytes - 1
    assert lib.lampa_gdr_bwd_chunk(*(ptr(x) for x in (q, k, v, g, beta, None, do, None, *got)), host, ptr(plan_dev), 3, 3, 64,
                                   64, 0, 0.2, gd.L2_CHUNK, *short, _capi.stream_of(q)) == -2


@pytest.mark.parametrize("token,value", [(700, float("inf")), (400, float("nan")), (767, float("-inf"))])
def test_values_that_are_not_finite_stay_out_of_earlier_gradients(device, token, value, monkeypatch):
    """A token whose v is not finite, with no loss on its chunk and the later ones: the gradients of the chunks before it are
    those of finite values, bit for bit (no v enters the gradient of a state), across the segments' boundaries."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 4)
    (q, k, v, g, beta, do), gen = _inputs(1, 768, 2, 2, 64, 64, torch.bfloat16, 5, unit=False, g_scale=0.02)
    h0 = torch.randn(1, 2, 64, 64, generator=gen)
    end = token // 64 * 64
    do[:, end:] = 0
    broken = v.clone()
    broken[0, token, 0, 3] = value
    want, got = (_gpu_grads(device, q, k, x, g, beta, do, h0, None, None, True) for x in (v, broken))
    for a, b in zip(got[:5], want[:5]):
        assert torch.equal(a[:, :end], b[:, :end])
    assert torch.equal(got[5], want[5])


@pytest.mark.parametrize("T,lens,H,dtype", [(14983, None, 6, torch.float16), (20000, None, 8, torch.bfloat16),
                                            (None, [5000, 0, 7001], 4, torch.bfloat16)])
def test_forward_of_a_training_step_gives_the_bits_of_the_plain_call(device, T, lens, H, dtype):
    """Outputs and final states of a forward that keeps what the backward pass needs: those of the call without gradients (the
    same segments, so M' is rounded at the same places), where a segment's states live on into the next ones."""
    cu = None if lens is None else torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), device=device)
    (q, k, v, g, beta, _), _ = _inputs(1, T or sum(lens), H, H, 64, 64, dtype, H, unit=False, g_scale=0.05)
    args = [x.to(device) for x in (q, k, v, g, beta)]
    call = lambda: gd.chunk_gated_delta_rule(*args, output_final_state=True, cu_seqlens=cu, use_qk_l2norm_in_kernel=True)
    o, s = call()
    for x in args:
        x.requires_grad_(True)
    ot, st = call()
    assert ot.requires_grad and torch.equal(o, ot) and torch.equal(s, st)


@pytest.mark.parametrize("dtype,cps,T", [(torch.bfloat16, 9, 64 * 9 * 3 - 9), (torch.float16, 9, 64 * 9 * 25), (torch.bfloat16, 66, 64 * 66 * 2 + 700)])
def test_sources_end_where_later_chunks_no_longer_count(device, dtype, cps, T, monkeypatch):
    """Segments whose first two (head 0) or four (head 1) chunks decay by more than the fp32 range, of which the pass for the
    segments' own gradients walks no others (and the walk over the segments behind starts at the next one); head 2 has next to
    no decay, head 3 one in its first half. Then a dO or a q that is not finite at either end of the chunks left out: none of
    the gradients that it belongs to in front of it are."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", cps)
    (q, k, v, g, beta, do), _ = _inputs(1, T, 4, 4, 64, 64, dtype, seed=cps, unit=False, g_scale=0.02)
    g[:, :, 0] *= 90
    g[:, :, 1] *= 35
    g[:, : T // 2, 3] *= 50
    got = _gpu_grads(device, q, k, v, g, beta, do, None, None, None, True)
    want = ob.backward_manual(q, k, v, g, beta, do, l2=og.L2_CHUNK)
    _check(got[:5], want[:5], dtype, chunked=True)
    assert all(torch.isfinite(x).all() for x in got[:5])
    seg = 64 * cps  # (of the second segment)
    for row in (seg + 64 * 2, seg + 64 * 4 + 3, 2 * seg - 1):
        bad = do.clone()
        bad[0, row, :2, 40] = float("inf")
        nan = _gpu_grads(device, q, k, v, g, beta, bad, None, None, None, True)
        assert not torch.isfinite(nan[2][0, :row, :2, 40]).any()
        assert all(torch.equal(a[:, :, 2:], b[:, :, 2:]) for a, b in zip(nan[:5], got[:5]))
        bad = q.clone()
        bad[0, row, :2, 3] = float("nan")
        nan = _gpu_grads(device, bad, k, v, g, beta, do, None, None, None, True)
        assert not torch.isfinite(nan[2][0, : row // 64 * 64, :2]).any()
        assert all(torch.equal(a[:, :, 2:], b[:, :, 2:]) for a, b in zip(nan[:5], got[:5]))


@pytest.mark.parametrize("q_exp,do_exp,edge", [(0, 115, -70), (60, 60, -72)])
def test_large_sources_behind_strong_decays(device, q_exp, do_exp, edge, monkeypatch):
    """Three chunks of 2^edge that write nothing in front of q and dO whose products are large, no dO before these: what is left
    of them there is small, but within the fp32 range."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 12)
    T, seg = 64 * 24, 64 * 12
    (q, k, v, g, beta, do), _ = _inputs(1, T, 2, 2, 64, 64, torch.bfloat16, seed=3, unit=True, g_scale=1e-4)
    q[:, seg:] *= 2.0 ** q_exp
    do *= 2.0 ** do_exp
    do[:, :seg + 64 * 3] = 0
    beta[:, seg:seg + 64 * 3] = 0
    g[:, seg:seg + 64 * 3] = edge * 0.6931471805599453 / 64
    got = _gpu_grads(device, q, k, v, g, beta, do, None, None, None, False)
    want = ob.backward_manual(q, k, v, g, beta, do)
    for a, b in zip(got[1:3], want[1:3]):  # dk, dv of the segment in front
        a, b = a[:, :seg].cpu().double(), b[:, :seg]
        assert 0 < b.abs().max() < 2.0 ** -80 and (a - b).norm() <= 2e-2 * b.norm()


@pytest.mark.parametrize("dtype,q_exp,do_exp,scale", [(torch.bfloat16, 70, 60, 1.0), (torch.bfloat16, 0, 100, 2.0 ** 40)])
def test_sources_that_overflow_behind_strong_decays(device, dtype, q_exp, do_exp, scale, monkeypatch):
    """Products of q, dO and the scale beyond the fp32 range behind three chunks of 2^-100: the gradients in front of these are
    none, as where every chunk is walked."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 12)
    T, seg = 64 * 24, 64 * 12
    (q, k, v, g, beta, do), _ = _inputs(1, T, 2, 2, 64, 64, dtype, seed=3, unit=True, g_scale=1e-4)
    q[:, seg:] *= 2.0 ** q_exp
    do *= 2.0 ** do_exp
    do[:, :seg + 64 * 3] = 0
    g[:, seg:seg + 64 * 3] = -100 * 0.6931471805599453 / 64
    got = _gpu_grads(device, q, k, v, g, beta, do, None, None, None, False, scale=scale)
    assert not torch.isfinite(got[2][:, :seg]).any()


@pytest.mark.parametrize("beta0", [3.0, 2.0])
def test_tokens_that_are_no_contraction_keep_the_gradient_behind_them(device, beta0, monkeypatch):
    """Five chunks at a segment's start whose log-decays sum up to 2^-320 and whose tokens all map one direction by 1 - beta0: with 3
    they take the decay back and hand the gradient of that row on as it was, with 2 nothing is left of it in front. (2e-2: the
    roundings of an ordinary call's gradients.)"""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 12)
    T, seg = 64 * 24, 64 * 12
    (q, k, v, g, beta, do), _ = _inputs(1, T, 2, 2, 64, 64, torch.bfloat16, seed=5, unit=True, g_scale=1e-3)
    start = slice(seg, seg + 64 * 5)
    k[:, start] = 0
    k[:, start, :, 5] = 1
    beta[:, start] = beta0
    g[:, start] = -0.6931471805599453
    do[:, :seg + 64 * 5] = 0
    got = _gpu_grads(device, q, k, v, g, beta, do, None, None, None, False)
    want = ob.backward_manual(q, k, v, g, beta, do)
    b = want[2][:, :seg]  # dv
    assert (b.abs().max() > 1e-2) == (beta0 == 3.0)
    assert (got[2][:, :seg].cpu().double() - b).norm() <= 2e-2 * b.norm() + 1e-30


def test_sources_of_grouped_heads_with_chunks_left_out(device, monkeypatch):
    """Two q / k heads of four value heads: the look at q of the chunks left out follows the group. A q of the second head that is
    not finite leaves the first head's gradients alone."""
    monkeypatch.setattr(gd, "CHUNKS_PER_SEGMENT", 9)
    T, seg = 64 * 9 * 3 - 20, 64 * 9
    (q, k, v, g, beta, do), _ = _inputs(1, T, 2, 4, 64, 64, torch.bfloat16, seed=7, unit=False, g_scale=2.0)
    got = _gpu_grads(device, q, k, v, g, beta, do, None, None, None, True)
    want = ob.backward_manual(q, k, v, g, beta, do, l2=og.L2_CHUNK)
    _check(got[:5], want[:5], torch.bfloat16, chunked=True)
    bad = q.clone()
    bad[0, 2 * seg - 1, 1, 3] = float("nan")
    nan = _gpu_grads(device, bad, k, v, g, beta, do, None, None, None, True)
    assert not torch.isfinite(nan[2][0, : 2 * seg - 64, 2:]).any() and not torch.isfinite(nan[1][0, : 2 * seg - 64, 1]).any()
    for i, heads in enumerate((1, 1, 2, 2, 2)):
        assert torch.equal(nan[i][:, :, :heads], got[i][:, :, :heads])
