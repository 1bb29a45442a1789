// Token-serial gated-delta-rule forward with an fp32 state held in registers (gfx950). Two kernels:
//
// gdr_recurrent_kernel: one wave owns up to 64 value columns of one (sequence, value head): lane = value column, and
// every lane keeps the K state rows of its column in registers, so the three contractions of a step (S^T k, the
// rank-one update and S^T q) are per-lane loops with no cross-lane traffic; k_t and q_t are loaded one element per
// lane, normalised with a wave reduction and broadcast with v_readlane.
// gdr_recurrent_split_kernel (further down, what nearly all launches take): 16 columns per wave, the state rows of a column
// split over eight or four lanes, the token's operands staged in LDS by the waves of a workgroup together. The first one serves
// sizes and alignments that cannot be staged in 16-byte pieces, head-wise beta, and one or two tokens each of very many
// sequences at 32 < K <= 64.
//
// Replaces fused_recurrent_gated_delta_rule_fwd_kernel, models/hattention/gated_delta_rule_ori.py:372-464
// (state layout [N, HV, K, V] fp32; grouped value heads HV >= H).  It is also the fp32 mode of the chunk operator and
// the on-GPU cross-check of the chunk kernels.
#include "gdr_common.h"

// value of lane `src` (a compile-time constant) in every lane: one v_readlane into a scalar register
__device__ __forceinline__ float bcast(float x, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), src));
}

// BETA_V: beta holds one value per value column, [tokens, HV, V] (IS_BETA_HEADWISE of the reference kernel,
// gated_delta_rule_ori.py:415-418,444-448), instead of one per (token, value head).
template <typename T, int KT, bool BETA_V = false>
__global__ void __launch_bounds__(64) gdr_recurrent_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                          const T* __restrict__ v, const float* __restrict__ g,
                                                          const float* __restrict__ beta, T* __restrict__ o,
                                                          const float* __restrict__ h0, float* __restrict__ ht,
                                                          const int64_t* __restrict__ cu_seqlens, int64_t t_len,
                                                          int H, int HV, int K, int V, float scale, int l2norm) {
  constexpr int KR = KT / 64 > 0 ? KT / 64 : 1;  // k/q elements held per lane
  const int lane = threadIdx.x;
  const int col = blockIdx.x * 64 + lane;
  const bool active = col < V;
  const int seq = blockIdx.y / HV, hv = blockIdx.y % HV;
  const int h = hv / (HV / H);
  const int64_t bos = cu_seqlens ? cu_seqlens[seq] : seq * t_len;
  const int64_t eos = cu_seqlens ? cu_seqlens[seq + 1] : bos + t_len;

  float S[KT];
#pragma unroll
  for (int i = 0; i < KT; ++i)
    S[i] = (h0 && active && i < K) ? h0[(((int64_t)seq * HV + hv) * K + i) * V + col] : 0.0f;

  // The inputs of the coming tokens are loaded PF tokens ahead into a ring of registers (a step depends on the
  // previous one through the state only, so without this every token pays a full memory latency). Loads past the end
  // of the sequence re-read its last token and are dropped.
  constexpr int PF = 8;
  struct Tok {
    float kv[KR], qv[KR], g, b, v;
  };
  Tok ring[PF];
  auto issue = [&](int64_t t, Tok& x) __attribute__((always_inline)) {
    t = t < eos ? t : eos - 1;
#pragma unroll
    for (int r = 0; r < KR; ++r) {
      const int i = r * 64 + lane;
      x.kv[r] = i < K ? GdrElem<T>::to_float(k[(t * H + h) * K + i]) : 0.0f;
      x.qv[r] = i < K ? GdrElem<T>::to_float(q[(t * H + h) * K + i]) : 0.0f;
    }
    x.g = g[t * HV + hv];
    if constexpr (BETA_V) x.b = active ? beta[(t * HV + hv) * V + col] : 0.0f;
    else x.b = beta[t * HV + hv];
    x.v = active ? GdrElem<T>::to_float(v[(t * HV + hv) * V + col]) : 0.0f;
  };
  auto step = [&](int64_t t, const Tok& x) __attribute__((always_inline)) {
    float kv[KR], qv[KR];
    float kss = 0.0f, qss = 0.0f;
#pragma unroll
    for (int r = 0; r < KR; ++r) {
      kv[r] = x.kv[r];
      qv[r] = x.qv[r];
      kss += kv[r] * kv[r];
      qss += qv[r] * qv[r];
    }
    float kinv = 1.0f, qinv = 1.0f;
    if (l2norm != GDR_L2_NONE) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        kss += __shfl_xor(kss, off);
        qss += __shfl_xor(qss, off);
      }
      if (l2norm == GDR_L2_CHUNK) {
        kinv = 1.0f / __fsqrt_rn(kss + 1e-6f);
        qinv = 1.0f / __fsqrt_rn(qss + 1e-6f);
      } else {
        kinv = 1.0f / (__fsqrt_rn(kss) + 1e-6f);
        qinv = 1.0f / (__fsqrt_rn(qss) + 1e-6f);
      }
    }
#pragma unroll
    for (int r = 0; r < KR; ++r) { kv[r] *= kinv; qv[r] *= qinv * scale; }
    const float decay = expf(x.g);
    const float b = x.b;
    const float vt = x.v;

    float dot4[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // four interleaved partial sums: a single chain of KT dependent FMAs
#pragma unroll                                  // would be the step's critical path
    for (int i = 0; i < KT; ++i) {
      const float ki = bcast(kv[i / 64], i % 64);
      S[i] *= decay;
      dot4[i & 3] = __builtin_fmaf(S[i], ki, dot4[i & 3]);
    }
    const float d = b * (vt - ((dot4[0] + dot4[1]) + (dot4[2] + dot4[3])));
    float out4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const float ki = bcast(kv[i / 64], i % 64);
      const float qi = bcast(qv[i / 64], i % 64);
      S[i] = __builtin_fmaf(ki, d, S[i]);
      out4[i & 3] = __builtin_fmaf(S[i], qi, out4[i & 3]);
    }
    const float out = (out4[0] + out4[1]) + (out4[2] + out4[3]);
    if (active) o[(t * HV + hv) * V + col] = GdrElem<T>::from_float(out);
  };
  if (bos < eos) {
#pragma unroll
    for (int p = 0; p < PF; ++p) issue(bos + p, ring[p]);
    for (int64_t t0 = bos; t0 < eos; t0 += PF) {
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const Tok cur = ring[p];
        issue(t0 + p + PF, ring[p]);
        if (t0 + p < eos) step(t0 + p, cur);
      }
    }
  }
  if (ht && active) {
#pragma unroll
    for (int i = 0; i < KT; ++i)
      if (i < K) ht[(((int64_t)seq * HV + hv) * K + i) * V + col] = S[i];
  }
}

// ---- the same recurrence with the state rows of a column split over eight or four lanes -------------------------------
// A wave owns 16 value columns of one (sequence, value head): lane = (column pair, row group), a
// lane keeps KT / 8 state rows of two columns, and the partial sums of S^T k and of S^T q meet over eight neighbouring lanes
// (three DPP additions each, no LDS); narrow heads have KT / 4 rows of one column to a lane (see NC). One wave per SIMD is bound by the instructions of a step, four cycles each, and by the
// dependent chain S^T k -> d -> S; the four waves of a CU, by the LDS reads of the token's k and q: with two columns to a lane
// those are KT / 8 values of each where a lane with one column reads twice as many. What is not the recurrence leaves the
// step: the waves of a workgroup, which own neighbouring columns of the same head, load a group of tokens ahead, widen q, k
// and v and park them in LDS together, and the per-token scalars (1 / |k|, scale / |q|, e^g, beta) are made with them: the
// squares are summed where the pieces of a row sit in neighbouring lanes, the decays scanned with lane = token. The l2 norms
// are applied as factors on the sums, not on the vectors. K a multiple of 4, q and k 16-byte aligned.
// Against two row groups, 32 columns and a workgroup per wave (us, 64 tokens, states in and out): 16 x 8 x 64 x 64 bf16
// 32.8 -> 20.7 (one token 8.0 -> 5.8), 32 x 4 x 128 x 128 110 -> 32, 128 x 8 x 64 x 64 82 -> 54, 40 x 6 x 32 x 64 fp32
// 20.8 -> 16.3, 128 x 8 x 16 x 32 17.5 -> 16.1. (Groups of 16 or 64 tokens at K = 16, four row groups of 32 columns a wave: slower.)
// x summed over aligned runs of N lanes, in every lane
template <int N>
__device__ __forceinline__ float rec_run_sum(float x) {
  x += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, x);
  x += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, x);
  if constexpr (N >= 8) x += dpp_f32<0x141, 0xF>(0.0f, x);   // row_half_mirror: the other quad of the 8
  if constexpr (N >= 16) x += dpp_f32<0x140, 0xF>(0.0f, x);  // row_mirror: the other 8 of the 16
  if constexpr (N >= 32) {
    const unsigned u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return x;
}

template <bool B>
struct RecLazy {
  static constexpr bool value = B;
};

// four elements as they come from memory, and widened
template <typename T>
struct RecRaw4 {
  typedef T type __attribute__((ext_vector_type(4)));
};
template <typename T>
__device__ __forceinline__ float4 rec_widen4(typename RecRaw4<T>::type x) {
  return make_float4(GdrElem<T>::to_float(x[0]), GdrElem<T>::to_float(x[1]), GdrElem<T>::to_float(x[2]),
                     GdrElem<T>::to_float(x[3]));
}

// COMPOSITE: the affine map of the sequence instead of its outputs. The state of a gated delta sequence is affine in
// the state it starts from, S_end = M S_0 + N: the wave's columns are columns of [M | N] (V = K + the value width),
// started from [I | 0], the M columns see v = 0; nothing is written but ht (fp32 [n_seq, HV, K, V]). ht_map (nullable)
// gives the row of ht that a sequence's final state goes to (negative: not stored).
template <typename T, int KT, int WAVES, bool COMPOSITE>
__global__ void __launch_bounds__(64 * WAVES, 2)
    gdr_recurrent_split_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                               const float* __restrict__ g, const float* __restrict__ beta, T* __restrict__ o,
                               const float* __restrict__ h0, float* __restrict__ ht,
                               const int64_t* __restrict__ cu_seqlens, int64_t t_len, int H, int HV, int K, int V,
                               float scale, int l2norm, const int32_t* __restrict__ ht_map, float lazy_span) {
  // Heads of 16 rows, and of 32 where a workgroup has two waves, give a lane a quarter of the rows of one column: with two
  // columns of two or four rows the sums over the lanes were the larger part of a step (64 tokens: 128 x 8 x 16 x 32 fp32
  // 18.7 -> 16.2 us, 64 x 8 x 16 x 128 29.1 -> 25.7, 128 x 8 x 32 x 32 22.9 -> 20.4). At K = 32 with four waves it is slower
  // (one token, 128 x 8 x 32 x 128 15.6 -> 17.1: a lane with one column reads twice as much of k and q from LDS).
  constexpr int NC = KT == 16 || (KT == 32 && WAVES == 2) ? 1 : 2;  // columns of a lane
  constexpr int RG = 4 * NC, WCOLS = 16;        // row groups and columns of a wave
  constexpr int NT = 64 * WAVES, COLS = WCOLS * WAVES;
  constexpr int RP = KT / RG;                   // state rows per lane
  constexpr int CHAINS = NC == 1 && RP >= 8 ? 2 : 1;  // sums a lane adds its rows in (two, where one would be of eight: the error)
  // Tokens per group. A workgroup of two waves (V <= 32) stages as much of k and q as one of four: with 32 tokens at K = 64 it
  // held 47 KB, three were all that a CU had room for, and 1 024 took two rounds (128 x 8 x 64 x 32 fp32, 64 tokens 48 us, one
  // 11; with 16 tokens 33 and 8.3).
  constexpr int G = KT < 64 || (KT == 64 && WAVES > 2) ? 32 : 16;
  constexpr int P = KT / 4;                     // 4-element pieces of a row of k
  constexpr int ROW4 = (2 * KT + 4) / 4;        // 16-byte pieces per token in LDS: k | q, padded against conflicts
  constexpr int PIECES = (G * P + NT - 1) / NT; // pieces of k (and of q) per thread and group
  constexpr int VALS = G * COLS / NT;           // v elements per thread and group
  static_assert((G * P) % NT == 0 || G * P < NT, "group shape");
  // two buffers of a group each; two more tokens' room behind each group, so that the reads ahead need no bound
  // (what they return for tokens after the group is never used)
  __shared__ float4 s_kq[2][(G + 2) * ROW4];
  __shared__ float4 s_sc[2][G + 2];
  __shared__ float s_v[2][(G + 2) * COLS];
  __shared__ T s_o[COMPOSITE ? 1 : G * COLS];  // o of a group, stored behind its last step
  static_assert(KT > 64 || (sizeof(s_kq) + sizeof(s_sc) + sizeof(s_v) + sizeof(s_o)) * 8 / WAVES <= 160 * 1024, "eight waves to a CU");
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, rg = lane % RG, cl = WCOLS * wave + NC * (lane / RG);
  const int wcol = (int)blockIdx.x * COLS, col = wcol + cl;  // (the first of) this lane's columns
  const int seq = blockIdx.y / HV, hv = blockIdx.y % HV;
  const int h = hv / (HV / H);
  const int64_t bos = cu_seqlens ? cu_seqlens[seq] : seq * t_len;
  const int64_t eos = cu_seqlens ? cu_seqlens[seq + 1] : bos + t_len;

  const int v_dim = COMPOSITE ? V - K : V;  // width of a row of v
  const bool even = V % 2 == 0 && ((reinterpret_cast<uintptr_t>(h0) | reinterpret_cast<uintptr_t>(ht)) & 7) == 0;  // columns in pairs
  float S[NC][RP];  // rows rg * RP + r
#pragma unroll
  for (int r = 0; r < RP; ++r) {
    const int i = rg * RP + r;
    if constexpr (COMPOSITE) {
#pragma unroll
      for (int c = 0; c < NC; ++c) S[c][r] = (i == col + c && i < K) ? 1.0f : 0.0f;
    } else {
      const float* at = h0 + (((int64_t)seq * HV + hv) * K + i) * V + col;
      float2 x = make_float2(0.0f, 0.0f);
      if (h0 && i < K && col < V) {
        if (NC == 1) x.x = at[0];
        else if (even) x = *reinterpret_cast<const float2*>(at);
        else x = make_float2(at[0], col + 1 < V ? at[1] : 0.0f);
      }
      S[0][r] = x.x;
      if constexpr (NC == 2) S[NC - 1][r] = x.y;
    }
  }
  if (bos < eos) {
    using Raw = typename RecRaw4<T>::type;
    Raw kp[PIECES], qp[COMPOSITE ? 1 : PIECES];  // (as they come: a conversion here would wait for the loads)
    T vals[VALS];
    float g_tok = 0.0f, b_tok = 0.0f;
    // loads of the group that starts at token t0: every address is inside the tensors (tokens past the end re-read the
    // last one, elements past K or V the last element) and what is out of range is replaced when it is parked. Uniform
    // base pointers and 32-bit offsets, the same for every whole group.
    int k_off[PIECES], v_off[VALS], g_off;
    auto offsets = [&](int last) __attribute__((always_inline)) {  // last: the group's last token that exists
#pragma unroll
      for (int n = 0; n < PIECES; ++n) {
        const int pi = tid + NT * n, c = 4 * (pi % P);
        k_off[n] = min(pi / P, last) * (H * K) + (c < K ? c : K - 4);
      }
#pragma unroll
      for (int n = 0; n < VALS; ++n) {
        const int vi = tid + NT * n, cc = wcol + vi % COLS - (COMPOSITE ? K : 0);
        v_off[n] = min(vi / COLS, last) * (HV * v_dim) + max(0, min(cc, v_dim - 1));
      }
      g_off = min(lane, last) * HV;
    };
    auto fetch = [&](int64_t t0) __attribute__((always_inline)) {
      const int64_t left = eos - t0;
      if (left < G) offsets((int)left - 1);
      const T* kb = k + (t0 * H + h) * K;
      const T* qb = q + (t0 * H + h) * K;
      const T* vb = v + (t0 * HV + hv) * v_dim;
#pragma unroll
      for (int n = 0; n < PIECES; ++n) {
        if (n > 0 && n * NT / P >= left) break;  // (a few tokens in all: nothing there)
        kp[n] = *reinterpret_cast<const Raw*>(kb + (unsigned)k_off[n]);
        if constexpr (!COMPOSITE) qp[n] = *reinterpret_cast<const Raw*>(qb + (unsigned)k_off[n]);
      }
#pragma unroll
      for (int n = 0; n < VALS; ++n) {
        if (n > 0 && n * NT / COLS >= left) break;
        vals[n] = vb[(unsigned)v_off[n]];
      }
      g_tok = g[t0 * HV + hv + (unsigned)g_off];
      b_tok = beta[t0 * HV + hv + (unsigned)g_off];
    };
    offsets(G - 1);
    // the fetched group, which starts at t0, into LDS buffer `buf`, with its per-token scalars.
    // The decay is not applied to the state token by token: within a run of eight tokens the registers hold S / c_j, c_j =
    // the decay from the run's start up to token j, and c_j goes into the token's scalars instead (a multiply per state
    // element and token less); the state is brought back to scale after the run. (Runs as long as the group, 16 to 64 tokens,
    // cost nothing less and up to 2.5 times the error against 64 bits, from the rounding of the longer sums in e^.) A group
    // with more than e^lazy_span of decay (or growth) in one of its runs takes the direct form: beyond e^60 1 / c_j would leave
    // the fp32 range; below zero every group does. c_run: of lane 8 r + 7, the decay over run r.
    float c_run = 1.0f;
    bool lazy = false;
    auto commit = [&](int64_t t0, int buf) __attribute__((always_inline)) {
      const float g_use = (lane < G && t0 + lane < eos) ? g_tok : 0.0f;  // (lane = token; every wave for itself)
      float cum = g_use;
      const float up1 = dpp_f32<GDR_DPP_ROW_SHR(1), 0xF>(0.0f, cum);  // (every lane enabled)
      cum += (lane & 7) >= 1 ? up1 : 0.0f;
      const float up2 = dpp_f32<GDR_DPP_ROW_SHR(2), 0xF>(0.0f, cum);
      cum += (lane & 7) >= 2 ? up2 : 0.0f;
      const float up4 = dpp_f32<GDR_DPP_ROW_SHR(4), 0xF>(0.0f, cum);
      cum += (lane & 7) >= 4 ? up4 : 0.0f;
      lazy = __ballot(!(rec_run_sum<8>(fabsf(g_use)) <= lazy_span)) == 0;  // (false for a NaN as well)
      const float c_tok = expf(lazy ? cum : g_tok), rc_tok = lazy ? expf(-cum) : 1.0f;
      c_run = c_tok;
#pragma unroll
      for (int n = 0; n < PIECES; ++n) {
        if (n > 0 && n * NT / P > eos - t0) break;  // (one token past an odd count is read as a step)
        const int pi = tid + NT * n, j = min(pi / P, G - 1), c4 = pi % P;
        const bool live = t0 + j < eos;
        // a token past the end is a step that changes nothing (d = 0, decay 1), so the steps need no branch
        const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float4 a = live && 4 * c4 < K ? rec_widen4<T>(kp[n]) : zero;
        float4 b = zero;
        if constexpr (!COMPOSITE) b = live && 4 * c4 < K ? rec_widen4<T>(qp[n]) : zero;
        const float kss = rec_run_sum<P>(a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w);
        const float qss = COMPOSITE ? 0.0f : rec_run_sum<P>(b.x * b.x + b.y * b.y + b.z * b.z + b.w * b.w);
        const float c = __shfl(c_tok, j), rc = __shfl(rc_tok, j), bt = __shfl(b_tok, j);
        float kinv = 1.0f, qinv = 1.0f;
        if (l2norm == GDR_L2_CHUNK) {
          kinv = 1.0f / __fsqrt_rn(kss + 1e-6f);
          qinv = 1.0f / __fsqrt_rn(qss + 1e-6f);
        } else if (l2norm == GDR_L2_RECURRENT) {
          kinv = 1.0f / (__fsqrt_rn(kss) + 1e-6f);
          qinv = 1.0f / (__fsqrt_rn(qss) + 1e-6f);
        }
        if (G * P >= NT || pi < G * P) {
          s_kq[buf][j * ROW4 + c4] = a;
          if constexpr (!COMPOSITE) s_kq[buf][j * ROW4 + P + c4] = b;
          // direct: 1 / |k|, scale / |q|, e^g, beta; lazy: c / |k|, c scale / |q|, 1 / (c |k|), beta
          float4 sc = lazy ? make_float4(kinv * c, qinv * scale * c, kinv * rc, bt) : make_float4(kinv, qinv * scale, c, bt);
          if (!live) sc = make_float4(0.0f, 0.0f, lazy ? 0.0f : 1.0f, 0.0f);
          if (c4 == 0) s_sc[buf][j] = sc;
        }
      }
#pragma unroll
      for (int n = 0; n < VALS; ++n) {
        if (n > 0 && n * NT / COLS > eos - t0) break;
        const int vi = tid + NT * n, cc = wcol + vi % COLS - (COMPOSITE ? K : 0);
        s_v[buf][vi] = (t0 + vi / COLS >= eos || (COMPOSITE && cc < 0)) ? 0.0f : GdrElem<T>::to_float(vals[n]);
      }
    };
    // a token's operands: its scalars, this lane's RP elements of k and of q, the v of its columns
    struct Operands {
      float4 sc;
      float kk[RP], qq[COMPOSITE ? 1 : RP];
      float v[NC];
    };
    auto read_row = [&](const float* p, float* to) __attribute__((always_inline)) {
      if constexpr (RP == 2) {
        const float2 x = *reinterpret_cast<const float2*>(p);
        to[0] = x.x; to[1] = x.y;
      } else {
#pragma unroll
        for (int r = 0; r < RP; r += 4) {
          const float4 x = *reinterpret_cast<const float4*>(p + r);
          to[r] = x.x; to[r + 1] = x.y; to[r + 2] = x.z; to[r + 3] = x.w;
        }
      }
    };
    auto read_token = [&](int buf, int j, Operands& x) __attribute__((always_inline)) {
      x.sc = s_sc[buf][j];  // the token's four scalars (direct or lazy form, see commit)
      const float* kr = reinterpret_cast<const float*>(&s_kq[buf][j * ROW4]) + rg * RP;
      read_row(kr, x.kk);
      if constexpr (!COMPOSITE) read_row(kr + KT, x.qq);
      if constexpr (NC == 2) {
        const float2 v2 = *reinterpret_cast<const float2*>(&s_v[buf][j * COLS + cl]);
        x.v[0] = v2.x; x.v[NC - 1] = v2.y;
      } else {
        x.v[0] = s_v[buf][j * COLS + cl];
      }
    };
    fetch(bos);
    commit(bos, 0);
    lds_barrier();
    // o of a group goes through LDS (the first NC row groups write the first of two tokens, the next the second) and leaves behind
    // the commit of the next group: stored token by token, the wait for that group's loads would be one for the stores too,
    // 2 us a group.
    const int o_tok = (rg / NC) & 1;
    T* const so = s_o + o_tok * COLS + cl + rg % NC;
    auto flush = [&](int64_t t0, int n_tok) __attribute__((always_inline)) {
      if constexpr (!COMPOSITE) {
        const int c = WCOLS * wave + lane % WCOLS, j0 = lane / WCOLS;  // this wave's columns, four tokens at a time
        T* ob = o + (t0 * HV + hv) * V + wcol;
        const unsigned at = (unsigned)(j0 * (HV * V) + c), step = (unsigned)(64 / WCOLS * HV * V);
#pragma unroll
        for (int n = 0; n < G * WCOLS / 64; ++n) {
          if (n * (64 / WCOLS) >= n_tok) break;
          const T x = s_o[(n * (64 / WCOLS) + j0) * COLS + c];
          if (n * (64 / WCOLS) + j0 < n_tok && wcol + c < V) ob[at + n * step] = x;
        }
      }
    };
    int buf = 0;
    for (int64_t t0 = bos; t0 < eos; t0 += G, buf ^= 1) {
      const bool more = t0 + G < eos;
      if (more) fetch(t0 + G);
      const int n_tok = eos - t0 < G ? (int)(eos - t0) : G;
      // two tokens per round on two operand sets: a token's operands are requested before the arithmetic of the token
      // before it starts, so their LDS latency hides behind it. The token after the last of an odd count is a step
      // that changes nothing.
      auto run_group = [&](auto lazy_tag) __attribute__((always_inline)) {
        constexpr bool LAZY = decltype(lazy_tag)::value;
        auto step = [&](const Operands& x) __attribute__((always_inline)) {
          float d[NC], dk[NC], out[NC];
          const float4 sc = x.sc;
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            float part[CHAINS];
#pragma unroll
            for (int r = 0; r < RP; ++r)
              part[r % CHAINS] = r < CHAINS ? S[c][r] * x.kk[r] : __builtin_fmaf(S[c][r], x.kk[r], part[r % CHAINS]);
            d[c] = CHAINS == 2 ? part[0] + part[CHAINS - 1] : part[0];
          }
#pragma unroll
          for (int c = 0; c < NC; ++c) d[c] = rec_run_sum<RG>(d[c]);
          // S <- e^g S, then d = beta (v - S^T k), S <- S + k d^T, o = S^T q, with k = k_raw / |k|; in the lazy form on
          // S / c_j, where the decay is part of the scalars
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const float dc = LAZY ? sc.w * (x.v[c] - sc.x * d[c]) : sc.w * (x.v[c] - sc.z * sc.x * d[c]);
            dk[c] = LAZY ? dc * sc.z : dc * sc.x;
          }
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            float part[CHAINS];
#pragma unroll
            for (int r = 0; r < RP; ++r) {
              S[c][r] = __builtin_fmaf(x.kk[r], dk[c], LAZY ? S[c][r] : sc.z * S[c][r]);
              if constexpr (!COMPOSITE)
                part[r % CHAINS] = r < CHAINS ? S[c][r] * x.qq[r] : __builtin_fmaf(S[c][r], x.qq[r], part[r % CHAINS]);
            }
            if constexpr (!COMPOSITE) out[c] = CHAINS == 2 ? part[0] + part[CHAINS - 1] : part[0];
          }
          if constexpr (COMPOSITE) return 0.0f;
          else {
#pragma unroll
            for (int c = 0; c < NC; ++c) out[c] = rec_run_sum<RG>(out[c]);
            return (rg % NC ? out[NC - 1] : out[0]) * sc.y;
          }
        };
        Operands xa, xb;
        read_token(buf, 0, xa);
#pragma unroll 1
        for (int run = 0; run < n_tok; run += 8) {
          const int end = min(n_tok, run + 8);
#pragma unroll 1
          for (int j = run; j < end; j += 2) {
            read_token(buf, j + 1, xb);
            __builtin_amdgcn_sched_barrier(0);
            const float oa = step(xa);
            read_token(buf, j + 2, xa);
            __builtin_amdgcn_sched_barrier(0);
            const float ob = step(xb);
            if constexpr (!COMPOSITE) {
              if (rg < 2 * NC) so[j * COLS] = GdrElem<T>::from_float(o_tok ? ob : oa);
            }
          }
          if constexpr (LAZY) {
            const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c_run), run + 7));
#pragma unroll
            for (int r = 0; r < RP; ++r) {  // back to scale: S = c_last (S / c_last)
#pragma unroll
              for (int x = 0; x < NC; ++x) S[x][r] *= c;
            }
          }
        }
      };
      if (lazy) run_group(RecLazy<true>{});
      else run_group(RecLazy<false>{});
      if (more) {
        commit(t0 + G, buf ^ 1);  // (that buffer was last read before the barrier in front of this group)
        lds_barrier();
      } else {
        lds_fence();
      }
      flush(t0, n_tok);
    }
  }
  const int out_row = ht_map ? ht_map[seq] : seq;
  if (ht && out_row >= 0) {
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      const int i = rg * RP + r;
      float* at = ht + (((int64_t)out_row * HV + hv) * K + i) * V + col;
      if (i < K && col < V) {
        if (NC == 2 && even) *reinterpret_cast<float2*>(at) = make_float2(S[0][r], S[NC - 1][r]);
        else {
          at[0] = S[0][r];
          if (NC == 2 && col + 1 < V) at[1] = S[NC - 1][r];
        }
      }
    }
  }
}

// Launch of the split kernel over `n_seq` runs of tokens; V: all the wave's columns (COMPOSITE: K + the value width).
// lazy_form: whether groups of tokens may apply their decays lazily (see commit).
template <typename T, bool COMPOSITE>
static void gdr_split_launch(const void* q, const void* k, const void* v, const float* g, const float* beta, void* o,
                             const float* h0, float* ht, const int64_t* cu, int n_seq, int64_t t_len, int H, int HV, int K,
                             int V, float scale, int l2norm, const int32_t* ht_map, hipStream_t s,
                             bool lazy_form = true) {
#define GDR_REC_SPLIT(KT, WAVES)                                                                                         \
  hipLaunchKernelGGL((gdr_recurrent_split_kernel<T, KT, WAVES, COMPOSITE>),                                              \
                     dim3((V + 16 * WAVES - 1) / (16 * WAVES), n_seq * HV), dim3(64 * WAVES), 0, s, (const T*)q,         \
                     (const T*)k, (const T*)v, g, beta, (T*)o, h0, ht, cu, t_len, H, HV, K, V, scale, l2norm, ht_map,   \
                     lazy_form ? 60.0f : -1.0f)
#define GDR_REC_SPLIT_K(WAVES)                  \
  do {                                          \
    if (K <= 16) GDR_REC_SPLIT(16, WAVES);      \
    else if (K <= 32) GDR_REC_SPLIT(32, WAVES); \
    else if (K <= 64) GDR_REC_SPLIT(64, WAVES); \
    else GDR_REC_SPLIT(128, WAVES);             \
  } while (0)
  if (V <= 32) GDR_REC_SPLIT_K(2);
  else GDR_REC_SPLIT_K(4);
#undef GDR_REC_SPLIT_K
#undef GDR_REC_SPLIT
}

template <typename T>
static int gdr_recurrent_launch(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                void* o, const float* h0, float* ht, const int64_t* cu, int n_seq, int64_t t_len,
                                int H, int HV, int K, int V, float scale, int l2norm, hipStream_t s) {
  LAMPA_PROF(s, "start");
  // The split form, but for one or two tokens each of very many sequences at K = 64 (a third of the registers, so more loads
  // of the states in flight: 1 024 x 8 x 64 x 64, one token 73 against 86 us, two 82 against 89, four 100 against 98; at half
  // as many sequences 37 against 44, a quarter 26 against 24; at K = 16, 32 and 128 the split form is faster throughout).
  const int64_t waves = (int64_t)((V + 31) / 32) * n_seq * HV, tokens = cu ? t_len / n_seq : t_len;
  const bool few_of_many = K > 32 && K <= 64 && tokens <= 2 && waves > 4096;
  // Launches of more than 2 048 waves of 32 columns take the direct form, the state times each token's own e^g as the lane-per-
  // column kernel has it. The lazy one takes ratios of decays from e^ of their sums: against 64 bits (64 tokens, K 16 to 128) its
  // states are 3.3 times as far off at e^-0.8 a token, 1.4 times at e^-0.24, 0.84 times at e^-0.04, and 5.9 times at e^-2.4; the
  // direct form's, 1.00 times. It costs a multiply per state element and token (fp32: 512 x 64 x 8 x 32 x 32 83 -> 87 us,
  // 128 x 64 x 8 x 128 x 128 182 -> 198, 1 024 x 64 x 8 x 64 x 64 383 -> 411; a lane per column 135, 285, 474). Smaller launches
  // are bound by the chain of a step; the two row groups that they took before were lazy over 8 to 64 tokens, and further off.
  if (K % 4 == 0 && ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) & 15) == 0 && !few_of_many) {
    gdr_split_launch<T, false>(q, k, v, g, beta, o, h0, ht, cu, n_seq, t_len, H, HV, K, V, scale, l2norm, nullptr, s,
                               waves <= 2048);
    LAMPA_PROF(s, "gdr_recurrent_split_kernel");
    return lampa_launch_status();
  }
  const dim3 grid((V + 63) / 64, n_seq * HV), block(64);
#define GDR_REC_CASE(KT)                                                                                         \
  hipLaunchKernelGGL((gdr_recurrent_kernel<T, KT>), grid, block, 0, s, (const T*)q, (const T*)k, (const T*)v, g, \
                     beta, (T*)o, h0, ht, cu, t_len, H, HV, K, V, scale, l2norm)
  if (K <= 32) GDR_REC_CASE(32);
  else if (K <= 64) GDR_REC_CASE(64);
  else GDR_REC_CASE(128);
#undef GDR_REC_CASE
  LAMPA_PROF(s, "gdr_recurrent_kernel");
  return lampa_launch_status();
}

// ---- long sequences in parallel ---------------------------------------------------------------------------------
// A token-serial kernel gives a (sequence, head) to one or two waves, so a few long sequences leave the chip idle. The
// state a run of tokens ends with is affine in the state it starts from, so the sequences are cut into segments:
//   A  every segment's map [M | N] from [I | 0]            (gdr_recurrent_split_kernel<COMPOSITE>, K + V columns)
//   S  S_{p+1} = M_p S_p + N_p over a sequence's segments  (gdr_segment_scan_kernel, serial, small)
//   B  every segment again from the state it really starts with, writing o (the plain kernel, segments as sequences)
// all in fp32: the same function as the token loop up to fp32 rounding.

// 16 columns of the state per workgroup; mn [n_seg, HV, K, K + V], sinit [n_seg, HV, K, V]. A step is a chain, so nothing
// else may be on it:
//  - M_p S runs on the fp32 MFMA (v_mfma_f32_16x16x4f32), with S in the accumulators it comes out in: register r of row
//    tile t of lane 16 g + j is row 16 t + 4 g + r of column j, which is what the next product wants as its B operand if it
//    takes the contraction index 16 t + 4 g + r in its step (t, r); the A operand of the four steps r is then one 16-byte
//    piece of a row of M_p, from memory straight to registers. A wave owns a row tile, and the tiles are exchanged through
//    LDS (double-buffered, one barrier per step) behind the wave's own four products;
//  - the maps are loaded DEPTH steps ahead into register sets that are fixed per step of an unrolled group (moving a set
//    would wait for its load), and every memory operation of a step is unconditional (under a condition it becomes a branch,
//    after which the compiler no longer counts the operations in flight and drains them).
// Before, with M through LDS, 32 columns per workgroup of four waves and three launches, 32 us of a call of 8 192 x 4 x 32 x 32
// tokens in 128 segments; now 5 + 10. (All rows on one wave up to K = 32: 7 + 15; eight steps of maps ahead instead of four:
// 8 + 16.) In the 256 segments that the operator makes of it 8 + 14, for 14 + 13 instead of 16 + 20 in the two other passes.
typedef float rs_f32x4 __attribute__((ext_vector_type(4)));
enum { RS_FINITE = 1, RS_ZERO = 2, RS_NOTE_LOADS = 4 };
template <int KT>
struct RsScanShape {
  static constexpr int NT = KT / 16;  // row tiles, a wave each
  static constexpr int DEPTH = 4;
};

// COMPOSE: workgroup (blockIdx.y = seq * maxg + grp) = group `grp` (gs consecutive segments) of sequence `seq`, on the K + V
// columns of [I | 0]: every map of the group is applied and the result, the group's own map [M | N], stored (V counts all
// K + V columns). Otherwise: the state every segment of the group starts from; a group in front of which there are others
// walks their maps (gmaps) first. A long sequence is scanned in groups of about sqrt(n / 2) segments, two launches of at
// most sqrt(2 n) dependent steps, any other as one group (gs >= its segments, maxg = 1) in one.
template <int KT, bool COMPOSE>
__global__ void __launch_bounds__(64 * RsScanShape<KT>::NT)
    gdr_segment_scan_kernel(const float* __restrict__ mn, const float* __restrict__ gmaps, const float* __restrict__ h0,
                            const int32_t* __restrict__ seq_seg0, int HV, int K, int V, float* __restrict__ out, int gs,
                            int maxg, int W, int* __restrict__ notes) {
  constexpr int NT = RsScanShape<KT>::NT, DEPTH = RsScanShape<KT>::DEPTH;
  __shared__ rs_f32x4 s_x[2][NT][64];
  __shared__ int s_note[NT];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g4 = lane >> 4, j16 = lane & 15;
  const int hv = blockIdx.z, seq = blockIdx.y / maxg, grp = blockIdx.y - seq * maxg;
  const int seg0 = seq_seg0[seq], seg1 = seq_seg0[seq + 1];
  const int p0 = seg0 + grp * gs, cnt = min(gs, seg1 - p0);  // this group's segments
  if (cnt <= 0 || (COMPOSE && p0 + gs >= seg1)) return;       // (no one asks for the map of a sequence's last group)
  const int lead = COMPOSE ? 0 : grp, n_apply = lead + (COMPOSE ? cnt : cnt - 1);
  // A row tile wholly past K (K = 36 .. 48, 68 .. 112): zeros for the products of the other waves, and their barriers. It may
  // not shadow rows of another tile as the lanes below do: a wave sums its own columns first, so it would store other last
  // bits to the same place, with no order between the two.
  if (16 * wave >= K) {
    s_x[0][wave][lane] = s_x[1][wave][lane] = rs_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int p = 0; p < n_apply; ++p) lds_barrier();
    return;
  }
  // Lanes past V shadow the last column, rows past K the last rows of the same place in their run of four, all in the same
  // wave: they load, compute and store the same as those. What they feed into a product is met by a zero of M.
  const int col = min((int)blockIdx.x * 16 + j16, V - 1);
  const bool is_m = COMPOSE && col < K;  // (a column of M: no additive term, starts from I)
  const int ncol = COMPOSE ? max(col - K, 0) : col;
  auto row_of = [&](int i) { return i < K ? i : K - 4 + (i & 3); };
  // offsets of this lane's 16-byte pieces of M (its tile's row j16; own tile's columns first) and of its four rows
  unsigned m_at[NT], row[4];
  bool inside[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int c = 16 * ((wave + t) % NT) + 4 * g4;
    inside[t] = c < K;
    m_at[t] = (unsigned)(row_of(16 * wave + j16) * W + min(c, K - 4));
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) row[r] = (unsigned)row_of(16 * wave + 4 * g4 + r);

  struct Set {
    rs_f32x4 m[NT];
    float n[4];
  };
  Set set[DEPTH];
  auto fetch = [&](int p, Set& x) __attribute__((always_inline)) {
    p = min(p, n_apply - 1);
    const float* M = p < lead ? gmaps + ((int64_t)(seq * maxg + p) * HV + hv) * K * W
                              : mn + ((int64_t)(p0 + p - lead) * HV + hv) * K * W;
#pragma unroll
    for (int t = 0; t < NT; ++t) x.m[t] = *reinterpret_cast<const rs_f32x4*>(M + m_at[t]);
#pragma unroll
    for (int r = 0; r < 4; ++r) x.n[r] = M[row[r] * W + K + ncol];
  };
  rs_f32x4 S;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (COMPOSE) S[r] = (is_m && (int)row[r] == col) ? 1.0f : 0.0f;
    else S[r] = h0 ? h0[(((int64_t)seq * HV + hv) * K + row[r]) * V + col] : 0.0f;
  }
  // Notes of the groups' maps, [HV][sequence][group][16 columns]: RS_FINITE, all entries are; RS_ZERO, those of M are zero. A
  // group behind maps that all are finite, the last of them without M (decays beyond the fp32 range), starts behind that one, on
  // the initial state as it is: 8 192 tokens x 4 at e^-0.8 a token, 32 x 32: scan 12.5 -> 7.4 us, call 45.1 -> 40.0; at
  // e^-0.04, where no map is zero, 45.7 -> 46.1, 64 x 64 93.1 -> 93.4. (Behind fewer than two groups there is nothing to leave out, and a
  // word that no one writes is read in their place: the loads are unconditional.)
  const int nb = (W + 15) / 16, n_notes = lead > 1 ? lead * nb : 1;
  const int* const seen = lead > 1 ? notes + ((int64_t)hv * (gridDim.y / maxg) + seq) * maxg * nb : seq_seg0;
  int note[RS_NOTE_LOADS];
  if constexpr (!COMPOSE) {
#pragma unroll
    for (int x = 0; x < RS_NOTE_LOADS; ++x) note[x] = seen[min(lane + 64 * x, n_notes - 1)];
  }
  auto store = [&](int64_t at, int width) __attribute__((always_inline)) {
    float* to = out + (at * HV + hv) * K * width + col;
#pragma unroll
    for (int r = 0; r < 4; ++r) to[row[r] * width] = S[r];
  };
  auto advance = [&](int p, Set& x) __attribute__((always_inline)) {
    // (in front of the group's own segments: to the place of the first of them, which is written again)
    if (!COMPOSE) store(p0 + max(p - lead, 0), V);
    s_x[p & 1][wave][lane] = S;
    // two sums, so that a product does not wait for the one in front of it; N joins last (the smaller roundings)
    rs_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, more = acc, n;
#pragma unroll
    for (int r = 0; r < 4; ++r) n[r] = is_m ? 0.0f : x.n[r];
    auto products = [&](int t, const rs_f32x4& b) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        rs_f32x4& to = r & 1 ? more : acc;
        to = __builtin_amdgcn_mfma_f32_16x16x4f32(inside[t] ? x.m[t][r] : 0.0f, b[r], to, 0, 0, 0);
      }
    };
    products(0, S);
    lds_barrier();
    rs_f32x4 b[NT];
#pragma unroll
    for (int t = 1; t < NT; ++t) b[t] = s_x[p & 1][(wave + t) % NT][lane];
#pragma unroll
    for (int t = 1; t < NT; ++t) products(t, b[t]);
    S = (acc + more) + n;
    fetch(p + DEPTH, x);
  };
  auto walk = [&](int p) __attribute__((always_inline)) {
    for (; p + DEPTH <= n_apply; p += DEPTH) {  // DEPTH steps on fixed register sets
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) advance(p + d, set[d]);
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (p + d < n_apply) advance(p + d, set[d]);
  };
  if (n_apply > 0) {
    bool cut = false;
    if constexpr (!COMPOSE) {
      int all = RS_FINITE | RS_ZERO;
#pragma unroll
      for (int x = 0; x < RS_NOTE_LOADS; ++x) all &= note[x] | (lane + 64 * x < n_notes - nb ? RS_ZERO : 0);
      cut = lead > 1 && n_notes <= 64 * RS_NOTE_LOADS && __ballot(all != (RS_FINITE | RS_ZERO)) == 0;
    }
    // (the maps are requested behind the look: with the first ones beside it, and a walk of its own for either way, scan 13.40 us of
    // 8 192 tokens x 4 x 64 x 64 at e^-0.04 a token, so 12.40, without any look 12.26; at e^-0.8, 32 x 32, 7.9 and 7.1)
    const int first = cut ? lead - 1 : 0;
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fetch(first + d, set[d]);
    walk(first);
  }
  if (COMPOSE) store(blockIdx.y, W);
  else store(p0 + cnt - 1, V);
  if constexpr (COMPOSE) {
    bool finite = true, zero = true;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      finite &= S[r] * 0.0f == 0.0f;
      zero &= !is_m || S[r] == 0.0f;
    }
    const int mine = (__ballot(!finite) ? 0 : RS_FINITE) | (__ballot(!zero) ? 0 : RS_ZERO);
    if (lane == 0) s_note[wave] = mine;
    lds_barrier();  // (of the waves whose rows exist)
    if (threadIdx.x == 0) {
      int all = mine;
      for (int w = 1; 16 * w < K; ++w) all &= s_note[w];
      notes[(((int64_t)hv * (gridDim.y / maxg) + seq) * maxg + grp) * nb + blockIdx.x] = all;
    }
  }
}

template <typename T>
static int gdr_recurrent_segmented(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                   void* o, const float* h0, float* ht, const int64_t* cu_seg,
                                   const int32_t* seq_seg0, const int32_t* seg_out, int n_seq, int n_seg, int H, int HV,
                                   int K, int V, float scale, int l2norm, float* mn, float* sinit, float* groups,
                                   hipStream_t s) {
  LAMPA_PROF(s, "start");
  gdr_split_launch<T, true>(k, k, v, g, beta, nullptr, nullptr, mn, cu_seg, n_seg, 0, H, HV, K, K + V, scale, l2norm, nullptr, s);
  LAMPA_PROF(s, "gdr_recurrent_split_kernel<composite>");
  if (gdr_segment_scan(mn, h0, seq_seg0, n_seq, n_seg, HV, K, V, sinit, groups, s) != LAMPA_OK) return LAMPA_ERR_LAUNCH;
  LAMPA_PROF(s, "start");
  gdr_split_launch<T, false>(q, k, v, g, beta, o, sinit, ht, cu_seg, n_seg, 0, H, HV, K, V, scale, l2norm, seg_out, s);
  LAMPA_PROF(s, "gdr_recurrent_split_kernel");
  return lampa_launch_status();
}

// The first two launches above on their own, for the backward pass (gdr_backward.hip), which needs the maps and the
// states the segments start from but not the outputs; the scan is also run a second time there, over the transposed
// maps in reverse segment order.
int gdr_segment_maps(const void* k, const void* v, const float* g, const float* beta, const int64_t* cu_seg, int n_seg,
                     int H, int HV, int K, int V, int dtype, int l2norm, float* mn, hipStream_t s) {
  LAMPA_PROF(s, "start");
#define GDR_MAPS(T)                                                                                                      \
  gdr_split_launch<T, true>(k, k, v, g, beta, nullptr, nullptr, mn, cu_seg, n_seg, 0, H, HV, K, K + V, 1.0f, l2norm, nullptr, s)
  switch (dtype) {
    case GDR_BF16: GDR_MAPS(__bf16); break;
    case GDR_FP16: GDR_MAPS(_Float16); break;
    case GDR_FP32: GDR_MAPS(float); break;
    default: return LAMPA_ERR_INVALID;
  }
#undef GDR_MAPS
  LAMPA_PROF(s, "gdr_recurrent_split_kernel<composite>");
  return lampa_launch_status();
}

// Group slots of the two-launch scan: at most GDR_SCAN_GROUP_SEQS sequences of together at most GDR_SCAN_GROUP_SEGS
// segments take it; groups of gs = ceil(sqrt(n_seg / (2 n_seq))) segments, at most maxg = ceil(n_seg / gs) of them in a
// sequence however the segments are spread, so n_seq * maxg <= n_seq^1.5 sqrt(2 n_seg) + n_seq slots of a map [K, K + V].
#define GDR_SCAN_GROUP_SEQS 4
#define GDR_SCAN_GROUP_SEGS 4096
int64_t gdr_scan_group_floats(int n_seg, int HV, int K, int V) {
  if (n_seg > GDR_SCAN_GROUP_SEGS) return 0;
  int64_t root = 1;
  while (root * root < n_seg) ++root;
  return (12 * root + GDR_SCAN_GROUP_SEQS) * HV * (K * (int64_t)(K + V) + (K + V + 15) / 16);  // maps, then notes
}

int gdr_segment_scan(const float* mn, const float* h0, const int32_t* seq_seg0, int n_seq, int n_seg, int HV, int K,
                     int V, float* sinit, float* groups, hipStream_t s) {
  const int W = K + V;
#define GDR_REC_SCAN(KT, COMPOSE, GROUPS, COLS, OUT, GS, MAXG)                                                          \
  hipLaunchKernelGGL((gdr_segment_scan_kernel<KT, COMPOSE>), dim3((COLS + 15) / 16, n_seq * (MAXG), HV),                \
                     dim3(64 * RsScanShape<KT>::NT), 0, s, mn, GROUPS, h0, seq_seg0, HV, K, COLS, OUT, GS, MAXG, W, notes)
#define GDR_REC_SCAN_ANY(...)                        \
  do {                                               \
    if (K <= 16) GDR_REC_SCAN(16, __VA_ARGS__);      \
    else if (K <= 32) GDR_REC_SCAN(32, __VA_ARGS__); \
    else if (K <= 64) GDR_REC_SCAN(64, __VA_ARGS__); \
    else GDR_REC_SCAN(128, __VA_ARGS__);             \
  } while (0)
  LAMPA_PROF(s, "start");
  int gs = n_seg, maxg = 1;
  int* notes = nullptr;
  if (groups && n_seq <= GDR_SCAN_GROUP_SEQS && n_seg <= GDR_SCAN_GROUP_SEGS && n_seg >= 24 * n_seq) {
    gs = 1;
    while (2 * gs * gs * n_seq < n_seg) ++gs;
    maxg = (n_seg + gs - 1) / gs;
    notes = (int*)(groups + (int64_t)n_seq * maxg * HV * K * W);
    GDR_REC_SCAN_ANY(true, (const float*)nullptr, W, groups, gs, maxg);
    LAMPA_PROF(s, "gdr_segment_scan_kernel<compose>");
  }
  GDR_REC_SCAN_ANY(false, (const float*)groups, V, sinit, gs, maxg);
#undef GDR_REC_SCAN_ANY
#undef GDR_REC_SCAN
  LAMPA_PROF(s, "gdr_segment_scan_kernel");
  return lampa_launch_status();
}

// Workspace of lampa_gdr_recurrent_segmented_fwd: the segments' maps [n_seg, HV, K, K + V] and the states they start
// from [n_seg, HV, K, V], fp32.
extern "C" int64_t lampa_gdr_recurrent_segmented_workspace_bytes(int n_seg, int HV, int K, int V) {
  if (n_seg < 0 || HV < 1 || K < 1 || V < 1) return LAMPA_ERR_INVALID;
  return lampa_align_up((int64_t)n_seg * HV * K * (K + V) * 4, 256) + lampa_align_up((int64_t)n_seg * HV * K * V * 4, 256) +
         lampa_align_up(gdr_scan_group_floats(n_seg, HV, K, V) * 4, 256);
}

// lampa_gdr_recurrent_fwd for a few long sequences: the caller cuts every sequence into segments (cu_seg: device int64,
// n_seg + 1 token offsets, every sequence boundary among them; seq_seg0: device int32, n_seq + 1, first segment of
// every sequence; seg_out: device int32, n_seg, the sequence whose last segment this is, else -1) and the segments run
// in parallel. Same arguments and results otherwise; K and V multiples of 4, q and k 16-byte aligned, K <= 128.
extern "C" int lampa_gdr_recurrent_segmented_fwd(const void* q, const void* k, const void* v, const float* g,
                                                 const float* beta, void* o, const float* h0, float* ht,
                                                 const int64_t* cu_seg, const int32_t* seq_seg0, const int32_t* seg_out,
                                                 int n_seq, int n_seg, int H, int HV, int K, int V, int dtype,
                                                 float scale, int l2norm, void* workspace, int64_t workspace_bytes,
                                                 void* stream) {
  if (!q || !k || !v || !g || !beta || !o || !cu_seg || !seq_seg0 || !seg_out) return LAMPA_ERR_INVALID;
  if (n_seq < 0 || n_seg < n_seq || H < 1 || HV < H || HV % H != 0 || K < 1 || V < 1) return LAMPA_ERR_INVALID;
  if (l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (K > 128 || K % 4 != 0 || V % 4 != 0 ||
      ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) & 15) != 0)
    return LAMPA_ERR_UNSUPPORTED;
  if (n_seq == 0 || n_seg == 0) return LAMPA_OK;
  if (!workspace || workspace_bytes < lampa_gdr_recurrent_segmented_workspace_bytes(n_seg, HV, K, V))
    return LAMPA_ERR_WORKSPACE;
  float* mn = (float*)workspace;
  float* sinit = (float*)((char*)workspace + lampa_align_up((int64_t)n_seg * HV * K * (K + V) * 4, 256));
  float* groups = (float*)((char*)sinit + lampa_align_up((int64_t)n_seg * HV * K * V * 4, 256));
  if (gdr_scan_group_floats(n_seg, HV, K, V) == 0) groups = nullptr;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case GDR_BF16:
      return gdr_recurrent_segmented<__bf16>(q, k, v, g, beta, o, h0, ht, cu_seg, seq_seg0, seg_out, n_seq, n_seg, H,
                                             HV, K, V, scale, l2norm, mn, sinit, groups, s);
    case GDR_FP16:
      return gdr_recurrent_segmented<_Float16>(q, k, v, g, beta, o, h0, ht, cu_seg, seq_seg0, seg_out, n_seq, n_seg, H,
                                               HV, K, V, scale, l2norm, mn, sinit, groups, s);
    case GDR_FP32:
      return gdr_recurrent_segmented<float>(q, k, v, g, beta, o, h0, ht, cu_seg, seq_seg0, seg_out, n_seq, n_seg, H, HV,
                                            K, V, scale, l2norm, mn, sinit, groups, s);
    default:
      return LAMPA_ERR_INVALID;
  }
}

// q, k [total_tokens, H, K]; v, o [total_tokens, HV, V]; g, beta fp32 [total_tokens, HV]; h0, ht fp32
// [n_seq, HV, K, V] (nullable). Sequences are [cu_seqlens[i], cu_seqlens[i+1]) (device int64, n_seq + 1 entries) or,
// when cu_seqlens is NULL, n_seq blocks of t_len tokens. dtype: 0 bf16, 1 fp16, 2 fp32 (q, k, v and o).
// l2norm: 0 none, 1 x / sqrt(sum x^2 + 1e-6), 2 x / (sqrt(sum x^2) + 1e-6).
extern "C" int lampa_gdr_recurrent_fwd(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                       void* o, const float* h0, float* ht, const int64_t* cu_seqlens, int n_seq,
                                       int64_t t_len, int H, int HV, int K, int V, int dtype, float scale, int l2norm,
                                       void* stream) {
  if (!q || !k || !v || !g || !beta || !o) return LAMPA_ERR_INVALID;
  if (n_seq < 0 || H < 1 || HV < H || HV % H != 0 || K < 1 || V < 1 || t_len < 0) return LAMPA_ERR_INVALID;
  if (K > 128) return LAMPA_ERR_UNSUPPORTED;
  if (l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (n_seq == 0) return LAMPA_OK;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case GDR_BF16:
      return gdr_recurrent_launch<__bf16>(q, k, v, g, beta, o, h0, ht, cu_seqlens, n_seq, t_len, H, HV, K, V, scale,
                                          l2norm, s);
    case GDR_FP16:
      return gdr_recurrent_launch<_Float16>(q, k, v, g, beta, o, h0, ht, cu_seqlens, n_seq, t_len, H, HV, K, V,
                                            scale, l2norm, s);
    case GDR_FP32:
      return gdr_recurrent_launch<float>(q, k, v, g, beta, o, h0, ht, cu_seqlens, n_seq, t_len, H, HV, K, V, scale,
                                         l2norm, s);
    default:
      return LAMPA_ERR_INVALID;
  }
}

// The same operator with one beta per value column: beta fp32 [total_tokens, HV, V] (the reference kernel's
// IS_BETA_HEADWISE, gated_delta_rule_ori.py:415-418,444-448). Always the lane-per-column kernel: a lane owns one
// value column, so its beta is one more load per token.
template <typename T>
static int gdr_recurrent_headwise_launch(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                         void* o, const float* h0, float* ht, const int64_t* cu, int n_seq,
                                         int64_t t_len, int H, int HV, int K, int V, float scale, int l2norm,
                                         hipStream_t s) {
  LAMPA_PROF(s, "start");
  const dim3 grid((V + 63) / 64, n_seq * HV), block(64);
#define GDR_REC_CASE(KT)                                                                                              \
  hipLaunchKernelGGL((gdr_recurrent_kernel<T, KT, true>), grid, block, 0, s, (const T*)q, (const T*)k, (const T*)v, g, \
                     beta, (T*)o, h0, ht, cu, t_len, H, HV, K, V, scale, l2norm)
  if (K <= 32) GDR_REC_CASE(32);
  else if (K <= 64) GDR_REC_CASE(64);
  else GDR_REC_CASE(128);
#undef GDR_REC_CASE
  LAMPA_PROF(s, "gdr_recurrent_kernel<headwise beta>");
  return lampa_launch_status();
}

extern "C" int lampa_gdr_recurrent_headwise_fwd(const void* q, const void* k, const void* v, const float* g,
                                                const float* beta, void* o, const float* h0, float* ht,
                                                const int64_t* cu_seqlens, int n_seq, int64_t t_len, int H, int HV,
                                                int K, int V, int dtype, float scale, int l2norm, void* stream) {
  if (!q || !k || !v || !g || !beta || !o) return LAMPA_ERR_INVALID;
  if (n_seq < 0 || H < 1 || HV < H || HV % H != 0 || K < 1 || V < 1 || t_len < 0) return LAMPA_ERR_INVALID;
  if (K > 128) return LAMPA_ERR_UNSUPPORTED;
  if (l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (n_seq == 0) return LAMPA_OK;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case GDR_BF16:
      return gdr_recurrent_headwise_launch<__bf16>(q, k, v, g, beta, o, h0, ht, cu_seqlens, n_seq, t_len, H, HV, K, V,
                                                   scale, l2norm, s);
    case GDR_FP16:
      return gdr_recurrent_headwise_launch<_Float16>(q, k, v, g, beta, o, h0, ht, cu_seqlens, n_seq, t_len, H, HV, K,
                                                     V, scale, l2norm, s);
    case GDR_FP32:
      return gdr_recurrent_headwise_launch<float>(q, k, v, g, beta, o, h0, ht, cu_seqlens, n_seq, t_len, H, HV, K, V,
                                                  scale, l2norm, s);
    default:
      return LAMPA_ERR_INVALID;
  }
}
