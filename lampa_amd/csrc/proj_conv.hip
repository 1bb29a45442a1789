// Fused input projection + depthwise causal short convolution + SiLU of a gated-delta layer on gfx950 (bf16, MFMA).
//
// Replaces, for one layer call, the q / k / v / g / b / a projections (nn.Linear, bias-free) and the three
// ShortConvolution calls that follow the first three (reference chengjiang123/Lampa,
// models/hattention/modeling_gated_deltaproduct.py:505-547 and models/hattention/short_convolution.py:39-99):
//   pre[t, n] = sum_k x[t, k] W[n, k]                 (fp32 accumulate on the matrix cores, rounded to bf16 as a
//                                                      bf16 nn.Linear output is)
//   conv columns:  y[t, n] = silu(bias[n] + sum_j cw[n, j] pre[t - 3 + j, n]),  taps before a sequence start are zero
//   plain columns: y[t, n] = pre[t, n]
// The projection output never goes to HBM: x is read once (K = 128 columns), the outputs are written once.
//
// A workgroup is four waves of 64 output columns (256 of a job's columns x a run of consecutive tokens). A wave keeps its
// columns of W in registers for the whole run (2 column tiles x K/16 operand fragments) and walks it in tiles of 32
// tokens (32 rows of x straight from HBM, next tile prefetched). The product is computed transposed, W x^T: a lane then
// holds one token and four neighbouring columns per quarter of its accumulators, so a tile goes to a private LDS tile as
// 8-byte pieces (8 writes instead of 32 of 2 bytes, and packed conversions); below the last 3 pre-activation rows of the
// previous tile it is turned into outputs, so the convolution needs no recomputation except one extra tile at the start of
// a run that does not begin a sequence.
//
// Bound by VALU issue in the convolution's epilogue (4 fma and a SiLU with a quarter-rate exp2 and rcp per output), which the
// plain columns do not have, at two workgroups per CU (256 registers). On a long input every workgroup therefore takes a
// run of convolution columns, then a shorter run of plain columns and a tile of the few columns behind them: with workgroups
// of one kind each the CUs that held two of the convolution worked on while the others were done.
// 60 000 tokens, 2064 columns of which 1536 with the convolution: 107.5 us with workgroups of one kind, 101.8 us this way,
// 89.5 us since the rows of x requested ahead are not waited for together with the stores behind them (see `tile`).
#include "gdr_common.h"
#include <atomic>
#include <type_traits>

#define PC_K 128            // contraction length (hidden size) this kernel is built for
#define PC_NKS (PC_K / 16)
#define PC_W 4              // convolution taps
#define PC_COLS_WG 256
#define PC_COLS_WAVE 64
#define PC_ROWS 32
#define PC_ROWS_LANE 4     // consecutive token rows of a tile that one lane turns into outputs (8 columns each)
#define PC_LD (PC_COLS_WAVE + 8)  // LDS row stride in elements: 144 bytes, keeps 16-byte alignment
#define PC_MAX_BLOCKS 16

struct PcBlock {   // one block of 256 consecutive rows of W
  __bf16* out;     // output tensor of the block's columns
  int out_stride;  // its row stride in elements
  int out_col0;    // column of `out` that the block's first column maps to
};
// The workgroups wg0 .. wg0 + n_wgs - 1 do the runs of a kind's blocks: workgroup wg0 + i block i % n_blocks, run i / n_blocks
struct PcJobs {
  int wg0, n_wgs, n_blocks, tokens;  // tokens per run
};
struct PcPlan {
  PcBlock blocks[PC_MAX_BLOCKS];  // convolution blocks, then plain blocks
  PcJobs conv, plain, tail;       // tail: the last columns of W (fewer than a wave's 64); a wave takes one tile at a time
  __bf16* tail_out;
  int tail_cols;
};

__device__ __forceinline__ float pc_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// 64 rows of W, w0 .. (the first n_valid of them; zero beyond), as operand fragments
__device__ __forceinline__ void pc_load_w(const __bf16* __restrict__ W, int64_t w0, int n_valid, int lane,
                                          bf16x8 (*wf)[PC_NKS]) {
  const int hh = lane >> 5, ln = lane & 31;
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int c = 32 * ct + ln;
    const bool ok = c < n_valid;
    const __bf16* wp = W + (w0 + (ok ? c : 0)) * PC_K + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < PC_NKS; ++ks) {
      wf[ct][ks] = *reinterpret_cast<const bf16x8*>(wp + 16 * ks);
      if (!ok) {
#pragma unroll
        for (int e = 0; e < 8; ++e) wf[ct][ks][e] = (__bf16)0.0f;
      }
    }
  }
}

// 32 rows of x from t0 on (clamped to the tensor)
__device__ __forceinline__ void pc_load_x(const __bf16* __restrict__ x, int64_t x_stride, int64_t n_tokens, int64_t t0, int lane,
                                          bf16x8* a) {
  int64_t row = t0 + (lane & 31);
  row = row < 0 ? 0 : (row >= n_tokens ? n_tokens - 1 : row);
  const __bf16* xp = x + row * x_stride + 8 * (lane >> 5);
#pragma unroll
  for (int ks = 0; ks < PC_NKS; ++ks) a[ks] = *reinterpret_cast<const bf16x8*>(xp + 16 * ks);
}

// pre-activations of a tile, rounded to bf16, below the rows of history
__device__ __forceinline__ void pc_tile(const bf16x8 (*wf)[PC_NKS], const bf16x8* xf, int lane, __bf16* sy) {
  const int hh = lane >> 5, ln = lane & 31;
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < PC_NKS; ++ks) acc = mfma32(wf[ct][ks], xf[ks], acc);
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      bf16x4 p;
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = (__bf16)acc[4 * q4 + e];
      *reinterpret_cast<bf16x4*>(&sy[(PC_W - 1 + ln) * PC_LD + 32 * ct + 8 * q4 + 4 * hh]) = p;
    }
  }
}

__global__ void __launch_bounds__(256, 2) pc_proj_conv_kernel(const __bf16* __restrict__ x, int64_t x_stride, int64_t n_tokens,
                                                          int64_t t_len, const __bf16* __restrict__ W,
                                                          const float* __restrict__ conv_w, const float* __restrict__ conv_b,
                                                          const PcPlan plan) {
  __shared__ __align__(16) __bf16 s_y[4][(PC_ROWS + PC_W - 1) * PC_LD];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wcol = PC_COLS_WAVE * wave;  // first column of this wave inside a block
  // (no workgroup-wide barrier below: a wave uses nothing but its own LDS tile)
  __bf16* sy = s_y[wave];
  // output role of the lane: 8 consecutive columns (cg) of the 4 consecutive token rows 4 tq .. 4 tq + 3 of a tile
  const int cg = lane & 7, tq = lane >> 3, col = wcol + 8 * cg;
  bf16x8 wf[2][PC_NKS], xf[PC_NKS], xnext[PC_NKS];

  int job = (int)blockIdx.x - plan.conv.wg0;
  if (job >= 0 && job < plan.conv.n_wgs) {
    const int b = job % plan.conv.n_blocks;
    const PcBlock blk = plan.blocks[b];
    const int64_t T0 = (int64_t)(job / plan.conv.n_blocks) * plan.conv.tokens;
    const int64_t T1 = T0 + plan.conv.tokens < n_tokens ? T0 + plan.conv.tokens : n_tokens;
    pc_load_w(W, (int64_t)b * PC_COLS_WG + wcol, PC_COLS_WAVE, lane, wf);
    float cw[PC_W][8], cb[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      cb[c] = conv_b ? conv_b[b * PC_COLS_WG + col + c] : 0.0f;
#pragma unroll
      for (int j = 0; j < PC_W; ++j) cw[j][c] = conv_w[(int64_t)(b * PC_COLS_WG + col + c) * PC_W + j];
    }
    auto carry = [&]() __attribute__((always_inline)) {  // the last 3 rows become the history of the next tile
      lds_fence();
      for (int i = lane; i < (PC_W - 1) * (PC_COLS_WAVE / 8); i += 64) {
        const int r = i / (PC_COLS_WAVE / 8), c8 = i % (PC_COLS_WAVE / 8);
        *reinterpret_cast<bf16x8*>(&sy[r * PC_LD + 8 * c8]) =
            *reinterpret_cast<const bf16x8*>(&sy[(PC_ROWS + r) * PC_LD + 8 * c8]);
      }
      lds_fence();
    };
    // token position inside the sequence, kept per tile in 32 bits (a 64-bit modulo per output row would cost more than
    // the convolution); sequences shorter than two tiles take the general modulo
    const int tl32 = (int)(t_len < INT32_MAX ? t_len : INT32_MAX);
    const bool small_seq = t_len < 2 * PC_ROWS;
    int ts0 = (int)(T0 % t_len);
    if (ts0 != 0) {  // the run starts inside a sequence: the tile before it, for its last rows only
      pc_load_x(x, x_stride, n_tokens, T0 - PC_ROWS, lane, xf);
      pc_tile(wf, xf, lane, sy);
      carry();
    } else {
      for (int i = lane; i < (PC_W - 1) * PC_LD; i += 64) sy[i] = (__bf16)0.0f;
    }
    // whole: all 32 rows exist. Stores without a condition: with one the compiler no longer knows how many are in flight
    // and waits for all of them before it uses the rows of x that were requested ahead of them.
    auto tile = [&](auto whole, int64_t t0, const bf16x8* xc, bf16x8* xn) __attribute__((always_inline)) {
      pc_load_x(x, x_stride, n_tokens, t0 + PC_ROWS, lane, xn);
      pc_tile(wf, xc, lane, sy);
      lds_fence();
      // the lane's 4 consecutive tokens share their taps: 7 rows of pre-activations for 4 outputs
      float pre[PC_ROWS_LANE + PC_W - 1][8];
#pragma unroll
      for (int r = 0; r < PC_ROWS_LANE + PC_W - 1; ++r) {
        const bf16x8 row = *reinterpret_cast<const bf16x8*>(&sy[(PC_ROWS_LANE * tq + r) * PC_LD + 8 * cg]);
#pragma unroll
        for (int c = 0; c < 8; ++c) pre[r][c] = (float)row[c];
      }
      // tokens closer than 3 to the start of their sequence lose the taps that reach across it; a tile that holds no
      // such token (all but the first of a long sequence) skips the masks
      const bool interior = ts0 >= PC_W - 1 && ts0 + PC_ROWS <= tl32;
      __bf16* out = blk.out + (t0 + PC_ROWS_LANE * tq) * blk.out_stride + blk.out_col0 + col;
#pragma unroll
      for (int i = 0; i < PC_ROWS_LANE; ++i) {
        const int tr = PC_ROWS_LANE * tq + i;
        float y[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) y[c] = cb[c];
        if (interior) {
#pragma unroll
          for (int j = 0; j < PC_W; ++j)
#pragma unroll
            for (int c = 0; c < 8; ++c) y[c] = __builtin_fmaf(pre[i + j][c], cw[j][c], y[c]);
        } else {
          int ts = ts0 + tr;
          if (ts >= tl32) ts = small_seq ? ts % tl32 : ts - tl32;
#pragma unroll
          for (int j = 0; j < PC_W; ++j) {
            const bool live = ts - (PC_W - 1) + j >= 0;
#pragma unroll
            for (int c = 0; c < 8; ++c) y[c] = __builtin_fmaf(live ? pre[i + j][c] : 0.0f, cw[j][c], y[c]);
          }
        }
        bf16x8 o;
#pragma unroll
        for (int c = 0; c < 8; ++c) o[c] = (__bf16)(y[c] * pc_sigmoid(y[c]));
        if (decltype(whole)::value || t0 + tr < T1) *reinterpret_cast<bf16x8*>(out + i * (int64_t)blk.out_stride) = o;
      }
      carry();
      ts0 = small_seq ? (ts0 + PC_ROWS) % tl32 : (ts0 + PC_ROWS >= tl32 ? ts0 + PC_ROWS - tl32 : ts0 + PC_ROWS);
    };
    int64_t t0 = T0;
    pc_load_x(x, x_stride, n_tokens, t0, lane, xf);
    if (t0 + 3 * PC_ROWS <= T1) {
      // (the first tile on its own: then loads and stores are in flight in the same order at both ends of the loop)
      tile(std::true_type{}, t0, xf, xnext);
      t0 += PC_ROWS;
      for (; t0 + 2 * PC_ROWS <= T1; t0 += 2 * PC_ROWS) {
        tile(std::true_type{}, t0, xnext, xf);
        tile(std::true_type{}, t0 + PC_ROWS, xf, xnext);
      }
#pragma unroll
      for (int ks = 0; ks < PC_NKS; ++ks) xf[ks] = xnext[ks];
    }
    for (; t0 < T1; t0 += PC_ROWS) {  // at most two
      tile(std::false_type{}, t0, xf, xnext);
#pragma unroll
      for (int ks = 0; ks < PC_NKS; ++ks) xf[ks] = xnext[ks];
    }
  }

  job = (int)blockIdx.x - plan.plain.wg0;
  if (job >= 0 && job < plan.plain.n_wgs) {  // the projection output itself
    const int b = plan.conv.n_blocks + job % plan.plain.n_blocks;
    const PcBlock blk = plan.blocks[b];
    const int64_t T0 = (int64_t)(job / plan.plain.n_blocks) * plan.plain.tokens;
    const int64_t T1 = T0 + plan.plain.tokens < n_tokens ? T0 + plan.plain.tokens : n_tokens;
    pc_load_w(W, (int64_t)b * PC_COLS_WG + wcol, PC_COLS_WAVE, lane, wf);
    pc_load_x(x, x_stride, n_tokens, T0, lane, xf);
    auto tile = [&](auto whole, int64_t t0, const bf16x8* xc, bf16x8* xn) __attribute__((always_inline)) {
      pc_load_x(x, x_stride, n_tokens, t0 + PC_ROWS, lane, xn);
      pc_tile(wf, xc, lane, sy);
      lds_fence();
#pragma unroll
      for (int i = 0; i < PC_ROWS_LANE; ++i) {
        const int tr = PC_ROWS_LANE * tq + i;
        const bf16x8 o = *reinterpret_cast<const bf16x8*>(&sy[(tr + PC_W - 1) * PC_LD + 8 * cg]);
        const int64_t t = t0 + tr;
        // (non-temporal: these columns, a layer's output gate, are read after its gated-delta kernels, in front of which they
        // would take the place of q, k and v in the caches. The block, 60 000 tokens, 4 layers:
        // 1 196 -> 1 167 us, kernels of 20 000 629 -> 628, of 6 000 437 -> 435; with the convolution's columns as well
        // 1 179, with those alone 1 179, and the gate and o read with the hint 1 178)
        if (decltype(whole)::value || t < T1)
          __builtin_nontemporal_store(o, reinterpret_cast<bf16x8*>(blk.out + t * blk.out_stride + blk.out_col0 + col));
      }
      lds_fence();
    };
    int64_t t0 = T0;
    if (t0 + 3 * PC_ROWS <= T1) {
      // (the first tile on its own: then loads and stores are in flight in the same order at both ends of the loop)
      tile(std::true_type{}, t0, xf, xnext);
      t0 += PC_ROWS;
      for (; t0 + 2 * PC_ROWS <= T1; t0 += 2 * PC_ROWS) {
        tile(std::true_type{}, t0, xnext, xf);
        tile(std::true_type{}, t0 + PC_ROWS, xf, xnext);
      }
#pragma unroll
      for (int ks = 0; ks < PC_NKS; ++ks) xf[ks] = xnext[ks];
    }
    for (; t0 < T1; t0 += PC_ROWS) {
      tile(std::false_type{}, t0, xf, xnext);
#pragma unroll
      for (int ks = 0; ks < PC_NKS; ++ks) xf[ks] = xnext[ks];
    }
  }

  job = (int)blockIdx.x - plan.tail.wg0;
  if (job >= 0 && job < plan.tail.n_wgs) {
    const int64_t w0 = (int64_t)(plan.conv.n_blocks + plan.plain.n_blocks) * PC_COLS_WG;
    for (int c0 = 0; c0 < plan.tail_cols; c0 += PC_COLS_WAVE) {
      pc_load_w(W, w0 + c0, plan.tail_cols - c0, lane, wf);
      for (int64_t t0 = (int64_t)(4 * job + wave) * PC_ROWS; t0 < n_tokens; t0 += (int64_t)4 * plan.tail.n_wgs * PC_ROWS) {
        pc_load_x(x, x_stride, n_tokens, t0, lane, xf);
        pc_tile(wf, xf, lane, sy);
        lds_fence();
        const int c = c0 + 8 * cg;
#pragma unroll
        for (int i = 0; i < PC_ROWS_LANE; ++i) {
          const int tr = PC_ROWS_LANE * tq + i;
          const bf16x8 o = *reinterpret_cast<const bf16x8*>(&sy[(tr + PC_W - 1) * PC_LD + 8 * cg]);
          const int64_t t = t0 + tr;
          if (t < n_tokens && c < plan.tail_cols) *reinterpret_cast<bf16x8*>(plan.tail_out + t * plan.tail_cols + c) = o;
        }
        lds_fence();
      }
    }
  }
}

// x [n_tokens, 128] bf16 (row stride x_stride elements), n_tokens / t_len dense sequences of t_len tokens;
// W [n_cols, 128] bf16 row-major (the rows of the projections one after the other); the first n_conv columns go
// through the convolution (conv_w fp32 [n_conv, 4], conv_b fp32 [n_conv] or NULL) and SiLU and are written as
// n_conv / conv_split tensors [n_tokens, conv_split] at conv_out + i * n_tokens * conv_split; the remaining columns
// are written as they are: the next plain_cols to plain_out [n_tokens, plain_cols], whatever is left (< 256 columns)
// to tail_out [n_tokens, tail_cols]. n_conv, conv_split and plain_cols are multiples of 256; tail_cols a multiple of 8.
extern "C" int lampa_proj_conv_fwd(const void* x, int64_t x_stride, int64_t n_tokens, int64_t t_len, int K, const void* W,
                                   int n_cols, const float* conv_w, const float* conv_b, int n_conv, int conv_split,
                                   void* conv_out, int plain_cols, void* plain_out, int tail_cols, void* tail_out,
                                   int tokens_per_wg, void* stream) {
  if (!x || !W || n_tokens < 0 || t_len < 1 || n_cols < 1) return LAMPA_ERR_INVALID;
  if (K != PC_K) return LAMPA_ERR_UNSUPPORTED;
  if (n_conv < 0 || plain_cols < 0 || tail_cols < 0 || n_conv + plain_cols + tail_cols != n_cols) return LAMPA_ERR_INVALID;
  if (n_conv % PC_COLS_WG || plain_cols % PC_COLS_WG || tail_cols >= PC_COLS_WG || tail_cols % 8) return LAMPA_ERR_UNSUPPORTED;
  if (n_conv && (!conv_w || !conv_out || conv_split < PC_COLS_WG || conv_split % PC_COLS_WG || n_conv % conv_split))
    return LAMPA_ERR_INVALID;
  if ((plain_cols && !plain_out) || (tail_cols && !tail_out)) return LAMPA_ERR_INVALID;
  if (x_stride < PC_K || x_stride % 8 || n_tokens % t_len) return LAMPA_ERR_INVALID;
  if (((uintptr_t)x | (uintptr_t)W | (uintptr_t)conv_out | (uintptr_t)plain_out | (uintptr_t)tail_out) % 16)
    return LAMPA_ERR_UNSUPPORTED;
  const int n_blocks = (n_cols + PC_COLS_WG - 1) / PC_COLS_WG;
  if (n_blocks > PC_MAX_BLOCKS) return LAMPA_ERR_UNSUPPORTED;
  if (n_tokens == 0) return LAMPA_OK;
  const int n_conv_blocks = n_conv / PC_COLS_WG, n_plain_blocks = plain_cols / PC_COLS_WG;
  static std::atomic<int> slots_of{0};  // workgroups the chip holds: two per CU (registers allow no more)
  int slots = slots_of.load();
  if (!slots) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
      cus = 256;
    slots = 2 * cus;
    slots_of.store(slots);
  }
  // runs of `tokens` per block of a kind, at least min_tokens and whole tiles
  auto runs_of = [&](PcJobs& j, int n_blocks, int64_t wgs, int64_t min_tokens) {
    j.n_blocks = n_blocks;
    if (n_blocks == 0) { j.wg0 = j.n_wgs = 0; j.tokens = PC_ROWS; return; }
    const int64_t runs = wgs / n_blocks > 0 ? wgs / n_blocks : 1;
    int64_t t = (n_tokens + runs - 1) / runs;
    t = ((t < min_tokens ? min_tokens : t) + PC_ROWS - 1) / PC_ROWS * PC_ROWS;
    j.tokens = (int)t;
    j.n_wgs = (int)((n_tokens + t - 1) / t) * n_blocks;
    j.wg0 = 0;
  };
  PcPlan plan;
  const int64_t tail_tiles = tail_cols ? (n_tokens + PC_ROWS - 1) / PC_ROWS : 0;
  // A workgroup with a run of every kind, one round of them, pays once all slots would be taken by one-kind workgroups of
  // more than the shortest run; below that the kinds side by side have fewer tiles in a row.
  const bool mixed = tokens_per_wg <= 0 && n_conv_blocks && n_tokens > (int64_t)slots / n_blocks * (4 * PC_ROWS);
  int64_t grid;
  if (mixed) {
    runs_of(plan.conv, n_conv_blocks, slots, 4 * PC_ROWS);
    runs_of(plan.plain, n_plain_blocks, plan.conv.n_wgs, PC_ROWS);
    plan.tail = {0, tail_cols ? plan.conv.n_wgs : 0, 1, PC_ROWS};
    grid = plan.conv.n_wgs > plan.plain.n_wgs ? plan.conv.n_wgs : plan.plain.n_wgs;
  } else {
    const int64_t min_tokens = tokens_per_wg > 0 ? tokens_per_wg : 4 * PC_ROWS;
    const int64_t wgs = tokens_per_wg > 0 ? INT32_MAX : slots / n_blocks;  // (per block)
    runs_of(plan.conv, n_conv_blocks, wgs * n_conv_blocks, min_tokens);
    runs_of(plan.plain, n_plain_blocks, wgs * n_plain_blocks, min_tokens);
    plan.plain.wg0 = plan.conv.n_wgs;
    plan.tail = {plan.conv.n_wgs + plan.plain.n_wgs, (int)((tail_tiles + 15) / 16), 1, PC_ROWS};
    grid = plan.tail.wg0 + plan.tail.n_wgs;
  }
  plan.tail_out = (__bf16*)tail_out;
  plan.tail_cols = tail_cols;
  for (int b = 0; b < n_conv_blocks + n_plain_blocks; ++b) {
    PcBlock& k = plan.blocks[b];
    const int c0 = b * PC_COLS_WG;
    if (c0 < n_conv) {
      const int part = c0 / conv_split;
      k = {(__bf16*)conv_out + (int64_t)part * n_tokens * conv_split, conv_split, c0 - part * conv_split};
    } else {
      k = {(__bf16*)plain_out, plain_cols, c0 - n_conv};
    }
  }
  hipStream_t s = (hipStream_t)stream;
  LAMPA_PROF(s, "start");
  hipLaunchKernelGGL(pc_proj_conv_kernel, dim3((unsigned)grid), dim3(256), 0, s, (const __bf16*)x, x_stride, n_tokens, t_len,
                     (const __bf16*)W, conv_w, conv_b, plan);
  LAMPA_PROF(s, "pc_proj_conv_kernel");
  return lampa_launch_status();
}

// ------------------------------------------------------------------------------- gated RMS norm + output projection
// y[t, :] = W_o * vec_h( rmsnorm(o[t, h, :]) * weight * swish(g[t, h, :]) ): the gated norm of every head
// (models/hattention/fused_norm.py:40-111 with IS_RMS_NORM and the swish gate) feeding the bias-free output projection
// (modeling_gated_deltaproduct.py:612-623) without writing the normalised tensor. One workgroup = 8 waves walks a run
// of 32-token tiles: all threads normalise and gate a tile into LDS (bf16; 8 lanes share a head's 64 channels), every
// wave multiplies it with its 16 rows of W_o, which it keeps in registers, and the result goes through LDS to whole rows,
// 16 lanes each, for the residual add, the next norm's sum of squares and the stores.
// Bound by latency: a tile is a chain of loads, norm, LDS, MFMA, LDS and stores on two waves per SIMD. The rows of o and g
// are therefore requested a tile ahead (32 registers), for which 16 rows of W_o per wave (64 registers, 128 for 32 rows)
// leave room; one workgroup per CU (with the 128 registers of two it spills 90). The sums over lanes are DPP moves. 60 000
// tokens with residual and norm: 50.4 us (four waves of 32 rows, two workgroups per CU, loads waited for where they are
// issued, two barriers that also drained them) -> 46 us.
#define NP_D 64        // channels per head
#define NP_KMAX 512    // heads * channels this kernel is built for (16 contraction steps of 32)
#define NP_OUT 128     // output columns (8 waves x 16)
#define NP_LDA (NP_KMAX + 8)
#define NP_LDO (NP_OUT + 8)
#define NP_THREADS 512
#define NP_PASSES 4    // rows of (token, head) a thread stages per tile: 64 per pass
#define NP_DPP_HALF_MIRROR 0x141
#define NP_DPP_ROW_LANE(n) (0x150 + (n))  /* lane n of each row of 16 -> the whole row */

// RES: with a residual and the next layer's norm
template <bool RES>
__global__ void __launch_bounds__(NP_THREADS, 2) pc_norm_proj_kernel(
    const __bf16* __restrict__ o, const __bf16* __restrict__ g, int64_t g_stride, const float* __restrict__ norm_w,
    const __bf16* __restrict__ W, int64_t n_tokens, float eps, __bf16* __restrict__ y, const __bf16* __restrict__ residual,
    const float* __restrict__ next_w, float next_eps, __bf16* __restrict__ res_out, int tokens_per_wg) {
  constexpr int NKS = NP_KMAX / 32;
  __shared__ __align__(16) __bf16 s_a[2][PC_ROWS * NP_LDA];
  __shared__ __align__(16) __bf16 s_out[PC_ROWS * NP_LDO];
  __shared__ __align__(16) float s_w[NP_D + NP_OUT];  // the weights of both norms (read where they are used, not held in registers)
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g4 = lane >> 4, ln = lane & 15;
  const int64_t T0 = (int64_t)blockIdx.x * tokens_per_wg;
  const int64_t T1 = T0 + tokens_per_wg < n_tokens ? T0 + tokens_per_wg : n_tokens;

  bf16x8 wf[NKS];  // rows 16 wave + ln of W_o
  {
    const __bf16* wp = W + (int64_t)(16 * wave + ln) * NP_KMAX + 8 * g4;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) wf[ks] = *reinterpret_cast<const bf16x8*>(wp + 32 * ks);
  }
  // norm role: 8 lanes per (token, head) row, 8 channels each
  const int sub = tid & 7, head = (tid >> 3) & 7, tok = wave;
  const int orow = tid >> 4, ocol = 8 * (tid & 15);  // output role: 8 columns of a row
  if (tid < NP_D) s_w[tid] = norm_w ? norm_w[tid] : 1.0f;
  if (RES && tid < NP_OUT) s_w[NP_D + tid] = next_w ? next_w[tid] : 1.0f;
  __syncthreads();

  bf16x8 ov[NP_PASSES], gv[NP_PASSES];
  auto request = [&](int64_t t0) __attribute__((always_inline)) {
    const int64_t first = t0 < n_tokens ? t0 : n_tokens - 1;
    const int last = n_tokens - 1 - first < PC_ROWS ? (int)(n_tokens - 1 - first) : PC_ROWS - 1;
    const __bf16 *ob = o + first * NP_KMAX, *gb = g + first * g_stride;
#pragma unroll
    for (int p = 0; p < NP_PASSES; ++p) {
      const int t = min(8 * p + tok, last);
      ov[p] = *reinterpret_cast<const bf16x8*>(ob + (uint32_t)(t * NP_KMAX + head * NP_D + 8 * sub));
      gv[p] = *reinterpret_cast<const bf16x8*>(gb + t * g_stride + (uint32_t)(head * NP_D + 8 * sub));
    }
  };
  auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP_PASSES; ++p) {
      float x[8], ss = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c) { x[c] = (float)ov[p][c]; ss = __builtin_fmaf(x[c], x[c], ss); }
      ss += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, ss);
      ss += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, ss);
      ss += dpp_f32<NP_DPP_HALF_MIRROR, 0xF>(0.0f, ss);
      const float rstd = 1.0f / sqrtf(ss * (1.0f / NP_D) + eps);
      bf16x8 out;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float gc = (float)gv[p][c];
        out[c] = (__bf16)(x[c] * rstd * s_w[8 * sub + c] * gc * pc_sigmoid(gc));
      }
      *reinterpret_cast<bf16x8*>(&s_a[buf][(8 * p + tok) * NP_LDA + head * NP_D + 8 * sub]) = out;
    }
  };
  auto request_residual = [&](int64_t t0) __attribute__((always_inline)) {
    bf16x8 r = {};
    if constexpr (RES) {
      int64_t t = t0 + orow;
      t = t < n_tokens ? t : n_tokens - 1;
      r = *reinterpret_cast<const bf16x8*>(residual + t * NP_OUT + ocol);
    }
    return r;
  };
  // One tile: buf holds it, the registers the rows of the next one; whole: all 32 rows exist (no condition on the stores, so
  // that the compiler can count them and does not wait for them with the rows requested ahead of them).
  auto tile = [&](auto whole, int64_t t0, int buf, const bf16x8& res, bf16x8& res_next) __attribute__((always_inline)) {
    stage(buf ^ 1);
    res_next = request_residual(t0 + PC_ROWS);
    request(t0 + 2 * PC_ROWS);
    f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    const __bf16* ap = &s_a[buf][ln * NP_LDA + 8 * g4];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int m = 0; m < 2; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            wf[ks], *reinterpret_cast<const bf16x8*>(ap + 16 * m * NP_LDA + 32 * ks), acc[m], 0, 0, 0);
#pragma unroll
    for (int m = 0; m < 2; ++m) {  // lane = token, registers = neighbouring columns
      bf16x4 p;
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = (__bf16)acc[m][e];
      *reinterpret_cast<bf16x4*>(&s_out[(16 * m + ln) * NP_LDO + 16 * wave + 4 * g4]) = p;
    }
    lds_barrier();  // the output tile is complete, the next A tile is staged
    const bf16x8 yv = *reinterpret_cast<const bf16x8*>(&s_out[orow * NP_LDO + ocol]);
    lds_barrier();  // the output tile has been read
    const int64_t t = t0 + orow;
    const bool live = decltype(whole)::value || t < T1;
    if constexpr (!RES) {
      if (live) *reinterpret_cast<bf16x8*>(y + t * NP_OUT + ocol) = yv;
    } else {
      // residual add and the next layer's RMS norm over the 128 output columns (fused_norm.py:1436-1506 with a
      // residual): res_out = residual + y, y = rmsnorm(res_out) * next_w, the sum of squares taken before rounding
      float sres[8], ss = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        sres[c] = (float)yv[c] + (float)res[c];
        ss = __builtin_fmaf(sres[c], sres[c], ss);
      }
      ss += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, ss);
      ss += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, ss);
      // every quad of lanes holds the sum over its 32 columns: added from the first to the last (another order changes the
      // bits of the norm now and then, and a stack of layers in bf16 spreads that over its whole output)
      ss = ((dpp_f32<NP_DPP_ROW_LANE(0), 0xF>(0.0f, ss) + dpp_f32<NP_DPP_ROW_LANE(4), 0xF>(0.0f, ss)) +
            dpp_f32<NP_DPP_ROW_LANE(8), 0xF>(0.0f, ss)) + dpp_f32<NP_DPP_ROW_LANE(12), 0xF>(0.0f, ss);
      const float rstd = 1.0f / sqrtf(ss * (1.0f / NP_OUT) + next_eps);
      bf16x8 ro, ho;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        ro[c] = (__bf16)sres[c];
        ho[c] = (__bf16)(sres[c] * rstd * s_w[NP_D + ocol + c]);
      }
      if (live) {
        *reinterpret_cast<bf16x8*>(res_out + t * NP_OUT + ocol) = ro;
        *reinterpret_cast<bf16x8*>(y + t * NP_OUT + ocol) = ho;
      }
    }
  };
  if (T0 >= T1) return;
  bf16x8 rA = request_residual(T0), rB;
  request(T0);
  stage(0);
  request(T0 + PC_ROWS);
  lds_barrier();
  int64_t t0 = T0;
  if (t0 + 3 * PC_ROWS <= T1) {
    // (the first tile on its own: then loads and stores are in flight in the same order at both ends of the loop)
    tile(std::true_type{}, t0, 0, rA, rB);
    t0 += PC_ROWS;
    for (; t0 + 2 * PC_ROWS <= T1; t0 += 2 * PC_ROWS) {
      tile(std::true_type{}, t0, 1, rB, rA);
      tile(std::true_type{}, t0 + PC_ROWS, 0, rA, rB);
    }
    rA = rB;
  }
  for (int buf = (int)((t0 - T0) / PC_ROWS) & 1; t0 < T1; t0 += PC_ROWS, buf ^= 1) {  // at most two
    tile(std::false_type{}, t0, buf, rA, rB);
    rA = rB;
  }
}

// o [n_tokens, 8, 64] bf16 contiguous; g the same shape with token stride g_stride elements; norm_w fp32 [64] or NULL;
// W [128, 512] bf16 row-major (the output projection); y [n_tokens, 128] bf16.
// With residual [n_tokens, 128] bf16: res_out = residual + projection (bf16) and y = rmsnorm(res_out) * next_w
// (next_w fp32 [128] or NULL, next_eps), i.e. the residual add and the next layer's pre-norm are applied as well.
extern "C" int lampa_norm_proj_fwd(const void* o, const void* g, int64_t g_stride, const float* norm_w, const void* W,
                                   int64_t n_tokens, int heads, int head_dim, int n_out, float eps, void* y,
                                   const void* residual, const float* next_w, float next_eps, void* res_out,
                                   int tokens_per_wg, void* stream) {
  if (!o || !g || !W || !y || n_tokens < 0) return LAMPA_ERR_INVALID;
  if (residual && (!res_out || ((uintptr_t)residual | (uintptr_t)res_out) % 16)) return LAMPA_ERR_INVALID;
  if (heads * head_dim != NP_KMAX || head_dim != NP_D || n_out != NP_OUT) return LAMPA_ERR_UNSUPPORTED;
  if (g_stride < NP_KMAX || g_stride % 8 || ((uintptr_t)o | (uintptr_t)g | (uintptr_t)W | (uintptr_t)y) % 16)
    return LAMPA_ERR_UNSUPPORTED;
  if (n_tokens == 0) return LAMPA_OK;
  if (tokens_per_wg <= 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
      cus = 256;
    tokens_per_wg = (int)((n_tokens + cus - 1) / cus);
    if (tokens_per_wg < 2 * PC_ROWS) tokens_per_wg = 2 * PC_ROWS;
  }
  tokens_per_wg = (tokens_per_wg + PC_ROWS - 1) / PC_ROWS * PC_ROWS;
  hipStream_t s = (hipStream_t)stream;
  LAMPA_PROF(s, "start");
  const dim3 grid((unsigned)((n_tokens + tokens_per_wg - 1) / tokens_per_wg));
#define NP_LAUNCH(RES)                                                                                                        \
  hipLaunchKernelGGL(pc_norm_proj_kernel<RES>, grid, dim3(NP_THREADS), 0, s, (const __bf16*)o, (const __bf16*)g, g_stride,    \
                     norm_w, (const __bf16*)W, n_tokens, eps, (__bf16*)y, (const __bf16*)residual, next_w, next_eps,          \
                     (__bf16*)res_out, tokens_per_wg)
  if (residual) NP_LAUNCH(true);
  else NP_LAUNCH(false);
#undef NP_LAUNCH
  LAMPA_PROF(s, "pc_norm_proj_kernel");
  return lampa_launch_status();
}
