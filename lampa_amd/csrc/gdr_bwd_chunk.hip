// Backward pass of the gated-delta forward in the chunked (WY) form on the MFMA (gfx950), K = V = 64, bf16 / fp16.
//
// Replaces chunk_gated_delta_rule_bwd (reference chengjiang123/Lampa, models/hattention/gated_delta_rule_ori.py:83-160:
// chunk_bwd_dv_local chunk_o.py:372, chunk_gated_delta_rule_bwd_dhu chunk_delta_h.py:209, chunk_bwd_dqkwg chunk_o.py:128,
// prepare_wy_repr_bwd wy_fast.py:27) and the l2norm_bwd calls of ChunkGatedDeltaRuleFunction.backward
// (gated_delta_rule_ori.py:205-233).
//
// Per chunk of 64 tokens of one head (Kh, Qh the l2-normalised rows, gamma the in-chunk cumulative log-decay, S the
// state entering the chunk, G' the gradient of the loss with respect to the state leaving it):
//   forward   A = strict_lower(beta_i (kh_i . kh_j) e^{gamma_i - gamma_j}),  T = (I + A)^-1,  E = diag(e^gamma),
//             D = diag(e^{gamma_L - gamma}),  R = B (V - E Kh S),  Vn = T R,  S' = e^{gamma_L} S + (D Kh)^T Vn,
//             O = E Qh S scale + P Vn,  P_ij = scale (qh_i . kh_j) e^{gamma_i - gamma_j}  (i >= j)
//   backward  dVn = P^T dO + D Kh G',   X = T^T dVn  (dV = B X),
//             dS = e^{gamma_L} G' + scale (E Qh)^T dO - (B E Kh)^T X,
//             grad A = -X Vn^T,  grad P = dO Vn^T,  and dKh, dQh from those and from X S^T, Vn G'^T, dO S^T
// The recurrence of dS is the transpose of the forward one and is cut into the same segments: a segment maps the gradient
// behind it to the gradient in front of it by G -> M^T G + N', with the M the forward composite pass already made.
//   forward   (gdr_chunk.hip, training form) leaves the chunks' records, the state in front of every chunk (16-bit operand
//             fragments) and the transposed M of every segment;
//   source    gdrb_source_kernel: every segment's N' (the walk below from a zero gradient, nothing else);
//   group     gdr_scan2_kernel, reversed: composites of groups of 8 segments of long sequences;
//   walk      gdrb_walk_kernel: a workgroup pushes the gradient behind the sequence through the composites of the
//             later segments, then walks its own chunks from the last to the first and writes every gradient of each.
#include "gdr_chunk_kernels.h"
#include "gdr_train.h"
#include <mutex>

#define GB_LS 72                    // row stride (16-bit elements) of the k, q and dO tiles: 16-byte aligned rows
#define GB_TS 36                    // row stride of a 32 x 32 block of T
#define GB_TRI 2048                 // bytes of one 32 x 32 tile in operand fragment order
#define GB_SOURCE_THREADS 512
#define GB_WALK_THREADS 768

// One set of a chunk's tiles in LDS (bytes). Fragment order of a 64 x 64 tile with rows r and columns c: fragment
// 4 (c / 32) + r / 16, lane 32 ((r / 4) % 2) + c % 32, element 4 ((r / 8) % 2) + r % 4 -- what a lane holds of an
// accumulator tile, rounded.
template <bool GRADS>
struct GbSet {
  static constexpr int TILE = 64 * GB_LS * 2;
  static constexpr int OFF_K = 0;                           // kh rows
  static constexpr int OFF_Q = OFF_K + TILE;                // qh rows
  static constexpr int OFF_DO = OFF_Q + TILE;
  static constexpr int OFF_T = OFF_DO + TILE;               // T11 | T21 | T22
  static constexpr int OFF_F = OFF_T + 3 * 32 * GB_TS * 2;  // rows of 64 floats: gamma, beta, e^gamma, e^{gamma_L - gamma}, rk, rq
  static constexpr int OFF_V = OFF_F + 6 * 256;             // v as two 64 x 32 tiles, then Vn (fragment order)
  static constexpr int OFF_S = OFF_V + (GRADS ? 8192 : 0);  // the state in front of the chunk (fragment order)
  static constexpr int BYTES = OFF_S + (GRADS ? 8192 : 0);
};

// The partial sums of a chunk (float offsets): every wave writes its own, wave 7 adds them up. (As LDS atomics they took
// half of the kernel's LDS cycles.)
struct GbSums {
  static constexpr int DOTK = 0;                 // [2][64] products of the rows of dKh with kh, per half of the columns
  static constexpr int DGAM = DOTK + 128;        // [6][32] d gamma: the two dQh waves, then the four dKh waves
  static constexpr int TILE_G = DGAM + 192;      // [3 tiles][32] d gamma of the tile's columns i
  static constexpr int TILE_C = TILE_G + 96;     // [3 tiles][32] and of its rows j (to be subtracted)
  static constexpr int TILE_B = TILE_C + 96;     // [3 tiles][32] d beta of the columns
  static constexpr int DBETA = TILE_B + 96;      // [four dKh waves][32] d beta of the wave's tokens
  static constexpr int XV = DBETA + 128;         // [64] X . v
  static constexpr int GL = XV + 64;             // [5][2] the terms of d gamma that belong to the chunk's last row: dKh waves, wave 7
  static constexpr int FLOATS = GL + 12;
};

// LDS of the walk: two sets of tiles, what the waves exchange inside a chunk, the rows of dq and dk on their way out.
struct GbWalkSmem {
  static constexpr int OFF_P = 2 * GbSet<true>::BYTES;  // P, N (grad P gated), M (grad A gated): three 32 x 32 tiles each
  static constexpr int OFF_N = OFF_P + 3 * GB_TRI;
  static constexpr int OFF_M = OFF_N + 3 * GB_TRI;
  static constexpr int OFF_G = OFF_M + 3 * GB_TRI;      // G' (fragment order)
  static constexpr int OFF_X = OFF_G + 8192;            // X (fragment order)
  static constexpr int OFF_OQ = OFF_X + 8192;
  static constexpr int OFF_OK = OFF_OQ + 64 * GB_LS * 2;
  static constexpr int OFF_SUM = OFF_OK + 64 * GB_LS * 2;
  static constexpr int BYTES = OFF_SUM + 4 * GbSums::FLOATS;
};
static_assert(GbWalkSmem::BYTES <= 163840, "LDS of a CU");
struct GbSourceSmem {
  static constexpr int OFF_P = 2 * GbSet<false>::BYTES;
  static constexpr int OFF_NOTE = OFF_P + 3 * GB_TRI;  // the waves' largest q and dO, the two waves of N'
  static constexpr int BYTES = OFF_NOTE + 80;
};
static_assert(GbSourceSmem::BYTES <= 81920, "two workgroups per CU");

// Transposing read of a tile in fragment order: operand row / column = tile row r0 + lane % 32, contraction over the tile
// columns c0 .. c0 + 15; KAPPA: in accumulator slot order, otherwise consecutive (slots of lane half hh: 8 hh ..).
template <typename OT, bool KAPPA>
__device__ __forceinline__ typename OpVec<OT>::x8 fr_tr(const unsigned char* tile, int r0, int c0, int lane) {
  const int L = lane & 15, blk = (lane >> 4) & 1, hh = lane >> 5;
  const int c = c0 + (KAPPA ? 4 : 8) * hh + (L >> 2);
  const OT* p = reinterpret_cast<const OT*>(tile + ((c >> 5) * 4 + (r0 >> 4) + blk) * 1024 +
                                            (32 * (L & 1) + (c & 31)) * 16 + ((L >> 1) & 1) * 8);
  const typename OpVec<OT>::x4 lo = op_lds_read_tr4<OT>(p), hi = op_lds_read_tr4<OT>(p + (KAPPA ? 8 : 4) * 8);
  typename OpVec<OT>::x8 out;
#pragma unroll
  for (int s = 0; s < 4; ++s) { out[s] = lo[s]; out[4 + s] = hi[s]; }
  return out;
}

// sum over the 32 lanes of this lane's half of the wave (every lane of the half receives it)
__device__ __forceinline__ float gb_half_sum(float x) {
  x += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, x);
  x += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, x);
  x += dpp_f32<0x141, 0xF>(0.0f, x);  // row_half_mirror
  x += dpp_f32<0x140, 0xF>(0.0f, x);  // row_mirror
  x += __shfl_xor(x, 16);
  return x;
}
// Sums of 16 registers over the 32 lanes of a half-wave, register by register: lane ln of the half receives the sum of
// register ln / 2. Every step halves the number of registers a lane still carries (16 swaps and adds, then selects and
// DPP adds: 38 instructions against 16 full reductions of 5 steps each).
__device__ __forceinline__ float gb_half_sums16(const float* x, int lane) {
  float y[8], z[4], w[2];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[r]), __float_as_uint(x[r + 8]), false, false);
    y[r] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  const bool b8 = lane & 8, b4 = lane & 4, b2 = lane & 2;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float keep = b8 ? y[r + 4] : y[r], give = b8 ? y[r] : y[r + 4];
    z[r] = keep + dpp_f32<0x128, 0xF>(0.0f, give);  // row_ror:8
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const float keep = b4 ? z[r + 2] : z[r], give = b4 ? z[r] : z[r + 2];
    w[r] = keep + dpp_f32<0x141, 0xF>(0.0f, give);  // row_half_mirror
  }
  const float keep = b2 ? w[1] : w[0], give = b2 ? w[0] : w[1];
  float t = keep + dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, give);
  t += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, t);
  return t;
}
// sum over the two half-waves
__device__ __forceinline__ float gb_both_halves(float x) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// sum over the 8 consecutive lanes that share lane / 8
__device__ __forceinline__ float gb_sum8(float x) {
  x += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, x);
  x += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, x);
  x += dpp_f32<0x141, 0xF>(0.0f, x);
  return x;
}

// this lane's 16 accumulator rows' worth of a per-row factor (rows r0 + 8 b + 4 hh + e)
__device__ __forceinline__ f32x4 gb_rows4(const float* f, int r0, int b4, int hh) {
  return *reinterpret_cast<const f32x4*>(&f[r0 + 8 * b4 + 4 * hh]);
}

// Fragments requested together: passing them through an asm behind all the reads keeps the MFMAs that use them there (an
// MFMA is no memory access, and left alone the compiler puts each one behind its own read and pays the LDS latency each time).
template <int N, typename X8>
__device__ __forceinline__ void gb_pin(X8 (&x)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) asm volatile("" : "+v"(x[j]));
}

// One 16-bit set of tiles in LDS
template <typename OT>
struct GbTiles {
  OT *k, *q, *dout, *t, *v;
  unsigned char* s;
  float *gam, *beta, *eg, *dk, *rk, *rq;
};
template <typename OT, bool GRADS>
__device__ __forceinline__ GbTiles<OT> gb_tiles(unsigned char* smem, int par) {
  unsigned char* b = smem + par * GbSet<GRADS>::BYTES;
  GbTiles<OT> t;
  t.k = reinterpret_cast<OT*>(b + GbSet<GRADS>::OFF_K);
  t.q = reinterpret_cast<OT*>(b + GbSet<GRADS>::OFF_Q);
  t.dout = reinterpret_cast<OT*>(b + GbSet<GRADS>::OFF_DO);
  t.t = reinterpret_cast<OT*>(b + GbSet<GRADS>::OFF_T);
  t.v = reinterpret_cast<OT*>(b + GbSet<GRADS>::OFF_V);
  t.s = b + GbSet<GRADS>::OFF_S;
  t.gam = reinterpret_cast<float*>(b + GbSet<GRADS>::OFF_F);
  t.beta = t.gam + 64;
  t.eg = t.gam + 128;
  t.dk = t.gam + 192;
  t.rk = t.gam + 256;
  t.rq = t.gam + 320;
  return t;
}

// operand fragments of the row-major tiles: rows in accumulator slot order / in consecutive order, and the transpose
template <typename OT>
__device__ __forceinline__ typename OpVec<OT>::x8 gb_rows_k(const OT* buf, int row, int c, int hh) {
  return op_ld_kappa<OT>(buf, GB_LS, row, c, hh);
}
template <typename OT>
__device__ __forceinline__ typename OpVec<OT>::x8 gb_rows_n(const OT* buf, int row, int c, int hh) {
  return *reinterpret_cast<const typename OpVec<OT>::x8*>(&buf[row * GB_LS + c + 8 * hh]);
}
template <typename OT>
__device__ __forceinline__ typename OpVec<OT>::x8 gb_cols(const OT* buf, int col0, int row0, int lane) {
  return op_ld_kappa_tr<OT, false>(buf, GB_LS, col0, row0, lane);
}
// a 32 x 32 product over 64 contraction steps, both operands from LDS, all eight fragments requested first
template <typename OT, typename FA, typename FB>
__device__ __forceinline__ f32x16 gb_mm(f32x16 acc, FA fa, FB fb) {
  typename OpVec<OT>::x8 a[4], b[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) { a[ks] = fa(ks); b[ks] = fb(ks); }
  gb_pin(a);
  gb_pin(b);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) acc = mfma32(a[ks], b[ks], acc);
  return acc;
}
// the same over the token steps a triangular tile leaves: lower (first 2 (tt + 1) of 4) or upper (from 2 tt on)
template <typename OT, bool LOWER, typename FA, typename FB>
__device__ __forceinline__ f32x16 gb_mm_tri(f32x16 acc, int tt, FA fa, FB fb) {
  if (tt == (LOWER ? 1 : 0)) return gb_mm<OT>(acc, fa, fb);
  typename OpVec<OT>::x8 a[2], b[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) { a[x] = fa(LOWER ? x : 2 + x); b[x] = fb(LOWER ? x : 2 + x); }
  gb_pin(a);
  gb_pin(b);
  acc = mfma32(a[0], b[0], acc);
  return mfma32(a[1], b[1], acc);
}

// The tile (j tile, i tile) of Q K^T (rows j, column i): scaled and gated it is P^T's operand and grad P's counterpart.
template <typename OT>
__device__ __forceinline__ f32x16 gb_pair(const OT* rows, int jt, const OT* colsb, int it, int ln, int hh) {
  return gb_mm<OT>(zero16(), [&](int ks) { return gb_rows_n<OT>(rows, 32 * jt + ln, 16 * ks, hh); },
                   [&](int ks) { return gb_rows_n<OT>(colsb, 32 * it + ln, 16 * ks, hh); });
}
// e^{gamma_i - gamma_j} of the tile for i >= j + e_min, else 0
__device__ __forceinline__ f32x16 gb_ratio(const float* gam, int jt, int it, int e_min, int ln, int hh) {
  const float gi = gam[32 * it + ln];
  const int lx = ln - 4 * hh - e_min + (jt != it ? 64 : 0);  // (the tile below the diagonal is full)
  f32x16 out;
#pragma unroll
  for (int b4 = 0; b4 < 4; ++b4) {
    const f32x4 gj = gb_rows4(gam, 32 * jt, b4, hh);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[4 * b4 + e] = __builtin_amdgcn_exp2f(lx >= 8 * b4 + e ? gi - gj[e] : -1e30f);
  }
  return out;
}
template <typename OT>
__device__ __forceinline__ void gb_store_tile(unsigned char* tile, const f32x16& x, int lane) {
  op_frag_store<OT>(tile, 0, lane, acc_to_op<OT>(x, 0));
  op_frag_store<OT>(tile, 1, lane, acc_to_op<OT>(x, 8));
}

// The gradient of the state: a wave's 32 value columns (all 64 rows) in accumulators. Every intermediate is handed on in
// registers: the accumulator tile of one product is the B operand of the next.
template <typename OT>
struct GbChain {
  using X8 = typename OpVec<OT>::x8;
  f32x16 G[2];  // the gradient behind the chunk
  f32x16 a[2];  // D Kh G', then dVn, then X
  X8 Xb[4];     // -beta e^gamma X as operand

  // a = D Kh G'; frags (nullable): G' goes there in fragment order
  __device__ __forceinline__ void state_rows(const GbTiles<OT>& t, unsigned char* frags, int slab, int lane, int hh, int ln) {
    X8 Gb[4], fk[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) fk[f] = gb_rows_k<OT>(t.k, 32 * (f >> 2) + ln, 16 * (f & 3), hh);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      Gb[ks] = acc_to_op<OT>(G[ks / 2], 8 * (ks % 2));
      if (frags) op_frag_store<OT>(frags, slab * 4 + ks, lane, Gb[ks]);
    }
    gb_pin(fk);
    a[0] = zero16();
    a[1] = zero16();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      a[0] = mfma32(fk[ks], Gb[ks], a[0]);
      a[1] = mfma32(fk[4 + ks], Gb[ks], a[1]);
    }
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        const f32x4 f = gb_rows4(t.dk, 32 * tm, b4, hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) a[tm][4 * b4 + e] *= f[e];
      }
  }
  // dVn = a + P^T dO, X = T^T dVn; X goes to frags (nullable) in fragment order
  __device__ __forceinline__ void chunk_rows(const GbTiles<OT>& t, const unsigned char* p, unsigned char* frags, int slab,
                                             int lane, int hh) {
    {
      X8 d[4], fp[6];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) d[ks] = gb_cols<OT>(t.dout, 32 * slab, 16 * ks, lane);
#pragma unroll
      for (int f = 0; f < 6; ++f) fp[f] = fr_tr<OT, true>(p + (f >> 1) * GB_TRI, 0, 16 * (f & 1), lane);
      gb_pin(d);
      gb_pin(fp);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        a[0] = mfma32(fp[ks], d[ks], a[0]);
        if (ks >= 2) a[1] = mfma32(fp[2 + ks], d[ks], a[1]);
      }
    }
    X8 ft[6];
#pragma unroll
    for (int f = 0; f < 6; ++f)
      ft[f] = op_ld_kappa_tr<OT, false>(t.t + (f >> 1) * 32 * GB_TS, GB_TS, 0, 16 * (f & 1), lane);
    X8 Rb[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) Rb[ks] = acc_to_op<OT>(a[ks / 2], 8 * (ks % 2));
    gb_pin(ft);
    a[0] = zero16();
    a[1] = zero16();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {  // (blocks T11, T21 | T22)
      a[0] = mfma32(ft[ks], Rb[ks], a[0]);
      if (ks >= 2) a[1] = mfma32(ft[2 + ks], Rb[ks], a[1]);
    }
#pragma unroll
    for (int tm = 0; tm < 2; ++tm) {
      if (frags) {
        op_frag_store<OT>(frags, slab * 4 + 2 * tm + 0, lane, acc_to_op<OT>(a[tm], 0));
        op_frag_store<OT>(frags, slab * 4 + 2 * tm + 1, lane, acc_to_op<OT>(a[tm], 8));
      }
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        const f32x4 fb = gb_rows4(t.beta, 32 * tm, b4, hh), fe = gb_rows4(t.eg, 32 * tm, b4, hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) a[tm][4 * b4 + e] *= -fb[e] * fe[e];
      }
      Xb[2 * tm + 0] = acc_to_op<OT>(a[tm], 0);
      Xb[2 * tm + 1] = acc_to_op<OT>(a[tm], 8);
    }
  }
  // the gradient in front of the chunk: e^{gamma_L} G' + (scale e^gamma Qh)^T dO - (beta e^gamma Kh)^T X
  __device__ __forceinline__ void update(const GbTiles<OT>& t, float scale, int slab, int lane, int hh) {
    const float dec = __builtin_amdgcn_exp2f(t.gam[63]);
#pragma unroll
    for (int km = 0; km < 2; ++km)
#pragma unroll
      for (int r = 0; r < 16; ++r) G[km][r] *= dec;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      X8 f[8], d[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int ks = 2 * half + x;
        d[x] = gb_cols<OT>(t.dout, 32 * slab, 16 * ks, lane);
#pragma unroll
        for (int km = 0; km < 2; ++km) {
          f[4 * x + km] = gb_cols<OT>(t.q, 32 * km, 16 * ks, lane);
          f[4 * x + 2 + km] = gb_cols<OT>(t.k, 32 * km, 16 * ks, lane);
        }
      }
      gb_pin(d);
      gb_pin(f);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int ks = 2 * half + x;
        const f32x4 f0 = *reinterpret_cast<const f32x4*>(&t.eg[16 * ks + 4 * hh]);
        const f32x4 f1 = *reinterpret_cast<const f32x4*>(&t.eg[16 * ks + 8 + 4 * hh]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          d[x][e] = (OT)((float)d[x][e] * (scale * f0[e]));
          d[x][4 + e] = (OT)((float)d[x][4 + e] * (scale * f1[e]));
        }
#pragma unroll
        for (int km = 0; km < 2; ++km) {
          G[km] = mfma32(f[4 * x + 2 + km], Xb[ks], G[km]);
          G[km] = mfma32(f[4 * x + km], d[x], G[km]);
        }
      }
    }
  }
};

// ---- staging of a chunk's tiles: loads into registers a chunk ahead, LDS writes when the other set is free ----------------
// k, q rows through the l2 normalisation: 256 threads, rows gt / 8 and 32 + gt / 8, 8-column piece gt % 8
template <typename T>
struct GbStageKQ {
  using OT = T;
  using X8 = typename OpVec<OT>::x8;
  typename Raw8<T>::type pk[2], pq[2];
  float prk[2];
  __device__ __forceinline__ void issue(const T* k, const T* q, const unsigned char* rec, int tok0, int len, int H, int h, int gt) {
    const float* rk = reinterpret_cast<const float*>(rec + T_BYTES) + 128;
    const size_t row0 = ((size_t)tok0 * H + h) * 64;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = 32 * u + (gt >> 3), r = min(row, len - 1);
      const uint32_t at = (uint32_t)(r * H * 64 + 8 * (gt & 7));  // (from the chunk's first row: one register per lane)
      pk[u] = *reinterpret_cast<const typename Raw8<T>::type*>(k + row0 + at);
      pq[u] = *reinterpret_cast<const typename Raw8<T>::type*>(q + row0 + at);
      prk[u] = rk[row];
    }
  }
  __device__ __forceinline__ void stage_k(const GbTiles<OT>& t, int len, int l2norm, int gt) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = 32 * u + (gt >> 3), part = gt & 7;
      const bool live = row < len;  // (rows past the end of a partial chunk become zero)
      const float ck = live ? prk[u] : 0.0f;
      X8 ok;
      if (l2norm != GDR_L2_NONE) {
#pragma unroll
        for (int e = 0; e < 8; ++e) ok[e] = (OT)((float)pk[u][e] * ck);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) ok[e] = live ? (OT)pk[u][e] : (OT)0.0f;
      }
      *reinterpret_cast<X8*>(&t.k[row * GB_LS + 8 * part]) = ok;
    }
  }
  __device__ __forceinline__ void stage_q(const GbTiles<OT>& t, int len, int l2norm, int gt) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = 32 * u + (gt >> 3), part = gt & 7;
      const bool live = row < len;
      float cq = 1.0f;
      X8 oq;
      if (l2norm != GDR_L2_NONE) {
        float fq[8], ss = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          fq[e] = live ? (float)pq[u][e] : 0.0f;
          ss = __builtin_fmaf(fq[e], fq[e], ss);
        }
        cq = l2_factor(gb_sum8(ss), l2norm);
#pragma unroll
        for (int e = 0; e < 8; ++e) oq[e] = (OT)(fq[e] * cq);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) oq[e] = live ? (OT)pq[u][e] : (OT)0.0f;
      }
      *reinterpret_cast<X8*>(&t.q[row * GB_LS + 8 * part]) = oq;
      if (part == 0) t.rq[row] = cq;
    }
  }
};
// dO rows and T (and v, S): NT threads
template <typename T, int NT, bool GRADS>
struct GbStageRest {
  using OT = T;
  using X8 = typename OpVec<OT>::x8;
  using X4 = typename OpVec<OT>::x4;
  static constexpr int NR = 512 / NT, NP = NT == 128 ? 3 : 2;  // (the last 32 pieces of T are loaded several times over)
  typename Raw8<T>::type pd[NR], pv[GRADS ? NR : 1];
  X8 ps[GRADS ? NR : 1], pt[NP];
  static __device__ __forceinline__ int t_piece(int u, int bt) { return NT * u + (u == NP - 1 ? (bt & 31) : bt); }
  static __device__ __forceinline__ int t_off(int p) {
    int row, pc;
    const int d = p - 128;
    tri_piece(d < 0 ? 0 : d < T_DIAG_PIECES ? d : d - T_DIAG_PIECES, row, pc);
    return d < 0 ? (32 + (p >> 2)) * GB_TS + 8 * (p & 3) : ((d < T_DIAG_PIECES ? 0 : 64) + row) * GB_TS + 8 * pc;
  }
  __device__ __forceinline__ void issue(const T* dout, const T* v, const unsigned char* rec, const unsigned char* state, int tok0,
                                        int len, int HV, int hv, int bt) {
    const size_t row0 = ((size_t)tok0 * HV + hv) * 64;
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      const int p = bt + NT * u, r = min(p >> 3, len - 1);
      const uint32_t at = (uint32_t)(r * HV * 64 + 8 * (p & 7));
      pd[u] = *reinterpret_cast<const typename Raw8<T>::type*>(dout + row0 + at);
      if constexpr (GRADS) {
        pv[u] = *reinterpret_cast<const typename Raw8<T>::type*>(v + row0 + at);
        ps[u] = reinterpret_cast<const X8*>(state)[p];
      }
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) pt[u] = reinterpret_cast<const X8*>(rec)[t_piece(u, bt)];
  }
  __device__ __forceinline__ void stage(const GbTiles<OT>& t, int len, int bt) {
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      const int p = bt + NT * u, row = p >> 3, part = p & 7;
      typename Raw8<T>::type z;
#pragma unroll
      for (int e = 0; e < 8; ++e) z[e] = (T)0.0f;
      const bool live = row < len;
      *reinterpret_cast<typename Raw8<T>::type*>(&t.dout[row * GB_LS + 8 * part]) = live ? pd[u] : z;
      if constexpr (GRADS) {
        *reinterpret_cast<typename Raw8<T>::type*>(&t.v[(part >> 2) * 2048 + row * 32 + 8 * (part & 3)]) = live ? pv[u] : z;
        *reinterpret_cast<X8*>(t.s + 16 * p) = ps[u];
      }
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int off = t_off(t_piece(u, bt));
      X4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) { lo[e] = pt[u][e]; hi[e] = pt[u][4 + e]; }
      *reinterpret_cast<X4*>(&t.t[off]) = lo;
      *reinterpret_cast<X4*>(&t.t[off + 4]) = hi;
    }
  }
};
// per-token factors: one wave
struct GbStageFactors {
  float g, b, r;
  __device__ __forceinline__ void issue(const unsigned char* rec, int lane) {
    const float* fact = reinterpret_cast<const float*>(rec + T_BYTES);
    g = fact[lane];
    b = fact[64 + lane];
    r = fact[128 + lane];
  }
  template <typename OT>
  __device__ __forceinline__ void stage(const GbTiles<OT>& t, int lane) {
    const float gl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), 63));
    t.gam[lane] = g;
    t.beta[lane] = b;
    t.rk[lane] = r;
    t.eg[lane] = __builtin_amdgcn_exp2f(g);
    t.dk[lane] = __builtin_amdgcn_exp2f(gl - g);
  }
};
// the pieces of T that lie entirely above the diagonals, in both sets: zero once
template <typename OT, bool GRADS>
__device__ __forceinline__ void gb_zero_upper(unsigned char* smem, int tid) {
  if (tid < 192) {
    const int u = tid % 96;
    int row, pc;
    tri_upper_piece(u % 48, row, pc);
    OT* at = &gb_tiles<OT, GRADS>(smem, tid / 96).t[((u < 48 ? 0 : 64) + row) * GB_TS + 8 * pc];
    typename OpVec<OT>::x4 z;
#pragma unroll
    for (int e = 0; e < 4; ++e) z[e] = (OT)0.0f;
    *reinterpret_cast<typename OpVec<OT>::x4*>(at) = z;
    *reinterpret_cast<typename OpVec<OT>::x4*>(at + 4) = z;
  }
}

// ---- source pass: every segment's N' (the walk from a zero gradient, no gradients written) --------------------------------
// Grid segments x heads (long segments first), eight waves: 0, 1 the gradient of the state (32 value columns each), 4-6 the
// tiles of P, 2 and 3 / 4-7 stage the next chunk into the other set of tiles. Two barriers per chunk, two workgroups per CU (80 KB
// of LDS, 128 registers). 52 - 57 us, by card, at 60 000 tokens x 8 heads (74 us with one set of tiles and the staging between the
// products), and 39 at e^-0.8 a token, where three of a segment's 15 chunks are walked and the q and dO of the others looked at (half
// of its traffic then); with the walk that starts at the next segment (197 -> 190) the training step 370 -> 352.
template <typename T>
__global__ void __launch_bounds__(GB_SOURCE_THREADS, 4)
    gdrb_source_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ dout,
                       const unsigned char* __restrict__ recs, const GdrPlanView pv, const int32_t* __restrict__ chunk_tok0,
                       const int32_t* __restrict__ chunk_len, unsigned char* __restrict__ Nr, int H, int HV, float scale,
                       int l2norm, const float* __restrict__ edges, const float* __restrict__ Dc, float* __restrict__ Dr) {
  using OT = T;
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char* const b_p = smem + GbSourceSmem::OFF_P;
  const int seg = pv.seg_order[blockIdx.x / HV], hv = blockIdx.x % HV, h = hv / (HV / H);
  if (pv.seg_flags[seg] & SEG_FIRST) return;  // nothing precedes the first segment of a sequence
  const int c0 = pv.seg_chunk0[seg], nc = pv.seg_nchunks[seg], cl = c0 + nc - 1;
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  // the chunks of a sequence follow one another, only its last one may be shorter: no table look-up in the loops
  const int tok_first = nc > 0 ? chunk_tok0[c0] : 0, len_last = nc > 0 ? chunk_len[cl] : 0;
  auto tok_of = [&](int c) { return tok_first + GDR_C * (c - c0); };
  auto len_of = [&](int c) { return c == cl ? len_last : GDR_C; };
  auto rec_of = [&](int c) { return recs + ((size_t)c * HV + hv) * REC_BYTES; };
  // chunk c from the set (cl - c) % 2; a chunk's tiles are staged while the one behind it is worked on, its loads issued a
  // chunk earlier still
  auto set_of = [&](int c) { return gb_tiles<OT, false>(smem, (cl - c) & 1); };
  gb_zero_upper<OT, false>(smem, tid);
  // Chunks at the segment's end that those in front of them leave nothing of are left out, as in the forward's composites, where a
  // look at their q and dO finds the sources scale q dO small enough: 128 chunks of these add up to less than 2^13 times the largest,
  // 2^58. With larger ones, or any that is not finite, all are walked.
  float* const note = reinterpret_cast<float*>(smem + GbSourceSmem::OFF_NOTE);
  int left = 0;
  if (nc >= GDR_EDGE_NC && nc <= GDR_EDGE_NC_MAX)
    left = uniform(gdr_chunks_left_out<true>(edges + (size_t)c0 * HV + hv, HV, nc, lane));
  if (left > 0) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 top_q = {0, 0}, top_d = {0, 0};
    const int row = tid >> 3, part = tid & 7;  // (a thread a 16-byte piece of the chunk's 64 rows)
    const T* qp = q + ((size_t)tok_of(cl - left + 1) * H + h) * 64 + 8 * part;
    const T* dp = dout + ((size_t)tok_of(cl - left + 1) * HV + hv) * 64 + 8 * part;
    const int rows = 64 * (left - 1) + len_last;
    for (int x = 0; x < left; x += 4) {
      uint4 rq[4], rd[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const size_t r = min(64 * (x + u) + row, rows - 1);
        rq[u] = *reinterpret_cast<const uint4*>(qp + r * H * 64);
        rd[u] = *reinterpret_cast<const uint4*>(dp + r * HV * 64);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t a[4] = {rq[u].x, rq[u].y, rq[u].z, rq[u].w}, d[4] = {rd[u].x, rd[u].y, rd[u].z, rd[u].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          top_q = __builtin_elementwise_max(top_q, __builtin_bit_cast(u16x2, a[e] & 0x7fff7fffu));
          top_d = __builtin_elementwise_max(top_d, __builtin_bit_cast(u16x2, d[e] & 0x7fff7fffu));
        }
      }
    }
    constexpr bool HALF = __is_same(T, _Float16);
    auto size_of = [](u16x2 top) {  // the largest of the wave (a NaN counts as infinity)
      const unsigned short x = min(max(top[0], top[1]), (unsigned short)(HALF ? 0x7c00 : 0x7f80));
      return wave_inclusive_max((float)__builtin_bit_cast(T, x));
    };
    const float wave_q = size_of(top_q), wave_d = size_of(top_d);
    if (lane == 63) { note[wave] = wave_q; note[8 + wave] = wave_d; }
    lds_barrier();
    float big_q = note[0], big_d = note[8];
#pragma unroll
    for (int w = 1; w < 8; ++w) { big_q = fmaxf(big_q, note[w]); big_d = fmaxf(big_d, note[8 + w]); }
    const float norm_q = l2norm == GDR_L2_NONE ? 8.0f * big_q : big_q <= 0x1p60f ? 1.0f : __builtin_inff();
    if (!(__builtin_fabsf(scale) * norm_q * big_d <= 0x1p45f)) left = 0;
  }
  const int ct = uniform(cl - left);  // the chunk the walk starts at
  if (wave < 2) {
    GbChain<OT> ch;
    ch.G[0] = zero16();
    ch.G[1] = zero16();
    if (nc > 0) lds_barrier();  // (0) the tiles of the first chunk are complete
    for (int c = ct; c >= c0; --c) {
      const GbTiles<OT> t = set_of(c);
      ch.state_rows(t, nullptr, wave, lane, hh, ln);
      lds_barrier();  // (1) P is complete
      ch.chunk_rows(t, b_p, nullptr, wave, lane, hh);
      ch.update(t, scale, wave, lane, hh);
      lds_barrier();  // (2) the tiles of chunk c have been read, those of chunk c - 1 are complete
    }
    // A segment without M (the forward's mark) and with a finite N' hands N' on whatever finite gradient comes from behind it
    const float dc = Dc[(size_t)seg * HV + hv];
    float dr = __builtin_fabsf(dc);
    if (gdr_d_cut(dc)) {
      float probe = 0.0f;
#pragma unroll
      for (int km = 0; km < 2; ++km)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(ch.G[km][r], 0.0f, probe);
      if (lane == 0) note[16 + wave] = __ballot(!(probe == 0.0f)) ? 1.0f : 0.0f;
      lds_barrier();  // (of the two waves that are left)
      if (note[16] + note[17] == 0.0f) dr = -0.0f;
    }
    if (tid == 0) Dr[(size_t)seg * HV + hv] = dr;
    // N' in accumulator order, as the forward composites keep N
    f32x4* out = reinterpret_cast<f32x4*>(Nr + (((size_t)seg * HV + hv) * 2 + wave) * GDR_STATE_BYTES);
#pragma unroll
    for (int km = 0; km < 2; ++km)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = ch.G[km][4 * q4 + e];
        out[(km * 4 + q4) * 64 + lane] = x;
      }
  } else if (nc == 0) {
    return;
  } else if (wave < 4) {
    GbStageRest<T, 128, false> st;
    const int bt = tid - 128;
    auto issue = [&](int c) {
      c = uniform(max(c, c0));
      st.issue(dout, nullptr, rec_of(c), nullptr, tok_of(c), len_of(c), HV, hv, bt);
    };
    issue(ct);
    st.stage(set_of(ct), len_of(ct), bt);
    issue(ct - 1);
    lds_barrier();  // (0)
    for (int c = ct; c >= c0; --c) {
      if (c > c0) st.stage(set_of(c - 1), len_of(c - 1), bt);
      issue(c - 2);
      lds_barrier();  // (1)
      lds_barrier();  // (2)
    }
  } else {
    GbStageKQ<T> st;
    GbStageFactors sf;
    const int gt = tid - 256, tw = wave - 4, jt = tw == 2 ? 1 : 0, it = tw == 0 ? 0 : 1;
    auto issue = [&](int c) {
      c = uniform(max(c, c0));
      st.issue(k, q, rec_of(c), tok_of(c), len_of(c), H, h, gt);
      sf.issue(rec_of(c), lane);  // (wave 7 stages them)
    };
    auto stage = [&](int c) {
      st.stage_k(set_of(c), len_of(c), l2norm, gt);
      st.stage_q(set_of(c), len_of(c), l2norm, gt);
      if (wave == 7) sf.stage(set_of(c), lane);
    };
    issue(ct);
    stage(ct);
    issue(ct - 1);
    lds_barrier();  // (0)
    for (int c = ct; c >= c0; --c) {
      const GbTiles<OT> t = set_of(c);
      if (wave < 7) {
        f32x16 p = gb_pair<OT>(t.k, jt, t.q, it, ln, hh);
        const f32x16 gm = gb_ratio(t.gam, jt, it, 0, ln, hh);
#pragma unroll
        for (int r = 0; r < 16; ++r) p[r] *= scale * gm[r];
        gb_store_tile<OT>(b_p + tw * GB_TRI, p, lane);
      }
      lds_barrier();  // (1)
      if (c > c0) stage(c - 1);
      issue(c - 2);
      lds_barrier();  // (2)
    }
  }
}

// ---- the walk: every gradient of a segment's chunks, from the last to the first --------------------------------------------
// Grid segments x heads (long segments first), twelve waves:
//   0, 1   the gradient of the state, 32 value columns each (GbChain)
//   2, 3   Vn = T B (V - E Kh S) for 32 value columns each, then dQh^T of 32 tokens each
//   4-6    the three token x token tiles (j tile, i tile) = (0,0), (0,1), (1,1), rows j in the registers, the lane holds i: P,
//          grad P and grad A with their gating and their sums over the rows and columns
//   7      per-token factors, e^{gamma_L} <G', S>, and the sums for d g and d beta
//   8-11   dKh^T, one 32 x 32 tile each (lane = token: per-token factors are one scalar, row sums mostly in-lane)
// Waves 4-7 stage k, q of the next chunk into the other set of tiles, waves 8-11 dO, v, S, T; waves 0, 1 write dv, waves 2, 3
// the rows of dq and dk of the chunk before. Barriers per chunk: (1) P, Vn, G' complete; (2) X, N complete; (3) M complete; (4)
// the partial row sums are complete; (5) the next chunk's tiles and the rows of dq and dk are complete.
// Bound by the latency of these five stages: 2.9 + 3.2 + 2.8 + 2.8 + 1.7 thousand cycles per chunk, of which a SIMD issues
// vector instructions for about 7 000 (one workgroup per CU: 160 KB of LDS). 184 - 205 us, by card, at 60 000 tokens x 8 heads; all roles on
// eight waves with one set of tiles and seven barriers took 256 us, two such workgroups per CU with 128 registers 395 us
// (they spill, and every reload waits for the tiles being prefetched). Each role has its own loop for that reason too: a loop
// shared by two roles copies the registers being loaded at its end and so waits for them (+7 us).
template <typename T>
__global__ void __launch_bounds__(GB_WALK_THREADS, 3)
    gdrb_walk_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ dout,
                     const unsigned char* __restrict__ recs, const unsigned char* __restrict__ states, const GdrPlanView pv,
                     const int32_t* __restrict__ chunk_tok0, const int32_t* __restrict__ chunk_len,
                     const unsigned char* __restrict__ Mt, const float* __restrict__ Dc, const unsigned char* __restrict__ Nr,
                     const unsigned char* __restrict__ Mgrp, const unsigned char* __restrict__ Ngrp,
                     const float* __restrict__ Dgrp, int gmax, const float* __restrict__ dht, T* __restrict__ dq,
                     T* __restrict__ dk, T* __restrict__ dv, float* __restrict__ dg, float* __restrict__ dbeta,
                     float* __restrict__ dh0, int H, int HV, float scale, int l2norm, int Kw, int Vw) {
  using OT = T;
  using X8 = typename OpVec<OT>::x8;
  using X4 = typename OpVec<OT>::x4;
  using SM = GbWalkSmem;
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char *const b_p = smem + SM::OFF_P, *const b_n = smem + SM::OFF_N, *const b_m = smem + SM::OFF_M;
  unsigned char *const b_g = smem + SM::OFF_G, *const b_x = smem + SM::OFF_X;
  OT* const b_oq = reinterpret_cast<OT*>(smem + SM::OFF_OQ);
  OT* const b_ok = reinterpret_cast<OT*>(smem + SM::OFF_OK);
  float* const s_sum = reinterpret_cast<float*>(smem + SM::OFF_SUM);

  const int seg = pv.seg_order[blockIdx.x / HV], hv = blockIdx.x % HV, h = hv / (HV / H);
  const int flags = pv.seg_flags[seg];
  const int c0 = pv.seg_chunk0[seg], nc = pv.seg_nchunks[seg], seq = pv.seg_seq[seg], cl = c0 + nc - 1;
  const int wave = uniform(threadIdx.x >> 6);
  // What depends on the lane is derived again for every chunk from a lane index the compiler cannot see through: left
  // alone it computes some hundred LDS addresses before the loops and spills them (and a reload from scratch memory waits
  // for every tile that is being prefetched).
  int tid, lane, hh, ln;
  auto lanes = [&]() __attribute__((always_inline)) {
    lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    tid = 64 * wave + lane;
    hh = lane >> 5;
    ln = lane & 31;
  };
  lanes();
  // the chunks of a sequence follow one another, only its last one may be shorter: no table look-up in the loops
  const int tok_first = nc > 0 ? chunk_tok0[c0] : 0, len_last = nc > 0 ? chunk_len[cl] : 0;
  auto tok_of = [&](int c) { return tok_first + GDR_C * (c - c0); };
  auto len_of = [&](int c) { return c == cl ? len_last : GDR_C; };
  auto rec_of = [&](int c) { return recs + ((size_t)c * HV + hv) * REC_BYTES; };
  auto set_of = [&](int c) { return gb_tiles<OT, true>(smem, (cl - c) & 1); };  // (as in the source pass)

  // (the result goes to waves 0, 1 through LDS: in registers it would be live through the loops of every other role)
  float* const xs = reinterpret_cast<float*>(b_g);
  static_assert(SM::OFF_X == SM::OFF_G + 8192, "two column slabs of 64 rows of float");
  {
    // The gradient behind the sequence pushed through the composites of the later segments: whole groups of
    // GDR_SCAN_GROUP first (gmax > 0), then the segments between them and this one; G <- d G + N' + M'^T G. Waves 0 .. 3:
    // wave w owns rows 32 (w / 2) .. of column slab w % 2 and takes the other rows as operand through LDS, so that the
    // composites of two steps fit the registers (one wave with all rows of a slab would need 128 for them).
    const int seg0 = pv.seq_seg0[seq], last = seg0 + pv.seq_nseg[seq] - 1, behind = last - seg;
    const int lead = gmax > 0 ? behind / GDR_SCAN_GROUP : 0, nst = lead + behind - lead * GDR_SCAN_GROUP;
    const int slab = wave & 1, km = (wave >> 1) & 1;
    // The walk starts at the last of the maps that cut off what lies behind them (from a gradient of zero behind the sequence; a
    // given one may not be finite). The look at the decays takes its time beside the first maps' loads (in front of them, where
    // nothing cuts off: pass 174.7 us, without any look 173.1, so 173.3; 60 000 tokens x 8).
    const bool look = nst > 1 && !dht;
    const int pl = min(lane, nst - 1);
    const size_t at = (size_t)(pl < lead ? seq * gmax + pl : last - lead * GDR_SCAN_GROUP - (pl - lead)) * HV + hv;
    const float dl = look ? (pl < lead ? Dgrp : Dc)[at] : 0.0f;
    auto start = [&]() __attribute__((always_inline)) { return look ? max(0, uniform(gdr_leading_cuts(dl, nst, lane)) - 1) : 0; };
    if (wave >= 4) {
      for (int p = start(); p < nst; ++p) lds_barrier();
      lds_barrier();
      lds_barrier();
    } else {
      f32x16 S = zero16();
      if (dht) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          S[r] = dht[(((size_t)seq * HV + hv) * 64 + 32 * km + acc_row(r, hh)) * 64 + 32 * slab + ln];
      }
      X8 rm[2][4];
      f32x4 rn[2][4];
      float rd[2];
      auto walk_issue = [&](int p, X8* m, f32x4* n, float& d) __attribute__((always_inline)) {
        p = uniform(max(0, min(p, nst - 1)));
        const bool top = p < lead;
        const size_t sh = (size_t)(top ? seq * gmax + p : last - lead * GDR_SCAN_GROUP - (p - lead)) * HV + hv;
        const X8* M = reinterpret_cast<const X8*>((top ? Mgrp : Mt) + sh * GDR_STATE_BYTES);
        const f32x4* N = reinterpret_cast<const f32x4*>((top ? Ngrp : Nr) + (sh * 2 + slab) * GDR_STATE_BYTES);
#pragma unroll
        for (int f = 0; f < 4; ++f) m[f] = M[(km * 4 + f) * 64 + lane];
#pragma unroll
        for (int f = 0; f < 4; ++f) n[f] = N[(km * 4 + f) * 64 + lane];
        d = (top ? Dgrp : Dc)[sh];
      };
      auto walk_step = [&](int p, const X8* m, const f32x4* n, float d) __attribute__((always_inline)) {
        unsigned char* xbuf = (p & 1 ? b_x : b_g) + slab * 4096;
        op_frag_store<OT>(xbuf, 2 * km + 0, lane, acc_to_op<OT>(S, 0));
        op_frag_store<OT>(xbuf, 2 * km + 1, lane, acc_to_op<OT>(S, 8));
        f32x16 acc;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * q4 + e] = __builtin_fmaf(d, S[4 * q4 + e], n[q4][e]);
        lds_barrier();
#pragma unroll
        for (int f = 0; f < 4; ++f) acc = mfma32(m[f], op_frag_load<OT>(xbuf, f, lane), acc);
        S = acc;
      };
      if (nst > 0) {
        __builtin_amdgcn_sched_barrier(0);
        walk_issue(0, rm[0], rn[0], rd[0]);
        walk_issue(1, rm[1], rn[1], rd[1]);
        __builtin_amdgcn_sched_barrier(0);
        const int from = start();
        asm volatile("" : "+s"(rd[0]), "+s"(rd[1]));  // (these loads stay in front of the branch)
        if (from > 0) {
          walk_issue(from, rm[0], rn[0], rd[0]);
          walk_issue(from + 1, rm[1], rn[1], rd[1]);
        }
        for (int p = from; p < nst; p += 2) {
          walk_step(p, rm[0], rn[0], rd[0]);
          walk_issue(p + 2, rm[0], rn[0], rd[0]);
          if (p + 1 < nst) walk_step(p + 1, rm[1], rn[1], rd[1]);
          walk_issue(p + 3, rm[1], rn[1], rd[1]);
        }
      }
      lds_barrier();  // (the last step's operands have been read)
#pragma unroll
      for (int r = 0; r < 16; ++r) xs[(32 * slab + 16 * km + r) * 64 + lane] = S[r];
      lds_barrier();
    }
  }
  gb_zero_upper<OT, true>(smem, tid);

  // ---- d v = beta X and the products X . v (waves 0, 1): 32 tokens per wave, 16 at a time
  typename Raw8<T>::type vre[2][2];
  auto load_v = [&](int tok0, int len) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const int xtok = 32 * wave + 16 * w + (lane & 15);
      const T* at = v + ((size_t)tok0 * HV + hv) * 64 + (uint32_t)(min(xtok, len - 1) * HV * 64 + 8 * (lane >> 4));
#pragma unroll
      for (int u = 0; u < 2; ++u) vre[w][u] = *reinterpret_cast<const typename Raw8<T>::type*>(at + 32 * u);
    }
  };
  auto rows_dv = [&](const GbTiles<OT>& t, int tok0, int len) __attribute__((always_inline)) {
    const int L = lane & 15, cc = 8 * (lane >> 4) + (L >> 2);
    const unsigned char* p = b_x + wave * 2048 + (32 * (L & 1) + cc) * 16 + ((L >> 1) & 1) * 8;
    X4 x4[2][4];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        x4[w][u] = op_lds_read_tr4<OT>(reinterpret_cast<const OT*>(p + w * 1024 + (u >> 1) * 4096 + (u & 1) * 64));
    // (X . v of both before the first store: the compiler cannot count conditional stores, and a wait for v behind them was
    // also one for them)
    float x[2] = {0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x[w] += (float)x4[w][2 * u][e] * (float)vre[w][u][e] + (float)x4[w][2 * u + 1][e] * (float)vre[w][u][4 + e];
    asm volatile("" : "+v"(x[0]), "+v"(x[1]));
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const int xtok = 32 * wave + 16 * w + L;
      const float b = t.beta[xtok];
      T* at = dv + ((size_t)tok0 * HV + hv) * Vw + (uint32_t)(xtok * HV * Vw + 8 * (lane >> 4));
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        typename Raw8<T>::type out;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out[e] = (T)(b * (float)x4[w][2 * u][e]);
          out[4 + e] = (T)(b * (float)x4[w][2 * u + 1][e]);
        }
        if (xtok < len && 32 * u + 8 * (lane >> 4) < Vw) *reinterpret_cast<typename Raw8<T>::type*>(at + 32 * u) = out;
      }
      x[w] += __shfl_xor(x[w], 16);
      x[w] = gb_both_halves(x[w]);
      if (lane < 16) s_sum[GbSums::XV + xtok] = x[w];
    }
  };
  // rows of a gradient tile (rows 32 kt .., lane = token tok) through the l2 normalisation: y the normalised input row, dot
  // the row's product with it, cn the normalisation factor (1 / (|x| + eps) in the recurrent form: |x| = 1 / c - eps)
  auto rows_out = [&](OT* to, const OT* y, const f32x16& acc, int kt, int tok, float dot, float cn) __attribute__((always_inline)) {
    float fy = 0.0f, fc = 1.0f;
    if (l2norm != GDR_L2_NONE) {
      fy = cn * dot;
      fc = cn;
      if (l2norm == GDR_L2_RECURRENT) fy = dot / fmaxf(1.0f / cn - 1e-6f, 1e-30f);
    }
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const int at = tok * GB_LS + 32 * kt + 8 * b4 + 4 * hh;
      const X4 y4 = *reinterpret_cast<const X4*>(&y[at]);
      X4 o4;
#pragma unroll
      for (int e = 0; e < 4; ++e) o4[e] = (OT)(fc * acc[4 * b4 + e] - fy * (float)y4[e]);
      *reinterpret_cast<X4*>(&to[at]) = o4;
    }
  };
  auto row_dot = [&](const OT* y, const f32x16& acc, int kt, int tok) __attribute__((always_inline)) {
    float dot = 0.0f;
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const X4 y4 = *reinterpret_cast<const X4*>(&y[tok * GB_LS + 32 * kt + 8 * b4 + 4 * hh]);
#pragma unroll
      for (int e = 0; e < 4; ++e) dot += (float)y4[e] * acc[4 * b4 + e];
    }
    return dot;
  };

  if (wave < 2) {
    // ======================================= the gradient of the state =======================================
    GbChain<OT> ch;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      ch.G[0][r] = xs[(32 * wave + r) * 64 + lane];
      ch.G[1][r] = xs[(32 * wave + 16 + r) * 64 + lane];
    }
    if (nc > 0) lds_barrier();  // (0) the tiles of the first chunk are complete
    for (int c = cl; c >= c0; --c) {
      lanes();
      const int tok0 = tok_of(c), len = len_of(c);
      const GbTiles<OT> t = set_of(c);
      ch.state_rows(t, b_g, wave, lane, hh, ln);
      lds_barrier();  // (1)
      ch.chunk_rows(t, b_p, b_x, wave, lane, hh);
      load_v(tok0, len);
      lds_barrier();  // (2)
      ch.update(t, scale, wave, lane, hh);
      lds_barrier();  // (3)
      rows_dv(t, tok0, len);
      lds_barrier();  // (4)
      lds_barrier();  // (5)
    }
    if (dh0 && (flags & SEG_FIRST)) {
#pragma unroll
      for (int km = 0; km < 2; ++km)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          dh0[(((size_t)seq * HV + hv) * 64 + 32 * km + acc_row(r, hh)) * 64 + 32 * wave + ln] = ch.G[km][r];
    }
  } else if (nc == 0) {
    return;
  } else if (wave < 4) {
    // =============================================== Vn, dQh^T ===============================================
    const int vn = wave - 2;
    auto store_rows = [&](int c) __attribute__((always_inline)) {  // dq, dk of chunk c
      const int tok0 = tok_of(c), len = len_of(c), row0 = 8 * vn + (lane >> 3), part = lane & 7;
      const size_t first = ((size_t)tok0 * HV + hv) * Kw;
      X8 o[8];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        o[u] = *reinterpret_cast<const X8*>(&b_oq[(16 * u + row0) * GB_LS + 8 * part]);
        o[4 + u] = *reinterpret_cast<const X8*>(&b_ok[(16 * u + row0) * GB_LS + 8 * part]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = 16 * u + row0;
        if (row < len && 8 * part < Kw) {
          const uint32_t at = (uint32_t)(row * HV * Kw + 8 * part);
          *reinterpret_cast<X8*>(dq + first + at) = o[u];
          *reinterpret_cast<X8*>(dk + first + at) = o[4 + u];
        }
      }
    };
    lds_barrier();  // (0)
    for (int c = cl; c >= c0; --c) {
      lanes();
      const int tok = 32 * vn + ln;
      const GbTiles<OT> t = set_of(c);
      {
        X8 Rb[4];
        OT* const vt = t.v + vn * 2048;
        {
          X8 Sb[4], fk[8];
#pragma unroll
          for (int f = 0; f < 8; ++f) fk[f] = gb_rows_k<OT>(t.k, 32 * (f >> 2) + ln, 16 * (f & 3), hh);
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) Sb[ks] = op_frag_load<OT>(t.s, vn * 4 + ks, lane);
          X4 vv[8];
#pragma unroll
          for (int b = 0; b < 8; ++b) vv[b] = op_ld_col4<OT>(vt, 32, 0, 8 * b, lane);
          gb_pin(fk);
          gb_pin(Sb);
          f32x16 r[2];
          r[0] = zero16();
          r[1] = zero16();
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            r[0] = mfma32(fk[ks], Sb[ks], r[0]);
            r[1] = mfma32(fk[4 + ks], Sb[ks], r[1]);
          }
#pragma unroll
          for (int tm = 0; tm < 2; ++tm) {
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4) {  // R = beta (v - e^gamma Kh S)
              const f32x4 fb = gb_rows4(t.beta, 32 * tm, b4, hh), fe = gb_rows4(t.eg, 32 * tm, b4, hh);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                r[tm][4 * b4 + e] = fb[e] * ((float)vv[4 * tm + b4][e] - fe[e] * r[tm][4 * b4 + e]);
            }
            Rb[2 * tm + 0] = acc_to_op<OT>(r[tm], 0);
            Rb[2 * tm + 1] = acc_to_op<OT>(r[tm], 8);
          }
        }
        X8 ft[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) ft[f] = op_ld_kappa<OT>(t.t + (f >> 1) * 32 * GB_TS, GB_TS, ln, 16 * (f & 1), hh);
        gb_pin(ft);
        f32x16 r[2];
        r[0] = zero16();
        r[1] = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          if (ks < 2) r[0] = mfma32(ft[ks], Rb[ks], r[0]);
          r[1] = mfma32(ft[2 + ks], Rb[ks], r[1]);
        }
        unsigned char* const vf = reinterpret_cast<unsigned char*>(t.v);  // (over this wave's own half of v, which it has read)
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) {
          op_frag_store<OT>(vf, vn * 4 + 2 * tm + 0, lane, acc_to_op<OT>(r[tm], 0));
          op_frag_store<OT>(vf, vn * 4 + 2 * tm + 1, lane, acc_to_op<OT>(r[tm], 8));
        }
      }
      lds_barrier();  // (1)
      f32x16 acc[2];  // rows 0-31, 32-63 of dQh^T: scale e^gamma S dO^T + Kh^T N^T
      float rs_g = 0.0f;
      const float fs = scale * t.eg[tok];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        acc[kt] = gb_mm<OT>(zero16(), [&](int ks) { return fr_tr<OT, false>(t.s, 32 * kt, 16 * ks, lane); },
                            [&](int ks) { return gb_rows_n<OT>(t.dout, tok, 16 * ks, hh); });
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[kt][r] *= fs;
        rs_g += row_dot(t.q, acc[kt], kt, tok);
      }
      if (c < cl) store_rows(c + 1);
      lds_barrier();  // (2)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        acc[kt] = gb_mm_tri<OT, true>(acc[kt], vn, [&](int ks) { return gb_cols<OT>(t.k, 32 * kt, 16 * ks, lane); },
                                      [&](int ks) { return op_frag_load<OT>(b_n + (vn + ks / 2) * GB_TRI, ks & 1, lane); });
      lds_barrier();  // (3)
      rs_g = gb_both_halves(rs_g);
      if (hh == 0) s_sum[GbSums::DGAM + 32 * vn + ln] = rs_g;
      const float dot = gb_both_halves(row_dot(t.q, acc[0], 0, tok) + row_dot(t.q, acc[1], 1, tok));
      const float cn = t.rq[tok];
      rows_out(b_oq, t.q, acc[0], 0, tok, dot, cn);
      rows_out(b_oq, t.q, acc[1], 1, tok, dot, cn);
      lds_barrier();  // (4)
      lds_barrier();  // (5)
    }
    store_rows(c0);
  } else if (wave < 7) {
    // ================================ the token x token tiles; staging of k, q ================================
    GbStageKQ<T> st;
    const int tw = wave - 4, jt = tw == 2 ? 1 : 0, it = tw == 0 ? 0 : 1;
    auto issue = [&](int c) __attribute__((always_inline)) {
      c = uniform(max(c, c0));
      st.issue(k, q, rec_of(c), tok_of(c), len_of(c), H, h, tid - 256);
    };
    issue(cl);
    st.stage_k(set_of(cl), len_of(cl), l2norm, tid - 256);
    st.stage_q(set_of(cl), len_of(cl), l2norm, tid - 256);
    issue(cl - 1);
    lds_barrier();  // (0)
    for (int c = cl; c >= c0; --c) {
      lanes();
      const GbTiles<OT> t = set_of(c);
      const int i = 32 * it + ln;
      f32x16 pm = gb_pair<OT>(t.k, jt, t.q, it, ln, hh), gm = gb_ratio(t.gam, jt, it, 0, ln, hh);
#pragma unroll
      for (int r = 0; r < 16; ++r) pm[r] *= scale * gm[r];
      gb_store_tile<OT>(b_p + tw * GB_TRI, pm, lane);
      const f32x16 gk = gb_pair<OT>(t.k, jt, t.k, it, ln, hh);
      lds_barrier();  // (1)
      const unsigned char* vf = reinterpret_cast<const unsigned char*>(t.v);
      float rs_g = 0.0f, rs_b = 0.0f, rs_c, cs[16];  // sums over the tile's rows (of column i) and columns (of a row)
      {  // grad P = dO Vn^T
        f32x16 n = gb_mm<OT>(zero16(), [&](int ks) { return fr_tr<OT, false>(vf, 32 * jt, 16 * ks, lane); },
                             [&](int ks) { return gb_rows_n<OT>(t.dout, i, 16 * ks, hh); });
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          cs[r] = n[r] * pm[r];
          rs_g += cs[r];
          n[r] *= scale * gm[r];
        }
        gb_store_tile<OT>(b_n + tw * GB_TRI, n, lane);
        rs_c = gb_half_sums16(cs, lane);
      }
      // (strictly below the diagonal for grad A)
      if (jt == it) {
#pragma unroll
        for (int r = 0; r < 16; ++r) gm[r] = ln == acc_row(r, hh) ? 0.0f : gm[r];
      }
      const float bi = t.beta[i];
      lds_barrier();  // (2)
      f32x16 da = gb_mm<OT>(zero16(), [&](int ks) { return fr_tr<OT, false>(vf, 32 * jt, 16 * ks, lane); },
                            [&](int ks) { return fr_tr<OT, false>(b_x, 32 * it, 16 * ks, lane); });
#pragma unroll
      for (int r = 0; r < 16; ++r) {  // grad A = -X Vn^T
        // grad A_ij Gamma_ij, and grad A_ij times A_ij / beta_i and times A_ij
        const float ga = -da[r] * gm[r], b = ga * gk[r], a = b * bi;
        rs_b += b;
        rs_g += a;
        cs[r] = a;
        da[r] = ga * bi;
      }
      gb_store_tile<OT>(b_m + tw * GB_TRI, da, lane);
      lds_barrier();  // (3)
      rs_c += gb_half_sums16(cs, lane);
      rs_g = gb_both_halves(rs_g);
      rs_b = gb_both_halves(rs_b);
      if (hh == 0) {
        s_sum[GbSums::TILE_G + 32 * tw + ln] = rs_g;
        s_sum[GbSums::TILE_B + 32 * tw + ln] = rs_b;
      }
      if (!(ln & 1)) s_sum[GbSums::TILE_C + 32 * tw + 8 * (ln >> 3) + 4 * hh + ((ln >> 1) & 3)] = rs_c;
      if (c > c0) st.stage_k(set_of(c - 1), len_of(c - 1), l2norm, tid - 256);
      lds_barrier();  // (4)
      if (c > c0) st.stage_q(set_of(c - 1), len_of(c - 1), l2norm, tid - 256);
      issue(c - 2);
      lds_barrier();  // (5)
    }
  } else if (wave == 7) {
    // ============================ per-token factors, d g, d beta; staging of k, q ============================
    // (a loop of its own: joined with the one above, the registers being loaded are copied at its end, waiting for them)
    GbStageKQ<T> st;
    GbStageFactors sf;
    auto issue = [&](int c) __attribute__((always_inline)) {
      c = uniform(max(c, c0));
      st.issue(k, q, rec_of(c), tok_of(c), len_of(c), H, h, tid - 256);
      sf.issue(rec_of(c), lane);
    };
    issue(cl);
    st.stage_k(set_of(cl), len_of(cl), l2norm, tid - 256);
    st.stage_q(set_of(cl), len_of(cl), l2norm, tid - 256);
    sf.stage(set_of(cl), lane);
    issue(cl - 1);
    lds_barrier();  // (0)
    for (int c = cl; c >= c0; --c) {
      lanes();
      const int tok0 = tok_of(c), len = len_of(c);
      const GbTiles<OT> t = set_of(c);
      lds_barrier();  // (1)
      float gs = 0.0f;  // e^{gamma_L} <G', S>
#pragma unroll
      for (int f = 0; f < 8; ++f) {
        const X8 xa = op_frag_load<OT>(b_g, f, lane), xb = op_frag_load<OT>(t.s, f, lane);
#pragma unroll
        for (int e = 0; e < 8; ++e) gs = __builtin_fmaf((float)xa[e], (float)xb[e], gs);
      }
      gs = gb_half_sum(gs) * __builtin_amdgcn_exp2f(t.gam[63]);
      if (ln == 0) s_sum[GbSums::GL + 8 + hh] = gs;
      lds_barrier();  // (2)
      lds_barrier();  // (3)
      if (c > c0) {
        st.stage_k(set_of(c - 1), len_of(c - 1), l2norm, tid - 256);
        st.stage_q(set_of(c - 1), len_of(c - 1), l2norm, tid - 256);
        sf.stage(set_of(c - 1), lane);
      }
      issue(c - 2);
      lds_barrier();  // (4)
      // d g = the sum of d gamma over the later rows of the chunk (gamma_i = g_0 + ... + g_i); d beta
      const float* w = s_sum + GbSums::DGAM + 32 * hh + ln;  // (lane = token 32 hh + ln; tiles (0,0), (0,1), (1,1))
      const float* s = s_sum + ln;
      float x = w[0] + (w[64] + w[128]);
      x += s[GbSums::TILE_G + 32 * hh] + (hh ? s[GbSums::TILE_G + 64] : 0.0f);
      x -= s[GbSums::TILE_C + 64 * hh] + (hh ? 0.0f : s[GbSums::TILE_C + 32]);
      const float db = (s[GbSums::TILE_B + 32 * hh] + (hh ? s[GbSums::TILE_B + 64] : 0.0f)) +
                       (s[GbSums::DBETA + 32 * hh] + s[GbSums::DBETA + 64 + 32 * hh]) +
                       s_sum[GbSums::XV + lane];
      if (lane == len - 1) {
        const float* g = s_sum + GbSums::GL;
        x += ((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7])) + (g[8] + g[9]);
      }
      if (lane >= len) x = 0.0f;
      const float incl = wave_inclusive_scan(x);  // (inclusive scan from the last lane down: total - exclusive prefix)
      const float total = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(incl), 63));
      if (lane < len) {
        dg[(size_t)(tok0 + lane) * HV + hv] = total - incl + x;
        dbeta[(size_t)(tok0 + lane) * HV + hv] = db;
      }
      lds_barrier();  // (5)
    }
  } else {
    // ============================ dKh^T; staging of dO, v, S, T; the rows of dq and dk ============================
    GbStageRest<T, 256, true> st;
    const int tw = wave - 8, kt = tw >> 1, tt = tw & 1;
    auto issue = [&](int c) {
      c = uniform(max(c, c0));
      st.issue(dout, v, rec_of(c), states + ((size_t)c * HV + hv) * GDR_STATE_BYTES, tok_of(c), len_of(c), HV, hv, tid - 512);
    };
    issue(cl);
    st.stage(set_of(cl), len_of(cl), tid - 512);
    issue(cl - 1);
    lds_barrier();  // (0)
    for (int c = cl; c >= c0; --c) {
      lanes();
      const int tok = 32 * tt + ln;
      const GbTiles<OT> t = set_of(c);
      if (c > c0) st.stage(set_of(c - 1), len_of(c - 1), tid - 512);
      issue(c - 2);
      lds_barrier();  // (1)
      const unsigned char* vf = reinterpret_cast<const unsigned char*>(t.v);
      float rs_g, rs_b = 0.0f;  // the terms of d gamma / d beta of this lane's token
      // D G' Vn^T
      f32x16 acc = gb_mm<OT>(zero16(), [&](int ks) { return fr_tr<OT, false>(b_g, 32 * kt, 16 * ks, lane); },
                             [&](int ks) { return fr_tr<OT, false>(vf, 32 * tt, 16 * ks, lane); });
      {
        const float fd = t.dk[tok];
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] *= fd;
        const float x = row_dot(t.k, acc, kt, tok);
        rs_g = -x;
        const float gl = gb_half_sum(x);
        if (ln == 0) s_sum[GbSums::GL + 2 * tw + hh] = gl;
      }
      lds_barrier();  // (2)
      {  // -(S X^T), the gradient of beta e^gamma Kh
        f32x16 xw = gb_mm<OT>(zero16(), [&](int ks) { return fr_tr<OT, false>(t.s, 32 * kt, 16 * ks, lane); },
                              [&](int ks) { return fr_tr<OT, false>(b_x, 32 * tt, 16 * ks, lane); });
        const float fe = -t.eg[tok], fb = t.beta[tok];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          xw[r] *= fe;
          acc[r] = __builtin_fmaf(fb, xw[r], acc[r]);
        }
        rs_b = row_dot(t.k, xw, kt, tok);
        rs_g = gb_both_halves(__builtin_fmaf(fb, rs_b, rs_g));
        rs_b = gb_both_halves(rs_b);
        if (hh == 0) {
          s_sum[GbSums::DBETA + 32 * tw + ln] = rs_b;
          s_sum[GbSums::DGAM + 64 + 32 * tw + ln] = rs_g;
        }
      }
      lds_barrier();  // (3)
      // + (N^T Qh)^T
      acc = gb_mm_tri<OT, false>(acc, tt, [&](int ks) { return gb_cols<OT>(t.q, 32 * kt, 16 * ks, lane); }, [&](int ks) {
        return fr_tr<OT, true>(b_n + (tt == 0 ? ks / 2 : 2) * GB_TRI, 0, 16 * (ks & 1), lane);
      });
      // + (M Kh)^T + (M^T Kh)^T
      acc = gb_mm_tri<OT, true>(acc, tt, [&](int ks) { return gb_cols<OT>(t.k, 32 * kt, 16 * ks, lane); }, [&](int ks) {
        return op_frag_load<OT>(b_m + (tt + ks / 2) * GB_TRI, ks & 1, lane);
      });
      acc = gb_mm_tri<OT, false>(acc, tt, [&](int ks) { return gb_cols<OT>(t.k, 32 * kt, 16 * ks, lane); }, [&](int ks) {
        return fr_tr<OT, true>(b_m + (tt == 0 ? ks / 2 : 2) * GB_TRI, 0, 16 * (ks & 1), lane);
      });
      float dot = gb_both_halves(row_dot(t.k, acc, kt, tok));
      if (hh == 0) s_sum[GbSums::DOTK + 64 * kt + tok] = dot;
      lds_barrier();  // (4)
      dot = s_sum[GbSums::DOTK + tok] + s_sum[GbSums::DOTK + 64 + tok];
      rows_out(b_ok, t.k, acc, kt, tok, dot, t.rk[tok]);
      lds_barrier();  // (5)
    }
  }
}

// ---- host ----------------------------------------------------------------------------------------------------------
struct GbWorkspace {
  int64_t nr, gm, gn, gd, dr, max_groups, bytes;
};
static GbWorkspace gb_workspace(int64_t segs, int HV) {
  GbWorkspace w;
  int64_t off = 0;
  auto take = [&](int64_t bytes) { const int64_t o = off; off += lampa_align_up(bytes, 256); return o; };
  w.max_groups = segs / GDR_SCAN_GROUP + 2;
  w.nr = take(segs * HV * 2 * (int64_t)GDR_STATE_BYTES);
  w.gm = take(w.max_groups * HV * (int64_t)GDR_STATE_BYTES);
  w.gn = take(w.max_groups * HV * 2 * (int64_t)GDR_STATE_BYTES);
  w.gd = take(w.max_groups * HV * 4);
  w.dr = take(segs * HV * 4);
  w.bytes = off;
  return w;
}

template <typename T>
static int gb_run(const void* q, const void* k, const void* v, const void* dout, const float* dht, void* dq, void* dk,
                  void* dv, float* dg, float* dbeta, float* dh0, const int32_t* ph, const int32_t* pd,
                  const unsigned char* saved, int H, int HV, int Kw, int Vw, float scale, int l2norm, unsigned char* ws,
                  hipStream_t s) {
  const int n_seq = ph[PLAN_N_SEQ], chunks = ph[PLAN_TOTAL_CHUNKS], segs = ph[PLAN_N_SEGMENTS];
  const GdrSaved sv = gdr_saved_layout(chunks, segs, HV);
  const GbWorkspace w = gb_workspace(segs, HV);
  static bool attr_set[64] = {};
  static std::mutex attr_lock;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return LAMPA_ERR_LAUNCH;
  {
    std::lock_guard<std::mutex> hold(attr_lock);
    if (!attr_set[dev]) {
      if (hipFuncSetAttribute((const void*)gdrb_source_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              GbSourceSmem::BYTES) != hipSuccess ||
          hipFuncSetAttribute((const void*)gdrb_walk_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              GbWalkSmem::BYTES) != hipSuccess)
        return LAMPA_ERR_LAUNCH;
      attr_set[dev] = true;
    }
  }
  const GdrPlanView pv = gdr_plan_view(ph, pd);
  int max_nseg = 0;
  for (int i = 0; i < n_seq; ++i) max_nseg = ph[ph[PLAN_OFF_SEQ_NSEG] + i] > max_nseg ? ph[ph[PLAN_OFF_SEQ_NSEG] + i] : max_nseg;
  const int groups = (max_nseg + GDR_SCAN_GROUP - 1) / GDR_SCAN_GROUP;
  const int gmax = max_nseg >= 3 * GDR_SCAN_GROUP && (int64_t)n_seq * groups <= w.max_groups ? groups : 0;
  unsigned char *Nr = ws + w.nr, *Gm = ws + w.gm, *Gn = ws + w.gn;
  float* Gd = (float*)(ws + w.gd);
  const unsigned char *recs = saved + sv.off_rec, *states = saved + sv.off_states, *Mt = saved + sv.off_mt;
  const float* Dc = (const float*)(saved + sv.off_d);
  float* Dr = (float*)(ws + w.dr);
  LAMPA_PROF(s, "start");
  if (segs > n_seq) {
    hipLaunchKernelGGL((gdrb_source_kernel<T>), dim3(segs * HV), dim3(GB_SOURCE_THREADS), GbSourceSmem::BYTES, s, (const T*)q,
                       (const T*)k, (const T*)dout, recs, pv, pv.chunk_tok0, pv.chunk_len, Nr, H, HV, scale, l2norm,
                       (const float*)(saved + sv.off_e), Dc, Dr);
    LAMPA_PROF(s, "gdrb_source_kernel");
    if (gmax > 0) {
      hipLaunchKernelGGL((gdr_scan2_kernel<T, 64, 64, 4, SCAN_GROUP, true>), dim3(4 * gmax, n_seq, HV), dim3(128), 0, s, pv, Mt,
                         Nr, (const float*)Dr, (const float*)nullptr, (float*)nullptr, Gm, Gn, Gd, HV, 0, gmax);
      LAMPA_PROF(s, "gdr_scan2_kernel<group, reversed>");
    }
  }
  hipLaunchKernelGGL((gdrb_walk_kernel<T>), dim3(segs * HV), dim3(GB_WALK_THREADS), GbWalkSmem::BYTES, s, (const T*)q,
                     (const T*)k, (const T*)v, (const T*)dout, recs, states, pv, pv.chunk_tok0, pv.chunk_len, Mt, (const float*)Dr, Nr, Gm, Gn,
                     Gd, gmax, dht, (T*)dq, (T*)dk, (T*)dv, dg, dbeta, dh0, H, HV, scale, l2norm, Kw, Vw);
  LAMPA_PROF(s, "gdrb_walk_kernel");
  return lampa_launch_status();
}

static bool gb_plan_ok(const int32_t* ph) {
  return ph && ph[PLAN_N_SEQ] >= 1 && ph[PLAN_N_SEGMENTS] >= ph[PLAN_N_SEQ] && ph[PLAN_TOTAL_CHUNKS] >= 0;
}

extern "C" int64_t lampa_gdr_bwd_saved_workspace_bytes(const int32_t* plan_host, int HV) {
  if (!gb_plan_ok(plan_host) || HV < 1) return LAMPA_ERR_INVALID;
  return gb_workspace(plan_host[PLAN_N_SEGMENTS], HV).bytes;
}

// Gradients from what lampa_gdr_chunk_fwd_train kept. q, k [tokens, H, 64]; v, dout [tokens, HV, 64]; dq, dk (one row per
// VALUE head) [tokens, HV, K], dv [tokens, HV, V] with K, V <= 64, multiples of 8 (the heads before they were padded); dg, dbeta fp32 [tokens, HV]; dht, dh0 fp32 [n_seq, HV, 64, 64] (nullable).
extern "C" int lampa_gdr_bwd_saved(const void* q, const void* k, const void* v, const void* saved, const void* dout,
                                   const float* dht, void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
                                   const int32_t* plan_host, const int32_t* plan_dev, int H, int HV, int K, int V, int dtype,
                                   float scale, int l2norm, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!q || !k || !v || !saved || !dout || !dq || !dk || !dv || !dg || !dbeta || !plan_host || !plan_dev)
    return LAMPA_ERR_INVALID;
  if (H < 1 || HV < H || HV % H != 0 || l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (!gdr_train_width(K) || !gdr_train_width(V) || (dtype != GDR_BF16 && dtype != GDR_FP16)) return LAMPA_ERR_UNSUPPORTED;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 15)
    return LAMPA_ERR_INVALID;
  if (!gb_plan_ok(plan_host)) return LAMPA_ERR_INVALID;
  if (!workspace || workspace_bytes < lampa_gdr_bwd_saved_workspace_bytes(plan_host, HV)) return LAMPA_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  unsigned char* ws = (unsigned char*)workspace;
  const unsigned char* sv = (const unsigned char*)saved;
  if (dtype == GDR_BF16)
    return gb_run<__bf16>(q, k, v, dout, dht, dq, dk, dv, dg, dbeta, dh0, plan_host, plan_dev, sv, H, HV, K, V, scale, l2norm, ws, s);
  return gb_run<_Float16>(q, k, v, dout, dht, dq, dk, dv, dg, dbeta, dh0, plan_host, plan_dev, sv, H, HV, K, V, scale, l2norm, ws, s);
}

// ---- the same from the inputs alone: the training form of the forward, then the pass above ------------------------------
#define GB_DEFAULT_CPS 16  // chunks per segment of the tables lampa_gdr_bwd_chunk_plan_fill makes (any plan will do)

extern "C" int64_t lampa_gdr_bwd_chunk_plan_size(const int64_t* cu_seqlens_host, int n_seq) {
  return lampa_gdr_plan_size(cu_seqlens_host, n_seq, GB_DEFAULT_CPS);
}
extern "C" int lampa_gdr_bwd_chunk_plan_fill(const int64_t* cu_seqlens_host, int n_seq, int32_t* plan) {
  return lampa_gdr_plan_fill(cu_seqlens_host, n_seq, GB_DEFAULT_CPS, plan);
}

struct GbChunkWorkspace {
  int64_t saved, fwd, bwd, o, fwd_bytes, bwd_bytes, bytes;
};
static GbChunkWorkspace gb_chunk_workspace(const int32_t* ph, int HV) {
  GbChunkWorkspace w;
  w.saved = 0;
  w.fwd = lampa_align_up(lampa_gdr_train_saved_bytes(ph, HV), 256);
  w.fwd_bytes = lampa_gdr_train_workspace_bytes(ph, HV);
  w.bwd = w.fwd + lampa_align_up(w.fwd_bytes, 256);
  w.bwd_bytes = lampa_gdr_bwd_saved_workspace_bytes(ph, HV);
  w.o = w.bwd + lampa_align_up(w.bwd_bytes, 256);
  w.bytes = w.o + (int64_t)ph[PLAN_TOTAL_TOKENS] * HV * 64 * 2 + 256;
  return w;
}
extern "C" int64_t lampa_gdr_bwd_chunk_workspace_bytes(const int32_t* plan_host, int HV) {
  if (!gb_plan_ok(plan_host) || HV < 1) return LAMPA_ERR_INVALID;
  return gb_chunk_workspace(plan_host, HV).bytes;
}
extern "C" int lampa_gdr_bwd_chunk(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                   const float* h0, const void* dout, const float* dht, void* dq, void* dk, void* dv,
                                   float* dg, float* dbeta, float* dh0, const int32_t* plan_host, const int32_t* plan_dev,
                                   int H, int HV, int K, int V, int dtype, float scale, int l2norm, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  if (!q || !k || !v || !g || !beta || !dout || !dq || !dk || !dv || !dg || !dbeta || !plan_host || !plan_dev)
    return LAMPA_ERR_INVALID;
  if (H < 1 || HV < 1 || l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (K != 64 || V != 64 || HV != H || (dtype != GDR_BF16 && dtype != GDR_FP16)) return LAMPA_ERR_UNSUPPORTED;
  if (!gb_plan_ok(plan_host)) return LAMPA_ERR_INVALID;
  if (!workspace || workspace_bytes < lampa_gdr_bwd_chunk_workspace_bytes(plan_host, HV)) return LAMPA_ERR_WORKSPACE;
  const GbChunkWorkspace w = gb_chunk_workspace(plan_host, HV);
  unsigned char* ws = (unsigned char*)workspace;
  const int rc = lampa_gdr_chunk_fwd_train(q, k, v, g, beta, ws + w.o, h0, nullptr, plan_host, plan_dev, H, HV, K, V, dtype,
                                           scale, l2norm, ws + w.saved, nullptr, ws + w.fwd, w.fwd_bytes, stream);
  if (rc != LAMPA_OK) return rc;
  return lampa_gdr_bwd_saved(q, k, v, ws + w.saved, dout, dht, dq, dk, dv, dg, dbeta, dh0, plan_host, plan_dev, H, HV, K, V,
                             dtype, scale, l2norm, ws + w.bwd, w.bwd_bytes, stream);
}
