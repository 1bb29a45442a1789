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
//   source    gdrb_segment_kernel<false>: every segment's N' (the walk below from a zero gradient, nothing else);
//   group     gdr_scan2_kernel, reversed: composites of groups of 8 segments of long sequences;
//   walk      gdrb_segment_kernel<true>: a workgroup pushes the gradient behind the sequence through the composites of the
//             later segments, then walks its own chunks from the last to the first and writes every gradient of each.
#include "gdr_chunk_kernels.h"
#include "gdr_train.h"
#include <mutex>

#define GB_THREADS 512
#define GB_LS 72                    // row stride (16-bit elements) of the k, q and dO tiles: 16-byte aligned rows
#define GB_TS 36                    // row stride of a 32 x 32 block of T
#define GB_TRI 2048                 // bytes of one 32 x 32 tile in operand fragment order

// LDS of the kernel (bytes). Fragment order of a 64 x 64 tile with rows r and columns c: fragment 4 (c / 32) + r / 16,
// lane 32 ((r / 4) % 2) + c % 32, element 4 ((r / 8) % 2) + r % 4 -- what a lane holds of an accumulator tile, rounded.
template <bool GRADS>
struct GbSmem {
  static constexpr int TILE = 64 * GB_LS * 2;
  static constexpr int OFF_K = 0;                           // kh rows; at the end of a chunk the rows of dk
  static constexpr int OFF_Q = OFF_K + TILE;                // qh rows; at the end of a chunk the rows of dq
  static constexpr int OFF_DO = OFF_Q + TILE;
  static constexpr int OFF_T = OFF_DO + TILE;               // T11 | T21 | T22; later M (grad A gated), three tiles
  static constexpr int OFF_P = OFF_T + 3 * 32 * GB_TS * 2;  // P, three tiles; later the waves' partial sums (GbSums)
  static constexpr int OFF_F = OFF_P + 3 * GB_TRI;
  static constexpr int OFF_N = OFF_F + 7 * 256;             // N (grad P gated), three tiles
  static constexpr int OFF_V = OFF_N + (GRADS ? 3 * GB_TRI : 0);  // v as two 64 x 32 tiles, then Vn (fragment order)
  static constexpr int OFF_S = OFF_V + (GRADS ? 8192 : 0);
  static constexpr int OFF_G = OFF_S + (GRADS ? 8192 : 0);
  static constexpr int OFF_X = OFF_G + (GRADS ? 8192 : 0);
  static constexpr int BYTES = OFF_X + (GRADS ? 8192 : 0);
};
static_assert(GbSmem<true>::BYTES <= 81920, "two workgroups per CU");

// The partial sums of a chunk (float offsets into the dead P tiles): every wave writes its own, wave 2 adds them up. (As
// LDS atomics they took a third of the kernel's LDS cycles.)
struct GbSums {
  static constexpr int DOTQ = 0;                 // [2][64] products of the rows of dQh / dKh with qh / kh, per half of the columns
  static constexpr int DOTK = DOTQ + 128;
  static constexpr int DGAM = DOTK + 128;        // [8 waves][32] d gamma of the wave's tokens 32 (wave % 2) ..
  static constexpr int TILE_G = DGAM + 256;      // [3 tiles][32] d gamma of the tile's columns i
  static constexpr int TILE_C = TILE_G + 96;     // [3 tiles][32] and of its rows j (to be subtracted)
  static constexpr int TILE_B = TILE_C + 96;     // [3 tiles][32] d beta of the columns
  static constexpr int DBETA = TILE_B + 96;      // [waves 4 .. 7][32] d beta of the wave's tokens
  static constexpr int XV = DBETA + 128;         // [2][64] X . v per half of the columns
  static constexpr int GL = XV + 128;            // [waves 4 .. 7][2] the terms of d gamma that belong to the chunk's last row
  static constexpr int FLOATS = GL + 8;
};
static_assert(GbSums::FLOATS * 4 <= 3 * GB_TRI, "partial sums over the P tiles");

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

// The walk of one (segment, head) from its last chunk to its first. Grid segments x heads (long segments first), eight
// waves. GRADS false: from a zero gradient, writes the segment's N' and nothing else.
//   waves 0, 1  the gradient of the state, 32 value columns each, in accumulators: dVn -> X -> the next gradient, every
//               intermediate handed on in registers (accumulator = operand, as in the forward pass)
//   waves 2, 3  Vn = T B (V - E Kh S) for 32 value columns each
//   waves 4-6   the three token x token tiles (j tile, i tile) = (0,0), (0,1), (1,1): P, then grad P and grad A with their
//               gating and their sums over the rows and columns (rows j in the registers, the lane holds i)
//   waves 0-3 / 4-7  one 32 x 32 tile each of dQh^T / dKh^T (lane = token: per-token factors and row sums are one scalar
//               or one in-lane sum)
// The tiles of the next chunk are loaded into registers while this one is worked on.
// Bound by the latency of a chunk's dependent stages (about 17 700 cycles per chunk, of which 2 000 stage, 10 000 are the
// four phases between barriers (0) and (4), and 3 900 the rows' normalisation and the stores). The gradients form takes one
// workgroup per CU (212 registers): two of them with 128 registers spill, and every reload waits for the tiles being
// prefetched (395 against 256 us at 60 000 tokens x 8 heads). The source form fits 128 and shares a CU (74 us).
template <typename T, bool GRADS>
__global__ void __launch_bounds__(GB_THREADS, GRADS ? 2 : 4)
    gdrb_segment_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                        const T* __restrict__ dout, const unsigned char* __restrict__ recs,
                        const unsigned char* __restrict__ states, const GdrPlanView pv,
                        const int32_t* __restrict__ chunk_tok0, const int32_t* __restrict__ chunk_len,
                        const unsigned char* __restrict__ Mt, const float* __restrict__ Dc,
                        unsigned char* __restrict__ Nr, const unsigned char* __restrict__ Mgrp,
                        const unsigned char* __restrict__ Ngrp, const float* __restrict__ Dgrp, int gmax,
                        const float* __restrict__ dht, T* __restrict__ dq, T* __restrict__ dk, T* __restrict__ dv,
                        float* __restrict__ dg, float* __restrict__ dbeta, float* __restrict__ dh0, int H, int HV,
                        float scale, int l2norm) {
  using OT = T;
  using X8 = typename OpVec<OT>::x8;
  using X4 = typename OpVec<OT>::x4;
  using SM = GbSmem<GRADS>;
  extern __shared__ __align__(16) unsigned char smem[];
  OT* const b_k = reinterpret_cast<OT*>(smem + SM::OFF_K);
  OT* const b_q = reinterpret_cast<OT*>(smem + SM::OFF_Q);
  OT* const b_do = reinterpret_cast<OT*>(smem + SM::OFF_DO);
  OT* const b_t = reinterpret_cast<OT*>(smem + SM::OFF_T);
  unsigned char* const b_m = smem + SM::OFF_T;
  unsigned char* const b_p = smem + SM::OFF_P;
  unsigned char* const b_n = smem + SM::OFF_N;
  unsigned char* const b_v = smem + SM::OFF_V;
  unsigned char* const b_s = smem + SM::OFF_S;
  unsigned char* const b_g = smem + SM::OFF_G;
  unsigned char* const b_x = smem + SM::OFF_X;
  float* const s_gam = reinterpret_cast<float*>(smem + SM::OFF_F);
  float* const s_beta = s_gam + 64;
  float* const s_eg = s_gam + 128;    // e^gamma
  float* const s_dk = s_gam + 192;    // e^{gamma_L - gamma}
  float* const s_rk = s_gam + 256;
  float* const s_rq = s_gam + 320;
  float* const s_sum = reinterpret_cast<float*>(b_p);  // GbSums (between barriers (2) and (6))

  const int seg = pv.seg_order[blockIdx.x / HV], hv = blockIdx.x % HV, h = hv / (HV / H);
  const int flags = pv.seg_flags[seg];
  if (!GRADS && (flags & SEG_FIRST)) return;  // nothing precedes the first segment of a sequence
  const int c0 = pv.seg_chunk0[seg], nc = pv.seg_nchunks[seg], seq = pv.seg_seq[seg];
  const int wave = uniform(threadIdx.x >> 6);
  const int kt = (wave >> 1) & 1, tt = wave & 1;  // this wave's tile of dQh^T / dKh^T: rows 32 kt, tokens 32 tt
  // Everything below that depends on the lane is derived again for every chunk from a thread index the compiler cannot see
  // through: left alone it computes some hundred LDS addresses before the loop and spills them.
  int tid, lane, hh, ln, srow, part, tok, xtok, xpart;
  auto lanes = [&]() __attribute__((always_inline)) {
    tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    lane = tid & 63;
    hh = lane >> 5;
    ln = lane & 31;
    srow = tid >> 3;  // staging: thread = (row, 8-column piece) of every tile
    part = tid & 7;
    tok = 32 * tt + ln;
    xtok = 16 * (wave & 3) + (lane & 15);  // this lane's piece of d v
    xpart = 4 * (wave >> 2) + (lane >> 4);
  };
  lanes();
  typename Raw8<T>::type pk, pq, pdo, pvv;
  X8 pt, ps;
  float pf0, pf1, pf2, prk;
  int t_off = 0;  // where this thread's piece of T goes (elements)
  {
    int row, pc;
    const int d = tid - 128;
    tri_piece(d < T_DIAG_PIECES ? max(d, 0) : min(d - T_DIAG_PIECES, T_DIAG_PIECES - 1), row, pc);
    t_off = tid < 128 ? (32 + (tid >> 2)) * GB_TS + 8 * (tid & 3)
                      : ((d < T_DIAG_PIECES ? 0 : 64) + row) * GB_TS + 8 * pc;
    if (tid >= 288) {  // the 96 pieces that lie entirely above the diagonals (written again for every chunk: M sits there)
      const int u = min(tid - 288, 95);
      tri_upper_piece(u % 48, row, pc);
      t_off = ((u < 48 ? 0 : 64) + row) * GB_TS + 8 * pc;
    }
  }
  auto issue = [&](int c) __attribute__((always_inline)) {
    c = uniform(c);
    const int tok0 = chunk_tok0[c], len = chunk_len[c];
    const int r = min(srow, len - 1);
    pk = *reinterpret_cast<const typename Raw8<T>::type*>(k + ((size_t)(tok0 + r) * H + h) * 64 + 8 * part);
    pq = *reinterpret_cast<const typename Raw8<T>::type*>(q + ((size_t)(tok0 + r) * H + h) * 64 + 8 * part);
    pdo = *reinterpret_cast<const typename Raw8<T>::type*>(dout + ((size_t)(tok0 + r) * HV + hv) * 64 + 8 * part);
    if constexpr (GRADS) {
      pvv = *reinterpret_cast<const typename Raw8<T>::type*>(v + ((size_t)(tok0 + r) * HV + hv) * 64 + 8 * part);
      ps = reinterpret_cast<const X8*>(states + ((size_t)c * HV + hv) * GDR_STATE_BYTES)[tid];
    }
    const unsigned char* rec = recs + ((size_t)c * HV + hv) * REC_BYTES;
    pt = reinterpret_cast<const X8*>(rec)[min(tid, 287)];
    const float* fact = reinterpret_cast<const float*>(rec + T_BYTES);
    if (wave >= 4) {  // (wave 7 stages them)
      pf0 = fact[lane];
      pf1 = fact[64 + lane];
      pf2 = fact[128 + lane];
    }
    prk = fact[128 + srow];
  };
  auto stage = [&](int len) __attribute__((always_inline)) {
    const bool live = srow < len;
    float fk[8], fq[8], ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      fk[e] = live ? (float)pk[e] : 0.0f;
      fq[e] = live ? (float)pq[e] : 0.0f;
      ss = __builtin_fmaf(fq[e], fq[e], ss);
    }
    const float cq = l2_factor(gb_sum8(ss), l2norm);
    X8 ok, oq, od;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      ok[e] = (OT)(fk[e] * prk);
      oq[e] = (OT)(fq[e] * cq);
      od[e] = live ? (OT)pdo[e] : (OT)0.0f;
    }
    *reinterpret_cast<X8*>(&b_k[srow * GB_LS + 8 * part]) = ok;
    *reinterpret_cast<X8*>(&b_q[srow * GB_LS + 8 * part]) = oq;
    *reinterpret_cast<X8*>(&b_do[srow * GB_LS + 8 * part]) = od;
    if (part == 0) s_rq[srow] = cq;
    if constexpr (GRADS) {
      X8 ov;
#pragma unroll
      for (int e = 0; e < 8; ++e) ov[e] = live ? (OT)pvv[e] : (OT)0.0f;
      *reinterpret_cast<X8*>(reinterpret_cast<OT*>(b_v) + (part >> 2) * 2048 + srow * 32 + 8 * (part & 3)) = ov;
      *reinterpret_cast<X8*>(b_s + 16 * tid) = ps;
    }
    if (tid < 384) {
      X4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = tid < 288 ? pt[e] : (OT)0.0f;
        hi[e] = tid < 288 ? pt[4 + e] : (OT)0.0f;
      }
      *reinterpret_cast<X4*>(&b_t[t_off]) = lo;
      *reinterpret_cast<X4*>(&b_t[t_off + 4]) = hi;
    }
    if (wave == 7) {
      const float gl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pf0), 63));
      s_gam[lane] = pf0;
      s_beta[lane] = pf1;
      s_rk[lane] = pf2;
      s_eg[lane] = __builtin_amdgcn_exp2f(pf0);
      s_dk[lane] = __builtin_amdgcn_exp2f(gl - pf0);
    }
  };

  f32x16 G[2];  // (waves 0, 1) the gradient of the state behind the chunk, value columns 32 wave + ln
  G[0] = zero16();
  G[1] = zero16();
  if (nc > 0) issue(c0 + nc - 1);
  if constexpr (GRADS) {
    // The gradient behind the sequence pushed through the composites of the later segments: whole groups of
    // GDR_SCAN_GROUP first (gmax > 0), then the segments between them and this one; G <- d G + N' + M'^T G. Waves 0 .. 3:
    // wave w owns rows 32 (w / 2) .. of column slab w % 2 and takes the other rows as operand through LDS, so that the
    // composites of two steps fit the registers (one wave with all rows of a slab would need 128 for them).
    const int seg0 = pv.seq_seg0[seq], last = seg0 + pv.seq_nseg[seq] - 1, behind = last - seg;
    const int lead = gmax > 0 ? behind / GDR_SCAN_GROUP : 0, nst = lead + behind - lead * GDR_SCAN_GROUP;
    const int slab = wave & 1, km = (wave >> 1) & 1;
    f32x16 S = zero16();
    if (dht && wave < 4) {
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
      unsigned char* xbuf = b_s + (p & 1) * 8192 + slab * 4096;
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
      if (wave < 4) {
        walk_issue(0, rm[0], rn[0], rd[0]);
        walk_issue(1, rm[1], rn[1], rd[1]);
        for (int p = 0; p < nst; p += 2) {
          walk_step(p, rm[0], rn[0], rd[0]);
          walk_issue(p + 2, rm[0], rn[0], rd[0]);
          if (p + 1 < nst) walk_step(p + 1, rm[1], rn[1], rd[1]);
          walk_issue(p + 3, rm[1], rn[1], rd[1]);
        }
      } else {
        for (int p = 0; p < nst; ++p) lds_barrier();
      }
    }
    lds_barrier();  // (the last step's operands have been read)
    float* xs = reinterpret_cast<float*>(b_s);  // rows 32 .. 63 go from waves 2, 3 to waves 0, 1
    if (wave == 2 || wave == 3) {
#pragma unroll
      for (int r = 0; r < 16; ++r) xs[(slab * 16 + r) * 64 + lane] = S[r];
    }
    lds_barrier();
    if (wave < 2) {
      G[0] = S;
#pragma unroll
      for (int r = 0; r < 16; ++r) G[1][r] = xs[(slab * 16 + r) * 64 + lane];
    }
    lds_barrier();
  }

  // operand pieces of the row-major tiles
  auto rows_k = [&](const OT* buf, int row, int c) __attribute__((always_inline)) {  // accumulator slot order
    return op_ld_kappa<OT>(buf, GB_LS, row, c, hh);
  };
  auto cols = [&](const OT* buf, int col0, int row0) __attribute__((always_inline)) {
    return op_ld_kappa_tr<OT, false>(buf, GB_LS, col0, row0, lane);
  };

  // steps k0 .. k1 - 1 (of 16) of a product: every operand fragment is requested before the first MFMA (left alone the
  // compiler requests them one by one and pays the LDS latency for each)
  auto mm = [&](f32x16 acc, int k0, int k1, auto fa, auto fb) __attribute__((always_inline)) {
    X8 a[4], b[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      if (ks >= k0 && ks < k1) { a[ks] = fa(ks); b[ks] = fb(ks); }
    // (an MFMA is no memory access: only passing its operands through an asm behind all the reads keeps it there)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      if (ks >= k0 && ks < k1) asm volatile("" : "+v"(a[ks]), "+v"(b[ks]));
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      if (ks >= k0 && ks < k1) acc = mfma32(a[ks], b[ks], acc);
    return acc;
  };
  auto rows_n = [&](const OT* buf, int row, int c) __attribute__((always_inline)) {  // consecutive columns
    return *reinterpret_cast<const X8*>(&buf[row * GB_LS + c + 8 * hh]);
  };

  // ---- what waves do alike at the end of a chunk: the rows of dq (waves 0-3) and dk (4-7) through the normalisation from
  //      this wave's tile acc (rows 32 kt, tokens 32 tt), the rows of d v, and the stores
  typename Raw8<T>::type vre;  // this lane's piece of v for d beta
  auto load_v = [&](int tok0, int len) __attribute__((always_inline)) {
    vre = *reinterpret_cast<const typename Raw8<T>::type*>(v + ((size_t)(tok0 + min(xtok, len - 1)) * HV + hv) * 64 +
                                                           8 * xpart);
  };
  auto finish = [&](f32x16& acc, float rs_g, int tok0, int len) __attribute__((always_inline)) {
    const OT* yin = wave < 4 ? b_q : b_k;
    float dot = 0.0f;
    X4 y4[4];
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      y4[b4] = *reinterpret_cast<const X4*>(&yin[tok * GB_LS + 32 * kt + 8 * b4 + 4 * hh]);
#pragma unroll
      for (int e = 0; e < 4; ++e) dot += (float)y4[b4][e] * acc[4 * b4 + e];
    }
    float* const s_dot = s_sum + (wave < 4 ? GbSums::DOTQ : GbSums::DOTK);
    dot = gb_both_halves(dot);
    rs_g = gb_both_halves(rs_g);
    if (hh == 0) {
      s_dot[64 * kt + tok] = dot;
      s_sum[GbSums::DGAM + 32 * wave + ln] = rs_g;
    }
    {  // d v = beta X and the product of X with v, 16 tokens x 4 pieces per wave
      const int L = lane & 15, r0 = 16 * (wave & 3) + 4 * (L & 3), cc = 8 * xpart + (L >> 2);
      const OT* p = reinterpret_cast<const OT*>(b_x + ((cc >> 5) * 4 + (r0 >> 4)) * 1024 +
                                                (32 * ((r0 >> 2) & 1) + (cc & 31)) * 16 + ((r0 >> 3) & 1) * 8);
      const X4 lo = op_lds_read_tr4<OT>(p), hi = op_lds_read_tr4<OT>(p + 4 * 8);
      const float b = s_beta[xtok];
      float t = 0.0f;
      typename Raw8<T>::type out;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        t += (float)lo[e] * (float)vre[e] + (float)hi[e] * (float)vre[4 + e];
        out[e] = (T)(b * (float)lo[e]);
        out[4 + e] = (T)(b * (float)hi[e]);
      }
      t += __shfl_xor(t, 16);
      t = gb_both_halves(t);
      if (lane < 16) s_sum[GbSums::XV + 64 * (wave >> 2) + xtok] = t;
      if (xtok < len) {
        *reinterpret_cast<typename Raw8<T>::type*>(dv + ((size_t)(tok0 + xtok) * HV + hv) * 64 + 8 * xpart) = out;
      }
    }
    lds_barrier();  // (4) the row sums are complete, every tile has been read
    {
      dot = s_dot[tok] + s_dot[64 + tok];
      const float cn = wave < 4 ? s_rq[tok] : s_rk[tok];
      // c = 1 / (|x| + eps) in the recurrent form: |x| = 1 / c - eps
      const float fy = l2norm == GDR_L2_CHUNK ? cn * dot
                       : l2norm == GDR_L2_RECURRENT ? dot / fmaxf(1.0f / cn - 1e-6f, 1e-30f) : 0.0f;
      OT* to = (wave < 4 ? b_q : b_k) + tok * GB_LS + 32 * kt;
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        X4 o4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gx = l2norm == GDR_L2_NONE ? acc[4 * b4 + e] : cn * acc[4 * b4 + e] - fy * (float)y4[b4][e];
          o4[e] = (OT)gx;
        }
        *reinterpret_cast<X4*>(&to[8 * b4 + 4 * hh]) = o4;
      }
    }
    lds_barrier();  // (5) the rows of dq and dk are complete
    const X8 o_k = *reinterpret_cast<const X8*>(&b_k[srow * GB_LS + 8 * part]);
    const X8 o_q = *reinterpret_cast<const X8*>(&b_q[srow * GB_LS + 8 * part]);
    if (srow < len) {
      const size_t at = ((size_t)(tok0 + srow) * HV + hv) * 64 + 8 * part;
      *reinterpret_cast<X8*>(dk + at) = o_k;
      *reinterpret_cast<X8*>(dq + at) = o_q;
    }
    if (wave == 2) {  // d g = the sum of d gamma over the later rows of the chunk (gamma_i = g_0 + ... + g_i); d beta
      const float* w = s_sum + GbSums::DGAM + 32 * hh + ln;  // (lane = token: its waves are hh, hh + 2, hh + 4, hh + 6)
      const float* t = s_sum + ln;                            // tiles (0,0), (0,1), (1,1)
      float x = (w[0] + w[64]) + (w[128] + w[192]);
      x += t[GbSums::TILE_G + 32 * hh] + (hh ? t[GbSums::TILE_G + 64] : 0.0f);
      x -= t[GbSums::TILE_C + 64 * hh] + (hh ? 0.0f : t[GbSums::TILE_C + 32]);
      const float db = (t[GbSums::TILE_B + 32 * hh] + (hh ? t[GbSums::TILE_B + 64] : 0.0f)) +
                       (t[GbSums::DBETA + 32 * hh] + t[GbSums::DBETA + 64 + 32 * hh]) +
                       (s_sum[GbSums::XV + lane] + s_sum[GbSums::XV + 64 + lane]);
      if (lane == len - 1) {
        const f32x4 ga = *reinterpret_cast<const f32x4*>(s_sum + GbSums::GL), gb = *reinterpret_cast<const f32x4*>(s_sum + GbSums::GL + 4);
        x += ((ga[0] + ga[1]) + (ga[2] + ga[3])) + ((gb[0] + gb[1]) + (gb[2] + gb[3]));
      }
      if (lane >= len) x = 0.0f;
      const float incl = wave_inclusive_scan(x);  // (inclusive scan from the last lane down: total - exclusive prefix)
      const float total = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(incl), 63));
      if (lane < len) {
        dg[(size_t)(tok0 + lane) * HV + hv] = total - incl + x;
        dbeta[(size_t)(tok0 + lane) * HV + hv] = db;
      }
    }
    lds_barrier();  // (6) every tile has been read: the next chunk's may be staged
  };
  // scale e^gamma S dO^T of this wave's tile, and its share of d gamma
  auto dq_state = [&](f32x16& acc, float& rs_g) __attribute__((always_inline)) {
    acc = mm(zero16(), 0, 4, [&](int ks) { return fr_tr<OT, false>(b_s, 32 * kt, 16 * ks, lane); },
             [&](int ks) { return rows_n(b_do, tok, 16 * ks); });
    const float fs = scale * s_eg[tok];
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const X4 y = *reinterpret_cast<const X4*>(&b_q[tok * GB_LS + 32 * kt + 8 * b4 + 4 * hh]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[4 * b4 + e] *= fs;
        rs_g += (float)y[e] * acc[4 * b4 + e];
      }
    }
  };
  // + Kh^T N^T
  auto dq_chunk = [&](f32x16& acc) __attribute__((always_inline)) {
    acc = mm(acc, 0, 2 * (tt + 1), [&](int ks) { return cols(b_k, 32 * kt, 16 * ks); },
             [&](int ks) { return op_frag_load<OT>(b_n + (tt + ks / 2) * GB_TRI, ks & 1, lane); });
  };

  // (every role has a chunk loop of its own, so that what one role carries from chunk to chunk takes no registers in the
  // others; the barriers pair up by their number)
  const int cl = c0 + nc - 1;
  if (wave < 2) {
    // ======================================= the gradient of the state =======================================
    for (int c = cl; c >= c0; --c) {
      const int tok0 = chunk_tok0[uniform(c)], len = chunk_len[uniform(c)];
      lanes();
      stage(len);
      if constexpr (GRADS) load_v(tok0, len);
      else issue(max(c - 1, c0));
      lds_barrier();  // (0) the tiles of chunk c are complete
      f32x16 a[2];  // D Kh G', then dVn, then X
      {
        X8 Gb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          Gb[ks] = acc_to_op<OT>(G[ks / 2], 8 * (ks % 2));
          if constexpr (GRADS) op_frag_store<OT>(b_g, wave * 4 + ks, lane, Gb[ks]);
        }
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) {
          a[tm] = mm(zero16(), 0, 4, [&](int ks) { return rows_k(b_k, 32 * tm + ln, 16 * ks); },
                     [&](int ks) { return Gb[ks]; });
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {
            const f32x4 f = gb_rows4(s_dk, 32 * tm, b4, hh);
#pragma unroll
            for (int e = 0; e < 4; ++e) a[tm][4 * b4 + e] *= f[e];
          }
        }
      }
      lds_barrier();  // (1) P, Vn and G' are complete
      {
        X8 dOb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) dOb[ks] = cols(b_do, 32 * wave, 16 * ks);
#pragma unroll
        for (int tm = 0; tm < 2; ++tm)  // + P^T dO
          a[tm] = mm(a[tm], 2 * tm, 4,
                     [&](int ks) { return fr_tr<OT, true>(b_p + (tm == 0 ? ks / 2 : 2) * GB_TRI, 0, 16 * (ks & 1), lane); },
                     [&](int ks) { return dOb[ks]; });
      }
      X8 Xb[4];
      {
        X8 Rb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) Rb[ks] = acc_to_op<OT>(a[ks / 2], 8 * (ks % 2));
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) {  // X = T^T dVn (blocks T11, T21 | T22)
          a[tm] = mm(zero16(), 2 * tm, 4,
                     [&](int ks) {
                       return op_ld_kappa_tr<OT, false>(b_t + (tm == 0 ? ks / 2 : 2) * 32 * GB_TS, GB_TS, 0, 16 * (ks & 1), lane);
                     },
                     [&](int ks) { return Rb[ks]; });
          if constexpr (GRADS) {
            op_frag_store<OT>(b_x, wave * 4 + 2 * tm + 0, lane, acc_to_op<OT>(a[tm], 0));
            op_frag_store<OT>(b_x, wave * 4 + 2 * tm + 1, lane, acc_to_op<OT>(a[tm], 8));
          }
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {  // -beta e^gamma X, the operand of the update
            const f32x4 fb = gb_rows4(s_beta, 32 * tm, b4, hh), fe = gb_rows4(s_eg, 32 * tm, b4, hh);
#pragma unroll
            for (int e = 0; e < 4; ++e) a[tm][4 * b4 + e] *= -fb[e] * fe[e];
          }
          Xb[2 * tm + 0] = acc_to_op<OT>(a[tm], 0);
          Xb[2 * tm + 1] = acc_to_op<OT>(a[tm], 8);
        }
      }
      if constexpr (GRADS) lds_barrier();  // (2) X and N are complete, T and P are dead
      {
        const float dec = __builtin_amdgcn_exp2f(s_gam[63]);
#pragma unroll
        for (int km = 0; km < 2; ++km)
#pragma unroll
          for (int r = 0; r < 16; ++r) G[km][r] *= dec;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {  // + (scale e^gamma Qh)^T dO - (beta e^gamma Kh)^T X
          X8 d = cols(b_do, 32 * wave, 16 * ks);
          const f32x4 f0 = *reinterpret_cast<const f32x4*>(&s_eg[16 * ks + 4 * hh]);
          const f32x4 f1 = *reinterpret_cast<const f32x4*>(&s_eg[16 * ks + 8 + 4 * hh]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            d[e] = (OT)((float)d[e] * (scale * f0[e]));
            d[4 + e] = (OT)((float)d[4 + e] * (scale * f1[e]));
          }
          X8 q0 = cols(b_q, 0, 16 * ks), q1 = cols(b_q, 32, 16 * ks), k0 = cols(b_k, 0, 16 * ks), k1 = cols(b_k, 32, 16 * ks);
          asm volatile("" : "+v"(q0), "+v"(q1), "+v"(k0), "+v"(k1));
          G[0] = mfma32(q0, d, G[0]);
          G[1] = mfma32(q1, d, G[1]);
          G[0] = mfma32(k0, Xb[ks], G[0]);
          G[1] = mfma32(k1, Xb[ks], G[1]);
        }
      }
      if constexpr (GRADS) {
        issue(max(c - 1, c0));
        f32x16 acc;
        float rs_g = 0.0f;
        dq_state(acc, rs_g);
        dq_chunk(acc);
        lds_barrier();  // (3)
        finish(acc, rs_g, tok0, len);
      } else {
        lds_barrier();  // every tile has been read: the next chunk's may be staged
      }
    }
    if constexpr (!GRADS) {  // N' in accumulator order, as the forward composites keep N
      f32x4* out = reinterpret_cast<f32x4*>(Nr + (((size_t)seg * HV + hv) * 2 + wave) * GDR_STATE_BYTES);
#pragma unroll
      for (int km = 0; km < 2; ++km)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          f32x4 t;
#pragma unroll
          for (int e = 0; e < 4; ++e) t[e] = G[km][4 * q4 + e];
          out[(km * 4 + q4) * 64 + lane] = t;
        }
    } else if (dh0 && (flags & SEG_FIRST)) {
#pragma unroll
      for (int km = 0; km < 2; ++km)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          dh0[(((size_t)seq * HV + hv) * 64 + 32 * km + acc_row(r, hh)) * 64 + 32 * wave + ln] = G[km][r];
    }
  } else if (GRADS && wave < 4) {
    // =============================================== Vn, dQh ===============================================
    const int vn = wave - 2;
    for (int c = cl; c >= c0; --c) {
      const int tok0 = chunk_tok0[uniform(c)], len = chunk_len[uniform(c)];
      lanes();
      stage(len);
      load_v(tok0, len);
      lds_barrier();  // (0)
      issue(max(c - 1, c0));
      X8 Rb[4];
      {
        X8 Sb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) Sb[ks] = op_frag_load<OT>(b_s, vn * 4 + ks, lane);
        const OT* vt = reinterpret_cast<const OT*>(b_v) + vn * 2048;
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) {
          f32x16 r = mm(zero16(), 0, 4, [&](int ks) { return rows_k(b_k, 32 * tm + ln, 16 * ks); },
                        [&](int ks) { return Sb[ks]; });
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {  // R = beta (v - e^gamma Kh S)
            const X4 vv = op_ld_col4<OT>(vt, 32, 0, 32 * tm + 8 * b4, lane);
            const f32x4 fb = gb_rows4(s_beta, 32 * tm, b4, hh), fe = gb_rows4(s_eg, 32 * tm, b4, hh);
#pragma unroll
            for (int e = 0; e < 4; ++e) r[4 * b4 + e] = fb[e] * ((float)vv[e] - fe[e] * r[4 * b4 + e]);
          }
          Rb[2 * tm + 0] = acc_to_op<OT>(r, 0);
          Rb[2 * tm + 1] = acc_to_op<OT>(r, 8);
        }
      }
      lds_fence();  // this wave's reads of its half of v are done: Vn goes over it
#pragma unroll
      for (int tm = 0; tm < 2; ++tm) {
        const f32x16 r = mm(zero16(), 0, 2 * (tm + 1),
                            [&](int ks) {
                              return op_ld_kappa<OT>(b_t + (tm == 0 ? 0 : 1 + ks / 2) * 32 * GB_TS, GB_TS, ln, 16 * (ks & 1), hh);
                            },
                            [&](int ks) { return Rb[ks]; });
        op_frag_store<OT>(b_v, vn * 4 + 2 * tm + 0, lane, acc_to_op<OT>(r, 0));
        op_frag_store<OT>(b_v, vn * 4 + 2 * tm + 1, lane, acc_to_op<OT>(r, 8));
      }
      lds_barrier();  // (1)
      f32x16 acc;
      float rs_g = 0.0f;
      dq_state(acc, rs_g);
      lds_barrier();  // (2)
      dq_chunk(acc);
      lds_barrier();  // (3)
      finish(acc, rs_g, tok0, len);
    }
  } else if (!GRADS && wave < 4) {
    for (int c = cl; c >= c0; --c) {
      lanes();
      stage(chunk_len[uniform(c)]);
      issue(max(c - 1, c0));
      lds_barrier();  // (0)
      lds_barrier();  // (1)
      lds_barrier();
    }
  } else {
    // ================================ the token x token tiles, dKh (waves 4-7) ================================
    const int tw = wave - 4, jt = tw == 2 ? 1 : 0, it = tw == 0 ? 0 : 1;
    for (int c = cl; c >= c0; --c) {
      const int tok0 = chunk_tok0[uniform(c)], len = chunk_len[uniform(c)];
      lanes();
      stage(len);
      if constexpr (GRADS) load_v(tok0, len);
      else issue(max(c - 1, c0));
      lds_barrier();  // (0)
      const int i = 32 * it + ln;
      // P of this wave's tile (rows j, column i): the product here and once more for grad P (16 registers less to carry)
      auto p_tile = [&]() __attribute__((always_inline)) {
        return mm(zero16(), 0, 4, [&](int ks) { return rows_n(b_k, 32 * jt + ln, 16 * ks); },
                  [&](int ks) { return rows_n(b_q, i, 16 * ks); });
      };
      // e^{gamma_i - gamma_j} for i >= j (strict: i > j), else 0, of accumulator registers 4 b4 .. + 3
      auto ratio = [&](int b4, float gi, int e_min, float* out) __attribute__((always_inline)) {
        const f32x4 gj = gb_rows4(s_gam, 32 * jt, b4, hh);
        const int lx = ln - 4 * hh - e_min + (jt != it ? 64 : 0);  // (the tile below the diagonal is full)
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = __builtin_amdgcn_exp2f(lx >= 8 * b4 + e ? gi - gj[e] : -1e30f);
      };
      if (wave < 7) {
        f32x16 pm = p_tile();
        const float gi = s_gam[i];
#pragma unroll
        for (int b4 = 0; b4 < 4; ++b4) {
          float gm[4];
          ratio(b4, gi, 0, gm);
#pragma unroll
          for (int e = 0; e < 4; ++e) pm[4 * b4 + e] *= scale * gm[e];
        }
        op_frag_store<OT>(b_p + tw * GB_TRI, 0, lane, acc_to_op<OT>(pm, 0));
        op_frag_store<OT>(b_p + tw * GB_TRI, 1, lane, acc_to_op<OT>(pm, 8));
      }
      lds_barrier();  // (1)
      if constexpr (GRADS) {
        f32x16 acc;
        float rs_g = 0.0f, rs_b = 0.0f;  // sums over the rows of the terms of d gamma / d beta: of token i, later of tok
        float rs_c = 0.0f, tg = 0.0f;    // sum over the columns for the tile's row gb_half_sums16 leaves here; of tok
        float gl = 0.0f;
        if (wave < 7) {  // grad P = dO Vn^T
          f32x16 n = mm(zero16(), 0, 4, [&](int ks) { return fr_tr<OT, false>(b_v, 32 * jt, 16 * ks, lane); },
                        [&](int ks) { return rows_n(b_do, i, 16 * ks); });
          const f32x16 pm = p_tile();
          const float gi = s_gam[i];
          float cs[16];  // the terms of d gamma, for their sums over the columns
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {
            float gm[4];
            ratio(b4, gi, 0, gm);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int r = 4 * b4 + e;
              n[r] *= scale * gm[e];
              cs[r] = n[r] * pm[r];
              rs_g += cs[r];
            }
          }
          op_frag_store<OT>(b_n + tw * GB_TRI, 0, lane, acc_to_op<OT>(n, 0));
          op_frag_store<OT>(b_n + tw * GB_TRI, 1, lane, acc_to_op<OT>(n, 8));
          rs_c = gb_half_sums16(cs, lane);
        } else {  // e^{gamma_L} <G', S>
          float x = 0.0f;
#pragma unroll
          for (int f = 0; f < 8; ++f) {
            const X8 xa = op_frag_load<OT>(b_g, f, lane), xb = op_frag_load<OT>(b_s, f, lane);
#pragma unroll
            for (int e = 0; e < 8; ++e) x = __builtin_fmaf((float)xa[e], (float)xb[e], x);
          }
          gl = x * __builtin_amdgcn_exp2f(s_gam[63]);
        }
        // dKh^T: D G' Vn^T first
        acc = mm(zero16(), 0, 4, [&](int ks) { return fr_tr<OT, false>(b_g, 32 * kt, 16 * ks, lane); },
                 [&](int ks) { return fr_tr<OT, false>(b_v, 32 * tt, 16 * ks, lane); });
        {
          const float fd = s_dk[tok];
          float t = 0.0f;
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {
            const X4 y = *reinterpret_cast<const X4*>(&b_k[tok * GB_LS + 32 * kt + 8 * b4 + 4 * hh]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              acc[4 * b4 + e] *= fd;
              t += (float)y[e] * acc[4 * b4 + e];
            }
          }
          gl += t;
          tg = -t;
        }
        lds_barrier();  // (2)
        if (wave < 7) {  // grad A = -X Vn^T
          f32x16 da = mm(zero16(), 0, 4, [&](int ks) { return fr_tr<OT, false>(b_v, 32 * jt, 16 * ks, lane); },
                         [&](int ks) { return fr_tr<OT, false>(b_x, 32 * it, 16 * ks, lane); });
          const f32x16 kk = mm(zero16(), 0, 4, [&](int ks) { return rows_n(b_k, 32 * jt + ln, 16 * ks); },
                               [&](int ks) { return rows_n(b_k, i, 16 * ks); });
          const float bi = s_beta[i], gi = s_gam[i];
          float cs[16];
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {
            float gm[4];
            ratio(b4, gi, 1, gm);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int r = 4 * b4 + e;
              // grad A_ij Gamma_ij, and grad A_ij times A_ij / beta_i and times A_ij
              const float ga = -da[r] * gm[e], b = ga * kk[r], a = b * bi;
              rs_b += b;
              rs_g += a;
              cs[r] = a;
              da[r] = ga * bi;
            }
          }
          op_frag_store<OT>(b_m + tw * GB_TRI, 0, lane, acc_to_op<OT>(da, 0));
          op_frag_store<OT>(b_m + tw * GB_TRI, 1, lane, acc_to_op<OT>(da, 8));
          rs_c += gb_half_sums16(cs, lane);
          rs_g = gb_both_halves(rs_g);
          rs_b = gb_both_halves(rs_b);
          if (hh == 0) {
            s_sum[GbSums::TILE_G + 32 * tw + ln] = rs_g;
            s_sum[GbSums::TILE_B + 32 * tw + ln] = rs_b;
          }
          if (!(ln & 1)) s_sum[GbSums::TILE_C + 32 * tw + 8 * (ln >> 3) + 4 * hh + ((ln >> 1) & 3)] = rs_c;
          rs_b = 0.0f;
        }
        issue(max(c - 1, c0));
        {  // -(S X^T), the gradient of beta e^gamma Kh
          const f32x16 xw = mm(zero16(), 0, 4, [&](int ks) { return fr_tr<OT, false>(b_s, 32 * kt, 16 * ks, lane); },
                               [&](int ks) { return fr_tr<OT, false>(b_x, 32 * tt, 16 * ks, lane); });
          const float fe = -s_eg[tok], fb = s_beta[tok];
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {
            const X4 y = *reinterpret_cast<const X4*>(&b_k[tok * GB_LS + 32 * kt + 8 * b4 + 4 * hh]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float t = fe * xw[4 * b4 + e];
              rs_b += (float)y[e] * t;
              acc[4 * b4 + e] = __builtin_fmaf(fb, t, acc[4 * b4 + e]);
            }
          }
          rs_g = __builtin_fmaf(fb, rs_b, tg);
          rs_b = gb_both_halves(rs_b);
          if (hh == 0) s_sum[GbSums::DBETA + 32 * tw + ln] = rs_b;
        }
        // + (N^T Qh)^T
        acc = mm(acc, 2 * tt, 4, [&](int ks) { return cols(b_q, 32 * kt, 16 * ks); },
                 [&](int ks) { return fr_tr<OT, true>(b_n + (tt == 0 ? ks / 2 : 2) * GB_TRI, 0, 16 * (ks & 1), lane); });
        {
          const float t = gb_half_sum(gl);
          if (ln == 0) s_sum[GbSums::GL + 2 * tw + hh] = t;
        }
        lds_barrier();  // (3) M is complete
        // + (M Kh)^T + (M^T Kh)^T
        acc = mm(acc, 0, 2 * (tt + 1), [&](int ks) { return cols(b_k, 32 * kt, 16 * ks); },
                 [&](int ks) { return op_frag_load<OT>(b_m + (tt + ks / 2) * GB_TRI, ks & 1, lane); });
        acc = mm(acc, 2 * tt, 4, [&](int ks) { return cols(b_k, 32 * kt, 16 * ks); },
                 [&](int ks) { return fr_tr<OT, true>(b_m + (tt == 0 ? ks / 2 : 2) * GB_TRI, 0, 16 * (ks & 1), lane); });
        finish(acc, rs_g, tok0, len);
      } else {
        lds_barrier();
      }
    }
  }

}

// ---- host ----------------------------------------------------------------------------------------------------------
struct GbWorkspace {
  int64_t nr, gm, gn, gd, max_groups, bytes;
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
  w.bytes = off;
  return w;
}

template <typename T>
static int gb_run(const void* q, const void* k, const void* v, const void* dout, const float* dht, void* dq, void* dk,
                  void* dv, float* dg, float* dbeta, float* dh0, const int32_t* ph, const int32_t* pd,
                  const unsigned char* saved, int H, int HV, float scale, int l2norm, unsigned char* ws, hipStream_t s) {
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
      if (hipFuncSetAttribute((const void*)gdrb_segment_kernel<T, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              GbSmem<false>::BYTES) != hipSuccess ||
          hipFuncSetAttribute((const void*)gdrb_segment_kernel<T, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              GbSmem<true>::BYTES) != hipSuccess)
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
  LAMPA_PROF(s, "start");
  if (segs > n_seq) {
    hipLaunchKernelGGL((gdrb_segment_kernel<T, false>), dim3(segs * HV), dim3(GB_THREADS), GbSmem<false>::BYTES, s,
                       (const T*)q, (const T*)k, (const T*)v, (const T*)dout, recs, states, pv, pv.chunk_tok0, pv.chunk_len,
                       Mt, Dc, Nr, Gm, Gn, Gd, 0, dht, (T*)dq, (T*)dk, (T*)dv, dg, dbeta, dh0, H, HV, scale, l2norm);
    LAMPA_PROF(s, "gdrb_segment_kernel<source>");
    if (gmax > 0) {
      hipLaunchKernelGGL((gdr_scan2_kernel<T, 64, 64, 4, SCAN_GROUP, true>), dim3(4 * gmax, n_seq, HV), dim3(128), 0, s, pv, Mt,
                         Nr, Dc, (const float*)nullptr, (float*)nullptr, Gm, Gn, Gd, HV, 0, gmax);
      LAMPA_PROF(s, "gdr_scan2_kernel<group, reversed>");
    }
  }
  hipLaunchKernelGGL((gdrb_segment_kernel<T, true>), dim3(segs * HV), dim3(GB_THREADS), GbSmem<true>::BYTES, s, (const T*)q,
                     (const T*)k, (const T*)v, (const T*)dout, recs, states, pv, pv.chunk_tok0, pv.chunk_len, Mt, Dc, Nr, Gm,
                     Gn, Gd, gmax, dht, (T*)dq, (T*)dk, (T*)dv, dg, dbeta, dh0, H, HV, scale, l2norm);
  LAMPA_PROF(s, "gdrb_segment_kernel<gradients>");
  return lampa_launch_status();
}

static bool gb_plan_ok(const int32_t* ph) {
  return ph && ph[PLAN_N_SEQ] >= 1 && ph[PLAN_N_SEGMENTS] >= ph[PLAN_N_SEQ] && ph[PLAN_TOTAL_CHUNKS] >= 0;
}

extern "C" int64_t lampa_gdr_bwd_saved_workspace_bytes(const int32_t* plan_host, int HV) {
  if (!gb_plan_ok(plan_host) || HV < 1) return LAMPA_ERR_INVALID;
  return gb_workspace(plan_host[PLAN_N_SEGMENTS], HV).bytes;
}

// Gradients from what lampa_gdr_chunk_fwd_train kept. q, k [tokens, H, 64]; v, dout, dv and dq, dk (one row per VALUE head)
// [tokens, HV, 64]; dg, dbeta fp32 [tokens, HV]; dht, dh0 fp32 [n_seq, HV, 64, 64] (nullable).
extern "C" int lampa_gdr_bwd_saved(const void* q, const void* k, const void* v, const void* saved, const void* dout,
                                   const float* dht, void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
                                   const int32_t* plan_host, const int32_t* plan_dev, int H, int HV, int K, int V, int dtype,
                                   float scale, int l2norm, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!q || !k || !v || !saved || !dout || !dq || !dk || !dv || !dg || !dbeta || !plan_host || !plan_dev)
    return LAMPA_ERR_INVALID;
  if (H < 1 || HV < H || HV % H != 0 || l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (K != 64 || V != 64 || (dtype != GDR_BF16 && dtype != GDR_FP16)) return LAMPA_ERR_UNSUPPORTED;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 15)
    return LAMPA_ERR_INVALID;
  if (!gb_plan_ok(plan_host)) return LAMPA_ERR_INVALID;
  if (!workspace || workspace_bytes < lampa_gdr_bwd_saved_workspace_bytes(plan_host, HV)) return LAMPA_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  unsigned char* ws = (unsigned char*)workspace;
  const unsigned char* sv = (const unsigned char*)saved;
  if (dtype == GDR_BF16)
    return gb_run<__bf16>(q, k, v, dout, dht, dq, dk, dv, dg, dbeta, dh0, plan_host, plan_dev, sv, H, HV, scale, l2norm, ws, s);
  return gb_run<_Float16>(q, k, v, dout, dht, dq, dk, dv, dg, dbeta, dh0, plan_host, plan_dev, sv, H, HV, scale, l2norm, ws, s);
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
