// One token of the hierarchical (level-weighted) gated delta rule on explicit level states.
//
// Replaces hattention_step (reference chengjiang123/Lampa, models/hattention/kernel.py:577-633) with
// step_state / step_output (recurrent.py:134-166) and HState.cascade_weak / insert (recurrent.py:44-97):
//   cascade   the full levels 0 .. z-1 are added into level z and emptied (lowest first);
//   gate      S_l <- a (S_l - b k (k^T S_l)) for every level, a = e^g;
//   insert    S_0 <- b k v^T;
//   output    o = q^T sum_l lambda_l S_l      (q l2-normalised and scaled, k l2-normalised, kernel.py:613-616).
// The level states are the reference's HState.states: fp32 [B, HV, K, V, L] with the level index fastest. Which levels
// are full depends only on the number of tokens seen, so the caller passes z (0 = nothing to merge).
// Workgroup per (sequence, value head, 16 value columns), 256 threads = 16 row groups x 16 columns: every thread walks
// the rows i = group, group + 16, ... of its column twice (k^T S_l first, summed over the groups through LDS, then the
// update); a row's L level values are contiguous, 16 columns of a row are one contiguous piece.
#include "gdr_common.h"

#define HGS_LMAX 32

#define HGS_COLS 16
#define HGS_GROUPS 16
#define HGS_LOADS 6  // 16-byte loads a thread of the LDS-staged form keeps in flight
#define HGS_ROWS 4   // rows of a thread's position whose LDS reads are in flight together
#define HGS_LDS_LIMIT (144 * 1024)  // dynamic LDS of the LDS-staged form at most (a CU has 160 KB)

template <typename T, int LM>
__global__ void __launch_bounds__(256)
    hgdn_step_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                     const float* __restrict__ g, const float* __restrict__ beta, const void* __restrict__ lam,
                     int lam_dtype, float lam_div, float* __restrict__ states, T* __restrict__ o, int H, int HV, int K,
                     int V, int L, int z, float scale, int l2norm) {
  extern __shared__ float s_qk[];  // q [K], k [K], lambda [HGS_LMAX], norm scratch [8], partial sums
  float* s_q = s_qk;
  float* s_k = s_qk + K;
  float* s_l = s_qk + 2 * K;
  float* s_red = s_l + HGS_LMAX;
  float* s_part = s_red + 8;  // [HGS_GROUPS][HGS_COLS][HGS_LMAX + 1]
  float* s_tot = s_part + HGS_GROUPS * HGS_COLS * (HGS_LMAX + 1);  // [HGS_COLS][HGS_LMAX + 1]
  float* s_m = s_tot + HGS_COLS * (HGS_LMAX + 1);                  // cascade coefficients, 3 x [HGS_LMAX]
  const int b = blockIdx.x / HV, hv = blockIdx.x % HV, h = hv / (HV / H);
  const int tid = threadIdx.x;
  const T* qp = q + ((size_t)b * H + h) * K;
  const T* kp = k + ((size_t)b * H + h) * K;
  float qs = 0.0f, ks = 0.0f;
  for (int i = tid; i < K; i += blockDim.x) {
    const float qi = GdrElem<T>::to_float(qp[i]), ki = GdrElem<T>::to_float(kp[i]);
    s_q[i] = qi;
    s_k[i] = ki;
    qs = __builtin_fmaf(qi, qi, qs);
    ks = __builtin_fmaf(ki, ki, ks);
  }
  for (int off = 32; off > 0; off >>= 1) {
    qs += __shfl_xor(qs, off);
    ks += __shfl_xor(ks, off);
  }
  if ((tid & 63) == 0) {
    s_red[2 * (tid >> 6)] = qs;
    s_red[2 * (tid >> 6) + 1] = ks;
  }
  if (tid < HGS_LMAX) {
    float x = 0.0f;  // levels past L weigh nothing
    if (tid < L) {
      const size_t li = ((size_t)b * HV + hv) * L + tid;
      x = lam_dtype == GDR_FP32   ? reinterpret_cast<const float*>(lam)[li]
          : lam_dtype == GDR_BF16 ? (float)reinterpret_cast<const __bf16*>(lam)[li]
                                  : (float)reinterpret_cast<const _Float16*>(lam)[li];
      if (lam_div != 1.0f) {  // lambda / scale, rounded to lambda's own type as the element-wise division would
        x = __fdiv_rn(x, lam_div);
        x = lam_dtype == GDR_FP32 ? x : lam_dtype == GDR_BF16 ? (float)(__bf16)x : (float)(_Float16)x;
      }
    }
    s_l[tid] = x;
    // the cascade as arithmetic on 0 / 1 coefficients (no branches in the row loops): the full levels below z are
    // summed, level z takes the sum, levels past L (loaded from a clamped index) are dropped
    s_m[tid] = (tid < L && tid < z) ? 1.0f : 0.0f;                 // enters the sum
    s_m[HGS_LMAX + tid] = (tid < L && tid >= z) ? 1.0f : 0.0f;     // keeps its value
    s_m[2 * HGS_LMAX + tid] = (z > 0 && tid == z) ? 1.0f : 0.0f;   // receives the sum
  }
  __syncthreads();
  qs = 0.0f;
  ks = 0.0f;
  for (int w = 0; w < 4; ++w) {
    qs += s_red[2 * w];
    ks += s_red[2 * w + 1];
  }
  float rq = scale, rk = 1.0f;
  if (l2norm == GDR_L2_CHUNK) {
    rq = scale / __fsqrt_rn(qs + 1e-6f);
    rk = 1.0f / __fsqrt_rn(ks + 1e-6f);
  } else if (l2norm == GDR_L2_RECURRENT) {
    rq = scale / (__fsqrt_rn(qs) + 1e-6f);
    rk = 1.0f / (__fsqrt_rn(ks) + 1e-6f);
  }
  const int grp = tid / HGS_COLS, jl = tid % HGS_COLS;
  const int j = blockIdx.y * HGS_COLS + jl;
  const bool live = j < V;
  const int jc = live ? j : V - 1;  // (idle threads shadow the last column and store nothing)
  const float a = __expf(g[(size_t)b * HV + hv]), bt = beta[(size_t)b * HV + hv];
  const float vj = GdrElem<T>::to_float(v[((size_t)b * HV + hv) * V + jc]);
  float* col = states + (((size_t)b * HV + hv) * K * V + jc) * L;  // row i of this column: col + i * V * L
  const size_t rs = (size_t)V * L;

  // A row's level values: LM unconditional loads (indices past L - 1 re-read the last level and are dropped), so that
  // all of them -- and those of the second row of a pair -- are in flight together; then the cascade.
  auto load_row = [&](const float* p, float* S) {
#pragma unroll
    for (int l = 0; l < LM; ++l) S[l] = p[min(l, L - 1)];
  };
  float m_sum[LM], m_keep[LM], m_take[LM];
#pragma unroll
  for (int l = 0; l < LM; ++l) {
    m_sum[l] = s_m[l];
    m_keep[l] = s_m[HGS_LMAX + l];
    m_take[l] = s_m[2 * HGS_LMAX + l];
  }
  auto cascade = [&](float* S) {
    float acc = m_sum[0] * S[0];
#pragma unroll
    for (int l = 1; l < LM; ++l) acc = __builtin_fmaf(m_sum[l], S[l], acc);  // S_1 + S_0, then + S_2 ...: exact 0 / 1 factors
#pragma unroll
    for (int l = 0; l < LM; ++l) S[l] = __builtin_fmaf(m_take[l], acc, m_keep[l] * S[l]);
  };
  float d[LM];
#pragma unroll
  for (int l = 0; l < LM; ++l) d[l] = 0.0f;
  for (int i = grp; i < K; i += 2 * HGS_GROUPS) {
    const int i2 = i + HGS_GROUPS;
    const bool two = i2 < K;
    float S[LM], S2[LM];
    load_row(col + i * rs, S);
    load_row(col + (two ? i2 : i) * rs, S2);
    cascade(S);
    cascade(S2);
    const float ki = s_k[i] * rk, ki2 = two ? s_k[i2] * rk : 0.0f;
#pragma unroll
    for (int l = 1; l < LM; ++l) d[l] = __builtin_fmaf(ki2, S2[l], __builtin_fmaf(ki, S[l], d[l]));
  }
  float* mine = s_part + (grp * HGS_COLS + jl) * (HGS_LMAX + 1);
  mine[0] = 0.0f;
#pragma unroll
  for (int l = 1; l < LM; ++l) mine[l] = d[l];
  __syncthreads();
  // sums over the row groups: one (column, level) pair per thread and round, then every thread takes its column's
  for (int pair = tid; pair < HGS_COLS * LM; pair += 256) {
    const int pc = pair / LM, pl = pair % LM;
    float t = 0.0f;
#pragma unroll
    for (int gq = 0; gq < HGS_GROUPS; ++gq) t += s_part[(gq * HGS_COLS + pc) * (HGS_LMAX + 1) + pl];
    s_tot[pc * (HGS_LMAX + 1) + pl] = t;
  }
  __syncthreads();
#pragma unroll
  for (int l = 1; l < LM; ++l) d[l] = s_tot[jl * (HGS_LMAX + 1) + l];
  float acc_o = 0.0f;
  auto update_row = [&](int i, float* S) {
    const float ki = s_k[i] * rk, qi = s_q[i] * rq;
    float sl = 0.0f;
    S[0] = bt * ki * vj;
#pragma unroll
    for (int l = 1; l < LM; ++l) S[l] = a * (S[l] - bt * ki * d[l]);
#pragma unroll
    for (int l = 0; l < LM; ++l) sl = __builtin_fmaf(s_l[l], S[l], sl);
    if (live) {
#pragma unroll
      for (int l = 0; l < LM; ++l)
        if (l < L) col[i * rs + l] = S[l];
    }
    acc_o = __builtin_fmaf(qi, sl, acc_o);
  };
  for (int i = grp; i < K; i += 2 * HGS_GROUPS) {
    const int i2 = i + HGS_GROUPS;
    const bool two = i2 < K;
    float S[LM], S2[LM];
    load_row(col + i * rs, S);
    load_row(col + (two ? i2 : i) * rs, S2);
    cascade(S);
    cascade(S2);
    update_row(i, S);
    if (two) update_row(i2, S2);
  }
  __syncthreads();  // every thread is done with the k^T S sums
  mine[0] = acc_o;
  __syncthreads();
  if (grp == 0 && live) {
    float t = 0.0f;
    for (int gq = 0; gq < HGS_GROUPS; ++gq) t += s_part[(gq * HGS_COLS + jl) * (HGS_LMAX + 1)];
    o[((size_t)b * HV + hv) * V + j] = GdrElem<T>::from_float(t);
  }
}

// The same token with the workgroup's part of the state staged in LDS: COLS value columns of every row are one
// contiguous piece of COLS * L floats, so the K pieces are read once with 16-byte accesses, worked on in LDS and written
// back once with 16-byte accesses. The cascade runs with a thread per (row, column) -- the only step that couples the
// levels of a row -- then a thread owns one (column, level) position of the piece and walks the rows
// i = group, group + 256 / (COLS * L), ...; k^T S_l and the output are sums of per-thread partial sums through LDS.
// Needs COLS * L <= 256, V * L a multiple of 4 floats, V a multiple of COLS and the pieces to fit in LDS; the kernel
// above covers the rest.
template <typename T, int COLS>
__global__ void __launch_bounds__(256)
    hgdn_step_lds_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                         const float* __restrict__ g, const float* __restrict__ beta, const void* __restrict__ lam,
                         int lam_dtype, float lam_div, float* __restrict__ states, T* __restrict__ o, int H, int HV,
                         int K, int V, int L, int z, float scale, int l2norm) {
  extern __shared__ float4 s_raw4[];
  const int PW = COLS * L;
  float* s_slab = reinterpret_cast<float*>(s_raw4);  // [K][PW], 16-byte aligned
  float* s_q = s_slab + K * PW;
  float* s_k = s_q + K;
  float* s_red = s_k + K;     // [8]
  float* s_part = s_red + 8;  // [256] partial sums of k^T S_l, then of the output
  const int b = blockIdx.x / HV, hv = blockIdx.x % HV, h = hv / (HV / H);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int groups = 256 / PW;
  const bool active = tid < groups * PW;
  const int grp = tid / PW, c = tid - grp * PW, jl = c / L, l = c - jl * L;
  // the token's own values first (short loads, in flight together with the pieces)
  const T* qp = q + ((size_t)b * H + h) * K;
  const T* kp = k + ((size_t)b * H + h) * K;
  float q0 = 0.0f, k0 = 0.0f, lam_l = 0.0f, vj = 0.0f;
  if (tid < K) {
    q0 = GdrElem<T>::to_float(qp[tid]);
    k0 = GdrElem<T>::to_float(kp[tid]);
  }
  if (active) {
    const size_t li = ((size_t)b * HV + hv) * L + l;
    lam_l = lam_dtype == GDR_FP32   ? reinterpret_cast<const float*>(lam)[li]
            : lam_dtype == GDR_BF16 ? (float)reinterpret_cast<const __bf16*>(lam)[li]
                                    : (float)reinterpret_cast<const _Float16*>(lam)[li];
    vj = GdrElem<T>::to_float(v[((size_t)b * HV + hv) * V + blockIdx.y * COLS + jl]);
  }
  const float g_tok = g[(size_t)b * HV + hv], bt = beta[(size_t)b * HV + hv];
  float* base = states + (((size_t)b * HV + hv) * K * V + (size_t)blockIdx.y * COLS) * L;  // row i: base + i * V * L
  const size_t rs = (size_t)V * L;
  const int p4 = PW / 4, n4 = K * p4;
  // the piece loads of a batch are all issued before the first is stored to LDS (one round trip per batch)
  for (int e0 = tid; e0 < n4; e0 += 256 * HGS_LOADS) {
    float4 r[HGS_LOADS];
#pragma unroll
    for (int u = 0; u < HGS_LOADS; ++u) {
      const int e = e0 + 256 * u;
      if (e < n4) {
        const int i = e / p4, c4 = e - i * p4;
        r[u] = reinterpret_cast<const float4*>(base + i * rs)[c4];
      }
    }
#pragma unroll
    for (int u = 0; u < HGS_LOADS; ++u) {
      const int e = e0 + 256 * u;
      if (e < n4) reinterpret_cast<float4*>(s_slab)[e] = r[u];
    }
  }
  float qs = q0 * q0, ks = k0 * k0;
  if (tid < K) {
    s_q[tid] = q0;
    s_k[tid] = k0;
  }
  for (int i = tid + 256; i < K; i += 256) {
    const float qi = GdrElem<T>::to_float(qp[i]), ki = GdrElem<T>::to_float(kp[i]);
    s_q[i] = qi;
    s_k[i] = ki;
    qs = __builtin_fmaf(qi, qi, qs);
    ks = __builtin_fmaf(ki, ki, ks);
  }
  for (int off = 32; off > 0; off >>= 1) {
    qs += __shfl_xor(qs, off);
    ks += __shfl_xor(ks, off);
  }
  if (lane == 0) {
    s_red[2 * wave] = qs;
    s_red[2 * wave + 1] = ks;
  }
  if (lam_div != 1.0f) {  // lambda / scale, rounded to lambda's own type as the element-wise division would
    lam_l = __fdiv_rn(lam_l, lam_div);
    lam_l = lam_dtype == GDR_FP32 ? lam_l : lam_dtype == GDR_BF16 ? (float)(__bf16)lam_l : (float)(_Float16)lam_l;
  }
  const float a = __expf(g_tok);
  __syncthreads();
  qs = 0.0f;
  ks = 0.0f;
  for (int w = 0; w < 4; ++w) {
    qs += s_red[2 * w];
    ks += s_red[2 * w + 1];
  }
  float rq = scale, rk = 1.0f;
  if (l2norm == GDR_L2_CHUNK) {
    rq = scale / __fsqrt_rn(qs + 1e-6f);
    rk = 1.0f / __fsqrt_rn(ks + 1e-6f);
  } else if (l2norm == GDR_L2_RECURRENT) {
    rq = scale / (__fsqrt_rn(qs) + 1e-6f);
    rk = 1.0f / (__fsqrt_rn(ks) + 1e-6f);
  }
  // cascade, a (row, column) pair per thread: the full levels below z are summed (S_1 + S_0, then + S_2 ...) into
  // level z and emptied
  if (z > 0) {
    for (int pr = tid; pr < K * COLS; pr += 256) {
      float* lv = s_slab + (pr / COLS) * PW + (pr % COLS) * L;
      float acc = lv[0];
      lv[0] = 0.0f;
      for (int m = 1; m < z; ++m) {
        acc += lv[m];
        lv[m] = 0.0f;
      }
      lv[z] += acc;
    }
    __syncthreads();
  }
  // k^T S_l on the unscaled key (the key's norm enters through the coefficients below); a thread's rows in batches
  // whose LDS reads are all issued before the first is used, the last rows one by one
  const int stride = groups * PW;
  const int n_rows = active ? (K - grp + groups - 1) / groups : 0;  // rows grp, grp + groups, ...
  float d = 0.0f;
  {
    const float* kr = s_k + grp;
    const float* sr = s_slab + grp * PW + c;
    int n = n_rows;
    for (; n >= HGS_ROWS; n -= HGS_ROWS, kr += HGS_ROWS * groups, sr += HGS_ROWS * stride) {
      float kk[HGS_ROWS], sv[HGS_ROWS];
#pragma unroll
      for (int u = 0; u < HGS_ROWS; ++u) {
        kk[u] = kr[u * groups];
        sv[u] = sr[u * stride];
      }
#pragma unroll
      for (int u = 0; u < HGS_ROWS; ++u) d = __builtin_fmaf(kk[u], sv[u], d);
    }
    for (; n > 0; --n, kr += groups, sr += stride) d = __builtin_fmaf(kr[0], sr[0], d);
  }
  s_part[tid] = d;
  __syncthreads();
  d = 0.0f;
  for (int gq = 0; gq < groups; ++gq) d += s_part[gq * PW + c];
  __syncthreads();  // every thread has its sum before the partial sums are used again
  // gate, insert, output: S <- c_a (c_m S + k_i c_b), with the coefficients of the thread's level
  //   l > 0: a (S - b k_i rk (rk d))      l = 0: b k_i rk v_j
  const float c_a = l == 0 ? 1.0f : a, c_m = l == 0 ? 0.0f : 1.0f, c_b = l == 0 ? bt * rk * vj : -(bt * rk) * (rk * d);
  float acc_o = 0.0f;
  {
    const float* kr = s_k + grp;
    const float* qr = s_q + grp;
    float* sr = s_slab + grp * PW + c;
    int n = n_rows;
    for (; n >= HGS_ROWS; n -= HGS_ROWS, kr += HGS_ROWS * groups, qr += HGS_ROWS * groups, sr += HGS_ROWS * stride) {
      float kk[HGS_ROWS], qq[HGS_ROWS], sv[HGS_ROWS];
#pragma unroll
      for (int u = 0; u < HGS_ROWS; ++u) {
        kk[u] = kr[u * groups];
        qq[u] = qr[u * groups];
        sv[u] = sr[u * stride];
      }
#pragma unroll
      for (int u = 0; u < HGS_ROWS; ++u) {
        const float x = c_a * __builtin_fmaf(kk[u], c_b, c_m * sv[u]);
        sr[u * stride] = x;
        acc_o = __builtin_fmaf(qq[u], x, acc_o);
      }
    }
    for (; n > 0; --n, kr += groups, qr += groups, sr += stride) {
      const float x = c_a * __builtin_fmaf(kr[0], c_b, c_m * sr[0]);
      sr[0] = x;
      acc_o = __builtin_fmaf(qr[0], x, acc_o);
    }
  }
  acc_o *= rq;
  s_part[tid] = lam_l * acc_o;
  __syncthreads();  // the updated rows and the output's partial sums are in LDS
  if (tid < COLS) {
    float t = 0.0f;
    for (int gq = 0; gq < groups; ++gq)
      for (int m = 0; m < L; ++m) t += s_part[gq * PW + tid * L + m];
    o[((size_t)b * HV + hv) * V + blockIdx.y * COLS + tid] = GdrElem<T>::from_float(t);
  }
  for (int e = tid; e < n4; e += 256) {
    const int i = e / p4, c4 = e - i * p4;
    reinterpret_cast<float4*>(base + i * rs)[c4] = reinterpret_cast<const float4*>(s_slab)[e];
  }
}

struct HgsArgs {
  const void *q, *k, *v;
  const float *g, *beta;
  const void* lam;
  int lam_dtype;
  float lam_div;
  float* states;
  void* o;
  int B, H, HV, K, V, L, z;
  float scale;
  int l2norm;
};

// One instantiation of the LDS-staged form: raises its dynamic LDS limit on the current device (set_attr) and launches
// it when it is the one picked.
template <typename TT, int CC>
static bool hgs_lds_one(const HgsArgs& a, bool set_attr, bool launch, size_t smem, hipStream_t s) {
  if (set_attr && hipFuncSetAttribute((const void*)hgdn_step_lds_kernel<TT, CC>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, HGS_LDS_LIMIT) != hipSuccess)
    return false;
  if (launch)
    hipLaunchKernelGGL((hgdn_step_lds_kernel<TT, CC>), dim3(a.B * a.HV, a.V / CC), dim3(256), smem, s, (const TT*)a.q,
                       (const TT*)a.k, (const TT*)a.v, a.g, a.beta, a.lam, a.lam_dtype, a.lam_div, a.states, (TT*)a.o,
                       a.H, a.HV, a.K, a.V, a.L, a.z, a.scale, a.l2norm);
  return true;
}

template <typename TT>
static bool hgs_lds_type(const HgsArgs& a, bool set_attr, bool mine, int cols, size_t smem, hipStream_t s) {
  return hgs_lds_one<TT, 4>(a, set_attr, mine && cols == 4, smem, s) &&
         hgs_lds_one<TT, 8>(a, set_attr, mine && cols == 8, smem, s);
}

// q, k [B, H, K]; v, o [B, HV, V] (dtype 0 bf16 / 1 fp16 / 2 fp32); g (log decay), beta fp32 [B, HV]; lam [B, HV, L] of
// lam_dtype, used as lam / lam_div rounded to its type; states fp32 [B, HV, K, V, L], updated in place;
// z: the levels 0 .. z-1 are full and cascade into level z (0: the state is empty). L <= 32.
extern "C" int lampa_hgdn_step(const void* q, const void* k, const void* v, const float* g, const float* beta,
                               const void* lam, int lam_dtype, float lam_div, float* states, void* o, int B, int H, int HV,
                               int K, int V, int L, int z, int dtype, float scale, int l2norm, void* stream) {
  if (!q || !k || !v || !g || !beta || !lam || !states || !o) return LAMPA_ERR_INVALID;
  if (B < 0 || H < 1 || HV < H || HV % H != 0 || K < 1 || V < 1 || L < 1 || z < 0 || z >= L) return LAMPA_ERR_INVALID;
  if (l2norm < 0 || l2norm > 2 || lam_dtype < 0 || lam_dtype > 2 || !(lam_div > 0.0f)) return LAMPA_ERR_INVALID;
  if (V > 1024 || L > HGS_LMAX || K > 4096 || dtype < 0 || dtype > 2) return LAMPA_ERR_UNSUPPORTED;
  if (B == 0) return LAMPA_OK;
  hipStream_t s = (hipStream_t)stream;
  LAMPA_PROF(s, "start");
  // the LDS-staged form where its layout conditions hold: 4 columns per workgroup (most workgroups, shortest loads)
  // unless the launch is large enough to fill the device with 8
  auto lds_bytes = [&](int cols) { return ((size_t)K * cols * L + 2 * (size_t)K + 8 + 256) * sizeof(float); };
  auto fits = [&](int cols) {
    return V % cols == 0 && cols * L <= 256 && ((size_t)V * L) % 4 == 0 &&
           (reinterpret_cast<uintptr_t>(states) & 15) == 0 && lds_bytes(cols) <= HGS_LDS_LIMIT;
  };
  const int cols = ((size_t)B * HV * (V / 4) > 8192 && fits(8)) ? 8 : fits(4) ? 4 : 0;
  if (cols) {
    static bool attr_set[64] = {};  // per device: the dynamic LDS limit of every instantiation (a repeated set is harmless)
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return LAMPA_ERR_LAUNCH;
    const HgsArgs a = {q, k, v, g, beta, lam, lam_dtype, lam_div, states, o, B, H, HV, K, V, L, z, scale, l2norm};
    const bool set_attr = !attr_set[dev];
    if (!hgs_lds_type<__bf16>(a, set_attr, dtype == GDR_BF16, cols, lds_bytes(cols), s) ||
        !hgs_lds_type<_Float16>(a, set_attr, dtype == GDR_FP16, cols, lds_bytes(cols), s) ||
        !hgs_lds_type<float>(a, set_attr, dtype == GDR_FP32, cols, lds_bytes(cols), s))
      return LAMPA_ERR_LAUNCH;
    attr_set[dev] = true;
    LAMPA_PROF(s, "hgdn_step_lds_kernel");
    return lampa_launch_status();
  }
  const size_t smem = (2 * (size_t)K + 4 * HGS_LMAX + 8 + (HGS_GROUPS + 1) * HGS_COLS * (HGS_LMAX + 1)) * sizeof(float);
#define HGS_LAUNCH(TT, LM)                                                                                         \
  hipLaunchKernelGGL((hgdn_step_kernel<TT, LM>), dim3(B * HV, (V + HGS_COLS - 1) / HGS_COLS), dim3(256), smem, s,  \
                     (const TT*)q, (const TT*)k, (const TT*)v, g, beta, lam, lam_dtype, lam_div, states, (TT*)o, H, \
                     HV, K, V, L, z, scale, l2norm)
#define HGS_CASE(TT)                    \
  do {                                  \
    if (L <= 16) HGS_LAUNCH(TT, 16);    \
    else if (L <= 24) HGS_LAUNCH(TT, 24); \
    else HGS_LAUNCH(TT, 32);            \
  } while (0)
  if (dtype == GDR_BF16) HGS_CASE(__bf16);
  else if (dtype == GDR_FP16) HGS_CASE(_Float16);
  else HGS_CASE(float);
#undef HGS_CASE
#undef HGS_LAUNCH
  LAMPA_PROF(s, "hgdn_step_kernel");
  return lampa_launch_status();
}

// ---- the tokens behind the whole chunks, in one launch -----------------------------------------------------------------
// A wavefront owns one value column of one (sequence, value head), in one of two layouts. What bounds both is the serial chain
// of a token (B * HV * V wavefronts, two per compute unit at 8 heads of 64 columns).
//
// hgdn_tail_kernel (up to 17 levels, sequences of up to 65 536 tokens): lane = (row group, level), a lane holds a quarter of
// the rows of one level > 0. All levels take a token's transition at once: k^T S_l is a lane's own sum over its rows and two
// register swaps over the row groups, the update a multiply and an fma per row. Level 0, the last token alone, is never
// stored: it enters the output as a scalar and the state of the level it cascades into as one fma per row; the levels
// between are summed over 16 lanes (DPP) every second token. k, q (normalised, fp32), the decays, the weights and v of 32
// tokens are staged in LDS by the workgroup's four waves, so a token waits for no load. Levels that hold no token yet are
// not read, and written as the zeros they are. RP, the rows of a lane: 4, 8, 16 or 32 as K asks. (With 16 rows for every
// K <= 64 and the loads of empty levels in front of the first token, many sequences of two or three tokens were slower than
// with the rows kernel: 128 x 2 tokens, 4 heads of 16 x 32, 34.3 us there, 47.6 so, 34.2 now; 4 of 32 x 64 78.7, 90.0, 66.5;
// 8 of 64 x 64 234, 174, 161.)
// hgdn_tail_rows_kernel (more levels): lane = state row (two rows for K > 64), the row's 32 level values in registers. Sums
// over the rows (k^T S_l for the levels > 0, the output, the two norms) are exchanges between lanes: 16 levels at a time are
// halved four times until a lane holds one level's sum over its group of 16 lanes (`wave_sums16`), and go back to all lanes
// as scalars; the next token's values are loaded while this one is worked on.
// A prefill of 15 000 tokens (24 behind its whole chunks, 8 heads of 64 x 64): 708 us with a launch of the single-token kernel
// and its copies per token, 188 us with the rows kernel (its own 38),
// 173 us with this one (25).
#define HGS_TAIL_LEVELS 17  // level 0 and one for each of 16 lanes: sequences up to 65 536 tokens
#define HGS_TAIL_WAVES 4
#define HGS_DPP_ROR8 0x128
#define HGS_DPP_HALF_MIRROR 0x141
#define HGS_DPP_MIRROR 0x140

__device__ __forceinline__ float hgs_fold32(float a, float b) {  // lanes < 32: both halves of a, lanes >= 32: of b
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

__device__ __forceinline__ float hgs_fold16(float a, float b) {  // even rows of 16 lanes: rows pairs of a, odd rows: of b
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

__device__ __forceinline__ float wave_sum_all(float x) {
  x = hgs_fold32(x, x);
  x = hgs_fold16(x, x);
  x += dpp_f32<HGS_DPP_ROR8, 0xF>(0.0f, x);
  x += dpp_f32<HGS_DPP_HALF_MIRROR, 0xF>(0.0f, x);
  x += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, x);
  return x + dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, x);
}

// Sums of 16 values over the wave: lanes 4n .. 4n + 3 return the sum of p[n] over all 64 lanes.
__device__ __forceinline__ float wave_sums16(float* p, int lane) {
#pragma unroll
  for (int n = 0; n < 8; ++n) p[n] = hgs_fold32(p[n], p[n + 8]);
#pragma unroll
  for (int n = 0; n < 4; ++n) p[n] = hgs_fold16(p[n], p[n + 4]);
  const bool b3 = lane & 8, b2 = lane & 4;
#pragma unroll
  for (int n = 0; n < 2; ++n)
    p[n] = (b3 ? p[n + 2] : p[n]) + dpp_f32<HGS_DPP_ROR8, 0xF>(0.0f, b3 ? p[n] : p[n + 2]);
  float x = (b2 ? p[1] : p[0]) + dpp_f32<HGS_DPP_HALF_MIRROR, 0xF>(0.0f, b2 ? p[0] : p[1]);
  x += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, x);
  return x + dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, x);
}

__device__ __forceinline__ float hgs_lane(float x, int n) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), n));
}

template <typename T, int ROWS>
__global__ void __launch_bounds__(64 * HGS_TAIL_WAVES)
    hgdn_tail_rows_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                     const float* __restrict__ g, const float* __restrict__ beta, const void* __restrict__ lam,
                     int lam_dtype, float lam_div, float* __restrict__ states, T* __restrict__ o, int n_tok, int tok0, int H,
                     int HV, int K, int V, int L, float scale, int l2norm) {
  const int lane = threadIdx.x & 63;
  const int j = blockIdx.y * HGS_TAIL_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (j >= V) return;
  const int b = blockIdx.x / HV, hv = blockIdx.x % HV, h = hv / (HV / H);
  float* col = states + (((size_t)b * HV + hv) * K * V + j) * L;  // row i: col + i * V * L
  // Loads come from clamped addresses without conditions on the lane, and are converted and masked where they are used: a
  // conditional load that is converted on the spot is a branch with a wait for memory inside (one per value: four round
  // trips per token, and one per level at either end).
  constexpr int LM = HGS_LMAX;
  float S[ROWS][LM];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int l = 0; l < LM; ++l) S[r][l] = col[(size_t)min(lane + 64 * r, K - 1) * V * L + min(l, L - 1)];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int l = 0; l < LM; ++l) S[r][l] = (lane + 64 * r < K && l < L) ? S[r][l] : 0.0f;
  struct Token {
    T q[ROWS], k[ROWS], v;
    uint32_t lam;
    float g, beta;
  };
  const int lam_at = min(lane, L - 1);
  auto load = [&](int t) {
    Token x;
    const size_t tok = (size_t)b * n_tok + t;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int i = min(lane + 64 * r, K - 1);
      x.q[r] = q[(tok * H + h) * K + i];
      x.k[r] = k[(tok * H + h) * K + i];
    }
    const size_t li = (tok * HV + hv) * L + lam_at;
    if (lam_dtype == GDR_FP32) x.lam = reinterpret_cast<const uint32_t*>(lam)[li];
    else x.lam = reinterpret_cast<const uint16_t*>(lam)[li];
    x.v = v[(tok * HV + hv) * V + j];
    x.g = g[tok * HV + hv];
    x.beta = beta[tok * HV + hv];
    return x;
  };
  auto lam_value = [&](uint32_t raw) {
    if (lane >= L) return 0.0f;
    return lam_dtype == GDR_FP32   ? __uint_as_float(raw)
           : lam_dtype == GDR_BF16 ? __uint_as_float(raw << 16)
                                   : (float)__builtin_bit_cast(_Float16, (uint16_t)raw);
  };
  // A token's output is stored at the start of the next token, ahead of the loads that are requested there: behind them the
  // wait for those loads would also be one for the store.
  float acc_o = 0.0f;
  auto store = [&](int t) {
    if (lane == 0) o[(((size_t)b * n_tok + t) * HV + hv) * V + j] = GdrElem<T>::from_float(acc_o);
  };
  Token next = load(tok0);
  for (int t = tok0; t < n_tok; ++t) {
    struct {
      float q[ROWS], k[ROWS], v, g, beta;
    } x;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      x.q[r] = lane + 64 * r < K ? GdrElem<T>::to_float(next.q[r]) : 0.0f;
      x.k[r] = lane + 64 * r < K ? GdrElem<T>::to_float(next.k[r]) : 0.0f;
    }
    x.v = GdrElem<T>::to_float(next.v);
    x.g = next.g;
    x.beta = next.beta;
    float lam_l = lam_value(next.lam);
    if (t > tok0) store(t - 1);
    next = load(min(t + 1, n_tok - 1));
    if (lam_div != 1.0f) {  // lambda / scale, rounded to lambda's own type as the element-wise division would
      lam_l = __fdiv_rn(lam_l, lam_div);
      lam_l = lam_dtype == GDR_FP32 ? lam_l : lam_dtype == GDR_BF16 ? (float)(__bf16)lam_l : (float)(_Float16)lam_l;
    }
    // cascade: after t tokens the levels below 1 + (trailing zero bits of t) are full
    const int z = t == 0 ? 0 : 1 + __builtin_ctz(t);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      float acc = S[r][0];
#pragma unroll
      for (int l = 1; l < LM; ++l) {
        const float s = S[r][l];
        S[r][l] = l < z ? 0.0f : l == z ? s + acc : s;
        acc = l < z ? acc + s : acc;
      }
      S[r][0] = 0.0f;  // (empty before the first token)
    }
    float qs = 0.0f, ks = 0.0f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      qs = __builtin_fmaf(x.q[r], x.q[r], qs);
      ks = __builtin_fmaf(x.k[r], x.k[r], ks);
    }
    float rq = scale, rk = 1.0f;
    if (l2norm == GDR_L2_CHUNK) {
      rq = scale / __fsqrt_rn(wave_sum_all(qs) + 1e-6f);
      rk = 1.0f / __fsqrt_rn(wave_sum_all(ks) + 1e-6f);
    } else if (l2norm == GDR_L2_RECURRENT) {
      rq = scale / (__fsqrt_rn(wave_sum_all(qs)) + 1e-6f);
      rk = 1.0f / (__fsqrt_rn(wave_sum_all(ks)) + 1e-6f);
    }
    const float a = __expf(x.g), bk = x.beta * rk;
    float sl[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      S[r][0] = x.k[r] * (bk * x.v);
      sl[r] = hgs_lane(lam_l, 0) * S[r][0];
    }
#pragma unroll
    for (int l0 = 1; l0 < LM; l0 += 16) {
      float p[16];
#pragma unroll
      for (int n = 0; n < 16; ++n) {
        p[n] = 0.0f;
        if (l0 + n < LM)
#pragma unroll
          for (int r = 0; r < ROWS; ++r) p[n] = __builtin_fmaf(x.k[r], S[r][l0 + n], p[n]);
      }
      const float d = wave_sums16(p, lane);
#pragma unroll
      for (int n = 0; n < 16; ++n) {
        const int l = l0 + n;
        if (l < LM) {
          const float c = -bk * (rk * hgs_lane(d, 4 * n)), al = l < L ? a : 0.0f;
#pragma unroll
          for (int r = 0; r < ROWS; ++r) {
            S[r][l] = al * __builtin_fmaf(x.k[r], c, S[r][l]);
            sl[r] = __builtin_fmaf(hgs_lane(lam_l, l), S[r][l], sl[r]);
          }
        }
      }
    }
    acc_o = 0.0f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) acc_o = __builtin_fmaf(x.q[r], sl[r], acc_o);
    acc_o = rq * wave_sum_all(acc_o);
  }
  store(n_tok - 1);
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int i = lane + 64 * r;
#pragma unroll
    for (int l = 0; l < LM; ++l)
      if (i < K && l < L) col[(size_t)i * V * L + l] = S[r][l];
  }
}

#define HGS_TAIL_BATCH 32  // tokens staged at a time

template <typename T, int RP>
__global__ void __launch_bounds__(64 * HGS_TAIL_WAVES)
    hgdn_tail_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                     const float* __restrict__ g, const float* __restrict__ beta, const void* __restrict__ lam,
                     int lam_dtype, float lam_div, float* __restrict__ states, T* __restrict__ o, int n_tok, int tok0, int H,
                     int HV, int K, int V, int L, float scale, int l2norm) {
  constexpr int KP = 4 * RP, NB = HGS_TAIL_BATCH, TPW = NB / HGS_TAIL_WAVES, NR = KP > 64 ? KP / 64 : 1;
  __shared__ __align__(16) float s_k[NB][KP], s_q[NB][KP];
  __shared__ float s_lam[NB][HGS_TAIL_LEVELS], s_v[NB][HGS_TAIL_WAVES];
  __shared__ float4 s_sc[NB];  // e^g, beta, k . q
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int rg = lane >> 4, level = 1 + (lane & 15);
  const int j = min((int)blockIdx.y * HGS_TAIL_WAVES + wave, V - 1);  // (waves past V work on the last column, storing nothing)
  const bool live = (int)blockIdx.y * HGS_TAIL_WAVES + wave < V;
  const int b = blockIdx.x / HV, hv = blockIdx.x % HV, h = hv / (HV / H);
  float* col = states + (((size_t)b * HV + hv) * K * V + j) * L;  // row i: col + i * V * L
  // (loads come from clamped addresses without conditions on the lane and are masked where they are used)
  const bool filled = level < L && tok0 > 0 && ((tok0 - 1) >> (level - 1)) & 1;  // tokens in this lane's level
  float S[RP], prev[RP];  // prev: the k of the token before (first token: level 0 as it was)
#pragma unroll
  for (int r = 0; r < RP; ++r) S[r] = prev[r] = 0.0f;
  if (tok0 > 0) {  // (else no level holds a token)
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      const size_t at = (size_t)min(rg * RP + r, K - 1) * V * L;
      S[r] = col[at + min(level, L - 1)];
      prev[r] = col[at];
    }
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      S[r] = filled && rg * RP + r < K ? S[r] : 0.0f;
      prev[r] = rg * RP + r < K ? prev[r] : 0.0f;
    }
  }
  float prev_v = 1.0f;  // beta v of the token before
  auto stage = [&](int t0) __attribute__((always_inline)) {  // tokens t0 .. t0 + NB - 1, TPW of them by each wave
    T kr[TPW][NR], qr[TPW][NR];
    uint32_t lr[TPW];
    float gr[TPW], br[TPW];
    T vr[TPW];
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const size_t tok = (size_t)b * n_tok + min(t0 + wave * TPW + i, n_tok - 1);
#pragma unroll
      for (int x = 0; x < NR; ++x) {
        const int e = min(lane + 64 * x, K - 1);
        kr[i][x] = k[(tok * H + h) * K + e];
        qr[i][x] = q[(tok * H + h) * K + e];
      }
      const size_t li = (tok * HV + hv) * L + min(lane, L - 1);
      lr[i] = lam_dtype == GDR_FP32 ? reinterpret_cast<const uint32_t*>(lam)[li] : reinterpret_cast<const uint16_t*>(lam)[li];
      gr[i] = g[tok * HV + hv];
      br[i] = beta[tok * HV + hv];
      vr[i] = v[(tok * HV + hv) * V + min((int)blockIdx.y * HGS_TAIL_WAVES + min(lane, HGS_TAIL_WAVES - 1), V - 1)];
    }
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int at = wave * TPW + i;
      float kf[NR], qf[NR], ks = 0.0f, qs = 0.0f, kq = 0.0f;
#pragma unroll
      for (int x = 0; x < NR; ++x) {
        kf[x] = lane + 64 * x < K ? GdrElem<T>::to_float(kr[i][x]) : 0.0f;
        qf[x] = lane + 64 * x < K ? GdrElem<T>::to_float(qr[i][x]) : 0.0f;
        ks = __builtin_fmaf(kf[x], kf[x], ks);
        qs = __builtin_fmaf(qf[x], qf[x], qs);
      }
      float rq = scale, rk = 1.0f;
      if (l2norm == GDR_L2_CHUNK) {
        rq = scale / __fsqrt_rn(wave_sum_all(qs) + 1e-6f);
        rk = 1.0f / __fsqrt_rn(wave_sum_all(ks) + 1e-6f);
      } else if (l2norm == GDR_L2_RECURRENT) {
        rq = scale / (__fsqrt_rn(wave_sum_all(qs)) + 1e-6f);
        rk = 1.0f / (__fsqrt_rn(wave_sum_all(ks)) + 1e-6f);
      }
#pragma unroll
      for (int x = 0; x < NR; ++x) {
        kf[x] *= rk;
        qf[x] *= rq;
        kq = __builtin_fmaf(kf[x], qf[x], kq);
        if (KP >= 64 || lane < KP) {
          s_k[at][lane + 64 * x] = kf[x];
          s_q[at][lane + 64 * x] = qf[x];
        }
      }
      kq = wave_sum_all(kq);
      float lam_l = lam_dtype == GDR_FP32   ? __uint_as_float(lr[i])
                    : lam_dtype == GDR_BF16 ? __uint_as_float(lr[i] << 16)
                                            : (float)__builtin_bit_cast(_Float16, (uint16_t)lr[i]);
      if (lam_div != 1.0f) {  // lambda / scale, rounded to lambda's own type as the element-wise division would
        lam_l = __fdiv_rn(lam_l, lam_div);
        lam_l = lam_dtype == GDR_FP32 ? lam_l : lam_dtype == GDR_BF16 ? (float)(__bf16)lam_l : (float)(_Float16)lam_l;
      }
      if (lane < HGS_TAIL_LEVELS) s_lam[at][lane] = lane < L ? lam_l : 0.0f;
      if (lane < HGS_TAIL_WAVES) s_v[at][lane] = GdrElem<T>::to_float(vr[i]);
      if (lane == 0) s_sc[at] = make_float4(__expf(gr[i]), br[i], kq, 0.0f);
    }
  };
  for (int t0 = tok0; t0 < n_tok; t0 += NB) {
    if (t0 > tok0) __syncthreads();  // (the batch before has been read)
    stage(t0);
    __syncthreads();
    const int n = min(NB, n_tok - t0);
    for (int i = 0; i < n; ++i) {
      const int t = t0 + i;
      float kk[RP], qq[RP];
#pragma unroll
      for (int r = 0; r < RP; r += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(&s_k[i][rg * RP + r]), y = *reinterpret_cast<const f32x4*>(&s_q[i][rg * RP + r]);
#pragma unroll
        for (int e = 0; e < 4; ++e) { kk[r + e] = x[e]; qq[r + e] = y[e]; }
      }
      const float4 sc = s_sc[i];
      const float lam_l = s_lam[i][level], lam_0 = s_lam[i][0], bv = sc.y * s_v[i][wave];
      // cascade: after t tokens the levels below z = 1 + (trailing zero bits of t) are full and go into level z
      const int z = t == 0 ? 0 : 1 + __builtin_ctz(t);
      if (z > 1) {
#pragma unroll
        for (int r = 0; r < RP; ++r) {
          float x = level < z ? S[r] : 0.0f;
          x += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, x);
          x += dpp_f32<GDR_DPP_QUAD_XOR2, 0xF>(0.0f, x);
          x += dpp_f32<HGS_DPP_HALF_MIRROR, 0xF>(0.0f, x);
          x += dpp_f32<HGS_DPP_MIRROR, 0xF>(0.0f, x);
          S[r] = level < z ? 0.0f : level == z ? S[r] + x : S[r];
        }
      }
      const float into = level == z ? prev_v : 0.0f;
      if (t == tok0) {  // (level 0 as it came may hold anything)
#pragma unroll
        for (int r = 0; r < RP; ++r) S[r] = level == z ? S[r] + prev[r] : S[r];
      } else {
#pragma unroll
        for (int r = 0; r < RP; ++r) S[r] = __builtin_fmaf(prev[r], into, S[r]);
      }
      float d0 = 0.0f, d1 = 0.0f;
#pragma unroll
      for (int r = 0; r < RP; r += 2) {
        d0 = __builtin_fmaf(kk[r], S[r], d0);
        d1 = __builtin_fmaf(kk[r + 1], S[r + 1], d1);
      }
      float d = d0 + d1;
      d = hgs_fold32(d, d);
      d = hgs_fold16(d, d);
      const float c = -sc.y * d;
      float y0 = 0.0f, y1 = 0.0f;
#pragma unroll
      for (int r = 0; r < RP; ++r) {
        S[r] = sc.x * __builtin_fmaf(kk[r], c, S[r]);
        prev[r] = kk[r];
        if (r & 1) y1 = __builtin_fmaf(qq[r], S[r], y1);
        else y0 = __builtin_fmaf(qq[r], S[r], y0);
      }
      prev_v = bv;
      const float y = wave_sum_all(lam_l * (y0 + y1)) + lam_0 * (bv * sc.z);
      if (lane == 0 && live) o[(((size_t)b * n_tok + t) * HV + hv) * V + j] = GdrElem<T>::from_float(y);
    }
  }
  if (!live) return;
#pragma unroll
  for (int r = 0; r < RP; ++r) {
    const int i = rg * RP + r;
    if (i < K && level < L) col[(size_t)i * V * L + level] = S[r];
  }
  // level 0, the last token alone: a row per lane (the last batch is still in LDS)
  const int last = (n_tok - 1 - tok0) % NB;
#pragma unroll
  for (int x = 0; x < NR; ++x)
    if (lane + 64 * x < K) col[(size_t)(lane + 64 * x) * V * L] = s_k[last][lane + 64 * x] * prev_v;
}

// Tokens tok0 .. n_tok - 1 of every sequence on the level states after its first tok0 tokens: q, k [B, n_tok, H, K],
// v, o [B, n_tok, HV, V], g, beta [B, n_tok, HV], lam [B, n_tok, HV, L], states [B, HV, K, V, L] updated in place.
extern "C" int lampa_hgdn_tail(const void* q, const void* k, const void* v, const float* g, const float* beta,
                               const void* lam, int lam_dtype, float lam_div, float* states, void* o, int B, int n_tok,
                               int tok0, int H, int HV, int K, int V, int L, int dtype, float scale, int l2norm,
                               void* stream) {
  if (!q || !k || !v || !g || !beta || !lam || !states || !o) return LAMPA_ERR_INVALID;
  if (B < 0 || H < 1 || HV < H || HV % H != 0 || K < 1 || V < 1 || L < 1 || tok0 < 0 || n_tok < tok0)
    return LAMPA_ERR_INVALID;
  if (l2norm < 0 || l2norm > 2 || lam_dtype < 0 || lam_dtype > 2 || !(lam_div > 0.0f)) return LAMPA_ERR_INVALID;
  if (V > 1024 || L > HGS_LMAX || K > 128 || dtype < 0 || dtype > 2) return LAMPA_ERR_UNSUPPORTED;
  if (B == 0 || n_tok == tok0) return LAMPA_OK;
  // the level that the fullest cascade of these tokens fills has to exist (token t fills level 1 + its trailing zero bits)
  for (int t = tok0 > 1 ? tok0 : 1; t < n_tok; ++t)
    if (1 + __builtin_ctz(t) >= L) return LAMPA_ERR_INVALID;
  hipStream_t s = (hipStream_t)stream;
  LAMPA_PROF(s, "start");
#define HGS_TAIL(KERNEL)                                                                                                   \
  hipLaunchKernelGGL((KERNEL), dim3(B * HV, (V + HGS_TAIL_WAVES - 1) / HGS_TAIL_WAVES), dim3(64 * HGS_TAIL_WAVES), 0, s,   \
                     (const TT*)q, (const TT*)k, (const TT*)v, g, beta, lam, lam_dtype, lam_div, states, (TT*)o, n_tok,    \
                     tok0, H, HV, K, V, L, scale, l2norm)
#define HGS_TAIL_CASE(TYPE)                                                      \
  do {                                                                           \
    typedef TYPE TT;                                                             \
    if (L <= HGS_TAIL_LEVELS) {                                                  \
      if (K <= 16) HGS_TAIL(hgdn_tail_kernel<TT HGS_COMMA 4>);                   \
      else if (K <= 32) HGS_TAIL(hgdn_tail_kernel<TT HGS_COMMA 8>);              \
      else if (K <= 64) HGS_TAIL(hgdn_tail_kernel<TT HGS_COMMA 16>);             \
      else HGS_TAIL(hgdn_tail_kernel<TT HGS_COMMA 32>);                          \
    } else {                                                                     \
      if (K <= 64) HGS_TAIL(hgdn_tail_rows_kernel<TT HGS_COMMA 1>);              \
      else HGS_TAIL(hgdn_tail_rows_kernel<TT HGS_COMMA 2>);                      \
    }                                                                            \
  } while (0)
#define HGS_COMMA ,
  if (dtype == GDR_BF16) HGS_TAIL_CASE(__bf16);
  else if (dtype == GDR_FP16) HGS_TAIL_CASE(_Float16);
  else HGS_TAIL_CASE(float);
#undef HGS_TAIL_CASE
#undef HGS_COMMA
#undef HGS_TAIL
  LAMPA_PROF(s, "hgdn_tail_kernel");
  return lampa_launch_status();
}
