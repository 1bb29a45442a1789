// Host side of the chunkwise gated-delta-rule forward: workspace layout, launch sequence and the C entry points.
// The kernels (and the description of the algorithm) are in gdr_chunk_kernels.h.
#include "gdr_chunk_kernels.h"
#include "gdr_train.h"
#include <algorithm>
#include <atomic>
#include <mutex>

struct GdrWorkspace {
  int64_t off_t, off_m, off_n, off_d, off_sinit, off_gm, off_gn, off_gd, max_groups, bytes;
};

// kept: the records and the edges are kept elsewhere (training form)
static GdrWorkspace gdr_workspace(int64_t chunks, int64_t segs, int HV, int K, int V, bool kept = false) {
  GdrWorkspace w;
  int64_t off = 0;
  w.off_t = off;     off += kept ? 0 : lampa_align_up(chunks * HV * (int64_t)REC_BYTES, 256);
  w.off_m = off;     off += lampa_align_up(segs * HV * (int64_t)K * K * 2, 256);
  w.off_n = off;     off += lampa_align_up(segs * HV * (int64_t)K * V * 4, 256);
  w.off_d = off;     off += lampa_align_up(segs * HV * 4, 256);
  // the segments' initial states + a spare slot (scan); before the scan the chunks' edges (GDR_EDGE_*)
  w.off_sinit = off; off += lampa_align_up(std::max((segs + 1) * HV * (int64_t)K * V, kept ? 0 : chunks * HV) * 4, 256);
  // two-level scan: composites of the groups of GDR_SCAN_GROUP segments
  w.max_groups = segs / GDR_SCAN_GROUP + 2;
  w.off_gm = off;    off += lampa_align_up(w.max_groups * HV * (int64_t)K * K * 2, 256);
  w.off_gn = off;    off += lampa_align_up(w.max_groups * HV * (int64_t)K * V * 4, 256);
  w.off_gd = off;    off += lampa_align_up(w.max_groups * HV * 4, 256);
  w.bytes = off > 0 ? off : 256;
  return w;
}

// Output pass with narrow chain waves (16 value columns per wave on the 16x16x32 MFMA; built for K >= 64).
// 0: never, 1: where it is the faster form (heads wider than 64 x 64), 2: wherever it is built.
static std::atomic<int> gdr_narrow_output{1};
extern "C" int lampa_gdr_chunk_config(int narrow_output) {
  if (narrow_output < 0 || narrow_output > 2) return LAMPA_ERR_INVALID;
  gdr_narrow_output.store(narrow_output);
  return LAMPA_OK;
}

static bool gdr_chunk_supported(int K, int V) {
  return ((K == 64 || K == 128) && (V == 64 || V == 128)) || (K == 32 && V == 32);
}

extern "C" int64_t lampa_gdr_chunk_workspace_bytes(int64_t total_chunks, int64_t n_segments, int HV, int K, int V) {
  if (total_chunks < 0 || n_segments < 0 || HV < 1) return LAMPA_ERR_INVALID;
  if (!gdr_chunk_supported(K, V)) return LAMPA_ERR_UNSUPPORTED;
  return gdr_workspace(total_chunks, n_segments, HV, K, V).bytes;
}

// chunks of the longest segment
static int gdr_max_chunks(const int32_t* plan_host) {
  return plan_host[plan_host[PLAN_OFF_SEG_NCHUNKS] + plan_host[plan_host[PLAN_OFF_SEG_ORDER]]];
}

// Buffers of the training form (gdr_train.h), or none.
struct GdrKeep {
  unsigned char *rec, *states, *mt;
  float *d, *edge;
  int32_t* positive_g;
  int o_width;
};

template <typename T, int KT, int VT, bool KEEP = false>
static int gdr_chunk_launch(const void* q, const void* k, const void* v, const float* g, const float* beta, void* o,
                            const float* h0, float* ht, const GdrPlanView pv, int n_seq, int chunks, int segs, int max_nseg,
                            int max_chunks, int H, int HV, float scale, int l2norm, unsigned char* ws, hipStream_t s,
                            const GdrKeep kp = GdrKeep{}) {
  const GdrWorkspace w = gdr_workspace(chunks, segs, HV, KT, VT, KEEP);
  unsigned char* tf = KEEP ? kp.rec : ws + w.off_t;
  unsigned char* Mc = ws + w.off_m;
  unsigned char* Nc = ws + w.off_n;
  float* Dc = KEEP ? kp.d : (float*)(ws + w.off_d);
  float* Si = (float*)(ws + w.off_sinit);
  constexpr int smem_a = GdrSegSmem<KT, VT, false>::BYTES, smem_b = GdrSegSmem<KT, VT, true>::BYTES;
  constexpr int CWN = KT >= 64 ? 16 : 32;  // chain-wave width of the narrow output pass (K = 32 has none)
  constexpr int smem_n = GdrSegSmem<KT, VT, true, false, GdrSegShape<KT, VT, true, CWN>::DOUBLE_Q ? 2 : 1>::BYTES;
  // the dynamic LDS limit is a per-device attribute of a kernel: set once per device and instantiation
  static bool attr_set[64] = {};
  static std::mutex attr_lock;  // (several host threads may call at once)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return LAMPA_ERR_LAUNCH;
  std::unique_lock<std::mutex> hold(attr_lock);
  if (!attr_set[dev]) {
    if (hipFuncSetAttribute((const void*)gdr_segment_kernel<T, KT, VT, false, true, T, 32, KEEP>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem_a) != hipSuccess ||
        hipFuncSetAttribute((const void*)gdr_segment_kernel<T, KT, VT, false, true, T, 32, KEEP, false>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem_a) != hipSuccess ||
        hipFuncSetAttribute((const void*)gdr_segment_kernel<T, KT, VT, true, false, T, 32, KEEP>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem_b) != hipSuccess ||
        hipFuncSetAttribute((const void*)gdr_segment_kernel<T, KT, VT, true, false, T, CWN>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem_n) != hipSuccess)
      return LAMPA_ERR_LAUNCH;
    attr_set[dev] = true;
  }
  hold.unlock();
  LAMPA_PROF(s, "start");
  float* const edges = KEEP ? kp.edge : Si;
  float* edge = segs > n_seq && max_chunks >= GDR_EDGE_NC ? edges : nullptr;  // (of shorter segments no one asks for them)
  if (chunks > 0) {
    hipLaunchKernelGGL((gdr_local_kernel<T, T, KT>), dim3(gdr_local_grid(chunks, HV)), dim3(64), 0, s, (const T*)k, g, beta,
                       pv.chunk_tok0, pv.chunk_len, tf, chunks, H, HV, l2norm, kp.positive_g, edge);
    LAMPA_PROF(s, "gdr_local_kernel");
    if (segs > n_seq) {
      hipLaunchKernelGGL((edge ? gdr_segment_kernel<T, KT, VT, false, true, T, 32, KEEP>
                               : gdr_segment_kernel<T, KT, VT, false, true, T, 32, KEEP, false>), dim3(segs * HV), dim3(64 * GdrSegShape<KT, VT, false>::WAVES), smem_a, s,
                         (const T*)q, (const T*)k, (const T*)v, g, beta, pv, pv.chunk_tok0, pv.chunk_len, tf, (const float*)edges, Mc, Nc, Dc,
                         (T*)nullptr, (float*)nullptr, H, HV, scale, l2norm, (const unsigned char*)nullptr,
                         (const unsigned char*)nullptr, (const float*)nullptr, (const float*)nullptr, 0, kp.mt, VT);
      LAMPA_PROF(s, "gdr_segment_kernel<composite>");
    }
  }
  const int gmax = (max_nseg + GDR_SCAN_GROUP - 1) / GDR_SCAN_GROUP;
  unsigned char* Gm = ws + w.off_gm;
  unsigned char* Gn = ws + w.off_gn;
  float* Gd = (float*)(ws + w.off_gd);
  // The output pass can walk the composites before its segment itself (K = 64: its chain waves hold whole columns
  // of the state in few enough registers); otherwise a leaf pass writes every segment's initial state.
  const bool two_level = max_nseg >= 3 * GDR_SCAN_GROUP && (int64_t)n_seq * gmax <= w.max_groups;
  const bool walk_in_output = two_level && KT == 64;
  if (two_level) {
    // long sequences: group composites, then every group's scan (which walks the earlier groups' composites first)
    const dim3 block(64 * (KT / 32));
    hipLaunchKernelGGL((gdr_scan2_kernel<T, KT, VT, 4, SCAN_GROUP>), dim3((KT + VT) / 32 * gmax, n_seq, HV), block, 0, s, pv, Mc,
                       Nc, Dc, (const float*)nullptr, (float*)nullptr, Gm, Gn, Gd, HV, 0, gmax);
    LAMPA_PROF(s, "gdr_scan2_kernel<group>");
    if (!walk_in_output) {
      hipLaunchKernelGGL((gdr_scan2_kernel<T, KT, VT, 4, SCAN_LEAF>), dim3(VT / 32 * gmax, n_seq, HV), block, 0, s, pv, Mc, Nc,
                         Dc, h0, Si, Gm, Gn, Gd, HV, segs, gmax);
      LAMPA_PROF(s, "gdr_scan2_kernel<leaf>");
    }
  } else if (segs > n_seq || h0) {  // (sequences of one segment without a state start from zero)
    hipLaunchKernelGGL((gdr_scan_kernel<T, KT, VT, 4>), dim3(n_seq, HV, VT / 32), dim3(64 * (KT / 32)), 0, s,
                       pv, Mc, Nc, Dc, h0, Si, HV, segs);
    LAMPA_PROF(s, "gdr_scan_kernel");
  }
  const int narrow = gdr_narrow_output.load();
  if (!KEEP && CWN == 16 && (narrow == 2 || (narrow == 1 && KT + VT > 128)))
    hipLaunchKernelGGL((gdr_segment_kernel<T, KT, VT, true, false, T, CWN>), dim3(segs * HV),
                       dim3(64 * GdrSegShape<KT, VT, true, CWN>::WAVES), smem_n, s, (const T*)q, (const T*)k, (const T*)v, g, beta,
                       pv, pv.chunk_tok0, pv.chunk_len, tf, Si, Mc, Nc, Dc, (T*)o, ht, H, HV, scale, l2norm,
                       (const unsigned char*)Gm, (const unsigned char*)Gn, (const float*)Gd, h0, walk_in_output ? gmax : 0, kp.states, KEEP ? kp.o_width : VT);
  else
  hipLaunchKernelGGL((gdr_segment_kernel<T, KT, VT, true, false, T, 32, KEEP>), dim3(segs * HV), dim3(64 * GdrSegShape<KT, VT, true>::WAVES), smem_b, s, (const T*)q,
                     (const T*)k, (const T*)v, g, beta, pv, pv.chunk_tok0, pv.chunk_len, tf, Si, Mc, Nc, Dc, (T*)o, ht, H, HV, scale,
                     l2norm, (const unsigned char*)Gm, (const unsigned char*)Gn, (const float*)Gd, h0, walk_in_output ? gmax : 0, kp.states, KEEP ? kp.o_width : VT);
  LAMPA_PROF(s, "gdr_segment_kernel<output>");
  return lampa_launch_status();
}

// Chunkwise forward. q, k [total_tokens, H, K]; v, o [total_tokens, HV, V] (dtype 0 bf16 / 1 fp16); g, beta fp32
// [total_tokens, HV]; h0, ht fp32 [n_seq, HV, K, V] (nullable). plan_host / plan_dev: the same plan
// (lampa_gdr_plan_fill) in host and in device memory. workspace: lampa_gdr_chunk_workspace_bytes bytes.
extern "C" int lampa_gdr_chunk_fwd(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                   void* o, const float* h0, float* ht, const int32_t* plan_host,
                                   const int32_t* plan_dev, int H, int HV, int K, int V, int dtype, float scale,
                                   int l2norm, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!q || !k || !v || !g || !beta || !o || !plan_host || !plan_dev) return LAMPA_ERR_INVALID;
  if (H < 1 || HV < H || HV % H != 0 || l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (!gdr_chunk_supported(K, V) || (dtype != GDR_BF16 && dtype != GDR_FP16)) return LAMPA_ERR_UNSUPPORTED;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) & 15) return LAMPA_ERR_INVALID;
  const int n_seq = plan_host[PLAN_N_SEQ], chunks = plan_host[PLAN_TOTAL_CHUNKS], segs = plan_host[PLAN_N_SEGMENTS];
  if (n_seq < 1 || segs < n_seq) return LAMPA_ERR_INVALID;
  if (!workspace || workspace_bytes < gdr_workspace(chunks, segs, HV, K, V).bytes) return LAMPA_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  unsigned char* ws = (unsigned char*)workspace;
  const GdrPlanView pv = gdr_plan_view(plan_host, plan_dev);
  int max_nseg = 0;
  for (int i = 0; i < n_seq; ++i) max_nseg = plan_host[plan_host[PLAN_OFF_SEQ_NSEG] + i] > max_nseg ? plan_host[plan_host[PLAN_OFF_SEQ_NSEG] + i] : max_nseg;
#define GDR_CASE(TT, KK, VV)                                                                                       \
  return gdr_chunk_launch<TT, KK, VV>(q, k, v, g, beta, o, h0, ht, pv, n_seq, chunks, segs, max_nseg, gdr_max_chunks(plan_host), H, HV, scale, \
                                      l2norm, ws, s)
  if (dtype == GDR_BF16) {
    if (K == 32 && V == 32) GDR_CASE(__bf16, 32, 32);
    if (K == 64 && V == 64) GDR_CASE(__bf16, 64, 64);
    if (K == 64 && V == 128) GDR_CASE(__bf16, 64, 128);
    if (K == 128 && V == 64) GDR_CASE(__bf16, 128, 64);
    if (K == 128 && V == 128) GDR_CASE(__bf16, 128, 128);
  } else {
    if (K == 32 && V == 32) GDR_CASE(_Float16, 32, 32);
    if (K == 64 && V == 64) GDR_CASE(_Float16, 64, 64);
    if (K == 64 && V == 128) GDR_CASE(_Float16, 64, 128);
    if (K == 128 && V == 64) GDR_CASE(_Float16, 128, 64);
    if (K == 128 && V == 128) GDR_CASE(_Float16, 128, 128);
  }
#undef GDR_CASE
  return LAMPA_ERR_UNSUPPORTED;
}

// ---- training form: the same forward, keeping what the backward pass needs (gdr_train.h) --------------------------------
GdrSaved gdr_saved_layout(int64_t chunks, int64_t segs, int HV) {
  GdrSaved v;
  int64_t off = 0;
  v.off_rec = off;    off += lampa_align_up(chunks * HV * (int64_t)REC_BYTES, 256);
  v.off_states = off; off += lampa_align_up(chunks * HV * (int64_t)GDR_STATE_BYTES, 256);
  v.off_mt = off;     off += lampa_align_up(segs * HV * (int64_t)GDR_STATE_BYTES, 256);
  v.off_d = off;      off += lampa_align_up(segs * HV * 4, 256);
  v.off_e = off;      off += lampa_align_up(chunks * HV * 4, 256);
  v.bytes = off > 0 ? off : 256;
  return v;
}

extern "C" int64_t lampa_gdr_train_saved_bytes(const int32_t* plan_host, int HV) {
  if (!plan_host || HV < 1) return LAMPA_ERR_INVALID;
  return gdr_saved_layout(plan_host[PLAN_TOTAL_CHUNKS], plan_host[PLAN_N_SEGMENTS], HV).bytes;
}
extern "C" int64_t lampa_gdr_train_workspace_bytes(const int32_t* plan_host, int HV) {
  if (!plan_host || HV < 1) return LAMPA_ERR_INVALID;
  return gdr_workspace(plan_host[PLAN_TOTAL_CHUNKS], plan_host[PLAN_N_SEGMENTS], HV, 64, 64, true).bytes;
}

// As lampa_gdr_chunk_fwd for q, k, v of 64 columns; the rows of o are V <= 64 columns, a multiple of 8 (K, V: the heads before
// they were padded to 64). saved: lampa_gdr_train_saved_bytes bytes for lampa_gdr_bwd_saved. positive_g_host
// (nullable): pinned host memory, zeroed by the caller; becomes 1 when an entry of g is positive.
extern "C" int lampa_gdr_chunk_fwd_train(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                         void* o, const float* h0, float* ht, const int32_t* plan_host,
                                         const int32_t* plan_dev, int H, int HV, int K, int V, int dtype, float scale,
                                         int l2norm, void* saved, int32_t* positive_g_host, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  if (!q || !k || !v || !g || !beta || !o || !plan_host || !plan_dev || !saved) return LAMPA_ERR_INVALID;
  if (H < 1 || HV < H || HV % H != 0 || l2norm < 0 || l2norm > 2) return LAMPA_ERR_INVALID;
  if (!gdr_train_width(K) || !gdr_train_width(V) || (dtype != GDR_BF16 && dtype != GDR_FP16)) return LAMPA_ERR_UNSUPPORTED;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o | (uintptr_t)saved) & 15) return LAMPA_ERR_INVALID;
  const int n_seq = plan_host[PLAN_N_SEQ], chunks = plan_host[PLAN_TOTAL_CHUNKS], segs = plan_host[PLAN_N_SEGMENTS];
  if (n_seq < 1 || segs < n_seq) return LAMPA_ERR_INVALID;
  if (!workspace || workspace_bytes < lampa_gdr_train_workspace_bytes(plan_host, HV)) return LAMPA_ERR_WORKSPACE;
  const GdrPlanView pv = gdr_plan_view(plan_host, plan_dev);
  int max_nseg = 0;
  for (int i = 0; i < n_seq; ++i) max_nseg = plan_host[plan_host[PLAN_OFF_SEQ_NSEG] + i] > max_nseg ? plan_host[plan_host[PLAN_OFF_SEQ_NSEG] + i] : max_nseg;
  const GdrSaved sv = gdr_saved_layout(chunks, segs, HV);
  unsigned char* sp = (unsigned char*)saved;
  GdrKeep kp{sp + sv.off_rec, sp + sv.off_states, sp + sv.off_mt, (float*)(sp + sv.off_d), (float*)(sp + sv.off_e), nullptr, V};
  if (positive_g_host && hipHostGetDevicePointer((void**)&kp.positive_g, positive_g_host, 0) != hipSuccess) {
    (void)hipGetLastError();
    return LAMPA_ERR_INVALID;
  }
  if (dtype == GDR_BF16)
    return gdr_chunk_launch<__bf16, 64, 64, true>(q, k, v, g, beta, o, h0, ht, pv, n_seq, chunks, segs, max_nseg, gdr_max_chunks(plan_host), H, HV, scale,
                                                  l2norm, (unsigned char*)workspace, (hipStream_t)stream, kp);
  return gdr_chunk_launch<_Float16, 64, 64, true>(q, k, v, g, beta, o, h0, ht, pv, n_seq, chunks, segs, max_nseg, gdr_max_chunks(plan_host), H, HV, scale,
                                                  l2norm, (unsigned char*)workspace, (hipStream_t)stream, kp);
}
