// What the training form of the chunk forward keeps for the backward pass (K = V = 64): the records of the chunks, the
// state in front of every chunk (16-bit operand fragments of the two 32-column slabs) and every segment's transposed M'
// (16-bit A-operand fragments) and decay, and the chunks' edges (GDR_EDGE_*; written where a segment has GDR_EDGE_NC chunks).
#pragma once
#include "common.h"
#include "gdr_plan.h"

#define GDR_STATE_BYTES 8192  // 64 x 64 elements of 2 bytes (and one 64 x 32 slab in fp32)

// widths of the rows that o and the gradients of padded heads can have
static inline bool gdr_train_width(int n) { return n >= 8 && n <= 64 && n % 8 == 0; }

struct GdrSaved {
  int64_t off_rec, off_states, off_mt, off_d, off_e, bytes;
};
GdrSaved gdr_saved_layout(int64_t chunks, int64_t segs, int HV);

extern "C" {
int64_t lampa_gdr_train_saved_bytes(const int32_t* plan_host, int HV);
int64_t lampa_gdr_train_workspace_bytes(const int32_t* plan_host, int HV);
int lampa_gdr_chunk_fwd_train(const void* q, const void* k, const void* v, const float* g, const float* beta, void* o,
                              const float* h0, float* ht, const int32_t* plan_host, const int32_t* plan_dev, int H, int HV,
                              int K, int V, int dtype, float scale, int l2norm, void* saved, int32_t* positive_g_host,
                              void* workspace, int64_t workspace_bytes, void* stream);
int64_t lampa_gdr_plan_size(const int64_t* cu_seqlens_host, int n_seq, int chunks_per_segment);
int lampa_gdr_plan_fill(const int64_t* cu_seqlens_host, int n_seq, int chunks_per_segment, int32_t* plan_host);
}
