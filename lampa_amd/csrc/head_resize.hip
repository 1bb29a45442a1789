// Heads copied to another width: up to four [rows, width] tensors of 16-bit elements in one launch, cut on the right or
// filled up with zeros. Operands and gradients of heads that the chunk kernels are not built for pass through it (the
// reference's layer uses d_k = 16, d_v = 32, models/hattention/modeling_gated_deltaproduct.py:583-587 of
// chengjiang123/Lampa, and its kernels mask the columns instead).
//
// Bound by HBM writes (q, k, v of 90 000 rows 16 / 16 / 32 -> 64 wide: 12 MB read, 35 MB written) and by being launched at
// all: a torch pad is a fill and a copy per tensor, so one training step of 14 983 x 6 x 16 x 32 fp16 spent 59 of its 201 us
// of GPU time and most of its 317 us of host time on twelve such launches. Four of these take their place.
#include "common.h"

#define HR_MAX 4
#define HR_MAX_ELEMENTS (INT64_C(1) << 40)  // far more than any memory holds: no tensor
#define HR_ROWS 4  // rows per thread: their loads are in flight together

struct HrArgs {
  const void* src[HR_MAX];
  void* dst[HR_MAX];
  int64_t rows[HR_MAX];
  int ws[HR_MAX], wd[HR_MAX];  // row widths in pieces
};

// grid (blocks, tensors), 256 threads: thread = (row of the block's pass, piece of the destination row)
template <typename P>
__global__ void __launch_bounds__(256) head_resize_kernel(const HrArgs a) {
  const int t = blockIdx.y, ws = a.ws[t], wd = a.wd[t];
  const int per_pass = 256 / wd, r = threadIdx.x / wd, c = threadIdx.x - r * wd;
  if (r >= per_pass) return;
  const P* src = reinterpret_cast<const P*>(a.src[t]);
  P* dst = reinterpret_cast<P*>(a.dst[t]);
  const int64_t rows = a.rows[t];
  // (one round, but for tensors of more rows than a grid holds)
  for (int64_t first = (int64_t)blockIdx.x * (per_pass * HR_ROWS) + r; first < rows;
       first += (int64_t)gridDim.x * (per_pass * HR_ROWS)) {
    P x[HR_ROWS];
#pragma unroll
    for (int i = 0; i < HR_ROWS; ++i) {
      const int64_t row = first + (int64_t)i * per_pass;
      x[i] = P{};
      if (c < ws && row < rows) x[i] = src[row * ws + c];
    }
#pragma unroll
    for (int i = 0; i < HR_ROWS; ++i) {
      const int64_t row = first + (int64_t)i * per_pass;
      if (row < rows) dst[row * wd + c] = x[i];
    }
  }
}

typedef unsigned int hr_u32x4 __attribute__((ext_vector_type(4)));

struct lampa_head_copy {
  const void* src;
  void* dst;
  int64_t rows;
  int32_t src_width, dst_width;
};

// n <= 4 tensors of 16-bit elements, packed: src [rows, src_width] -> dst [rows, dst_width], columns beyond the source's
// width zero. Widths 1 .. 256; src and dst must not overlap.
extern "C" int lampa_head_resize(int n, const lampa_head_copy* copies, void* stream) {
  if (n < 1 || n > HR_MAX || !copies) return LAMPA_ERR_INVALID;
  HrArgs a;
  int piece = 8;  // elements: 16 bytes where every row of every tensor starts on 16, else one element
  for (int i = 0; i < n; ++i) {
    const lampa_head_copy& c = copies[i];
    if (!c.src || !c.dst || c.rows < 0) return LAMPA_ERR_INVALID;
    if (c.src_width < 1 || c.dst_width < 1 || c.src_width > 256 || c.dst_width > 256) return LAMPA_ERR_UNSUPPORTED;
    if (c.rows > HR_MAX_ELEMENTS / (c.src_width > c.dst_width ? c.src_width : c.dst_width)) return LAMPA_ERR_UNSUPPORTED;
    if (((uintptr_t)c.src | (uintptr_t)c.dst) & 1) return LAMPA_ERR_INVALID;
    if ((c.src_width | c.dst_width) % 8 || (((uintptr_t)c.src | (uintptr_t)c.dst) & 15)) piece = 1;
  }
  int64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    a.src[i] = copies[i].src;
    a.dst[i] = copies[i].dst;
    a.rows[i] = copies[i].rows;
    a.ws[i] = copies[i].src_width / piece;
    a.wd[i] = copies[i].dst_width / piece;
    const int64_t per_block = (int64_t)(256 / a.wd[i]) * HR_ROWS, b = (a.rows[i] + per_block - 1) / per_block;
    blocks = b > blocks ? b : blocks;
  }
  if (blocks == 0) return LAMPA_OK;
  if (blocks > INT32_MAX / 256) blocks = INT32_MAX / 256;  // (a grid holds fewer than 2^31 threads per dimension here)
  const dim3 grid((unsigned)blocks, n);
  if (piece == 8)
    hipLaunchKernelGGL(head_resize_kernel<hr_u32x4>, grid, dim3(256), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(head_resize_kernel<uint16_t>, grid, dim3(256), 0, (hipStream_t)stream, a);
  return lampa_launch_status();
}
