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
#define HR_MAX_BLOCKS (1 << 20)  // blocks of a grid; of more rows than those take in one turn a block takes several spans
#define HR_MAX_ELEMENTS (INT64_C(1) << 40)  // far more than any memory holds: no tensor
#define HR_ROUNDS(bytes) ((bytes) == 16 ? 4 : (bytes) == 8 ? 8 : 16)  // pieces per thread

struct HrArgs {
  const void* src[HR_MAX];
  void* dst[HR_MAX];
  int64_t rows[HR_MAX];
  int ws[HR_MAX], wd[HR_MAX];  // row widths in pieces
};

// grid (blocks, tensors), 256 threads. A block takes as many rows of the destination as HR_ROUNDS rounds of its threads have
// pieces for; a thread goes from piece to piece 256 at a time. Pieces are as wide as every row of every tensor allows, 16 to 2
// bytes, and the narrower they are the more rounds there are: few bytes in flight bound them otherwise. Addresses are 32 bits
// from the block's first row on, loads come from clamped ones without a condition (which made each one a branch).
// 480 000 rows, us: torch's pad or slice / pieces of 16 or 2 bytes only, with conditions and four rounds / this:
//   48 -> 64 28 / 18 / 17    100 -> 128 52 / 66 / 34    33 -> 64 27 / 37 / 24    65 -> 128 42 / 66 / 38
//   128 -> 100 35 / 67 / 33  128 -> 65 29 / 47 / 31     64 -> 33 16 / 23 / 17    64 -> 20 14 / 16 / 14
template <typename P>
__global__ void __launch_bounds__(256) head_resize_kernel(const HrArgs a) {
  constexpr int ROUNDS = HR_ROUNDS(sizeof(P));
  const int t = blockIdx.y, ws = a.ws[t], wd = a.wd[t];
  const P* src = reinterpret_cast<const P*>(a.src[t]);
  P* dst = reinterpret_cast<P*>(a.dst[t]);
  const int64_t rows = a.rows[t];
  const int span = 256 * ROUNDS / wd, row_step = 256 / wd, col_step = 256 - row_step * wd;
  const int first_row = threadIdx.x / wd, first_col = threadIdx.x - first_row * wd;
  for (int64_t row0 = (int64_t)blockIdx.x * span; row0 < rows; row0 += (int64_t)gridDim.x * span) {
    const int left = rows - row0 < span ? (int)(rows - row0) : span;
    const P* from = src + row0 * ws;
    P* to = dst + row0 * wd;
    P x[ROUNDS];
    int row = first_row, col = first_col;
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
      x[i] = from[(uint32_t)(min(row, left - 1) * ws + min(col, ws - 1))];
      if (col >= ws) x[i] = P{};
      row += row_step;
      col += col_step;
      if (col >= wd) { col -= wd; ++row; }
    }
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
      const int at = threadIdx.x + 256 * i;
      if (at < left * wd) to[(uint32_t)at] = x[i];
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
  uintptr_t bits = 16;  // (of the sizes and addresses in bytes: the lowest one set is the widest piece)
  for (int i = 0; i < n; ++i) {
    const lampa_head_copy& c = copies[i];
    if (!c.src || !c.dst || c.rows < 0) return LAMPA_ERR_INVALID;
    if (c.src_width < 1 || c.dst_width < 1 || c.src_width > 256 || c.dst_width > 256) return LAMPA_ERR_UNSUPPORTED;
    if (c.rows > HR_MAX_ELEMENTS / (c.src_width > c.dst_width ? c.src_width : c.dst_width)) return LAMPA_ERR_UNSUPPORTED;
    if (((uintptr_t)c.src | (uintptr_t)c.dst) & 1) return LAMPA_ERR_INVALID;
    bits |= (uintptr_t)c.src | (uintptr_t)c.dst | 2 * (uintptr_t)(c.src_width | c.dst_width);
  }
  const int bytes = (int)(bits & (~bits + 1));
  int64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    a.src[i] = copies[i].src;
    a.dst[i] = copies[i].dst;
    a.rows[i] = copies[i].rows;
    a.ws[i] = 2 * copies[i].src_width / bytes;
    a.wd[i] = 2 * copies[i].dst_width / bytes;
    const int64_t per_block = 256 * HR_ROUNDS(bytes) / a.wd[i], b = (a.rows[i] + per_block - 1) / per_block;
    blocks = b > blocks ? b : blocks;
  }
  if (blocks == 0) return LAMPA_OK;
  if (blocks > HR_MAX_BLOCKS) blocks = HR_MAX_BLOCKS;
  const dim3 grid((unsigned)blocks, n);
#define HR_LAUNCH(P) hipLaunchKernelGGL(head_resize_kernel<P>, grid, dim3(256), 0, (hipStream_t)stream, a)
  if (bytes == 16) HR_LAUNCH(hr_u32x4);
  else if (bytes == 8) HR_LAUNCH(uint64_t);
  else if (bytes == 4) HR_LAUNCH(uint32_t);
  else HR_LAUNCH(uint16_t);
#undef HR_LAUNCH
  return lampa_launch_status();
}
