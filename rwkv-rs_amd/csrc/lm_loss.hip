// The language model's loss: cross entropy of the next-token logits with
// l2wrap's gradient term (examples/rwkv-lm/src/model.rs:158-169,
// kernels/l2wrap/mod.rs:38-66), one forward and one backward pass over the
// logits instead of a cast to fp32, a softmax, its backward, a cast back and
// l2wrap's max / clone / scatter.
//
// A row is walked in pieces of 8 logits (one 16-byte access for bf16, two for
// fp32). Rows of a vocabulary that is no multiple of 8 begin anywhere, so the
// pieces begin at the row's first 16-byte boundary, and the few logits before
// it and after the last whole piece go one to a thread (RowSpan). Forward: a
// block per row; each thread keeps a running maximum m, the sum s of exp(x - m)
// rescaled whenever m grows, and the first index of m. The threads' triples
// are combined by wave shuffles and then across the waves in a fixed order, so
// a row's result does not depend on scheduling. The backward recomputes
// exp(x - lse) from the saved log-sum-exp and writes each gradient once; a
// row's pieces are independent there, so with few rows several blocks share
// one.
//
// HBM bounds it once the rows fill the chip: 8192 x 65536 bf16, forward 187 us
// (5.7 TB/s), backward 420 us (5.1). With the logits of a ragged row taken one
// by one instead of in pieces, 8192 x 65529 took 545 + 1,271 us in bf16 and 898
// + 2,070 in fp32; in pieces 189 + 450 and 361 + 916 (its rows' edges share
// cache lines with their neighbours').
#include <algorithm>
#include <climits>
#include <cmath>

#include "lm_loss_launch.hpp"

namespace rwkv_loss {
namespace {

struct Piece {
  float v[kPiece];
};

template <bool BF>
__device__ __forceinline__ Piece load_piece(const void* base, int64_t i) {
  Piece p;
  if constexpr (BF) {
    const uint4 raw = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + i);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      p.v[2 * k] = __builtin_bit_cast(float, w[k] << 16);
      p.v[2 * k + 1] = __builtin_bit_cast(float, w[k] & 0xffff0000u);
    }
  } else {
    const float4* f = reinterpret_cast<const float4*>(static_cast<const float*>(base) + i);
    const float4 a = f[0], b = f[1];
    p.v[0] = a.x; p.v[1] = a.y; p.v[2] = a.z; p.v[3] = a.w;
    p.v[4] = b.x; p.v[5] = b.y; p.v[6] = b.z; p.v[7] = b.w;
  }
  return p;
}

template <bool BF>
__device__ __forceinline__ void store_piece(void* base, int64_t i, const Piece& p) {
  if constexpr (BF) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w[k] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<__bf16>(p.v[2 * k]))) |
             (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<__bf16>(p.v[2 * k + 1])))
              << 16);
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(base) + i) = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    float4* f = reinterpret_cast<float4*>(static_cast<float*>(base) + i);
    f[0] = make_float4(p.v[0], p.v[1], p.v[2], p.v[3]);
    f[1] = make_float4(p.v[4], p.v[5], p.v[6], p.v[7]);
  }
}

template <bool BF>
__device__ __forceinline__ float load_one(const void* base, int64_t i) {
  if constexpr (BF) return __builtin_bit_cast(float, static_cast<uint32_t>(static_cast<const uint16_t*>(base)[i]) << 16);
  else return static_cast<const float*>(base)[i];
}

template <bool BF>
__device__ __forceinline__ void store_one(void* base, int64_t i, float v) {
  if constexpr (BF) static_cast<uint16_t*>(base)[i] = __builtin_bit_cast(uint16_t, static_cast<__bf16>(v));
  else static_cast<float*>(base)[i] = v;
}

// Elements [0, head) and [tail, V) of a row are taken one by one, the pieces
// between them start on a 16-byte boundary. head and V - tail are below kPiece.
struct RowSpan {
  int64_t pieces, tail;
  int head;
};
// kWhole: every row is whole pieces from a 16-byte boundary on.
template <bool BF, bool kWhole>
__device__ __forceinline__ RowSpan row_span(const void* base, int64_t row0, int64_t V) {
  if constexpr (kWhole) return {V / kPiece, V, 0};
  constexpr int kSize = BF ? 2 : 4;
  const uintptr_t at = reinterpret_cast<uintptr_t>(base) + row0 * kSize;
  const int head = static_cast<int>(min(static_cast<int64_t>((16 - (at & 15)) & 15) / kSize, V));
  const int64_t pieces = (V - head) / kPiece;
  return {pieces, head + pieces * kPiece, head};
}

// running (max, sum of exp(x - max), first index of max)
struct Run {
  float m, s;
  int idx;
};

__device__ __forceinline__ float scaled(float s, float m, float to) {
  return s == 0.f ? 0.f : s * __expf(m - to);
}

// b covers indices after a's when they come from one thread; across threads
// the smaller index wins a tie
__device__ __forceinline__ Run combine(const Run& a, const Run& b) {
  Run r;
  r.m = fmaxf(a.m, b.m);
  r.s = scaled(a.s, a.m, r.m) + scaled(b.s, b.m, r.m);
  r.idx = a.m > b.m ? a.idx : b.m > a.m ? b.idx : min(a.idx, b.idx);
  return r;
}

// How a row is walked: element by element, in pieces between a head and a tail,
// or in pieces alone (kWholePieces: it begins and ends on a 16-byte boundary).
enum { kElements, kPieces, kWholePieces };

template <bool BF, int kWidth, int kForm>
__global__ __launch_bounds__(kWidth) void xent_forward_kernel(XentArgs a) {
  __shared__ Run part[kWidth / 64];
  const int64_t row = blockIdx.x;
  const int64_t V = a.vocab, base = row * V;
  constexpr bool kWhole = kForm == kWholePieces;
  const RowSpan span = kForm == kElements ? RowSpan{0, V, 0} : row_span<BF, kWhole>(a.logits, base, V);
  const int tid = threadIdx.x;
  Run run{-INFINITY, 0.f, INT_MAX};
  // a logit of -inf adds nothing (and is no maximum), NaN makes the sum NaN
  auto single = [&](int64_t j) {
    const float x = load_one<BF>(a.logits, base + j);
    const Run one{x, x == -INFINITY ? 0.f : __expf(x - x), static_cast<int>(j)};
    const Run both = combine(run, one);
    run = {both.m, both.s, x > run.m ? one.idx : run.idx};
  };
  // each thread sees its logits by rising index: head, pieces, tail
  if (kForm == kElements)
    for (int64_t j = tid; j < V; j += kWidth) single(j);
  if (!kWhole && tid < span.head) single(tid);
  for (int64_t q = tid; q < span.pieces; q += kWidth) {
    const int64_t j0 = span.head + q * kPiece;
    const Piece p = load_piece<BF>(a.logits, base + j0);
    float cm = p.v[0];
    int ci = 0;
#pragma unroll
    for (int k = 1; k < kPiece; ++k)
      if (p.v[k] > cm) {
        cm = p.v[k];
        ci = k;
      }
    const float m = fmaxf(run.m, cm);
    const float to = m == -INFINITY ? 0.f : m;   // nothing but -inf so far: the exponentials are 0
    float s = scaled(run.s, run.m, m);
#pragma unroll
    for (int k = 0; k < kPiece; ++k) s += __expf(p.v[k] - to);
    if (cm > run.m) run.idx = static_cast<int>(j0) + ci;
    run.m = m;
    run.s = s;
  }
  if (!kWhole && span.tail + tid < V) single(span.tail + tid);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    Run o;
    o.m = __shfl_xor(run.m, off);
    o.s = __shfl_xor(run.s, off);
    o.idx = __shfl_xor(run.idx, off);
    run = combine(run, o);
  }
  if ((tid & 63) == 0) part[tid >> 6] = run;
  __syncthreads();
  if (tid == 0) {
    Run r = part[0];
#pragma unroll
    for (int w = 1; w < kWidth / 64; ++w) r = combine(r, part[w]);
    const float lse = r.m + logf(r.s);
    const int64_t t = a.targets[row];
    const float xt = t >= 0 && t < V ? load_one<BF>(a.logits, base + t) : NAN;
    a.row_loss[row] = lse - xt;
    a.row_lse[row] = lse;
    a.row_max[row] = r.m;
    a.row_argmax[row] = r.idx;
  }
}

// kPieces: the rows of the logits and of their gradient begin alike within 16
// bytes. kShared: blocks (row, y) take every gridDim.y-th run of kThreads pieces
// or elements.
template <bool BF, int kForm, bool kShared>
__global__ __launch_bounds__(kThreads) void xent_backward_kernel(XentArgs a) {
  const int64_t row = blockIdx.x;
  const int64_t V = a.vocab, base = row * V;
  const float lse = a.lse[row], g = a.row_grad[row];
  const float l2 = a.l2wrap_scale * a.max[row];
  const int64_t t = a.targets[row], am = a.argmax[row];
  const int64_t first = (kShared ? static_cast<int64_t>(blockIdx.y) * kThreads : 0) + threadIdx.x;
  const int64_t stride = kShared ? static_cast<int64_t>(gridDim.y) * kThreads : kThreads;
  auto grad = [&](float x, int64_t j) {
    float d = g * __expf(x - lse);
    if (j == t) d -= g;
    if (j == am) d += l2;
    return d;
  };
  auto single = [&](int64_t j) { store_one<BF>(a.logits_grad, base + j, grad(load_one<BF>(a.logits, base + j), j)); };
  if constexpr (kForm == kElements) {
    for (int64_t j = first; j < V; j += stride) single(j);
  } else {
    constexpr bool kWhole = kForm == kWholePieces;
    const RowSpan span = row_span<BF, kWhole>(a.logits, base, V);
    if (!kWhole && first < span.head) single(first);
    for (int64_t q = first; q < span.pieces; q += stride) {
      const int64_t j0 = span.head + q * kPiece;
      Piece p = load_piece<BF>(a.logits, base + j0);
#pragma unroll
      for (int k = 0; k < kPiece; ++k) p.v[k] = grad(p.v[k], j0 + k);
      store_piece<BF>(a.logits_grad, base + j0, p);
    }
    if (!kWhole && span.tail + first < V) single(span.tail + first);
  }
}

// A few long rows leave most of the chip idle and each is a chain of loads: four
// times the threads a row. us, 256 / 1024 threads, bf16: 65536 logits, 64 rows
// 11.9 / 9.1, 256 rows 12.5 / 9.6, 1024 rows 25.4 / 26.4; 32000 logits, 256 rows
// 7.6 / 6.9 (fp32 10.0 / 7.4). At 512 rows bf16 gains 0.7-3 and fp32 loses 1.6-2.
// The line is where every one of 1024 threads has at least three pieces, 24576:
// 1 row 6.6 / 6.2, 256 rows 7.3 / 7.2; at 16384 they were 5.4 / 5.6 and 6.1 / 6.5.
constexpr int64_t kWideRows = 256;
constexpr int kWideThreads = 1024;
constexpr int64_t kWideVocab = 3 * kWideThreads * kPiece;

// every row of x begins and ends on a 16-byte boundary
bool whole_pieces(const void* x, int64_t vocab) {
  return vocab % kPiece == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
}

// Short ragged rows go one by one: their heads and tails are a pass each. us, 8192
// rows, pieces / elements: fp32 97 logits forward 12.8 / 11.2, backward 6.1 / 4.0;
// 509 logits 12.7 / 12.9 and 8.6 / 8.9; bf16 13.0 / 13.0 and 6.9 / 6.1. Rows that
// are whole pieces walk them without looking for a head and a tail: 256 logits,
// bf16, backward 5.8 with, 4.3 without (1024 rows 2.5 / 2.3).
constexpr int64_t kShortVocab = 2 * kThreads;
int row_form(const void* x, int64_t vocab) {
  return whole_pieces(x, vocab) ? kWholePieces : vocab <= kShortVocab ? kElements : kPieces;
}

template <bool BF, int kWidth>
void forward(const XentArgs& a, hipStream_t s) {
  const int form = row_form(a.logits, a.vocab);
  auto* const kernel = form == kElements ? xent_forward_kernel<BF, kWidth, kElements>
                       : form == kPieces ? xent_forward_kernel<BF, kWidth, kPieces>
                                         : xent_forward_kernel<BF, kWidth, kWholePieces>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.rows)), dim3(kWidth), 0, s, a);
}

template <bool BF>
hipError_t forward(const XentArgs& a, hipStream_t s) {
  if (a.rows <= kWideRows && a.vocab >= kWideVocab) forward<BF, kWideThreads>(a, s);
  else forward<BF, kThreads>(a, s);
  return hipGetLastError();
}

// Blocks enough to fill the chip (eight of 256 threads a compute unit); a row has
// at most one for each run of pieces. us without / with, bf16, 65536 logits: 16
// rows 13.9 / 4.2, 64 rows 14.4 / 4.6, 256 rows 18.5 / 11.3, 1024 rows 46 / 44.
// fp32 rows, twice the bytes, fill it by themselves from 512 on: 8192 logits, 256
// rows 4.9 / 4.3, 768 rows 9.0 / 9.7, 65536 logits 22.0 / 21.6 and 83 / 86.
constexpr int64_t kFillBlocks = 2048;
constexpr int64_t kShareRowsF32 = 256;

template <bool BF, bool kShared>
hipError_t backward(const XentArgs& a, int form, unsigned split, hipStream_t s) {
  auto* const kernel = form == kElements ? xent_backward_kernel<BF, kElements, kShared>
                       : form == kPieces ? xent_backward_kernel<BF, kPieces, kShared>
                                         : xent_backward_kernel<BF, kWholePieces, kShared>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.rows), split), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

template <bool BF>
hipError_t backward(const XentArgs& a, hipStream_t s) {
  const bool alike = ((reinterpret_cast<uintptr_t>(a.logits) ^ reinterpret_cast<uintptr_t>(a.logits_grad)) & 15) == 0;
  const int form = alike ? row_form(a.logits, a.vocab) : kElements;
  const int64_t runs = (a.vocab / (form == kElements ? 1 : kPiece) + kThreads - 1) / kThreads;
  const int64_t fill = BF || a.rows <= kShareRowsF32 ? kFillBlocks / a.rows : 1;
  const int64_t split = std::max<int64_t>(1, std::min<int64_t>(fill, runs));
  if (split > 1) return backward<BF, true>(a, form, static_cast<unsigned>(split), s);
  return backward<BF, false>(a, form, 1, s);
}

}  // namespace

hipError_t launch_xent_forward(const XentArgs& a, hipStream_t s) {
  if (a.rows == 0) return hipSuccess;
  return a.bf16 ? forward<true>(a, s) : forward<false>(a, s);
}

hipError_t launch_xent_backward(const XentArgs& a, hipStream_t s) {
  if (a.rows == 0) return hipSuccess;
  return a.bf16 ? backward<true>(a, s) : backward<false>(a, s);
}

}  // namespace rwkv_loss
