// One decode step of a cell (include/rwkv_decode.h) in nine launches.
//
// A step of a few sequences reads every weight once and does almost nothing
// with it, so it is bound by launches and by the latency of each: through the
// modules it took about 60 launches a cell (weight casts, products, token
// shift, element-wise ends), issued from Python, 0.73 ms a cell. Here:
//   norm + token shift + six mixes      one workgroup a row
//   receptance, key, value and the four LoRAs' first products   16 columns a
//   the LoRAs' second products + weight preparation's end       a head a
//   recurrence (wkv7_infer.hip), gated readout (neighbors.hip)
//   output product + residual
//   norm + token shift + mix, key product + relu^2, value product + residual
// The weights are read as they are stored, fp32, and rounded to bf16 in
// registers, so no bf16 copy of them is made or kept. At 12 cells, C = 768, 8
// sequences, vocabulary 65536, a step took 9,150 us through the modules and
// takes 835 so. Its kernels sum to 684 us, of which the head's 201 MB of
// weights are 49; the rest is each launch's own latency, 3-9 us. The host, which
// reads the modules' parameters and issues them, takes about as long.
#include "decode_launch.hpp"

#include "neighbors_device.hpp"
#include "neighbors_launch.hpp"
#include "wkv7_launch.hpp"

namespace rwkv_decode {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf(bf16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ bf16_t to_bf(float x) { return __builtin_bit_cast(bf16_t, (__bf16)x); }
__device__ __forceinline__ float rbf(float x) { return (float)(__bf16)x; }

// ------------------------------------------------- norm, token shift, mixes
struct NormArgs {
  const float *x, *weight, *bias;
  float eps;
  int rows, C;
  // mixes (NM > 0): out_i = h + (shift[slot] - h) * mix_i; the new shift is h
  const int32_t* batch_ids;
  const float* shift_in;
  float* shift_out;
  int full_batch;
  const float* mix[6];
  bf16_t* out[6];     // NM = 0: out[0] = h
};

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Blocks 0 .. rows - 1 take a row each; with a token shift, block rows + s
// copies slot s unless a row writes it. A thread holds kChannels channels, and
// loads all that they need before the first sum, so that the sums wait for one
// memory latency (at C = 768, six mixes / one: 5.2 / 5.7 us a launch with the
// row in LDS and the parameters loaded after the sums, 4.2 / 3.3 us so). Six
// mixes / one, us a launch with 4 channels a thread: C = 1024 4.2 / 3.4; with 8:
// 1088 4.9 / 3.6, 2048 5.0 / 3.8; with 32, most of a wave's registers and one
// wave a SIMD: 2112 7.5 / 4.9, 4096 8.5 / 5.7, beside 87 us of products a cell
// at 2112 and 194 at 4096.
template <int NM, int kChannels>
__global__ __launch_bounds__(256) void norm_mix_kernel(const NormArgs a) {
  __shared__ float red[4];
  const int C = a.C, tid = threadIdx.x;
  if (NM > 0 && (int)blockIdx.x >= a.rows) {
    const int s = blockIdx.x - a.rows;
    bool written = false;
    for (int b = 0; b < a.rows; ++b) written |= a.batch_ids[b] == s;
    if (!written)
      for (int c = tid; c < C; c += 256) a.shift_out[(int64_t)s * C + c] = a.shift_in[(int64_t)s * C + c];
    return;
  }
  const int row = blockIdx.x;
  int slot = -1;
  if (NM > 0) {
    const int id = a.batch_ids[row];
    if (id >= 0 && id < a.full_batch) slot = id;
  }
  float x[kChannels], w[kChannels], b[kChannels], prev[kChannels], mix[NM > 0 ? NM : 1][kChannels];
#pragma unroll
  for (int i = 0; i < kChannels; ++i) {
    const int c = min(tid + 256 * i, C - 1);   // past the end: the last channel, not counted or stored
    x[i] = a.x[(int64_t)row * C + c];
    w[i] = a.weight[c];
    b[i] = a.bias[c];
    if (NM > 0) prev[i] = a.shift_in[(int64_t)max(slot, 0) * C + c];
#pragma unroll
    for (int k = 0; k < NM; ++k) mix[k][i] = a.mix[k][c];
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kChannels; ++i) sum += tid + 256 * i < C ? x[i] : 0.f;
  const float mean = block_sum(sum, red) / C;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < kChannels; ++i) {
    const float d = x[i] - mean;
    sq += tid + 256 * i < C ? d * d : 0.f;
  }
  const float rstd = 1.f / sqrtf(block_sum(sq, red) / C + a.eps);
#pragma unroll
  for (int i = 0; i < kChannels; ++i) {
    const int c = tid + 256 * i;
    if (c >= C) break;
    const float v = (x[i] - mean) * rstd * w[i] + b[i];
    const int64_t at = (int64_t)row * C + c;
    if (NM == 0) {
      a.out[0][at] = to_bf(v);
    } else {
      const float d = (slot >= 0 ? prev[i] : 0.f) - v;
#pragma unroll
      for (int k = 0; k < NM; ++k) a.out[k][at] = to_bf(v + d * mix[k][i]);
      if (slot >= 0) a.shift_out[(int64_t)slot * C + c] = v;
    }
  }
}

template <int NM>
hipError_t norm_mix(const NormArgs& a, hipStream_t s) {
  const dim3 grid(NM > 0 ? a.rows + a.full_batch : a.rows), block(256);
  if (a.C <= 1024) hipLaunchKernelGGL((norm_mix_kernel<NM, 4>), grid, block, 0, s, a);
  else if (a.C <= 2048) hipLaunchKernelGGL((norm_mix_kernel<NM, 8>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((norm_mix_kernel<NM, RWKV_DECODE_MAX_DIM / 256>), grid, block, 0, s, a);
  return hipGetLastError();
}

// ------------------------------------------------------------- row products
// out [rows, N] = act(x [rows, K] W), W as [N, K] (a linear layer's) or [K, N]
// (a LoRA factor's), rounded to bf16 as it is read.
enum Act { kNone, kTanh, kSigmoid, kSquaredRelu, kResidual };
struct Job {
  const float* w;
  const bf16_t* x;
  void* out;          // bf16, or (kResidual) the fp32 rows the result is added to
  int K, N;
  int tile0;          // first 16-column tile of this job in the launch
  int act;
  bool in_out;        // W is [K, N]
};
constexpr int kMaxJobs = 7;
struct GemmArgs {
  Job job[kMaxJobs];
  int jobs, rows;
};

// eight weights of column n at k .. k + 7, one load step of an MFMA's B operand
__device__ __forceinline__ bf16x8 weights8(const Job& j, int n, int k) {
  f32x8 w;
  if (j.in_out) {
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = j.w[(int64_t)(k + e) * j.N + n];
  } else {
    const f32x4* const q = reinterpret_cast<const f32x4*>(j.w + (int64_t)n * j.K + k);
    const f32x4 lo = __builtin_nontemporal_load(q), hi = __builtin_nontemporal_load(q + 1);
    w = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  return __builtin_convertvector(w, bf16x8);
}

// A workgroup forms 16 columns of up to 16 MT rows; its eight waves split the
// inner axis in steps of 32 (one MFMA a step and row tile) and add up through
// LDS in wave order. Wave w's loads are four steps deep, so a wave has up to
// 8 KB of weights in flight. v_mfma_f32_16x16x32_bf16: lane l holds A[row l %
// 16] and B[column l % 16] at k = 8 (l / 16) .. + 7, the result D[row 4 (l /
// 16) + r][column l % 16] (any order of k serves, the same for A and B).
constexpr int kGemmWaves = 8, kDepth = 4;
template <int MT>
__global__ __launch_bounds__(64 * kGemmWaves) void rows_gemm_kernel(const GemmArgs a) {
  __shared__ float part[kGemmWaves][MT * 256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int ji = 0;
  while (ji + 1 < a.jobs && (int)blockIdx.x >= a.job[ji + 1].tile0) ++ji;
  const Job& j = a.job[ji];
  const int n0 = 16 * (blockIdx.x - j.tile0);
  const int n = min(n0 + (lane & 15), j.N - 1), k0 = 8 * (lane >> 4);
  const int steps = j.K / 32;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = wave; s0 < steps; s0 += kGemmWaves * kDepth) {
    bf16x8 w[kDepth], x[kDepth][MT];
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      const int s = s0 + d * kGemmWaves;
      if (s < steps) {
        w[d] = weights8(j, n, 32 * s + k0);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int row = min(16 * m + (lane & 15), a.rows - 1);
          x[d][m] = *reinterpret_cast<const bf16x8*>(j.x + (int64_t)row * j.K + 32 * s + k0);
        }
      }
    }
#pragma unroll
    for (int d = 0; d < kDepth; ++d)
      if (s0 + d * kGemmWaves < steps) {
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[d][m], w[d], acc[m], 0, 0, 0);
      }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(&part[wave][m * 256 + 4 * lane]) = acc[m];
  __syncthreads();
  for (int i = threadIdx.x; i < MT * 256; i += 64 * kGemmWaves) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kGemmWaves; ++w) v += part[w][i];
    const int l = (i >> 2) & 63, row = 16 * (i >> 8) + 4 * (l >> 4) + (i & 3), col = n0 + (l & 15);
    if (row >= a.rows || col >= j.N) continue;
    const int64_t at = (int64_t)row * j.N + col;
    v = rbf(v);
    if (j.act == kResidual) {
      static_cast<float*>(j.out)[at] += v;
      continue;
    }
    if (j.act == kTanh) v = tanhf(v);
    else if (j.act == kSigmoid) v = rwkv_nb::sigmoid1(v);
    else if (j.act == kSquaredRelu) v = v > 0.f ? v * v : v == v ? 0.f : v;   // NaN stays
    static_cast<bf16_t*>(j.out)[at] = to_bf(v);
  }
}

// ------------------------------- LoRAs' second products, preparation's end
struct PrepareArgs {
  const bf16_t *key, *value;          // projections [rows, C]
  bf16_t* value_first;                // [rows, C]: written by the first cell, read by the others
  // hidden rows [rows, rank] and second factors [rank, C]: learning rate,
  // decay, gate, value residual (null in the first cell)
  const bf16_t* hid[4];
  const float* w[4];
  int rank[4];
  const float *rate_bias, *decay_bias, *residual_bias, *key_replacement, *key_removal;
  bf16_t *decay, *rkey, *val, *removal, *replacement, *gate;
  int rows, C;
};

// One workgroup of sixteen waves a head. Wave 4 i + q forms LoRA i's product
// for the head's channels 16 q .. (row tiles of 16) and leaves it in LDS; then
// the waves take the rows in turn, a lane a channel. (Four waves that formed
// the four products one after another waited for one after another's loads:
// 11.3 us a launch at C = 768, 5.8 us so.)
template <int MT, bool kFirst>
__global__ __launch_bounds__(1024) void lora_prepare_kernel(const PrepareArgs a) {
  __shared__ float y[4][16 * MT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int C = a.C;
  const int i = wave >> 2;
  if (i < (kFirst ? 3 : 4)) {
    const int t = lane & 15, qd = lane >> 4, n = 16 * (wave & 3) + t, c = 64 * blockIdx.x + n;
    const int rank = a.rank[i];
    const float* const w0 = a.w[i] + c;
    const bf16_t* const h0 = a.hid[i];
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 8 * qd; k < rank; k += 32) {
      f32x8 w;
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = w0[(int64_t)(k + e) * C];
      const bf16x8 wb = __builtin_convertvector(w, bf16x8);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = min(16 * m + t, a.rows - 1);
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(h0 + (int64_t)row * rank + k), wb, acc[m], 0, 0, 0);
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) y[i][16 * m + 4 * qd + r][n] = rbf(acc[m][r]);
  }
  const int c = 64 * blockIdx.x + lane;
  const float rate_b = a.rate_bias[c], decay_b = a.decay_bias[c], ka = a.key_replacement[c], kk = a.key_removal[c];
  const float residual_b = kFirst ? 0.f : a.residual_bias[c];
  __syncthreads();
  for (int row = wave; row < a.rows; row += 16) {
    const int64_t at = (int64_t)row * C + c;
    const float key = bf(a.key[at]), u = key * kk;
    float v = bf(a.value[at]);
    const float first = kFirst ? 0.f : bf(a.value_first[at]);
    float ss = u * u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float n = sqrtf(ss);
    const float un = u / (n >= rwkv_nb::kNormEps ? n : rwkv_nb::kNormEps);
    const float rate = rwkv_nb::sigmoid1(y[0][row][lane] + rate_b);
    if (kFirst)
      a.value_first[at] = a.value[at];
    else
      v += (first - v) * rwkv_nb::sigmoid1(y[3][row][lane] + residual_b);
    a.decay[at] = to_bf(-rwkv_nb::softplus1(-(y[1][row][lane] + decay_b)) - 0.5f);
    a.rkey[at] = to_bf(key * (ka * (rate - 1.f) + 1.f));
    a.val[at] = to_bf(v);
    a.removal[at] = to_bf(-un);
    a.replacement[at] = to_bf(un * rate);
    a.gate[at] = to_bf(y[2][row][lane]);
  }
}

hipError_t gemm(GemmArgs& a, hipStream_t s) {
  int tiles = 0;
  for (int i = 0; i < a.jobs; ++i) {
    a.job[i].tile0 = tiles;
    tiles += (a.job[i].N + 15) / 16;
  }
  const dim3 grid(tiles), block(64 * kGemmWaves);
  if (a.rows <= 16) hipLaunchKernelGGL(rows_gemm_kernel<1>, grid, block, 0, s, a);
  else if (a.rows <= 32) hipLaunchKernelGGL(rows_gemm_kernel<2>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(rows_gemm_kernel<4>, grid, block, 0, s, a);
  return hipGetLastError();
}

template <bool kFirst>
hipError_t prepare(const PrepareArgs& a, int H, hipStream_t s) {
  if (a.rows <= 16) hipLaunchKernelGGL((lora_prepare_kernel<1, kFirst>), dim3(H), dim3(1024), 0, s, a);
  else if (a.rows <= 32) hipLaunchKernelGGL((lora_prepare_kernel<2, kFirst>), dim3(H), dim3(1024), 0, s, a);
  else hipLaunchKernelGGL((lora_prepare_kernel<4, kFirst>), dim3(H), dim3(1024), 0, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_cell(const CellCall& c, hipStream_t stream) {
  const rwkv_decode_cell_params& p = *c.p;
  const int R = c.rows, C = c.H * 64;
  // the workspace: the first cell's value rows, nine rows of C reused through
  // the step, and 4 C that the LoRAs' hidden rows share
  bf16_t* const base = static_cast<bf16_t*>(c.workspace);
  auto buf = [&](int i) { return base + (int64_t)i * R * C; };
  bf16_t* const first = buf(0);
  bf16_t *const mix = buf(1), *const rec = buf(7), *const key = buf(8), *const val = buf(9), *const hid = buf(10);
  const bool is_first = p.residual_a == nullptr;

  NormArgs n{};
  n.x = c.x;
  n.weight = p.norm_time_weight;
  n.bias = p.norm_time_bias;
  n.eps = p.norm_time_eps;
  n.rows = R;
  n.C = C;
  n.batch_ids = c.batch_ids;
  n.shift_in = c.shift_time_in;
  n.shift_out = c.shift_time_out;
  n.full_batch = c.full_batch;
  for (int i = 0; i < 6; ++i) {
    n.mix[i] = p.mix[i];
    n.out[i] = mix + (int64_t)i * R * C;
  }
  hipError_t e = norm_mix<6>(n, stream);
  if (e != hipSuccess) return e;

  const int64_t RC = (int64_t)R * C;
  bf16_t* const h_rate = hid;
  bf16_t* const h_decay = h_rate + R * p.rate_rank;
  bf16_t* const h_gate = h_decay + R * p.decay_rank;
  bf16_t* const h_res = h_gate + R * p.gate_rank;
  GemmArgs g{};
  g.rows = R;
  auto add = [&](const float* w, const bf16_t* x, void* out, int64_t K, int64_t N, int act, bool in_out) {
    g.job[g.jobs++] = Job{w, x, out, (int)K, (int)N, 0, act, in_out};
  };
  add(p.receptance, mix, rec, C, C, kNone, false);
  add(p.key, mix + 2 * RC, key, C, C, kNone, false);
  add(p.value, mix + 3 * RC, val, C, C, kNone, false);
  add(p.rate_a, mix + 4 * RC, h_rate, C, p.rate_rank, kNone, true);
  add(p.decay_a, mix + RC, h_decay, C, p.decay_rank, kTanh, true);
  add(p.gate_a, mix + 5 * RC, h_gate, C, p.gate_rank, kSigmoid, true);
  if (!is_first) add(p.residual_a, mix + 3 * RC, h_res, C, p.residual_rank, kNone, true);
  if ((e = gemm(g, stream)) != hipSuccess) return e;

  // the mixes are used up: their rows take the recurrence's operands
  bf16_t *const decay = mix, *const rkey = mix + RC, *const v = mix + 2 * RC, *const removal = mix + 3 * RC,
         *const replacement = mix + 4 * RC, *const gate = mix + 5 * RC;
  PrepareArgs q{};
  q.key = key;
  q.value = val;
  q.value_first = first;
  const bf16_t* const hids[4] = {h_rate, h_decay, h_gate, h_res};
  const float* const ws[4] = {p.rate_b, p.decay_b, p.gate_b, p.residual_b};
  const int64_t ranks[4] = {p.rate_rank, p.decay_rank, p.gate_rank, is_first ? 0 : p.residual_rank};
  for (int i = 0; i < 4; ++i) {
    q.hid[i] = hids[i];
    q.w[i] = ws[i];
    q.rank[i] = (int)ranks[i];
  }
  q.rate_bias = p.rate_bias;
  q.decay_bias = p.decay_bias;
  q.residual_bias = p.residual_bias;
  q.key_replacement = p.key_replacement;
  q.key_removal = p.key_removal;
  q.decay = decay;
  q.rkey = rkey;
  q.val = v;
  q.removal = removal;
  q.replacement = replacement;
  q.gate = gate;
  q.rows = R;
  q.C = C;
  if ((e = is_first ? prepare<true>(q, c.H, stream) : prepare<false>(q, c.H, stream)) != hipSuccess) return e;

  bf16_t* const y = key;   // the projections are used up too
  wkv7::InferDesc d{};
  d.dtype = wkv7::Dtype::BF16;
  d.state_dtype = c.state_bf16 ? wkv7::Dtype::BF16 : wkv7::Dtype::F32;
  d.Ba = R;
  d.T = 1;
  d.H = c.H;
  d.full_batch = c.full_batch;
  d.w = decay;
  d.r = rec;
  d.k = rkey;
  d.v = v;
  d.a = removal;
  d.b = replacement;
  d.batch_ids = c.batch_ids;
  d.state = c.state;
  d.elapsed_t = c.elapsed_t;
  d.use_dither = c.use_dither;
  d.y = y;
  if ((e = wkv7::launch_infer(d, stream)) != hipSuccess) return e;

  bf16_t* const read = val;
  rwkv_nb::ReadoutArgs o{};
  o.y = y;
  o.r = rec;
  o.k = rkey;
  o.v = v;
  o.gate = gate;
  o.bonus = p.bonus;
  o.weight = p.group_norm_weight;
  o.bias = p.group_norm_bias;
  o.eps = p.group_norm_eps;
  o.rows = R;
  o.H = c.H;
  o.op_bf16 = o.act_bf16 = true;
  o.out = read;
  if ((e = rwkv_nb::launch_readout_forward(o, stream)) != hipSuccess) return e;

  g = GemmArgs{};
  g.rows = R;
  add(p.output, read, c.x, C, C, kResidual, false);
  if ((e = gemm(g, stream)) != hipSuccess) return e;

  // channel mixer
  n.weight = p.norm_channel_weight;
  n.bias = p.norm_channel_bias;
  n.eps = p.norm_channel_eps;
  n.shift_in = c.shift_channel_in;
  n.shift_out = c.shift_channel_out;
  n.mix[0] = p.channel_mix;
  n.out[0] = mix;
  if ((e = norm_mix<1>(n, stream)) != hipSuccess) return e;
  bf16_t* const hidden = mix + RC;   // [rows, 4 C]
  g = GemmArgs{};
  g.rows = R;
  add(p.channel_key, mix, hidden, C, 4 * (int64_t)C, kSquaredRelu, false);
  if ((e = gemm(g, stream)) != hipSuccess) return e;
  g = GemmArgs{};
  g.rows = R;
  add(p.channel_value, hidden, c.x, 4 * (int64_t)C, C, kResidual, false);
  return gemm(g, stream);
}

hipError_t launch_head(const HeadCall& c, hipStream_t stream) {
  const int C = c.H * 64;
  NormArgs n{};
  n.x = c.x;
  n.weight = c.norm_weight;
  n.bias = c.norm_bias;
  n.eps = c.eps;
  n.rows = c.rows;
  n.C = C;
  n.out[0] = static_cast<bf16_t*>(c.workspace);
  if (hipError_t e = norm_mix<0>(n, stream)) return e;
  GemmArgs g{};
  g.rows = c.rows;
  g.jobs = 1;
  g.job[0] = Job{c.unembed, n.out[0], c.logits, C, (int)c.vocab, 0, kNone, false};
  return gemm(g, stream);
}

}  // namespace rwkv_decode
