// WKV7 slot-mapped inference over several steps with a bf16 state: the prompts
// of a serving loop (T > 1), on few enough (row, head) pairs that each can
// have a compute unit.
//
// Semantics as in wkv7_infer.hip's bf16 kernel (wkv7_infer/kernel.rs:15-114 at
// F = bf16): every product and sum rounded to bf16 in the reference's order,
// the sums over the key index left to right, masked steps skipped. The results
// are the same bit for bit.
//
// What bounds it is latency. Rows of the state are independent, but a row's
// step is a chain: 64 rounded additions for the removal state, the update, and
// 64 more for the output. That kernel's one wave per pair also issues the
// update of all 64 keys, about 1,024 instructions a step, and a wave alone on
// its SIMD issues one every 6-8 cycles: 2.69 us a step. Here the step of a
// pair's rows is shared by the waves of a workgroup:
//   wave 0 (lane = row)  the removal-state sum: 64 links of two instructions,
//                        "round the running sum" and "add the next rounded
//                        product" (a bf16 value in the high half of a register
//                        is its own fp32 value, so the packed conversion of
//                        (0, z) is rb(z));
//   wave 1 (lane = row)  the output sum, two steps behind, beside it;
//   update waves         a lane has one row and eight keys: the state, its
//                        update, the rounded products that the sums read;
//   last wave (lane = key)  the unmasked steps in order: decay, dither, widening.
// Two barriers a step: after the sum (the update needs it) and after the
// update's products (the next sum needs them). What does not depend on the
// sum, S w and k v and the output's products, is formed beside it.
// The update's instructions, beside the sums', then bound it, so where CUs are
// free a pair's rows go to two workgroups (kSplit).
//
// Measured per step, 36 pairs, T = 256: 2.65 us on the one-wave kernel, 0.87
// here with 64 rows a workgroup, 0.68 with 32, 0.69 with 16 (not kept).
#include "wkv7_device.hpp"
#include "wkv7_launch.hpp"

namespace wkv7 {
namespace {

constexpr int kKeys = 8;                             // of an update lane
constexpr int kRing = 8;                             // staged steps
constexpr int kLead = 3;                             // a step is staged this many steps ahead
constexpr int kLdp = kHead + 4;                      // padded product rows: 4 banks apart

struct PromptParams {
  const bf16_t *w, *r, *k, *v, *a, *b;
  const int32_t* batch_ids;
  bf16_t* state;
  const bf16_t* mask;
  const int32_t* elapsed_t;
  bf16_t* y;
  int T, H, full_batch, use_dither;
};

// one unmasked step's operands as fp32 values (w: the rounded decay)
struct Step {
  float w[kHead], a[kHead], b[kHead], k[kHead], r[kHead], v[kHead];
};

template <int kRows>
struct PromptLds {
  Step ring[kRing];
  int at[kRing];                      // the staged step's index t, -1 past the last one
  float ap[kRows][kLdp];              // rounded S a, [row][key]
  float yp[2][kRows][kLdp];           // rounded S r
  float sa[kRows];
};

// x rounded to bf16, as an fp32 value: the packed conversion puts it in the
// high half over a zero
__device__ __forceinline__ float rbf(float x) {
  return __builtin_bit_cast(float, __builtin_convertvector(f32x2_t{0.0f, x}, bf16x2_t));
}

// the reference's rounded sum of 64 rounded products, left to right; returns
// rb of it
__device__ __forceinline__ float rounded_sum(const float* p) {
  float4 x[kHead / 4];
#pragma unroll
  for (int i = 0; i < kHead / 4; ++i) x[i] = reinterpret_cast<const float4*>(p)[i];
  float z = 0.0f;
#pragma unroll
  for (int i = 0; i < kHead / 4; ++i) {
    z = rbf(z) + x[i].x;
    z = rbf(z) + x[i].y;
    z = rbf(z) + x[i].z;
    z = rbf(z) + x[i].w;
  }
  return rbf(z);
}

__device__ __forceinline__ void load8(const float* p, float (&x)[kKeys]) {
  const float4 lo = reinterpret_cast<const float4*>(p)[0], hi = reinterpret_cast<const float4*>(p)[1];
  x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w;
  x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
}
__device__ __forceinline__ void store8(float* p, const float (&x)[kKeys]) {
  reinterpret_cast<float4*>(p)[0] = make_float4(x[0], x[1], x[2], x[3]);
  reinterpret_cast<float4*>(p)[1] = make_float4(x[4], x[5], x[6], x[7]);
}

// Grid (H, rows of the batch, kSplit): workgroup z takes the state's value
// rows z kRows .. of its pair. An update wave's lanes hold kRows rows times
// kSplit groups of eight keys.
constexpr int prompt_waves(int split) { return 3 + kHead / (kKeys * split); }
template <int kSplit>
__global__ __launch_bounds__(64 * prompt_waves(kSplit)) void wkv7_infer_bf16_prompt_kernel(const PromptParams p) {
  constexpr int kRows = kHead / kSplit, kWaves = prompt_waves(kSplit);
  __shared__ PromptLds<kRows> L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane % kRows, j0 = kRows * blockIdx.z;
  const int h = blockIdx.x, bi = blockIdx.y, T = p.T;
  const int64_t tstride = (int64_t)p.H * kHead;
  const int64_t tok0 = ((int64_t)bi * T * p.H + h) * kHead;
  const int64_t slot = p.batch_ids[bi];
  // an out-of-range slot is refused: zero output, no state touched
  if (slot < 0 || slot >= p.full_batch) {
    for (int t = wave; t < T; t += kWaves) p.y[tok0 + (int64_t)t * tstride + j0 + row] = 0;
    return;
  }
  bf16_t* const st = p.state + (slot * p.H + h) * (kHead * kHead);

  // Each role runs its own loop over the steps (a shared loop with the roles
  // as branches made the sums wait for the other roles' memory accesses where
  // the branches join: 1.19 against 1.02 us a step). All of them pass the same
  // barriers: two before the first step, two a step, one after the last.
  auto step_at = [&](int e) { return L.at[e % kRing]; };

  if (wave == kWaves - 1) {
    // ------------------------------------------------------------- operands
    // `live`: the mask of the 64 steps from `base` on, without those already
    // handed out
    uint64_t live = 0;
    int64_t base = -64;
    auto next_live = [&]() -> int {
      while (live == 0) {
        base += 64;
        if (base >= T) return -1;
        const bool in = base + lane < T;
        const bool on = in && (!p.mask || (p.mask[(int64_t)bi * T + base + lane] & 0x7fffu) != 0u);
        live = __ballot(on);
        uint64_t dead = __ballot(in && !on);   // masked steps: y = 0
        while (dead) {
          p.y[tok0 + (base + __builtin_ctzll(dead)) * tstride + j0 + row] = 0;
          dead &= dead - 1;
        }
      }
      const int t = (int)base + __builtin_ctzll(live);
      live &= live - 1;
      return t;
    };
    struct Raw { bf16_t w, a, b, k, r, v; };
    auto fetch = [&](int t) {
      const int64_t off = tok0 + (int64_t)max(t, 0) * tstride + lane;
      return Raw{p.w[off], p.a[off], p.b[off], p.k[off], p.r[off], p.v[off]};
    };
    uint32_t seed = p.elapsed_t ? (uint32_t)p.elapsed_t[slot] : 0u;   // + unmasked steps so far
    auto stage = [&](int e, int t, const Raw& x) {
      Step& s = L.ring[e % kRing];
      float wd = decay_f(sigmoid_f(bf16_to_f32(x.w)));
      if (p.use_dither) wd += dither_f(seed);
      ++seed;
      s.w[lane] = rbf(wd);
      s.a[lane] = bf16_to_f32(x.a);
      s.b[lane] = bf16_to_f32(x.b);
      s.k[lane] = bf16_to_f32(x.k);
      s.r[lane] = bf16_to_f32(x.r);
      s.v[lane] = bf16_to_f32(x.v);
      if (lane == 0) L.at[e % kRing] = t;
    };
    for (int e = 0; e < kLead; ++e) {
      const int t = next_live();
      stage(e, t, fetch(t));
    }
    int tn = next_live();
    Raw xn = fetch(tn);
    lds_barrier();
    lds_barrier();
    int t = __builtin_amdgcn_readfirstlane(step_at(0));
    for (int e = 0; t >= 0; ++e) {
      const int t1 = step_at(e + 1);
      stage(e + kLead, tn, xn);
      tn = tn < 0 ? -1 : next_live();
      xn = fetch(tn);
      lds_barrier();
      t = __builtin_amdgcn_readfirstlane(t1);
      lds_barrier();
    }
    lds_barrier();
  } else if (wave == 0) {
    // ----------------------------------------------------- removal-state sum
    __builtin_amdgcn_s_setprio(3);   // the sums are the step's critical path
    lds_barrier();
    lds_barrier();
    int t = __builtin_amdgcn_readfirstlane(step_at(0));
    for (int e = 0; t >= 0; ++e) {
      const int t1 = step_at(e + 1);
      L.sa[row] = rounded_sum(L.ap[row]);
      lds_barrier();
      t = __builtin_amdgcn_readfirstlane(t1);
      lds_barrier();
    }
    lds_barrier();
  } else if (wave == 1) {
    // ------------------------------------------- output sum, two steps behind
    __builtin_amdgcn_s_setprio(3);
    auto output = [&](int e, int t) {
      p.y[tok0 + (int64_t)t * tstride + j0 + row] = (bf16_t)(__float_as_uint(rounded_sum(L.yp[e & 1][row])) >> 16);
    };
    lds_barrier();
    lds_barrier();
    int e = 0, t = __builtin_amdgcn_readfirstlane(step_at(0)), ta = -1, tb = -1;   // ta, tb: the two before t
    for (; t >= 0; ++e) {
      const int t1 = step_at(e + 1);
      if (e >= 2) output(e - 2, tb);
      lds_barrier();
      tb = ta;
      ta = t;
      t = __builtin_amdgcn_readfirstlane(t1);
      lds_barrier();
    }
    if (e >= 2) output(e - 2, tb);
    lds_barrier();
    if (e >= 1) output(e - 1, ta);
  } else {
    // ------------------------------- update: keys k0 .. k0 + 7 of the lane's row
    const int k0 = kKeys * ((wave - 2) * kSplit + lane / kRows);
    float S[kKeys];
    bf16_t* const mine = st + (j0 + row) * kHead + k0;
    {
      const uint4 x = *reinterpret_cast<const uint4*>(mine);
      const uint32_t u[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        S[2 * i] = __uint_as_float(u[i] << 16);
        S[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
      }
    }
    auto products = [&](const float (&x)[kKeys], float* to) {
      float o[kKeys];
#pragma unroll
      for (int i = 0; i < kKeys; ++i) o[i] = rbf(S[i] * x[i]);
      store8(to, o);
    };
    // a step's operands: a is the next step's
    struct Ops { float w[kKeys], k[kKeys], b[kKeys], r[kKeys], a[kKeys], v; };
    auto load = [&](int e, Ops& o) {
      const Step& s = L.ring[e % kRing];
      load8(s.w + k0, o.w);
      load8(s.k + k0, o.k);
      load8(s.b + k0, o.b);
      load8(s.r + k0, o.r);
      load8(L.ring[(e + 1) % kRing].a + k0, o.a);
      o.v = s.v[j0 + row];
    };
    float* const ap = &L.ap[row][k0];
    int t;
    // step e with its operands x; y holds the step before's, and then the next's
    auto step = [&](int e, Ops& x, Ops& y) {
      const int t1 = step_at(e + 1);
      // beside the removal-state sum: what does not need it
      float sw[kKeys], kv[kKeys];
#pragma unroll
      for (int i = 0; i < kKeys; ++i) {
        sw[i] = rbf(S[i] * x.w[i]);
        kv[i] = rbf(x.k[i] * x.v);
      }
      if (e > 0) products(y.r, &L.yp[(e - 1) & 1][row][k0]);
      load(e + 1, y);
      lds_barrier();
      // S = rb(rb(rb(S w) + rb(sa b)) + rb(k v)), and the next step's products
      const float sa = L.sa[row];
#pragma unroll
      for (int i = 0; i < kKeys; ++i) S[i] = rbf(rbf(sw[i] + rbf(sa * x.b[i])) + kv[i]);
      products(x.a, ap);
      t = __builtin_amdgcn_readfirstlane(t1);
      lds_barrier();
    };
    Ops x, y;
    lds_barrier();
    load8(L.ring[0].a + k0, x.a);
    products(x.a, ap);
    load(0, x);
    lds_barrier();
    t = __builtin_amdgcn_readfirstlane(step_at(0));
    int e = 0;
    while (t >= 0) {   // two steps an iteration, so that x and y need no moves
      step(e++, x, y);
      if (t < 0) break;
      step(e++, y, x);
    }
    if (e > 0) {
      products((e & 1) ? x.r : y.r, &L.yp[(e - 1) & 1][row][k0]);
      uint32_t u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        u[i] = (__float_as_uint(S[2 * i]) >> 16) | (__float_as_uint(S[2 * i + 1]) & 0xffff0000u);
      *reinterpret_cast<uint4*>(mine) = make_uint4(u[0], u[1], u[2], u[3]);
    }
    lds_barrier();
  }
}

}  // namespace

// A CU's registers hold one workgroup, so past 256 pairs they queue. us, the
// one-wave kernel and this one:
//          T = 1       T = 2       T = 4        T = 5        T = 8        T = 16       T = 256
//   12     5.4 / 5.1   8.0 / 5.8   13.3 / 7.0   16.1 / 7.7   24.0 / 9.6   45.1 / 15.0  679 / 173
//   256    5.7 / 5.9   8.4 / 6.7   13.6 / 8.5   16.6 / 9.5   24.5 / 11.9  45.4 / 19.2  684 / 229
//   288    5.8 / 9.2   8.6 / 10.9  14.1 / 14.4  16.9 / 16.4  25.1 / 21.3  47.2 / 35.0  701 / 446
//   512    6.1 / 9.7   9.0 / 11.5  14.4 / 14.8  17.4 / 16.7  25.5 / 21.8  47.7 / 35.8  701 / 451
//   576    6.2 / 13.0  9.1 / 15.9  14.4 / 21.0  17.3 / 23.6  25.4 / 31.1  47.5 / 51.9  701 / 668
// (pairs to the left). One step, where at most 6% are to be had and only up to
// 128 pairs, stays on the one-wave kernel.
bool infer_prompt_preferred(const InferDesc& d) {
  const int64_t pairs = (int64_t)d.Ba * d.H;
  return d.state_dtype == Dtype::BF16 && (d.T > 4 ? pairs <= 512 : d.T > 1 && pairs <= 256);
}

hipError_t launch_infer_prompt(const InferDesc& d, hipStream_t stream) {
  PromptParams p;
  p.w = static_cast<const bf16_t*>(d.w);
  p.r = static_cast<const bf16_t*>(d.r);
  p.k = static_cast<const bf16_t*>(d.k);
  p.v = static_cast<const bf16_t*>(d.v);
  p.a = static_cast<const bf16_t*>(d.a);
  p.b = static_cast<const bf16_t*>(d.b);
  p.batch_ids = d.batch_ids;
  p.state = static_cast<bf16_t*>(d.state);
  p.mask = static_cast<const bf16_t*>(d.context_mask);
  p.elapsed_t = d.elapsed_t;
  p.y = static_cast<bf16_t*>(d.y);
  p.T = d.T;
  p.H = d.H;
  p.full_batch = d.full_batch;
  p.use_dither = d.use_dither;
  // half the rows a workgroup while every one still has a CU (T = 256: 177
  // against 228 us at 128 pairs, 275 against 239 at 256)
  if ((int64_t)d.Ba * d.H <= 128)
    hipLaunchKernelGGL(wkv7_infer_bf16_prompt_kernel<2>, dim3(d.H, d.Ba, 2), dim3(64 * prompt_waves(2)), 0, stream, p);
  else
    hipLaunchKernelGGL(wkv7_infer_bf16_prompt_kernel<1>, dim3(d.H, d.Ba, 1), dim3(64 * prompt_waves(1)), 0, stream, p);
  return hipGetLastError();
}

}  // namespace wkv7
