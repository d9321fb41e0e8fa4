// Sequences cut into segments that run side by side. The transition kernel
// here is for bf16 operands; the one with fp32 products is in
// wkv7_f32_chunk.hip, and the combine and poison kernels serve both.
//
// One workgroup per (batch, head) walks a whole sequence, so a call with few
// pairs leaves most of the chip idle for as long as one chain of chunks takes.
// The recurrence (wkv7_common/kernel.rs:51-103) is affine in the state: over
// a run of chunks
//   S_end = S_start M + N,
// with M (64 x 64) and N independent of S_start, and the state's gradient
// runs backwards the same way with M^T and another N. So the sequence is cut
// into segments and a call becomes three launches:
//   1. transition kernel (here): per (batch, head) and segment, M and N;
//   2. combine kernel (here): the segments' start states (or end gradients),
//      S_(g+1) = S_g M_g + N_g, fp32 products and sums;
//   3. the chunked forward / backward kernel on each segment as if it were a
//      sequence of its own.
//
// The transition kernel is the chunked forward's two-group pipeline (see
// wkv7_chunk_forward.hip) without its outputs: eight prep waves form each chunk's
// operands, chain waves carry two states per value tile, N's (which starts
// from the segment's known start state, or zero) and M's (which starts from
// the identity and sees no values), so the two dependency chains fill each
// other's latency. Forward, per chunk (notation of wkv7_chunk.hpp):
//   SA = W S^T + U,  W = P A^,  U = P A_ak V,
//   S <- (S + V^T K~ + SA^T B~) diag(gamma_L).
// Backward, with dS' = dS diag(gamma_L):
//   dSA = W dS'^T + U,  W = P^T B~,  U = P^T A_rb^T dY,
//   dS <- dS' + dY^T R^ + dSA^T A^,
// the same form with the roles of the rows exchanged and the decay applied
// first. Products are the chunked kernels' split-bf16 ones, so a segment's
// start state has the accuracy the sequential chain gives it (against float64
// at B=1, T=4096, H=32: final state 2.6e-6, removal_state 5.6e-6, initial-
// state gradient 2.6e-6, with and without segments).
//
// At B=1, T=4096, H=32 (8 segments of 32 chunks) forward + backward went from
// 1,100 to 305 us of kernel time: transition 46 + 48, combine 7 + 7, forward
// 347 -> 65, backward 743 -> 125. The transition kernel first had four prep
// waves, whose work (a wave alone on its half of a SIMD issues every 6-8
// cycles) the chain waves waited for 40% of the time: 53 us; with eight, two
// per chain wave and SIMD, 46 us, and the chain waits for its own products.
// Raising the chain waves' issue priority changed nothing.
#include <algorithm>
#include <type_traits>

#include "wkv7_chunk.hpp"
#include "wkv7_launch.hpp"

namespace wkv7 {
namespace {

using namespace chunk;

constexpr int kChainWaves = 4;            // value tile = wave
constexpr int kSlots = 4;                 // operand slots
constexpr int kPrepWaves = 8;
constexpr int kWaves = kChainWaves + kPrepWaves;
constexpr int kBlock = 64 * kWaves;
constexpr int kVecs = 5;
// x, a, b; then k and v (forward) or r and dy (backward)
enum { S_X, S_A, S_B, S_K, S_V };
constexpr int kPieces = kVecs * kL * 8 / 64;   // 16-byte loads per prep lane and chunk

// One chunk's operands, in the fragment order the chain loads (index [lane]
// last). f: the rows that meet the values (K~ or R^), g: those that meet SA
// (B~ or A^), both transposed and stacked hi | lo.
struct SegOps {
  bf16x8 w[2][2][64];     // W, x32 A operand: [key half][hi/lo]
  bf16x8 f[4][64];
  bf16x8 g[4][64];
  bf16x4 v[4][64];        // values, x16 B operand per value tile
  f32x4 u[4][64];         // U per value tile, result layout
  float gl[64];           // gamma_L
};
struct SegPrep {
  PadTile stg[kVecs];     // the chunk's raw rows; all but the values' tile are reused for the
                          // hi/lo rows of the decayed tensors
  float gl[64];
};
struct Flags {
  int ready[kSlots];
  int taken[kSlots][kChainWaves];
  int fault;
};

struct SegParams {
  const bf16_t* in[kVecs];
  const float* edge;      // [B,H,64,64]: the state the first segment starts from (forward), the
                          // gradient the last one ends with (backward), or null (zeros)
  float* bound;           // [B,H,G,64,64]: N, at the index of the segment it is handed to
  float* trans;           // [B,H,G,64,64]: M of segment g
  int* fault;             // [B,H,G]: segment g's wait gave up
  int T, H, G, cps;       // cps: chunks per segment (the last may have fewer)
  uint32_t spin_limit;    // polls per hand-over wait (> 0)
};

__device__ __forceinline__ const uint4* seg_piece(const SegParams& p, int64_t tok0, int64_t tstride, int c,
                                                  int lane, int k) {
  const int vec = k >> 1, step = 8 * (k & 1) + (lane >> 3);
  const int oct = ((lane & 7) - tile_rot(step)) & 7;
  return reinterpret_cast<const uint4*>(p.in[vec] + tok0 + (int64_t)(kL * c + step) * tstride + 8 * oct);
}

// `free_slot` returns once the slot may be overwritten.
template <bool kBwd, typename FreeSlot>
__device__ __forceinline__ void prepare_segment_chunk(SegPrep& my, SegOps& o, int lane, FreeSlot free_slot) {
  const int t = lane & 15, qd = lane >> 4;
  PadTile* const stg = my.stg;
  auto raw = [&](int vec, int m, int hh) -> f32x4 {
    const uint2 u = *reinterpret_cast<const uint2*>(tile_at(stg[vec].r, t, 32 * m + 16 * hh + 4 * qd));
    return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
                 __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
  };
  // A^ = a gamma_(t-1), B~ = b / gamma_t, and K~ = k / gamma_t or R^ = r gamma_t
  Split8 AH[2], BT[2], FR[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    f32x4 ah[2], bt[2], fr[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const f32x4 x = raw(S_X, m, hh);
      f32x4 gam, gin, gpv, gl;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float g = row_scan16(log2_decay(x[c]));
        const float e = exp2_f(g);
        gam[c] = e;
        gin[c] = exp2_f(-g);
        gpv[c] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
            __builtin_bit_cast(int, 1.0f), __builtin_bit_cast(int, e), 0x111, 0xf, 0xf, false));
        gl[c] = row_last16(e);
      }
      if (t == 0) *reinterpret_cast<f32x4*>(&my.gl[32 * m + 16 * hh + 4 * qd]) = gl;
      ah[hh] = raw(S_A, m, hh) * gpv;
      bt[hh] = raw(S_B, m, hh) * gin;
      fr[hh] = raw(S_K, m, hh) * (kBwd ? gam : gin);
    }
    AH[m] = split8(ah[0], ah[1]);
    BT[m] = split8(bt[0], bt[1]);
    FR[m] = split8(fr[0], fr[1]);
  }
  // step products: A_ab in both orientations; q is A_ak (forward) or A_rb^T
  // (backward) as an A operand (the lane's row, contraction over 4 qd + r)
  f32x4 aab = {0.f, 0.f, 0.f, 0.f}, aabT = aab, q = aab;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    aabT = mma32x3(BT[m], AH[m], aabT);
    aab = mma32x3(AH[m], BT[m], aab);
    q = kBwd ? mma32x3(FR[m], BT[m], q) : mma32x3(FR[m], AH[m], q);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = 4 * qd + r;
    if (!(s < t)) aabT[r] = 0.f;
    if (!(t < s)) aab[r] = 0.f;
    if (kBwd ? !(t <= s) : !(s < t)) q[r] = 0.f;
  }
  // forward: lane (qd, t) holds P[t][4 qd + r], i.e. P as an A operand and
  // P^T as a B operand; backward: P[4 qd + r][t], P^T as A and P as B
  const Split4 P = split4(kBwd ? unit_lower_inverse(aab, aabT, t, qd) : unit_lower_inverse(aabT, aab, t, qd));

  // hi/lo rows into LDS, then their transposed fragments (row = key, k =
  // step): A^ and B~ first, K~ / R^ in the same tiles after them
  bf16_t (*rows[4])[64] = {stg[S_X].r, stg[S_A].r, stg[S_B].r, stg[S_K].r};
  auto put = [&](int i, const Split8 (&x)[2]) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const Split4 h4 = half_of(x[m], hh);
        write4(rows[i], t, 32 * m + 16 * hh + 4 * qd, h4.hi);
        write4(rows[i + 1], t, 32 * m + 16 * hh + 4 * qd, h4.lo);
      }
  };
  auto tr = [&](bf16_t (*tile)[64], int ib) { return tr_frag(tile, 0, 16 * ib, lane); };
  put(0, AH);
  put(2, BT);
  wave_lds_sync();
  free_slot();
  // W^T = A^^T P^T (forward) or B~^T P (backward): rows = keys, column = step
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    f32x4 Wt[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int ib = 2 * m + hh;
      const Split4 aT{tr(rows[0], ib), tr(rows[1], ib)}, bT{tr(rows[2], ib), tr(rows[3], ib)};
      Wt[hh] = mma_s3(stack(kBwd ? bT : aT), P, f32x4{0.f, 0.f, 0.f, 0.f});
      o.g[ib][lane] = stack(kBwd ? aT : bT);
    }
    const Split8 w8 = split8(Wt[0], Wt[1]);
    o.w[m][0][lane] = w8.hi;
    o.w[m][1][lane] = w8.lo;
  }
  wave_lds_sync();
  put(0, FR);
  wave_lds_sync();
#pragma unroll
  for (int ib = 0; ib < 4; ++ib) o.f[ib][lane] = cat8(tr(rows[0], ib), tr(rows[1], ib));
  o.gl[lane] = my.gl[lane];
  const bf16x8 qs = stack(split4(q)), Ps = stack(P);
#pragma unroll
  for (int vb = 0; vb < 4; ++vb) {
    const bf16x4 vt = tr(stg[S_V].r, vb);
    o.v[vb][lane] = vt;
    const f32x4 X = mma_s2(qs, vt, f32x4{0.f, 0.f, 0.f, 0.f});
    o.u[vb][lane] = mma_s3(Ps, split4(X), f32x4{0.f, 0.f, 0.f, 0.f});
  }
}

// Grid (H, B, G - 1): the segment whose result nobody needs (the last one
// forward, the first one backward) is not run.
template <bool kBwd>
__global__ __launch_bounds__(kBlock, 1) void wkv7_transition_kernel(const SegParams p) {
  __shared__ SegOps ops[kSlots];
  __shared__ __attribute__((aligned(16))) SegPrep prep[kPrepWaves];
  __shared__ Flags flags;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: roles branch on it
  const int t = lane & 15, qd = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.y, H = p.H, T = p.T;
  const int g = kBwd ? blockIdx.z + 1 : blockIdx.z;
  const int64_t bh = (int64_t)b * H + h;
  const int64_t tstride = (int64_t)H * kHead;
  const int total = T / kL;
  const int c0 = g * p.cps, n = min(p.cps, total - c0);   // chunks of this segment (n >= 1)
  const int64_t tok0 = (((int64_t)b * T + (int64_t)kL * c0) * H + h) * kHead;
  // the i-th chunk in the order of the chain
  auto chunk_of = [&](int i) { return kBwd ? n - 1 - i : i; };
  // the segment at the known end of the sequence: N starts from the given
  // state, and M is not needed
  const bool edge = kBwd ? g == p.G - 1 : g == 0;

  if (tid < kSlots) flags.ready[tid] = -1;
  if (tid == 0) flags.fault = 0;
  if (tid < kSlots * kChainWaves) flags.taken[tid / kChainWaves][tid % kChainWaves] = tid / kChainWaves - kSlots;
  __syncthreads();

  float* const out_n = p.bound + (bh * p.G + (kBwd ? g - 1 : g + 1)) * (kHead * kHead);
  float* const out_m = p.trans + (bh * p.G + g) * (kHead * kHead);
  if (wave >= kChainWaves) {
    // chunks s, s + 8, ... of the chain's order, into slot s % 4
    const int s = wave - kChainWaves, slot = s % kSlots;
    SegPrep& my = prep[s];
    static_assert(kPieces == 10, "ten 16-byte pieces per lane and chunk");
    if (s < n) {
      // the next chunk's raw rows are loaded while this one is prepared; kept
      // by the caches for the main kernel, which reads them again
      uint4 r0, r1, r2, r3, r4, r5, r6, r7, r8, r9;
#define RWKV_SEG_LOAD(c) \
  r0 = *seg_piece(p, tok0, tstride, c, lane, 0); r1 = *seg_piece(p, tok0, tstride, c, lane, 1); \
  r2 = *seg_piece(p, tok0, tstride, c, lane, 2); r3 = *seg_piece(p, tok0, tstride, c, lane, 3); \
  r4 = *seg_piece(p, tok0, tstride, c, lane, 4); r5 = *seg_piece(p, tok0, tstride, c, lane, 5); \
  r6 = *seg_piece(p, tok0, tstride, c, lane, 6); r7 = *seg_piece(p, tok0, tstride, c, lane, 7); \
  r8 = *seg_piece(p, tok0, tstride, c, lane, 8); r9 = *seg_piece(p, tok0, tstride, c, lane, 9);
      RWKV_SEG_LOAD(chunk_of(s))
      for (int i = s; i < n; i += kPrepWaves) {
        auto dst = [&](int k) { return reinterpret_cast<uint4*>(&my.stg[k >> 1].r[8 * (k & 1)][0]) + lane; };
        *dst(0) = r0; *dst(1) = r1; *dst(2) = r2; *dst(3) = r3; *dst(4) = r4;
        *dst(5) = r5; *dst(6) = r6; *dst(7) = r7; *dst(8) = r8; *dst(9) = r9;
        const int in = i + kPrepWaves < n ? i + kPrepWaves : i;   // the last reloads itself
        RWKV_SEG_LOAD(chunk_of(in))
        wave_lds_sync();
        prepare_segment_chunk<kBwd>(my, ops[slot], lane, [&] {
          bool ok = true;
          for (int w = 0; w < kChainWaves; ++w) ok &= wait_flag(&flags.taken[slot][w], i - kSlots, p.spin_limit);
          if (!ok && lane == 0) lds_store_flag(&flags.fault, 1);
          lds_acquire();
        });
        lds_release();
        if (lane == 0) lds_store_flag(&flags.ready[slot], i);
      }
#undef RWKV_SEG_LOAD
    }
  } else {
    // value tile jb; key tiles ib in the result layout (rows = key i = 16 ib
    // + 4 qd + r, columns = value j = 16 jb + t)
    const int jb = wave, jcol = 16 * jb + t;
    f32x4 SN[4], SM[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      if (edge && p.edge)
        SN[ib] = *reinterpret_cast<const f32x4*>(p.edge + bh * (kHead * kHead) + jcol * kHead + 16 * ib + 4 * qd);
      else
        SN[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) SM[ib][r] = 16 * ib + 4 * qd + r == jcol ? 1.f : 0.f;
    }
    auto chain = [&](auto both) {
      constexpr bool kBoth = decltype(both)::value;   // M's state too
      for (int i = 0; i < n; ++i) {
        const int slot = i % kSlots;
        if (!wait_flag(&flags.ready[slot], i, p.spin_limit) && lane == 0) lds_store_flag(&flags.fault, 1);
        lds_acquire();
        const SegOps& o = ops[slot];
        const Split8 w0{o.w[0][0][lane], o.w[0][1][lane]}, w1{o.w[1][0][lane], o.w[1][1][lane]};
        const f32x4 u = o.u[jb][lane];
        const bf16x4 v = o.v[jb][lane];
        bf16x8 f[4], gg[4];
        f32x4 gl[4];
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          f[ib] = o.f[ib][lane];
          gg[ib] = o.g[ib][lane];
          gl[ib] = *reinterpret_cast<const f32x4*>(&o.gl[16 * ib + 4 * qd]);
        }
        if (kBwd) {
#pragma unroll
          for (int ib = 0; ib < 4; ++ib) {
            SN[ib] *= gl[ib];
            if (kBoth) SM[ib] *= gl[ib];
          }
        }
        const Split8 n0 = split8(SN[0], SN[1]), n1 = split8(SN[2], SN[3]);
        f32x4 sn = mma32x3(w0, n0, u), sm = {0.f, 0.f, 0.f, 0.f};
        sn = mma32x3(w1, n1, sn);
        if (kBoth) {
          const Split8 m0 = split8(SM[0], SM[1]), m1 = split8(SM[2], SM[3]);
          sm = mma32x3(w0, m0, sm);
          sm = mma32x3(w1, m1, sm);
        }
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) SN[ib] = mma_s2(f[ib], v, SN[ib]);
        const Split4 sns = split4(sn), sms = split4(sm);
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          SN[ib] = mma_s3(gg[ib], sns, SN[ib]);
          if (kBoth) SM[ib] = mma_s3(gg[ib], sms, SM[ib]);
          if (!kBwd) {
            SN[ib] *= gl[ib];
            if (kBoth) SM[ib] *= gl[ib];
          }
        }
        // every operand has been used, so its load has completed
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
        lds_release();
        if (lane == 0) lds_store_flag(&flags.taken[slot][jb], i);
      }
    };
    if (edge) chain(std::false_type{});
    else chain(std::true_type{});
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      const int at = jcol * kHead + 16 * ib + 4 * qd;
      *reinterpret_cast<f32x4*>(out_n + at) = SN[ib];
      if (!edge) *reinterpret_cast<f32x4*>(out_m + at) = SM[ib];
    }
  }
  // a wave that gave up a wait: N becomes NaN, so every result that depends on
  // it does, and the segment's word says so
  __syncthreads();
  const bool bad = lds_load_flag(&flags.fault) != 0;
  if (bad)
    for (int i = tid; i < kHead * kHead; i += kBlock) out_n[i] = __builtin_nanf("");
  if (tid == 0) {
    p.fault[bh * p.G + g] = bad ? 1 : 0;
    // the segment that is not run here has its word cleared by its neighbour
    if (g == (kBwd ? 1 : p.G - 2)) p.fault[bh * p.G + (kBwd ? 0 : p.G - 1)] = 0;
  }
}

// The segments' boundary states in order: bound[g + 1] += bound[g] M[g]
// (forward, g = 1 .. G - 2), bound[g - 1] += bound[g] M[g] (backward, g =
// G - 2 .. 1). State rows are independent: one workgroup per (batch, head)
// and 16 rows, wave w the key tile 16 w ..; fp32 matrix products, four
// accumulators so that the sixteen steps over the inner axis overlap. The
// chain is one small product per segment, so M and N are loaded kAhead
// segments before they are multiplied.
constexpr int kAhead = 4;
template <bool kBwd>
__global__ __launch_bounds__(256) void wkv7_combine_kernel(float* bound, const float* trans, int G) {
  __shared__ float row[2][16][kHead + 4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = lane & 15, qd = lane >> 4;
  const int64_t bh = blockIdx.x;
  const int j0 = 16 * blockIdx.y;
  float* const bd = bound + bh * G * (kHead * kHead) + (j0 + 4 * qd) * kHead + 16 * w + t;
  const float* const tm = trans + bh * G * (kHead * kHead) + qd * kHead + 16 * w + t;
  const int step = kBwd ? -1 : 1, count = G - 2;
  // the i-th segment multiplied; past the last one, the last one again
  auto seg = [&](int i) { return kBwd ? G - 2 - min(i, count - 1) : 1 + min(i, count - 1); };
  float m[kAhead][16];
  f32x4 nn[kAhead];
  auto load = [&](int i, float (&mi)[16], f32x4& ni) {
    const int g = seg(i);
#pragma unroll
    for (int s = 0; s < 16; ++s) mi[s] = tm[g * (kHead * kHead) + 4 * s * kHead];
#pragma unroll
    for (int r = 0; r < 4; ++r) ni[r] = bd[(g + step) * (kHead * kHead) + r * kHead];
  };
#pragma unroll
  for (int r = 0; r < 4; ++r) row[0][4 * qd + r][16 * w + t] = bd[seg(0) * (kHead * kHead) + r * kHead];
#pragma unroll
  for (int a = 0; a < kAhead; ++a) load(a, m[a], nn[a]);
  for (int i0 = 0; i0 < count; i0 += kAhead) {
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      const int i = i0 + a;
      if (i >= count) break;
      __syncthreads();
      f32x4 acc[4] = {nn[a], {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int s = 0; s < 16; ++s)
        acc[s & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(row[i & 1][t][4 * s + qd], m[a][s], acc[s & 3], 0, 0, 0);
      const f32x4 o = (acc[0] + acc[1]) + (acc[2] + acc[3]);
      const int g = seg(i);
#pragma unroll
      for (int r = 0; r < 4; ++r) row[(i + 1) & 1][4 * qd + r][16 * w + t] = o[r];
      // loads before the stores: a wait for a load also waits for older stores
      load(i + kAhead, m[a], nn[a]);
#pragma unroll
      for (int r = 0; r < 4; ++r) bd[(g + step) * (kHead * kHead) + r * kHead] = o[r];
    }
  }
}

// One wave per (batch, head), after a segmented forward.
template <typename Tio>
__global__ __launch_bounds__(64) void wkv7_segment_poison_kernel(const int* fault, int G, Tio* y, float* sa,
                                                                  float* ckpt, float* sT, int T, int C,
                                                                  unsigned int* faults) {
  const int64_t bh = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
  bool bad = false;
  for (int i = threadIdx.x; i < G; i += 64) bad |= fault[bh * G + i] != 0;
  if (!__any(bad)) return;
  poison_forward(y, sa, ckpt, sT, blockIdx.y, blockIdx.x, gridDim.x, T, T / C, threadIdx.x, 64);
  if (threadIdx.x == 0) atomicAdd(faults, 1u);
}

template <bool kBwd>
hipError_t launch_bounds(const TransitionCall& c, bool f32, hipStream_t stream) {
  hipError_t e;
  if (f32) {
    e = launch_transition_f32(c, stream);
  } else {
    SegParams p;
    for (int i = 0; i < kVecs; ++i) p.in[i] = static_cast<const bf16_t*>(c.in[i]);
    p.edge = c.edge;
    p.bound = c.seg.bound;
    p.trans = c.seg.trans;
    p.fault = c.seg.fault;
    p.T = c.T;
    p.H = c.H;
    p.G = c.seg.G;
    p.cps = c.seg.cps;
    p.spin_limit = c.spin_limit;
    hipLaunchKernelGGL(wkv7_transition_kernel<kBwd>, dim3(c.H, c.B, p.G - 1), dim3(kBlock), 0, stream, p);
    e = hipGetLastError();
  }
  if (e != hipSuccess || c.seg.G < 3) return e;
  hipLaunchKernelGGL(wkv7_combine_kernel<kBwd>, dim3(c.B * c.H, 4), dim3(256), 0, stream, c.seg.bound, c.seg.trans,
                     c.seg.G);
  return hipGetLastError();
}

// What a call takes, in microseconds, fitted to timings of 1 to 192 pairs and
// 4 to 256 chunks (back-to-back Python calls, workspace allocation included):
// n chunks in one piece cost a + b n; in G segments of cps chunks, c + d G +
// e cps (d: the combine kernel's step). Neither is below what issuing the
// launches takes the host.
struct Cost {
  float whole_host, a, b;
  float seg_host, c, d, e;
};
// Forward, 32 pairs, us: n = 256: 354 in one piece, 137 in 8 segments; n = 32:
// 52 and 40; n = 16: 30 and 34. 64 pairs, n = 256: 359 and 224 (4 segments).
constexpr Cost kForwardCost = {22.f, 4.5f, 1.36f, 34.f, 16.f, 0.65f, 3.6f};
// Backward, 32 pairs: n = 256: 748 and 171; n = 32: 106 and 48; n = 16: 60 and
// 38. 128 pairs, n = 64: 201 and 150 (2 segments).
constexpr Cost kBackwardCost = {28.f, 13.f, 2.88f, 37.f, 25.f, 0.65f, 4.38f};

// The fp32 chunked kernels. Forward, 32 pairs: n = 256: 725 in one piece and
// 222 in 8 segments; n = 32: 101 and 53; n = 16: 54 and 40; 85 pairs, n = 16:
// 59 and 63 (3 segments).
constexpr Cost kForwardCost32 = {22.f, 9.f, 2.8f, 34.f, 27.f, 0.5f, 5.7f};
// Backward, 32 pairs: n = 256: 1922 and 359; n = 16: 130 and 48. 128 pairs, n =
// 64: 492 and 319 (2 segments).
constexpr Cost kBackwardCost32 = {28.f, 5.f, 7.6f, 37.f, 25.f, 0.5f, 9.6f};

// The cheapest number of segments, among those whose workgroups (one per pair
// and segment, each filling a CU's LDS) all run at once: more would queue, and
// the transition pass would be paid for nothing. q: chunks per checkpoint
// interval, of which a segment holds a whole number.
Segments plan(int64_t pairs, int n, int q, const Cost& k) {
  constexpr int kCus = 256;
  Segments best;
  best.cps = n;
  float cost = std::max(k.whole_host, k.a + k.b * n);
  const int units = n / q, most = (int)std::min<int64_t>(kCus / std::max<int64_t>(pairs, 1), units);
  for (int g = 2; g <= most; ++g) {
    const int cps = (units + g - 1) / g * q, G = (n + cps - 1) / cps;
    const float c = std::max(k.seg_host, k.c + k.d * G + k.e * cps);
    if (G > 1 && c < cost) {
      cost = c;
      best.G = G;
      best.cps = cps;
    }
  }
  return best;
}

}  // namespace

Segments plan_segments(const ForwardDesc& d) {
  const int64_t pairs = (int64_t)d.B * d.H;
  if (d.kc.step_only) return Segments{};
  if (chunk_forward_supported(d)) return plan(pairs, d.T / kL, 1, kForwardCost);
  if (chunk_f32_forward_supported(d)) return plan(pairs, d.T / kL, d.C / kL, kForwardCost32);
  return Segments{};
}
Segments plan_segments(const BackwardDesc& d) {
  const int64_t pairs = (int64_t)d.B * d.H;
  if (d.kc.step_only) return Segments{};
  if (chunk_backward_supported(d)) return plan(pairs, d.T / kL, d.C / kL, kBackwardCost);
  if (chunk_f32_backward_supported(d) && chunk_f32_backward_preferred(d))
    return plan(pairs, d.T / kL, d.C / kL, kBackwardCost32);
  return Segments{};
}

int64_t segment_bytes(const Segments& s, int B, int H) {
  if (s.G < 2) return 0;
  return (int64_t)B * H * s.G * (2 * kHead * kHead * (int64_t)sizeof(float) + (int64_t)sizeof(int));
}
void place_segments(Segments* s, int B, int H, void* workspace) {
  const int64_t states = (int64_t)B * H * s->G * kHead * kHead;
  s->bound = static_cast<float*>(workspace);
  s->trans = s->bound + states;
  s->fault = reinterpret_cast<int*>(s->trans + states);
}

hipError_t launch_segment_bounds(const ForwardDesc& d, hipStream_t stream) {
  return launch_bounds<false>(TransitionCall{{d.w, d.a, d.b, d.k, d.v}, d.s0, d.seg, d.B, d.T, d.H, d.dtype, false,
                                             d.kc.spin_limit ? d.kc.spin_limit : kSpinLimit},
                              !chunk_forward_supported(d), stream);
}
hipError_t launch_segment_bounds(const BackwardDesc& d, hipStream_t stream) {
  return launch_bounds<true>(TransitionCall{{d.w, d.a, d.b, d.r, d.dy}, d.dsT, d.seg, d.B, d.T, d.H, d.dtype, true,
                                            d.kc.spin_limit ? d.kc.spin_limit : kSpinLimit},
                             !chunk_backward_supported(d), stream);
}
hipError_t launch_segment_poison(const ForwardDesc& d, hipStream_t stream) {
  unsigned int* faults;
  if (hipError_t e = handover_fault_counter(&faults)) return e;
  auto go = [&](auto* y) {
    typedef typename std::remove_pointer<decltype(y)>::type Tio;
    hipLaunchKernelGGL(wkv7_segment_poison_kernel<Tio>, dim3(d.H, d.B), dim3(64), 0, stream, d.seg.fault, d.seg.G, y,
                       d.sa, d.ckpt, d.sT, d.T, d.C, faults);
    return hipGetLastError();
  };
  return d.dtype == Dtype::BF16 ? go(static_cast<bf16_t*>(d.y)) : go(static_cast<float*>(d.y));
}

}  // namespace wkv7
