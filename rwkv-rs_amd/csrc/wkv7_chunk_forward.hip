// Chunked WKV7 forward on the matrix cores (bf16 operands, fp32 state).
//
// Computes what wkv7_forward_kernel does (crates/rwkv-nn/src/kernels/
// wkv7_common/kernel.rs:6-114, launched by wkv7_common/host.rs:29-183): the
// per-step removal_state sa_t = S_{t-1} a_t, the output y_t = S_t r_t, the
// transposed state every chunk_len steps, the optional initial state load and
// final state store. It takes the matrix form of 16-step chunks (wkv7_chunk.hpp)
// instead of stepping the state 4096 times, so the state's dependency chain is
// 37 small matrix products per chunk instead of 16 rank-2 updates with
// reductions.
//
// Work layout: one workgroup of eight waves per (batch, head), two per SIMD,
// in two groups that run concurrently and hand chunks over through LDS:
//   prep waves 4-7  wave 4 + s prepares chunks c = s, s + 4, ... on its own:
//                   stages the chunk's raw rows in its LDS region (loaded
//                   into registers during the previous chunk), forms the
//                   decays, the four 16x16 step-by-step products, P on the
//                   matrix cores, W and U, and writes every operand the chain
//                   needs to slot s, in fragment order (one 16-byte or 8-byte
//                   load per lane); then it marks the slot ready;
//   chain waves 0-3 take the chunks in order; wave w owns value columns
//                   16w..16w+15 of the state (state rows are independent in
//                   the forward), loads chunk c's operands from slot c % 4,
//                   computes SA, Y and the next state, and marks the slot
//                   taken once every operand has been used.
// A prep wave overwrites its slot only after all four chain waves have taken
// the chunk in it, so preparing chunk c overlaps the chain of chunks c-4 ..
// c-1. The hand-over uses two LDS flags per slot and no barriers; every wait
// is bounded, so a kernel whose flags went wrong ends instead of hanging. A
// wave that gives up a wait raises a workgroup fault flag; after a final
// barrier the workgroup then overwrites all of its (batch, head)'s outputs
// with NaN and counts the event in a device counter the host reads back
// (wkv7_take_faults), so a broken hand-over is never silent.
#include "wkv7_chunk.hpp"
#include "wkv7_launch.hpp"

namespace wkv7 {
namespace {

using namespace chunk;

constexpr int kChainWaves = 4;            // value tile = wave
constexpr int kSlots = 4;                 // operand slots = prep waves
constexpr int kWaves = kChainWaves + kSlots;
constexpr int kBlock = 64 * kWaves;
constexpr int kVecs = 6;                  // staged inputs: x, r, k, a, b, v
enum { S_X, S_R, S_K, S_A, S_B, S_V };
constexpr int kPieces = kVecs * kL * 8 / 64;   // 16-byte loads per prep lane and chunk
// hand-over faults of chunked forwards and segmented calls on this device since
// the host last took them, and the value the last take read
__device__ unsigned int handover_faults;
__device__ unsigned int handover_faults_taken;

// Phase-1 products of one chunk, each in the fragment order its phase-2
// consumer loads (index [lane] last). K~ and B~ are kept without the chunk's
// total decay gamma_L, which phase 2 applies to the updated state instead:
// S_L^T = diag(gamma_L) (S0^T + K~^T V + B~^T SA).
struct ChunkOps {
  bf16x8 w[2][2][64];     // W = P A^, x32 A operand: [key half][hi/lo]
  bf16x8 r[2][2][64];     // R^, x32 A operand
  bf16x8 ark[64];         // A_rk stacked (hi | lo), contraction over steps
  bf16x8 arb[64];         // A_rb stacked
  bf16x8 kt[4][64];       // K~^T stacked, per key tile (row = key, k = step)
  bf16x8 bt[4][64];       // B~^T stacked
  bf16x4 v[4][64];        // V, x16 B operand per value tile (k = step)
  f32x4 u[4][64];         // U per value tile, result layout (SA's start)
  float gl[64];           // gamma_L
};

struct FwdChunkParams {
  const bf16_t* in[kVecs];   // [B,T,H,64] each, in S_* order
  const float* s0;
  float* ckpt;
  float* sa;
  bf16_t* y;
  float* sT;
  int T, H;
  // segmented calls only:
  int cps;                   // chunks per segment
  const float* bound;        // segment g > 0 of [B,H,G,64,64]: its start state
  int* fault;                // [B,H,G]
  uint32_t spin_limit;       // polls per hand-over wait (> 0)
};

// The preparation of one chunk, run by one wave. `stg` holds the chunk's raw
// rows; after they are read, the chunk's x, r, k, a, b rows and the wave's
// scratch `scr` are reused for the hi/lo rows of A^, K~ and B~, from which the
// transposed fragments are read.
__device__ __forceinline__ void prepare_chunk(PadTile* stg, float (*scr)[kL][kL],
                                              ChunkOps& o, int lane) {
  const int t = lane & 15, qd = lane >> 4;
  // the lane's step row t, keys 32 m + 16 hh + 4 qd + c (c < 4), as raw bf16
  auto raw = [&](int vec, int m, int hh) -> uint2 {
    return *reinterpret_cast<const uint2*>(tile_at(stg[vec].r, t, 32 * m + 16 * hh + 4 * qd));
  };
  auto widen = [](uint2 u) -> f32x4 {
    return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
                 __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
  };

  // decays: gamma_t (prefix product over the chunk's steps, via log2 sums),
  // 1/gamma_t, gamma_{t-1} (previous lane of the row; 1 at t = 0), gamma_L
  f32x4 gam[2][2], gin[2][2], gpv[2][2];
  float gL[2][2][4];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const f32x4 x = widen(raw(S_X, m, hh));
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float g = row_scan16(log2_decay(x[c]));
        const float e = exp2_f(g);
        gam[m][hh][c] = e;
        gin[m][hh][c] = exp2_f(-g);
        gpv[m][hh][c] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
            __builtin_bit_cast(int, 1.0f), __builtin_bit_cast(int, e), 0x111, 0xf, 0xf, false));
        gL[m][hh][c] = row_last16(e);
      }
    }
  Split8 AH[2], RH[2], KT[2], BT[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    f32x4 ah[2], rh[2], kt[2], bt[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      ah[hh] = widen(raw(S_A, m, hh)) * gpv[m][hh];
      rh[hh] = widen(raw(S_R, m, hh)) * gam[m][hh];
      kt[hh] = widen(raw(S_K, m, hh)) * gin[m][hh];
      bt[hh] = widen(raw(S_B, m, hh)) * gin[m][hh];
    }
    AH[m] = split8(ah[0], ah[1]);
    RH[m] = split8(rh[0], rh[1]);
    KT[m] = split8(kt[0], kt[1]);
    BT[m] = split8(bt[0], bt[1]);
  }
  // step-by-step products, computed transposed: result row = step s, lane
  // column = step t, which is the x16 A operand (row t, k = s) of A_xx[t][s]
  f32x4 akT = {0.f, 0.f, 0.f, 0.f}, arkT = akT, arbT = akT, aabT = akT, aab = akT;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    akT = mma32x3(KT[m], AH[m], akT);
    arkT = mma32x3(KT[m], RH[m], arkT);
    arbT = mma32x3(BT[m], RH[m], arbT);
    aabT = mma32x3(BT[m], AH[m], aabT);
    aab = mma32x3(AH[m], BT[m], aab);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = 4 * qd + r;
    if (!(s < t)) { akT[r] = 0.f; aabT[r] = 0.f; }
    if (!(s <= t)) { arkT[r] = 0.f; arbT[r] = 0.f; }
    if (!(t < s)) aab[r] = 0.f;
  }
  // P^T = (I - A_ab^T)^{-1} on the matrix cores, in the result layout: lane
  // (qd, t) holds P[t][4 qd + r], which is P as an A operand and P^T as a B
  // operand
  const Split4 P = split4(unit_lower_inverse(aabT, aab, t, qd));

  // hi/lo rows of A^, K~, B~ into LDS (the chunk's raw rows are consumed),
  // then their transposed fragments (row = key, k = step) by transposed loads
  bf16_t (*rows[6])[64] = {stg[S_X].r, stg[S_R].r, stg[S_K].r, stg[S_A].r, stg[S_B].r,
                           reinterpret_cast<bf16_t (*)[64]>(&scr[0][0][0])};
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int c0 = 32 * m + 16 * hh + 4 * qd;
      const Split4 a = half_of(AH[m], hh), k = half_of(KT[m], hh), b = half_of(BT[m], hh);
      *reinterpret_cast<bf16x4*>(tile_at(rows[0], t, c0)) = a.hi;
      *reinterpret_cast<bf16x4*>(tile_at(rows[1], t, c0)) = a.lo;
      *reinterpret_cast<bf16x4*>(tile_at(rows[2], t, c0)) = k.hi;
      *reinterpret_cast<bf16x4*>(tile_at(rows[3], t, c0)) = k.lo;
      *reinterpret_cast<bf16x4*>(tile_at(rows[4], t, c0)) = b.hi;
      *reinterpret_cast<bf16x4*>(tile_at(rows[5], t, c0)) = b.lo;
    }
  wave_lds_sync();
  // lane (group g, c) addresses row 4 g + c / 4, columns 16 ib + 4 (c % 4)
  const int tr_t = 4 * qd + (t >> 2), tr_c = 4 * (t & 3);
  auto tr = [&](bf16_t (*tile)[64], int ib) { return read_tr16(tile_at(tile, tr_t, 16 * ib + tr_c)); };

  // W^T tile ib = A^T P^T (result rows = keys, lane column = step t), which
  // is W in the x32 A-operand order
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    f32x4 Wt[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int ib = 2 * m + hh;
      const Split4 aT{tr(rows[0], ib), tr(rows[1], ib)};
      Wt[hh] = mma_s3(stack(aT), P, f32x4{0.f, 0.f, 0.f, 0.f});
      o.kt[ib][lane] = cat8(tr(rows[2], ib), tr(rows[3], ib));
      o.bt[ib][lane] = cat8(tr(rows[4], ib), tr(rows[5], ib));
    }
    const Split8 w8 = split8(Wt[0], Wt[1]);
    o.w[m][0][lane] = w8.hi;
    o.w[m][1][lane] = w8.lo;
    o.r[m][0][lane] = RH[m].hi;
    o.r[m][1][lane] = RH[m].lo;
  }
  const bf16x8 ak = stack(split4(akT));
  o.ark[lane] = stack(split4(arkT));
  o.arb[lane] = stack(split4(arbT));
  // U = P (A_ak V), per value tile
  const bf16x8 Ps = stack(P);
#pragma unroll
  for (int vb = 0; vb < 4; ++vb) {
    const bf16x4 vt = tr(stg[S_V].r, vb);
    o.v[vb][lane] = vt;
    const f32x4 X = mma_s2(ak, vt, f32x4{0.f, 0.f, 0.f, 0.f});
    o.u[vb][lane] = mma_s3(Ps, split4(X), f32x4{0.f, 0.f, 0.f, 0.f});
  }
  if (t == 0) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
        *reinterpret_cast<f32x4*>(&o.gl[32 * m + 16 * hh + 4 * qd]) =
            f32x4{gL[m][hh][0], gL[m][hh][1], gL[m][hh][2], gL[m][hh][3]};
  }
}

// Phase-2 operands of one chunk for value tile jb, in registers
struct ChainOps {
  Split8 w[2], r[2];
  bf16x8 ark, arb, kt[4], bt[4];
  bf16x4 v;
  f32x4 u, gl[4];
};
__device__ __forceinline__ ChainOps load_chain_ops(const ChunkOps& o, int jb, int lane) {
  const int qd = lane >> 4;
  ChainOps c;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    c.w[m] = Split8{o.w[m][0][lane], o.w[m][1][lane]};
    c.r[m] = Split8{o.r[m][0][lane], o.r[m][1][lane]};
  }
  c.ark = o.ark[lane];
  c.arb = o.arb[lane];
#pragma unroll
  for (int ib = 0; ib < 4; ++ib) {
    c.kt[ib] = o.kt[ib][lane];
    c.bt[ib] = o.bt[ib][lane];
    c.gl[ib] = *reinterpret_cast<const f32x4*>(&o.gl[16 * ib + 4 * qd]);
  }
  c.v = o.v[jb][lane];
  c.u = o.u[jb][lane];
  return c;
}

// a prep wave's LDS: the raw rows of the chunk it prepares, then (reused)
// the hi/lo rows of A^, K~, B~; 16-byte pieces of a row rotated by the step
// index so that row and transposed reads spread over the banks
struct PrepLds {
  PadTile stg[kVecs];
  float scr[2][kL][kL];
};

// hand-over flags: ready[s] = the chunk whose operands are in slot s,
// taken[s][w] = the last chunk chain wave w loaded from slot s
struct Flags {
  int ready[kSlots];
  int taken[kSlots][kChainWaves];
  int fault;                 // a wave gave up a wait
};

// A prep lane's share of a chunk's raw rows: piece k is row 8 k + lane / 8
// of the chunk's 6 x 16 rows (vec k / 2, step 8 (k % 2) + lane / 8); LDS slot
// lane % 8 of that row holds global 16-byte piece (slot - tile_rot(step)) % 8.
// Kept as named values so that the compiler holds them in registers across
// the preparation of a chunk.
__device__ __forceinline__ const uint4* raw_piece(const FwdChunkParams& p, int64_t tok0,
                                                  int64_t tstride, int c, int lane, int k) {
  const int vec = k >> 1, step = 8 * (k & 1) + (lane >> 3);
  const int oct = ((lane & 7) - tile_rot(step)) & 7;
  return reinterpret_cast<const uint4*>(p.in[vec] + tok0 + (int64_t)(kL * c + step) * tstride +
                                        8 * oct);
}
// The raw rows are read once per launch: loaded with the non-temporal hint
// (measured at config[1]: forward 0.503 -> 0.477 ms, the following backward
// 1% slower, the pair 1.2% faster; the same hint on the checkpoint stores made
// the forward 18% slower).
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 load_stream(const uint4* q) {
  const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(q));
  return make_uint4(x[0], x[1], x[2], x[3]);
}

// Grid (H, B, G): workgroup (h, b, g) runs segment g of the sequence, chunks
// g cps ..
template <int kStart>
__global__ __launch_bounds__(kBlock, 1) void wkv7_fwd_chunk_kernel(const FwdChunkParams p) {
  __shared__ ChunkOps ops[kSlots];
  __shared__ __attribute__((aligned(16))) PrepLds prep[kSlots];
  __shared__ Flags flags;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t = lane & 15, qd = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.y, H = p.H, T = p.T;
  const int64_t bh = (int64_t)b * H + h;
  const int64_t tstride = (int64_t)H * kHead;              // elements per step
  constexpr bool kSeg = kStart == start::kSegment;
  const int g = kSeg ? blockIdx.z : 0, total = T / kL;
  const int c0 = kSeg ? g * p.cps : 0, nchunks = kSeg ? min(p.cps, total - c0) : total;   // this segment's chunks
  // step 0 of (b, h)'s segment
  const int64_t tok0 = (((int64_t)b * T + (int64_t)kL * c0) * H + h) * kHead;
  const float* const s0 = start_state<kStart>(p.s0, p.bound, bh, g);
  const bool has_s0 = kStart == start::kGiven || (kSeg && s0);

  if (tid < kSlots) flags.ready[tid] = -1;
  if (tid == 0) flags.fault = 0;
  if (tid < kSlots * kChainWaves) flags.taken[tid / kChainWaves][tid % kChainWaves] = tid / kChainWaves - kSlots;
  __syncthreads();

  if (wave >= kChainWaves) {
    // ================================================= prep wave for slot s
    const int s = wave - kChainWaves;
    PrepLds& my = prep[s];
    // The raw rows of the next chunk are loaded into registers while this one
    // is prepared (one chunk of loads in flight hides their latency; LDS has no
    // room for a second staging region per wave).
    static_assert(kPieces == 12, "twelve 16-byte pieces per lane and chunk");
    if (s < nchunks) {
#define RWKV_RAW_LOAD(c) \
  r0 = load_stream(raw_piece(p, tok0, tstride, c, lane, 0)); r1 = load_stream(raw_piece(p, tok0, tstride, c, lane, 1)); \
  r2 = load_stream(raw_piece(p, tok0, tstride, c, lane, 2)); r3 = load_stream(raw_piece(p, tok0, tstride, c, lane, 3)); \
  r4 = load_stream(raw_piece(p, tok0, tstride, c, lane, 4)); r5 = load_stream(raw_piece(p, tok0, tstride, c, lane, 5)); \
  r6 = load_stream(raw_piece(p, tok0, tstride, c, lane, 6)); r7 = load_stream(raw_piece(p, tok0, tstride, c, lane, 7)); \
  r8 = load_stream(raw_piece(p, tok0, tstride, c, lane, 8)); r9 = load_stream(raw_piece(p, tok0, tstride, c, lane, 9)); \
  r10 = load_stream(raw_piece(p, tok0, tstride, c, lane, 10)); r11 = load_stream(raw_piece(p, tok0, tstride, c, lane, 11));
      uint4 r0, r1, r2, r3, r4, r5, r6, r7, r8, r9, r10, r11;
      RWKV_RAW_LOAD(s)
      for (int c = s; c < nchunks; c += kSlots) {
        // piece k: rows 8 (k % 2) .. of input k / 2
        auto dst = [&](int k) { return reinterpret_cast<uint4*>(&my.stg[k >> 1].r[8 * (k & 1)][0]) + lane; };
        *dst(0) = r0; *dst(1) = r1; *dst(2) = r2; *dst(3) = r3; *dst(4) = r4; *dst(5) = r5;
        *dst(6) = r6; *dst(7) = r7; *dst(8) = r8; *dst(9) = r9; *dst(10) = r10; *dst(11) = r11;
        // the last chunk reloads itself (harmless) so that the loads need no branch
        const int cn = c + kSlots < nchunks ? c + kSlots : c;
        RWKV_RAW_LOAD(cn)
        // the slot is free once every chain wave has taken chunk c - kSlots
        bool ok = true;
        for (int w = 0; w < kChainWaves; ++w) ok &= wait_flag(&flags.taken[s][w], c - kSlots, p.spin_limit);
        if (!ok && lane == 0) lds_store_flag(&flags.fault, 1);
        lds_acquire();
        prepare_chunk(my.stg, my.scr, ops[s], lane);
        lds_release();
        if (lane == 0) lds_store_flag(&flags.ready[s], c);
      }
#undef RWKV_RAW_LOAD
    }
  } else {
    // ===================================================== chain wave: value tile jb
    // state: key tiles ib = 0..3 in the result layout (rows = key i =
    // 16 ib + 4 qd + r, columns = value j = 16 jb + t)
    const int jb = wave, jcol = 16 * jb + t;
    f32x4 S[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      if (has_s0)
        S[ib] = *reinterpret_cast<const f32x4*>(s0 + jcol * kHead + 16 * ib + 4 * qd);
      else
        S[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint32_t tok_row = (uint32_t)tstride;                       // one step
    const uint32_t tok_off = 4 * qd * tok_row + jcol;                  // row 4 qd, column jcol
    const uint32_t ck_off = 4 * qd * kHead + jcol;
    const uint32_t yt_off = t * tok_row + 16 * jb + 4 * qd;            // row t, 4 values
    // the checkpoint after chunk c (chunk_len is 16 here: one per chunk),
    // transposed ([key][value]): rows = keys 16 ib + 4 qd + r, column jcol
    auto store_ckpt = [&](int c, const f32x4 (&st)[4]) {
      float* const ck = p.ckpt + (bh * total + c0 + c) * (kHead * kHead);
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int r = 0; r < 4; ++r) ck[ck_off + (16 * ib + r) * kHead] = st[ib][r];
    };

    for (int cidx = 0; cidx < nchunks; ++cidx) {
      const int slot = cidx % kSlots;
      if (!wait_flag(&flags.ready[slot], cidx, p.spin_limit) && lane == 0)
        lds_store_flag(&flags.fault, 1);
      lds_acquire();
      const ChainOps cur = load_chain_ops(ops[slot], jb, lane);

      const Split8 Sx0 = split8(S[0], S[1]), Sx1 = split8(S[2], S[3]);
      // the previous chunk's checkpoint (the state this chunk starts from),
      // stored here so that the stores overlap this chunk's products
      if (cidx > 0) store_ckpt(cidx - 1, S);
      f32x4 sa = mma32x3(cur.w[0], Sx0, cur.u);
      sa = mma32x3(cur.w[1], Sx1, sa);
      // Y^T = S0 R^T + V^T A_rk^T + SA^T A_rb^T: the same registers with the
      // operand roles swapped (a result tile as the A operand is its
      // transpose), so each lane holds 4 consecutive values of one step
      f32x4 yt = mma32x3(Sx0, cur.r[0], f32x4{0.f, 0.f, 0.f, 0.f});
      yt = mma32x3(Sx1, cur.r[1], yt);
      yt = mma32(twice(cur.v), cur.ark, yt);
      const Split4 sas = split4(sa);
      yt = mma32(cat8(sas.lo, bf16x4{0, 0, 0, 0}), cur.arb, yt);
      yt = mma32(twice(sas.hi), cur.arb, yt);
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        f32x4 st = mma_s2(cur.kt[ib], cur.v, S[ib]);
        st = mma_s3(cur.bt[ib], sas, st);
        S[ib] = st * cur.gl[ib];
      }
      // every operand has been used, so its load has completed (the wait costs
      // nothing here); the slot goes back to its prep wave
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
      lds_release();
      if (lane == 0) lds_store_flag(&flags.taken[slot][jb], cidx);
      // outputs: sa rows = steps 16 cidx + 4 qd + r, column = value jcol;
      // y at step 16 cidx + t, values 16 jb + 4 qd .. + 3 (one 8-byte store)
      const int64_t cbase = tok0 + (int64_t)kL * cidx * tstride;
      float* const sa_c = p.sa + cbase;
      bf16_t* const y_c = p.y + cbase;
#pragma unroll
      for (int r = 0; r < 4; ++r) sa_c[tok_off + r * tok_row] = sa[r];
      *reinterpret_cast<bf16x4*>(y_c + yt_off) = to_bf16x4(yt);
    }
    if (nchunks > 0) store_ckpt(nchunks - 1, S);

    if (p.sT && (!kSeg || c0 + nchunks == total)) {
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
        *reinterpret_cast<f32x4*>(p.sT + bh * (kHead * kHead) + jcol * kHead + 16 * ib + 4 * qd) = S[ib];
    }
  }

  // every wave ends here: if any wave gave up a wait, the whole (batch,
  // head)'s outputs are unreliable, so they are overwritten with NaN and the
  // event is counted for the host; a segment leaves its word for the kernel
  // that does this after all segments
  __syncthreads();
  if (kSeg) {
    if (tid == 0 && lds_load_flag(&flags.fault)) p.fault[bh * gridDim.z + g] = 1;
  } else if (lds_load_flag(&flags.fault)) {
    poison_forward(p.y, p.sa, p.ckpt, p.sT, b, h, H, T, total, tid, kBlock);
    if (tid == 0) atomicAdd(&handover_faults, 1u);
  }
}

__global__ void take_faults_kernel() {
  handover_faults_taken = atomicExch(&handover_faults, 0u);
}

}  // namespace

// bf16 operands and chunk_len 16. The checkpoints feed the reference-order
// backward, which rebuilds states between checkpoints by dividing by the
// decay and so amplifies a checkpoint's deviation by about 1.35x per step.
// The split-bf16 products leave the checkpoints ~2.5e-6 from the fp32
// algorithm's (~6e-8): harmless at chunk_len 16, where no state is rebuilt
// except chunk 0's, but measured at chunk_len 32 / 48 / 64 the rebuilt-state
// gradients (dw, dr, da) end up 4x / 30x / 30x further from exact than the
// reference algorithm's own. Longer chunk lengths therefore keep the
// step-by-step fp32 forward (the chunked backward takes them).
bool chunk_forward_supported(const ForwardDesc& d) {
  return d.dtype == Dtype::BF16 && d.C == kL && d.T % kL == 0;
}

hipError_t launch_forward_chunked(const ForwardDesc& d, hipStream_t stream) {
  FwdChunkParams p;
  p.in[S_X] = static_cast<const bf16_t*>(d.w);
  p.in[S_R] = static_cast<const bf16_t*>(d.r);
  p.in[S_K] = static_cast<const bf16_t*>(d.k);
  p.in[S_A] = static_cast<const bf16_t*>(d.a);
  p.in[S_B] = static_cast<const bf16_t*>(d.b);
  p.in[S_V] = static_cast<const bf16_t*>(d.v);
  p.s0 = d.s0;
  p.ckpt = d.ckpt;
  p.sa = d.sa;
  p.y = static_cast<bf16_t*>(d.y);
  p.sT = d.sT;
  p.T = d.T;
  p.H = d.H;
  p.cps = d.seg.cps;
  p.bound = d.seg.bound;
  p.fault = d.seg.fault;
  p.spin_limit = d.kc.spin_limit ? d.kc.spin_limit : kSpinLimit;
  const dim3 grid(d.H, d.B, d.seg.G), block(kBlock, 1, 1);
  if (d.seg.G > 1)
    if (hipError_t e = launch_segment_bounds(d, stream)) return e;
  auto* const kernel = d.seg.G > 1 ? wkv7_fwd_chunk_kernel<start::kSegment>
                       : d.s0 ? wkv7_fwd_chunk_kernel<start::kGiven> : wkv7_fwd_chunk_kernel<start::kZero>;
  hipLaunchKernelGGL(kernel, grid, block, 0, stream, p);
  hipError_t e = hipGetLastError();
  return e == hipSuccess && d.seg.G > 1 ? launch_segment_poison(d, stream) : e;
}

hipError_t handover_fault_counter(unsigned int** counter) {
  return hipGetSymbolAddress(reinterpret_cast<void**>(counter), HIP_SYMBOL(handover_faults));
}

hipError_t take_handover_faults(hipStream_t stream, uint32_t* count) {
  hipLaunchKernelGGL(take_faults_kernel, dim3(1), dim3(1), 0, stream);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  e = hipMemcpyFromSymbolAsync(count, HIP_SYMBOL(handover_faults_taken), sizeof(uint32_t), 0,
                               hipMemcpyDeviceToHost, stream);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(stream);
}

}  // namespace wkv7
