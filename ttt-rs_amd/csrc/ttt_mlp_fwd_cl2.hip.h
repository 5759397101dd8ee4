// TTT-MLP multi-stage forward for head_dim 128 (and 96) on gfx950: the register-resident kernel of
// ttt_mlp_fwd_rr.hip.h spread over a PAIR of workgroups (two CUs) per (batch, head).
//
// Arithmetic: reference rust/core/src/mlp.rs:127-208 looped as rust/core/src/inner.rs:25-50.
//
// At d = 128 the f32 state (W1 [128,512], W2 [512,128]: 512 KiB) equals the whole register file of
// one CU, so the hidden axis is cut in two: workgroup `cu` of a pair owns hidden units
// [2d cu, 2d cu + 2d), i.e. W1[:, half], W2[half, :], b1[half] (128 VGPRs of state per lane), and
// runs the register-resident scheme on its half.  A workgroup has d/16 waves: one per d-feature tile
// (reducer and output roles) and two hidden tiles each.  At d = 96 (six waves, 96 VGPRs of state) the
// state fits one CU and the pair is an option for launches with at most half as many units as CUs.
// What crosses the pair, once per mini-batch:
//   X1  (recurrence)  each CU's locally reduced Z2^T tiles [d x 16]: both CUs add the two halves
//       (always in the order cu 0 + cu 1, so both hold bit-identical Z2, G2, b2);
//   X2  (output path) CU 1's locally reduced Zbar2^T tiles and A2 tile go to CU 0, which finishes
//       and stores the output.
// The exchange runs through global memory without fences or separate flags: every f32 travels in a
// 64-bit word together with a tag (mini-batch index + 1), written and polled with relaxed agent-scope
// atomics, so a word is either old or complete and the caches are never flushed or invalidated (an
// agent-scope release / acquire pair per mini-batch cost about 30 us here).  Lane l of wave I only
// ever waits for lane l of wave I of the other CU (A2: wave 2 for wave 2).  There is no workspace argument in ttt_mlp_fwd, so
// the exchange area is the unit's W2_out buffer, which is not needed until the final state is stored:
// everything a CU polls lies in the rows of W2_out that this CU itself overwrites at the end, so its
// final store is ordered after its last read by program order, and the partner never writes there
// again after its last mini-batch.  The host zeroes W2_out (tag 0 = nothing sent) before the launch.
// Pairs are blocks (i, i + 8): with workgroups dealt round-robin to the eight XCDs both land on the
// same XCD (shared L2), and the exchange then never leaves that L2 (workgroup-scope stores, see send_tagged).
// That placement is checked, not assumed: at start the two workgroups tell each other which XCD they run on
// (device-scope words), and a pair that sits on two XCDs stores at device scope for the whole launch -- slower,
// same results.  Every wait for the partner is bounded, so a missing partner ends in NaN outputs, never in a hang.
//
// What bounds it.  The products by the issue of a SIMD's two waves, as in ttt_mlp_fwd_rr.hip.h; between the first and the
// second barrier a round trip through the L2, about 1.6 k cycles from the send to the tile in registers.  Cycles of a
// mini-batch at d = 128 with all 256 CUs at work, before -> after the last revision: A 4.0 -> 5.2 k (XQ W1 moved here, where
// it shares XK W1's operands), B 8.9 -> 4.0 k, C 1.8 -> 1.1 k, D 5.8 -> 6.7 k (CU 0; CU 1 6.0 k).  What it took in B: one load
// of the tile when it is needed instead of a watch on one word first, the words of a tile next to each other in each load,
// loads of a sum issued together, A2 and M1 formed by the older waves, which would wait at the first barrier, and the output
// finished a phase later, its stores where the waves wait for the partner.  128 units x 2048 tokens: d = 128 1078 -> 826 us,
// d = 96 838 -> 623 us.
#pragma once
#include "ttt_mlp_fwd_rr.hip.h"

namespace ttt {

template <int D, int ES>
struct MlpCl2Lds {
  static constexpr int NW = D / 16, NT = D / 16, FH = 2 * D;  // FH: hidden units of one CU; one wave per d-feature tile
  static constexpr int TILE = 16 * D * ES;
  static constexpr int IN1 = 3 * TILE;
  static constexpr int IN = 0;                  // [2 buffers][3][16][d]
  static constexpr int LR = IN + 2 * IN1;       // [2][16] floats
  static constexpr int P1 = LR + 2 * 64 + 128;  // [NW][NT][64] f32x4: partial Z2^T tiles
  static constexpr int P2 = P1 + NW * NT * 1024;  // [NW][NT][64] bf16x4: partial Zbar2^T tiles
  static constexpr int PA = P2 + NW * NT * 512;   // [NW][64] f32x4: partial A2^T
  static constexpr int EX = PA + NW * 1024;       // [6 sums][2][16 tokens] f32x4 (reducer index % 4)
  static constexpr int EXO = EX + 6 * 2 * 16 * 16;
  static constexpr int GT = EXO + 2 * 2 * 16 * 16;       // [2][NT][64] frag: G2^T tiles
  static constexpr int X2S = GT + 2 * NT * 64 * 4 * ES;  // [NW][FH / 16 / NW][64] frag: X2^T tiles
  static constexpr int M1 = X2S + FH / 16 * 64 * 4 * ES;  // [2][64] frag: M1 of this mini-batch
  static constexpr int M2 = M1 + 2 * 64 * 4 * ES;     // [64] frag: M2 of the previous one
  static constexpr int ID = M2 + 64 * 4 * ES;     // [64] frag: identity
  static constexpr int RHO = ID + 64 * 4 * ES;    // [16] token_eta / sc
  static constexpr int PRM = RHO + 64;            // gamma[d], beta[d], b1[FH] floats
  static constexpr int LOST = PRM + (2 * D + FH) * 4;  // one word: a wait for the partner ran out
  static constexpr int FL = LOST + 16;            // [NW] counters
  static constexpr int BYTES = FL + 32;
  static_assert(BYTES <= 160 * 1024, "exceeds the 160 KiB of LDS of a gfx950 CU");
  static_assert(NT == NW && NW <= 8 && D % 32 == 0 && ES == 2, "one reducer and one output tile per wave, bf16 I/O");
  static_assert(FH % (32 * NW) == 0, "an even number of hidden tiles per wave");
  static_assert(TILE % 1024 == 0 && P1 % 16 == 0, "input tiles are staged in 1 KiB wave blocks");
  // exchange area inside this CU's rows of W2_out (bytes): two parities of X1 tiles, X2 tiles, A2 tile,
  // each tile as 64 lanes x 4 tagged 64-bit words
  static constexpr int XTILE = 2048, XSLOT = (2 * NT + 1) * XTILE;
  static constexpr int XHELLO = 2 * XSLOT;  // one tagged word behind the tiles: the partner's XCD
  static_assert(XHELLO + 16 <= FH * D * 4, "exchange area exceeds this CU's rows of W2_out");
};

// One [16 x 16] f32 tile (this lane's four values) as four (value, tag) words, value r of lane l at word 64 r + l.
// The two workgroups of a pair sit on CUs of one XCD (see the block numbering in the kernel), which share an L2.
// The stores therefore carry workgroup scope: they leave the CU (its L1 writes through) and stay in that L2, where
// the partner's device-scope loads, which bypass its own L1, find them.  Device-scope stores would also be written
// through to memory, every one of them: measured at 2.8 GB of writes per launch of 128 units x 2048 tokens, which
// made the kernel 40 % slower on a full GPU than on a quarter of it.  `same_xcd` is what the two workgroups found
// out about each other at start (see the kernel): a pair on two XCDs stores at device scope.
__device__ __forceinline__ void send_tagged(unsigned long long* slot, f32x4 v, unsigned tag, bool same_xcd) {
  if (same_xcd) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      __hip_atomic_store(slot + 64 * r, ((unsigned long long)tag << 32) | __float_as_uint(v[r]), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WORKGROUP);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      __hip_atomic_store(slot + 64 * r, ((unsigned long long)tag << 32) | __float_as_uint(v[r]), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
}
// A tile on its way in: the four words as last loaded.
struct Inbound {
  unsigned long long wd[4];
  __device__ __forceinline__ void load(const unsigned long long* slot) {
#pragma unroll
    for (int r = 0; r < 4; ++r) wd[r] = __hip_atomic_load(slot + 64 * r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // Loads again until the four words of every lane carry the tag.  The wait is bounded; after one wait has run out
  // (`alive` cleared) no further wait is attempted: a lost partner costs one time-out per wave, not one per
  // mini-batch, and ends in NaN outputs, never in a hang.
  __device__ __forceinline__ f32x4 wait(const unsigned long long* slot, unsigned tag, bool& alive, int spin_limit) {
    int it = 0;
    while (true) {
      bool ok = true;
#pragma unroll
      for (int r = 0; r < 4; ++r) ok = ok && (unsigned)(wd[r] >> 32) == tag;
      // the whole wave leaves together: its lanes poll neighbouring words of the same tile
      if (__all(ok) || !alive) break;
      if (++it >= spin_limit) {
        alive = false;
        break;
      }
      load(slot);
    }
    return f32x4{__uint_as_float((unsigned)wd[0]), __uint_as_float((unsigned)wd[1]), __uint_as_float((unsigned)wd[2]),
                 __uint_as_float((unsigned)wd[3])};
  }
};

// see ttt_mlp_fwd_rr.hip.h: lane coordinates and constants held across the loop spill here as well (62 registers)
#define RELANE()                       \
  do {                                 \
    asm volatile("" : "+v"(lane));     \
    c = lane & 15;                     \
    g = lane >> 4;                     \
    own = own_offset<1>(w, 0, g);      \
  } while (0)

template <class T, int D>
__global__ void __launch_bounds__(64 * (D / 16)) ttt_mlp_fwd_cl2_kernel(Problems<MlpFwdArgs> problems) {
  const MlpFwdArgs& a = problems.p[blockIdx.y];
  using IO = Io<T>;
  using frag = typename IO::frag;
  using elem = typename IO::elem;
  constexpr int ES = sizeof(elem);
  using L = MlpCl2Lds<D, ES>;
  constexpr int NW = L::NW, NT = D / 16, F = 4 * D, FH = L::FH, HT = FH / 16 / NW, NTHR = 64 * NW;
  constexpr float inv_d = 1.0f / D;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63;
  int c = lane & 15, g = lane >> 4;
  // blocks (i, i + 8) of every group of sixteen form a pair
  const int blk = blockIdx.x;
  const int cu = (blk >> 3) & 1;
  const size_t bh = (size_t)a.unit_base + (size_t)(blk >> 4) * 8 + (blk & 7);
  if (bh >= (size_t)a.B * a.H) return;
  int& lost = *reinterpret_cast<int*>(smem + L::LOST);  // set by a wave whose wait for the partner ran out
  if (tid == 0) lost = 0;
  const int h = (int)(bh % a.H), K = a.K, spin_limit = held(a.spin_limit);
  const float eps = held(a.eps);
  const int hoff = cu * FH;  // first hidden unit of this CU

  f32x4* const P1 = reinterpret_cast<f32x4*>(smem + L::P1);
  frag* const P2 = reinterpret_cast<frag*>(smem + L::P2);
  f32x4* const PA = reinterpret_cast<f32x4*>(smem + L::PA);
  float* const EX = reinterpret_cast<float*>(smem + L::EX);
  float* const EXO = reinterpret_cast<float*>(smem + L::EXO);
  frag* const GT = reinterpret_cast<frag*>(smem + L::GT);
  frag* const X2S = reinterpret_cast<frag*>(smem + L::X2S) + w * HT * 64;
  frag* const M1s = reinterpret_cast<frag*>(smem + L::M1);
  frag* const M2s = reinterpret_cast<frag*>(smem + L::M2);
  frag* const IDs = reinterpret_cast<frag*>(smem + L::ID);
  lds_int* const FL = (lds_int*)(smem + L::FL);
  float* const RHO = reinterpret_cast<float*>(smem + L::RHO);
  uint32_t* const LRs = reinterpret_cast<uint32_t*>(smem + L::LR);
  float* const GAM = reinterpret_cast<float*>(smem + L::PRM);
  float* const BET = GAM + D;
  float* const B1s = BET + D;  // this CU's half of b1

  // exchange areas: what this CU receives lies in its own rows of W2_out, what it sends in the partner's
  unsigned char* const xin = reinterpret_cast<unsigned char*>(a.W2 + (bh * F + hoff) * (size_t)D);
  unsigned char* const xout = reinterpret_cast<unsigned char*>(a.W2 + (bh * F + (FH - hoff)) * (size_t)D);

  // ---- which XCD does the partner run on?  One device-scope word each way (tag 0xffffffff: no mini-batch uses it),
  // sent before the state is loaded and read after, so the round trip costs nothing.  The answer decides the scope
  // of every later store to the partner.
  unsigned my_xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(my_xcc));
  my_xcc &= 15u;
  if (tid == 0)
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(xout + L::XHELLO), (0xffffffffull << 32) | my_xcc, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);

  const float te_last = a.token_eta[K - 1];
  const bool upd = te_last != 0.f;
  const float sc = upd ? te_last : 1.f;
  if (tid < 8) FL[tid] = tid < NW ? 0 : 0x7fffffff;
  if (tid < 16) RHO[tid] = tid < K ? a.token_eta[tid] / sc : 0.f;
  if (w == 0) IDs[lane] = identity_frag<T>(c, g);
  const size_t sb = a.state_per_batch ? bh : (size_t)h;
  int own = own_offset<1>(w, 0, g);  // first of this lane's four features of d-feature tile w

  // ---- state and parameters
  f32x4 W1c[NT][HT], W2c[HT][NT];
  {
    const float* W1 = a.W1_0 + sb * (size_t)D * F;
    const float* W2 = a.W2_0 + sb * (size_t)D * F;
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const int hb = hoff + 16 * (w * HT + j);
#pragma unroll
      for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          W1c[I][j][r] = W1[(size_t)feat(I, 4 * g + r) * F + hb + c];
          W2c[j][I][r] = W2[(size_t)(hb + 4 * g + r) * D + feat(I, c)];
        }
    }
  }
  f32x4 b2T;
  float sum_a = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) b2T[r] = a.b2_0[sb * D + own + r];
  // the second layer is carried centred (see row_means16 in ttt_mlp_fwd_rr.hip.h)
#pragma unroll
  for (int j = 0; j < HT; ++j) {
    const f32x4 m = row_means16<NT>(W2c[j], inv_d);
#pragma unroll
    for (int I = 0; I < NT; ++I) W2c[j][I] -= m;
  }
  b2T -= mean_of(a.b2_0 + sb * D, D, inv_d);
  for (int f = 0; f < D; ++f) sum_a += a.gamma[h * D + f] * a.gamma[h * D + f];
  sum_a = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(sum_a)));
  for (int i = tid; i < D; i += NTHR) {
    GAM[i] = a.gamma[h * D + i];
    BET[i] = a.beta[h * D + i];
  }
  for (int i = tid; i < FH; i += NTHR) B1s[i] = a.b1_0[sb * F + hoff + i];

  // ---- staging of the xq / xk / xv rows: global -> LDS, two buffers.  The fetch of mini-batch st+1 is
  // issued after the first barrier of mini-batch st (every wave has then finished reading the buffer it
  // overwrites) and has landed before the third.
  // Per wave block a running source address, scalar like everything but the lane's offset.
  constexpr int NBLK = L::IN1 / 1024, NBI = (NBLK + NW - 1) / NW;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem);
  const unsigned step = (unsigned)(K * D * ES);
  const size_t unit0 = bh * (size_t)a.seq_stride * (D * ES);
  const unsigned char* srcp[NBI];
#pragma unroll
  for (int it = 0; it < NBI; ++it) {
    const int b = w + NW * it, ten = (1024 * b) / L::TILE;
    srcp[it] = static_cast<const unsigned char*>(ten == 0 ? a.xq : ten == 1 ? a.xk : a.xv) + unit0;
  }
  const unsigned char* lrp = static_cast<const unsigned char*>(a.lr) + bh * (size_t)a.seq_stride * ES;
  unsigned char* const outp = static_cast<unsigned char*>(a.out) + unit0;
  const int n_stages = a.n_stages;
  auto fetch = [&](int stage) {
    if (stage >= n_stages) return;
    const unsigned dst = lds0 + L::IN + (stage & 1) * L::IN1 + 1024 * w;
#pragma unroll
    for (int it = 0; it < NBI; ++it) {
      const int b = w + NW * it;
      const unsigned off = (1024u * b) % L::TILE + 16u * lane;
      if (b < NBLK && off < step) lds_dma16(srcp[it], off, dst + 1024 * NW * it);
      srcp[it] += step;
    }
    // lr as zero-extended bf16 words, copied like the tiles (a register load here would make the compiler
    // wait for every copy in flight); absent tokens read a clamped position and are zeroed at use
    if (w == 0 && lane < 16) lds_dma2(lrp, 2u * (unsigned)min(lane, K - 1), lds0 + L::LR + (stage & 1) * 64);
    lrp += K * ES;
  };
  auto row = [&](int buf, int ten) -> const elem* {
    return reinterpret_cast<const elem*>(smem + L::IN + buf * L::IN1 + ten * L::TILE) + c * D;
  };

  for (int i = tid; i < (L::P1 - L::IN) / 4; i += NTHR) reinterpret_cast<float*>(smem)[i] = 0.f;
  for (int i = tid; i < 6 * 2 * 16 * 4; i += NTHR) EX[i] = 0.f;
  if (tid < 2 * 2 * 16 * 4) EXO[tid] = 0.f;
  int& partner_xcc = *reinterpret_cast<int*>(smem + L::LOST + 4);  // -1: the partner never said
  if (tid == 0) {
    const unsigned long long* hello = reinterpret_cast<const unsigned long long*>(xin + L::XHELLO);
    unsigned long long wd = 0;
    int it = 0;
    while ((unsigned)((wd = __hip_atomic_load(hello, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >> 32) != 0xffffffffu) {
      if (++it >= spin_limit) break;
      __builtin_amdgcn_s_sleep(1);
    }
    partner_xcc = (unsigned)(wd >> 32) == 0xffffffffu ? (int)(wd & 15u) : -1;
  }
  __syncthreads();
  // a partner that never said where it runs is treated like one on another XCD; the first wait for it will run out
  const bool same_xcd = !a.assume_other_xcd && __builtin_amdgcn_readfirstlane(partner_xcc) == (int)my_xcc;
  fetch(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  auto publish = [&](const float (&S)[6]) {
    const float v0 = xg_sum4_scatter(S[0], S[1], S[2], S[3]);
    const float v1 = xg_sum2_scatter(S[4], S[5]);
    EX[(((g)*2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = v0;
    EX[(((4 + (g >> 1)) * 2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = v1;  // two lane groups write the same value
  };  // (with this and every sum from its first term, same bits: 128 units x 2048 tokens, d = 96 615 -> 608 us, d = 128 812 -> 807)
  // sums i and j of those exchanged at ex
  auto collect2 = [&](const float* ex, int i, int j, float& a, float& b) {
    f32x4 v[4];
    v[0] = *reinterpret_cast<const f32x4*>(ex + ((i * 2 + 0) * 16 + c) * 4);
    v[1] = *reinterpret_cast<const f32x4*>(ex + ((j * 2 + 0) * 16 + c) * 4);
    v[2] = *reinterpret_cast<const f32x4*>(ex + ((i * 2 + 1) * 16 + c) * 4);
    v[3] = *reinterpret_cast<const f32x4*>(ex + ((j * 2 + 1) * 16 + c) * 4);
    together(v);
    a = ((v[0][0] + v[0][1]) + (v[0][2] + v[0][3])) + ((v[2][0] + v[2][1]) + (v[2][2] + v[2][3]));
    b = ((v[1][0] + v[1][1]) + (v[1][2] + v[1][3])) + ((v[3][0] + v[3][1]) + (v[3][2] + v[3][3]));
  };
  // tile slot `idx` of parity `par`: X1 tiles 0..NT-1, X2 tiles NT..2NT-1, the A2 tile 2NT
  bool alive = spin_limit > 0;
  auto send_tile = [&](int par_, int idx, f32x4 v, unsigned tag) {
    send_tagged(reinterpret_cast<unsigned long long*>(xout + par_ * L::XSLOT + idx * L::XTILE) + lane, v, tag, same_xcd);
  };
  auto slot_in = [&](int par_, int idx) -> const unsigned long long* {
    return reinterpret_cast<const unsigned long long*>(xin + par_ * L::XSLOT + idx * L::XTILE) + lane;
  };

  // ---- output path, wave w owns d-feature tile w.  While the Z2 tiles of mini-batch t + 1 cross, each CU sums its partial
  // Zbar2 tiles of t and CU 1 sends its half off; CU 0 adds it in phase D, applies the causal correction and forms the row
  // moments, and stores the output while the tiles of t + 2 cross.  A2 is summed by wave 2 of each CU at the end of phase
  // A, as soon as every wave has written its partial block.  There is no barrier between: each wave waits for its block to
  // be in LDS (lds_done) and then counts up its own word there, which wave 2 reads.  Block and word both have to be LDS
  // instructions (FL carries the address space: through a generic pointer the word goes another way than the block).  This
  // wait needs no bound: on its way from B3 to the counter a wave waits for nothing but, bounded, the partner's tile.
  f32x4 zb = {0.f, 0.f, 0.f, 0.f};
  frag qo1 = IO::zero(), qo2 = qo1;  // xq tiles of the last mini-batch and of the one before
  auto a2_sum = [&]() -> f32x4 {
    f32x4 v[NW];
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) v[ww] = PA[ww * 64 + lane];
    together(v);
    return sum_tiles(v);
  };
  auto a2_early = [&](int stage) -> f32x4 {
    while (__builtin_amdgcn_ballot_w64(__hip_atomic_load(FL + (lane & 7), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= stage) != 0) {
    }
    lds_done();
    const f32x4 at = a2_sum();
    if (cu == 1) send_tile(stage & 1, 2 * NT, at, (unsigned)stage + 1);
    return at;
  };
  auto output_local = [&](int stage) {
    const int par_ = stage & 1;
    frag v[NW];
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) v[ww] = P2[(ww * NT + w) * 64 + lane];
    zb = IO::to_f32(v[0]);
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) zb += IO::to_f32(v[ww]);
    pin(zb);
    if (cu == 1) send_tile(par_, NT + w, zb, (unsigned)stage + 1);
  };
  // wave 2 of CU 0: M2[s][t] = (token_eta[t] / sc)(1 + A2[t][s]) for s <= t
  auto output_m2 = [&](f32x4 at) {
    const float rho_c = RHO[c];
    f32x4 m;
#pragma unroll
    for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? rho_c * (1.f + at[r]) : 0.f;
    M2s[lane] = IO::to_frag(m);
  };
  // CU 0: add CU 1's half, causal correction, row moments
  auto output_finish = [&](int stage, f32x4 zb_part) {
    zb += zb_part;
    IO::mma(zb, read_tr(GT + ((stage & 1) * NT + w) * 64 + tr_lane(lane)), M2s[lane]);
    float s0;
#pragma unroll
    for (int r = 0; r < 4; ++r) sum_term(s0, r == 0, zb[r]);
    EXO[(((g >> 1) * 2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = xg_sum2_scatter(s0, sum_squares(zb));
  };
  auto output_emit = [&](int stage) {
    float mu, ms;
    collect2(EXO, 0, 1, mu, ms);
    mu *= inv_d;
    const float rstd = __builtin_amdgcn_rsqf(fmaxf(ms * inv_d - mu * mu, 0.f) + eps);
    if (c < K) {
      const f32x4 gam = *reinterpret_cast<const f32x4*>(GAM + own), bet = *reinterpret_cast<const f32x4*>(BET + own);
      elem* po = reinterpret_cast<elem*>(outp + (size_t)stage * step) + (c * D + own);
      store4<T>(po, IO::to_f32(qo2) + bet + gam * ((zb - mu) * rstd));
    }
  };
  // partial tiles of X W2 over this wave's hidden units, two at a time (HT is even here)
  auto partials = [&](const frag (&x)[HT], auto put) {
#pragma unroll
    for (int I = 0; I < NT; I += 2) {
      f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
#pragma unroll
      for (int j = 0; j < HT; j += 2) {
        IO::mma2(p0, IO::to_frag(W2c[j][I]), IO::to_frag(W2c[j + 1][I]), x[j], x[j + 1]);
        IO::mma2(p1, IO::to_frag(W2c[j][I + 1]), IO::to_frag(W2c[j + 1][I + 1]), x[j], x[j + 1]);
      }
      put(I, p0);
      put(I + 1, p1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  for (int st = 0; st < n_stages; ++st) {
    const int buf = st & 1, par = st & 1;
    frag* const GTc = GT + par * NT * 64;
    RELANE();

    // ================= phase A: everything that needs only W1, W2 and the inputs
    f32x4 z1[HT], zq[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) zq[j] = z1[j] = *reinterpret_cast<const f32x4*>(B1s + 16 * (w * HT + j) + 4 * g);
#pragma unroll
    for (int q = 0; q < NT / 2; ++q) {
      frag k0, k1, q0, q1;
      IO::load8(row(buf, 1) + 32 * q + 8 * g, true, k0, k1);
      IO::load8(row(buf, 0) + 32 * q + 8 * g, true, q0, q1);
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        const frag w0 = IO::to_frag(W1c[2 * q][j]), w1 = IO::to_frag(W1c[2 * q + 1][j]);
        IO::mma2(z1[j], w0, w1, k0, k1);
        IO::mma2(zq[j], w0, w1, q0, q1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    frag x2f[HT];
    f32x4 dg[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      f32x4 y, dy;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float yy, dd;
        gelu_fast_pair(z1[j][r], yy, dd);
        y[r] = yy;
        dy[r] = dd;
      }
      x2f[j] = IO::to_frag(y);
      dg[j] = dy;
      asm volatile("" : "+v"(x2f[j]), "+v"(dg[j]));
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < HT; ++j) X2S[j * 64 + lane] = x2f[j];
    partials(x2f, [&](int I, f32x4 p) { P1[(w * NT + I) * 64 + lane] = p; });
    f32x4 at = {0.f, 0.f, 0.f, 0.f};
    if (w == 2 && st > 0) at = a2_early(st - 1);
    // M1[s][t] = (token_eta[t] / sc)(1 + A1[t][s]) for s <= t
    if (w == 3) {
      const float rho_c = RHO[c];
      f32x4 At = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < NT / 2; ++q) {
        frag k0, k1, q0, q1;
        IO::load8(row(buf, 1) + 32 * q + 8 * g, true, k0, k1);
        IO::load8(row(buf, 0) + 32 * q + 8 * g, true, q0, q1);
        IO::mma2(At, k0, k1, q0, q1);
      }
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? rho_c * (1.f + At[r]) : 0.f;
      M1s[par * 64 + lane] = IO::to_frag(m);
    }
    lds_barrier();  // ---- B1
    RELANE();

    // ================= phase B: this CU's half of Z2 tile w, exchange with the partner, row moments
    f32x4 z, bq;
    Inbound zb_in;
    {
      f32x4 zloc;
      {
        f32x4 v[NW];
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) v[ww] = P1[(ww * NT + w) * 64 + lane];
        together(v);
        zloc = sum_tiles(v);
      }
      send_tile(par, w, zloc, (unsigned)st + 1);
      // everything that does not need the partner goes between the send and the wait: the local half of the previous
      // output
      if (cu == 0 && st > 1) output_emit(st - 2);
      if (st > 0) output_local(st - 1);
      const frag ko = load4<T>(row(buf, 1) + own), vo = load4<T>(row(buf, 2) + own);
      const f32x4 gam = *reinterpret_cast<const f32x4*>(GAM + own), bet = *reinterpret_cast<const f32x4*>(BET + own);
      const f32x4 tgt = bet - (IO::to_f32(vo) - IO::to_f32(ko));
      bq = gam * tgt;
      const bool m2w = cu == 0 && w == 2 && st > 0;  // CU 1 sent its A2 before its Z2 tiles
      Inbound in, in2;
      in.load(slot_in(par, w));
      if (m2w) in2.load(slot_in(par ^ 1, 2 * NT));
      const f32x4 zpart = in.wait(slot_in(par, w), (unsigned)st + 1, alive, spin_limit);
      z = b2T + (cu == 0 ? zloc + zpart : zpart + zloc);  // same order of the halves on both CUs
      float S[6];
      const f32x4 a2 = gam * gam, az = a2 * z;
      S[1] = sum_squares(z);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sum_term(S[0], r == 0, z[r]);
        sum_term(S[2], r == 0, a2[r], z[r]);
        sum_term(S[3], r == 0, az[r], z[r]);
        sum_term(S[4], r == 0, gam[r], tgt[r]);
        sum_term(S[5], r == 0, bq[r], z[r]);
      }
      publish(S);
      if (cu == 0 && st > 0) {
        if (m2w) output_m2(at + in2.wait(slot_in(par ^ 1, 2 * NT), (unsigned)st, alive, spin_limit));
        zb_in.load(slot_in(par ^ 1, NT + w));
      }
      fetch(st + 1);
    }
    lds_barrier();  // ---- B2
    RELANE();

    // ================= phase C: G2''
    {
      const float lrc = (c < K) ? __uint_as_float(LRs[buf * 16 + c] << 16) : 0.f;
      float S[6];
      {
        // lane group g adds up sums g and 4 + (g & 1), then all groups get all six
        float v0, v1;
        collect2(EX, g, 4 + (g & 1), v0, v1);
        const uint32_t u = __float_as_uint(v0), v = __float_as_uint(v1);
        const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);  // rows: 0 0 2 2 / 1 1 3 3
        const uint32_t p0 = p[0], p1 = p[1];
        const auto q = __builtin_amdgcn_permlane32_swap(p0, p0, false, false);
        const auto r = __builtin_amdgcn_permlane32_swap(p1, p1, false, false);
        const auto t2 = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // rows: 4 4 4 4 / 5 5 5 5
        const uint32_t q0 = q[0], q1 = q[1], r0 = r[0], r1 = r[1], t0 = t2[0], t1 = t2[1];
        S[0] = __uint_as_float(q0);
        S[2] = __uint_as_float(q1);
        S[1] = __uint_as_float(r0);
        S[3] = __uint_as_float(r1);
        S[4] = __uint_as_float(t0);
        S[5] = __uint_as_float(t1);
      }
      const float mu = S[0] * inv_d;
      const float var = S[1] * inv_d - mu * mu;
      const float rstd = __builtin_amdgcn_rsqf(fmaxf(var, 0.f) + eps);
      const float s1 = rstd * (S[2] - mu * sum_a) + S[4];
      const float m5 = S[5] - mu * S[4], q3 = S[3] - 2.f * mu * S[2] + mu * mu * sum_a, r2 = rstd * rstd;
      const float s2 = __builtin_fmaf(m5, rstd, r2 * q3);
      const float p = -sc * lrc * rstd;
      const float c1 = p * rstd, c2 = -c1 * s2 * inv_d, c3 = -p * s1 * inv_d;
      const f32x4 gam = *reinterpret_cast<const f32x4*>(GAM + own);
      const f32x4 G = (z - mu) * (gam * gam * c1 + c2) + (bq * p + c3);
      GTc[w * 64 + lane] = IO::to_frag(G);
    }
    // the next mini-batch's rows must have landed before anybody passes B3
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();  // ---- B3
    RELANE();

    // ================= phase D: G1, Zbar1, Xbar2, split-k partials of the output path, updates
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W2c[j][I]);
    // G1''^T = (W2 G2''^T) gelu'(Z1)
    frag G1d[HT];
    {
      const frag ident = IDs[lane];
      f32x4 acc[HT];
#pragma unroll
      for (int j = 0; j < HT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < NT / 2; ++q) {
        const frag g0 = GTc[(2 * q) * 64 + lane], g1 = GTc[(2 * q + 1) * 64 + lane];
        f32x4 t0[HT], t1[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          t0[j] = t1[j] = f32x4{0.f, 0.f, 0.f, 0.f};
          IO::mma(t0[j], IO::to_frag(W2c[j][2 * q]), ident);
          IO::mma(t1[j], IO::to_frag(W2c[j][2 * q + 1]), ident);
        }
#pragma unroll
        for (int j = 0; j < HT; ++j) IO::mma2(acc[j], IO::to_frag(t0[j]), IO::to_frag(t1[j]), g0, g1);
        __builtin_amdgcn_sched_barrier(0);
      }
      f32x4 t[HT];
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        t[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        IO::mma(t[j], IO::to_frag(acc[j] * dg[j]), ident);
      }
#pragma unroll
      for (int j = 0; j < HT; ++j) G1d[j] = IO::to_frag(t[j]);
    }
    // Zbar1^T = (XQ W1 + b1)^T + G1''^T M1
    {
      const frag Mf = M1s[par * 64 + lane];
#pragma unroll
      for (int j = 0; j < HT; ++j) IO::mma(zq[j], G1d[j], Mf);
    }
    if (cu == 0) {
      if (st > 0) output_finish(st - 1, zb_in.wait(slot_in(par ^ 1, NT + w), (unsigned)st, alive, spin_limit));
      qo2 = qo1;
      qo1 = load4<T>(row(buf, 0) + own);
    }
    frag xbf[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      f32x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = gelu_fast(zq[j][r]);
      xbf[j] = IO::to_frag(y);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W2c[j][I]);
    {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < HT; j += 2) IO::mma2(p, x2f[j], x2f[j + 1], xbf[j], xbf[j + 1]);
      PA[w * 64 + lane] = p;
      lds_done();  // the block is in LDS before its counter says so
      if (lane == 0) __hip_atomic_store(FL + w, st + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    // (b2 enters the sum once: through wave I of CU 0)
    partials(xbf, [&](int I, f32x4 p) { P2[(w * NT + I) * 64 + lane] = IO::to_frag(I == w && cu == 0 ? p + b2T : p); });
    if (upd) {
      frag x2d[HT];
      {
        const frag ones = splat_frag<T>(1.f);
        f32x4 b[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          x2d[j] = read_tr(X2S + j * 64 + tr_lane(lane));
          b[j] = *reinterpret_cast<const f32x4*>(B1s + 16 * (w * HT + j) + 4 * g);
        }
#pragma unroll
        for (int j = 0; j < HT; ++j) IO::mma(b[j], G1d[j], ones);
#pragma unroll
        for (int j = 0; j < HT; ++j)
          if (c == 0) *reinterpret_cast<f32x4*>(B1s + 16 * (w * HT + j) + 4 * g) = b[j];
      }
      // XK tiles with tokens along k, straight from the staged rows: lane l supplies four features of token 4g + c / 4
      const elem* const kr = reinterpret_cast<const elem*>(smem + L::IN + buf * L::IN1 + L::TILE) + (4 * g + (c >> 2)) * D + 8 * (c & 3);
      const frag* const gr = GTc + tr_lane(lane);
      frag kd = read_tr(kr), g2d = read_tr(gr);
#pragma unroll
      for (int I = 0; I < NT; ++I) {
        const int In = I + 1 < NT ? I + 1 : I;
        const frag kn = read_tr(kr + 32 * (In >> 1) + 4 * (In & 1)), gn = read_tr(gr + (I + 1 < NT ? I + 1 : w) * 64);
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          IO::mma(W1c[I][j], kd, G1d[j]);
          IO::mma(W2c[j][I], x2d[j], g2d);
        }
        kd = kn;
        g2d = gn;
        __builtin_amdgcn_sched_barrier(0);
      }
      IO::mma(b2T, g2d, splat_frag<T>(1.f));
    }
  }

  // ---- the last mini-batch's output
  lds_barrier();
  if (cu == 0 && n_stages > 1) output_emit(n_stages - 2);
  qo2 = qo1;
  output_local(n_stages - 1);
  f32x4 at = {0.f, 0.f, 0.f, 0.f};
  if (w == 2) at = a2_early(n_stages - 1);
  if (cu == 0 && w == 2) {
    const unsigned long long* const sl = slot_in((n_stages - 1) & 1, 2 * NT);
    Inbound in;
    in.load(sl);
    output_m2(at + in.wait(sl, (unsigned)n_stages, alive, spin_limit));
  }
  lds_barrier();
  if (cu == 0) {
    const unsigned long long* const sl = slot_in((n_stages - 1) & 1, NT + w);
    Inbound in;
    in.load(sl);
    output_finish(n_stages - 1, in.wait(sl, (unsigned)n_stages, alive, spin_limit));
  }
  lds_barrier();
  if (cu == 0) output_emit(n_stages - 1);

  // ---- final state: this CU's hidden half.  Its rows of W2_out held the exchange area; every read of
  // it by this workgroup is above, every write of the partner into it was awaited above.
  if (!alive) lost = 1;
  __syncthreads();
  // A wait for the partner that ran out (the two workgroups of a pair were not resident together long enough)
  // must not pass for a result: the workgroup that saw it turns everything it owns of the unit into NaN -- its
  // half of W1, b1, W2, b2 and the whole output of the unit (both workgroups do, as a rule: the partner then finds
  // NaN tags where it polls and times out too).  The caller sees NaN in every output tensor of that unit.
  const float poison = lost ? __builtin_nanf("") : 0.f;
  {
    float* W1 = a.W1 + bh * (size_t)D * F;
    float* W2 = a.W2 + bh * (size_t)D * F;
    const float* W2i = a.W2_0 + sb * (size_t)D * F;
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const int hb = hoff + 16 * (w * HT + j);
      // second layer: initial value + (centred value now - centred value at the start); see ttt_mlp_fwd_rr.hip.h
      f32x4 w0[NT];
#pragma unroll
      for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) w0[I][r] = W2i[(size_t)(hb + 4 * g + r) * D + feat(I, c)];
      const f32x4 m = row_means16<NT>(w0, inv_d);
#pragma unroll
      for (int I = 0; I < NT; ++I) {
        const f32x4 start = w0[I] - m;
        const f32x4 fin = w0[I] + (W2c[j][I] - start);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          W1[(size_t)feat(I, 4 * g + r) * F + hb + c] = W1c[I][j][r] + poison;
          W2[(size_t)(hb + 4 * g + r) * D + feat(I, c)] = fin[r] + poison;
        }
      }
      if (c == 0)
        store4<F32>(a.b1 + bh * F + hb + 4 * g, *reinterpret_cast<const f32x4*>(B1s + 16 * (w * HT + j) + 4 * g) + poison);
    }
    {
      const float bb = mean_of(a.b2_0 + sb * D, D, inv_d);
      const f32x4 v0 = *reinterpret_cast<const f32x4*>(a.b2_0 + sb * D + own);
      const f32x4 start = v0 - bb;
      if ((cu == 0 || lost) && c == 0) store4<F32>(a.b2 + bh * D + own, v0 + (b2T - start) + poison);
    }
    if (lost) {
      if (tid == 0) atomicAdd(&g_mlp_fwd_lost_workgroups, 1u);
      elem* po = static_cast<elem*>(a.out) + bh * (size_t)a.seq_stride * D;
      const size_t n = (size_t)a.n_stages * K * D;
      for (size_t i = tid; i < n; i += NTHR) IO::store1(po + i, poison);
    }
  }
}

#undef RELANE

}  // namespace ttt
