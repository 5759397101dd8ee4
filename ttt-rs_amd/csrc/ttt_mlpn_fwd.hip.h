// TTT-MLP with NL hidden layers (NL = 2, 3, 4), multi-stage forward: the reference's TTTMLP2 / TTTMLP3 / TTTMLP4 inner
// models (rust/core/src/mlp2.rs:152-243, mlp3.rs:162-279, mlp4.rs:186-324) looped as rust/core/src/inner.rs:25-50.
// The reference has no fused kernel for them; this is their Burn-op mini-batch restated as one persistent kernel with the
// weights in registers, the NL-layer generalisation of the loop that ttt_mlp_fwd_kernel (ttt_engine_fwd.hip.h) runs on tiles
// in memory:
//
//   weight layer i = 0 .. NL:  W[i] [in_i x out_i], in_0 = d, out_NL = d, every other side M = 4 d
//   forward chain   X[0] = XK;  Z[i] = X[i] W[i] + b[i];  X[i+1] = gelu(Z[i])  (i < NL)
//   gradients       G[NL] = LN-L2 gradient of Z[NL] against XV - XK;  G[i] = (G[i+1] W[i+1]^T) * gelu'(Z[i])
//   output chain    Xb[0] = XQ;  Zb[i] = Xb[i] W[i] - (eta (1 + tril(Xb[i] X[i]^T))) G[i] + b[i];  Xb[i+1] = gelu(Zb[i])
//   out = XQ + LN(Zb[NL]);   W[i] -= (eta_last X[i])^T G[i];   b[i] -= colsum(eta_last G[i])
//
// One workgroup of 8 waves per (batch, head).  The weights stay in registers over the whole sequence, as accumulator
// tiles of the f32 matrix instructions: register r of lane 16 g + c holds row 4 g + r, column c of a 16 x 16 tile, which
// is at the same time a B operand over the rows (k step r takes row 4 g + r; the A operand is one 16-byte LDS read for
// four k steps) and the accumulator of the rank-16 update.  A wave owns M / 8 hidden columns: the same columns of
// W[0 .. NL-1] and the same rows of W[NL], so that elementwise work, gradients, biases and updates of a layer need no
// exchange; products over k = M take the other waves' columns of X from LDS, products with W[NL] and the attention
// blocks are summed over the waves.  G[i+1] W[i+1]^T contracts over the columns, the one product the layout does not
// give: the tiles go through LDS (CH tile rows at a time) and are read back transposed.  (By 32 columns, written by two
// waves while the others multiply the chunk before, half the barriers: 2138 us against 2087; the two writers hold up the
// rest.)  At head_dim 64 all of it is 192 registers of a wave's 256; W[0], 32 of them, is therefore written to the output
// buffer at the end of a mini-batch and read back for the next update.
//
// Bound by the f32 matrix instructions, 774 per wave and mini-batch at head_dim 64 with two hidden layers: two waves to
// a SIMD, 32 cycles each, 20.6 of 32.2 us at 2.4 GHz; the rest are the barriers and the activations between the
// products.  96 units of 64 mini-batches, bf16: 3128 us with the state read from the L2 for every product and update,
// 2062 so.  All products are f32 for both I/O types.  LDS bounds the shapes: head_dim 32 with up to four hidden layers,
// head_dim 64 with two.
//
// A unit on two workgroups (ttt_mlpn_fwd_pair_kernel), where the device has two CUs for each.  Nothing of the output chain is
// needed for the state, so one workgroup, the producer, runs the forward chain, the gradients and the updates; the other, the
// consumer, takes X[i] and G[i] from it, runs the output chain and the same updates on a state of its own (542 and 424
// matrix instructions per wave and mini-batch).  Nothing flows back, so neither waits for a round trip of the other: the
// producer runs up to SLOTS mini-batches ahead.  Wave w hands over to wave w in the layout of its registers, through a ring in
// the unit's W_out (MlpNPair); two words per pair of waves say how far each has come.  The producer's stores stay in the L2 that
// both share (each publishes its XCD number) or are written back by a device-scope release while that is not known; the
// consumer loads at device scope.  Every wait is bounded: a side that waits in vain marks its words, both run to their end
// without waiting, the consumer marks the unit in W[NL], and a status word counts both.  A launch of the one-workgroup kernel
// behind the pair's does the marked units again, from inputs that no output overlaps (the caller's rule), and finds none where
// nothing held the device's CUs for seconds: 1.5 us.
// The arithmetic is that of one workgroup, bit for bit.  64 mini-batches of 16 tokens, bf16, us on one / on two workgroups:
// head_dim 64, 12 units 2066 / 1505, 96 units 2094 / 1533, 128 units 2093 / 1543; head_dim 32, 96 units two hidden layers
// 704 / 523, three 1069 / 804, four 1429 / 1063.
#pragma once
#include "ttt_engine_fwd.hip.h"

namespace ttt {

constexpr int kMlpNMaxLayers = 5;  // weight layers of the deepest variant (four hidden layers)

struct MlpNFwdArgs {
  const void* xq;
  const void* xk;
  const void* xv;
  const float* W0[kMlpNMaxLayers];  // initial state of weight layer i: [H,in,out] or [B,H,in,out]
  const float* b0[kMlpNMaxLayers];  // [H,out] or [B,H,out]
  float* W[kMlpNMaxLayers];         // [B,H,in,out]: live state during the call, final state after it
  float* b[kMlpNMaxLayers];         // [B,H,out]
  const float* token_eta;
  const void* lr;
  const float* gamma;
  const float* beta;
  void* out;
  int B, H, seq, seq_stride, K, n_stages, state_per_batch;  // seq_stride: tokens between consecutive (b, h) units
  float eps;
  // a unit on two workgroups
  unsigned spin_limit;   // polls before a wait for the partner gives up; 0: give up at once (tests of that path)
  int agent_release;     // 1: always publish with a device-scope release
  unsigned* lost_count;  // counts workgroups that waited in vain
  int only_lost;         // 1: the launch behind the pair's, for the units marked kMlpNLost
};

template <int D, int NL>
struct MlpNLds {
  static constexpr int NW = 8, M = 4 * D, LD = D + 4, LM = M + 4;  // pitches: 4 mod 16 banks, 16-byte rows
  static constexpr int TD = 16 * LD, TM = 16 * LM;
  static constexpr int NTD = D / 16, NTM = M / 16, NBM = NTM / NW;
  static constexpr int CH = D == 32 ? NTM : 4;  // tile rows of W[i+1] in LDS at a time for G[i+1] W[i+1]^T
  static constexpr int XI = 0;                  // X[1 .. NL]
  static constexpr int GT = XI + NL * TM;       // G[i+1] as an operand
  // one after the other: partials of Z[NL]; W[NL] transposed per wave; W[i+1] transposed and its partials; Xb[i] (two,
  // in turn) beside the partials of Zb[NL]
  static constexpr int POOL = GT + TM, PZ = POOL + 2 * TM;
  static constexpr int S0 = CH * 16 * LM, S1 = NW * NBM * 16 * LD, S2 = 2 * TM + NW * NTD * 256, S3 = 4 * TM;
  static constexpr int S01 = S0 > S1 ? S0 : S1, S23 = S2 > S3 ? S2 : S3, POOL_N = S01 > S23 ? S01 : S23;
  static constexpr int XQ = POOL + POOL_N, XK = XQ + TD, TG = XK + TD, ZL = TG + TD, ZBL = ZL + TD;
  static constexpr int PART = ZBL + TD;         // partials of an attention block, two blocks in turn
  static constexpr int bl = PART + 2 * NW * 256;  // bias of the last layer
  static constexpr int gam = bl + D, bet = gam + D, lr = bet + D, te = lr + 16, END = te + 16;
  static constexpr size_t BYTES = sizeof(float) * END;
  static_assert(BYTES <= 160 * 1024, "exceeds the 160 KiB of LDS of a gfx950 CU");
};

// What crosses between the two workgroups of a unit lies in its W_out until the consumer stores the final state over it: a
// ring of SLOTS mini-batches of X[1 .. NL] and G[0 .. NL-1] (W[1], W[2]), the same of G[NL], and the progress words.  W[0] and
// W[NL] are taken at head_dim 64, where W[0] waits in memory on either side.
template <int D, int NL>
struct MlpNPair {
  using L = MlpNLds<D, NL>;
  static constexpr bool STREAM = D == 64;
  static constexpr int SLOTS = STREAM ? 3 : 2, NJD = D / 32;
  static constexpr int PIECE = 512 * 4 * 2 * L::NBM, PP = L::M * L::M / PIECE;  // floats of a layer's X and G; pieces to a W[i]
  static constexpr int GR = STREAM ? (SLOTS * NL) * PIECE : 0, GSLOT = 512 * NJD;  // G[NL], in W[1] or W[0]
  static constexpr int FL = GR + SLOTS * GSLOT, FL_WORDS = 64;
  static_assert(SLOTS * NL <= (NL == 2 ? 1 : 2) * PP && FL + FL_WORDS <= (STREAM ? L::M : D) * L::M, "the hand-over must fit");
  // words: progress of the producer's waves, its XCD; the same of the consumer
  enum { COUNT = 0, XCD = 8, SIDE = 32 };
};
constexpr unsigned kMlpNPoison = 0xffffffffu;
constexpr unsigned kMlpNLost = 0x7fc60b5eu;  // first word of a unit's W[NL], which no producer writes (a NaN that comes to have these
                                             // bits by itself costs a computation, not the result)

// acc += A B over 16 k: k step r takes the four k with index 4 g + r
__device__ __forceinline__ void mlpn_mma(f32x4& acc, f32x4 a, f32x4 b) {
#pragma unroll
  for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mlpn_ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void mlpn_st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
// rows 4 g .. 4 g + 3 of a column: the transposed operand of a rank-16 update, or its B operand
__device__ __forceinline__ f32x4 mlpn_col4(const float* p, int ld) { return f32x4{p[0], p[ld], p[2 * ld], p[3 * ld]}; }
// LDS written by a wave's lanes and read by other lanes of the same wave
__device__ __forceinline__ void mlpn_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a wave's own piece of the ring, stored by another CU: two device-scope loads, which do not look in the CU's vector cache
__device__ __forceinline__ f32x4 mlpn_ld4_dev(const float* p) {
  const unsigned long long* q = reinterpret_cast<const unsigned long long*>(p);
  const unsigned long long u = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long v = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return f32x4{__uint_as_float((unsigned)u), __uint_as_float((unsigned)(u >> 32)), __uint_as_float((unsigned)v),
               __uint_as_float((unsigned)(v >> 32))};
}

// ROLE 0: the whole unit.  1: the producer of a unit on two workgroups, 2: its consumer.
template <class T, int D, int NL, int ROLE>
__device__ __forceinline__ void mlpn_fwd_body(const MlpNFwdArgs& a, const size_t bh) {
  using IO = Io<T>;
  using elem = typename IO::elem;
  using L = MlpNLds<D, NL>;
  using P = MlpNPair<D, NL>;
  constexpr int M = L::M, LD = L::LD, LM = L::LM, TM = L::TM, NW = L::NW;
  constexpr int GW = 32, NJD = D / GW, NTD = L::NTD, NTM = L::NTM, NBM = L::NBM;
  constexpr int CH = L::CH, NCH = NTM / CH, SPLIT = NW / CH;
  constexpr bool STREAM = D == 64;  // W[0] waits in the output buffer while the other products run
  constexpr int W0S = ROLE == 2 ? NL : 0;  // (the consumer's copy in that of W[NL], of the same size)
  static_assert(NTM % NW == 0 && NTM % CH == 0 && NW % CH == 0 && (SPLIT > 1 || NBM == 1), "tiles must divide among the waves");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int t = tid >> 5, cg = tid & 31, c = lane & 15, g = lane >> 4;
  const int h = (int)(bh % a.H), K = a.K;
  float *sbl = lds + L::bl, *sgam = lds + L::gam, *sbet = lds + L::bet, *slr = lds + L::lr, *ste = lds + L::te;
  const size_t sbase = a.state_per_batch ? bh : (size_t)h;

  // tile (row tile q, column tile n) of a row-major matrix of ld columns <-> registers.  q and n are known at compile
  // time; the lane's own part of the address is the 32-bit offset o.
  auto lane_off = [&](int ld, int row, int col) { return (unsigned)((row + 4 * g) * ld + col + c); };
  auto load_tile = [&](const float* p, int ld, int q, int n, unsigned o) {
    p += 16 * q * ld + 16 * n;
    return f32x4{p[o], (p + ld)[o], (p + 2 * ld)[o], (p + 3 * ld)[o]};
  };
  auto store_tile = [&](float* p, int ld, int q, int n, unsigned o, f32x4 v) {
    p += 16 * q * ld + 16 * n;
#pragma unroll
    for (int r = 0; r < 4; ++r) (p + r * ld)[o] = v[r];
  };

  // ---- initial state
  f32x4 w0[NTD][NBM], w[NL - 1][NTM][NBM], wl[NBM][NTD];  // W[0], W[1 .. NL-1]: own columns; W[NL]: own rows
  float bias[NL][NBM];
  const unsigned oc = lane_off(M, 0, 16 * NBM * wave), orow = lane_off(D, 16 * NBM * wave, 0);
#pragma unroll
  for (int j = 0; j < NBM; ++j) {
#pragma unroll
    for (int q = 0; q < NTD; ++q) {
      w0[q][j] = load_tile(a.W0[0] + sbase * D * M, M, q, j, oc);
      if (STREAM) store_tile(a.W[W0S] + bh * D * M, M, q, j, oc, w0[q][j]);
    }
#pragma unroll
    for (int i = 1; i < NL; ++i)
#pragma unroll
      for (int q = 0; q < NTM; ++q) w[i - 1][q][j] = load_tile(a.W0[i] + sbase * M * M, M, q, j, oc);
#pragma unroll
    for (int q = 0; q < NTD; ++q) wl[j][q] = load_tile(a.W0[NL] + sbase * M * D, D, j, q, orow);
#pragma unroll
    for (int i = 0; i < NL; ++i) bias[i][j] = a.b0[i][sbase * M + 16 * (wave * NBM + j) + c];
  }
  for (int e = tid; e < D; e += 512) {
    sbl[e] = a.b0[NL][sbase * D + e];
    sgam[e] = a.gamma[h * D + e];
    sbet[e] = a.beta[h * D + e];
  }
  if (tid < 16) ste[tid] = (tid < K) ? a.token_eta[tid] : 0.f;
  __syncthreads();
  const float te_last = ste[K - 1];

  // ---- the partner: wave w hands over to wave w, in the layout of the registers, so the only barriers are those of the products
  float* const gring = STREAM ? a.W[1] + bh * M * M + P::GR : a.W[0] + bh * D * M + P::GR;
  unsigned* const fl = reinterpret_cast<unsigned*>(gring + P::SLOTS * P::GSLOT);
  unsigned* const mine = fl + (ROLE == 2 ? P::SIDE : 0);
  unsigned* const theirs = fl + (ROLE == 2 ? 0 : P::SIDE);
  unsigned known = 0, my_xcd = 0;
  bool lost = false, fast = false;  // fast: the partner is known to sit behind the same L2
  if constexpr (ROLE != 0) {
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(my_xcd));
    my_xcd = 0x100u | (my_xcd & 15u);
    lost = a.spin_limit == 0;
    if (tid == 0) __hip_atomic_store(mine + P::XCD, my_xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  auto look = [&](const unsigned* p) {
    return (unsigned)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  };
  auto wait_partner = [&](unsigned want) {  // until the partner's wave has come so far
    if (lost || known >= want) return;
    for (unsigned n = 0; ; ++n) {
      const unsigned v = look(theirs + P::COUNT + (threadIdx.x >> 6));
      if (v == kMlpNPoison || n >= a.spin_limit) {
        lost = true;
        return;
      }
      if (v >= want) {
        known = v;
        return;
      }
      __builtin_amdgcn_s_sleep(2);
    }
  };
  auto publish = [&](unsigned count) {  // every store of this wave has been acknowledged, or written back
    if (ROLE == 1 && !fast && a.agent_release == 0) fast = look(theirs + P::XCD) == my_xcd;
    if (ROLE == 1 && !fast) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if ((threadIdx.x & 63) == 0)
      __hip_atomic_store(mine + P::COUNT + (threadIdx.x >> 6), lost ? kMlpNPoison : count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  int slot = 0;
  auto hand = [&](int i, int kind, int j) {  // X[i+1] (kind 0) or G[i] (1), tile j of the own columns
    const int p = slot * NL + i;
    float* base = NL > 2 && p >= P::PP ? a.W[NL > 2 ? 2 : 1] + bh * M * M + (p - P::PP) * P::PIECE : a.W[1] + bh * M * M + p * P::PIECE;
    return base + (unsigned)(4 * ((kind * NBM + j) * 512 + tid));
  };

  // Where the staged rows wait: what the role does not use otherwise, or X[1]
  constexpr int SQ = ROLE == 2 ? L::GT : L::XI, SK = ROLE == 1 ? L::XQ : SQ + L::TD;
  constexpr int ST = ROLE == 1 ? L::ZBL : SQ + 2 * L::TD, SL = ROLE == 1 ? L::PART : SQ + 3 * L::TD;
  // The next mini-batch's xq/xk/xv/lr are fetched into registers while the last W[i] is updated, wait where X[1] lay while
  // W[0] is in registers, and go to their places when the mini-batch begins.  All by the thread that fetched them.
  elem pq[NJD], pk[NJD], pv[NJD], plr;
  auto fetch = [&](int stage) {  // rows K .. 15 are zero
    int x = tid;  // opaque: the offsets are formed here and not kept from the loop's beginning
    asm volatile("" : "+v"(x));
    const size_t r0 = bh * (size_t)a.seq_stride + (size_t)stage * K;
    const elem* xq = static_cast<const elem*>(a.xq) + r0 * D;
    const elem* xk = static_cast<const elem*>(a.xk) + r0 * D;
    const elem* xv = static_cast<const elem*>(a.xv) + r0 * D;
    const elem* lr = static_cast<const elem*>(a.lr) + r0;
    const unsigned o = ((x >> 5) < K ? x >> 5 : 0) * D + (x & 31);
#pragma unroll
    for (int j = 0; j < NJD; ++j) {
      if (ROLE != 1) pq[j] = xq[o + GW * j];
      pk[j] = xk[o + GW * j];
      if (ROLE != 2) pv[j] = xv[o + GW * j];
    }
    plr = lr[(unsigned)((x & 15) < K ? x & 15 : 0)];
  };
  auto stage_rows = [&]() {
    float* S = lds + SQ + t * LD + cg;
#pragma unroll
    for (int j = 0; j < NJD; ++j) {
      const float k = IO::load1(pk + j);
      if (ROLE != 1) S[GW * j] = t < K ? IO::load1(pq + j) : 0.f;
      S[SK - SQ + GW * j] = t < K ? k : 0.f;
      if (ROLE != 2) S[ST - SQ + GW * j] = t < K ? IO::load1(pv + j) - k : 0.f;
    }
    if (tid < 16) lds[SL + tid] = tid < K ? IO::load1(&plr) : 0.f;
  };
  static_assert(3 * L::TD + 16 <= TM, "the staged rows take the place of X[1]");
  fetch(0);
  stage_rows();

  for (int st = 0; st < a.n_stages; ++st) {
    // re-derived from an opaque copy every mini-batch, so that address arithmetic is recomputed here instead of being
    // hoisted out of the scan into (spilled) registers
    asm volatile("" : "+v"(tid));
    lane = tid & 63, wave = tid >> 6, t = tid >> 5, cg = tid & 31, c = lane & 15, g = lane >> 4;
    const int own = 16 * NBM * wave;               // first own hidden column
    const int am = c * LM + 4 * g, ad = c * LD + 4 * g;  // A operand: row c, k = 4 g ..
    const int um = 4 * g * LM + c, ud = 4 * g * LD + c;  // rows 4 g .., column c
#pragma unroll
    for (int j = 0; j < NJD; ++j) {
      const int o = t * LD + cg + GW * j;
      if (ROLE != 1) lds[L::XQ + o] = lds[SQ + o];
      lds[L::XK + o] = lds[SK + o];
      if (ROLE != 2) lds[L::TG + o] = lds[ST + o];
    }
    if (tid < 16) slr[tid] = lds[SL + tid];
    __syncthreads();

    // ---- forward chain: Z[i] = X[i] W[i]; X[i+1] = gelu(Z[i] + b[i]); gelu' stays in registers.  XQ W[0] rides along.
    // Attention blocks are held transposed, element [s = 4 g + r][t = c]: as registers they are the A operand of MX G.
    f32x4 G[NL][NBM], zq[NBM];  // G: gelu'(Z[i]), later G[i]
    auto hidden = [&](int i, const f32x4 (&z)[NBM]) {
      float* X = lds + L::XI + i * TM + own;
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float y, dy;
          gelu_tanh_pair(z[j][r] + bias[i][j], y, dy);
          X[um + r * LM + 16 * j] = y;
          if constexpr (ROLE == 1) x[r] = y;
          G[i][j][r] = dy;
        }
        if constexpr (ROLE == 1) mlpn_st4(hand(i, 0, j), x);
      }
    };
    // X W over k = M, the operand read one tile ahead (the compiler, short of registers, would wait for each read)
    auto product = [&](f32x4 (&z)[NBM], const float* X, const f32x4 (&W)[NTM][NBM]) {
      f32x4 fx = mlpn_ld4(X + am);
#pragma unroll
      for (int j = 0; j < NBM; ++j) z[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < NTM; ++q) {
        const f32x4 nx = mlpn_ld4(X + am + 16 * (q + 1 < NTM ? q + 1 : q));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_mma(z[j], fx, W[q][j]);
        __builtin_amdgcn_sched_barrier(0);
        fx = nx;
      }
    };
    if (ROLE == 1 && st >= P::SLOTS) wait_partner((unsigned)(st - P::SLOTS + 1));  // the slot is free
    if constexpr (ROLE == 1) {
      f32x4 z[NBM];
#pragma unroll
      for (int j = 0; j < NBM; ++j) z[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < NTD; ++q) {
        const f32x4 fk = mlpn_ld4(lds + L::XK + ad + 16 * q);
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_mma(z[j], fk, w0[q][j]);
      }
      hidden(0, z);
    } else {
      f32x4 z[NBM], at = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NBM; ++j) z[j] = zq[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (ROLE == 0) {
#pragma unroll
      for (int q = 0; q < NTD; ++q) {
        const f32x4 fk = mlpn_ld4(lds + L::XK + ad + 16 * q);
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_mma(z[j], fk, w0[q][j]);
      }
      }
      // the attention block XQ XK^T: the waves share its k steps
#pragma unroll
      for (int e = 0; e < D / 4 / NW; ++e) {
        const int ks = wave * (D / 4 / NW) + e, o = ad + 16 * (ks >> 2) + (ks & 3);
        at = __builtin_amdgcn_mfma_f32_16x16x4f32(lds[L::XK + o], lds[L::XQ + o], at, 0, 0, 0);
      }
      mlpn_st4(lds + L::PART + wave * 256 + 4 * lane, at);
      __builtin_amdgcn_sched_barrier(0);
      // XQ W[0] runs beside the activations: a product of four matrix instructions, then an activation
      static_assert(NTD <= 4, "products to go with the activations");
      float* X = lds + L::XI + own;
#pragma unroll
      for (int e = 0; e < 4 * NBM; ++e) {
        if (e < NTD * NBM) mlpn_mma(zq[e % NBM], mlpn_ld4(lds + L::XQ + ad + 16 * (e / NBM)), w0[e / NBM][e % NBM]);
        if (ROLE == 2) continue;
        float y, dy;
        gelu_tanh_pair(z[e >> 2][e & 3] + bias[0][e >> 2], y, dy);
        X[um + (e & 3) * LM + 16 * (e >> 2)] = y;
        G[0][e >> 2][e & 3] = dy;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (ROLE == 2) {
      // what the producer has made of this mini-batch
      wait_partner((unsigned)(st + 1));
      if (!fast) {
        if (a.agent_release == 0) fast = look(theirs + P::XCD) == my_xcd;
        if (!fast) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      }
      f32x4 x[NL][NBM];
      unsigned long long gv = 0;
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int j = 0; j < NBM; ++j) {
          x[i][j] = mlpn_ld4_dev(hand(i, 0, j));
          G[i][j] = mlpn_ld4_dev(hand(i, 1, j));
        }
      const float* gp = gring + slot * P::GSLOT + NJD * tid;
      if constexpr (NJD == 2)
        gv = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(gp), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        gv = __hip_atomic_load(reinterpret_cast<const unsigned*>(gp), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      publish((unsigned)(st + 1));  // all of it has landed
      slot = slot + 1 < P::SLOTS ? slot + 1 : 0;
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int j = 0; j < NBM; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) lds[L::XI + i * TM + own + um + r * LM + 16 * j] = x[i][j][r];
#pragma unroll
      for (int j = 0; j < NJD; ++j) lds[L::ZL + t * LD + cg + GW * j] = __uint_as_float((unsigned)(gv >> (32 * j)));
    }
    __syncthreads();
    if constexpr (ROLE != 2) {
#pragma unroll
      for (int i = 1; i < NL; ++i) {
        f32x4 z[NBM];
        product(z, lds + L::XI + (i - 1) * TM, w[i - 1]);
        hidden(i, z);
        if (i + 1 < NL) __syncthreads();
      }
      mlpn_wave_sync();
    }
    // X W[NL] over the wave's own rows
    auto last_product = [&](const float* X) {
      f32x4 z[NTD];
#pragma unroll
      for (int n = 0; n < NTD; ++n) z[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        const f32x4 fx = mlpn_ld4(X + am + own + 16 * j);
#pragma unroll
        for (int n = 0; n < NTD; ++n) mlpn_mma(z[n], fx, wl[j][n]);
      }
#pragma unroll
      for (int n = 0; n < NTD; ++n) mlpn_st4(lds + L::PZ + (wave * NTD + n) * 256 + 4 * lane, z[n]);
    };
    if constexpr (ROLE != 2) {
    // ---- Z[NL] = X[NL] W[NL]; G[NL] = LN-L2 gradient of Z[NL] + b[NL] against the target
    last_product(lds + L::XI + (NL - 1) * TM);
    __syncthreads();
    {
      float Gv[NJD], z[NJD][NW];
#pragma unroll
      for (int j = 0; j < NJD; ++j) {
        const int o = cg + GW * j;
        const float* p = lds + L::PZ + (o >> 4) * 256 + 4 * (16 * (t >> 2) + (o & 15)) + (t & 3);
#pragma unroll
        for (int v = 0; v < NW; ++v) z[j][v] = p[v * NTD * 256];
      }
      __builtin_amdgcn_sched_barrier(0);  // all reads first: the compiler would wait for each
#pragma unroll
      for (int j = 0; j < NJD; ++j) {
#pragma unroll
        for (int v = 1; v < NW; ++v) z[j][0] += z[j][v];
        lds[L::ZL + t * LD + cg + GW * j] = z[j][0];
      }
      ln_l2_grad<D, GW>(lds + L::ZL + t * LD, sbl, lds + L::TG + t * LD, sgam, sbet, cg, a.eps, Gv);
#pragma unroll
      for (int j = 0; j < NJD; ++j) lds[L::ZL + t * LD + cg + GW * j] = Gv[j];
      if constexpr (ROLE == 1) {
        float* gp = gring + slot * P::GSLOT + NJD * tid;
        if constexpr (NJD == 2)
          *reinterpret_cast<float2*>(gp) = float2{Gv[0], Gv[1]};
        else
          *gp = Gv[0];
      }
    }
    __syncthreads();
    // ---- G[NL-1] = (G[NL] W[NL]^T) * gelu'(Z[NL-1]): own rows, transposed in the wave's own part of the pool
    {
      float* S = lds + L::POOL + wave * NBM * 16 * LD;
#pragma unroll
      for (int j = 0; j < NBM; ++j)
#pragma unroll
        for (int n = 0; n < NTD; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[16 * j * LD + ud + r * LD + 16 * n] = wl[j][n][r];
      mlpn_wave_sync();
      f32x4 z[NBM];
#pragma unroll
      for (int j = 0; j < NBM; ++j) z[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < NTD; ++n) {
        const f32x4 fg = mlpn_ld4(lds + L::ZL + ad + 16 * n);
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_mma(z[j], fg, mlpn_ld4(S + 16 * j * LD + ad + 16 * n));
      }
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        G[NL - 1][j] *= z[j];
        if (ROLE == 1) mlpn_st4(hand(NL - 1, 1, j), G[NL - 1][j]);
#pragma unroll
        for (int r = 0; r < 4; ++r) lds[L::GT + um + r * LM + own + 16 * j] = G[NL - 1][j][r];
      }
    }
    __syncthreads();
    // ---- G[i] = (G[i+1] W[i+1]^T) * gelu'(Z[i]): a wave takes one tile row of each chunk, SPLIT waves share its k
#pragma unroll
    for (int i = NL - 2; i >= 0; --i) {
      f32x4 z[NCH];
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
#pragma unroll
        for (int q = 0; q < CH; ++q)
#pragma unroll
          for (int j = 0; j < NBM; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              lds[L::POOL + 16 * q * LM + um + r * LM + own + 16 * j] = w[i][ch * CH + q][j][r];
        __syncthreads();
        const int k0 = (wave / CH) * (M / SPLIT);
        const float* Gp = lds + L::GT + am + k0;
        const float* Wp = lds + L::POOL + 16 * (wave % CH) * LM + am + k0;
        f32x4 z0[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, fg = mlpn_ld4(Gp), fw = mlpn_ld4(Wp);
#pragma unroll
        for (int k = 0; k < M / SPLIT; k += 16) {  // reads one tile ahead, as above
          const int kn = k + 16 < M / SPLIT ? k + 16 : k;
          const f32x4 ng = mlpn_ld4(Gp + kn), nw = mlpn_ld4(Wp + kn);
          __builtin_amdgcn_sched_barrier(0);
          mlpn_mma(z0[(k >> 4) & 1], fg, fw);
          __builtin_amdgcn_sched_barrier(0);
          fg = ng;
          fw = nw;
        }
        z[ch] = z0[0] + z0[1];
        __syncthreads();
      }
      if constexpr (SPLIT == 1) {
        G[i][0] *= z[0];
      } else {
        // (G[1] waited in LDS: eight registers more for the products)
#pragma unroll
        for (int j = 0; j < NBM; ++j) G[NL - 1][j] = mlpn_col4(lds + L::GT + um + own + 16 * j, LM);
        static_assert(SPLIT == 1 || (SPLIT == 2 && NL == 2), "the partials lie where the next layer's chunk would");
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            lds[L::PZ + (wave / CH) * TM + um + r * LM + 16 * (ch * CH + wave % CH)] = z[ch][r];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NBM; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float* p = lds + L::PZ + um + r * LM + own + 16 * j;
            G[i][j][r] *= p[0] + p[TM];
          }
      }
      if (ROLE == 1)
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_st4(hand(i, 1, j), G[i][j]);
      if (i > 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < NBM; ++j) lds[L::GT + um + r * LM + own + 16 * j] = G[i][j][r];
      }
    }
    }
    // ---- output chain; W[i] is updated right behind its last product of the mini-batch
    auto last = [&]() { return te_last * mlpn_ld4(slr + 4 * g); };  // of rows 4 g ..
    auto sum8 = [&](const float* p, int stride) {  // the waves' partials of a tile
      f32x4 v[NW];
#pragma unroll
      for (int u = 0; u < NW; ++u) v[u] = mlpn_ld4(p + u * stride);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 1; u < NW; ++u) v[0] += v[u];
      return v[0];
    };
    auto attention = [&](int i) {  // -eta (1 + tril(Xb[i] X[i]^T)), transposed
      const float* p = lds + L::PART + (i & 1) * NW * 256 + 4 * lane;
      const f32x4 at = sum8(p, 256), l = mlpn_ld4(slr + 4 * g);
      const float te = -ste[c];
      f32x4 mx;
#pragma unroll
      for (int r = 0; r < 4; ++r) mx[r] = 4 * g + r <= c ? te * l[r] * (1.f + at[r]) : 0.f;
      return mx;
    };
    auto step = [&](int i) {  // the update's gradient and the bias
      const f32x4 lst = last();
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        G[i][j] *= lst;
        float s = (G[i][j][0] + G[i][j][1]) + (G[i][j][2] + G[i][j][3]);
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
        bias[i][j] -= s;
      }
    };
    auto hidden_out = [&](int i, f32x4 (&z)[NBM]) {  // z -> Xb[i+1] and the own part of its attention block
      const f32x4 mx = attention(i);
      float* X = lds + L::POOL + (i & 1) * TM + own;
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        mlpn_mma(z[j], mx, G[i][j]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float y, dy;
          gelu_tanh_pair(z[j][r] + bias[i][j], y, dy);
          X[um + r * LM + 16 * j] = y;
        }
      }
      mlpn_wave_sync();
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NBM; ++j)
        mlpn_mma(p, mlpn_ld4(lds + L::XI + i * TM + am + own + 16 * j), mlpn_ld4(X + am + 16 * j));
      mlpn_st4(lds + L::PART + ((i + 1) & 1) * NW * 256 + wave * 256 + 4 * lane, p);
      step(i);
    };
    if constexpr (ROLE == 1) {
      if (st + 1 == a.n_stages) publish((unsigned)(st + 1));  // (otherwise behind the updates, where nothing waits for the stores)
      step(0);
    } else {
      hidden_out(0, zq);
    }
#pragma unroll
    for (int i = 1; i < NL; ++i) {
      if constexpr (ROLE == 1) {
        step(i);
      } else {
        __syncthreads();
        f32x4 z[NBM];
        product(z, lds + L::POOL + ((i - 1) & 1) * TM, w[i - 1]);
        hidden_out(i, z);
      }
      if (i == NL - 1) fetch(st + 1 < a.n_stages ? st + 1 : st);  // no branch: the registers would be kept through it
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < NTM; ++q) {
        const f32x4 fx = -mlpn_col4(lds + L::XI + (i - 1) * TM + um + 16 * q, LM);
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_mma(w[i - 1][q][j], fx, G[i][j]);
      }
    }
    if constexpr (ROLE != 1) {
      last_product(lds + L::POOL + ((NL - 1) & 1) * TM);
      __syncthreads();
    }
    stage_rows();
    if (ROLE != 1 && wave < NTD) {
      f32x4 z = sum8(lds + L::PZ + wave * 256 + 4 * lane, NTD * 256);
      mlpn_mma(z, attention(NL), mlpn_col4(lds + L::ZL + ud + 16 * wave, LD));
#pragma unroll
      for (int r = 0; r < 4; ++r) lds[L::ZBL + ud + r * LD + 16 * wave] = z[r];
    }
    if (STREAM) {
#pragma unroll
      for (int q = 0; q < NTD; ++q)
#pragma unroll
        for (int j = 0; j < NBM; ++j) w0[q][j] = load_tile(a.W[W0S] + bh * D * M, M, q, j, lane_off(M, 0, own));
    }
    __builtin_amdgcn_sched_barrier(0);
    {
      const f32x4 lst = last();
      f32x4 fx[NBM];
#pragma unroll
      for (int j = 0; j < NBM; ++j) fx[j] = -mlpn_col4(lds + L::XI + (NL - 1) * TM + um + own + 16 * j, LM);
#pragma unroll
      for (int n = 0; n < NTD; ++n) {
        const f32x4 gl = mlpn_col4(lds + L::ZL + ud + 16 * n, LD) * lst;
#pragma unroll
        for (int j = 0; j < NBM; ++j) mlpn_mma(wl[j][n], fx[j], gl);
      }
    }
    if constexpr (ROLE == 1) {
      if (st + 1 < a.n_stages) publish((unsigned)(st + 1));
      slot = slot + 1 < P::SLOTS ? slot + 1 : 0;
    }
#pragma unroll
    for (int q = 0; q < NTD; ++q) {
      const f32x4 fx = -mlpn_col4(lds + L::XK + ud + 16 * q, LD);
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        mlpn_mma(w0[q][j], fx, G[0][j]);
        if (STREAM) store_tile(a.W[W0S] + bh * D * M, M, q, j, lane_off(M, 0, own), w0[q][j]);
      }
    }
    float db = 0.f;
    if (tid >= 512 - D)  // a wave that had no tile of Zb[NL]
#pragma unroll
      for (int r = 0; r < 16; ++r) db += lds[L::ZL + r * LD + tid - (512 - D)] * (te_last * slr[r]);
    __syncthreads();
    // ---- out = XQ + LN(Zb[NL] + b[NL])
    if constexpr (ROLE != 1) {
      const size_t row = bh * (size_t)a.seq_stride + (size_t)st * K + t;
      float xh[NJD], rstd;
      ln_stats<D, GW>(lds + L::ZBL + t * LD, sbl, cg, a.eps, xh, rstd);
#pragma unroll
      for (int j = 0; j < NJD; ++j) {
        const int o = cg + GW * j;
        if (t < K)
          IO::store1(static_cast<elem*>(a.out) + row * D + o, lds[L::XQ + t * LD + o] + (sgam[o] * xh[j] + sbet[o]));
      }
    }
    if (ROLE != 1) __syncthreads();
    if (tid >= 512 - D) sbl[tid - (512 - D)] -= db;
  }

  if constexpr (ROLE != 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this side's stores into W_out lie in front of the final state's
    lane = tid & 63, wave = tid >> 6;
    float* S = lds + L::PZ;
    __syncthreads();
    if (lane == 0) S[wave] = lost ? 1.f : 0.f;
    __syncthreads();
    float any = 0.f;
#pragma unroll
    for (int v = 0; v < NW; ++v) any += S[v];
    if (__builtin_amdgcn_readfirstlane((int)any) != 0) {  // a wait was in vain: the unit is done again
      if (tid == 0) {
        atomicAdd(a.lost_count, 1u);
        if (ROLE == 2) *reinterpret_cast<unsigned*>(a.W[NL] + bh * M * D) = kMlpNLost;
      }
      return;
    }
    if (ROLE == 1) return;
  }

  // ---- final state
  const unsigned oc1 = lane_off(M, 0, 16 * NBM * wave), orow1 = lane_off(D, 16 * NBM * wave, 0);
#pragma unroll
  for (int j = 0; j < NBM; ++j) {
    const int n = wave * NBM + j;
    if (!STREAM) {
#pragma unroll
      for (int q = 0; q < NTD; ++q) store_tile(a.W[0] + bh * D * M, M, q, j, oc1, w0[q][j]);
    }
#pragma unroll
    for (int i = 1; i < NL; ++i)
#pragma unroll
      for (int q = 0; q < NTM; ++q) store_tile(a.W[i] + bh * M * M, M, q, j, oc1, w[i - 1][q][j]);
#pragma unroll
    for (int q = 0; q < NTD; ++q) store_tile(a.W[NL] + bh * M * D, D, j, q, orow1, wl[j][q]);
#pragma unroll
    for (int i = 0; i < NL; ++i)
      if (g == 0) a.b[i][bh * M + 16 * n + c] = bias[i][j];
  }
  __syncthreads();
  if (tid < D) a.b[NL][bh * D + tid] = sbl[tid];
}

// The arguments where they lie in the argument segment: through the parameter the compiler loads all of them at the start, and
// the f32 kernel at head_dim 64 spills 200 registers instead of 20.
__device__ __forceinline__ const MlpNFwdArgs& mlpn_args() {
  return *(const MlpNFwdArgs*)__builtin_amdgcn_kernarg_segment_ptr();
}

template <class T, int D, int NL>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) ttt_mlpn_fwd_kernel(MlpNFwdArgs) {
  const MlpNFwdArgs& a = mlpn_args();
  if (a.only_lost != 0) {
    const unsigned* mark = reinterpret_cast<const unsigned*>(a.W[NL] + blockIdx.x * (size_t)(4 * D * D));
    if (__builtin_amdgcn_readfirstlane((int)*mark) != (int)kMlpNLost) return;
  }
  mlpn_fwd_body<T, D, NL, 0>(a, blockIdx.x);
}

// Workgroups b and b + 8 of every 16 share a unit: consecutive workgroups go to the XCDs in turn, so both run behind one L2.
template <class T, int D, int NL>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) ttt_mlpn_fwd_pair_kernel(MlpNFwdArgs) {
  const MlpNFwdArgs& a = mlpn_args();
  const size_t bh = (size_t)(blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
  if (bh >= (size_t)a.B * a.H) return;
  if (((blockIdx.x >> 3) & 1) == 0)
    mlpn_fwd_body<T, D, NL, 1>(a, bh);
  else
    mlpn_fwd_body<T, D, NL, 2>(a, bh);
}

template <int D, int NL>
__global__ void ttt_mlpn_fwd_clear_kernel(MlpNFwdArgs a) {  // the progress words of every unit
  using P = MlpNPair<D, NL>;
  constexpr int M = 4 * D;
  float* fl = (P::STREAM ? a.W[1] + (size_t)blockIdx.x * M * M : a.W[0] + (size_t)blockIdx.x * D * M) + P::FL;
  fl[threadIdx.x] = 0.f;
}

hipError_t launch_mlpn_fwd(bool f32, int head_dim, int n_hidden, bool pair, const MlpNFwdArgs& a, hipStream_t s);  // ttt_mlpn_fwd.hip

}  // namespace ttt
