// TTT-MLP multi-stage forward for gfx950 with the whole state resident in registers.
//
// Arithmetic: reference rust/core/src/mlp.rs:127-208 (one mini-batch) looped over the sequence as
// rust/core/src/inner.rs:25-50; GELU constants rust/thundercube/src/unary_ops.rs:136-173.
//
// One workgroup of eight waves per (batch, head).  The hidden axis (4 d units) is cut into eight
// slices; wave w keeps, as MFMA accumulator tiles in VGPRs for the whole sequence,
//     W1[:, slice]  (d x 4d/8)   rows (d features) in registers, hidden units across lanes
//     W2[slice, :]  (4d/8 x d)   hidden units in registers, d features across lanes
//     b1[slice]
// which is 2 * (d/16) * (d/32) tiles = 144 VGPRs at d = 96.  Everything that is elementwise in the
// hidden axis (Z1, GELU, G1, Zbar1, Xbar2, both state updates) stays inside the wave.  The three
// contractions OVER the hidden axis (Z2 = X2 W2, Zbar2 = Xbar2 W2, A2 = Xbar2 X2^T) are split-k:
// every wave writes its partial tiles to LDS and wave I < d/16 (a "reducer") adds up d-feature
// tile I, owns b2 / gamma / beta of those sixteen features and does the LayerNorm work on them.
//
// Per mini-batch there are three barriers on the recurrence W -> Z1 -> X2 -> Z2 -> G2 -> G1 -> W':
//   B1  partial Z2 tiles (and last mini-batch's partial Zbar2 / A2) are in LDS
//   B2  the reducers' row moments for the LN-L2 gradient are in LDS
//   B3  G2 (already scaled by -eta_last) is in LDS, and the row moments of last mini-batch's output
// The output of mini-batch t needs nothing the recurrence waits for: it is finished one mini-batch late, where waves have time.
// At d = 96 its sums are formed at the end of phase A by the older waves (0 - 3: of the two waves of a SIMD they run 2 k cycles
// ahead and would wait at B1) and stored between B1 and B3 by the two waves that reduce nothing; at d = 32 and 64 there are
// more such waves, and all of it is theirs.
//
// What bounds it.  Phases A and D (the products) by the issue of a SIMD's two waves: matrix instructions and vector
// instructions of 16x16 tiles hardly overlap, not across waves either (probe: a matrix instruction and three FMAs, two
// waves, 23.3 cycles against 16 + 7.5).  Phases B and C by latency.  Cycles of a mini-batch at d = 96 and 128 units:
// XQ W1 sharing the operands of XK W1 took A from 4.9 to 4.7 k, sums by lane group B from 2.9 to 2.0 k and C from 2.2 to 1.3 k,
// independent products side by side and transposes read from LDS D from 7.4 to 6.4 k: 8 x 16 units x 2048 tokens, d = 96 840 -> 661 us,
// d = 64 488 -> 428, d = 32 286 -> 260.  The output taken out of B (three tiles of sums by two waves were its longest path, 2.1 k) and
// D, the staging copies from the younger waves, a load of eps through the scalar cache from C and the sums of the prologue from
// one load each: 636, 413, 247; saving d = 96 715 -> 674, d = 64 467 -> 444, d = 32 284 -> 270.
//
// An odd hidden tile at the end of a split-k chain is issued as a k = 32 MFMA with a zero second
// half, not as a k = 16 one: a 16x16x16 bf16 MFMA accumulating straight onto the result of a
// 16x16x32 one was measured to give wrong sums on gfx950 with this toolchain.
//
// Operands that are needed with their axes exchanged.  What lies in LDS anyway (the staged rows of XK, G2) or is not waited
// for (X2 at d = 96) is read with the transposing LDS load.  W2 tiles with d in the k position (G1 = G2 W2^T) and G1 are
// transposed on the matrix pipe, one 16x16x16 MFMA against an identity fragment each: G1 is on the chain, where a round trip
// through LDS takes longer, and for W2 (74 KB at d = 96) LDS has no room beside the partial tiles.  (Shared by the two kinds
// of partial tile, it has: 726 us, the waits for the region cost what the transposes save.)
#pragma once
#include "ttt_engine_fwd.hip.h"
#include "ttt_linear_fwd_mw.hip.h"

namespace ttt {

template <int D, int ES>
struct MlpRrLds {
  static constexpr int NW = 8, NT = D / 16;
  static constexpr int XS = D > 64 ? 2 : 0;   // hidden tiles of a wave whose X2 is transposed by LDS: as many as there is room for
  static constexpr int TILE = 16 * D * ES;    // one [16 x d] input tile, rows unpadded
  static constexpr int IN1 = 3 * TILE;        // xq, xk, xv tiles of one mini-batch
  static constexpr int IN = 0;                // [3 buffers][3][16][d]
  static constexpr int LR = IN + 3 * IN1;     // [3][16] floats
  static constexpr int PRM = LR + 3 * 64 + 64;  // gamma[d], beta[d], b1[4d] floats
  static constexpr int EX = PRM + 6 * D * 4;    // [6 sums][2][16 tokens] f32x4 (reducer index % 4)
  static constexpr int EXO = EX + 6 * 2 * 16 * 16;      // [2 sums][2][16 tokens] f32x4 (output tile % 4)
  static constexpr int P1 = EXO + 2 * 2 * 16 * 16;  // [NW][NT][64] f32x4: partial Z2^T tiles
  static constexpr int P2 = P1 + NW * NT * 1024;  // partial Zbar2^T tiles
  static constexpr int PA = P2 + NW * NT * 1024;  // [NW][64] f32x4: partial A2^T
  static constexpr int ZB = PA + NW * 1024;       // [NT][64] f32x4: Zbar2^T tiles of the previous mini-batch
  static constexpr int GT = ZB + NT * 1024;       // [2][NT][64] frag: G2^T tiles (d along k)
  static constexpr int X2S = GT + 2 * NT * 64 * 4 * ES;  // [NW][XS][64] frag: X2^T tiles
  static constexpr int M1 = X2S + NW * XS * 64 * 4 * ES;  // [2][64] frag: M1 of this mini-batch
  static constexpr int ID = M1 + 2 * 64 * 4 * ES;  // [64] frag: identity
  static constexpr int RHO = ID + 64 * 4 * ES;  // [16] token_eta / sc
  static constexpr int FL = RHO + 64;           // [NW] counters
  static constexpr int BYTES = FL + 4 * NW;
  static_assert(BYTES <= 160 * 1024, "exceeds the 160 KiB of LDS of a gfx950 CU");
  static_assert(NT <= NW && D % 32 == 0, "one reducer wave per d-feature tile");
  static_assert(ES == 2, "the transposing LDS load takes 16-bit elements");
  static_assert(TILE % 1024 == 0 && P1 % 16 == 0, "input tiles are staged in 1 KiB wave blocks");
};

// Makes the compiler forget what it knows about v.  The bf16 operand copies of the W2 tiles are
// needed at three places of a mini-batch; without this the compiler keeps the converted copies
// (36 VGPRs at d = 96) alive across the barriers and spills state tiles to scratch instead.
__device__ __forceinline__ void forget(f32x4& v) { asm volatile("" : "+v"(v)); }
// Orders memory accesses around the point where v is complete: keeps a reduction loop from issuing
// all its LDS loads (four VGPRs each) before the first add.
__device__ __forceinline__ void pin(f32x4& v) { asm volatile("" : "+v"(v)::"memory"); }
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)::"memory"); }

// ---- Centred second layer.  The TTT-MLP loop looks at W2 and b2 only through LayerNorm (Z2 = X2 W2 + b2 feeds the
// LN-L2 gradient, Zbar2 the output LayerNorm) and through G1 = (G2 W2^T) gelu'(Z1), where the rows of G2 sum to zero.
// So, exactly as for the TTT-Linear state (centre_state in ttt_linear_fwd_mw.hip.h), the kernels carry
// W2 - m 1^T (m_i = mean over the d columns of row i) and b2 - mean(b2): the dropped part shifts every feature of a
// token by the same amount (discarded by both LayerNorms) and meets only zero row sums in G2 W2^T; the updates
// W2 += X2^T G2'', b2 += colsum G2'' do not move m or mean(b2).  Z2 and Zbar2 then have row means at rounding
// level, which keeps the one-pass statistics and the bf16 operand images of W2 accurate for any offset of its rows.
//
// Mean of each of the four rows (4g + r of a 16-row tile) of a [16 x d] tile held as NT accumulator tiles
// (columns: tile I, lane c), the same float in all sixteen lanes of a row.  Made opaque so that the subtraction
// that follows is a subtraction of this rounded number wherever it is repeated (no fused multiply-add).
template <int NT>
__device__ __forceinline__ f32x4 row_means16(const f32x4 (&t)[NT], float inv_d) {
  f32x4 m;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float p = 0.f;
#pragma unroll
    for (int I = 0; I < NT; ++I) p += t[I][r];
    m[r] = row16_first(row16_sum_dpp(p)) * inv_d;
  }
  asm volatile("" : "+v"(m));
  return m;
}
// mean of d floats in global memory, the same float in every lane, opaque as above
__device__ __forceinline__ float mean_of(const float* p, int d, float inv_d) {
  float s = 0.f;
  for (int f = 0; f < d; ++f) s += p[f];
  s *= inv_d;
  asm volatile("" : "+v"(s));
  return s;
}

// The LDS addresses derived from the lane index are many (the regions span 150 KiB, beyond the
// 64 KiB reach of an instruction offset) and all loop-invariant: hoisted out of the loop they are
// spilled and reloaded from scratch.  Hiding the lane index from the optimiser at the start of each
// phase makes them cheap phase-local recomputations instead.  At d = 96 the lane coordinates and the constant operands
// (identity, rho) are formed anew or read from LDS as well: held in registers they spill, and a reload from scratch waits for
// the copies in flight (871 against 770 us); at d <= 64 there is room for them (471 against 434 us), but for one register
// too many in the saving kernel at d = 32 (see the kernel's launch bounds).
#define RELANE()                               \
  do {                                         \
    asm volatile("" : "+v"(lane));             \
    if constexpr (D == 32 && SAVE) g = lane >> 4; \
    if constexpr (D > 64) {                    \
      c = lane & 15;                           \
      g = lane >> 4;                           \
      own = own_offset<1>(red ? w : 0, 0, g);  \
    }                                          \
  } while (0)

// SAVE: also leave what a backward starts from (MlpFwdArgs::fac_save or G1_save).  A compilation of its own: the pointers
// and branches cost the plain forward 3 % of its time in registers.
// d = 32 is held to 128 registers, so that a CU takes two workgroups (LDS has room for them): each hides the other's waits
// between the barriers.  512 units x 2048 tokens, with 130 registers -> 128: 530 -> 353 us, saving 574 -> 382 us; 128 units,
// which have a CU each, 266 -> 261 and 287 -> 285 us.
template <class T, int D, bool SAVE>
__global__ void __launch_bounds__(512, D == 32 ? 4 : 2) ttt_mlp_fwd_rr_kernel(Problems<MlpFwdArgs> problems) {
  const MlpFwdArgs& a = problems.p[blockIdx.y];
  using IO = Io<T>;
  using frag = typename IO::frag;
  using elem = typename IO::elem;
  constexpr int ES = sizeof(elem);
  using L = MlpRrLds<D, ES>;
  constexpr int NW = 8, NT = D / 16, F = 4 * D, HT = F / 16 / NW;
  constexpr float inv_d = 1.0f / D;
  if (SAVE && already_saved(a)) return;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  // the wave index is read through an SGPR so that everything keyed on it is scalar control flow
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63;  // refreshed (see RELANE) at every phase of the main loop
  int c = lane & 15, g = lane >> 4;
  const size_t bh = blockIdx.x;
  const int h = (int)(bh % a.H), K = a.K;
  const float eps = held(a.eps);
  const bool red = w < NT;  // this wave reduces d-feature tile w
  // this wave stores output tiles (at d = 32 there are more waves left than tiles)
  const bool outw = !red && (2 * NT >= NW || w < 2 * NT);
  const bool older = w < 4;               // the first wave of its SIMD
  constexpr bool LATE = D <= 64;
  const bool outs = LATE ? outw : older;   // this wave adds up output tiles

  f32x4* const P1 = reinterpret_cast<f32x4*>(smem + L::P1);
  f32x4* const P2 = reinterpret_cast<f32x4*>(smem + L::P2);
  f32x4* const PA = reinterpret_cast<f32x4*>(smem + L::PA);
  float* const EX = reinterpret_cast<float*>(smem + L::EX);
  float* const EXO = reinterpret_cast<float*>(smem + L::EXO);
  frag* const IDs = reinterpret_cast<frag*>(smem + L::ID);
  float* const RHO = reinterpret_cast<float*>(smem + L::RHO);
  frag* const M1s = reinterpret_cast<frag*>(smem + L::M1);
  lds_int* const FL = (lds_int*)(smem + L::FL);
  f32x4* const ZB = reinterpret_cast<f32x4*>(smem + L::ZB);
  frag* const GT = reinterpret_cast<frag*>(smem + L::GT);
  frag* const X2S = reinterpret_cast<frag*>(smem + L::X2S) + w * L::XS * 64;
  uint32_t* const LRs = reinterpret_cast<uint32_t*>(smem + L::LR);
  float* const GAM = reinterpret_cast<float*>(smem + L::PRM);
  float* const BET = GAM + D;
  float* const B1s = BET + D;  // b1: each wave reads and updates only its own slice

  // scale folding as in the TTT-Linear kernels: G'' = -sc lr G, M'' = (token_eta[t] / sc)(1 + A)
  const float te_last = a.token_eta[K - 1];
  const bool upd = te_last != 0.f;
  const float sc = upd ? te_last : 1.f;
  const float rho_r = (c < K) ? a.token_eta[c] / sc : 0.f;
  const frag ident_r = identity_frag<T>(c, g);
  auto rho = [&]() { return D > 64 ? RHO[c] : rho_r; };
  auto identity = [&]() { return D > 64 ? IDs[lane] : ident_r; };
  const size_t sb = a.state_per_batch ? bh : (size_t)h;
  int own = own_offset<1>(red ? w : 0, 0, g);  // first of this lane's four features of tile w

  // ---- state and parameters
  f32x4 W1c[NT][HT], W2c[HT][NT];
  {
    const float* W1 = a.W1_0 + sb * (size_t)D * F;
    const float* W2 = a.W2_0 + sb * (size_t)D * F;
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const int hb = 16 * (w * HT + j);
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
  if (tid < 16) RHO[tid] = tid < K ? a.token_eta[tid] / sc : 0.f;
  if (w == 0) IDs[lane] = identity_frag<T>(c, g);
#pragma unroll
  for (int r = 0; r < 4; ++r) b2T[r] = a.b2_0[sb * D + own + r];
  // the second layer is carried centred (see row_means16)
#pragma unroll
  for (int j = 0; j < HT; ++j) {
    const f32x4 m = row_means16<NT>(W2c[j], inv_d);
#pragma unroll
    for (int I = 0; I < NT; ++I) W2c[j][I] -= m;
  }
  // Formed by whole waves from one load each; in the chain of loads 128 units x 2048 tokens took 647 instead of 637 us (d = 96).  Not
  // so in the backward kernels and on pairs of CUs, where it changes nothing or costs 0.2 %.
  float b2_mean = sum_in_order<D>(a.b2_0 + sb * D) * inv_d;  // as mean_of
  asm volatile("" : "+v"(b2_mean));
  b2T -= b2_mean;
  const float sum_a = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(sum_in_order<D, true>(a.gamma + h * D))));
  for (int i = tid; i < D; i += 512) {
    GAM[i] = a.gamma[h * D + i];
    BET[i] = a.beta[h * D + i];
  }
  for (int i = tid; i < F; i += 512) B1s[i] = a.b1_0[sb * F + i];

  // ---- staging of the xq / xk / xv rows of a mini-batch: global -> LDS without passing through
  // registers, in wave blocks of 64 lanes x 16 bytes.  A block never straddles two tensors; lanes
  // whose token is past a short mini-batch are masked off and their LDS rows keep the zeros
  // written below.  Three buffers: mini-batch st+1 is fetched while st is computed, and rows of
  // st are still read (for the W1 update) after the slowest wave has started st+1's fetch.
  // Per wave block a running source address, scalar like everything but the lane's offset.
  constexpr int NBLK = L::IN1 / 1024, NBI = (NBLK + 3) / 4;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem);
  const unsigned step = (unsigned)(K * D * ES);
  const unsigned char* srcp[NBI];
#pragma unroll
  for (int it = 0; it < NBI; ++it) {
    const int b = (w & 3) + 4 * it, ten = (1024 * b) / L::TILE;
    srcp[it] = static_cast<const unsigned char*>(ten == 0 ? a.xq : ten == 1 ? a.xk : a.xv) + bh * (size_t)a.seq_stride * (D * ES);
  }
  const unsigned char* lrp = static_cast<const unsigned char*>(a.lr) + bh * (size_t)a.seq_stride * ES;
  unsigned char* const outp = static_cast<unsigned char*>(a.out) + bh * (size_t)a.seq_stride * (D * ES);
  unsigned fdst = lds0 + L::IN + 1024 * (w & 3), flr = lds0 + L::LR;  // where the next mini-batch goes
  const int n_stages = a.n_stages;
  auto fetch = [&](int stage) {
    if (stage >= n_stages) return;
#pragma unroll
    for (int it = 0; it < NBI; ++it) {
      const int b = w + 4 * it;
      const unsigned off = (1024u * b) % L::TILE + 16u * lane;
      if (b < NBLK && off < step) lds_dma16(srcp[it], off, fdst + 4096 * it);
      srcp[it] += step;
    }
    // lr as zero-extended bf16 words, copied like the tiles (a register load here would make the compiler
    // wait for every copy in flight); absent tokens read a clamped position and are zeroed at use
    if (w == 0 && lane < 16) lds_dma2(lrp, 2u * (unsigned)min(lane, K - 1), flr);
    lrp += K * ES;
    const bool wrap = stage % 3 == 2;
    fdst += wrap ? -2 * L::IN1 : L::IN1;
    flr += wrap ? -128 : 64;
  };
  // staged row of token c of tensor ten (0 xq, 1 xk, 2 xv)
  auto row = [&](int buf, int ten) -> const elem* {
    return reinterpret_cast<const elem*>(smem + L::IN + buf * L::IN1 + ten * L::TILE) + c * D;
  };

  for (int i = tid; i < (L::PRM - L::IN) / 4; i += 512) reinterpret_cast<float*>(smem)[i] = 0.f;
  for (int i = tid; i < 6 * 2 * 16 * 4; i += 512) EX[i] = 0.f;
  if (tid < 2 * 2 * 16 * 4) EXO[tid] = 0.f;
  if (tid < NW) FL[tid] = 0;
  __syncthreads();
  if (older) fetch(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- reducers: lane group g publishes sums g and g + 4 (six in all) of reducer w
  auto publish = [&](const float (&S)[6]) {
    const float v0 = xg_sum4_scatter(S[0], S[1], S[2], S[3]);
    const float v1 = xg_sum2_scatter(S[4], S[5]);
    EX[(((g)*2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = v0;
    EX[(((4 + (g >> 1)) * 2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = v1;  // two lane groups write the same value
  };  // (with this and every sum from its first term, 128 units x 2048 tokens: d = 64 418 -> 413 us; saving, d = 96 682 -> 674)
  // sums i and j of those exchanged at ex
  auto collect2 = [&](const float* ex, int i, int j, float& a, float& b) {
    f32x4 v[4] = {};
    v[0] = *reinterpret_cast<const f32x4*>(ex + ((i * 2 + 0) * 16 + c) * 4);
    v[1] = *reinterpret_cast<const f32x4*>(ex + ((j * 2 + 0) * 16 + c) * 4);
    if (NT > 4) {
      v[2] = *reinterpret_cast<const f32x4*>(ex + ((i * 2 + 1) * 16 + c) * 4);
      v[3] = *reinterpret_cast<const f32x4*>(ex + ((j * 2 + 1) * 16 + c) * 4);
    }
    together(v);
    a = (v[0][0] + v[0][1]) + (v[0][2] + v[0][3]);
    b = (v[1][0] + v[1][1]) + (v[1][2] + v[1][3]);
    if (NT > 4) {
      a += (v[2][0] + v[2][1]) + (v[2][2] + v[2][3]);
      b += (v[3][0] + v[3][1]) + (v[3][2] + v[3][3]);
    }
  };

  // ---- output path: the sums, causal correction and row moments of mini-batch t by the older waves at the end of phase A of
  // t + 1, wave w the tiles w + 4 i; the stores by the waves that reduce no Z2 tile, beside the reducers in phase B.
  // There is no barrier between a wave's partial blocks and the wave that adds them up: each wave waits for its blocks to
  // be in LDS (lds_done) and then counts up its own word there.  Blocks and word are LDS instructions both (FL carries the
  // address space).  The wait needs no bound: on its way from B3 to the counter a wave waits for nobody.
  constexpr int EW = NW - NT, EPW = (NT + EW - 1) / EW, OPW = LATE ? 1 : (NT + 3) / 4;
  static_assert(!LATE || EPW == 1, "one tile per wave");
  auto otile = [&](int i) { return LATE ? w - NT : w + 4 * i; };
  auto output_finish = [&](int stage) {
    if (!LATE) {
      while (__builtin_amdgcn_ballot_w64(__hip_atomic_load(FL + (lane & 7), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= stage) != 0) {
      }
      lds_done();
    }
    frag m2f;
    {
      // M2[s][t] = (token_eta[t] / sc)(1 + A2[t][s]) for s <= t
      const float rho_c = rho();
      f32x4 v[NW];
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) v[ww] = PA[ww * 64 + lane];
      together(v);
      const f32x4 at = sum_tiles(v);
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? rho_c * (1.f + at[r]) : 0.f;
      m2f = IO::to_frag(m);
    }
    float s[2 * OPW];
#pragma unroll
    for (int i = 0; i < OPW; ++i) {
      const int I = otile(i);
      s[2 * i] = s[2 * i + 1] = 0.f;
      if (I >= NT) continue;
      f32x4 v[NW];
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) v[ww] = P2[(ww * NT + I) * 64 + lane];
      together(v);
      f32x4 zo = sum_tiles(v);
      IO::mma(zo, read_tr(GT + (((stage & 1) * NT) + I) * 64 + tr_lane(lane)), m2f);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sum_term(s[2 * i], r == 0, zo[r]);
        sum_term(s[2 * i + 1], r == 0, zo[r], zo[r]);
      }
      ZB[I * 64 + lane] = zo;
    }
    // lane group g: sum g & 1 of this wave's tile g / 2
    static_assert(OPW <= 2, "two sums of two tiles, a lane group each");
    if constexpr (OPW > 1) {
      const float v = xg_sum4_scatter(s[0], s[1], s[2], s[3]);
      const int I = otile(g >> 1);
      if (I < NT) EXO[(((g & 1) * 2 + (I >> 2)) * 16 + c) * 4 + (I & 3)] = v;
    } else {
      const float v = xg_sum2_scatter(s[0], s[1]);
      const int I = otile(0);
      if (I < NT) EXO[(((g >> 1) * 2 + (I >> 2)) * 16 + c) * 4 + (I & 3)] = v;
    }
  };
  // out = xq + gamma (zbar - mu) rstd + beta, tiles (w - NT) + EW i for i in [i0, i1)
  float o_mu = 0.f, o_rstd = 0.f;
  auto output_stats = [&]() {
    float ms;
    collect2(EXO, 0, 1, o_mu, ms);
    o_mu *= inv_d;
    o_rstd = __builtin_amdgcn_rsqf(fmaxf(ms * inv_d - o_mu * o_mu, 0.f) + eps);
  };
  auto output_emit = [&](int stage, int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      const int I = (w - NT) + EW * i;
      if (I >= NT) continue;
      const int own_o = own_offset<1>(I, 0, g);
      const f32x4 zb = ZB[I * 64 + lane];
      const frag qo = load4<T>(row(stage % 3, 0) + own_o);
      const f32x4 gam = *reinterpret_cast<const f32x4*>(GAM + own_o), bet = *reinterpret_cast<const f32x4*>(BET + own_o);
      const f32x4 o = IO::to_f32(qo) + bet + gam * ((zb - o_mu) * o_rstd);
      elem* po = reinterpret_cast<elem*>(outp + (size_t)stage * step) + (c * D + own_o);
      if (c < K) store4<T>(po, o);
    }
  };
  // partial tiles of X W2 over this wave's hidden units, two at a time
  auto partials = [&](f32x4* P, const frag (&x)[HT], bool bias) {
    f32x4* p = P + w * NT * 64 + lane;
#pragma unroll
    for (int I = 0; I < NT; I += 2) {
      f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
      if (bias && I == w) p0 = b2T;
      if (bias && I + 1 == w) p1 = b2T;
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2) {
        IO::mma2(p0, IO::to_frag(W2c[j][I]), IO::to_frag(W2c[j + 1][I]), x[j], x[j + 1]);
        IO::mma2(p1, IO::to_frag(W2c[j][I + 1]), IO::to_frag(W2c[j + 1][I + 1]), x[j], x[j + 1]);
      }
      if (HT & 1) {
        IO::mma2(p0, IO::to_frag(W2c[HT - 1][I]), IO::zero(), x[HT - 1], IO::zero());
        IO::mma2(p1, IO::to_frag(W2c[HT - 1][I + 1]), IO::zero(), x[HT - 1], IO::zero());
      }
      p[I * 64] = p0;
      p[(I + 1) * 64] = p1;
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  for (int st = 0; st < n_stages; ++st) {
    const int buf = st % 3;
    frag* const GTc = GT + (st & 1) * NT * 64;
    RELANE();
    if (older) fetch(st + 1);

    // ================= phase A: everything that needs only W1, W2 and the inputs
    f32x4 z1[HT], zq[HT];
    // Z1^T and (XQ W1 + b1)^T for this wave's hidden units
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
    // X2 = gelu(Z1), gelu'(Z1)
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
      // materialise both now: left to itself the compiler postpones gelu' to its use after the
      // barriers and keeps (or spills) twice as many intermediates until then
      asm volatile("" : "+v"(x2f[j]), "+v"(dg[j]));
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < L::XS; ++j) X2S[j * 64 + lane] = x2f[j];
    partials(P1, x2f, false);
    // of the two waves of a SIMD the older runs ahead and would wait at B1 for 2 k cycles
    if (!LATE && outs && st > 0) output_finish(st - 1);
    // M1[s][t] = (token_eta[t] / sc)(1 + A1[t][s]) for s <= t
    if (w == 3) {
      const float rho_c = rho();
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
      M1s[(st & 1) * 64 + lane] = IO::to_frag(m);
    }
    lds_barrier();  // ---- B1
    RELANE();

    // ================= phase B: reducers: full Z2 tile and its row moments;
    //                          the other waves: stores of the previous mini-batch's output
    f32x4 z = {0.f, 0.f, 0.f, 0.f}, bq = z;
    if (red) {
      const f32x4* p = P1 + w * 64 + lane;
      const frag ko = load4<T>(row(buf, 1) + own), vo = load4<T>(row(buf, 2) + own);
      const f32x4 gam = *reinterpret_cast<const f32x4*>(GAM + own), bet = *reinterpret_cast<const f32x4*>(BET + own);
      f32x4 v[NW];
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) v[ww] = p[ww * NT * 64];
      together(v);
      z = b2T;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) z += v[ww];
      const f32x4 tgt = bet - (IO::to_f32(vo) - IO::to_f32(ko));
      bq = gam * tgt;
      float S[6];
      const f32x4 a2 = gam * gam, az = a2 * z;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sum_term(S[0], r == 0, z[r]);
        sum_term(S[1], r == 0, z[r], z[r]);
        sum_term(S[2], r == 0, a2[r], z[r]);
        sum_term(S[3], r == 0, az[r], z[r]);
        sum_term(S[4], r == 0, gam[r], tgt[r]);
        sum_term(S[5], r == 0, bq[r], z[r]);
      }
      publish(S);
    } else if (outw && st > 0) {
      if (LATE) {
        output_finish(st - 1);
      } else {
        output_stats();
        output_emit(st - 1, 0, 1);
      }
    }
    lds_barrier();  // ---- B2
    RELANE();

    // ================= phase C: reducers: G2''
    if (red) {
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
    } else if (outw && st > 0) {
      if (LATE) output_stats();
      output_emit(st - 1, LATE ? 0 : 1, EPW);
    }
    // the next mini-batch's rows must have landed before anybody passes B3
    if (older) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();  // ---- B3
    RELANE();

    // ================= phase D: G1, Zbar1, Xbar2, split-k partials of the output path, updates
    // The factors of this mini-batch's state update for ttt_mlp_bwd, eta_last * G1 [16 x 4d] and eta_last * G2
    // [16 x d] (row = token), exactly as the update applies them: rounded to the operand type, sign undone
    // (G'' = -eta_last * lr * G); zeros when token_eta[K-1] = 0 switches the update off.
    const size_t saved_at = bh * (size_t)n_stages + st;
    unsigned char* const facp = SAVE && a.fac_save != nullptr ? a.fac_save + saved_at * ((NW * HT + NT) * 512) : nullptr;
    if (SAVE && facp != nullptr && red)
      *reinterpret_cast<frag*>(facp + (NW * HT + w) * 512 + 8u * lane) = read_tr(GTc + w * 64 + tr_lane(lane));
    if (SAVE && a.G2_save != nullptr && red) {
      const f32x4 v = upd ? -IO::to_f32(GTc[w * 64 + lane]) : f32x4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(a.G2_save + saved_at * (16 * D) + (unsigned)(c * D + own)) = v;
    }
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W2c[j][I]);
    // G1''^T = (W2 G2''^T) gelu'(Z1)
    frag G1d[HT];
    {
      const frag ident = identity();
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
        const frag g1b = IO::to_frag(acc[j] * dg[j]);
        t[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        IO::mma(t[j], g1b, ident);
        if (SAVE && a.G1_save != nullptr) {
          const f32x4 v = upd ? -IO::to_f32(g1b) : f32x4{0.f, 0.f, 0.f, 0.f};
          *reinterpret_cast<f32x4*>(a.G1_save + saved_at * (16 * F) + 16 * (w * HT + j) + (unsigned)(c * F + 4 * g)) = v;
        }
      }
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        G1d[j] = IO::to_frag(t[j]);
        if (SAVE && facp != nullptr) *reinterpret_cast<frag*>(facp + (w * HT + j) * 512 + 8u * lane) = G1d[j];
      }
    }
    // Zbar1^T = (XQ W1 + b1)^T + G1''^T M1
    frag xbf[HT];
    {
      const frag Mf = M1s[(st & 1) * 64 + lane];
#pragma unroll
      for (int j = 0; j < HT; ++j) IO::mma(zq[j], G1d[j], Mf);
    }
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
      for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, x2f[j], x2f[j + 1], xbf[j], xbf[j + 1]);
      if (HT & 1) IO::mma2(p, x2f[HT - 1], IO::zero(), xbf[HT - 1], IO::zero());
      PA[w * 64 + lane] = p;
    }
    partials(P2, xbf, true);
    if (!LATE) {
      lds_done();  // the blocks are in LDS before their counter says so
      if (lane == 0) __hip_atomic_store(FL + w, st + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (upd) {
      frag x2d[HT];
      {
        const frag ones = splat_frag<T>(1.f);
        f32x4 b[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          if (j < L::XS) {
            x2d[j] = read_tr(X2S + j * 64 + tr_lane(lane));
          } else {
            f32x4 t = {0.f, 0.f, 0.f, 0.f};
            IO::mma(t, x2f[j], identity());
            x2d[j] = IO::to_frag(t);
          }
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
        const frag kn = read_tr(kr + 32 * (In >> 1) + 4 * (In & 1)), gn = read_tr(gr + (I + 1 < NT ? I + 1 : w < NT ? w : 0) * 64);
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          IO::mma(W1c[I][j], kd, G1d[j]);
          IO::mma(W2c[j][I], x2d[j], g2d);
        }
        kd = kn;
        g2d = gn;
        __builtin_amdgcn_sched_barrier(0);
      }
      if (red) IO::mma(b2T, g2d, splat_frag<T>(1.f));
    }
  }

  // ---- the last mini-batch's output
  if (LATE) lds_barrier();
  if (outs) output_finish(n_stages - 1);
  lds_barrier();
  if (outw) {
    output_stats();
    output_emit(n_stages - 1, 0, EPW);
  }

  if (SAVE && a.state_save != nullptr) {
    f32x4* s1 = reinterpret_cast<f32x4*>(a.state_save + bh * (size_t)(2 * D * F)) + (w * NT * HT) * 64 + lane;
    f32x4* s2 = s1 + NW * NT * HT * 64;
#pragma unroll
    for (int j = 0; j < HT; ++j) {
#pragma unroll
      for (int I = 0; I < NT; ++I) {
        s1[(I * HT + j) * 64] = W1c[I][j];
        s2[(j * NT + I) * 64] = W2c[j][I];
      }
      const int hb = 16 * (w * HT + j);
      if (c == 0) store4<F32>(a.b1_save + bh * F + hb + 4 * g, *reinterpret_cast<const f32x4*>(B1s + hb + 4 * g));
    }
    if (red && c == 0) store4<F32>(a.b2_save + bh * D + own, b2T);
  }
  if (SAVE && a.W1 == nullptr) return;
  // ---- final state.  Second layer: initial value + (centred value now - centred value at the start), the start
  // value formed again exactly as above, so a sequence that never updates the state returns it bit for bit.
  {
    float* W1 = a.W1 + bh * (size_t)D * F;
    float* W2 = a.W2 + bh * (size_t)D * F;
    const float* W2i = a.W2_0 + sb * (size_t)D * F;
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const int hb = 16 * (w * HT + j);
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
          W1[(size_t)feat(I, 4 * g + r) * F + hb + c] = W1c[I][j][r];
          W2[(size_t)(hb + 4 * g + r) * D + feat(I, c)] = fin[r];
        }
      }
      if (c == 0) store4<F32>(a.b1 + bh * F + hb + 4 * g, *reinterpret_cast<const f32x4*>(B1s + hb + 4 * g));
    }
    if (red) {
      const float bb = mean_of(a.b2_0 + sb * D, D, inv_d);
      const f32x4 v0 = *reinterpret_cast<const f32x4*>(a.b2_0 + sb * D + own);
      const f32x4 start = v0 - bb;
      if (c == 0) store4<F32>(a.b2 + bh * D + own, v0 + (b2T - start));
    }
  }
}

#undef RELANE

}  // namespace ttt
