// TTT-MLP fused backward with the state and its gradient resident in registers (bf16 I/O, head_dim 32 / 64 / 96).
//
// Arithmetic: the gradient of the inner loop of reference rust/core/src/mlp.rs:127-208 looped as
// rust/core/src/inner.rs:25-50 (the reference differentiates it with Burn autodiff), as a reverse scan over mini-batches
// with the second-order LayerNorm (rust/fused/src/linear_fused_tile/layer_norm.rs:428-709) and GELU'' terms.
//
// Why: the scan on tiles in memory (ttt_mlp_bwd.hip.h) passes over W1, W2, dW1, dW2 21 times per mini-batch, 57 GB at
// 128 units x 2048 tokens of d = 96, and is bound by that traffic: 9.3 ms.  This kernel: 2.07 ms there, 1.76 ms for 16
// units: bound by the producer's products, and on a full chip by the hand-over of 289 KB per mini-batch and unit besides
// (more than the L2 of 16 units holds).  Nothing of the state moves here: a unit is worked on by two roles, each of which keeps its
// matrices as MFMA accumulator tiles in the
// registers of one workgroup of eight waves, the hidden axis (4 d) cut into eight slices as in the forward
// (ttt_mlp_fwd_rr.hip.h):
//   producer  W1[:, slice], W2[slice, :]: walks the state back (the update factors the forward saved), recomputes the
//             forward's intermediates, and carries out everything that needs no gradient of the state: the output
//             LayerNorm backward, dXbar2, dZbar1, d_xq
//   consumer  dW1[:, slice], dW2[slice, :]: S = X dW, the second-order LayerNorm, dZ2, dZ1, d_xk, d_xv, the rank-48 /
//             rank-32 updates
// Elementwise work in the hidden axis stays inside a wave.  Contractions over the hidden axis are split over the waves
// (partial tiles in LDS, wave I < d/16 adds up feature tile I).  What crosses is a slot of global memory per mini-batch
// (fragments exactly as the consumer's lanes hold them, 1 KiB per wave instruction): the transposed bf16 images of W1 and
// W2, which the producer forms for its own products, the hidden tiles and the LayerNorm tiles.
//
// All matrix operands are rounded to bf16, once for all products that take them, and accumulated in f32; state, gradients
// and elementwise tiles are f32 (G2 in the sum behind d_lr: two bf16 parts).  Against float64 every gradient's error is
// that of the scan on tiles with bf16 operands: ratios 0.93 - 1.01 over 24 cases of 9 - 128 mini-batches.
// W2 and b2 are carried centred (ttt_mlp_fwd_rr.hip.h): every use of W2 here meets rows that sum to zero or a LayerNorm.
//
// Two workgroups per unit (up to 128 units): producer and consumer run side by side on two CUs of one XCD, the producer a
// mini-batch ahead, and follow each other through two counters (see ttt_mlp_bwd.hip.h for the placement, the XCD
// check, the bounded waits and the poison value; they are the same here).  One workgroup per unit: the roles run in
// turn, launch by launch, over as many mini-batches as there are slots; the matrices are stored in accumulator order
// between launches.  The same code and the same bits.
//
// Registers.  At d = 96 a role holds 144 of 256 in its matrices, and a value spilled inside the loop is dear: its reload waits
// for every load and store of the wave that is in flight, up to 5 k cycles on a full chip.  Hence what is read from LDS
// (transposing loads of the staged rows, sums of gradients, parked tiles) or formed again rather than held, and the
// scheduler's register tracking that the d = 96 instance is compiled with (build.py).  128 units x 2048 tokens, d = 96:
// 2645 us with fourteen reloads in the two loops, 2167 with two, 2066 with none; d = 64 1440 -> 1375, d = 32 845 -> 818 us.
#pragma once
#include "ttt_engine.hip.h"
#include "ttt_frag.hip.h"
#include "ttt_linear_fwd_mw.hip.h"

namespace ttt {

constexpr unsigned kMlpRpPoison = 0xffffffffu;
constexpr int kMlpRpFlagWords = 32;  // per unit: [0] producer's count, [1] consumer's count, [2], [3] XCD ids

// sizes that the host plans with too
template <int D>
struct MlpRp {
  static constexpr int NW = 8, NT = D / 16, F = 4 * D, HT = F / 16 / NW, NQ = NT / 2;
  // update factors of a mini-batch: [wave][hidden tile] fragments of G1'', then [feature tile] fragments of G2''
  static constexpr int FAC = (NW * HT + NT) * 512;
  // hand-over slot: per wave W2^T, W1^T images, hidden tiles; per feature tile LayerNorm tiles; small matrices, scalars
  static constexpr int W2T = 0, W1T = W2T + HT * NQ * 1024, XT = W1T + HT * NQ * 1024, DG = XT + HT * 1024,
                       UG = DG + HT * 1024, G1 = UG + HT * 1024, DT = G1 + HT * 1024, WAVE = DT + HT * 512;
  static constexpr int XH = 0, GO = 1024, G2 = 2048, MZ = 3072, GG = 4096, ZD = 5120, TILE = ZD + 512;
  static constexpr int TILES = NW * WAVE, SMALL = TILES + NT * TILE;
  static constexpr int M1T = SMALL, A2T = M1T + 512, A1T = A2T + 512, SCAL = A1T + 512;  // SCAL: six rows of 16 floats
  static constexpr int ZB1 = SCAL + 6 * 64, ZB2 = ZB1 + F * 4;  // column sums of dZbar1 [4d] and dZbar2 [d], f32
  static constexpr int SLOT = (ZB2 + D * 4 + 1023) / 1024 * 1024;
};

struct MlpBwdRpArgs {
  const void *xq, *xk, *xv, *d_out, *lr;
  const float *token_eta, *gamma, *beta;
  const unsigned char* fac;  // [units][n_stages][MlpRp::FAC]
  float* state;              // [units][2 * d * 4d]: W1, W2 (centred) in accumulator order, the state entering `last`
  float *b1, *b2;            // [units][4d], [units][d] (centred): its biases
  unsigned char* hand;       // [units][slots][MlpRp::SLOT]
  const float *up_W1, *up_b1, *up_W2, *up_b2;  // upstream gradients of the final state, or null
  float *d_W1, *d_b1, *d_W2, *d_b2;
  void *d_xq, *d_xk, *d_xv, *d_lr;
  float *d_token_eta, *d_gamma, *d_beta;
  unsigned *flags, *lost_count;
  int B, H, K, n_stages, seq_stride, slots;
  int first, last;  // mini-batches last - 1 .. first of this launch
  int role;         // 0 producer, 1 consumer, 2: two workgroups per unit
  float eps;
  unsigned spin_limit;
  int agent_release;
};

template <int D>
struct MlpRpLds {
  using S = MlpRp<D>;
  static constexpr int NT = S::NT, NW = S::NW;
  static constexpr int TILE = 16 * D * 2, IN1 = 4 * TILE;
  static constexpr int IN = 0;                     // [2 buffers][xq, xk, xv, d_out][16][d] bf16
  static constexpr int LR = IN + 2 * IN1;          // [2][16] bf16 words
  static constexpr int PA = LR + 2 * 64 + 128;     // [NW][64] f32x4: partial [16 x 16] blocks
  static constexpr int PB = PA + NW * 1024;        // [2][NW][NT][64] f32x4: partial [16 x d] tiles
  static constexpr int GT = PB + 2 * NW * NT * 1024;  // fragments by feature tile
  static constexpr int ZT = GT + NT * 512, DG = ZT + NT * 512;  // DG: producer: [NT][64] f32x4, d gamma by lane
  static constexpr int GS = DG + NT * 1024;
  static constexpr int EX = GS + NT * 512;         // [8 sums][2][16 tokens] f32x4 (reducer index % 4)
  static constexpr int PRM = EX + 8 * 2 * 16 * 16;  // gamma[d], beta[d], b1[4d]
  static constexpr int QS = PRM + 6 * D * 4;       // [NW][16] floats
  static constexpr int CTL = QS + NW * 64;
  static constexpr int DB = CTL + 16;              // [NT][64] f32x4, d beta by lane (the consumer's d gamma: in PA)
  static constexpr int B2 = DB + NT * 1024;        // consumer: d b2 [d]
  static constexpr int GL = B2 + D * 4;            // consumer: [NT][64] fragments of what G2 loses as an operand
  static constexpr int BYTES = GL + NT * 512;
  static_assert(BYTES <= 160 * 1024, "exceeds the 160 KiB of LDS of a gfx950 CU");
  static_assert(2 * S::HT <= NT, "what waits for phase D fits a wave's partial tiles");
};

// gelu_tanh_pair and gelu_tanh_all with their common factors taken out: the producer evaluates them twice per element and
// mini-batch and is bound by its vector instructions at head_dim 32 and 64 (128 units of 2048 tokens, d = 64, forward and
// backward: 1902 -> 1879 us).  Against float64 the 2-norm errors of y, y', y'' on N(0, s^2) inputs, s = 0.02 .. 10, are theirs
// or smaller.
__device__ __forceinline__ void gelu_of_tanh(float x, float& y, float& dy, float& hp, float& du, float& s, float& sdu, float& t) {
  const float c = 0.7978845608f, ca = 0.7978845608f * 0.044715f;
  const float x2 = x * x;
  t = tanh_nobranch(x * __builtin_fmaf(ca, x2, c));
  hp = __builtin_fmaf(0.5f, t, 0.5f);
  s = __builtin_fmaf(-t, t, 1.f);
  du = __builtin_fmaf(3.f * ca, x2, c);
  sdu = s * du;
  y = x * hp;
  dy = __builtin_fmaf(0.5f * x, sdu, hp);
}
__device__ __forceinline__ void gelu_pair(float x, float& y, float& dy) {
  float hp, du, s, sdu, t;
  gelu_of_tanh(x, y, dy, hp, du, s, sdu, t);
}
__device__ __forceinline__ void gelu_all(float x, float& y, float& dy, float& ddy) {
  float hp, du, s, sdu, t;
  gelu_of_tanh(x, y, dy, hp, du, s, sdu, t);
  ddy = __builtin_fmaf(x, __builtin_fmaf(3.f * 0.7978845608f * 0.044715f * x, s, -(t * du) * sdu), sdu);
}

// Lane coordinates formed anew: the addresses derived from them are many and all loop-invariant; hoisted out of the loop
// they would be spilled and reloaded, and a reload waits for every load in flight (see ttt_mlp_fwd_rr.hip.h).
#define RP_RELANE() x.relane()
#define RP_FENCE() __builtin_amdgcn_sched_barrier(0)

namespace rp {
using IO = Io<BF16>;
using frag = IO::frag;

__device__ __forceinline__ frag neg(frag f) {
  const u32x2 v = __builtin_bit_cast(u32x2, f);
  return __builtin_bit_cast(frag, u32x2{v[0] ^ 0x80008000u, v[1] ^ 0x80008000u});
}
// A-side fragment X[m, k] -> the fragment of X^T (exact: the values are bf16 already)
__device__ __forceinline__ frag flip(frag x, frag ident) {
  f32x4 t = {0.f, 0.f, 0.f, 0.f};
  IO::mma(t, x, ident);
  return IO::to_frag(t);
}
// one 16-deep product accumulated by the 32-deep instruction: for accumulators that other 32-deep products write
__device__ __forceinline__ void mmz(f32x4& acc, frag a, frag b) { IO::mma2(acc, a, IO::zero(), b, IO::zero()); }
__device__ __forceinline__ u32x4 pair(frag a, frag b) {
  const u32x2 x = __builtin_bit_cast(u32x2, a), y = __builtin_bit_cast(u32x2, b);
  return u32x4{x[0], x[1], y[0], y[1]};
}
__device__ __forceinline__ frag lo(u32x4 v) { return __builtin_bit_cast(frag, u32x2{v[0], v[1]}); }
__device__ __forceinline__ frag hi(u32x4 v) { return __builtin_bit_cast(frag, u32x2{v[2], v[3]}); }
__device__ __forceinline__ void forget(f32x4& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(f32x4& v) { asm volatile("" : "+v"(v)::"memory"); }

// an element of a slot: uniform base + 32-bit offset
template <class V>
__device__ __forceinline__ V& at(const unsigned char* base, unsigned off) {
  return *reinterpret_cast<V*>(const_cast<unsigned char*>(base) + off);
}

// lds_dma4 with device scope (see Slot)
__device__ __forceinline__ void lds_dma4_dev(const void* base, unsigned lane_off, unsigned lds_base) {
  unsigned saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2 sc1\n\ts_nop 0\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(lane_off), "s"(uniform_ptr(base)), "s"(lds_base)
      : "memory");
}
// The consumer's reads of a slot: device-scope loads (sc1), which do not look in the CU's vector cache and so see what the
// producer's CU stored into the L2 behind both.  (Dropping the cache instead takes an instruction of device scope, which
// also drops lines of the L2; what one of workgroup scope does is not for other workgroups to rely on.)  A slot is read once
// or twice, so the cache holds nothing worth keeping of it: forward and backward at 128 units of 2048 tokens, d = 96, take
// 3554 us, with a device-scope acquire per mini-batch 3908 us.  Scalar offset + lane offset.
struct Slot {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ Slot(const unsigned char* base, int bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(base), 0, bytes, 0x00027000)) {}
  template <class V>
  __device__ __forceinline__ V get(unsigned lane_off, unsigned off) const {
    static_assert(sizeof(V) == 4 || sizeof(V) == 8 || sizeof(V) == 16, "");
    if constexpr (sizeof(V) == 16)
      return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_off, off, 16));
    else if constexpr (sizeof(V) == 8)
      return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane_off, off, 16));
    else
      return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane_off, off, 16));
  }
};

// What both roles need of their place: lane coordinates, LDS regions, input staging, exchange of row sums.
template <int D, int TENSORS>
struct Base {
  using S = MlpRp<D>;
  using L = MlpRpLds<D>;
  static constexpr int NW = S::NW, NT = S::NT, F = S::F, HT = S::HT, NQ = S::NQ;
  static constexpr float inv_d = 1.0f / D;
  static constexpr bool ROOM = D <= 64;  // registers for more loads in flight beside the state (d = 96: spills, 2.3 ms)
  const MlpBwdRpArgs& a;
  unsigned char* smem;
  size_t bh;
  int tid, w, lane, c, g, K, h, own;
  bool red, pair;
  f32x4 *PA, *PB;
  frag *GT, *ZT, *GS;
  float *EX, *GAM, *BET, *B1s, *QS;
  uint32_t* LRs;
  int* lost;
  frag ident, ones;
  float te_last, te_c, sum_a;
  const unsigned char* src[TENSORS];  // first row of the unit
  const unsigned char* lrp;

  __device__ __forceinline__ void relane() {
    asm volatile("" : "+v"(lane));
    c = lane & 15;
    g = lane >> 4;
    own = own_offset<1>(red ? w : 0, 0, g);
  }
  __device__ __forceinline__ Base(const MlpBwdRpArgs& a_, unsigned char* sm, size_t bh_, bool pair_)
      : a(a_), smem(sm), bh(bh_), pair(pair_) {
    tid = threadIdx.x;
    w = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    c = lane & 15;
    g = lane >> 4;
    K = a.K;
    h = (int)(bh % a.H);
    red = w < NT;
    own = own_offset<1>(red ? w : 0, 0, g);
    PA = reinterpret_cast<f32x4*>(smem + L::PA);
    PB = reinterpret_cast<f32x4*>(smem + L::PB);
    GT = reinterpret_cast<frag*>(smem + L::GT);
    ZT = reinterpret_cast<frag*>(smem + L::ZT);
    GS = reinterpret_cast<frag*>(smem + L::GS);
    EX = reinterpret_cast<float*>(smem + L::EX);
    GAM = reinterpret_cast<float*>(smem + L::PRM);
    BET = GAM + D;
    B1s = BET + D;
    QS = reinterpret_cast<float*>(smem + L::QS);
    LRs = reinterpret_cast<uint32_t*>(smem + L::LR);
    lost = reinterpret_cast<int*>(smem + L::CTL);
    ident = identity_frag<BF16>(c, g);
    ones = splat_frag<BF16>(1.f);
    te_last = a.token_eta[K - 1];
    te_c = c < K ? a.token_eta[c] : 0.f;
    sum_a = 0.f;
    for (int f = 0; f < D; ++f) sum_a += a.gamma[h * D + f] * a.gamma[h * D + f];
    for (int i = tid; i < D; i += 512) {
      GAM[i] = a.gamma[h * D + i];
      BET[i] = a.beta[h * D + i];
    }
    for (int i = tid; i < (L::PA - L::IN) / 4; i += 512) reinterpret_cast<float*>(smem)[i] = 0.f;
    for (int i = tid; i < 8 * 2 * 16 * 4; i += 512) EX[i] = 0.f;
    const size_t r0 = bh * (size_t)a.seq_stride * (D * 2);
    const void* const t[4] = {a.xq, a.xk, a.xv, a.d_out};
#pragma unroll
    for (int i = 0; i < TENSORS; ++i) src[i] = static_cast<const unsigned char*>(t[i]) + r0;
    lrp = static_cast<const unsigned char*>(a.lr) + bh * (size_t)a.seq_stride * 2;
  }
  // the LDS address of the dynamic allocation, as a scalar
  __device__ __forceinline__ unsigned lds0() const {
    return __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem);
  }
  // rows of a mini-batch, global -> LDS without passing registers; tokens past a short mini-batch keep the zeros
  __device__ __forceinline__ void fetch(int stage) {
    if (stage < a.first) return;
    const unsigned in0 = lds0();
    const unsigned dst = in0 + L::IN + (stage & 1) * L::IN1;
    const size_t tok0 = (size_t)stage * (unsigned)(K * D * 2);
    // a tensor's tile is TILE / 1024 wave blocks; the blocks of all tensors are dealt to the waves in turn
    constexpr int PER = L::TILE / 1024;
#pragma unroll
    for (int i = 0; i < TENSORS; ++i)
#pragma unroll
      for (int b = 0; b < PER; ++b)
        if (w == (i * PER + b) % NW) {
          const int off = 1024 * b + 16 * lane;
          if (off < K * D * 2) lds_dma16(src[i] + tok0, (unsigned)off, dst + i * L::TILE + 1024 * b);
        }
    if (tid < 16) lds_dma2(lrp + 2 * (size_t)stage * K, 2u * (unsigned)(tid < K ? tid : K - 1), in0 + L::LR + (stage & 1) * 64);
  }
  __device__ __forceinline__ const uint16_t* row(int stage, int ten) const {
    return reinterpret_cast<const uint16_t*>(smem + L::IN + (stage & 1) * L::IN1 + ten * L::TILE) + c * D;
  }
  // tile I of a staged tensor with tokens along k: lane l supplies four features of token 4g + c / 4
  __device__ __forceinline__ frag token_k(int stage, int ten, int I) const {
    const unsigned char* t = smem + L::IN + (stage & 1) * L::IN1 + ten * L::TILE;
    return read_tr(reinterpret_cast<const uint16_t*>(t) + (4 * g + (c >> 2)) * D + 8 * (c & 3) + 32 * (I >> 1) + 4 * (I & 1));
  }
  __device__ __forceinline__ float lr_of(int stage, int t) const {
    return t < K ? __uint_as_float(LRs[(stage & 1) * 16 + t] << 16) : 0.f;
  }
  // the slot of a mini-batch, as a scalar address: accesses are then scalar base + 32-bit lane offset (a divided or
  // otherwise vector-computed base costs a register pair and a 64-bit addition per access, and spills)
  __device__ __forceinline__ unsigned char* slot(int stage) const {
    const unsigned n = __builtin_amdgcn_readfirstlane((unsigned)stage % (unsigned)a.slots);
    return a.hand + (bh * (size_t)a.slots + n) * S::SLOT;
  }
  // the own features of token c of a mini-batch in an output tensor
  __device__ __forceinline__ uint16_t* out_row(void* t, int stage) const {
    unsigned char* base = static_cast<unsigned char*>(t) + (bh * (size_t)a.seq_stride + (size_t)stage * K) * (D * 2);
    return reinterpret_cast<uint16_t*>(base + (unsigned)(c * (D * 2) + own * 2));
  }
  // reducers: lane group g publishes sums g and g + 4 of reducer w; any wave collects
  __device__ __forceinline__ void publish(const float (&Q)[8]) {
    const float v0 = xg_sum4_scatter(Q[0], Q[1], Q[2], Q[3]);
    const float v1 = xg_sum4_scatter(Q[4], Q[5], Q[6], Q[7]);
    EX[((g * 2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = v0;
    EX[(((g + 4) * 2 + (w >> 2)) * 16 + c) * 4 + (w & 3)] = v1;
  }
  __device__ __forceinline__ float collect(int i) const {
    const f32x4 l = *reinterpret_cast<const f32x4*>(EX + ((i * 2 + 0) * 16 + c) * 4);
    float s = (l[0] + l[1]) + (l[2] + l[3]);
    if (NT > 4) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(EX + ((i * 2 + 1) * 16 + c) * 4);
      s += (u[0] + u[1]) + (u[2] + u[3]);
    }
    return s;
  }
  __device__ __forceinline__ f32x4 sum_tile(int buf, int I) const {
    f32x4 v[NW], z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (ROOM) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) v[ww] = PB[((buf * NW + ww) * NT + I) * 64 + lane];
      together(v);
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) z += v[ww];
    } else {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        z += PB[((buf * NW + ww) * NT + I) * 64 + lane];
        if ((ww & 3) == 3) pin(z);
      }
    }
    return z;
  }
  __device__ __forceinline__ f32x4 sum_block() const {
    f32x4 v[NW], z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (ROOM) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) v[ww] = PA[ww * 64 + lane];
      together(v);
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) z += v[ww];
    } else {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) z += PA[ww * 64 + lane];
      pin(z);
    }
    return z;
  }
  // (moved to a scalar register by hand: see isa_check.py, the scalar select on a vector comparison)
  __device__ __forceinline__ bool is_lost() const { return __builtin_amdgcn_readfirstlane(*lost) != 0; }
  // A look at the counter ahead of time: the poll that follows finds it in LDS and is spared the round trip it would begin
  // with, up to 5 k cycles on a full chip (d = 96 2167 -> 2122 us).  Through LDS because a register for it spills others.
  __device__ __forceinline__ void peek(const unsigned* fl, int which) {
    if (pair && w == 0 && lane == 0) lds_dma4_dev(fl, 4u * which, lds0() + L::CTL + 4);
  }
  // bounded wait of thread 0 for the partner's counter; the barrier behind it is the caller's
  __device__ __forceinline__ void poll(unsigned* fl, int which, int want) {
    if (!pair || want <= 0 || tid != 0 || is_lost()) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // as the copy left it (the wait above is a memory clobber); in a scalar register, as in is_lost: d = 32 803 -> 793 us
    const unsigned seen = (unsigned)__builtin_amdgcn_readfirstlane(lost[1]);
    bool got = seen != kMlpRpPoison && seen >= (unsigned)want;
    if (got) return;
    for (unsigned i = 0; i < a.spin_limit; ++i) {
      const unsigned v = __hip_atomic_load(fl + which, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (v == kMlpRpPoison) break;
      if (v >= (unsigned)want) {
        got = true;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    if (!got) *lost = 1;
  }
  __device__ __forceinline__ void raise(unsigned* fl, int which, int value) {
    if (pair && tid == 0)
      __hip_atomic_store(fl + which, is_lost() ? kMlpRpPoison : (unsigned)value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // sums over tokens and batch elements
  __device__ __forceinline__ void add_norm_grads(f32x4 dgam, f32x4 dbet) {
    if (!red) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float x = dgam[r], y = dbet[r];
      const float sx = row16_sum_dpp(x), sy = row16_sum_dpp(y);
      if (c == 0) {
        atomicAdd(a.d_gamma + h * D + own + r, sx);
        atomicAdd(a.d_beta + h * D + own + r, sy);
      }
    }
  }
};

template <int D>
__device__ __forceinline__ void producer(const MlpBwdRpArgs& a, unsigned char* smem, size_t bh, bool pair) {
  using B = Base<D, 4>;
  using S = MlpRp<D>;
  constexpr int NW = B::NW, NT = B::NT, F = B::F, HT = B::HT, NQ = B::NQ;
  constexpr float inv_d = B::inv_d;
  B x(a, smem, bh, pair);
  const int w = x.w, tid = x.tid, K = x.K;
  int &lane = x.lane, &c = x.c, &g = x.g;
  const bool red = x.red;
  unsigned* const fl = a.flags + bh * (size_t)kMlpRpFlagWords;
  unsigned my_xcc = 0;
  bool fast_release = !pair;  // the consumer is known to sit behind the same L2
  if (pair) {
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(my_xcc));
    my_xcc &= 15u;
    if (tid == 0) __hip_atomic_store(fl + 2, 0x100u | my_xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid == 0) x.lost[0] = pair && a.spin_limit == 0 ? 1 : 0, x.lost[1] = 0;
  const bool upd = x.te_last != 0.f;

  f32x4 W1c[NT][HT], W2c[HT][NT], b2T = {0.f, 0.f, 0.f, 0.f};
  f32x4* const st1 = reinterpret_cast<f32x4*>(a.state + bh * (size_t)(2 * D * F)) + (w * NT * HT) * 64 + lane;
  f32x4* const st2 = st1 + NW * NT * HT * 64;
#pragma unroll
  for (int I = 0; I < NT; ++I)
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      W1c[I][j] = st1[(I * HT + j) * 64];
      W2c[j][I] = st2[(j * NT + I) * 64];
    }
  for (int i = tid; i < F; i += 512) x.B1s[i] = a.b1[bh * F + i];
  if (red) b2T = *reinterpret_cast<const f32x4*>(a.b2 + bh * D + x.own);
  // sums that only the reducers touch, once per mini-batch, live in LDS: the registers are short
  auto dgam = [&]() -> f32x4& { return reinterpret_cast<f32x4*>(smem + B::L::DG)[(red ? w : 0) * 64 + lane]; };
  auto dbet = [&]() -> f32x4& { return reinterpret_cast<f32x4*>(smem + B::L::DB)[(red ? w : 0) * 64 + lane]; };
  if (red) dgam() = dbet() = f32x4{0.f, 0.f, 0.f, 0.f};

  const unsigned char* const fac = a.fac + bh * (size_t)a.n_stages * S::FAC;
  frag G1d[HT], gd = IO::zero();
  auto load_factors = [&](int st) {
    const unsigned char* f = fac + (size_t)st * S::FAC;
#pragma unroll
    for (int j = 0; j < HT; ++j) G1d[j] = at<const frag>(f + w * HT * 512, j * 512 + 8u * lane);
    if (red) gd = at<const frag>(f + (NW * HT + w) * 512, 8u * lane);
  };
  __syncthreads();
  x.fetch(a.last - 1);
  load_factors(a.last - 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (red) {
    x.GS[w * 64 + lane] = gd;
  }

  for (int st = a.last - 1; st >= a.first; --st) {
    const int par = st & 1;
    unsigned char* const sl = x.slot(st);
    unsigned char* const sw = sl + w * S::WAVE;
    unsigned char* const stl = sl + S::TILES + (red ? w : 0) * S::TILE;
    lds_barrier();  // ---- T: factors and XK tiles are in LDS
    RP_RELANE();

    // ================= A: walk W1, b1 back; Z1, X2; walk W2, b2 back; partial Z2
    f32x4 z1[HT], zq[HT];
    frag kd[NT];
#pragma unroll
    for (int I = 0; I < NT; ++I) kd[I] = x.token_k(st, 1, I);
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const frag ng = upd ? neg(G1d[j]) : IO::zero();
#pragma unroll
      for (int I = 0; I < NT; ++I) IO::mma(W1c[I][j], kd[I], ng);
      f32x4* const bp = reinterpret_cast<f32x4*>(x.B1s + 16 * (w * HT + j) + 4 * g);
      z1[j] = *bp;
      IO::mma(z1[j], ng, x.ones);
      if (c == 0) *bp = z1[j];
      asm volatile("s_nop 4" : "+v"(z1[j]));
      zq[j] = z1[j];
      RP_FENCE();
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      frag k0, k1, q0, q1;
      IO::load8(x.row(st, 1) + 32 * q + 8 * g, true, k0, k1);
      IO::load8(x.row(st, 0) + 32 * q + 8 * g, true, q0, q1);
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        const frag w0 = IO::to_frag(W1c[2 * q][j]), w1 = IO::to_frag(W1c[2 * q + 1][j]);
        IO::mma2(z1[j], w0, w1, k0, k1);
        IO::mma2(zq[j], w0, w1, q0, q1);
      }
      RP_FENCE();
    }
    frag x2f[HT];
    f32x4 dg[HT], ddg[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      f32x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float yy, d1, d2;
        gelu_all(z1[j][r], yy, d1, d2);
        y[r] = yy;
        dg[j][r] = d1;
        ddg[j][r] = d2;
      }
      x2f[j] = IO::to_frag(y);
      asm volatile("" : "+v"(x2f[j]), "+v"(dg[j]), "+v"(ddg[j]));
      const frag nx = upd ? neg(flip(x2f[j], x.ident)) : IO::zero();
#pragma unroll
      for (int I = 0; I < NT; ++I) IO::mma(W2c[j][I], nx, x.GS[I * 64 + lane]);
      RP_FENCE();
    }
    if constexpr (D < 96) {  // (d = 96: more instructions of the loop above lie behind the first products than the states)
#pragma unroll
      for (int I = 0; I < NT; ++I) asm volatile("" : "+v"(W2c[HT - 1][I]));
      settle();
    }
    if (red) IO::mma(b2T, upd ? neg(x.GS[w * 64 + lane]) : IO::zero(), x.ones);
#pragma unroll
    for (int I = 0; I < NT; ++I) {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, IO::to_frag(W2c[j][I]), IO::to_frag(W2c[j + 1][I]), x2f[j], x2f[j + 1]);
      if (HT & 1) mmz(p, IO::to_frag(W2c[HT - 1][I]), x2f[HT - 1]);
      x.PB[((par * NW + w) * NT + I) * 64 + lane] = p;
      RP_FENCE();
    }
    // the stores of the mini-batch before have had all of phase A to be acknowledged
    if (fast_release) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      if (a.agent_release == 0 && st + 2 < a.last) {
        const unsigned other = __hip_atomic_load(fl + 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        fast_release = __builtin_amdgcn_readfirstlane(other) == (0x100u | my_xcc);
      }
    }
    lds_barrier();  // ---- B1
    x.raise(fl, 0, a.n_stages - 1 - st);
    // the slot was last read by the consumer `slots` mini-batches ago; the first store to it comes behind B2.
    // (Behind the raise: the consumer may be waiting for it before it can report that the slot is free.)
    x.poll(fl, 1, a.n_stages - st - a.slots);
    RP_RELANE();
    x.fetch(st - 1);

    // ================= B, C: reducers: LayerNorm of Z2, G2
    f32x4 z = {0.f, 0.f, 0.f, 0.f}, bq = z, dlt = z;
    if (red) {
      z = x.sum_tile(par, w) + b2T;
      const frag ko = load4<BF16>(x.row(st, 1) + x.own), vo = load4<BF16>(x.row(st, 2) + x.own);
      const f32x4 gam = *reinterpret_cast<const f32x4*>(x.GAM + x.own);
      dlt = *reinterpret_cast<const f32x4*>(x.BET + x.own) - (IO::to_f32(vo) - IO::to_f32(ko));
      bq = gam * dlt;
      const f32x4 az = gam * gam * z;
      float Q[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        Q[0] += z[r];
        Q[1] += z[r] * z[r];
        Q[2] += az[r];
        Q[3] += az[r] * z[r];
        Q[4] += bq[r];
        Q[5] += bq[r] * z[r];
      }
      x.publish(Q);
    }
    lds_barrier();  // ---- B2
    RP_RELANE();
    if (red) {
      const float q0 = x.collect(0), q1 = x.collect(1), q2 = x.collect(2), q3 = x.collect(3), q4 = x.collect(4), q5 = x.collect(5);
      const float mu = q0 * inv_d;
      const float rstd = __builtin_amdgcn_rsqf(fmaxf(q1 * inv_d - mu * mu, 0.f) + a.eps);
      const float sa1 = rstd * (q2 - mu * x.sum_a), sa2 = rstd * rstd * (q3 - 2.f * mu * q2 + mu * mu * x.sum_a);
      const float s1 = sa1 + q4, s2 = sa2 + rstd * (q5 - mu * q4);  // sums of g_x and of g_x x_hat
      const f32x4 gam = *reinterpret_cast<const f32x4*>(x.GAM + x.own);
      const f32x4 xh = (z - mu) * rstd, gO = gam * xh + dlt;
      const f32x4 G = (gam * gO - s1 * inv_d - xh * (s2 * inv_d)) * rstd;
      const frag gt = IO::to_frag(G), gn = flip(gt, x.ident);
      x.GT[w * 64 + lane] = gt;
      x.GS[w * 64 + lane] = gn;
      at<f32x4>(stl, S::XH + 16u * lane) = xh;
      at<f32x4>(stl, S::GO + 16u * lane) = gO;
      at<f32x4>(stl, S::G2 + 16u * lane) = G;
      at<u32x4>(stl, S::GG + 16u * lane) = rp::pair(gt, gn);
      if (w == 0 && g == 0) {
        const unsigned so = S::SCAL + 4u * c;
        at<float>(sl, so) = rstd, at<float>(sl, so + 64) = s1, at<float>(sl, so + 128) = s2, at<float>(sl, so + 192) = sa1,
        at<float>(sl, so + 256) = sa2;
      }
    }
    lds_barrier();  // ---- B3
    RP_RELANE();

    // ================= D: U = G2 W2^T, G1; Zbar1, Xbar2; partial A2, Zbar2
    // (Zbar1 and Zbar2 take G1, G2 and the causal blocks M1, M2 as the very operands that the gradient's products take: what
    // an operand loses then shifts the point at which the gradient is taken, instead of adding to its error)
    float lrs[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) lrs[r] = x.lr_of(st, 4 * g + r);
    frag g1b[HT], g1n[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W2c[j][I]);
    {
      f32x4 acc[HT];
#pragma unroll
      for (int j = 0; j < HT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const frag g0 = x.GT[(2 * q) * 64 + lane], g1 = x.GT[(2 * q + 1) * 64 + lane];
        f32x4 f0[HT], f1[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          f0[j] = f1[j] = f32x4{0.f, 0.f, 0.f, 0.f};
          IO::mma(f0[j], IO::to_frag(W2c[j][2 * q]), x.ident);
          IO::mma(f1[j], IO::to_frag(W2c[j][2 * q + 1]), x.ident);
        }
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          const frag t0 = IO::to_frag(f0[j]), t1 = IO::to_frag(f1[j]);
          at<u32x4>(sw, S::W2T + (j * NQ + q) * 1024 + 16u * lane) = rp::pair(t0, t1);
          IO::mma2(acc[j], t0, t1, g0, g1);
        }
        RP_FENCE();
      }
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        const f32x4 g1 = acc[j] * dg[j];
        g1b[j] = IO::to_frag(g1);
        at<f32x4>(sw, S::DG + j * 1024 + 16u * lane) = dg[j];
        at<f32x4>(sw, S::UG + j * 1024 + 16u * lane) = acc[j] * ddg[j];
        at<f32x4>(sw, S::G1 + j * 1024 + 16u * lane) = g1;
      }
#pragma unroll
      for (int j = 0; j < HT; ++j) g1n[j] = flip(g1b[j], x.ident);
    }
    RP_FENCE();
    f32x4 At = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      frag k0, k1, q0, q1;
      IO::load8(x.row(st, 1) + 32 * q + 8 * g, true, k0, k1);
      IO::load8(x.row(st, 0) + 32 * q + 8 * g, true, q0, q1);
      IO::mma2(At, k0, k1, q0, q1);
    }
    {
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? x.te_c * lrs[r] * (1.f + At[r]) : 0.f;
      const frag Mf = neg(IO::to_frag(m));
#pragma unroll
      for (int j = 0; j < HT; ++j) mmz(zq[j], g1n[j], Mf);
    }
    frag xbf[HT];
    f32x4 dgz[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      f32x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float yy, d1;
        gelu_pair(zq[j][r], yy, d1);
        y[r] = yy;
        dgz[j][r] = d1;
      }
      xbf[j] = IO::to_frag(y);
      asm volatile("" : "+v"(xbf[j]), "+v"(dgz[j]));
      at<u32x4>(sw, S::XT + j * 1024 + 16u * lane) = rp::pair(x2f[j], xbf[j]);
      RP_FENCE();
    }
    {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, x2f[j], x2f[j + 1], xbf[j], xbf[j + 1]);
      if (HT & 1) mmz(p, x2f[HT - 1], xbf[HT - 1]);
      x.PA[w * 64 + lane] = p;
    }
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W2c[j][I]);
#pragma unroll
    for (int I = 0; I < NT; ++I) {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, IO::to_frag(W2c[j][I]), IO::to_frag(W2c[j + 1][I]), xbf[j], xbf[j + 1]);
      if (HT & 1) mmz(p, IO::to_frag(W2c[HT - 1][I]), xbf[HT - 1]);
      x.PB[(((par ^ 1) * NW + w) * NT + I) * 64 + lane] = p;
      RP_FENCE();
    }
    lds_barrier();  // ---- B4
    RP_RELANE();

    // ================= E: reducers: output LayerNorm backward, dZbar2 (and the wave that forms d lr keeps A2)
    f32x4 at2 = {0.f, 0.f, 0.f, 0.f}, dO = at2, zb = at2;
    if (red || w == NW - 1) at2 = x.sum_block();
#pragma unroll
    for (int r = 0; r < 4; ++r) lrs[r] = x.lr_of(st, 4 * g + r);
    frag M2f = IO::zero();
    if (red) {
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? x.te_c * lrs[r] * (1.f + at2[r]) : 0.f;
      M2f = IO::to_frag(m);
      zb = x.sum_tile(par ^ 1, w) + b2T;
      IO::mma(zb, x.GS[w * 64 + lane], neg(M2f));
      dO = IO::to_f32(load4<BF16>(x.row(st, 3) + x.own));
      const f32x4 gam = *reinterpret_cast<const f32x4*>(x.GAM + x.own);
      float Q[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float gx = gam[r] * dO[r];
        Q[0] += zb[r];
        Q[1] += zb[r] * zb[r];
        Q[2] += gx;
        Q[3] += gx * zb[r];
      }
      x.publish(Q);
    }
    lds_barrier();  // ---- B5
    RP_RELANE();
    if (red) {
      const float q0 = x.collect(0), q1 = x.collect(1), q2 = x.collect(2), q3 = x.collect(3);
      const float mu = q0 * inv_d;
      const float rstd = __builtin_amdgcn_rsqf(fmaxf(q1 * inv_d - mu * mu, 0.f) + a.eps);
      const float s1 = q2 * inv_d, s2 = rstd * (q3 - mu * q2) * inv_d;
      const f32x4 gam = *reinterpret_cast<const f32x4*>(x.GAM + x.own);
      const f32x4 xh = (zb - mu) * rstd;
      const f32x4 dz = (gam * dO - s1 - xh * s2) * rstd, zs = over_tokens(dz);
      if (c == 0) at<f32x4>(sl, S::ZB2 + 4u * x.own) = zs;
      const frag zt = IO::to_frag(dz), zd = flip(zt, x.ident);
      dgam() += dO * xh;
      dbet() += dO;
      x.ZT[w * 64 + lane] = zt;
      at<frag>(stl, S::ZD + 8u * lane) = zd;
      f32x4 mz = {0.f, 0.f, 0.f, 0.f};  // M2^T dZbar2
      IO::mma(mz, zd, flip(M2f, x.ident));
      at<f32x4>(stl, S::MZ + 16u * lane) = mz;
    }
    // the next mini-batch's rows have landed: every wave has issued at least the stores of phase D behind their copies
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(HT * NQ + 4 * HT) : "memory");
    lds_barrier();  // ---- B6
    RP_RELANE();

    // ================= F: dXbar2, dZbar1; partial P1 and dQ
    if (st > a.first) load_factors(st - 1);
    x.peek(fl, 1);
    f32x4 Pm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      IO::mma2(Pm, x.GT[(2 * q) * 64 + lane], x.GT[(2 * q + 1) * 64 + lane], x.ZT[(2 * q) * 64 + lane], x.ZT[(2 * q + 1) * 64 + lane]);
    frag dA2f;
    {
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? -Pm[r] * (x.te_c * lrs[r]) : 0.f;
      dA2f = IO::to_frag(m);
    }
    frag dzb[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W2c[j][I]);
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        IO::mma2(acc, flip(IO::to_frag(W2c[j][2 * q]), x.ident), flip(IO::to_frag(W2c[j][2 * q + 1]), x.ident),
                 x.ZT[(2 * q) * 64 + lane], x.ZT[(2 * q + 1) * 64 + lane]);
      mmz(acc, flip(x2f[j], x.ident), dA2f);
      const f32x4 dz = acc * dgz[j], zs = over_tokens(dz);
      if (c == 0) at<f32x4>(sl, S::ZB1 + (w * HT + j) * 64 + 16u * g) = zs;
      dzb[j] = IO::to_frag(dz);
      at<frag>(sw, S::DT + j * 512 + 8u * lane) = dzb[j];
      RP_FENCE();
    }
    {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, g1b[j], g1b[j + 1], dzb[j], dzb[j + 1]);
      if (HT & 1) mmz(p, g1b[HT - 1], dzb[HT - 1]);
      x.PA[w * 64 + lane] = p;
    }
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(W1c[I][j]);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      frag t[2 * HT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < HT; ++j) t[u * HT + j] = flip(IO::to_frag(W1c[2 * q + u][j]), x.ident);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, t[u * HT + j], t[u * HT + j + 1], dzb[j], dzb[j + 1]);
        if (HT & 1) mmz(p, t[u * HT + HT - 1], dzb[HT - 1]);
        x.PB[((par * NW + w) * NT + 2 * q + u) * 64 + lane] = p;
      }
#pragma unroll
      for (int n = 0; n < HT; ++n)
        at<u32x4>(sw, S::W1T + (q * HT + n) * 1024 + 16u * lane) = rp::pair(t[2 * n], t[2 * n + 1]);
      RP_FENCE();
    }
    lds_barrier();  // ---- B7
    RP_RELANE();

    // ================= G: reducers: d_xq; last wave: the causal blocks' gradients
    if (red || w == NW - 1) {
      const f32x4 p1 = x.sum_block();
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? -p1[r] * (x.te_c * lrs[r]) : 0.f;
      const frag dA1f = IO::to_frag(m);
      if (red) {
        f32x4 dq = x.sum_tile(par, w) + dO;
        IO::mma(dq, x.token_k(st, 1, w), dA1f);
        if (c < K)
          store4<BF16>(x.out_row(a.d_xq, st), dq);
        x.GS[w * 64 + lane] = gd;
      } else {
        float dte = 0.f;
        f32x4 m1, dl;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool ok = 4 * g + r <= c;
          const float de = ok ? -(Pm[r] * (1.f + at2[r]) + p1[r] * (1.f + At[r])) : 0.f;
          dte += de * lrs[r];
          const float v = de * x.te_c;
          dl[r] = row16_sum_dpp(v);
          m1[r] = ok ? x.te_c * lrs[r] * (1.f + At[r]) : 0.f;
        }
        dte = xg_sum(dte);
        if (g == 0 && c < K) atomicAdd(a.d_token_eta + (size_t)st * K + c, dte);
        if (c == 0) at<f32x4>(sl, S::SCAL + 320 + 16u * g) = dl;
        at<frag>(sl, S::M1T + 8u * lane) = flip(IO::to_frag(m1), x.ident);
        at<frag>(sl, S::A2T + 8u * lane) = flip(dA2f, x.ident);
        at<frag>(sl, S::A1T + 8u * lane) = flip(dA1f, x.ident);
      }
    }
  }
  if (pair) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!fast_release) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    lds_barrier();
    x.raise(fl, 0, a.n_stages - a.first);
    if (tid == 0 && x.is_lost()) atomicAdd(a.lost_count, 1u);
  } else {
    // the state entering `first`, for the next launch
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        st1[(I * HT + j) * 64] = W1c[I][j];
        st2[(j * NT + I) * 64] = W2c[j][I];
      }
    lds_barrier();
    for (int i = tid; i < F; i += 512) a.b1[bh * F + i] = x.B1s[i];
    if (red && c == 0) *reinterpret_cast<f32x4*>(a.b2 + bh * D + x.own) = b2T;
  }
  x.add_norm_grads(dgam(), dbet());
}

template <int D>
__device__ __forceinline__ void consumer(const MlpBwdRpArgs& a, unsigned char* smem, size_t bh, bool pair) {
  using B = Base<D, 2>;
  using S = MlpRp<D>;
  constexpr int NW = B::NW, NT = B::NT, F = B::F, HT = B::HT, NQ = B::NQ;
  constexpr float inv_d = B::inv_d;
  B x(a, smem, bh, pair);
  const int w = x.w, tid = x.tid, K = x.K;
  int &lane = x.lane, &c = x.c, &g = x.g;
  const bool red = x.red;
  unsigned* const fl = a.flags + bh * (size_t)kMlpRpFlagWords;
  unsigned my_xcc = 0;
  bool same_l2 = false;  // the producer is known to sit behind the same L2 (it publishes its XCD before its first count)
  if (pair) {
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(my_xcc));
    my_xcc &= 15u;
    if (tid == 0) __hip_atomic_store(fl + 3, 0x100u | my_xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid == 0) x.lost[0] = pair && a.spin_limit == 0 ? 1 : 0, x.lost[1] = 0;
  // sums that only the reducers touch, once per mini-batch, live in LDS: the registers are short
  auto dgam = [&]() -> f32x4& { return x.PA[(red ? w : 0) * 64 + lane]; };
  auto dbet = [&]() -> f32x4& { return reinterpret_cast<f32x4*>(smem + B::L::DB)[(red ? w : 0) * 64 + lane]; };
  auto db2 = [&]() -> f32x4& { return *reinterpret_cast<f32x4*>(smem + B::L::B2 + 4 * x.own); };
  // second use of an LDS region: dZ2 beside its other orientation
  frag* const ZDs = x.GT;
  // G2 in both orientations and dZbar2: where the staging area has room for two tensors more than are staged here
  frag* const GTs = reinterpret_cast<frag*>(smem + B::L::IN + 2 * B::L::TILE);
  frag* const GNs = GTs + NT * 64;
  frag* const GLs = reinterpret_cast<frag*>(smem + B::L::GL);
  frag* const ZNs = reinterpret_cast<frag*>(smem + B::L::IN + B::L::IN1 + 2 * B::L::TILE);
  float* const DB1 = x.B1s;

  f32x4 dW1c[NT][HT], dW2c[HT][NT];
  float* const g1 = a.d_W1 + bh * (size_t)D * F;
  float* const g2 = a.d_W2 + bh * (size_t)D * F;
  const bool top = a.last == a.n_stages;
  {
    const f32x4* s1 = reinterpret_cast<const f32x4*>(g1) + (w * NT * HT) * 64 + lane;
    const f32x4* s2 = reinterpret_cast<const f32x4*>(g2) + (w * NT * HT) * 64 + lane;
    const bool up = a.up_W1 != nullptr;
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const int hb = 16 * (w * HT + j);
#pragma unroll
      for (int I = 0; I < NT; ++I) {
        if (!top) {
          dW1c[I][j] = s1[(I * HT + j) * 64];
          dW2c[j][I] = s2[(j * NT + I) * 64];
        } else if (up) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            dW1c[I][j][r] = a.up_W1[bh * (size_t)D * F + (size_t)feat(I, 4 * g + r) * F + hb + c];
            dW2c[j][I][r] = a.up_W2[bh * (size_t)D * F + (size_t)(hb + 4 * g + r) * D + feat(I, c)];
          }
        } else {
          dW1c[I][j] = dW2c[j][I] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
    const float* b1 = top ? (up ? a.up_b1 : nullptr) : a.d_b1;
    const float* b2 = top ? (up ? a.up_b2 : nullptr) : a.d_b2;
    for (int i = tid; i < F; i += 512) DB1[i] = b1 != nullptr ? b1[bh * F + i] : 0.f;
    if (red) {
      f32x4 b = {0.f, 0.f, 0.f, 0.f};
      dgam() = b;
      dbet() = b;
      if (b2 != nullptr)
#pragma unroll
        for (int r = 0; r < 4; ++r) b[r] = b2[bh * D + x.own + r];
      if (c == 0) db2() = b;
    }
  }
  // pending d_xk of the mini-batch before (its partial tiles are in LDS)
  f32x4 dk_p = {0.f, 0.f, 0.f, 0.f};  // its terms of the own features
  float dl_p = 0.f;
  __syncthreads();
  x.fetch(a.last - 1);

  auto finish = [&](int st) {  // d_xk and d_lr of mini-batch st
    if (red) {
      const f32x4 dk = x.sum_tile(1, w) + dk_p;
      if (c < K)
        store4<BF16>(x.out_row(a.d_xk, st), dk);
    }
    if (w == NW - 1) {
      float q = 0.f;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) q += x.QS[ww * 16 + c];
      if (g == 0 && c < K) {
        const size_t tok = bh * (size_t)a.seq_stride + (size_t)st * K;
        IO::store1(static_cast<uint16_t*>(a.d_lr) + tok + c, dl_p - x.te_last * q);
        // (the rows of the staged lr belong to another mini-batch by now)
      }
      const float l = c < K ? IO::load1(static_cast<const uint16_t*>(a.lr) + bh * (size_t)a.seq_stride + (size_t)st * K + c) : 0.f;
      const float v = -q * l;
      const float s = row16_sum_dpp(v);
      if (lane == 0) atomicAdd(a.d_token_eta + (size_t)st * K + K - 1, s);
    }
  };

  for (int st = a.last - 1; st >= a.first; --st) {
    const Slot sl(x.slot(st), S::SLOT);
    const unsigned sw = w * S::WAVE, stl = S::TILES + (red ? w : 0) * S::TILE;
    x.poll(fl, 0, a.n_stages - st);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();  // ---- T: the slot is filled, this mini-batch's rows have landed, the slot before is no longer read
    // a producer behind another L2 writes its L2 back: drop the lines that this one's L2 and vector cache hold.  Behind one
    // L2 nothing need go: the hand-over is read with device-scope loads (see Slot), which do not look in the vector cache
    if (pair && !same_l2) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (pair && !same_l2 && a.agent_release == 0)
      same_l2 = __builtin_amdgcn_readfirstlane(__hip_atomic_load(fl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == (0x100u | my_xcc);
    x.raise(fl, 1, a.n_stages - 1 - st);
    RP_RELANE();
    x.fetch(st - 1);

    // ================= A: d_xk, d_lr of the mini-batch before; S1 = XK dW1, dG1, dU; partial -last X2 dW2 + dU W2
    frag x2f[HT];
    frag dt[HT];  // dZbar1: fetched again for the last part of phase D
    f32x4 dg[HT], ug[HT], gg1[HT];
    // the images of W2 and W1 are fetched a feature-tile pair ahead of their use
    auto load_w2 = [&](u32x4 (&t)[HT], int q) {
#pragma unroll
      for (int j = 0; j < HT; ++j) t[j] = sl.get<u32x4>(16u * lane, sw + S::W2T + (j * NQ + q) * 1024);
    };
    auto load_w1 = [&](u32x4 (&t)[HT], int q) {
#pragma unroll
      for (int n = 0; n < HT; ++n) t[n] = sl.get<u32x4>(16u * lane, sw + S::W1T + (q * HT + n) * 1024);
    };
    u32x4 wt[2][HT];
    // column sums of dZbar1 (own hidden slice) and, reducers, of dZbar2 (own features): one value a lane
    const float zb1 = sl.get<float>(4u * (lane < 16 * HT ? lane : 0), S::ZB1 + w * HT * 64);
    const int fb2 = own_offset<1>(red ? w : 0, 0, (lane >> 2) & 3) + (lane & 3);
    const float zb2 = sl.get<float>(4u * fb2, S::ZB2);
    RP_FENCE();
    if (st + 1 < a.last) finish(st + 1);
    RP_FENCE();
    // gelu'(Z1) and U gelu''(Z1) wait in LDS, in the wave's own part of the partial tiles it is about to form
    {
      const unsigned char* const hs = x.slot(st) + sw;
      const unsigned park = x.lds0() + B::L::PB + w * NT * 1024;
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        lds_dma16_dev(hs + S::DG + j * 1024, 16u * lane, park + j * 1024);
        lds_dma16_dev(hs + S::UG + j * 1024, 16u * lane, park + (HT + j) * 1024);
      }
    }
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      x2f[j] = sl.get<frag>(16u * lane, sw + S::XT + j * 1024);
      dt[j] = sl.get<frag>(8u * lane, sw + S::DT + j * 512);
      gg1[j] = sl.get<f32x4>(16u * lane, sw + S::G1 + j * 1024);
    }
    const frag m1t = sl.get<frag>(8u * lane, S::M1T);
    load_w2(wt[0], 0);
    RP_FENCE();
    const float last_c = x.te_last * x.lr_of(st, c);
    f32x4 s1[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) s1[j] = *reinterpret_cast<const f32x4*>(DB1 + 16 * (w * HT + j) + 4 * g);
    // (S1 takes db1 as it was; a wave's slice is its own)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      frag k0, k1;
      IO::load8(x.row(st, 1) + 32 * q + 8 * g, true, k0, k1);
#pragma unroll
      for (int j = 0; j < HT; ++j) IO::mma2(s1[j], IO::to_frag(dW1c[2 * q][j]), IO::to_frag(dW1c[2 * q + 1][j]), k0, k1);
      RP_FENCE();
    }
    if (lane < 16 * HT) DB1[16 * w * HT + lane] += zb1;
    float qs = 0.f;
    frag duf[HT], g1b[HT];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what was copied to LDS has landed
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      dg[j] = x.PB[(w * NT + j) * 64 + lane];
      ug[j] = x.PB[(w * NT + HT + j) * 64 + lane];
    }
#pragma unroll
    for (int j = 0; j < HT; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) qs += gg1[j][r] * s1[j][r];
      g1b[j] = IO::to_frag(gg1[j]);
      f32x4 m = {0.f, 0.f, 0.f, 0.f};
      IO::mma(m, flip(dt[j], x.ident), m1t);
      const f32x4 dG1 = -(last_c * s1[j] + m);
      duf[j] = IO::to_frag(dG1 * dg[j]);
      ug[j] = dG1 * ug[j];  // first term of dZ1
    }
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(dW2c[j][I]);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (q + 1 < NQ) load_w2(wt[(q + 1) & 1], q + 1);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int I = 2 * q + u;
        f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j + 1 < HT; j += 2)
          IO::mma2(p, IO::to_frag(dW2c[j][I]), IO::to_frag(dW2c[j + 1][I]), x2f[j], x2f[j + 1]);
        if (HT & 1) mmz(p, IO::to_frag(dW2c[HT - 1][I]), x2f[HT - 1]);
        p *= -last_c;
        frag wn[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) wn[j] = flip(u == 0 ? lo(wt[q & 1][j]) : hi(wt[q & 1][j]), x.ident);
#pragma unroll
        for (int j = 0; j + 1 < HT; j += 2) IO::mma2(p, wn[j], wn[j + 1], duf[j], duf[j + 1]);
        if (HT & 1) mmz(p, wn[HT - 1], duf[HT - 1]);
        x.PB[(w * NT + I) * 64 + lane] = p;
      }
      RP_FENCE();
    }
    f32x4 xh = {0.f, 0.f, 0.f, 0.f}, gO = xh, uu = xh, G = xh, mz = xh;
    u32x4 gg = {0u, 0u, 0u, 0u};
    frag zdn = IO::zero();
    const unsigned so = 4u * c;
    const float rstd = sl.get<float>(so, S::SCAL), sg = sl.get<float>(so, S::SCAL + 64), sgx = sl.get<float>(so, S::SCAL + 128),
                sa1 = sl.get<float>(so, S::SCAL + 192), sa2 = sl.get<float>(so, S::SCAL + 256), dlp = sl.get<float>(so, S::SCAL + 320);
    if (red) {
      xh = sl.get<f32x4>(16u * lane, stl + S::XH);
      gO = sl.get<f32x4>(16u * lane, stl + S::GO);
      G = sl.get<f32x4>(16u * lane, stl + S::G2);
      mz = sl.get<f32x4>(16u * lane, stl + S::MZ);
      gg = sl.get<u32x4>(16u * lane, stl + S::GG);
      zdn = sl.get<frag>(8u * lane, stl + S::ZD);
    }
    lds_barrier();  // ---- C1
    RP_RELANE();

    // ================= B: reducers: dG2, row sums of the second-order LayerNorm
    if (red) {
      GTs[w * 64 + lane] = lo(gg);
      GNs[w * 64 + lane] = hi(gg);
      GLs[w * 64 + lane] = IO::to_frag(G - IO::to_f32(lo(gg)));
      ZNs[w * 64 + lane] = zdn;
      const f32x4 db2T = db2();
      if (lane < 16) reinterpret_cast<float*>(smem + B::L::B2)[fb2] += zb2;  // behind the read: dG2 takes db2 as it was
      const f32x4 dG = x.sum_tile(0, w) - last_c * db2T - mz;
      const f32x4 gam = *reinterpret_cast<const f32x4*>(x.GAM + x.own);
      uu = dG * -rstd;
      const f32x4 gu = gam * gam * uu;
      float Q[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        Q[0] += uu[r];
        Q[1] += uu[r] * xh[r];
        Q[2] += gu[r];
        Q[3] += gu[r] * xh[r];
        Q[4] += dG[r] * G[r];
        qs += G[r] * db2T[r];
      }
      x.publish(Q);
    }
    // the first term of dZ1, dU and G1 as an operand wait for phase D in the wave's part of the partial dK tiles, which are
    // summed by now
    auto wait_frag = [&](int n) -> frag& { return reinterpret_cast<frag*>(x.PB + ((NW + w) * NT + HT) * 64)[n * 64 + lane]; };
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      x.PB[((NW + w) * NT + j) * 64 + lane] = ug[j];
      wait_frag(j) = duf[j];
      wait_frag(HT + j) = g1b[j];
    }
    lds_barrier();  // ---- C2
    RP_RELANE();
    u32x4 xd[HT];  // (X2, Xbar2), fetched again rather than held since phase A
    constexpr int AH = B::ROOM ? 2 : 1;  // feature-tile pairs of W2^T on their way
#pragma unroll
    for (int q = 0; q < AH && q < NQ; ++q) load_w2(wt[q], q);
#pragma unroll
    for (int j = 0; j < HT; ++j) xd[j] = sl.get<u32x4>(16u * lane, sw + S::XT + j * 1024);
    const frag a2t = sl.get<frag>(8u * lane, S::A2T), a1t = sl.get<frag>(8u * lane, S::A1T);

    // ================= C: reducers: dZ2, dT
    if (red) {
      const float q0 = x.collect(0), q1 = x.collect(1), q2 = x.collect(2), q3 = x.collect(3), q4 = x.collect(4);
      const float m1 = q0 * inv_d, m2 = q1 * inv_d, m3 = sgx * inv_d;  // means of u, u x_hat, g_x x_hat
      const f32x4 gam = *reinterpret_cast<const f32x4*>(x.GAM + x.own);
      const f32x4 dgx = m1 + xh * m2 - uu, dy = gam * dgx;
      dgam() += gO * dgx + dy * xh;
      dbet() += dy;
      const f32x4 dxh = gam * dy + (gam * gO) * m2 + uu * m3;
      const float t1 = (-q2 + m1 * x.sum_a + m2 * sa1 + m2 * sg + m3 * q0) * inv_d;
      const float t2 = -q3 + m1 * sa1 + m2 * sa2 + m2 * sgx + m3 * q1 + q4;
      const float dsig = -t2 * rstd;
      const f32x4 dZ2 = (dxh - t1) * rstd + xh * (dsig * inv_d);
      const f32x4 dT = -dy;
      if (c < K)
        store4<BF16>(x.out_row(a.d_xv, st), dT);
      const frag zt = IO::to_frag(dZ2), zd = flip(zt, x.ident);
      x.ZT[w * 64 + lane] = zt;
      ZDs[w * 64 + lane] = zd;
      const f32x4 b = db2() + over_tokens(dZ2);
      if (c == 0) db2() = b;
      dk_p = dy;  // -d target
      IO::mma(dk_p, x.token_k(st, 0, w), a1t);
    }
    dl_p = dlp;
    lds_barrier();  // ---- C3
    RP_RELANE();

    x.peek(fl, 0);
    // ================= D: T2, dX2, dZ1; partial dK; updates
    // (X2 : T2 is the sum G2 : X2 dW2 behind d lr; it takes G2 in two bf16 parts, 16 bits of it, so that only the operands
    // X2 and dW2 are rounded there)
    frag dz1[HT], xbd[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(dW2c[j][I]);
    {
      f32x4 t[HT], acc[HT], dd[HT];  // T2; dX2; gelu'(Z1), fetched again
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        xbd[j] = flip(hi(xd[j]), x.ident);
        t[j] = acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        mmz(acc[j], xbd[j], a2t);
      }
      RP_FENCE();
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const frag z0 = x.ZT[(2 * q) * 64 + lane], z1 = x.ZT[(2 * q + 1) * 64 + lane];
#pragma unroll
        for (int j = 0; j < HT; ++j) IO::mma2(acc[j], lo(wt[q % AH][j]), hi(wt[q % AH][j]), z0, z1);
        RP_FENCE();
        if (q + AH < NQ) load_w2(wt[q % AH], q + AH);
        if (q + 1 == NQ) {
#pragma unroll
          for (int j = 0; j < HT; ++j) dd[j] = sl.get<f32x4>(16u * lane, sw + S::DG + j * 1024);
        }
        const frag g0 = GTs[(2 * q) * 64 + lane], g1 = GTs[(2 * q + 1) * 64 + lane], l0 = GLs[(2 * q) * 64 + lane],
                   l1 = GLs[(2 * q + 1) * 64 + lane];
        frag w0[HT], w1[HT];
        {
          f32x4 f[HT];
#pragma unroll
          for (int j = 0; j < HT; ++j) {
            f[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            IO::mma(f[j], IO::to_frag(dW2c[j][2 * q]), x.ident);
          }
#pragma unroll
          for (int j = 0; j < HT; ++j) w0[j] = IO::to_frag(f[j]);
#pragma unroll
          for (int j = 0; j < HT; ++j) {
            f[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            IO::mma(f[j], IO::to_frag(dW2c[j][2 * q + 1]), x.ident);
          }
#pragma unroll
          for (int j = 0; j < HT; ++j) w1[j] = IO::to_frag(f[j]);
        }
#pragma unroll
        for (int j = 0; j < HT; ++j) IO::mma2(t[j], w0[j], w1[j], g0, g1);
#pragma unroll
        for (int j = 0; j < HT; ++j) IO::mma2(t[j], w0[j], w1[j], l0, l1);
        RP_FENCE();
      }
      load_w1(wt[0], 0);
#pragma unroll
      for (int n = 0; n < HT; ++n) dt[n] = sl.get<frag>(8u * lane, sw + S::DT + n * 512);
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        const f32x4 xf = IO::to_f32(lo(xd[j]));
#pragma unroll
        for (int r = 0; r < 4; ++r) qs += xf[r] * t[j][r];
        const f32x4 dx2 = acc[j] - last_c * t[j];
        const f32x4 dz = x.PB[((NW + w) * NT + j) * 64 + lane] + dx2 * dd[j];
        {
          f32x4* const bp = reinterpret_cast<f32x4*>(DB1 + 16 * (w * HT + j) + 4 * g);
          const f32x4 b = *bp + over_tokens(dz);  // (bias gradients are sums of f32 terms)
          if (c == 0) *bp = b;
        }
        dz1[j] = IO::to_frag(dz);
      }
    }
    RP_FENCE();
    // dW2 += [X2 | dU]^T [dZ2 ; G2] + Xbar2^T dZbar2
    {
      frag x2d[HT], dud[HT];
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        x2d[j] = flip(lo(xd[j]), x.ident);
        dud[j] = flip(wait_frag(j), x.ident);
      }
      frag zd = ZDs[lane], gn = GNs[lane], zn = ZNs[lane];
#pragma unroll
      for (int I = 0; I < NT; ++I) {
        const int In = (I + 1 < NT ? I + 1 : I) * 64;
        const frag zd_ = ZDs[In + lane], gn_ = GNs[In + lane], zn_ = ZNs[In + lane];
#pragma unroll
        for (int j = 0; j < HT; ++j) IO::mma2(dW2c[j][I], x2d[j], dud[j], zd, gn);
#pragma unroll
        for (int j = 0; j < HT; ++j) mmz(dW2c[j][I], xbd[j], zn);
        zd = zd_;
        gn = gn_;
        zn = zn_;
        RP_FENCE();
      }
    }
    {
      const float s = xg_sum(qs);
      if (g == 0) x.QS[w * 16 + c] = s;
    }
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) forget(dW1c[I][j]);
#pragma unroll
    for (int j = 0; j < HT; ++j) g1b[j] = wait_frag(HT + j);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (q + 1 < NQ) load_w1(wt[(q + 1) & 1], q + 1);
f32x4 f[2][HT], p[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        p[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          f[u][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          IO::mma(f[u][j], IO::to_frag(dW1c[2 * q + u][j]), x.ident);
        }
      }
      frag tn[2][HT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < HT; ++j) tn[u][j] = IO::to_frag(f[u][j]);
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2)
#pragma unroll
        for (int u = 0; u < 2; ++u) IO::mma2(p[u], tn[u][j], tn[u][j + 1], g1b[j], g1b[j + 1]);
      if (HT & 1)
#pragma unroll
        for (int u = 0; u < 2; ++u) mmz(p[u], tn[u][HT - 1], g1b[HT - 1]);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        p[u] *= -last_c;
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          const int n = u * HT + j;
          tn[u][j] = (n & 1) ? hi(wt[q & 1][n >> 1]) : lo(wt[q & 1][n >> 1]);
        }
      }
#pragma unroll
      for (int j = 0; j + 1 < HT; j += 2)
#pragma unroll
        for (int u = 0; u < 2; ++u) IO::mma2(p[u], tn[u][j], tn[u][j + 1], dz1[j], dz1[j + 1]);
      if (HT & 1)
#pragma unroll
        for (int u = 0; u < 2; ++u) mmz(p[u], tn[u][HT - 1], dz1[HT - 1]);
#pragma unroll
      for (int u = 0; u < 2; ++u) x.PB[((NW + w) * NT + 2 * q + u) * 64 + lane] = p[u];
      RP_FENCE();
    }
    // dW1 += [XQ | XK]^T [dZbar1 ; dZ1]
    frag dzd[HT], dz1d[HT];
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      dzd[j] = flip(dt[j], x.ident);
      dz1d[j] = flip(dz1[j], x.ident);
    }
#pragma unroll
    for (int I = 0; I < NT; ++I) {
      const frag qd = x.token_k(st, 0, I), kd = x.token_k(st, 1, I);
#pragma unroll
      for (int j = 0; j < HT; ++j) IO::mma2(dW1c[I][j], qd, kd, dzd[j], dz1d[j]);
      RP_FENCE();
    }
  }
  lds_barrier();
  RP_RELANE();
  finish(a.first);
  const bool poison = pair && x.is_lost();
  if (pair) {
    if (tid == 0 && poison) atomicAdd(a.lost_count, 1u);
    x.raise(fl, 1, a.n_stages - a.first);
  }
  // the gradient of the state entering `first`: of the initial state, or for the next launch
  if (a.first == 0) {
#pragma unroll
    for (int j = 0; j < HT; ++j) {
      const int hb = 16 * (w * HT + j);
#pragma unroll
      for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          g1[(size_t)feat(I, 4 * g + r) * F + hb + c] = dW1c[I][j][r];
          g2[(size_t)(hb + 4 * g + r) * D + feat(I, c)] = dW2c[j][I][r];
        }
    }
  } else {
    f32x4* s1 = reinterpret_cast<f32x4*>(g1) + (w * NT * HT) * 64 + lane;
    f32x4* s2 = reinterpret_cast<f32x4*>(g2) + (w * NT * HT) * 64 + lane;
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int I = 0; I < NT; ++I) {
        s1[(I * HT + j) * 64] = dW1c[I][j];
        s2[(j * NT + I) * 64] = dW2c[j][I];
      }
  }
  for (int i = tid; i < F; i += 512) a.d_b1[bh * F + i] = poison ? __builtin_nanf("") : DB1[i];
  if (red && c == 0) *reinterpret_cast<f32x4*>(a.d_b2 + bh * D + x.own) = db2();
  x.add_norm_grads(dgam(), dbet());
}

}  // namespace rp

template <int D>
__global__ void __launch_bounds__(512) ttt_mlp_bwd_rp_kernel(MlpBwdRpArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  size_t bh = blockIdx.x;
  int role = a.role;
  const bool pair = role == 2;
  if (pair) {
    bh = (size_t)(blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
    role = (blockIdx.x >> 3) & 1;
    if (bh >= (size_t)a.B * a.H) return;
  }
  if (role == 0)
    rp::producer<D>(a, smem, bh, pair);
  else
    rp::consumer<D>(a, smem, bh, pair);
}

#undef RP_RELANE
#undef RP_FENCE

template <int D>
hipError_t launch_mlp_bwd_rp_d(const MlpBwdRpArgs& a, hipStream_t s) {
  constexpr auto kern = ttt_mlp_bwd_rp_kernel<D>;
  constexpr int bytes = MlpRpLds<D>::BYTES;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  // two workgroups per unit: workgroups b and b + 8 of every 16 share a unit
  const unsigned units = (unsigned)(a.B * a.H), grid = a.role == 2 ? (units + 7) / 8 * 16 : units;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), bytes, s, a);
  return hipGetLastError();
}

}  // namespace ttt
