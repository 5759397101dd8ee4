// TTT-Linear multi-stage forward for gfx950: the workgroup kernel of ttt_linear_fwd_mw.hip.h with
// the output path skewed by one mini-batch.
//
// Per mini-batch t a wave has two dependency chains:
//   recurrence  W_t -> Z1 -> LayerNorm statistics -> G -> W_{t+1}     (must finish before t+1 starts)
//   output      Zbar_t -> LayerNorm statistics -> out_t               (nothing waits for it)
// Each needs its own cross-wave exchange of row sums.  Here the output chain of mini-batch t-1 runs
// inside iteration t: its two sums travel in the same LDS exchange as the six sums of the
// recurrence (lane group g publishes sums g and g+4: eight in all), so there is ONE barrier per
// mini-batch, and between two barriers the instruction stream always holds two independent chains
// for the in-order issue to interleave.  The exchange buffer is double-buffered by parity because
// one barrier per iteration does not separate a fast wave's next write from a slow wave's read.
#pragma once
#include <type_traits>

#include "ttt_linear_fwd_mw.hip.h"

namespace ttt {

// RAW = 0: the operands are given (xq, xk, xv [B,H,seq,d], lr, token_eta of LinearFwdArgs).
// RAW > 0: the kernel forms them from the projections (FusedInputsArgs: head split by addressing, rotary embedding
// of xq and xk, lr gate, token_eta), i.e. it does the work of ttt_inner_inputs_kernel inside its tile loads:
//   * a wave loads only the features it owns of the raw xq, xk, xv rows (strided [B,seq,H,d] rows), three
//     mini-batches ahead, rotates its xq and xk features in the shadow of the state update two mini-batches ahead
//     of their use, and puts them into LDS; behind the next barrier (the one the recurrence has anyway) every wave
//     reads the full rotated rows back.  The rotation is therefore done once per unit, not once per wave, and no
//     barrier is added;
//   * RAW = 1: the position of a token repeats with the mini-batch (pos_wrap divides K: the reference's default),
//     cosines and sines stay in registers; RAW = 2: positions run over the sequence (pos_wrap = 0), cosines and sines
//     are loaded with the rows;
//   * the operands as used (rotated xq, xk; xv; lr) are written out in [B,H,seq,d] order when the caller asks for them
//     (ttt_linear_bwd needs them): the wave that owns a feature stores it.
// RAW = 3: the operands are given, and fetched the same way: every wave loads only the features it owns and the
// full xq, xk rows reach the waves through LDS (half the vector loads of RAW = 0, where every wave loads every row).
// RAW = 4: as RAW = 3 with the operands formed as x + xq, x + xk, x + xv (LinearFwdArgs::xin: a layer of a stack whose
// input is the output of the layer below plus its own projections); x may be the memory `out` is written to: a wave
// reads a row's own features three mini-batches before it writes that row's own features, and no other wave
// touches them.
// RAW = 5: the operands are given, and a CONTROL WAVE beside the NW compute waves brings them in: it copies the rows of
// xq, xk, xv and lr of a mini-batch global -> LDS without passing registers (one 1 KiB row per feature tile and
// tensor, 16 bytes per lane: exactly the fragment that lane holds of the tile), four mini-batches ahead into a ring of
// four slots, and takes part in every barrier.  The compute waves issue no global load at all: behind the barrier of a
// mini-batch they read the next one's fragments from LDS.  (A load costs the wave that issues it up to a hundred
// cycles of stalled issue, nine of them per wave and mini-batch with f32 I/O.)  For f32 I/O with one feature tile per
// wave, where a unit has a CU to itself (the control wave shares a SIMD with a compute wave: the kernel must stay
// within 256 registers) and whole mini-batches of 16 tokens.
// ADAM: the state update W -= XK^T (eta_last G) is replaced by one Adam step on that gradient per mini-batch
// (reference rust/core/src/linear_adam.rs:76-128): the gradient tile is formed by the same matrix instructions into a
// zero accumulator, the moments live in registers beside the state (three times the state's registers), bias
// corrections come from running powers of beta1, beta2.  Everything else -- products, LayerNorm, output -- is the
// plain kernel's; the output of a mini-batch does not see its own update in either.
// COMPACT: one loop body per ring slot, with the branches of the first and the last pass (see `pass` below).
// STATES: only the recurrence runs, from a given state, and the state entering every one of n_stages + 1 mini-batches is
// written as a checkpoint: no output, no attention block, no final state (see ttt_linear_states_kernel).  The unit and the
// index of its initial state are then given (unit, state) instead of following from the workgroup's index.
template <class T, int D, int NW, int PF, bool FULL, bool FAC, int RAW, bool ADAM = false, bool STATES = false, bool COMPACT = false, bool CKPT = !ADAM>
__device__ __forceinline__ void linear_fwd_sk_body(const LinearFwdArgs& a, const FusedInputsArgs* fip,
                                                   const AdamArgs* adam = nullptr, size_t unit = 0, size_t state = 0) {
  static_assert(!ADAM || (D <= 64 && !FAC && (RAW == 0 || RAW == 3 || RAW == 5)), "Adam inner optimiser: head_dim <= 64, operands given, no checkpoints");
  static_assert(!STATES || (D <= 64 && !FAC && RAW == 0 && !ADAM), "states alone: head_dim <= 64, operands given");
  using IO = Io<T>;
  using frag = typename IO::frag;
  using elem = typename IO::elem;
  constexpr int NT = D / 16, TPW = NT / NW;
  constexpr bool BF = sizeof(elem) == 2;
  constexpr float inv_d = 1.0f / D;
  static_assert(NW > 1, "the skewed kernel is for two or more waves per unit");
  __shared__ __attribute__((aligned(16))) float ex[2][8 * 16 * NW];
  // f32 products with one feature tile per wave are bound by the f32 matrix instructions: the waves then share what
  // each would otherwise compute for itself.  Every wave transposes its own XK tile and forms the attention block over
  // its own 16 features; both cross LDS with the row sums (same barrier, same double buffering) and are read back
  // behind it: 8 matrix instructions per wave and mini-batch instead of 32.
  constexpr bool SHARE = !BF && TPW == 1;
  __shared__ f32x4 kdx[SHARE ? 2 : 1][SHARE ? NT : 1][64];
  __shared__ f32x4 atx[SHARE ? 2 : 1][SHARE ? NW : 1][64];

  constexpr bool DMA = RAW == 5;
  // XK with tokens along k, for the state update: where the rows are shared through LDS anyway, the transposing LDS load
  // gives it, instead of a matrix instruction and two conversions per tile (the waves are bound by what they issue; 384 units
  // x 2048 tokens, d = 64: 128.3 -> 127.3 us, saving update factors 148.7 -> 140.6 us; runs of one side differ by 0.3 us).  A zero token_eta[K-1] then masks G'' in the
  // update, where it makes the transpose zero otherwise.  Not where the operands are formed here (a layer 199.3 -> 200.1 us)
  // and not with the Adam step (230 -> 240 us), whose loops are scheduled worse with it.
  constexpr bool TRK = RAW >= 3 && !DMA && BF && !ADAM;
  const int lane = threadIdx.x & 63, w = (threadIdx.x >> 6) % NW;
  // RAW = 5: the wave behind the compute waves is the control wave; up to the point where it branches off it does what
  // wave 0 does (w == 0: valid loads) and it stores nothing
  const bool ctlw = DMA && __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) == NW;
  const int c = lane & 15, g = lane >> 4;
  const size_t bh = STATES ? unit : blockIdx.x;
  const int h = (int)(bh % a.H);
  // Arguments of every mini-batch held in scalar registers (see held).  384 units x 2048 tokens, d = 64: 127 -> 117 us, saving
  // update factors 142 -> 128; d = 32 99 -> 97; f32, 96 units 215.4 -> 214.2.  Not with the Adam step (230 -> 231), and the length
  // only where the loop has a branch-free middle: held in the other loops (wide heads, d = 128: 193 -> 230 us; f32 215 -> 218; the
  // Adam step 230 -> 258) it has the compiler take them apart.
  constexpr bool HOLD_EPS = !ADAM, HOLD_N = BF && !ADAM && NT <= 4;
  const int K = a.K, n_held = HOLD_N ? held(a.n_stages) : 0, n_stages_ = (HOLD_N ? n_held : a.n_stages) + (STATES ? 1 : 0);
  const float eps_held = HOLD_EPS ? held(a.eps) : 0.f;
  auto n_st = [&]() { return HOLD_N ? n_held : a.n_stages; };
  auto eps = [&]() { return HOLD_EPS ? eps_held : a.eps; };
  const UnitBase<T, D> ub(a, bh);

  // same scale folding as the unskewed kernel: G'' = -sc lr G, M'' = (token_eta[t]/sc)(1 + A)
  constexpr bool FORM = RAW == 1 || RAW == 2;  // the operands are formed here from the projections
  auto tok_eta = [&](int i) {
    if constexpr (FORM) return fmaxf(fip->token_idx[i] + fip->learnable_token_idx[i], 0.f);
    else return a.token_eta[i];
  };
  const float te_last = tok_eta(K - 1);
  const bool upd = te_last != 0.f;
  const float sc = upd ? te_last : 1.f;
  const float rho_c = (c < K) ? tok_eta(c) / sc : 0.f;
  const frag ident = identity_frag<T>(c, g);
  const frag nident = identity_frag<T>(c, g, -1.f);
  const frag ones = splat_frag<T>(1.f);
  const size_t sb = STATES ? state : a.state_per_batch ? bh : (size_t)h;
  f32x4 gam[TPW], bet[TPW], bT[TPW], a2[TPW];
#pragma unroll
  for (int jj = 0; jj < TPW; ++jj)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int f = own_offset<TPW>(w, jj, g) + r;
      gam[jj][r] = a.gamma[h * D + f];
      bet[jj][r] = a.beta[h * D + f];
      bT[jj][r] = a.b0[sb * D + f];
      a2[jj][r] = gam[jj][r] * gam[jj][r];
    }
  f32x4 Wc[NT][TPW];
  load_state_slice<D, TPW>(Wc, a.W0 + sb * D * D, w, c, g);
  // the kernel carries the centred state (see centre_state): row means in LDS, the exchange buffer as scratch
  __shared__ __attribute__((aligned(16))) float m0s[D + 4];
  static_assert((NW + 2) * D <= 2 * 8 * 16 * NW, "the exchange buffer doubles as scratch of centre_state");
  float sum_a;  // of gamma^2, from centre_state

  // ADAM: first and second moments of this wave's W tiles and bias rows, and the running powers beta^step
  f32x4 Wm[ADAM ? NT : 1][TPW], Wv[ADAM ? NT : 1][TPW], bm[TPW], bv[TPW];
  float pw1 = 1.f, pw2 = 1.f;
  if constexpr (ADAM) {
    const bool have = adam->Wm0 != nullptr;
    const float um = 1.f / (1.f - adam->beta1), uv = 1.f / (1.f - adam->beta2);
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const size_t at = bh * D * D + feat(I, 4 * g + r) * D + feat(w * TPW + jj, c);
          Wm[I][jj][r] = have ? adam->Wm0[at] * um : 0.f;
          Wv[I][jj][r] = have ? adam->Wv0[at] * uv : 0.f;
        }
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const size_t at = bh * D + own_offset<TPW>(w, jj, g) + r;
        bm[jj][r] = have ? adam->bm0[at] * um : 0.f;
        bv[jj][r] = have ? adam->bv0[at] * uv : 0.f;
      }
    for (int i = 0; i < adam->step0; ++i) {
      pw1 *= adam->beta1;
      pw2 *= adam->beta2;
    }
  }
  // One Adam step on a tile: gneg = -gradient (what the plain kernel would add to the state).  The moments are carried
  // as m / (1 - beta1) and v / (1 - beta2), so that each decays and takes its new term in one or two instructions, and
  // lr m^ / (sqrt(v^) + eps) is taken as ad_k m / (sqrt(v) + ad_e) with the bias corrections in the two scalars: eight
  // instructions per element, two of them transcendental, where the step as written has eleven.
  float ad_k = 0.f, ad_e = 0.f;
  auto adam_tile = [&](f32x4& x, f32x4& m, f32x4& v, f32x4 gneg) {
    if constexpr (ADAM) {
      const float b1 = adam->beta1, b2 = adam->beta2;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        m[r] = __builtin_fmaf(b1, m[r], -gneg[r]);
        v[r] = __builtin_fmaf(b2, v[r], gneg[r] * gneg[r]);
        const float den = __builtin_amdgcn_sqrtf(v[r]) + ad_e;  // 1 ulp; v is far above the denormals
        x[r] = __builtin_fmaf(ad_k, m[r] * __builtin_amdgcn_rcpf(den), x[r]);
      }
    }
  };
  // pending output of the previous mini-batch (its LayerNorm sums travel in the next exchange) and of the
  // one before (sums known: it is finished while the next exchange is in flight)
  f32x4 zbp[TPW], zbo[TPW];
  frag qop[TPW], qoo[TPW];
  float so0 = 0.f, so1 = 0.f;
#pragma unroll
  for (int jj = 0; jj < TPW; ++jj) {
    zbp[jj] = zbo[jj] = f32x4{0.f, 0.f, 0.f, 0.f};
    qop[jj] = qoo[jj] = IO::zero();
  }

  // Every sum starts from its first term, not from zero: a wave is bound by the number of instructions it issues, and each
  // sum from zero has one that adds nothing (d = 32, 384 units x 2048 tokens: 97.4 -> 95.4 us, d = 64 116.5 -> 114.7, d = 96, 128
  // units 146.5 -> 143.6, d = 128, 64 units 193.7 -> 190.6; f32, d = 64, 96 units 215.7 -> 211.9).  Not with the Adam step (230 -> 235).
  constexpr bool FIRST = !ADAM;
  // publish this lane group's two sums ...
  auto exchange8_publish = [&](const float (&S)[8], int parity) {
    // lane group g ends up with sums g and g+4 reduced over the wave, and publishes them
    const float v0 = xg_sum4_scatter(S[0], S[1], S[2], S[3]);
    const float v1 = xg_sum4_scatter(S[4], S[5], S[6], S[7]);
    float* e = ex[parity];
    e[(g * 16 + c) * NW + w] = v0;
    e[((g + 4) * 16 + c) * NW + w] = v1;
  };
  // ... wait for the other waves, add up
  auto exchange8_collect = [&](float (&S)[8], int parity) {
    const float* e = ex[parity];
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float s = FIRST ? e[(i * 16 + c) * NW] : 0.f;
#pragma unroll
      for (int ww = FIRST; ww < NW; ++ww) s += e[(i * 16 + c) * NW + ww];
      S[i] = s;
    }
  };
  auto exchange8 = [&](float (&S)[8], int parity) {
    exchange8_publish(S, parity);
    exchange8_collect(S, parity);
  };
  // In-lane sums of a pending Zbar.  One routine with explicit fused multiply-adds for every place that forms
  // them: a sequence processed in several calls must give the same bits as one call.
  auto pend_sums = [&](const f32x4 (&z)[TPW], float& s0, float& s1) {
    s0 = s1 = 0.f;
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool first = FIRST && jj == 0 && r == 0;
        s0 = first ? z[jj][r] : s0 + z[jj][r];
        s1 = first ? z[jj][r] * z[jj][r] : __builtin_fmaf(z[jj][r], z[jj][r], s1);
      }
  };
  // the six moments of Z1, feature tile jj
  float z_first = 0.f;
  auto moments = [&](float (&S)[8], int jj, const f32x4& z, const f32x4& uu, const f32x4& bq) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float az = a2[jj][r] * z[r];
      if (jj == 0 && r == 0) z_first = z[r];
      if (FIRST && jj == 0 && r == 0) {
        S[0] = z[r];
        S[2] = az;
        S[3] = az * z[r];
        S[4] = bq[r];
        S[5] = bq[r] * z[r];
      } else {
        S[0] += z[r];
        if (jj != 0 || r != 0) S[1] = jj == 0 && r == 1 ? __builtin_fmaf(z_first, z_first, z[r] * z[r]) : __builtin_fmaf(z[r], z[r], S[1]);
        S[2] = __builtin_fmaf(a2[jj][r], z[r], S[2]);
        S[3] = __builtin_fmaf(az, z[r], S[3]);
        S[4] = __builtin_fmaf(gam[jj][r], uu[r], S[4]);
        S[5] = __builtin_fmaf(bq[r], z[r], S[5]);
      }
    }
  };
  // out = xq + gamma (zbar - mu) rstd + beta for the pending mini-batch
  auto emit_output = [&](float s0, float s1, int stage, const f32x4 (&zbp)[TPW], const frag (&qop)[TPW]) {
    const float mu = s0 * inv_d;
    const float rstd = __builtin_amdgcn_rsqf(fmaxf(s1 * inv_d - mu * mu, 0.f) + eps());
    if (FULL || c < K) {
      elem* po = reinterpret_cast<elem*>(ub.out + UnitBase<T, D>::row_off(stage, K, c));
      f32x4 o[TPW];
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        f32x4 qb;
        if (BF) {
          qb = bet[jj];
          IO::mma(qb, ident, qop[jj]);
        } else {
          qb = IO::to_f32(qop[jj]) + bet[jj];
        }
        o[jj] = qb + gam[jj] * ((zbp[jj] - mu) * rstd);
      }
      if (TPW == 1) {
        store4<T>(po + own_offset<TPW>(w, 0, g), o[0]);
      } else {
#pragma unroll
        for (int qq = 0; qq < TPW / 2; ++qq)
          IO::store8(po + own_offset<TPW>(w, 2 * qq, g), o[2 * qq], o[2 * qq + 1]);
      }
    }
  };

  // b += colsum G''.  The bias is the accumulator input of the next mini-batch's Z1 and Zbar products, which are
  // k = 32 matrix instructions with bf16 I/O, and the scheduler is free to place them right behind this k = 16 update:
  // a matrix instruction that takes its accumulator from one of ANOTHER shape less than five wait states earlier
  // reads a stale value (the hardware interlocks only equal shapes; measured, see ttt_selftest.hip.h).  The wait
  // states are therefore put behind the update by hand, tied to the bias registers so that no reader of the bias can
  // be scheduled in front of them: nothing measurable at any size.  (Issuing the update as a k = 32 instruction with
  // a zero half, the other way to make the shapes equal, cost 10 % of the kernel's time at every size.)  In most
  // instantiations the scheduler leaves the W update's matrix instructions between the pair anyway; the one that had
  // them adjacent gave outputs 1 % off from the sixth mini-batch on.  The build's assembly scan (isa_check.py) refuses
  // any code in which such a pair is closer than five wait states.
  auto bias_update = [&](f32x4 (&b)[TPW], const frag (&gd)[TPW], frag ones_or_zero) {
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) IO::mma(b[jj], gd[jj], ones_or_zero);
    if constexpr (BF) {
      if constexpr (TPW == 1) asm volatile("s_nop 4" : "+v"(b[0]));
      else if constexpr (TPW == 2) asm volatile("s_nop 4" : "+v"(b[0]), "+v"(b[1]));
      else
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) asm volatile("s_nop 4" : "+v"(b[jj]));
    }
  };
  // token_eta[K-1] == 0 means "no state update": instead of a branch inside the loop the two operands
  // that carry tokens into the update (XK^T, the ones column of the bias update) are made zero
  const unsigned upd_mask = upd ? ~0u : 0u;
  auto and_mask = [](frag f, unsigned m) -> frag {
    if constexpr (BF) {
      const u32x2 v = __builtin_bit_cast(u32x2, f);
      return __builtin_bit_cast(frag, u32x2{v[0] & m, v[1] & m});
    } else {
      return f;
    }
  };
  // s2 of the LN-L2 gradient, a sum of two products of which one is rounded before the other is added: written out, or the
  // compiler decides it in each copy of the body, and a mini-batch is rounded by its place in the loop.  Wide heads keep what
  // the compiler once chose for their loop (two of three mini-batches the other way): any other rounding there is as good, but a
  // stack of six TTT-Linear and two TTT-MLP layers at d = 128 carries a last bit on to 1.0 % of its output, as much as callers who
  // compare one version's results with the next's allow for.
  auto g_norm_sum = [&](const float (&S)[8], float mu, float rstd, bool square_fused) {
    const float m = S[5] - mu * S[4], q = S[3] - 2.f * mu * S[2] + mu * mu * sum_a, r2 = rstd * rstd;
    return square_fused ? __builtin_fmaf(r2, q, rstd * m) : __builtin_fmaf(m, rstd, r2 * q);
  };
  const frag ident_upd = upd ? ident : IO::zero();
  const frag ones_upd = upd ? ones : IO::zero();

  constexpr int R = PF + 1;
  StageInMw<T, NT, TPW> buf[R];
  // ---- RAW: the raw rows of the own features, three mini-batches ahead (ring index = mini-batch % R, as for buf)
  struct RawIn {
    frag q[TPW], k[TPW], v[TPW];
    frag x[TPW];                // RAW = 4 only
    float z;                    // lr logit of the lane's token
    f32x2 cs[TPW], sn[TPW];     // RAW = 2 only
  };
  RawIn raw[RAW != 0 ? R : 1];
  f32x2 cs_fix[TPW], sn_fix[TPW];  // RAW = 1: cosines and sines of the lane's token position and own feature pairs
  u32x4* xrot = nullptr;           // rotated rows in LDS: [2 buffers][xq, xk][feature pair][lane]
  float lr_bias_h = 0.f;
  if constexpr (RAW != 0 && !DMA) {
    static_assert(BF && PF == 2, "rows shared through LDS: bf16 I/O");
    static_assert(!FORM || NT <= 4, "operands formed from the projections: head_dim <= 64");
    __shared__ u32x4 xrot_s[2][2][NT / 2][64];
    xrot = &xrot_s[0][0][0][0];
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) {
      cs_fix[jj] = f32x2{1.f, 1.f};
      sn_fix[jj] = f32x2{0.f, 0.f};
    }
  }
  if constexpr (FORM) {
    lr_bias_h = fip->lr_bias[h];
    if (RAW == 1 && fip->cos != nullptr) {
      const int pos = (fip->pos_offset + c) % fip->pos_wrap;
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        const size_t o = (size_t)pos * (D / 2) + own_offset<TPW>(w, jj, g) / 2;
        cs_fix[jj] = *reinterpret_cast<const f32x2*>(fip->cos + o);
        sn_fix[jj] = *reinterpret_cast<const f32x2*>(fip->sin + o);
      }
    }
    if (fip->token_eta_out != nullptr && bh == 0)
      for (int i = threadIdx.x; i < a.seq; i += 64 * NW) fip->token_eta_out[i] = tok_eta(i % K);
  }
  const bool has_x = a.xin != nullptr;  // RAW = 4: a problem without x takes the operands as they are (x = 0)
  // raw rows of unit (b, h): token t of the unit is row (b * seq + t) * H + h of the [B,seq,H,d] tensors
  const size_t bidx = bh / a.H;
  const unsigned raw_row = (unsigned)a.H * (unsigned)(D * sizeof(elem));  // bytes from one token to the next
  auto load_raw = [&](RawIn& r, int stage) {
    if constexpr (RAW != 0 && !DMA) {
      if (FULL) stage = min(stage, n_stages_ - 1);
      const bool ok = FULL || ((c < K) && (stage < n_stages_));
      const unsigned t = (unsigned)stage * (unsigned)K + (unsigned)c;
      const unsigned char *bq, *bk, *bv;
      unsigned off;
      if constexpr (FORM) {
        const size_t row0 = (bidx * (size_t)a.seq * a.H + h) * (D * sizeof(elem));
        bq = static_cast<const unsigned char*>(fip->xq) + row0;
        bk = static_cast<const unsigned char*>(fip->xk) + row0;
        bv = static_cast<const unsigned char*>(fip->xv) + row0;
        off = t * raw_row;
      } else {
        bq = ub.xq;
        bk = ub.xk;
        bv = ub.xv;
        off = UnitBase<T, D>::row_off(stage, K, c);
      }
      if (TPW == 1) {
        const unsigned o1 = off + own_offset<TPW>(w, 0, g) * (unsigned)sizeof(elem);
        r.q[0] = ok ? load4<T>(reinterpret_cast<const elem*>(bq + o1)) : IO::zero();
        r.k[0] = ok ? load4<T>(reinterpret_cast<const elem*>(bk + o1)) : IO::zero();
        r.v[0] = ok ? load4<T>(reinterpret_cast<const elem*>(bv + o1)) : IO::zero();
        if constexpr (RAW == 4) r.x[0] = (ok && has_x) ? load4<T>(reinterpret_cast<const elem*>(ub.xin + o1)) : IO::zero();
      } else {
#pragma unroll
        for (int qq = 0; qq < TPW / 2; ++qq) {
          const unsigned o2 = off + own_offset<TPW>(w, 2 * qq, g) * (unsigned)sizeof(elem);
          IO::load8(reinterpret_cast<const elem*>(bq + o2), ok, r.q[2 * qq], r.q[2 * qq + 1]);
          IO::load8(reinterpret_cast<const elem*>(bk + o2), ok, r.k[2 * qq], r.k[2 * qq + 1]);
          IO::load8(reinterpret_cast<const elem*>(bv + o2), ok, r.v[2 * qq], r.v[2 * qq + 1]);
          if constexpr (RAW == 4) IO::load8(reinterpret_cast<const elem*>(ub.xin + o2), ok && has_x, r.x[2 * qq], r.x[2 * qq + 1]);
        }
      }
      if constexpr (FORM) {
        const elem* zl = static_cast<const elem*>(fip->lr_logits) + (bidx * (size_t)a.seq * a.H + h);
        r.z = ok ? IO::load1(zl + (size_t)t * a.H) : 0.f;
      } else {
        r.z = ok ? IO::load1(reinterpret_cast<const elem*>(ub.lr + t * (unsigned)sizeof(elem))) : 0.f;  // lr itself
      }
      if constexpr (RAW == 2) {
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          const size_t o = (size_t)(fip->pos_offset + (int)t) * (D / 2) + own_offset<TPW>(w, jj, g) / 2;
          r.cs[jj] = fip->cos != nullptr ? *reinterpret_cast<const f32x2*>(fip->cos + o) : f32x2{1.f, 1.f};
          r.sn[jj] = fip->sin != nullptr ? *reinterpret_cast<const f32x2*>(fip->sin + o) : f32x2{0.f, 0.f};
        }
      }
    }
  };
  // own features of a mini-batch: rotate, keep (own-feature operands of dst), share through LDS buffer `pb`, store
  auto rotate_share = [&](const RawIn& r, StageInMw<T, NT, TPW>& dst, int stage, int pb) {
    if constexpr (RAW != 0 && !DMA) {
      const bool tok = FULL || c < K;
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        if constexpr (FORM) {
          const f32x2 cs = RAW == 2 ? r.cs[jj] : cs_fix[jj], sn = RAW == 2 ? r.sn[jj] : sn_fix[jj];
          dst.qo[jj] = IO::to_frag(rope_rotate4(IO::to_f32(r.q[jj]), cs, sn));
          dst.ko[jj] = IO::to_frag(rope_rotate4(IO::to_f32(r.k[jj]), cs, sn));
          dst.vo[jj] = r.v[jj];
        } else if constexpr (RAW == 4) {
          const f32x4 x = IO::to_f32(r.x[jj]);
          dst.qo[jj] = IO::to_frag(x + IO::to_f32(r.q[jj]));
          dst.ko[jj] = IO::to_frag(x + IO::to_f32(r.k[jj]));
          dst.vo[jj] = IO::to_frag(x + IO::to_f32(r.v[jj]));
        } else {
          dst.qo[jj] = r.q[jj];
          dst.ko[jj] = r.k[jj];
          dst.vo[jj] = r.v[jj];
        }
      }
      // the gate in the precision the operand has when it is a tensor of its own
      // (a token past the end of a short mini-batch has no learning rate: it must not reach the state update)
      if constexpr (FORM) dst.lr = tok ? IO::rounded(lr_gate(r.z + lr_bias_h, fip->lr_scale)) : 0.f;
      else dst.lr = r.z;
      u32x4* xb = xrot + (size_t)pb * 2 * (NT / 2) * 64;
      if (TPW == 1) {
        const int J = w;
        unsigned char* pq_ = reinterpret_cast<unsigned char*>(xb + (0 * (NT / 2) + (J >> 1)) * 64 + lane) + 8 * (J & 1);
        unsigned char* pk_ = reinterpret_cast<unsigned char*>(xb + (1 * (NT / 2) + (J >> 1)) * 64 + lane) + 8 * (J & 1);
        *reinterpret_cast<u32x2*>(pq_) = __builtin_bit_cast(u32x2, dst.qo[0]);
        *reinterpret_cast<u32x2*>(pk_) = __builtin_bit_cast(u32x2, dst.ko[0]);
      } else {
#pragma unroll
        for (int qq = 0; qq < TPW / 2; ++qq) {
          const int q = w * (TPW / 2) + qq;
          const u32x2 a0 = __builtin_bit_cast(u32x2, dst.qo[2 * qq]), a1 = __builtin_bit_cast(u32x2, dst.qo[2 * qq + 1]);
          const u32x2 b0 = __builtin_bit_cast(u32x2, dst.ko[2 * qq]), b1 = __builtin_bit_cast(u32x2, dst.ko[2 * qq + 1]);
          xb[(0 * (NT / 2) + q) * 64 + lane] = u32x4{a0[0], a0[1], a1[0], a1[1]};
          xb[(1 * (NT / 2) + q) * 64 + lane] = u32x4{b0[0], b0[1], b1[0], b1[1]};
        }
      }
      if (FORM && stage < n_stages_ && tok) {
        const unsigned off = UnitBase<T, D>::row_off(stage, K, c);
        const size_t u0 = bh * (size_t)a.seq * (D * sizeof(elem));
        auto put = [&](void* base, const frag (&x)[TPW]) {
          if (base == nullptr) return;
          unsigned char* pb_ = static_cast<unsigned char*>(base) + u0 + off;
          if (TPW == 1) {
            *reinterpret_cast<u32x2*>(pb_ + own_offset<TPW>(w, 0, g) * sizeof(elem)) = __builtin_bit_cast(u32x2, x[0]);
          } else {
#pragma unroll
            for (int qq = 0; qq < TPW / 2; ++qq) {
              const u32x2 a0 = __builtin_bit_cast(u32x2, x[2 * qq]), a1 = __builtin_bit_cast(u32x2, x[2 * qq + 1]);
              *reinterpret_cast<u32x4*>(pb_ + own_offset<TPW>(w, 2 * qq, g) * sizeof(elem)) = u32x4{a0[0], a0[1], a1[0], a1[1]};
            }
          }
        };
        put(fip->xq_out, dst.qo);
        put(fip->xk_out, dst.ko);
        put(fip->xv_out, dst.vo);
        if (fip->lr_out != nullptr && w == 0 && g == 0)
          IO::store1(static_cast<elem*>(fip->lr_out) + bh * (size_t)a.seq + (size_t)stage * K + c, dst.lr);
      }
    }
  };
  // the full rotated rows of a mini-batch, from LDS buffer `pb` (behind a barrier that follows rotate_share)
  auto gather_rows = [&](StageInMw<T, NT, TPW>& dst, int pb) {
    if constexpr (RAW != 0 && !DMA) {
      const u32x4* xb = xrot + (size_t)pb * 2 * (NT / 2) * 64;
#pragma unroll
      for (int q = 0; q < NT / 2; ++q) {
        const u32x4 vq = xb[(0 * (NT / 2) + q) * 64 + lane], vk = xb[(1 * (NT / 2) + q) * 64 + lane];
        dst.q[2 * q] = __builtin_bit_cast(frag, u32x2{vq[0], vq[1]});
        dst.q[2 * q + 1] = __builtin_bit_cast(frag, u32x2{vq[2], vq[3]});
        dst.k[2 * q] = __builtin_bit_cast(frag, u32x2{vk[0], vk[1]});
        dst.k[2 * q + 1] = __builtin_bit_cast(frag, u32x2{vk[2], vk[3]});
      }
    }
  };
  // ---- RAW = 5: the ring the control wave fills, and the control wave itself
  constexpr int RS = 4;                                  // slots = mini-batches in flight
  constexpr int kCopies = 3 * NT + 1;                    // copies per mini-batch: the tile rows of xq, xk, xv, and lr
  __shared__ f32x4 ring_s[DMA ? RS : 1][3][DMA ? NT : 1][64];  // [slot][xq, xk, xv][feature tile][lane]
  __shared__ float ringlr_s[DMA ? RS : 1][64];           // lr of the lane's token c
  auto gather_dma = [&](StageInMw<T, NT, TPW>& dst, int stage) {
    if constexpr (DMA) {
      static_assert(!BF && TPW == 1 && FULL && !FAC, "control-wave loads: f32 I/O, one feature tile per wave, whole mini-batches");
      const int sl = stage & (RS - 1);
#pragma unroll
      for (int J = 0; J < NT; ++J) {
        dst.q[J] = ring_s[sl][0][J][lane];
        dst.k[J] = ring_s[sl][1][J][lane];
      }
      dst.qo[0] = ring_s[sl][0][w][lane];
      dst.ko[0] = ring_s[sl][1][w][lane];
      dst.vo[0] = ring_s[sl][2][w][lane];
      dst.lr = ringlr_s[sl][c];
    }
  };
  // The first rows are asked for before the state is centred: a launch of few mini-batches consists of round trips to memory, and
  // this one then overlaps those of the state (and sums over d features go through LDS, see centre_state, and the final state's
  // reference is read while the last output is exchanged).  One mini-batch, 12 units, launch to launch (an empty kernel 3.7): bf16
  // d = 64 10.3 -> 6.8 us, d = 128 17.0 -> 10.8, f32 d = 64 9.5 -> 6.6, d = 128 26.3 -> 19.9; 384 units x 2048 tokens, bf16, d = 64
  // 117.8 -> 114.0.
  if constexpr (RAW != 0 && !DMA) {
#pragma unroll
    for (int u = 0; u < R; ++u) load_raw(raw[u], u);
  } else if constexpr (!DMA) {
#pragma unroll
    for (int u = 0; u < (PF > 0 ? PF : 1); ++u) load_stage_mw<T, D, NW, FULL>(buf[u], ub, K, n_stages_, u, c, g, w);
  }
  if constexpr (DMA) {
    if (ctlw) {
      const unsigned ring0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)&ring_s[0][0][0][0];
      const unsigned lr0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)&ringlr_s[0][0];
      // the copies of one mini-batch (past the end: the last one again, into a slot nobody reads)
      auto copy_in = [&](int stage) {
        const unsigned dst = ring0 + (unsigned)(stage & (RS - 1)) * (3 * NT * 1024);
        const int st_ld = min(stage, n_stages_ - 1);
        const unsigned off = UnitBase<T, D>::row_off(st_ld, K, c);
#pragma unroll
        for (int J = 0; J < NT; ++J) {
          const unsigned fo = (unsigned)(32 * (J >> 1) + 8 * g + 4 * (J & 1)) * 4u;  // the lane's four features of tile J
          lds_dma16(ub.xq, off + fo, dst + (0 * NT + J) * 1024);
          lds_dma16(ub.xk, off + fo, dst + (1 * NT + J) * 1024);
          lds_dma16(ub.xv, off + fo, dst + (2 * NT + J) * 1024);
        }
        // every lane issues (the count of copies in flight must not depend on the lane): lanes 16.. repeat token c's
        lds_dma4(ub.lr, ((unsigned)st_ld * (unsigned)K + (unsigned)c) * 4u, lr0 + (unsigned)(stage & (RS - 1)) * 256u);
      };
#pragma unroll
      for (int u = 0; u < RS; ++u) copy_in(u);
      centre_state<D, NW, TPW, false>(Wc, bT, a.b0 + sb * D, m0s, a.gamma + h * D, sum_a, &ex[0][0], w, c, g);  // (the others do)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - 1) * kCopies) : "memory");  // mini-batch 0 has landed
      asm volatile("s_barrier" ::: "memory");
      for (int st = 0; st < n_stages_; ++st) {
        // mini-batch st + 1 has landed (st + 2 .. st + RS - 1 may be in flight); behind the barrier the compute waves
        // read it, and the slot of mini-batch st, read behind the barrier before, is free
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - 2) * kCopies) : "memory");
        asm volatile("s_barrier" ::: "memory");
        copy_in(st + RS);
      }
      asm volatile("s_barrier" ::: "memory");  // the exchange that flushes the last output
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      return;
    }
  }
  centre_state<D, NW, TPW>(Wc, bT, a.b0 + sb * D, m0s, a.gamma + h * D, sum_a, &ex[0][0], w, c, g);
  if constexpr (DMA) {
    lds_barrier();
    gather_dma(buf[0], 0);
  } else if constexpr (RAW != 0) {
    // mini-batch 0 complete, mini-batch 1 rotated and on its way through LDS (read behind the first barrier of the
    // loop), the raw rows of mini-batch 2 in flight
    rotate_share(raw[0], buf[0], 0, 0);
    lds_barrier();
    gather_rows(buf[0], 0);
    rotate_share(raw[1], buf[1], 1, 1);
  }

  // One pass over R mini-batches (the ring of prefetch registers is indexed at compile time).  CHECKED:
  // the first and the last pass, which test for "no pending output yet" and "past the end"; the passes in
  // between run without any branch, so that everything between two barriers -- the tail of one mini-batch
  // (pending output, G, state update) and the head of the next (products, moments) -- is one basic block and
  // the compiler can interleave the two dependency chains.
  float ps0 = 0.f, ps1 = 0.f;
  CkptCursor<D> ck(a, bh);
  const float b_mean = __builtin_amdgcn_readfirstlane(m0s[D]);  // mean of the initial bias (split off by centre_state)
  static_assert(!FAC || BF, "update factors are saved with bf16 I/O only");
  unsigned char* fac = FAC ? factor_base<D>(a.W_ckpt, a.n_ckpt, bh) : nullptr;
  auto pass = [&](auto checked_tag, int st0) {
    constexpr bool CHECKED = decltype(checked_tag)::value;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int st = st0 + u;
      if constexpr (RAW != 0)
        load_raw(raw[u], st + R);  // its previous content, mini-batch st, was rotated two mini-batches ago
      else
        load_stage_mw<T, D, NW, FULL>(buf[(u + PF) % R], ub, K, n_stages_, st + PF, c, g, w);
      if (CHECKED && st >= n_st()) continue;
      const StageInMw<T, NT, TPW>& cur = buf[u];

      // ---- XK with tokens along k for the state update: depends on nothing computed here, so it
      // is issued first and fills the gaps of the dependent chain below
      frag kd[NT];
      if constexpr (SHARE) {
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
        IO::mma(t, cur.ko[0], ident_upd);  // the own tile; the others come back from LDS behind the barrier
        kdx[st & 1][w][lane] = t;
      } else if constexpr (TRK) {
        // (the rows lie there as fragments, tokens across lanes; they are overwritten behind the next barrier)
        const u32x4* const xk = xrot + ((st & 1) * 2 + 1) * (NT / 2) * 64 + tr_lane(lane);
#pragma unroll
        for (int I = 0; I < NT; ++I) kd[I] = read_tr(reinterpret_cast<const unsigned char*>(xk + (I >> 1) * 64) + 8 * (I & 1));
      } else {
#pragma unroll
        for (int I = 0; I < NT; ++I) {
          f32x4 t = {0.f, 0.f, 0.f, 0.f};
          IO::mma(t, cur.k[I], ident_upd);  // t[r] = XK[s = 4g+r][feat(I,c)]
          kd[I] = IO::to_frag(t);
        }
      }
      // ---- Z1^T, Zbar^T (this wave's feature rows) and the attention block
      f32x4 z1[TPW], zb[TPW], At = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        z1[jj] = bT[jj];
        zb[jj] = bT[jj];
      }
#pragma unroll
      for (int q = 0; q < NT / 2; ++q) {
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          const frag w0 = IO::to_frag(Wc[2 * q][jj]), w1 = IO::to_frag(Wc[2 * q + 1][jj]);
          IO::mma2(z1[jj], w0, w1, cur.k[2 * q], cur.k[2 * q + 1]);
          if constexpr (!STATES) IO::mma2(zb[jj], w0, w1, cur.q[2 * q], cur.q[2 * q + 1]);
        }
        if constexpr (!SHARE && !STATES) IO::mma2(At, cur.k[2 * q], cur.k[2 * q + 1], cur.q[2 * q], cur.q[2 * q + 1]);
      }
      if constexpr (SHARE && !STATES) {
        IO::mma(At, cur.ko[0], cur.qo[0]);  // over the own 16 features
        atx[st & 1][w][lane] = At;
      }
      f32x4 bq[TPW], uu[TPW];  // uu = beta - (xv - xk)
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        if (BF) {
          uu[jj] = bet[jj];
          IO::mma2(uu[jj], nident, ident, cur.vo[jj], cur.ko[jj]);
        } else {
          uu[jj] = bet[jj] - (IO::to_f32(cur.vo[jj]) - IO::to_f32(cur.ko[jj]));
        }
      }
      if constexpr (FORM && NT == 2) settle(kd[0], kd[1]);
      // ---- checkpoint of the state entering this mini-batch (W and b change only behind the barrier);
      // placed at the barrier so that its branch does not cut the stretch in two
      if (CKPT && ck.due()) {
        if (ck.packed) {
          store_ckpt_packed<T, NT, TPW>(ck.W, Wc, w, lane);
          store_bias_true<D, TPW>(ck.b, bT, b_mean, w, c, g);
        } else {
          store_state_f32<D, TPW>(ck.W, ck.b, Wc, bT, m0s, w, c, g);
        }
        ck.advance();
      }
      if constexpr (CKPT) ck.next_stage();
      // (without checkpoints the stretch is cut here all the same: as one, 208.5 us instead of 206)
      if constexpr (!CKPT && !ADAM) __builtin_amdgcn_sched_barrier(0);
      // The wait states of settle() for what the sums read, but behind the branch, which counts as one of them
      if constexpr (BF && !ADAM) {
        if constexpr (TPW == 1) asm volatile("s_nop 5" : "+v"(z1[0]), "+v"(uu[0]));
        else asm volatile("s_nop 5" : "+v"(z1[0]), "+v"(uu[0]), "+v"(z1[1]), "+v"(uu[1]));
      }
      // ---- row sums: six raw moments of Z1 (this mini-batch), two of the pending Zbar
      float S[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, ps0, ps1};  // the pending Zbar's in-lane sums are ready
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        bq[jj] = gam[jj] * uu[jj];
        moments(S, jj, z1[jj], uu[jj], bq[jj]);
      }
      exchange8_publish(S, st & 1);
      // ---- the output pending since two mini-batches (sums known since the last exchange): nothing waits
      // for it, and here it runs while this exchange is in flight (LDS write, barrier, LDS read)
      if constexpr (!STATES) {
        if (!CHECKED || st > 1) emit_output(so0, so1, st - 2, zbo, qoo);
      }
      exchange8_collect(S, st & 1);
      // RAW: the rows of the next mini-batch, rotated by their owners before this barrier
      if constexpr (DMA) gather_dma(buf[(u + 1) % R], st + 1);
      else if constexpr (RAW != 0) gather_rows(buf[(u + 1) % R], (st + 1) & 1);
      so0 = S[6];
      so1 = S[7];
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        zbo[jj] = zbp[jj];
        qoo[jj] = qop[jj];
      }
      if constexpr (SHARE) {
#pragma unroll
        for (int I = 0; I < NT; ++I) kd[I] = IO::to_frag(kdx[st & 1][I][lane]);
        if constexpr (!STATES) {
          At = atx[st & 1][0][lane];
#pragma unroll
          for (int ww = 1; ww < NW; ++ww) At += atx[st & 1][ww][lane];
        }
      }

      // ---- recurrence: G'' , causal correction, state update
      f32x4 G[TPW];
      {
        const float mu = S[0] * inv_d;
        const float var = S[1] * inv_d - mu * mu;
        const float rstd = __builtin_amdgcn_rsqf(fmaxf(var, 0.f) + eps());
        const float s1 = rstd * (S[2] - mu * sum_a) + S[4];
        const float s2 = g_norm_sum(S, mu, rstd, true);
        const float p = -sc * cur.lr * rstd;
        const float c1 = p * rstd, c2 = -c1 * s2 * inv_d, c3 = -p * s1 * inv_d;
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) G[jj] = (z1[jj] - mu) * (a2[jj] * c1 + c2) + (bq[jj] * p + c3);
      }
      frag Gd[TPW];
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
        IO::mma(t, IO::to_frag(G[jj]), ident);
        Gd[jj] = IO::to_frag(t);
      }
      if constexpr (FAC) {
        store_factor<TPW>(fac, Gd, w, lane);
        fac += 32 * D;
      }
      if constexpr (!STATES) {
        f32x4 m;
#pragma unroll
        for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? rho_c * (1.f + At[r]) : 0.f;
        const frag Mf = IO::to_frag(m);
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) IO::mma(zb[jj], Gd[jj], Mf);
      }
      if constexpr (ADAM) {
        pw1 *= adam->beta1;
        pw2 *= adam->beta2;
        {
          // v^ = v c2, m^ = m c1: lr m^ / (sqrt(v^) + eps) = (lr c1 / sqrt(c2)) m / (sqrt(v) + eps / sqrt(c2))
          const float c1 = (1.f - adam->beta1) / (1.f - pw1), rc2 = sqrtf((1.f - pw2) / (1.f - adam->beta2));
          ad_k = -adam->lr * c1 * rc2;
          ad_e = adam->eps * rc2;
        }
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
          for (int jj = 0; jj < TPW; ++jj) {
            f32x4 gneg = {0.f, 0.f, 0.f, 0.f};
            IO::mma(gneg, kd[I], Gd[jj]);
            adam_tile(Wc[I][jj], Wm[I][jj], Wv[I][jj], gneg);
          }
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          f32x4 gneg = {0.f, 0.f, 0.f, 0.f};
          IO::mma(gneg, Gd[jj], ones_upd);
          adam_tile(bT[jj], bm[jj], bv[jj], gneg);
        }
      } else {
        frag Gu[TPW];
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) Gu[jj] = TRK ? and_mask(Gd[jj], upd_mask) : Gd[jj];
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
          for (int jj = 0; jj < TPW; ++jj) IO::mma(Wc[I][jj], kd[I], Gu[jj]);
        bias_update(bT, Gd, ones_upd);
      }
      // this mini-batch's Zbar and xq become the pending output; its in-lane sums are formed here, in the
      // shadow of the state update, not between the next Z1 and its exchange
      if constexpr (!STATES) {
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          zbp[jj] = zb[jj];
          qop[jj] = cur.qo[jj];
        }
        pend_sums(zbp, ps0, ps1);
      }
      // RAW: the own features of the mini-batch after the next, loaded during the previous pass of the loop; read
      // back by every wave behind the next barrier.  LDS buffer st & 1 was last read behind the barrier of the
      // previous mini-batch (TRK: in front of this one's), which every wave has left.
      if constexpr (RAW != 0) rotate_share(raw[(u + 2) % R], buf[(u + 2) % R], st + 2, st & 1);
    }
  };
  if constexpr (COMPACT) {
    for (int st0 = 0; st0 < n_st(); st0 += R) pass(std::true_type{}, st0);
  } else if constexpr (NT <= 4) {
    int st0 = 0;
    pass(std::true_type{}, st0);
    for (st0 = R; st0 + R <= n_st(); st0 += R) pass(std::false_type{}, st0);
    if (st0 < n_st()) pass(std::true_type{}, st0);
  } else {
    // Wide heads (d = 96, 128) keep the loop with its branches: in one long basic block the scheduler overlaps
    // so much that the state tiles no longer fit the register file (d = 128: 30 spilled registers).
    for (int st0 = 0; st0 < n_st(); st0 += R) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int st = st0 + u;
        if constexpr (RAW != 0)
          load_raw(raw[u], st + R);
        else if (PF > 0)
          load_stage_mw<T, D, NW, FULL>(buf[(u + PF) % R], ub, K, n_stages_, st + PF, c, g, w);
        if (st >= n_st()) continue;
        const StageInMw<T, NT, TPW>& cur = buf[u];

        if (ck.due()) {
          if (ck.packed) {
            store_ckpt_packed<T, NT, TPW>(ck.W, Wc, w, lane);
            store_bias_true<D, TPW>(ck.b, bT, b_mean, w, c, g);
          } else {
            store_state_f32<D, TPW>(ck.W, ck.b, Wc, bT, m0s, w, c, g);
          }
          ck.advance();
        }
        ck.next_stage();

        // ---- XK with tokens along k for the state update: depends on nothing computed here, so it
        // is issued first and fills the gaps of the dependent chain below
        frag kd[NT];
        if constexpr (TRK) {
          const u32x4* const xk = xrot + ((st & 1) * 2 + 1) * (NT / 2) * 64 + tr_lane(lane);
#pragma unroll
          for (int I = 0; I < NT; ++I) kd[I] = read_tr(reinterpret_cast<const unsigned char*>(xk + (I >> 1) * 64) + 8 * (I & 1));
        } else {
#pragma unroll
          for (int I = 0; I < NT; ++I) {
            f32x4 t = {0.f, 0.f, 0.f, 0.f};
            IO::mma(t, cur.k[I], ident);  // t[r] = XK[s = 4g+r][feat(I,c)]
            kd[I] = IO::to_frag(t);
          }
        }
        // ---- Z1^T, Zbar^T (this wave's feature rows) and the attention block
        f32x4 z1[TPW], zb[TPW], At = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          z1[jj] = bT[jj];
          zb[jj] = bT[jj];
        }
#pragma unroll
        for (int q = 0; q < NT / 2; ++q) {
#pragma unroll
          for (int jj = 0; jj < TPW; ++jj) {
            const frag w0 = IO::to_frag(Wc[2 * q][jj]), w1 = IO::to_frag(Wc[2 * q + 1][jj]);
            IO::mma2(z1[jj], w0, w1, cur.k[2 * q], cur.k[2 * q + 1]);
            IO::mma2(zb[jj], w0, w1, cur.q[2 * q], cur.q[2 * q + 1]);
          }
          IO::mma2(At, cur.k[2 * q], cur.k[2 * q + 1], cur.q[2 * q], cur.q[2 * q + 1]);
        }
        // ---- row sums: six raw moments of Z1 (this mini-batch), two of the pending Zbar
        f32x4 bq[TPW];
        float S[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          f32x4 uu;  // beta - (xv - xk)
          if (BF) {
            uu = bet[jj];
            IO::mma2(uu, nident, ident, cur.vo[jj], cur.ko[jj]);
          } else {
            uu = bet[jj] - (IO::to_f32(cur.vo[jj]) - IO::to_f32(cur.ko[jj]));
          }
          bq[jj] = gam[jj] * uu;
          moments(S, jj, z1[jj], uu, bq[jj]);
        }
        pend_sums(zbp, S[6], S[7]);
        const float lr_st = cur.lr;
        frag qo_st[TPW];
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) qo_st[jj] = cur.qo[jj];
        // PF = 0: one set of rows, filled anew as soon as its products are done
        if constexpr (PF == 0) load_stage_mw<T, D, NW, FULL>(buf[0], ub, K, n_stages_, st + 1, c, g, w);
        exchange8_publish(S, st & 1);
        if (st > 1) emit_output(so0, so1, st - 2, zbo, qoo);  // inside the exchange window, as above
        exchange8_collect(S, st & 1);
        if constexpr (RAW != 0) gather_rows(buf[(u + 1) % R], (st + 1) & 1);
        so0 = S[6];
        so1 = S[7];
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          zbo[jj] = zbp[jj];
          qoo[jj] = qop[jj];
        }

        // ---- recurrence: G'' , causal correction, state update
        f32x4 G[TPW];
        {
          const float mu = S[0] * inv_d;
          const float var = S[1] * inv_d - mu * mu;
          const float rstd = __builtin_amdgcn_rsqf(fmaxf(var, 0.f) + eps());
          const float s1 = rstd * (S[2] - mu * sum_a) + S[4];
          const float s2 = g_norm_sum(S, mu, rstd, FULL && u == 2);
          const float p = -sc * lr_st * rstd;
          const float c1 = p * rstd, c2 = -c1 * s2 * inv_d, c3 = -p * s1 * inv_d;
#pragma unroll
          for (int jj = 0; jj < TPW; ++jj) G[jj] = (z1[jj] - mu) * (a2[jj] * c1 + c2) + (bq[jj] * p + c3);
        }
        frag Gd[TPW];
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          f32x4 t = {0.f, 0.f, 0.f, 0.f};
          IO::mma(t, IO::to_frag(G[jj]), ident);
          Gd[jj] = IO::to_frag(t);
        }
        if constexpr (FAC) {
          store_factor<TPW>(fac, Gd, w, lane);
          fac += 32 * D;
        }
        {
          f32x4 m;
#pragma unroll
          for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? rho_c * (1.f + At[r]) : 0.f;
          const frag Mf = IO::to_frag(m);
#pragma unroll
          for (int jj = 0; jj < TPW; ++jj) IO::mma(zb[jj], Gd[jj], Mf);
        }
        if (upd) {
#pragma unroll
          for (int I = 0; I < NT; ++I)
#pragma unroll
            for (int jj = 0; jj < TPW; ++jj) IO::mma(Wc[I][jj], kd[I], Gd[jj]);
          bias_update(bT, Gd, ones);
        }
        // this mini-batch's Zbar and xq become the pending output
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj) {
          zbp[jj] = zb[jj];
          qop[jj] = qo_st[jj];
        }
        if constexpr (RAW != 0) rotate_share(raw[(u + 2) % R], buf[(u + 2) % R], st + 2, st & 1);
      }
    }

  }

  if constexpr (STATES) {  // the state entering the last mini-batch
    store_ckpt_packed<T, NT, TPW>(ck.W, Wc, w, lane);
    store_bias_true<D, TPW>(ck.b, bT, b_mean, w, c, g);
    return;
  }
  // ---- flush the last mini-batch's output
  f32x4 W0[NT][TPW];
  int c_w0 = c, g_w0 = g;
  // Formed from the same lane indices as the prologue's, the compiler keeps the addresses in 32 registers through the loop.  With
  // the Adam step and four waves those are not there: without it f32 spills 18 instead of 44 (384 units, 1 mini-batch 20.4 -> 18.0
  // us; 96 units, 128 mini-batches 274.9 -> 272.0), bf16, 96 units 158.9 -> 154.9.  Two waves and the other kernels gain nothing.
  if constexpr (ADAM && NW == 4) asm volatile("" : "+v"(c_w0), "+v"(g_w0));
  load_state_slice<D, TPW>(W0, a.W0 + sb * D * D, w, c_w0, g_w0);
  {
    float S[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    pend_sums(zbp, S[6], S[7]);
    exchange8(S, n_st() & 1);
    if (n_st() >= 2) emit_output(so0, so1, n_st() - 2, zbo, qoo);
    emit_output(S[6], S[7], n_st() - 1, zbp, qop);
  }
  store_state_final<D, TPW>(a.W_out + bh * D * D, a.b_out + bh * D, W0, a.b0 + sb * D, Wc, bT, m0s, w, c, g);
  if constexpr (ADAM) {
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const size_t at = bh * D * D + feat(I, 4 * g + r) * D + feat(w * TPW + jj, c);
          adam->Wm_out[at] = Wm[I][jj][r] * (1.f - adam->beta1);
          adam->Wv_out[at] = Wv[I][jj][r] * (1.f - adam->beta2);
        }
    if (c == 0) {
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        const size_t at = bh * D + own_offset<TPW>(w, jj, g);
        *reinterpret_cast<f32x4*>(adam->bm_out + at) = bm[jj] * (1.f - adam->beta1);
        *reinterpret_cast<f32x4*>(adam->bv_out + at) = bv[jj] * (1.f - adam->beta2);
      }
    }
  }
  if constexpr (FAC)
    store_state_tiles<D, TPW>(a.W_ckpt + bh * (size_t)a.n_ckpt * (D * D), a.b_ckpt + bh * (size_t)a.n_ckpt * D, Wc, bT, w, lane);
}

// OWN = 1: every wave loads only the features it owns, full rows through LDS (RAW = 3); OWN = 2: the same with the
// operands formed as x + xq, x + xk, x + xv (RAW = 4)
template <class T, int D, int NW, int PF, bool FULL, bool FAC = false, int OWN = 0>
__global__ void __launch_bounds__(64 * NW) ttt_linear_fwd_sk_kernel(Problems<LinearFwdArgs> problems) {
  linear_fwd_sk_body<T, D, NW, PF, FULL, FAC, OWN == 0 ? 0 : OWN + 2>(problems.p[blockIdx.y], nullptr);
}

// The forward with a control wave that brings the operands in: see RAW = 5 above.
template <class T, int D, int NW, int PF, bool CKPT>
__global__ void __launch_bounds__(64 * (NW + 1)) ttt_linear_fwd_dma_kernel(Problems<LinearFwdArgs> problems) {
  linear_fwd_sk_body<T, D, NW, PF, true, false, 5, false, false, false, CKPT>(problems.p[blockIdx.y], nullptr);
}

// TTT-Linear with the Adam inner optimiser: see ADAM above.  Bound by the chain of a mini-batch, and in it by the issue
// of the optimiser's step (eight instructions per element of the state, two of them transcendental at a quarter of the
// rate) and by fetching instructions.  Hence one wave per feature tile where a unit has a CU to itself, rows loaded by
// their owners and shared through LDS (bf16) or copied in by a control wave (f32), and the loop without its branch-free
// copies where a body is long (COMPACT: 207 us instead of 161).  OCC: waves per SIMD that the register allocation
// allows; with one, the two waves of a second workgroup on a CU land on the other two SIMDs (d = 32, 384 units: 174 us
// with two, 114 with one).  2048 tokens, d = 64, bf16: 96 units 260 -> 162 us, 384 units 263 -> 231; f32: 96 units 534 ->
// 285, 384 units 545 -> 538.
template <class T, int D, int NW, int PF, bool FULL, int RAW, bool COMPACT, int OCC>
__global__ void __launch_bounds__(64 * (NW + (RAW == 5))) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) ttt_linear_adam_fwd_kernel(LinearFwdArgs a, AdamArgs ad) {
  linear_fwd_sk_body<T, D, NW, PF, FULL, false, RAW, true, false, COMPACT>(a, nullptr, &ad);
}

// The same forward on the projections as they leave the GEMMs: see RAW above.
template <class T, int D, int NW, int PF, bool FULL, bool FAC, int RAW>
__global__ void __launch_bounds__(64 * NW) ttt_linear_fwd_fi_kernel(LinearFwdArgs a, FusedInputsArgs fi) {
  static_assert(RAW == 1 || RAW == 2, "RAW selects how positions are looked up");
  linear_fwd_sk_body<T, D, NW, PF, FULL, FAC, RAW>(a, &fi);
}

// The states between two sparse checkpoints, for a backward that was given a checkpoint every ci mini-batches only: a
// workgroup takes one segment (the mini-batches from one checkpoint to the next) and writes the state entering each of
// them as a packed checkpoint, which the dense-checkpoint backward kernels then read.  Segments are independent, so the
// launch has units x segments workgroups where the reverse scan has one or two per unit: at 96 units and 8 segments of 16
// mini-batches (d = 64, f32) the 12 288 states take 90 us, bound by the chain of 15 dependent mini-batches and by writing
// 200 MB.  Same arithmetic as the forward that wrote the checkpoints.
struct LinearSegments {
  const float* W_in;  // [units, n_in, d, d]: the sparse checkpoints
  const float* b_in;  // [units, n_in, d]
  int n_in, first;    // checkpoints per unit; the first segment of this launch
  int n_seg, every;   // segments per unit in this launch; mini-batches of a segment
};
// a: rows, lr, ... at the first token of the launch; W_ckpt, b_ckpt [units, n_ckpt, ..] for its n_ckpt mini-batches
template <class T, int D, int NW, bool FULL>
__global__ void __launch_bounds__(64 * NW, 2) ttt_linear_states_kernel(LinearFwdArgs a, LinearSegments sg) {
  using elem = typename Io<T>::elem;
  const size_t unit = blockIdx.x / (unsigned)sg.n_seg, seg = blockIdx.x % (unsigned)sg.n_seg;
  const size_t at = seg * (size_t)sg.every, tok = at * (size_t)a.K;
  LinearFwdArgs b = a;
  b.xq = static_cast<const elem*>(a.xq) + tok * D;
  b.xk = static_cast<const elem*>(a.xk) + tok * D;
  b.xv = static_cast<const elem*>(a.xv) + tok * D;
  b.lr = static_cast<const elem*>(a.lr) + tok;
  b.W0 = sg.W_in;
  b.b0 = sg.b_in;
  b.W_ckpt = a.W_ckpt + at * (D * D);
  b.b_ckpt = a.b_ckpt + at * D;
  b.n_stages = __builtin_amdgcn_readfirstlane(min(sg.every, a.n_ckpt - (int)at) - 1);  // (the division leaves it in a vector register)
  linear_fwd_sk_body<T, D, NW, 2, FULL, false, 0, false, true>(b, nullptr, nullptr, unit,
                                                               unit * (size_t)sg.n_in + sg.first + seg);
}

}  // namespace ttt
