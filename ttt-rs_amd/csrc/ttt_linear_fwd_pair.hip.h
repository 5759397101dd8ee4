// TTT-Linear forward with f32 I/O, a (batch, head) unit on two workgroups on two CUs (head_dim 32 / 64, mini-batches of 16).
//
// The f32 matrix instructions bound the kernel with one workgroup per unit (ttt_linear_fwd_dma_kernel): 68 of 32 cycles per
// wave and mini-batch at head_dim 64, 24 of them for the output, of which nothing is needed for the state.  Here a PRODUCER
// runs the recurrence alone (40 instructions) and hands G'' of every mini-batch to a CONSUMER on a second CU, which follows with
// the same updates on a state of its own and forms the output (40).  Nothing flows back: the producer waits for nobody.
//
// G'' of a mini-batch [16 x d] is as large as that mini-batch's rows of `out`, which nobody reads before the consumer writes
// them: it is handed over there, in register layout, so there is no ring to run full.  One word per unit, in W_out, says how many
// mini-batches have been handed over; the consumer writes the final state over it at the end.  The producer's stores stay in the
// L2 that both share (the consumer publishes its XCD number) or are written back by a device-scope release while that is not
// known; the consumer loads at device scope.  The consumer's wait is bounded: if it was in vain it runs to its end without
// waiting and marks the unit in W_out, and a launch of the one-workgroup form behind the pair's does the marked units
// again, from inputs that no output overlaps (the caller's rule).
//
// Beside its NW = d / 16 compute waves a workgroup has two that only move data, so that the compute waves issue no global load and,
// in the producer, no store but checkpoints: one copies rows global -> LDS (as in ttt_linear_fwd_dma_kernel), the
// COURIER stores G'' and the word, or watches the word and copies G'' global -> LDS.  One barrier per mini-batch.
//
// A sequence may end in a short mini-batch (REST), which is then the last one of both workgroups instead of a launch of its own:
// the lanes without a token have rows of zeros and a learning rate of zero, and the state in front of it is what two launches would hand
// over (StateBetween, 1.3 us of the call).  63 mini-batches and five tokens, 24 units, head_dim 64, with a launch of its own 89.6 us, in
// this one 83.3.
//
// The arithmetic is that of one workgroup, and with a short mini-batch that of two launches, bit for bit.
#pragma once
#include "ttt_linear_fwd_sk.hip.h"

namespace ttt {

struct LinearPairArgs {
  unsigned spin_limit;  // polls before the consumer gives up
  int lose_at;          // the mini-batch from which on it does not wait at all (tests of that path), or INT_MAX
  int agent_release;    // 1: always publish with a device-scope release
  int rest;             // REST: tokens of the short mini-batch behind the a.n_stages whole ones, 1 .. 15
};
// words of the last 64 floats of a unit's W_out, and the mark in its first (a final state that comes to have these bits by
// itself costs a computation, not the result)
constexpr int kLinPairWords = 64, kLinPairCount = 0, kLinPairXcd = 32;
constexpr unsigned kLinPairLost = 0x7fc60b5fu;

template <int D, bool REST>
struct LinearPairLds {
  static constexpr int NT = D / 16, RS = 4;
  f32x4 rows[RS][2][NT][64];  // producer: xk, xv; consumer: xq, xk.  Four features of a token each, see `at_row`
  f32x4 g[RS][NT][64];        // G'' with tokens along k: on its way out (two slots) or in
  f32x4 at[2][NT][64];        // consumer: a wave's share of the attention block
  float lr[RS][64];
  __attribute__((aligned(16))) float ex[2][8 * 16 * NT];
  __attribute__((aligned(16))) float m0s[D + 4];
  std::conditional_t<REST, StateBetween<D, NT, 1>, NoStateBetween> between;
  int lost;
};

template <int D, bool PRODUCER, bool CKPT, bool REST>
__device__ __forceinline__ void linear_fwd_pair_body(const LinearFwdArgs& a, const LinearPairArgs& pa, LinearPairLds<D, REST>& L, size_t bh) {
  using IO = Io<F32>;
  constexpr int NT = D / 16, NW = NT, RS = LinearPairLds<D, REST>::RS;
  constexpr float inv_d = 1.0f / D;
  constexpr int K = 16;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int w = wave % NW, c = lane & 15, g = lane >> 4;  // (the two other waves do what a compute wave does up to where they branch off)
  const int h = (int)(bh % a.H), n = a.n_stages + (REST ? 1 : 0);
  const UnitBase<F32, D> ub(a, bh);
  unsigned* const words = reinterpret_cast<unsigned*>(a.W_out + bh * D * D + (D * D - kLinPairWords));
  // where G'' of a mini-batch crosses: its rows of `out`; a short one has fewer rows than G'', which goes into W_out, behind the
  // mark (a producer may write it when a consumer that waited in vain has set the mark)
  const auto crossing = [&](int st) {
    return REST && st == n - 1 ? reinterpret_cast<unsigned char*>(a.W_out + bh * D * D + kLinPairWords)
                               : ub.out + (unsigned)st * (unsigned)(K * D * 4);
  };
  static_assert(kLinPairWords + 16 * D <= D * D - kLinPairWords, "G'' lies between the mark and the words");

  if (wave >= NW) {
    float sum_a;
    f32x4 Wn[NT][1], bn[1];
    const auto centre = [&]() { centre_state<D, NW, 1, false>(Wn, bn, a.b0, L.m0s, a.gamma, sum_a, &L.ex[0][0], w, c, g); };
    if (wave == NW) {  // rows: mini-batch st + RS behind the barrier of mini-batch st
      constexpr int kCopies = 2 * NT + (PRODUCER ? 1 : 0);
      const unsigned rows0 = lds_addr(&L.rows[0][0][0][0]), lr0 = lds_addr(&L.lr[0][0]);
      const auto copy_in = [&](int stage) {  // (past the end: the last one again, into a slot nobody reads)
        const unsigned slot = (unsigned)(stage & (RS - 1)), dst = rows0 + slot * (2 * NT * 1024);
        const int st_ld = min(stage, n - 1);
        // (a short mini-batch's last token again in the lanes without one, until they are cleared below)
        const int last = REST && st_ld == n - 1 ? pa.rest - 1 : K - 1, row = min(c, last);
        const unsigned off = UnitBase<F32, D>::row_off(st_ld, K, min((c - g) & 15, last));
#pragma unroll
        for (int J = 0; J < NT; ++J) {
          const unsigned fo = (unsigned)(32 * (J >> 1) + 8 * g + 4 * (J & 1)) * 4u;  // the lane's four features of tile J
          lds_dma16(PRODUCER ? ub.xk : ub.xq, off + fo, dst + J * 1024);
          lds_dma16(PRODUCER ? ub.xv : ub.xk, off + fo, dst + (NT + J) * 1024);
        }
        if constexpr (PRODUCER) lds_dma4(ub.lr, ((unsigned)st_ld * (unsigned)K + (unsigned)row) * 4u, lr0 + slot * 256u);
      };
#pragma unroll
      for (int u = 0; u < RS; ++u) copy_in(u);
      centre();
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - 1) * kCopies) : "memory");  // mini-batch 0 has landed
      asm volatile("s_barrier" ::: "memory");
      for (int st = 0; st < n; ++st) {
        if (REST && st == n - 1) asm volatile("s_barrier" ::: "memory");           // of StateBetween
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - 2) * kCopies) : "memory");  // mini-batch st + 1 has landed
        if (REST && st == n - 2) {  // the short one: zeros in the lanes without a token
          const int sl = (n - 1) & (RS - 1);
          if (((c - g) & 15) >= pa.rest) {
#pragma unroll
            for (int i = 0; i < 2 * NT; ++i) L.rows[sl][i / NT][i % NT][lane] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
          if (PRODUCER && c >= pa.rest) L.lr[sl][lane] = 0.f;
          lds_done();
        }
        asm volatile("s_barrier" ::: "memory");
        copy_in(st + RS);
      }
      asm volatile("s_barrier" ::: "memory");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      return;
    }
    // the courier
    const auto look = [&](const unsigned* p) {
      return (unsigned)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    };
    unsigned xcd;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcd));
    xcd = 0x100u | (xcd & 15u);
    const unsigned lane16 = (unsigned)lane * 16u;
    if constexpr (PRODUCER) {
      bool fast = false;  // the consumer is known to sit behind the same L2
      const auto hand_over = [&](int st) {
#pragma unroll
        for (int J = 0; J < NT; ++J)
          *reinterpret_cast<f32x4*>(crossing(st) + J * 1024 + lane16) = L.g[st & 1][J][lane];
        if (!fast && pa.agent_release == 0) fast = look(words + kLinPairXcd) == xcd;
        if (!fast) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane == 0) __hip_atomic_store(words + kLinPairCount, (unsigned)(st + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      centre();
      asm volatile("s_barrier" ::: "memory");
      // G'' of mini-batch st lies in LDS behind the barrier of st + 1, until behind that of st + 2
      asm volatile("s_barrier" ::: "memory");
      for (int st = 1; st <= n; ++st) {
        asm volatile("s_barrier" ::: "memory");
        hand_over(st - 1);
        if (REST && st == n - 2) {  // StateBetween has a barrier: G'' of n - 2 need not wait for the next, nor the consumer's state
          asm volatile("s_barrier" ::: "memory");
          hand_over(st);
          ++st;
          asm volatile("s_barrier" ::: "memory");
        }
      }
    } else {
      if (lane == 0) __hip_atomic_store(words + kLinPairXcd, xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned g0 = lds_addr(&L.g[0][0][0]);
      bool lost = false;
      int known = 0, next = 0;  // mini-batches handed over; the next to copy
      centre();
      asm volatile("s_barrier" ::: "memory");
      for (int st = 0; st < n; ++st) {
        if (REST && st == n - 1) asm volatile("s_barrier" ::: "memory");  // of StateBetween
        // G'' of mini-batch st in LDS in front of the barrier of st, and of the next two if they are there: the slot of st + 2 was
        // last read behind the barrier of st - 2, which every wave left in front of that of st - 1
        if (st >= pa.lose_at) lost = true;
        if (!lost && known < n) {
          for (unsigned polls = 0;; ++polls) {
            known = (int)look(words + kLinPairCount);
            if (known > st) break;
            if (polls >= pa.spin_limit) {
              lost = true;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
        if (!lost) {
          for (; next < known && next <= st + 2; ++next) {
#pragma unroll
            for (int J = 0; J < NT; ++J)
              lds_dma16_dev(crossing(next), J * 1024u + lane16, g0 + (unsigned)(next & (RS - 1)) * (NT * 1024) + J * 1024);
          }
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        asm volatile("s_barrier" ::: "memory");
      }
      if (lane == 0) L.lost = lost ? 1 : 0;
      lds_done();
      asm volatile("s_barrier" ::: "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  // ---- compute waves: tile w of the features (the names are those of linear_fwd_sk_body)
  const float te_last = a.token_eta[K - 1];
  bool upd = te_last != 0.f;
  float sc = upd ? te_last : 1.f, rho_c = a.token_eta[c] / sc;
  const f32x4 ident = identity_frag<F32>(c, g), ones = splat_frag<F32>(1.f);
  f32x4 ones_upd = upd ? ones : IO::zero();
  unsigned upd_mask = upd ? ~0u : 0u;  // zero token_eta[K-1]: no update
  // the short mini-batch's token_eta, loaded here and taken up in front of it
  float te_rest_last = 0.f, te_rest_c = 0.f;
  if constexpr (REST) {
    const float* te = a.token_eta + a.n_stages * K;
    te_rest_last = te[pa.rest - 1];
    te_rest_c = te[min(c, pa.rest - 1)];
  }
  const auto take_rest = [&]() {
    upd = te_rest_last != 0.f;
    sc = upd ? te_rest_last : 1.f;
    rho_c = te_rest_c / sc;
    ones_upd = upd ? ones : IO::zero();
    upd_mask = upd ? ~0u : 0u;
  };
  const auto masked = [&](const f32x4& x) {
    u32x4 v = __builtin_bit_cast(u32x4, x);
    v &= upd_mask;
    return __builtin_bit_cast(f32x4, v);
  };
  const size_t sb = a.state_per_batch ? bh : (size_t)h;
  const float eps = held(a.eps);
  const int fo = own_offset<1>(w, 0, g);
  f32x4 gam, bet, a2, bT[1], Wc[NT][1];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    gam[r] = a.gamma[h * D + fo + r];
    bet[r] = a.beta[h * D + fo + r];
    bT[0][r] = a.b0[sb * D + fo + r];
    a2[r] = gam[r] * gam[r];
  }
  load_state_slice<D, 1>(Wc, a.W0 + sb * D * D, w, c, g);
  if constexpr (REST) L.between.keep(Wc, bT, w, lane);
  float sum_a;  // of gamma^2
  centre_state<D, NW, 1>(Wc, bT, a.b0 + sb * D, L.m0s, a.gamma + h * D, sum_a, &L.ex[0][0], w, c, g);
  lds_barrier();

  // Features 4 j .. of a tile of token s lie at 16 j + (s + j) mod 16: sixteen lanes that read a row's features and sixteen that read a
  // feature of four tokens (four lanes each, all four j) both meet all banks.
  const int at_row = 16 * g + ((c + g) & 15);
  // XK with tokens along k, from the rows, not by four matrix instructions in front of Z1, and a write for the other waves (24 units, 63 mini-
  // batches and five tokens 83.9 -> 82.4 us, a training step of 96 units x 2048 tokens 619 -> 617): element r is feature c of a tile of token 4 g + r
  const auto tokens_along_k = [&](f32x4 (&kd)[NT], int stage) {
    const float* const x = reinterpret_cast<const float*>(&L.rows[stage & (RS - 1)][PRODUCER ? 0 : 1][0][0]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = 4 * (16 * (c >> 2) + ((4 * g + r + (c >> 2)) & 15)) + (c & 3);
#pragma unroll
      for (int I = 0; I < NT; ++I) kd[I][r] = x[256 * I + o];
    }
  };
  // rows of a mini-batch: full rows of what is multiplied by the state, own features of the others
  f32x4 x[2][NT], xo[2], yo[2];  // producer: xk, own xk, own xv; consumer: xq, own xq, own xk
  float lr[2];
  const auto gather = [&](int u, int stage) {
    const int sl = stage & (RS - 1);
#pragma unroll
    for (int J = 0; J < NT; ++J) x[u][J] = L.rows[sl][0][J][at_row];
    xo[u] = L.rows[sl][0][w][at_row];
    yo[u] = L.rows[sl][1][w][at_row];
    if constexpr (PRODUCER) lr[u] = L.lr[sl][c];
  };
  gather(0, 0);

  // all mini-batches
  const auto run = [&](const auto& mini_batch) {
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    int st = 0;
    for (; st + 2 <= a.n_stages; st += 2) {
      mini_batch(even, st);
      mini_batch(odd, st + 1);
    }
    if (st < a.n_stages) mini_batch(even, st);
    if constexpr (REST) {
      take_rest();
      L.between.form(Wc, bT, L.m0s, w, c, g);
      lds_barrier();
      L.between.centre(Wc, bT, w, c, g);
      if (st < a.n_stages)
        mini_batch(odd, n - 1);
      else
        mini_batch(even, n - 1);
    }
  };

  if constexpr (PRODUCER) {
    CkptCursor<D> ck(a, bh);
    const float b_mean = __builtin_amdgcn_readfirstlane(L.m0s[D]);
    const auto mini_batch = [&](auto u_tag, int st) {
      constexpr int u = decltype(u_tag)::value;
      f32x4 kd[NT];
      tokens_along_k(kd, st);
      f32x4 z1 = bT[0];
#pragma unroll
      for (int J = 0; J < NT; ++J) IO::mma(z1, Wc[J][0], x[u][J]);
      const f32x4 uu = bet - (yo[u] - xo[u]);
      if (CKPT && ck.due()) {
        if (ck.packed) {
          store_ckpt_packed<F32, NT, 1>(ck.W, Wc, w, lane);
          store_bias_true<D, 1>(ck.b, bT, b_mean, w, c, g);
        } else {
          store_state_f32<D, 1>(ck.W, ck.b, Wc, bT, L.m0s, w, c, g);
        }
        ck.advance();
      }
      if constexpr (CKPT) {
        ck.next_stage();
        settle_f32(z1);
      }
      // the six moments of Z1
      float S[6];
      const f32x4 bq = gam * uu;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float az = a2[r] * z1[r];
        if (r == 0) {
          S[0] = z1[0];
          S[2] = az;
          S[3] = az * z1[0];
          S[4] = bq[0];
          S[5] = bq[0] * z1[0];
        } else {
          S[0] += z1[r];
          S[1] = r == 1 ? __builtin_fmaf(z1[0], z1[0], z1[1] * z1[1]) : __builtin_fmaf(z1[r], z1[r], S[1]);
          S[2] = __builtin_fmaf(a2[r], z1[r], S[2]);
          S[3] = __builtin_fmaf(az, z1[r], S[3]);
          S[4] = __builtin_fmaf(gam[r], uu[r], S[4]);
          S[5] = __builtin_fmaf(bq[r], z1[r], S[5]);
        }
      }
      float* const e = L.ex[u];
      const float v0 = xg_sum4_scatter(S[0], S[1], S[2], S[3]), v1 = xg_sum2_scatter(S[4], S[5]);
      e[(g * 16 + c) * NW + w] = v0;
      if ((g & 1) == 0) e[((4 + (g >> 1)) * 16 + c) * NW + w] = v1;
      lds_barrier();
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        float s = e[(i * 16 + c) * NW];
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) s += e[(i * 16 + c) * NW + ww];
        S[i] = s;
      }
      gather(u ^ 1, st + 1);
      const float mu = S[0] * inv_d;
      const float var = S[1] * inv_d - mu * mu;
      const float rstd = __builtin_amdgcn_rsqf(fmaxf(var, 0.f) + eps);
      const float s1 = rstd * (S[2] - mu * sum_a) + S[4];
      const float m = S[5] - mu * S[4], q = S[3] - 2.f * mu * S[2] + mu * mu * sum_a, r2 = rstd * rstd;
      const float s2 = __builtin_fmaf(r2, q, rstd * m);
      const float p = -sc * lr[u] * rstd;
      const float c1 = p * rstd, c2 = -c1 * s2 * inv_d, c3 = -p * s1 * inv_d;
      const f32x4 G = (z1 - mu) * (a2 * c1 + c2) + (bq * p + c3);
      f32x4 Gd = {0.f, 0.f, 0.f, 0.f};
      IO::mma(Gd, G, ident);
#pragma unroll
      for (int I = 0; I < NT; ++I) IO::mma(Wc[I][0], kd[I], masked(Gd));
      IO::mma(bT[0], Gd, ones_upd);
      L.g[u][w][lane] = Gd;
    };
    run(mini_batch);
    lds_barrier();  // the last G''
  } else {
    // pending output of the last mini-batch (its sums travel in the next exchange) and of the one before (sums known)
    f32x4 zbp = {0.f, 0.f, 0.f, 0.f}, zbo = zbp, qop = zbp, qoo = zbp;
    float so0 = 0.f, so1 = 0.f;
    const auto publish = [&](int u) {
      const float s0 = ((zbp[0] + zbp[1]) + zbp[2]) + zbp[3];
      const float s1 = __builtin_fmaf(zbp[3], zbp[3], __builtin_fmaf(zbp[2], zbp[2], __builtin_fmaf(zbp[1], zbp[1], zbp[0] * zbp[0])));
      const float v = xg_sum2_scatter(s0, s1);
      if ((g & 1) == 0) L.ex[u][((g >> 1) * 16 + c) * NW + w] = v;
    };
    const auto collect = [&](int u, float& s0, float& s1) {
      const float* e = L.ex[u];
      s0 = e[c * NW];
      s1 = e[(16 + c) * NW];
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) {
        s0 += e[c * NW + ww];
        s1 += e[(16 + c) * NW + ww];
      }
    };
    const auto emit = [&](float s0, float s1, int stage, const f32x4& zb, const f32x4& qo) {
      const float mu = s0 * inv_d;
      const float rstd = __builtin_amdgcn_rsqf(fmaxf(s1 * inv_d - mu * mu, 0.f) + eps);
      float* po = reinterpret_cast<float*>(ub.out + UnitBase<F32, D>::row_off(stage, K, c));
      const f32x4 qb = qo + bet;
      *reinterpret_cast<f32x4*>(po + fo) = qb + gam * ((zb - mu) * rstd);
    };
    const auto mini_batch = [&](auto u_tag, int st) {
      constexpr int u = decltype(u_tag)::value;
      f32x4 At = {0.f, 0.f, 0.f, 0.f}, kd[NT];
      tokens_along_k(kd, st);
      IO::mma(At, yo[u], xo[u]);
      L.at[u][w][lane] = At;
      f32x4 zb = bT[0];
#pragma unroll
      for (int J = 0; J < NT; ++J) IO::mma(zb, Wc[J][0], x[u][J]);
      publish(u);
      if (st > 1) emit(so0, so1, st - 2, zbo, qoo);
      lds_barrier();
      collect(u, so0, so1);
      At = L.at[u][0][lane];
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) At += L.at[u][ww][lane];
      const f32x4 Gd = L.g[st & (RS - 1)][w][lane];
      gather(u ^ 1, st + 1);
      zbo = zbp;
      qoo = qop;
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = (4 * g + r <= c) ? rho_c * (1.f + At[r]) : 0.f;
#pragma unroll
      for (int I = 0; I < NT; ++I) IO::mma(Wc[I][0], kd[I], masked(Gd));
      IO::mma(bT[0], Gd, ones_upd);
      IO::mma(zb, Gd, m);
      zbp = zb;
      qop = xo[u];
    };
    run(mini_batch);
    f32x4 W0[NT][1];
    if constexpr (!REST) load_state_slice<D, 1>(W0, a.W0 + sb * D * D, w, c, g);
    publish(n & 1);
    lds_barrier();
    float s0, s1;
    collect(n & 1, s0, s1);
    if (n >= 2) emit(so0, so1, n - 2, zbo, qoo);
    if (!REST || c < pa.rest) emit(s0, s1, n - 1, zbp, qop);
    if constexpr (REST) {
      L.between.weights(W0, w, lane);
      store_state_final<D, 1>(a.W_out + bh * D * D, a.b_out + bh * D, W0, L.between.b, Wc, bT, L.between.m0s, w, c, g);
    } else {
      store_state_final<D, 1>(a.W_out + bh * D * D, a.b_out + bh * D, W0, a.b0 + sb * D, Wc, bT, L.m0s, w, c, g);
    }
    // element (0, 0) of W_out is written by the lane that marks the unit
    if (L.lost != 0 && threadIdx.x == 0) *reinterpret_cast<unsigned*>(a.W_out + bh * D * D) = kLinPairLost;
  }
}

// Workgroups b and b + 8 of every 16 share a unit: consecutive workgroups go to the XCDs in turn, so both run behind one L2, and
// the producer, which waits for nobody, is dispatched first.
template <int D, bool CKPT, bool REST>
__global__ void __launch_bounds__(64 * (D / 16 + 2)) ttt_linear_fwd_pair_kernel(LinearFwdArgs a, LinearPairArgs pa) {
  __shared__ LinearPairLds<D, REST> L;
  const size_t bh = (size_t)(blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
  if (bh >= (size_t)a.B * a.H) return;
  if (((blockIdx.x >> 3) & 1) == 0)
    linear_fwd_pair_body<D, true, CKPT, REST>(a, pa, L, bh);
  else
    linear_fwd_pair_body<D, false, false, REST>(a, pa, L, bh);
}

// the word of every unit, and the consumer's XCD number
template <int D>
__global__ void ttt_linear_fwd_pair_clear_kernel(float* W_out, int units) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < units) {
    float* words = W_out + (size_t)i * D * D + (D * D - kLinPairWords);
    words[kLinPairCount] = words[kLinPairXcd] = 0.f;
  }
}

// the units whose consumer waited in vain, on one workgroup
template <int D, bool CKPT>
__global__ void __launch_bounds__(64 * (D / 16 + 1)) ttt_linear_fwd_redo_kernel(LinearFwdArgs a) {
  const unsigned* mark = reinterpret_cast<const unsigned*>(a.W_out + blockIdx.x * (size_t)(D * D));
  if (__builtin_amdgcn_readfirstlane((int)*mark) != (int)kLinPairLost) return;
  linear_fwd_sk_body<F32, D, D / 16, 2, true, false, 5, false, false, false, CKPT>(a, nullptr);
}

// the same where a short mini-batch of `rest` tokens follows: as two calls would, without the wave that copies rows
template <int D>
__global__ void __launch_bounds__(64 * (D / 16)) ttt_linear_fwd_redo_rest_kernel(LinearFwdArgs a, int rest) {
  const unsigned* mark = reinterpret_cast<const unsigned*>(a.W_out + blockIdx.x * (size_t)(D * D));
  if (__builtin_amdgcn_readfirstlane((int)*mark) != (int)kLinPairLost) return;
  linear_fwd_sk_body<F32, D, D / 16, 2, true, false, 0, false, false, false, false>(a, nullptr);
  __threadfence();  // the state in between goes from wave to wave through memory
  __syncthreads();
  const size_t at = (size_t)a.n_stages * a.K, row = at * (D * 4);
  a.xq = static_cast<const unsigned char*>(a.xq) + row;
  a.xk = static_cast<const unsigned char*>(a.xk) + row;
  a.xv = static_cast<const unsigned char*>(a.xv) + row;
  a.lr = static_cast<const unsigned char*>(a.lr) + at * 4;
  a.out = static_cast<unsigned char*>(a.out) + row;
  a.token_eta += at;
  a.W0 = a.W_out;
  a.b0 = a.b_out;
  a.state_per_batch = 1;
  a.seq = a.K = rest;
  a.n_stages = 1;
  linear_fwd_sk_body<F32, D, D / 16, 2, false, false, 0, false, false, false, false>(a, nullptr);
}

hipError_t launch_linear_fwd_pair(int head_dim, const LinearFwdArgs& a, const LinearPairArgs& pa, hipStream_t s);  // ttt_linear_fwd_pair.hip

}  // namespace ttt
