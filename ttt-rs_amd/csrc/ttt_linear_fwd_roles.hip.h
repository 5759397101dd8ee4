// TTT-Linear forward with bf16 I/O, the waves of a (batch, head) unit in roles on one CU (head_dim 32 / 64, mini-batches of 16).
//
// With two waves per unit (ttt_linear_fwd_sk_kernel) each wave issues the recurrence, the output and the loads of its features, and is
// bound by what it issues, while two of the CU's four SIMDs have nothing to do.  Here two CHAIN waves run the recurrence alone
// and leave G'' of every mini-batch in LDS; two OUTPUT waves follow two mini-batches behind with the same updates on a state
// of their own, form the output and save states or factors; a COPY wave brings the rows in, global -> LDS, without passing
// registers.  One barrier per mini-batch, which the recurrence has anyway.  The output waves come first, so that the copy wave shares a
// SIMD with one of them.  Bound by the chain waves: 0.62 us per mini-batch at head_dim 64 (counted over chain and output waves, 34 % of their
// time is waiting, 45 % vector issue).
//
// 128 mini-batches, us with two waves / in roles: head_dim 64, 12 units 110.0 / 77.9, 64 111.2 / 78.8, 256 113.0 / 80.7, saving
// update factors 116.5 / 81.5; head_dim 32, 12 units 71.6 / 52.6, 256 72.8 / 54.0.  One mini-batch, head_dim 64, 12 units 6.9 / 6.1.
// Rows brought in by the output waves instead: 82.7 and 58.1 at 256 units, a mini-batch 7.7.
//
// TWO: two units per CU (head_dim 32).  Wave i of a workgroup goes to SIMD i mod 4, so the second half of the workgroups has the roles the
// other way round: a chain wave shares its SIMD with an output wave and has priority.  384 units 94.9 / 64.8.  At head_dim 64 a wave needs
// more registers than five waves of two workgroups leave it (two rounds, 164 us), and without the copy wave it is even with two
// waves per unit: 272 units 113.1 / 107.3, 384 113.8 / 114.0, 512 121.0 / 130.2.
//
// FORM: head split, rotary embedding and lr gate go to a second copy wave, which forms the operands of the next mini-batch in LDS, in
// place; in the two-wave kernel (RAW = 1) they are instructions of the waves that carry the recurrence.  128 mini-batches, head_dim 64, 12
// units 135.0 -> 78.1 us, 256 138.6 -> 81.6; head_dim 32, 256 units 97.1 -> 53.7, 384 126.8 -> 73.3.
//
// REST: a short mini-batch behind the whole ones is the last one, as in ttt_linear_fwd_pair.hip.h; the chain waves form the state in
// front of it (StateBetween) and the output waves take it over.  24 units, five tokens behind four mini-batches, two launches with two
// waves / one in roles: head_dim 64 16.0 / 10.1 us, 32 11.1 / 6.4; behind 63 63.8 / 44.4 and 42.4 / 29.3.
//
// The arithmetic is that of ttt_linear_fwd_sk_kernel, and with a short mini-batch that of two launches of it, bit for bit.
#pragma once
#include "ttt_linear_fwd_sk.hip.h"

namespace ttt {

template <int D, bool REST = false>
struct LinearRolesLds {
  static constexpr int NT = D / 16, NW = 2, TPW = NT / NW, RS = 8;
  u32x4 rows[RS][3][NT / 2][64];  // xq, xk, xv: lane (c, g) the features 32 q + 8 g .. + 7 of token c
  unsigned lr[RS][64];
  u32x2 g[2][NT][64];             // G'' with tokens along k
  __attribute__((aligned(16))) float ex[2][6 * 16 * NW];
  __attribute__((aligned(16))) float ez[2][2 * 16 * NW];
  __attribute__((aligned(16))) float m0s[D + 4];
  std::conditional_t<REST, StateBetweenShared<D, NW, TPW>, NoStateBetween> between;
};

// SAVE 0: nothing.  1: states.  2: update factors.
// FORM: the operands are formed from the projections (FusedInputsArgs, no copies of them asked for, positions that repeat with the
// mini-batch), by a second copy wave.
template <int D, int SAVE, bool TWO, bool REST, bool FORM = false>
__device__ __forceinline__ void linear_fwd_roles_body(const LinearFwdArgs& a, LinearRolesLds<D, REST>& L, bool flip, int rest,
                                                      const FusedInputsArgs* fi = nullptr) {
  using IO = Io<BF16>;
  using frag = IO::frag;
  using LD = LinearRolesLds<D, REST>;
  constexpr int NT = D / 16, NW = LD::NW, TPW = LD::TPW, RS = LD::RS, K = 16;
  constexpr float inv_d = 1.0f / D;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int w = wave % NW, c = lane & 15, g = lane >> 4;
  const size_t bh = blockIdx.x;
  const int h = (int)(bh % a.H), whole = held(a.n_stages), n = whole + (REST ? 1 : 0);
  const UnitBase<BF16, D> ub(a, bh);
  float* const scratch = reinterpret_cast<float*>(&L.g[0][0][0]);
  static_assert(sizeof(L.g) >= (NW + 2) * D * sizeof(float), "scratch of centre_state");
  static_assert(64 * NW >= D, "centre_state's sums are the first NW waves'");
  float sum_a;  // of gamma^2

  if (FORM && wave == 2 * NW + 1) {  // xq, xk and the learning rates of mini-batch st + 1 between the barriers of st - 1 and st, in place
    const size_t pos = fi->cos != nullptr ? (size_t)((fi->pos_offset + c) % fi->pos_wrap) * (D / 2) + 4 * g : 0;
    f32x4 cs[NT / 2], sn[NT / 2];
#pragma unroll
    for (int q = 0; q < NT / 2; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        cs[q][i] = fi->cos != nullptr ? fi->cos[pos + 16 * q + i] : 1.f;
        sn[q][i] = fi->cos != nullptr ? fi->sin[pos + 16 * q + i] : 0.f;
      }
    const float bias = fi->lr_bias[h], scale = fi->lr_scale;
    const auto form = [&](int stage) {
      const int sl = stage & (RS - 1);
#pragma unroll
      for (int what = 0; what < 2; ++what)
#pragma unroll
        for (int q = 0; q < NT / 2; ++q) {
          const u32x4 v = L.rows[sl][what][q][lane];
          const f32x4 lo = IO::to_f32(__builtin_bit_cast(frag, u32x2{v[0], v[1]})), hi = IO::to_f32(__builtin_bit_cast(frag, u32x2{v[2], v[3]}));
          const u32x2 x = __builtin_bit_cast(u32x2, IO::to_frag(rope_rotate4(lo, f32x2{cs[q][0], cs[q][1]}, f32x2{sn[q][0], sn[q][1]})));
          const u32x2 y = __builtin_bit_cast(u32x2, IO::to_frag(rope_rotate4(hi, f32x2{cs[q][2], cs[q][3]}, f32x2{sn[q][2], sn[q][3]})));
          L.rows[sl][what][q][lane] = u32x4{x[0], x[1], y[0], y[1]};
        }
      const float z = __uint_as_float(L.lr[sl][lane] << 16);
      L.lr[sl][lane] = __float_as_uint(IO::rounded(lr_gate(z + bias, scale))) >> 16;
    };
    f32x4 Wn[NT][TPW], bn[TPW];
    centre_state<D, NW, TPW, false>(Wn, bn, a.b0, L.m0s, a.gamma, sum_a, scratch, w, c, g);
    asm volatile("s_barrier" ::: "memory");
    form(0);
    lds_barrier();
    for (int st = 0; st < n; ++st) {
      form(st + 1);
      lds_barrier();
    }
    asm volatile("s_barrier\n\ts_barrier" ::: "memory");
    return;
  }
  if (wave == 2 * NW) {  // rows: mini-batch st + RS - 2 behind the barrier of mini-batch st
    constexpr int kCopies = 3 * (NT / 2) + 1;
    // (FORM: token t of the unit is row (b seq + t) H + h of the [B,seq,H,d] projections and of the [B,seq,H] logits)
    const size_t row0 = FORM ? bh / a.H * (size_t)a.seq * a.H + h : 0;
    const unsigned char* const xq = FORM ? static_cast<const unsigned char*>(fi->xq) + row0 * (D * 2) : ub.xq;
    const unsigned char* const xk = FORM ? static_cast<const unsigned char*>(fi->xk) + row0 * (D * 2) : ub.xk;
    const unsigned char* const xv = FORM ? static_cast<const unsigned char*>(fi->xv) + row0 * (D * 2) : ub.xv;
    const unsigned char* const lr = FORM ? static_cast<const unsigned char*>(fi->lr_logits) + row0 * 2 : ub.lr;
    const unsigned pitch = FORM ? (unsigned)a.H : 1u;
    const unsigned rows0 = lds_addr(&L.rows[0][0][0][0]), lr0 = lds_addr(&L.lr[0][0]);
    const auto copy_in = [&](int stage) {  // (past the end: the last one again, into a slot nobody reads)
      const unsigned slot = (unsigned)(stage & (RS - 1)), dst = rows0 + slot * (3 * (NT / 2) * 1024);
      const int st_ld = min(stage, n - 1);
      // (a short mini-batch's last token again in the lanes without one, until they are cleared below)
      const int row = REST && st_ld == n - 1 ? min(c, rest - 1) : c;
      const unsigned t = ((unsigned)st_ld * (unsigned)K + (unsigned)row) * pitch, off = t * (D * 2u) + 16u * (unsigned)g;
#pragma unroll
      for (int q = 0; q < NT / 2; ++q) {
        lds_dma16(xk, off + 64u * q, dst + (1 * (NT / 2) + q) * 1024);
        lds_dma16(xv, off + 64u * q, dst + (2 * (NT / 2) + q) * 1024);
        lds_dma16(xq, off + 64u * q, dst + (0 * (NT / 2) + q) * 1024);
      }
      lds_dma2(lr, t * 2u, lr0 + slot * 256u);
    };
#pragma unroll
    for (int u = 0; u < RS - 2; ++u) copy_in(u);
    f32x4 Wn[NT][TPW], bn[TPW];
    centre_state<D, NW, TPW, false>(Wn, bn, a.b0, L.m0s, a.gamma, sum_a, scratch, w, c, g);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - (FORM ? 4 : 3)) * kCopies) : "memory");  // mini-batch 0 has landed (FORM: and 1)
    asm volatile("s_barrier" ::: "memory");
    if constexpr (FORM) asm volatile("s_barrier" ::: "memory");
    for (int st = 0; st < n; ++st) {
      if (REST && st == n - 1) asm volatile("s_barrier" ::: "memory");  // of StateBetween
      // mini-batch st + 1 has landed (FORM: st + 2); the slot of mini-batch st - 2 was last read in front of this barrier, by the output waves
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - (FORM ? 5 : 4)) * kCopies) : "memory");
      if (REST && st == n - 2) {  // the short one: zeros in the lanes without a token
        const int sl = (n - 1) & (RS - 1);
        if (c >= rest) {
#pragma unroll
          for (int i = 0; i < 3 * (NT / 2); ++i) L.rows[sl][i / (NT / 2)][i % (NT / 2)][lane] = u32x4{0u, 0u, 0u, 0u};
          L.lr[sl][lane] = 0u;
        }
        lds_done();
      }
      asm volatile("s_barrier" ::: "memory");
      copy_in(st + RS - 2);
    }
    asm volatile("s_barrier\n\ts_barrier" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  const auto tok_eta = [&](int i) {
    if constexpr (FORM) return fmaxf(fi->token_idx[i] + fi->learnable_token_idx[i], 0.f);
    else return a.token_eta[i];
  };
  const float te_last = tok_eta(K - 1);
  bool upd = te_last != 0.f;
  float sc = upd ? te_last : 1.f, rho_c = tok_eta(c) / sc;
  const frag ident = identity_frag<BF16>(c, g), nident = identity_frag<BF16>(c, g, -1.f), ones = splat_frag<BF16>(1.f);
  frag ones_upd = upd ? ones : IO::zero();
  unsigned upd_mask = upd ? ~0u : 0u;
  // the short mini-batch's token_eta, loaded here and taken up in front of it
  float te_rest_last = 0.f, te_rest_c = 0.f;
  if constexpr (REST) {
    const float* te = a.token_eta + whole * K;
    te_rest_last = te[rest - 1];
    te_rest_c = te[min(c, rest - 1)];
  }
  const auto take_rest = [&]() {
    upd = te_rest_last != 0.f;
    sc = upd ? te_rest_last : 1.f;
    rho_c = te_rest_c / sc;
    ones_upd = upd ? ones : IO::zero();
    upd_mask = upd ? ~0u : 0u;
  };
  const size_t sb = a.state_per_batch ? bh : (size_t)h;
  const float eps = held(a.eps);
  f32x4 gam[TPW], bet[TPW], a2[TPW], bT[TPW], Wc[NT][TPW];
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
  load_state_slice<D, TPW>(Wc, a.W0 + sb * D * D, w, c, g);
  if constexpr (REST) L.between.keep(Wc, bT, w, lane);
  centre_state<D, NW, TPW>(Wc, bT, a.b0 + sb * D, L.m0s, a.gamma + h * D, sum_a, scratch, w, c, g);
  lds_barrier();
  if constexpr (FORM) lds_barrier();

  const auto full_rows = [&](frag (&x)[NT], int sl, int what) {
#pragma unroll
    for (int q = 0; q < NT / 2; ++q) {
      const u32x4 v = L.rows[sl][what][q][lane];
      x[2 * q] = __builtin_bit_cast(frag, u32x2{v[0], v[1]});
      x[2 * q + 1] = __builtin_bit_cast(frag, u32x2{v[2], v[3]});
    }
  };
  const auto own_rows = [&](frag (&x)[TPW], int sl, int what) {
    if constexpr (TPW == 1) {
      x[0] = __builtin_bit_cast(frag, reinterpret_cast<const u32x2*>(&L.rows[sl][what][w >> 1][lane])[w & 1]);
    } else {
#pragma unroll
      for (int qq = 0; qq < TPW / 2; ++qq) {
        const u32x4 v = L.rows[sl][what][w * (TPW / 2) + qq][lane];
        x[2 * qq] = __builtin_bit_cast(frag, u32x2{v[0], v[1]});
        x[2 * qq + 1] = __builtin_bit_cast(frag, u32x2{v[2], v[3]});
      }
    }
  };
  const auto tokens_along_k = [&](frag (&kd)[NT], int sl) {
    const u32x4* const xk = &L.rows[sl][1][0][0] + tr_lane(lane);
#pragma unroll
    for (int I = 0; I < NT; ++I) kd[I] = read_tr(reinterpret_cast<const unsigned char*>(xk + (I >> 1) * 64) + 8 * (I & 1));
  };
  // W += XK^T G'', b += colsum G'' (zero token_eta[K-1]: nothing), see linear_fwd_sk_body
  const auto update = [&](const frag (&kd)[NT], const frag (&Gd)[TPW]) {
    frag Gu[TPW];
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) {
      const u32x2 v = __builtin_bit_cast(u32x2, Gd[jj]);
      Gu[jj] = __builtin_bit_cast(frag, u32x2{v[0] & upd_mask, v[1] & upd_mask});
    }
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) IO::mma(Wc[I][jj], kd[I], Gu[jj]);
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) IO::mma(bT[jj], Gd[jj], ones_upd);
    if constexpr (TPW == 1) asm volatile("s_nop 4" : "+v"(bT[0]));
    else asm volatile("s_nop 4" : "+v"(bT[0]), "+v"(bT[1]));
  };

  if ((wave >= NW) != (TWO && flip)) {  // ---- the recurrence
    if constexpr (TWO) __builtin_amdgcn_s_setprio(2);
    frag k[NT], ko[TPW], vo[TPW];  // of the next mini-batch from the barrier on
    float lr_next;
    const auto gather = [&](int stage) {
      const int sl = stage & (RS - 1);
      full_rows(k, sl, 1);
      own_rows(ko, sl, 1);
      own_rows(vo, sl, 2);
      lr_next = __uint_as_float(L.lr[sl][c] << 16);
    };
    const auto mini_batch = [&](auto u_tag, int st) {
      constexpr int u = decltype(u_tag)::value;
      frag kd[NT];
      tokens_along_k(kd, st & (RS - 1));
      f32x4 z1[TPW], uu[TPW], bq[TPW];
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) z1[jj] = bT[jj];
#pragma unroll
      for (int q = 0; q < NT / 2; ++q)
#pragma unroll
        for (int jj = 0; jj < TPW; ++jj)
          IO::mma2(z1[jj], IO::to_frag(Wc[2 * q][jj]), IO::to_frag(Wc[2 * q + 1][jj]), k[2 * q], k[2 * q + 1]);
      float S[6], z_first = 0.f;
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        uu[jj] = bet[jj];
        IO::mma2(uu[jj], nident, ident, vo[jj], ko[jj]);
        bq[jj] = gam[jj] * uu[jj];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float z = z1[jj][r], az = a2[jj][r] * z;
          if (jj == 0 && r == 0) {
            z_first = z;
            S[0] = z;
            S[2] = az;
            S[3] = az * z;
            S[4] = bq[jj][r];
            S[5] = bq[jj][r] * z;
          } else {
            S[0] += z;
            S[1] = jj == 0 && r == 1 ? __builtin_fmaf(z_first, z_first, z * z) : __builtin_fmaf(z, z, S[1]);
            S[2] = __builtin_fmaf(a2[jj][r], z, S[2]);
            S[3] = __builtin_fmaf(az, z, S[3]);
            S[4] = __builtin_fmaf(gam[jj][r], uu[jj][r], S[4]);
            S[5] = __builtin_fmaf(bq[jj][r], z, S[5]);
          }
        }
      }
      float* const e = L.ex[u];
      const float v0 = xg_sum4_scatter(S[0], S[1], S[2], S[3]), v1 = xg_sum2_scatter(S[4], S[5]);
      e[(g * 16 + c) * NW + w] = v0;
      if ((g & 1) == 0) e[((4 + (g >> 1)) * 16 + c) * NW + w] = v1;
      lds_barrier();
#pragma unroll
      for (int i = 0; i < 6; ++i) S[i] = e[(i * 16 + c) * NW] + e[(i * 16 + c) * NW + 1];
      const float lr = lr_next;
      gather(st + 1);
      const float mu = S[0] * inv_d;
      const float var = S[1] * inv_d - mu * mu;
      const float rstd = __builtin_amdgcn_rsqf(fmaxf(var, 0.f) + eps);
      const float s1 = rstd * (S[2] - mu * sum_a) + S[4];
      const float m = S[5] - mu * S[4], q = S[3] - 2.f * mu * S[2] + mu * mu * sum_a, r2 = rstd * rstd;
      const float s2 = __builtin_fmaf(r2, q, rstd * m);
      const float p = -sc * lr * rstd;
      const float c1 = p * rstd, c2 = -c1 * s2 * inv_d, c3 = -p * s1 * inv_d;
      frag Gd[TPW];
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) {
        const f32x4 G = (z1[jj] - mu) * (a2[jj] * c1 + c2) + (bq[jj] * p + c3);
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
        IO::mma(t, IO::to_frag(G), ident);
        Gd[jj] = IO::to_frag(t);
      }
      update(kd, Gd);
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) L.g[u][w * TPW + jj][lane] = __builtin_bit_cast(u32x2, Gd[jj]);
    };
    gather(0);
    int st = 0;
    for (; st + 2 <= whole; st += 2) {
      mini_batch(std::integral_constant<int, 0>{}, st);
      mini_batch(std::integral_constant<int, 1>{}, st + 1);
    }
    if (st < whole) mini_batch(std::integral_constant<int, 0>{}, st);
    if constexpr (REST) {
      take_rest();
      L.between.form(Wc, bT, L.m0s, w, c, g);
      lds_barrier();
      L.between.centre(Wc, bT, w, c, g);
      L.between.give(Wc, bT, w, lane);
      if (st < whole)
        mini_batch(std::integral_constant<int, 1>{}, whole);
      else
        mini_batch(std::integral_constant<int, 0>{}, whole);
    }
    lds_barrier();
    f32x4 W0[NT][TPW];
    if constexpr (!REST) load_state_slice<D, TPW>(W0, a.W0 + sb * D * D, w, c, g);
    lds_barrier();
    if constexpr (REST) {
      int c_end = c, g_end = g;  // (or the addresses, formed from the same lane indices as the prologue's, are kept: 16 spilled registers)
      asm volatile("" : "+v"(c_end), "+v"(g_end));
      L.between.weights(W0, w, lane);
      store_state_final<D, TPW>(a.W_out + bh * D * D, a.b_out + bh * D, W0, L.between.b, Wc, bT, L.between.m0s, w, c_end, g_end);
    } else {
      store_state_final<D, TPW>(a.W_out + bh * D * D, a.b_out + bh * D, W0, a.b0 + sb * D, Wc, bT, L.m0s, w, c, g);
    }
    if constexpr (SAVE == 2)
      store_state_tiles<D, TPW>(a.W_ckpt + bh * (size_t)a.n_ckpt * (D * D), a.b_ckpt + bh * (size_t)a.n_ckpt * D, Wc, bT, w, lane);
    return;
  }

  // ---- the output: mini-batch m behind the barrier of m + 1
  CkptCursor<D> ck(a, bh);
  const float b_mean = __builtin_amdgcn_readfirstlane(L.m0s[D]);
  unsigned char* fac = SAVE == 2 ? factor_base<D>(a.W_ckpt, a.n_ckpt, bh) : nullptr;
  f32x4 zb[TPW];
  frag qo[TPW];
  const auto emit = [&](int m) {  // out = xq + gamma (zbar - mu) rstd + beta
    const float* const e = L.ez[m & 1];
    const float s0 = e[c * NW] + e[c * NW + 1], s1 = e[(16 + c) * NW] + e[(16 + c) * NW + 1];
    const float mu = s0 * inv_d;
    const float rstd = __builtin_amdgcn_rsqf(fmaxf(s1 * inv_d - mu * mu, 0.f) + eps);
    uint16_t* const po = reinterpret_cast<uint16_t*>(ub.out + UnitBase<BF16, D>::row_off(m, K, c));
    f32x4 o[TPW];
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) {
      f32x4 qb = bet[jj];
      IO::mma(qb, ident, qo[jj]);
      o[jj] = qb + gam[jj] * ((zb[jj] - mu) * rstd);
    }
    if constexpr (TPW == 1) {
      store4<BF16>(po + own_offset<TPW>(w, 0, g), o[0]);
    } else {
#pragma unroll
      for (int qq = 0; qq < TPW / 2; ++qq) IO::store8(po + own_offset<TPW>(w, 2 * qq, g), o[2 * qq], o[2 * qq + 1]);
    }
  };
  lds_barrier();
  lds_barrier();
  for (int m = 0; m < n; ++m) {
    const int sl = m & (RS - 1);
    if (m > 0) emit(m - 1);
    if constexpr (REST) {
      if (m == whole) {  // the recurrence left its state two barriers ago
        take_rest();
        L.between.take(Wc, bT, w, lane);
      }
    }
    frag q[NT], k[NT], kd[NT], Gd[TPW];
    full_rows(q, sl, 0);
    full_rows(k, sl, 1);
    own_rows(qo, sl, 0);
    tokens_along_k(kd, sl);
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) Gd[jj] = __builtin_bit_cast(frag, L.g[m & 1][w * TPW + jj][lane]);
    if constexpr (SAVE == 1) {
      if (ck.due()) {
        if (ck.packed) {
          store_ckpt_packed<BF16, NT, TPW>(ck.W, Wc, w, lane);
          store_bias_true<D, TPW>(ck.b, bT, b_mean, w, c, g);
        } else {
          store_state_f32<D, TPW>(ck.W, ck.b, Wc, bT, L.m0s, w, c, g);
        }
        ck.advance();
      }
      ck.next_stage();
    }
    if constexpr (SAVE == 2) {
      store_factor<TPW>(fac, Gd, w, lane);
      fac += 32 * D;
    }
    f32x4 At = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) zb[jj] = bT[jj];
#pragma unroll
    for (int t = 0; t < NT / 2; ++t) {
#pragma unroll
      for (int jj = 0; jj < TPW; ++jj) IO::mma2(zb[jj], IO::to_frag(Wc[2 * t][jj]), IO::to_frag(Wc[2 * t + 1][jj]), q[2 * t], q[2 * t + 1]);
      IO::mma2(At, k[2 * t], k[2 * t + 1], q[2 * t], q[2 * t + 1]);
    }
    f32x4 cm;
#pragma unroll
    for (int r = 0; r < 4; ++r) cm[r] = (4 * g + r <= c) ? rho_c * (1.f + At[r]) : 0.f;
    const frag Mf = IO::to_frag(cm);
    // five wait states between matrix instructions of two shapes on one accumulator, as behind the bias in `update`
    if constexpr (TPW == 1) asm volatile("s_nop 4" : "+v"(zb[0]));
    else asm volatile("s_nop 4" : "+v"(zb[0]), "+v"(zb[1]));
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj) IO::mma(zb[jj], Gd[jj], Mf);
    update(kd, Gd);
    if (REST && m == n - 3) asm volatile("s_barrier" ::: "memory");  // of StateBetween (the recurrence is two mini-batches ahead)
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int jj = 0; jj < TPW; ++jj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s0 = jj + r == 0 ? zb[0][0] : s0 + zb[jj][r];
        s1 = jj + r == 0 ? zb[0][0] * zb[0][0] : __builtin_fmaf(zb[jj][r], zb[jj][r], s1);
      }
    const float v = xg_sum2_scatter(s0, s1);
    if ((g & 1) == 0) L.ez[m & 1][((g >> 1) * 16 + c) * NW + w] = v;
    lds_barrier();
  }
  if (!REST || c < rest) emit(n - 1);
}

template <int D, int SAVE, bool TWO, bool REST>
__global__ void __launch_bounds__(64 * 5, TWO ? 3 : 2) ttt_linear_fwd_roles_kernel(Problems<LinearFwdArgs> P, int cus, int rest) {
  __shared__ LinearRolesLds<D, REST> L;
  linear_fwd_roles_body<D, SAVE, TWO, REST>(P.p[blockIdx.y], L, TWO && (int)(blockIdx.y * gridDim.x + blockIdx.x) >= cus, rest);
}

template <int D, bool TWO>
__global__ void __launch_bounds__(64 * 6, TWO ? 3 : 2) ttt_linear_fwd_roles_form_kernel(LinearFwdArgs a, FusedInputsArgs fi, int cus) {
  __shared__ LinearRolesLds<D> L;
  linear_fwd_roles_body<D, 0, TWO, false, true>(a, L, TWO && (int)blockIdx.x >= cus, 0, &fi);
}

hipError_t launch_linear_fwd_roles_form(int head_dim, const LinearFwdArgs& a, const FusedInputsArgs& fi, int cus, hipStream_t s);
// rest: tokens of a short mini-batch behind the whole ones (no checkpoints then), or 0
hipError_t launch_linear_fwd_roles(int head_dim, const LinearFwdArgs* probs, unsigned ny, int cus, int rest, hipStream_t s);  // ttt_linear_fwd_roles.hip

}  // namespace ttt
