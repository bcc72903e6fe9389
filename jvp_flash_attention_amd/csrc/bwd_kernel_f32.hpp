// Backward kernels for fp32, D in {32, 64, 128}, on the forward's direct-to-LDS pipeline (fwd_kernel_f32.hpp: row-major tiles
// of 32 rows, two stages, one barrier per tile, both reads from the one copy, contraction order chosen for them).  Up to D = 64 what
// bwd_kernel_f32x3.hpp falls back on for gradients that are not finite.
// Mathematics and modes: bwd_kernel.hpp; statistics arrive negated.  What bounds them: the fp32 matrix rate, 8 (dq) and 10
// (dk/dv) executed products of which the register-staged kernels these replace reached 60 - 65 %.
// Measured, B4 H8 L1024 D64 dual with an additive bias per head: dq 325 -> 257 us, dk/dv 432 -> 333 us (87 and 84 % of
// the rate of a large fp32 matrix product); whole backward B4 H16 L2048 D64 5.56 -> 4.47 ms, D128 17.0 -> 9.4 ms.
#pragma once
#include "fwd_kernel_f32.hpp"

namespace jvpfa {

#if defined(__HIP_DEVICE_COMPILE__)
template <int NJ> __device__ __forceinline__ void load_own_row(f32x4 (&f)[NJ], const void *base, size_t off, int g) {
#pragma unroll
  for (int j = 0; j < NJ; ++j) f[j] = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(base) + off + 8 * j + 4 * g);
#pragma unroll
  for (int j = 0; j < NJ; ++j) pin_acc(f[j]);
}
template <int DB> __device__ __forceinline__ void zero_accs(f32x16 (&x)[DB]) {
#pragma unroll
  for (int db = 0; db < DB; ++db) {
#pragma unroll
    for (int e = 0; e < 16; ++e) x[db][e] = 0.f;
    pin_acc(x[db]);
  }
}
// A row of the output: registers 4q .. 4q + 3 of block db are columns DB (8q + 4g + 0..3) + db.
template <int DB> __device__ __forceinline__ void store_own_row(float *row, const f32x16 (&acc)[DB], float scale, int g) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int x = 0; x < 4 * DB; x += 4) {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = acc[(x + i) % DB][4 * q + (x + i) / DB] * scale;
      *reinterpret_cast<f32x4 *>(row + DB * (8 * q + 4 * g) + x) = v;
    }
  }
}
template <typename V> __device__ __forceinline__ void lds_done(V (&a)[4], V (&b)[4], V (&c)[4], V (&d)[4]) {
  lds_done(a, b);
  lds_done(c, d);
}

// dq (PLAIN / DUAL) or dq' (TANGENT): workgroup = 128 query rows, loop over key tiles K, V (, K', V').
template <int D, int MODE, int MASK, bool GO, bool DROP, bool SPLIT = false>
__device__ __forceinline__ void bwd_f32_dq_body(const BwdParams &p, const int bid, const BwdSplit sp = {}, const int total = 0) {
  using C = F32Cfg<D>;
  constexpr bool DUAL = MODE == BWD_DUAL, TAN = MODE == BWD_TANGENT;
  constexpr int BT = C::BT, NJ = C::NJ, DB = C::DB, NTILE = DUAL ? 4 : 2, STAGEB = NTILE * C::TILEB;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;  // stage s: [K | V | K' | V']

  const Problem &pr = p.pr;
  const int L = pr.L, Lk = pr.Lk;
  const int nqb = (L + C::BLK - 1) / C::BLK;
  const Dealt share = SPLIT ? deal_query_block(sp.q, bid, total, nqb, pr.Z * pr.H, pr.causal != 0, more_than_units(gridDim.x, pr.units)) : Dealt{xcd_remap(bid, nqb, pr.Z * pr.H, pr.causal != 0), 1, 0};
  const bool split = SPLIT && share.count > 1;
  const int zh = share.id / nqb;
  const int qb = pr.causal ? nqb - 1 - share.id % nqb : share.id % nqb;
  const int z = zh / pr.H, h = zh % pr.H;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int r = lane % 32, g = lane / 32;

  const size_t head = (size_t)zh * L * D, srow = (size_t)zh * L;
  const size_t kvhead = ((size_t)z * pr.Hk + h / (pr.H / pr.Hk)) * Lk * D;
  const float *Kg = reinterpret_cast<const float *>(p.k) + kvhead, *Vg = reinterpret_cast<const float *>(p.v) + kvhead;
  const float *Ktg = DUAL ? reinterpret_cast<const float *>(p.kt) + kvhead : nullptr;
  const float *Vtg = DUAL ? reinterpret_cast<const float *>(p.vt) + kvhead : nullptr;
  const int q0 = qb * C::BLK, qrow = q0 + wave * 32 + r, qld = qrow < L ? qrow : L - 1;

  f32x4 Qf[NJ], gOf[TAN ? 1 : NJ], Qtf[DUAL ? NJ : 1], gTf[(DUAL || TAN) ? NJ : 1];
  const size_t own = head + (size_t)qld * D;
  load_own_row(Qf, p.q, own, g);
  if constexpr (!TAN && GO) load_own_row(gOf, p.go, own, g);
  if constexpr (DUAL) load_own_row(Qtf, p.qt, own, g);
  if constexpr (DUAL || TAN) load_own_row(gTf, p.gt, own, g);
  const float Mq = qrow < L ? p.M[srow + qld] : __builtin_inff();
  const float nd1 = MODE == BWD_PLAIN ? p.neg_d1[srow + qld] : 0.f;
  const float mu = DUAL ? p.mu[srow + qld] : 0.f;
  const float na = (DUAL || TAN) ? p.neg_a[srow + qld] : 0.f;
  const float nd2 = DUAL ? p.neg_d2[srow + qld] : 0.f;
  f32x16 acc[DB];
  zero_accs(acc);

  const float sl2 = pr.scale * LOG2E;
  const int64_t mrow = MASK != MASK_NONE ? z * pr.ms[0] + h * pr.ms[1] + (int64_t)qld * pr.ms[2] : 0;
  const uint32_t drop_row = DROP ? drop_row_word(pr, zh, qld) : 0u;
  bool mask_al = false;
  if constexpr (MASK != MASK_NONE) mask_al = mask_rows_aligned<float, MASK>(pr);
  int kend = pr.causal ? min(Lk, q0 + C::BLK) : Lk;
  TileWalk<BT> walk;  // key tiles visited, see fwd_kernel_f32.hpp
  {
    const int *tl = nullptr;
    if constexpr (MASK != MASK_NONE) {
      if (pr.klimit) kend = min(kend, max(pr.klimit[z], 1));
      if (pr.tiles_q) tl = pr.tiles_q + tile_list_offset_q(pr, z, h, qb);
    }
    walk.init(tl, 0, kend, Lk);
    if (split) walk.take(share.index, share.count, ((pr.causal ? min(Lk, q0 + C::BLK) : Lk) + TILE_W - 1) / TILE_W);
  }
  const int ntiles = __builtin_amdgcn_readfirstlane(walk.n);
  auto tile_at = [&](int it) { return __builtin_amdgcn_readfirstlane(walk.at(min(it, max(ntiles - 1, 0)))); };

  F32Tiles<D, NTILE> tiles;
  tiles.init(wave, lane);
  constexpr int NLOAD = C::IPW * NTILE;
  auto aim = [&](int stage, int j0, bool on) {
    const int rows = on ? Lk - j0 : 0;
    tiles.ld_dst = lds0 + stage * STAGEB + (wave * C::IPW) * 1024;
    tiles.aim(0, Kg, j0, rows), tiles.aim(1, Vg, j0, rows);
    if constexpr (DUAL) tiles.aim(2, Ktg, j0, rows), tiles.aim(3, Vtg, j0, rows);
  };
  MaskAhead<float, MASK> mcur[2], mnext[2];
  auto fetch_masks = [&](int jn) {
    if constexpr (MASK != MASK_NONE) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
        mnext[c] = (mask_al && jn + BT <= Lk) ? mask_fetch8<float, MASK>(pr, mrow, jn + 16 * c + 8 * g) : mask_fetch8_any<float, MASK>(pr, mrow, jn + 16 * c + 8 * g);
    }
  };

  int jcur = tile_at(0), jnext = tile_at(1);
  fetch_masks(jcur);
  aim(0, jcur, ntiles > 0);
  static_for<NLOAD>([&](auto pc) { tiles.template load<decltype(pc)::value>(); });
  for (int t = 0; t < ntiles; ++t) {
    const int j0 = jcur;
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    if constexpr (MASK != MASK_NONE) {
      mcur[0] = mnext[0], mcur[1] = mnext[1];
      fetch_masks(jnext);
    }
    aim((t + 1) & 1, jnext, t + 1 < ntiles);
    const uint32_t sb = lds0 + (t & 1) * STAGEB, rowa = sb + tiles.row0;

    // ---- recompute S, (S', dP, A, B): dP also collects V' gT^T --------------------------------------------
    f32x16 S, Sp, dP, At;
    f32x4 fk[2], fv[2], fkt[2], fvt[2];
    auto issue_n = [&](auto jc) {
      constexpr int j = decltype(jc)::value, sl = j % 2;
      const uint32_t a = rowa ^ (32 * j);
      lds_row<0>(fk[sl], a);
      lds_row<C::TILEB>(fv[sl], a);
      if constexpr (DUAL) {
        lds_row<2 * C::TILEB>(fkt[sl], a);
        lds_row<3 * C::TILEB>(fvt[sl], a);
      }
    };
    typename F32Row<DB>::type tk[2][4], tkt[2][4];  // rows of 4 registers' keys
    auto issue_t = [&](auto ic) {
      constexpr int i = decltype(ic)::value;
      static_for<4>([&](auto ec) {
        constexpr int e = decltype(ec)::value;
        const uint32_t a = sb + tiles.col[4 * (i % 2) + e];
        lds_row<(i / 2) * 16 * C::ROWB>(tk[i % 2][e], a);
        if constexpr (DUAL) lds_row<2 * C::TILEB + (i / 2) * 16 * C::ROWB>(tkt[i % 2][e], a);
      });
    };
    issue_n(std::integral_constant<int, 0>{});
    static_for<NJ>([&](auto jc) {
      constexpr int j = decltype(jc)::value, sl = j % 2;
      if constexpr (DUAL) lds_done(fk[sl], fv[sl], fkt[sl], fvt[sl]);
      else lds_done(fk[sl], fv[sl]);
      if constexpr (j + 1 < NJ) issue_n(std::integral_constant<int, j + 1>{});
      else issue_t(std::integral_constant<int, 0>{});
      static_for<(NLOAD + NJ - 1) / NJ>([&](auto pc) {
        constexpr int P = j * ((NLOAD + NJ - 1) / NJ) + decltype(pc)::value;
        if constexpr (P < NLOAD) tiles.template load<P>();
      });
      static_for<4>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        constexpr bool F = j == 0 && i == 0;
        mma_f32_s<F, false, D == 128>(S, fk[sl][i], Qf[j][i]);
        if constexpr (MODE == BWD_PLAIN) mma_f32_s<F, false, D == 128>(dP, fv[sl][i], gOf[j][i]);
        if constexpr (TAN) mma_f32_s<F, false, D == 128>(At, fv[sl][i], gTf[j][i]);
        if constexpr (DUAL) {
          if constexpr (GO) mma_f32_s<F, false, D == 128>(dP, fv[sl][i], gOf[j][i]);
          mma_f32_s<F, false, D == 128>(Sp, fk[sl][i], Qtf[j][i]);
          mma_f32_s<F, false, D == 128>(At, fv[sl][i], gTf[j][i]);
          mma_f32_s<false, false, D == 128>(Sp, fkt[sl][i], Qf[j][i]);
          mma_f32_s<F && !GO, false, D == 128>(dP, fvt[sl][i], gTf[j][i]);
        }
      });
    });
    if constexpr (DUAL) tiles_ready(S, dP, Sp, At);
    else if constexpr (TAN) tiles_ready(S, At);
    else tiles_ready(S, dP);

    // ---- P and the score gradients (register e: key 16 (e / 8) + 8g + e % 8 of the tile) -------------------
    const bool edge = (pr.causal && j0 + BT - 1 > q0 + wave * 32) || j0 + BT > Lk;
    const int klim = min(pr.causal ? qrow : 0x7fffffff, Lk - 1);
    float pv[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if constexpr (MASK == MASK_ADD) pv[e] = fast_exp2(__builtin_fmaf(S[e], sl2, __builtin_fmaf(mcur[e / 8].f[e % 8], LOG2E, -Mq)));
      else pv[e] = fast_exp2(__builtin_fmaf(S[e], sl2, -Mq));
      if constexpr (MASK == MASK_BOOL) pv[e] = mask_keep_of<float, MASK>(mcur[e / 8], e % 8) ? pv[e] : 0.f;
    }
    if (edge) {
#pragma unroll
      for (int e = 0; e < 16; ++e) pv[e] = (j0 + 16 * (e / 8) + 8 * g + e % 8 <= klim) ? pv[e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if constexpr (DROP) {  // gO V^T, gT V^T, gT V'^T reach the logits through the kept, rescaled entries only
        const float ks = drop_scale_of(pr, drop_row + (uint32_t)(j0 + 16 * (e / 8) + 8 * g + e % 8) * DROP_C_KEY);
        if constexpr (!TAN) dP[e] *= ks;
        if constexpr (DUAL || TAN) At[e] *= ks;
      }
      if constexpr (MODE == BWD_PLAIN) {
        S[e] = pv[e] * (dP[e] + nd1);
      } else if constexpr (DUAL) {
        const float u = __builtin_fmaf(Sp[e], pr.scale, -mu), am = At[e] + na;
        Sp[e] = pv[e] * am;
        S[e] = pv[e] * __builtin_fmaf(am, u, dP[e] + nd2);
      } else {
        S[e] = pv[e] * (At[e] + na);
      }
    }
    if constexpr (DUAL) asm volatile("s_nop 1" : "+v"(S), "+v"(Sp));
    else asm volatile("s_nop 1" : "+v"(S));

    // ---- dQ^T += K^T dS^T (+ K'^T dS'^T) --------------------------------------------------------------------
    static_for<4>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (DUAL) lds_done(tk[i % 2], tkt[i % 2]);
      else lds_done(tk[i % 2]);
      if constexpr (i + 1 < 4) issue_t(std::integral_constant<int, i + 1>{});
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int db = 0; db < DB; ++db) mma_f32_acc(acc[db], f32_at(tk[i % 2][e], db), S[4 * i + e]);
        if constexpr (DUAL) {
#pragma unroll
          for (int db = 0; db < DB; ++db) mma_f32_acc(acc[db], f32_at(tkt[i % 2][e], db), Sp[4 * i + e]);
        }
      }
    });
    jcur = jnext;
    jnext = tile_at(t + 2);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  accs_ready(acc);
  float *out = split ? sp.part_q + (size_t)share.index * pr.Z * pr.H * L * D : reinterpret_cast<float *>(TAN ? p.dqt : p.dq);
  if (qrow < L) store_own_row(out + head + (size_t)qrow * D, acc, pr.scale, g);
}

// dk, dv (PLAIN / DUAL) or dk', dv' (TANGENT): workgroup = 128 key rows, loop over query tiles Q, G (, Q', gT),
// G = gO (gT in TANGENT).  Scores are S = Q K^T (lane = key).  The query heads of a group are visited one after
// another (this workgroup's share of them, see split.hpp).
template <int D, int MODE, int MASK, bool GO, bool DROP, bool SPLIT = false>
__device__ __forceinline__ void bwd_f32_dkdv_body(const BwdParams &p, const int bid, const BwdSplit sp = {}, const int total = 0) {
  using C = F32Cfg<D>;
  constexpr bool DUAL = MODE == BWD_DUAL, TAN = MODE == BWD_TANGENT;
  constexpr int BT = C::BT, NJ = C::NJ, DB = C::DB, NTILE = DUAL ? 4 : 2, STAGEB = NTILE * C::TILEB;
  constexpr int NSTAT = DUAL ? 4 : 2, STATB = NSTAT * 64 * 4;  // row statistics: 64 lanes a load, 32 of them used
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;  // stage s: [Q | G | Q' | gT], then two stages of statistics
  const uint32_t stat0 = lds0 + 2 * STAGEB;

  const Problem &pr = p.pr;
  const int L = pr.L, Lk = pr.Lk;
  const int nkb = (Lk + C::BLK - 1) / C::BLK;
  const int shares = pr.Z * pr.Hk * pr.chunks;
  const Dealt share = SPLIT ? deal_key_block(sp.k, bid, total, nkb, shares, pr.causal != 0, more_than_units(gridDim.x, pr.units)) : Dealt{xcd_remap(bid, nkb, shares, pr.causal != 0), 1, 0};
  const bool split = SPLIT && share.count > 1;
  const int zhk = share.id / nkb / pr.chunks, chunk = share.id / nkb % pr.chunks;
  const int kb = share.id % nkb;  // causal: the first key blocks have the longest query loops
  const int z = zhk / pr.Hk, hk = zhk % pr.Hk, group = group_share(pr, chunk + 1) - group_share(pr, chunk);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int r = lane % 32, g = lane / 32;

  const size_t kvhead = (size_t)zhk * Lk * D;
  const int k0 = kb * C::BLK, krow = k0 + wave * 32 + r, kld = krow < Lk ? krow : Lk - 1;
  const uint32_t drop_lane = DROP ? (uint32_t)kld * DROP_C_KEY + (uint32_t)(8 * g) * DROP_C_ROW : 0u;
  f32x4 Kf[NJ], Vf[NJ], Ktf[DUAL ? NJ : 1], Vtf[DUAL ? NJ : 1];
  const size_t own = kvhead + (size_t)kld * D;
  load_own_row(Kf, p.k, own, g);
  load_own_row(Vf, p.v, own, g);
  if constexpr (DUAL) {
    load_own_row(Ktf, p.kt, own, g);
    load_own_row(Vtf, p.vt, own, g);
  }
  f32x16 dK[DB], dV[DB];
  zero_accs(dK);
  zero_accs(dV);

  const float sl2 = pr.scale * LOG2E;
  const int istart = pr.causal ? (k0 / BT) * BT : 0;
  F32Tiles<D, NTILE> tiles;
  tiles.init(wave, lane);
  constexpr int NLOAD = C::IPW * NTILE;

  for (int gi = 0; gi < group; ++gi) {
    const int h = hk * (pr.H / pr.Hk) + group_share(pr, chunk) + gi;  // query head
    const size_t head = ((size_t)z * pr.H + h) * L * D, srow = ((size_t)z * pr.H + h) * L;
    const float *Qg = reinterpret_cast<const float *>(p.q) + head;
    const float *Qtg = DUAL ? reinterpret_cast<const float *>(p.qt) + head : nullptr;
    const float *gTg = (DUAL || TAN) ? reinterpret_cast<const float *>(p.gt) + head : nullptr;
    const float *Gg = TAN ? gTg : (GO ? reinterpret_cast<const float *>(p.go) + head : Qg);
    const float *st_p[4] = {p.M + srow, (MODE == BWD_PLAIN ? p.neg_d1 : DUAL ? p.mu : p.neg_a) + srow, DUAL ? p.neg_a + srow : nullptr, DUAL ? p.neg_d2 + srow : nullptr};
    TileWalk<BT> walk;  // query tiles visited: all from istart on, or those of the caller's list
    {
      const int *tl = nullptr;
      if constexpr (MASK != MASK_NONE) {
        if (pr.tiles_k) tl = pr.tiles_k + tile_list_offset_k(pr, z, h, kb);
      }
      walk.init(tl, istart, L, L);
      if constexpr (MASK != MASK_NONE) {
        if (pr.klimit && k0 >= pr.klimit[z]) walk.n = 0;  // a key block the caller's hint declares fully masked: zeros
      }
      if (split) walk.take(share.index, share.count, (max(L - istart, 0) + TILE_W - 1) / TILE_W);
    }
    const int ntiles = __builtin_amdgcn_readfirstlane(walk.n);
    auto tile_at = [&](int it) { return __builtin_amdgcn_readfirstlane(walk.at(min(it, max(ntiles - 1, 0)))); };
    auto aim = [&](int stage, int i0, bool on) {
      const int rows = on ? L - i0 : 0;
      tiles.ld_dst = lds0 + stage * STAGEB + (wave * C::IPW) * 1024;
      tiles.aim(0, Qg, i0, rows), tiles.aim(1, Gg, i0, (DUAL && !GO) ? 0 : rows);
      if constexpr (DUAL) tiles.aim(2, Qtg, i0, rows), tiles.aim(3, gTg, i0, rows);
    };
    auto load_stats = [&](int stage, int i0) {  // wave s brings statistic s (rows past the end: the last one's)
      if (wave < NSTAT)
        __builtin_amdgcn_global_load_lds((JVPFA_GLB(const void))(st_p[wave] + min(i0 + lane, L - 1)),
                                         (JVPFA_LDS(void))(uintptr_t)(stat0 + stage * STATB + wave * 256), 4, 0, 0);
    };
    // mask entries of this lane's key against the 16 queries of its registers, a tile ahead
    float mcur_a[MASK == MASK_ADD ? 16 : 1], mnext_a[MASK == MASK_ADD ? 16 : 1];
    uint8_t mcur_b[MASK == MASK_BOOL ? 16 : 1], mnext_b[MASK == MASK_BOOL ? 16 : 1];
    auto fetch_masks = [&](int in) {
      if constexpr (MASK != MASK_NONE) {
        const int64_t col = z * pr.ms[0] + h * pr.ms[1] + (int64_t)kld * pr.ms[3];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t off = col + (int64_t)min(in + 16 * (e / 8) + 8 * g + e % 8, L - 1) * pr.ms[2];
          if constexpr (MASK == MASK_ADD) mnext_a[e] = reinterpret_cast<const float *>(pr.mask)[off];
          if constexpr (MASK == MASK_BOOL) mnext_b[e] = reinterpret_cast<const uint8_t *>(pr.mask)[off];
        }
      }
    };

    if (gi > 0) __syncthreads();  // every wave is done with the previous head's last tile
    int icur = tile_at(0), inext = tile_at(1);
    if (ntiles > 0) {
      fetch_masks(icur);
      aim(0, icur, true);
      static_for<NLOAD>([&](auto pc) { tiles.template load<decltype(pc)::value>(); });
      load_stats(0, icur);
    }
    for (int t = 0; t < ntiles; ++t) {
      const int i0 = icur;
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
      if constexpr (MASK != MASK_NONE) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          if constexpr (MASK == MASK_ADD) mcur_a[e] = mnext_a[e];
          if constexpr (MASK == MASK_BOOL) mcur_b[e] = mnext_b[e];
        }
        fetch_masks(inext);
      }
      aim((t + 1) & 1, inext, t + 1 < ntiles);
      load_stats((t + 1) & 1, inext);
      const uint32_t sb = lds0 + (t & 1) * STAGEB, rowa = sb + tiles.row0;
      const uint32_t sta = stat0 + (t & 1) * STATB + 8 * g * 4;

      // ---- recompute: dP also collects gT V'^T ------------------------------------------------------------
      f32x16 S, Sp, dP, At;
      f32x4 fq[2], fg[2], fqt[2], fgt[2];
      auto issue_n = [&](auto jc) {
        constexpr int j = decltype(jc)::value, sl = j % 2;
        const uint32_t a = rowa ^ (32 * j);
        lds_row<0>(fq[sl], a);
        lds_row<C::TILEB>(fg[sl], a);
        if constexpr (DUAL) {
          lds_row<2 * C::TILEB>(fqt[sl], a);
          lds_row<3 * C::TILEB>(fgt[sl], a);
        }
      };
      f32x4 st[2][4];  // statistics of registers 4q .. 4q + 3 (queries 16 (q / 2) + 8g + 4 (q % 2) + 0..3)
      auto issue_s = [&](auto qc) {
        constexpr int q = decltype(qc)::value, O = (q / 2) * 64 + (q % 2) * 16;
        lds_row<O>(st[q % 2][0], sta);
        lds_row<O + 256>(st[q % 2][1], sta);
        if constexpr (DUAL) {
          lds_row<O + 512>(st[q % 2][2], sta);
          lds_row<O + 768>(st[q % 2][3], sta);
        }
      };
      auto stats_done = [&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (DUAL) lds_done(st[q % 2]);
        else lds_done(st[q % 2][0], st[q % 2][1]);
      };
      issue_n(std::integral_constant<int, 0>{});
      static_for<NJ>([&](auto jc) {
        constexpr int j = decltype(jc)::value, sl = j % 2;
        if constexpr (DUAL) lds_done(fq[sl], fg[sl], fqt[sl], fgt[sl]);
        else lds_done(fq[sl], fg[sl]);
        if constexpr (j + 1 < NJ) issue_n(std::integral_constant<int, j + 1>{});
        else issue_s(std::integral_constant<int, 0>{});
        static_for<(NLOAD + NJ - 1) / NJ>([&](auto pc) {
          constexpr int P = j * ((NLOAD + NJ - 1) / NJ) + decltype(pc)::value;
          if constexpr (P < NLOAD) tiles.template load<P>();
        });
        static_for<4>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          constexpr bool F = j == 0 && i == 0;
          mma_f32_s<F, false, D == 128>(S, fq[sl][i], Kf[j][i]);
          if constexpr (MODE == BWD_PLAIN) mma_f32_s<F, false, D == 128>(dP, fg[sl][i], Vf[j][i]);
          if constexpr (TAN) mma_f32_s<F, false, D == 128>(At, fg[sl][i], Vf[j][i]);
          if constexpr (DUAL) {
            if constexpr (GO) mma_f32_s<F, false, D == 128>(dP, fg[sl][i], Vf[j][i]);
            mma_f32_s<F, false, D == 128>(Sp, fqt[sl][i], Kf[j][i]);
            mma_f32_s<F, false, D == 128>(At, fgt[sl][i], Vf[j][i]);
            mma_f32_s<false, false, D == 128>(Sp, fq[sl][i], Ktf[j][i]);
            mma_f32_s<F && !GO, false, D == 128>(dP, fgt[sl][i], Vtf[j][i]);
          }
        });
      });
      if constexpr (DUAL) tiles_ready(S, dP, Sp, At);
      else if constexpr (TAN) tiles_ready(S, At);
      else tiles_ready(S, dP);

      // ---- P, P' and the score gradients, four registers at a time -----------------------------------------
      const bool edge = (pr.causal && i0 < k0 + wave * 32 + 31) || i0 + BT > L;
      const int qmin = pr.causal ? krow : 0;  // queries below this index do not see this key
      const uint32_t drop_tile = DROP ? drop_row_word(pr, z * pr.H + h, i0) + drop_lane : 0u;  // 32 queries: one block of the pattern
      f32x16 Pp;  // DUAL: P (S' - mu)
      static_for<4>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        stats_done(qc);
        if constexpr (q + 1 < 4) issue_s(std::integral_constant<int, q + 1>{});
        const f32x4(&s_)[4] = st[q % 2];
        float pv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = 4 * q + i;
          if constexpr (MASK == MASK_ADD) pv[i] = fast_exp2(__builtin_fmaf(S[e], sl2, __builtin_fmaf(mcur_a[e], LOG2E, -s_[0][i])));
          else pv[i] = fast_exp2(__builtin_fmaf(S[e], sl2, -s_[0][i]));
          if constexpr (MASK == MASK_BOOL) pv[i] = mcur_b[e] != 0 ? pv[i] : 0.f;
        }
        if (edge) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int qi = i0 + 16 * (q / 2) + 8 * g + 4 * (q % 2) + i;
            pv[i] = (qi >= qmin && qi < L) ? pv[i] : 0.f;
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = 4 * q + i;
          float ks = 1.f;  // dropout: 1 / (1 - p) for a kept entry, 0 for a dropped one
          if constexpr (DROP) {
            ks = drop_scale_of(pr, drop_tile + (uint32_t)(16 * (e / 8) + e % 8) * DROP_C_ROW);
            if constexpr (!TAN) dP[e] *= ks;
            if constexpr (DUAL || TAN) At[e] *= ks;
          }
          S[e] = DROP ? pv[i] * ks : pv[i];
          if constexpr (MODE == BWD_PLAIN) {
            dP[e] = pv[i] * (dP[e] + s_[1][i]);
          } else if constexpr (DUAL) {
            const float u = __builtin_fmaf(Sp[e], pr.scale, -s_[1][i]), am = At[e] + s_[2][i];
            Pp[e] = DROP ? pv[i] * u * ks : pv[i] * u;
            Sp[e] = pv[i] * am;
            dP[e] = pv[i] * __builtin_fmaf(am, u, dP[e] + s_[3][i]);
          } else {
            Sp[e] = pv[i] * (At[e] + s_[1][i]);
          }
        }
      });
      // query rows of KT registers (one where four tensors' rows of 128 columns would not fit twice)
      constexpr int KT = DUAL && D == 128 ? 1 : 2;
      typename F32Row<DB>::type tq[2][2], tg[2][2], tqt[2][2], tgt[2][2];
      auto issue_t = [&](auto ic) {
        constexpr int i = decltype(ic)::value, sl = i % 2, O = (KT * i / 8) * 16 * C::ROWB;
        static_for<KT>([&](auto ec) {
          constexpr int e = decltype(ec)::value;
          const uint32_t a = sb + tiles.col[KT * i % 8 + e];
          lds_row<O>(tq[sl][e], a);
          if constexpr (!DUAL || GO) lds_row<C::TILEB + O>(tg[sl][e], a);
          if constexpr (DUAL) {
            lds_row<2 * C::TILEB + O>(tqt[sl][e], a);
            lds_row<3 * C::TILEB + O>(tgt[sl][e], a);
          }
        });
      };
      issue_t(std::integral_constant<int, 0>{});
      if constexpr (DUAL) asm volatile("s_nop 1" : "+v"(S), "+v"(Sp), "+v"(dP), "+v"(Pp));
      else if constexpr (TAN) asm volatile("s_nop 1" : "+v"(S), "+v"(Sp));
      else asm volatile("s_nop 1" : "+v"(S), "+v"(dP));

      // ---- dK^T += Q^T dS (+ Q'^T dS'), dV^T += G^T P (+ gT^T P') -------------------------------------------
      static_for<16 / KT>([&](auto ic) {
        constexpr int i = decltype(ic)::value, sl = i % 2;
        static_for<KT>([&](auto ec) {
          constexpr int e = decltype(ec)::value;
          lds_done(tq[sl][e]);
          if constexpr (!DUAL || GO) lds_done(tg[sl][e]);
          if constexpr (DUAL) lds_done(tqt[sl][e], tgt[sl][e]);
        });
        if constexpr (i + 1 < 16 / KT) issue_t(std::integral_constant<int, i + 1>{});
#pragma unroll
        for (int e = 0; e < KT; ++e) {
          const int x = KT * i + e;
#pragma unroll
          for (int db = 0; db < DB; ++db) {
            if constexpr (MODE == BWD_PLAIN) {
              mma_f32_acc(dK[db], f32_at(tq[sl][e], db), dP[x]);
              mma_f32_acc(dV[db], f32_at(tg[sl][e], db), S[x]);
            } else if constexpr (DUAL) {
              mma_f32_acc(dK[db], f32_at(tq[sl][e], db), dP[x]);
              if constexpr (GO) mma_f32_acc(dV[db], f32_at(tg[sl][e], db), S[x]);
              mma_f32_acc(dK[db], f32_at(tqt[sl][e], db), Sp[x]);
              mma_f32_acc(dV[db], f32_at(tgt[sl][e], db), Pp[x]);
            } else {
              mma_f32_acc(dK[db], f32_at(tq[sl][e], db), Sp[x]);
              mma_f32_acc(dV[db], f32_at(tg[sl][e], db), S[x]);
            }
          }
        }
      });
      icur = inext;
      inext = tile_at(t + 2);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  }
  accs_ready(dK, dV);
  if (krow < Lk) {
    const size_t elems = (size_t)pr.Z * pr.Hk * Lk * D;
    float *partk = split ? sp.part_k + share.index * 2 * elems : kv_part(pr, D, 2, 0, chunk), *partv = split ? partk + elems : kv_part(pr, D, 2, 1, chunk);
    const size_t off = kvhead + (size_t)krow * D;
    store_own_row((partk ? partk : reinterpret_cast<float *>(TAN ? p.dkt : p.dk)) + off, dK, pr.scale, g);
    store_own_row((partv ? partv : reinterpret_cast<float *>(TAN ? p.dvt : p.dv)) + off, dV, 1.f, g);
  }
}
#endif

template <int D, int MODE> struct BwdF32Lds {
  static constexpr size_t DQ = 2 * (MODE == BWD_DUAL ? 4 : 2) * (size_t)F32Cfg<D>::TILEB;
  static constexpr size_t DKV = DQ + 2 * (MODE == BWD_DUAL ? 4 : 2) * 256;
};
template <int D, int MODE, int MASK, bool GO, bool DROP = false>
__global__ __launch_bounds__(256, 1) void bwd_f32_dq_kernel(const BwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  bwd_f32_dq_body<D, MODE, MASK, GO, DROP>(p, blockIdx.x);
#endif
}
template <int D, int MODE, int MASK, bool GO, bool DROP = false>
__global__ __launch_bounds__(256, 1) void bwd_f32_dkdv_kernel(const BwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  bwd_f32_dkdv_body<D, MODE, MASK, GO, DROP>(p, blockIdx.x);
#endif
}

// Both roles in one launch (see bwd2_both_kernel): the first kv_blocks workgroups are dk/dv workgroups.  SPLIT: blocks' tiles split
// (split.hpp), compiled apart: what it needs takes 15 - 80 scalar registers that the others' loops have to spill (B2 H6 L777 D64 first
// order with a bias, whose rows are not aligned: 124 -> 159 us).
template <int D, int MODE, int MASK, bool GO, bool SPLIT>
__global__ __launch_bounds__(256, 1) void bwd_f32_both_kernel(const BwdParams p, const BwdSplit sp, const int kv_blocks) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int b = __builtin_amdgcn_readfirstlane(blockIdx.x);
  if (b < kv_blocks) bwd_f32_dkdv_body<D, MODE, MASK, GO, false, SPLIT>(p, b, sp, kv_blocks);
  else bwd_f32_dq_body<D, MODE, MASK, GO, false, SPLIT>(p, b - kv_blocks, sp, gridDim.x - kv_blocks);
#endif
}

}  // namespace jvpfa
