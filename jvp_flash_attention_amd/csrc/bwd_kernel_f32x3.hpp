// Backward kernels for fp32, D in {32, 64}, on the 16-bit matrix instructions: every operand as three bf16 parts, six products
// for one (fwd_kernel_f32x3.hpp: why, and with which error).  Mathematics, work split and modes as in bwd_kernel_f32.hpp.
//
// A workgroup's own rows stay resident as parts; the streamed 32-row tiles go global -> registers (a tile ahead) -> three
// bf16 planes each in LDS, two stages, one barrier per tile, and are read both ways from the one copy.  A tile is four
// groups of matrix instructions, each with vector work between them that depends on the group before:
//     S, S'  |  staging of the next tile      dP, A  |  P (and, dk/dv, P' and their parts)
//     dk/dv: dV | dS, dS' and their parts     dK | the rest of the staging
//     dq:    half of dS, dS', then dQ of that half | the other half, then dQ of it
// The small products of the six go first into the one accumulator there is room for: sums over 8192 terms are then off by
// 1.4e-6 (2-norm, signs mixed; 0.77e-6 for terms of one sign) where the fp32 instructions are by 1.6e-6 (1.2e-6).
// What bounds them: one wave per SIMD, which pays most of an issue slot for each vector instruction between the matrix ones.
// Measured, B4 H8 L1024 D64 dual, kernels alone: key padding dq 251 -> 153 us, dk/dv 326 -> 200 us; bias per head dq 263 ->
// 172 us, dk/dv 339 -> 228 us (without a mask the whole backward takes as long).
#pragma once
#include "bwd_kernel_f32.hpp"
#include "fwd_kernel_f32x3.hpp"

namespace jvpfa {

#if defined(__HIP_DEVICE_COMPILE__)
// Own rows as parts, resident in the accumulation file.
template <int KK> __device__ __forceinline__ void x3_own_row(bf16x8 (&f)[KK][3], const void *base, size_t off, int g) {
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    const float *src = reinterpret_cast<const float *>(base) + off + 16 * kk + 8 * g;
    u32x4 x[3];
    x3_split8(*reinterpret_cast<const f32x4 *>(src), *reinterpret_cast<const f32x4 *>(src + 4), x);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      f[kk][i] = x3_frag(x[i]);
      pin_acc(f[kk][i]);
    }
  }
}

// Staging and fragment reads of the streamed tiles of NTILE tensors; SKIP: this one is absent.
template <int D, int NTILE, int SKIP> struct X3Tiles {
  using C = X3Cfg<D>;
  static constexpr int KK = D / 16, DB = D / 32, STAGEB = NTILE * C::OPB, NTASK = NTILE * C::TASKS / C::NT;
  static_assert(C::TASKS == C::NT || 2 * C::TASKS == C::NT, "the tensor of a task is the same in every lane of a wave");
  static constexpr bool PAIRED = C::TASKS != C::NT;  // two tensors to a task, one for either half of the waves
  static constexpr int NLIVE = NTASK - (!PAIRED && SKIP >= 0 ? 1 : 0), NU = 10 * NLIVE;
  const float *base[NTASK];
  uint32_t src, dst[NTASK], roff[KK], toff[DB][2];
  f32x4 raw[NTASK][2];
  u32x4 sp[3];
  float sa = 0.f, sb = 0.f;

  __device__ __forceinline__ void init(uint32_t lds0, int tid, int lane) {
    const int r = lane % 32, g = lane / 32, pr32 = perm32(r), row = (tid % C::TASKS) / C::CH, ch = tid % C::CH;
    src = (tid % C::TASKS) * 32;
#pragma unroll
    for (int i = 0; i < NTASK; ++i) dst[i] = lds0 + (PAIRED ? 2 * i * C::OPB + (tid / C::TASKS) * C::OPB : i * C::OPB) + row * C::ROWB + ((ch ^ swz_u<C::CH>(row)) * 16);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) roff[kk] = lds0 + pr32 * C::ROWB + (((2 * kk + g) ^ swz_u<C::CH>(pr32)) * 16);
    const int a = (lane >> 4) & 1, j = lane & 15;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int rw = 8 * g + 4 * hh + (j >> 2);
        toff[db][hh] = lds0 + rw * C::ROWB + (((4 * db + 2 * a + (j & 1)) ^ swz_u<C::CH>(rw)) * 16) + 8 * ((j >> 1) & 1);
      }
    }
  }
  __device__ __forceinline__ void tensors(int wave, const float *const (&t)[4]) {
#pragma unroll
    for (int i = 0; i < NTASK; ++i) base[i] = PAIRED ? (wave < 2 ? t[2 * i] : t[2 * i + 1]) : t[i];
  }
  static constexpr bool live(int i) { return PAIRED || i != SKIP; }
  // task i's rows of the tile whose first is j of len (rows past the end, and tiles that do not exist: zeros)
  template <int I> __device__ __forceinline__ void load(int j, int len, bool on) {
    const int bytes = __builtin_amdgcn_readfirstlane(min(max(on ? len - j : 0, 0), C::BT) * (D * 4));
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)(base[I] + (size_t)j * D), 0, bytes, 0x00020000);
    raw[I][0] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, src, 0, 0));
    raw[I][1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, src + 16, 0, 0));
  }
  template <int I> __device__ __forceinline__ void store(uint32_t stage) {
#pragma unroll
    for (int x = 0; x < 3; ++x) *(JVPFA_LDS(u32x4))(uintptr_t)(dst[I] + stage + x * C::PLANE) = sp[x];
  }
  // unit u of splitting what the registers hold into `stage` and requesting the tile at j
  template <int U> __device__ __forceinline__ void unit(uint32_t stage, int j, int len, bool on) {
    constexpr int n = U / 10, i = (!PAIRED && SKIP >= 0 && n >= SKIP) ? n + 1 : n, s = U % 10, w = s / 2;
    if constexpr (s < 8) {
      if constexpr (s % 2 == 0) {
        sa = raw[i][w / 2][2 * (w % 2)], sb = raw[i][w / 2][2 * (w % 2) + 1];
        sp[0][w] = x3_take(sa, sb);
        anchor(sa), anchor(sb);
      } else {
        sp[1][w] = x3_take(sa, sb);
        sp[2][w] = x3_last(sa, sb);
        anchor(sp[2][w]);
      }
    } else if constexpr (s == 8) {
      store<i>(stage);
    } else {
      load<i>(j, len, on);
    }
  }
  // first tile of a walk at once, the second one requested
  __device__ __forceinline__ void first(int j, int jnext, int len, bool next) {
    static_for<NTASK>([&](auto ic) {
      if constexpr (live(decltype(ic)::value)) load<decltype(ic)::value>(j, len, true);
    });
    static_for<NTASK>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (live(i)) {
        x3_split8(raw[i][0], raw[i][1], sp);
        store<i>(0);
        load<i>(jnext, len, next);
      }
    });
  }
  template <int T> __device__ __forceinline__ void rows(u32x4 (&f)[3], int kk, uint32_t stage) const {
    const uint32_t a = roff[kk] + stage;
    static_for<3>([&](auto xc) { f[decltype(xc)::value] = lds_b128<T * C::OPB + decltype(xc)::value * C::PLANE>(a); });
  }
  template <int T, int CHUNK> __device__ __forceinline__ void cols(u32x2 (&f)[3][2], int db, uint32_t stage) const {
    const uint32_t a0 = toff[db][0] + stage, a1 = toff[db][1] + stage;
    static_for<3>([&](auto xc) {
      constexpr int O = T * C::OPB + decltype(xc)::value * C::PLANE + CHUNK * 16 * C::ROWB;
      f[decltype(xc)::value][0] = lds_tr64<O>(a0);
      f[decltype(xc)::value][1] = lds_tr64<O>(a1);
    });
  }
};
// Behind matrix instruction number G of a group of NG: its share of the NU units of vector work.  AFTER: units start behind the
// third instruction, when the results of the group before are through.
template <int G, int NG, int NU, bool AFTER, typename F> __device__ __forceinline__ void x3_gap(F &&unit) {
  constexpr int S = AFTER ? 2 : 0, lo = G < S ? 0 : (G - S) * NU / (NG - S), hi = G < S ? 0 : (G - S + 1) * NU / (NG - S);
  static_for<hi - lo>([&](auto dc) { unit(std::integral_constant<int, lo + decltype(dc)::value>{}); });
  __builtin_amdgcn_sched_barrier(0);
}
// dq (PLAIN / DUAL) or dq' (TANGENT).  Returns whether every output is finite.
template <int D, int MODE, int MASK, bool GO, bool DROP, bool SPLIT = false>
__device__ __forceinline__ bool bwd_f32x3_dq_body(const BwdParams &p, const int bid, const BwdSplit sp = {}, const int total = 0) {
  using C = X3Cfg<D>;
  constexpr bool DUAL = MODE == BWD_DUAL, TAN = MODE == BWD_TANGENT;
  constexpr int BT = C::BT, KK = D / 16, DB = D / 32, NTILE = DUAL ? 4 : 2;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;  // stage s: [K | V | K' | V'], three planes each

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
  const int q0 = qb * C::BLK, qrow = q0 + wave * 32 + r, qld = qrow < L ? qrow : L - 1;

  bf16x8 Qf[KK][3], gOf[TAN || !GO ? 1 : KK][3], Qtf[DUAL ? KK : 1][3], gTf[(DUAL || TAN) ? KK : 1][3];
  const size_t own = head + (size_t)qld * D;
  x3_own_row(Qf, p.q, own, g);
  if constexpr (!TAN && GO) x3_own_row(gOf, p.go, own, g);
  if constexpr (DUAL) x3_own_row(Qtf, p.qt, own, g);
  if constexpr (DUAL || TAN) x3_own_row(gTf, p.gt, own, g);
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

  using Tiles = X3Tiles<D, NTILE, -1>;
  Tiles tiles;
  tiles.init(lds0, tid, lane);
  {
    const float *t[4] = {reinterpret_cast<const float *>(p.k) + kvhead, reinterpret_cast<const float *>(p.v) + kvhead,
                         DUAL ? reinterpret_cast<const float *>(p.kt) + kvhead : nullptr, DUAL ? reinterpret_cast<const float *>(p.vt) + kvhead : nullptr};
    tiles.tensors(wave, t);
  }
  MaskAhead<float, MASK> mk[2];
  const int klim = min(pr.causal ? qrow : 0x7fffffff, Lk - 1);
  const uint32_t vzero = 0u, vninf = 0xff800000u;

  // One tile: its first key is j0, the next but one's jn.
  auto tile = [&](int t, int j0, int jn, auto LIMc) {
    x3_barrier();
    if constexpr (MASK != MASK_NONE) {  // (keys past the end come masked)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        mk[c] = (mask_al && j0 + BT <= Lk) ? mask_fetch8<float, MASK>(pr, mrow, j0 + 16 * c + 8 * g) : mask_fetch8_lim<float, MASK>(pr, mrow, j0 + 16 * c + 8 * g);
    }
    const uint32_t st = (t & 1) * Tiles::STAGEB, stn = ((t + 1) & 1) * Tiles::STAGEB;
    f32x16 S, Sp, dP, At;
    // ---- S, S' of K, K', with the staging of the next tile; then dP, A of V, V', with P ---------------------
    u32x4 fr[2][3];
    constexpr int NPAIR = DUAL ? 2 : 1, NS = KK * NPAIR;  // steps of a group: (contraction step, tensor)
    auto read_row = [&](auto ic) {  // step i of both groups
      constexpr int i = decltype(ic)::value, kk = (i % NS) / NPAIR, T = (i / NS) + 2 * (i % NPAIR);
      tiles.template rows<T>(fr[i % 2], kk, st);
    };
    auto unit_st = [&](auto uc) { tiles.template unit<decltype(uc)::value>(stn, jn, Lk, t + 2 < ntiles); };
    float x1 = 0.f;
    auto unit_p = [&](auto uc) {  // S becomes P, S' becomes S' - mu: two units per pair of entries
      constexpr int u = decltype(uc)::value, e = u & ~1;
      auto arg = [&](auto ec) {
        constexpr int y = decltype(ec)::value;
        float m = -Mq;
        if constexpr (MASK == MASK_ADD) m = __builtin_fmaf(mk[y / 8].f[y % 8], LOG2E, -Mq);
        if constexpr (MASK == MASK_BOOL) m += mask_term_of_byte<y % 4>((y % 8) < 4 ? (uint32_t)mk[y / 8].w : (uint32_t)(mk[y / 8].w >> 32), vzero, vninf);
        float x = __builtin_fmaf(S[y], sl2, m);
        if constexpr (decltype(LIMc)::value) x = (j0 + 16 * (y / 8) + 8 * g + y % 8 <= klim) ? x : -__builtin_inff();
        return x;
      };
      if constexpr (u % 2 == 0) {
        const float x0 = arg(std::integral_constant<int, e>{});
        x1 = arg(std::integral_constant<int, e + 1>{});
        S[e] = fast_exp2(x0);
        anchor(x1);
        anchor(S[e]);
      } else {
        S[e + 1] = fast_exp2(x1);
        if constexpr (DUAL) {
          Sp[e] = __builtin_fmaf(Sp[e], pr.scale, -mu);
          Sp[e + 1] = __builtin_fmaf(Sp[e + 1], pr.scale, -mu);
          anchor(Sp[e + 1]);
        }
        anchor(S[e + 1]);
      }
    };
    // dS (and dS') in parts
    constexpr int UPP = (DUAL ? 5 : 3), NU_DS = 4 * UPP;  // units per pair of entries; per half of the tile
    u32x4 ds[2][3], dt[2][3];
    float a0 = 0.f, a1 = 0.f, b0 = 0.f, b1 = 0.f;
    auto unit_ds = [&](auto cc, auto uc) {
      constexpr int c = decltype(cc)::value, u = decltype(uc)::value, w = u / UPP, s = u % UPP, e = 8 * c + 2 * w;
      if constexpr (s == 0) {
        auto one = [&](auto ec, float &a, float &b) {
          constexpr int y = decltype(ec)::value;
          if constexpr (DROP) {  // gO V^T, gT V^T, gT V'^T reach the logits through the kept, rescaled entries only
            const float ks = drop_scale_of(pr, drop_row + (uint32_t)(j0 + 16 * (y / 8) + 8 * g + y % 8) * DROP_C_KEY);
            if constexpr (!TAN) dP[y] *= ks;
            if constexpr (DUAL || TAN) At[y] *= ks;
          }
          if constexpr (MODE == BWD_PLAIN) {
            a = S[y] * (dP[y] + nd1);
          } else if constexpr (DUAL) {
            const float am = At[y] + na;
            b = S[y] * am;
            a = S[y] * __builtin_fmaf(am, Sp[y], dP[y] + nd2);
            anchor(b);
          } else {
            a = S[y] * (At[y] + na);
          }
          anchor(a);
        };
        one(std::integral_constant<int, e>{}, a0, b0);
        one(std::integral_constant<int, e + 1>{}, a1, b1);
      } else if constexpr (s == 1) {
        ds[c][0][w] = x3_take(a0, a1);
        anchor(a0), anchor(a1);
      } else if constexpr (s == 2) {
        ds[c][1][w] = x3_take(a0, a1);
        ds[c][2][w] = x3_last(a0, a1);
        anchor(ds[c][2][w]);
      } else if constexpr (s == 3) {
        dt[c][0][w] = x3_take(b0, b1);
        anchor(b0), anchor(b1);
      } else {
        dt[c][1][w] = x3_take(b0, b1);
        dt[c][2][w] = x3_last(b0, b1);
        anchor(dt[c][2][w]);
      }
    };
    u32x2 ca[2][3][2], cb[2][3][2];
    auto read_col = [&](auto ic) {
      constexpr int i = decltype(ic)::value, c = i / DB, db = i % DB;
      tiles.template cols<0, c>(ca[i % 2], db, st);
      if constexpr (DUAL) tiles.template cols<2, c>(cb[i % 2], db, st);
    };

    read_row(std::integral_constant<int, 0>{});
    static_for<2 * NS>([&](auto ic) {
      constexpr int i = decltype(ic)::value, G = i / NS, kk = (i % NS) / NPAIR, pair = i % NPAIR, sl = i % 2;
      x3_wait(fr[sl]);
      if constexpr (i + 1 < 2 * NS) read_row(std::integral_constant<int, i + 1>{});
      else read_col(std::integral_constant<int, 0>{});
      __builtin_amdgcn_sched_barrier(0);
      static_for<6>([&](auto xc) {
        constexpr int x = decltype(xc)::value;
        constexpr bool F = kk == 0 && x == 0;
        const bf16x8 a = x3_frag(fr[sl][X3_A[x]]);
        // number of this product's first instruction within its group: the first tensor of a step makes TWO, the second one
        constexpr int TWO = DUAL && (G == 0 || GO) ? 2 : 1, PER = 6 * (TWO + NPAIR - 1), N0 = kk * PER + (pair == 0 ? x * TWO : 6 * TWO + x);
        auto gap = [&](auto nc) {
          if constexpr (G == 0) x3_gap<decltype(nc)::value, KK * PER, Tiles::NU, false>(unit_st);
          else x3_gap<decltype(nc)::value, KK * PER, 16, true>(unit_p);
        };
        if constexpr (G == 0) {
          if constexpr (pair == 0) {
            if constexpr (DUAL) {
              mfma_s<F>(Sp, a, Qtf[kk][X3_B[x]]);
              gap(std::integral_constant<int, N0>{});
              mfma_s<F>(S, a, Qf[kk][X3_B[x]]);
              gap(std::integral_constant<int, N0 + 1>{});
            } else {
              mfma_s<F>(S, a, Qf[kk][X3_B[x]]);
              gap(std::integral_constant<int, N0>{});
            }
          } else {
            mfma_s<false>(Sp, a, Qf[kk][X3_B[x]]);
            gap(std::integral_constant<int, N0>{});
          }
        } else if constexpr (pair == 0) {
          if constexpr (MODE == BWD_PLAIN) {
            mfma_s<F>(dP, a, gOf[kk][X3_B[x]]);
            gap(std::integral_constant<int, N0>{});
          } else if constexpr (TAN) {
            mfma_s<F>(At, a, gTf[kk][X3_B[x]]);
            gap(std::integral_constant<int, N0>{});
          } else {
            mfma_s<F>(At, a, gTf[kk][X3_B[x]]);
            gap(std::integral_constant<int, N0>{});
            if constexpr (GO) {
              mfma_s<F>(dP, a, gOf[kk][X3_B[x]]);
              gap(std::integral_constant<int, N0 + 1>{});
            }
          }
        } else {
          mfma_s<F && !GO>(dP, a, gTf[kk][X3_B[x]]);
          gap(std::integral_constant<int, N0>{});
        }
      });
    });
    if constexpr (DUAL) tiles_ready(dP, At);
    else if constexpr (TAN) tiles_ready(At);
    else tiles_ready(dP);
    static_for<NU_DS>([&](auto uc) { unit_ds(std::integral_constant<int, 0>{}, uc); });
    __builtin_amdgcn_sched_barrier(0);
    // ---- dQ^T += K^T dS^T (+ K'^T dS'^T), the second half of dS behind the products of the first -------------
    static_for<2 * DB>([&](auto ic) {
      constexpr int i = decltype(ic)::value, c = i / DB, db = i % DB, sl = i % 2, MPS = DUAL ? 2 : 1;
      if constexpr (DUAL) x3_wait(ca[sl], cb[sl]);
      else x3_wait(ca[sl]);
      if constexpr (i + 1 < 2 * DB) read_col(std::integral_constant<int, i + 1>{});
      __builtin_amdgcn_sched_barrier(0);
      static_for<6>([&](auto xc) {
        constexpr int x = decltype(xc)::value, n = (db * 6 + x) * MPS;
        auto gap = [&](auto nc) {
          if constexpr (c == 0) x3_gap<decltype(nc)::value, DB * 6 * MPS, NU_DS, false>([&](auto uc) { unit_ds(std::integral_constant<int, 1>{}, uc); });
          else __builtin_amdgcn_sched_barrier(0);
        };
        mfma_acc(acc[db], x3_frag(ca[sl][X3_A[x]]), x3_frag(ds[c][X3_B[x]]));
        gap(std::integral_constant<int, n>{});
        if constexpr (DUAL) {
          mfma_acc(acc[db], x3_frag(cb[sl][X3_A[x]]), x3_frag(dt[c][X3_B[x]]));
          gap(std::integral_constant<int, n + 1>{});
        }
      });
    });
  };

  int j0 = tile_at(0), j1 = tile_at(1), j2 = tile_at(2);
  tiles.first(j0, j1, Lk, 1 < ntiles);
  auto step = [&](int t, auto LIMc) {
    tile(t, j0, j2, LIMc);
    j0 = j1, j1 = j2, j2 = tile_at(t + 3);
  };
  int t = 0;
  if constexpr (MASK == MASK_NONE) {  // the causal diagonal and the end form the tail of the walk
    int t_lim = Lk / BT;
    if (pr.causal) t_lim = min(t_lim, q0 / BT);
    t_lim -= walk.first;
    for (; t < min(t_lim, ntiles); ++t) step(t, std::false_type{});
    for (; t < ntiles; ++t) step(t, std::true_type{});
  } else {
    for (; t < ntiles; ++t) step(t, std::false_type{});
  }
  accs_ready(acc);
  float check = 0.f;  // not zero once an output is not finite
  if (qrow < L) {
    float *out = (split ? sp.part_q + (size_t)share.index * pr.Z * pr.H * L * D : reinterpret_cast<float *>(TAN ? p.dqt : p.dq)) + head + (size_t)qrow * D;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        float x8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x8[e] = acc[db][8 * hf + e] * pr.scale;
          check = __builtin_fmaf(x8[e], 0.f, check);
        }
        store8<float>(out + 32 * db + 16 * hf + 8 * g, x8);
      }
    }
  }
  return !x3_any(!(check == 0.f), lds0, wave, lane);
}

// dk, dv (PLAIN / DUAL) or dk', dv' (TANGENT).  Returns whether every output is finite.
template <int D, int MODE, int MASK, bool GO, bool DROP, bool SPLIT = false>
__device__ __forceinline__ bool bwd_f32x3_dkdv_body(const BwdParams &p, const int bid, const BwdSplit sp = {}, const int total = 0) {
  using C = X3Cfg<D>;
  constexpr bool DUAL = MODE == BWD_DUAL, TAN = MODE == BWD_TANGENT;
  constexpr int BT = C::BT, KK = D / 16, DB = D / 32, NTILE = DUAL ? 4 : 2;
  constexpr int NSTAT = DUAL ? 4 : 2, STATB = NSTAT * BT * 4;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;  // stage s: [Q | G | Q' | gT], three planes each; then two stages of statistics
  using Tiles = X3Tiles<D, NTILE, (DUAL && !GO) ? 1 : -1>;
  const uint32_t stat0 = lds0 + 2 * Tiles::STAGEB;

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
  bf16x8 Kf[KK][3], Vf[KK][3], Ktf[DUAL ? KK : 1][3], Vtf[DUAL ? KK : 1][3];
  const size_t own = kvhead + (size_t)kld * D;
  x3_own_row(Kf, p.k, own, g);
  x3_own_row(Vf, p.v, own, g);
  if constexpr (DUAL) {
    x3_own_row(Ktf, p.kt, own, g);
    x3_own_row(Vtf, p.vt, own, g);
  }
  f32x16 dK[DB], dV[DB];
  zero_accs(dK);
  zero_accs(dV);

  const float sl2 = pr.scale * LOG2E;
  const int istart = pr.causal ? (k0 / BT) * BT : 0;
  Tiles tiles;
  tiles.init(lds0, tid, lane);
  const uint32_t vzero = 0u;

  for (int gi = 0; gi < group; ++gi) {
    const int h = hk * (pr.H / pr.Hk) + group_share(pr, chunk) + gi;  // query head
    const size_t head = ((size_t)z * pr.H + h) * L * D, srow = ((size_t)z * pr.H + h) * L;
    {
      const float *qg = reinterpret_cast<const float *>(p.q) + head;
      const float *gt = (DUAL || TAN) ? reinterpret_cast<const float *>(p.gt) + head : nullptr;
      const float *t[4] = {qg, TAN ? gt : (GO ? reinterpret_cast<const float *>(p.go) + head : qg), DUAL ? reinterpret_cast<const float *>(p.qt) + head : nullptr, gt};
      tiles.tensors(wave, t);
    }
    // wave s brings statistic s of the tile's rows
    const float *st_p = nullptr;
    if (wave == 0) st_p = p.M + srow;
    else if (wave == 1) st_p = (MODE == BWD_PLAIN ? p.neg_d1 : DUAL ? p.mu : p.neg_a) + srow;
    else if (DUAL) st_p = (wave == 2 ? p.neg_a : p.neg_d2) + srow;
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
    float raw_stat = 0.f;
    auto load_stat = [&](int i) {  // (rows past the end: a log-sum-exp of plus infinity, so that their P is zero)
      if (wave < NSTAT && lane < BT) {
        raw_stat = st_p[min(i + lane, L - 1)];
        if (wave == 0 && i + lane >= L) raw_stat = __builtin_inff();
      }
    };
    auto store_stat = [&](int stage) {
      if (wave < NSTAT && lane < BT) *(JVPFA_LDS(float))(uintptr_t)(stat0 + stage * STATB + wave * BT * 4 + lane * 4) = raw_stat;
    };
    // mask entries of this lane's key against the 16 queries of its registers
    float mka[MASK == MASK_ADD ? 16 : 1];
    uint8_t mkb[MASK == MASK_BOOL ? 16 : 1];
    auto fetch_masks = [&](int in) {
      if constexpr (MASK != MASK_NONE) {
        const int64_t col = z * pr.ms[0] + h * pr.ms[1] + (int64_t)kld * pr.ms[3];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t off = col + (int64_t)min(in + 16 * (e / 8) + 8 * g + e % 8, L - 1) * pr.ms[2];
          if constexpr (MASK == MASK_ADD) mka[e] = reinterpret_cast<const float *>(pr.mask)[off];
          if constexpr (MASK == MASK_BOOL) mkb[e] = reinterpret_cast<const uint8_t *>(pr.mask)[off];
        }
      }
    };

    // One tile: its first query is i0, the next but one's in.
    auto tile = [&](int t, int i0, int i1, int in, auto LIMc) {
      x3_barrier();
      fetch_masks(i0);
      const uint32_t st = (t & 1) * Tiles::STAGEB, stn = ((t + 1) & 1) * Tiles::STAGEB;
      const uint32_t sta = stat0 + (t & 1) * STATB + 8 * g * 4;
      f32x16 S, Sp, dP, At;
      u32x4 fr[2][3];
      constexpr int NPAIR = DUAL ? 2 : 1, NS = KK * NPAIR;
      constexpr bool NOG = DUAL && !GO;
      // group 0: Q (S, S'), Q' (S'); group 1: G (dP), gT (A, dP).  PLAIN, TANGENT: Q; G
      auto read_row = [&](auto ic) {
        constexpr int i = decltype(ic)::value, G = i / NS, kk = (i % NS) / NPAIR, pair = i % NPAIR, T = G + 2 * pair;
        if constexpr (!(NOG && T == 1)) tiles.template rows<T>(fr[i % 2], kk, st);
      };
      constexpr int NST = Tiles::NU + 1;  // staging: half of it here, the rest with dK; then the statistics
      auto unit_st = [&](auto uc) {
        constexpr int u = decltype(uc)::value;
        if constexpr (u < Tiles::NU) {
          tiles.template unit<u>(stn, in, L, t + 2 < ntiles);
        } else {
          store_stat((t + 1) & 1);
          load_stat(in);
        }
      };
      constexpr int NST1 = DUAL ? NST / 2 : NST, NST4 = NST - NST1;
      // P (and S' - mu, P'): S and S' are overwritten; parts of P (and P')
      constexpr int UPP = DUAL ? 7 : 4, NU_P = 8 * UPP;
      f32x4 s0, s1, s2, s3;  // statistics of registers 4q .. 4q + 3 (queries 16 (q / 2) + 8g + 4 (q % 2) + 0..3)
      auto stat = [&](int q, int which) { return *(JVPFA_LDS(const f32x4))(uintptr_t)(sta + which * BT * 4 + (q / 2) * 64 + (q % 2) * 16); };
      const uint32_t drop_tile = DROP ? drop_row_word(pr, z * pr.H + h, i0) + drop_lane : 0u;  // 32 queries: one block of the pattern
      const int dist = i0 + 8 * g - krow;
      u32x4 pf[2][3], tf[2][3];
      float x1 = 0.f, a0 = 0.f, a1 = 0.f, b0 = 0.f, b1 = 0.f;
      auto kept = [&](auto ec) { return drop_scale_of(pr, drop_tile + (uint32_t)(16 * (decltype(ec)::value / 8) + decltype(ec)::value % 8) * DROP_C_ROW); };
      auto unit_p = [&](auto uc) {
        constexpr int u = decltype(uc)::value, q = u / UPP, s = u % UPP, e = 2 * q, c = e / 8, w = (e % 8) / 2, i = e % 4;
        auto arg = [&](auto ec) {
          constexpr int y = decltype(ec)::value;
          float m = -s0[y % 4];
          if constexpr (MASK == MASK_ADD) m = __builtin_fmaf(mka[y], LOG2E, m);
          float x = __builtin_fmaf(S[y], sl2, m);
          if constexpr (MASK == MASK_BOOL) x = mkb[y] != 0 ? x : -__builtin_inff();
          if constexpr (decltype(LIMc)::value) x = (dist >= -(16 * (y / 8) + y % 8)) ? x : -__builtin_inff();
          return x;
        };
        if constexpr (s == 0) {
          if constexpr (i == 0) {
            s0 = stat(e / 4, 0);
            if constexpr (DUAL) s1 = stat(e / 4, 1);
          }
          const float x0 = arg(std::integral_constant<int, e>{});
          x1 = arg(std::integral_constant<int, e + 1>{});
          S[e] = fast_exp2(x0);
          anchor(x1);
          anchor(S[e]);
        } else if constexpr (s == 1) {
          S[e + 1] = fast_exp2(x1);
          if constexpr (DUAL) {
            Sp[e] = __builtin_fmaf(Sp[e], pr.scale, -s1[i]);
            Sp[e + 1] = __builtin_fmaf(Sp[e + 1], pr.scale, -s1[i + 1]);
            anchor(Sp[e + 1]);
          }
          anchor(S[e + 1]);
        } else if constexpr (s == 2) {
          a0 = S[e], a1 = S[e + 1];
          if constexpr (DROP) a0 *= kept(std::integral_constant<int, e>{}), a1 *= kept(std::integral_constant<int, e + 1>{});
          if constexpr (DUAL) {
            b0 = a0 * Sp[e], b1 = a1 * Sp[e + 1];
            anchor(b0), anchor(b1);
          }
          pf[c][0][w] = x3_take(a0, a1);
          anchor(a0), anchor(a1);
        } else if constexpr (s == 3) {
          pf[c][1][w] = x3_take(a0, a1);
          pf[c][2][w] = x3_last(a0, a1);
          anchor(pf[c][2][w]);
        } else if constexpr (s == 4) {
          tf[c][0][w] = x3_take(b0, b1);
          anchor(b0), anchor(b1);
        } else if constexpr (s == 5) {
          tf[c][1][w] = x3_take(b0, b1);
          anchor(b0), anchor(b1);
        } else {
          tf[c][2][w] = x3_last(b0, b1);
          anchor(tf[c][2][w]);
        }
      };
      // dS (and dS') in parts
      constexpr int UPD = DUAL ? 5 : 3, NU_DS = 8 * UPD;
      u32x4 ds[2][3], dt[2][3];
      auto unit_ds = [&](auto uc) {
        constexpr int u = decltype(uc)::value, q = u / UPD, s = u % UPD, e = 2 * q, c = e / 8, w = (e % 8) / 2, i = e % 4;
        if constexpr (s == 0) {
          if constexpr (i == 0) {
            s2 = stat(e / 4, DUAL ? 2 : 1);
            if constexpr (DUAL) s3 = stat(e / 4, 3);
          }
          auto one = [&](auto ec, float &a, float &b) {
            constexpr int y = decltype(ec)::value;
            if constexpr (DROP) {
              const float ks = kept(ec);
              if constexpr (!TAN) dP[y] *= ks;
              if constexpr (DUAL || TAN) At[y] *= ks;
            }
            if constexpr (MODE == BWD_PLAIN) {
              a = S[y] * (dP[y] + s2[y % 4]);
            } else if constexpr (DUAL) {
              const float am = At[y] + s2[y % 4];
              b = S[y] * am;
              a = S[y] * __builtin_fmaf(am, Sp[y], dP[y] + s3[y % 4]);
              anchor(b);
            } else {
              a = S[y] * (At[y] + s2[y % 4]);
            }
            anchor(a);
          };
          one(std::integral_constant<int, e>{}, a0, b0);
          one(std::integral_constant<int, e + 1>{}, a1, b1);
        } else if constexpr (s == 1) {
          ds[c][0][w] = x3_take(a0, a1);
          anchor(a0), anchor(a1);
        } else if constexpr (s == 2) {
          ds[c][1][w] = x3_take(a0, a1);
          ds[c][2][w] = x3_last(a0, a1);
          anchor(ds[c][2][w]);
        } else if constexpr (s == 3) {
          dt[c][0][w] = x3_take(b0, b1);
          anchor(b0), anchor(b1);
        } else {
          dt[c][1][w] = x3_take(b0, b1);
          dt[c][2][w] = x3_last(b0, b1);
          anchor(dt[c][2][w]);
        }
      };
      // column fragments, step i: (chunk c, block db) of G (and gT), then of Q (and Q')
      u32x2 ca[2][3][2], cb[2][3][2];
      auto read_col = [&](auto ic) {
        constexpr int i = decltype(ic)::value, G = i / (2 * DB), c = i % (2 * DB) / DB, db = i % DB;
        if constexpr (!(NOG && G == 0)) tiles.template cols<G == 0 ? 1 : 0, c>(ca[i % 2], db, st);
        if constexpr (DUAL) tiles.template cols<G == 0 ? 3 : 2, c>(cb[i % 2], db, st);
      };

      read_row(std::integral_constant<int, 0>{});
      static_for<2 * NS>([&](auto ic) {
        constexpr int i = decltype(ic)::value, G = i / NS, kk = (i % NS) / NPAIR, pair = i % NPAIR, sl = i % 2;
        constexpr bool ABSENT = NOG && G == 1 && pair == 0;
        if constexpr (!ABSENT) x3_wait(fr[sl]);
        if constexpr (i + 1 < 2 * NS) read_row(std::integral_constant<int, i + 1>{});
        else read_col(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        static_for<6>([&](auto xc) {
          constexpr int x = decltype(xc)::value;
          constexpr bool F = kk == 0 && x == 0;
          const bf16x8 a = x3_frag(fr[sl][X3_A[x]]);
          // products of a step: group 0: two by Q, one by Q'; group 1: one by G (if there is one), two by gT
          constexpr int N1ST = !DUAL ? 1 : G == 0 ? 2 : GO ? 1 : 0, N2ND = !DUAL ? 0 : G == 0 ? 1 : 2, PER = 6 * (N1ST + N2ND);
          constexpr int N0 = kk * PER + (pair == 0 ? x * N1ST : 6 * N1ST + x * N2ND);
          auto gap = [&](auto nc) {
            if constexpr (G == 0) x3_gap<decltype(nc)::value, KK * PER, NST1, false>(unit_st);
            else x3_gap<decltype(nc)::value, KK * PER, NU_P, true>(unit_p);
          };
          if constexpr (G == 0) {
            if constexpr (pair == 0) {
              if constexpr (DUAL) {
                mfma_s<F>(Sp, a, Ktf[kk][X3_B[x]]);
                gap(std::integral_constant<int, N0>{});
                mfma_s<F>(S, a, Kf[kk][X3_B[x]]);
                gap(std::integral_constant<int, N0 + 1>{});
              } else {
                mfma_s<F>(S, a, Kf[kk][X3_B[x]]);
                gap(std::integral_constant<int, N0>{});
              }
            } else {
              mfma_s<false>(Sp, a, Kf[kk][X3_B[x]]);
              gap(std::integral_constant<int, N0>{});
            }
          } else if constexpr (pair == 0) {
            if constexpr (TAN) mfma_s<F>(At, a, Vf[kk][X3_B[x]]);
            else if constexpr (!NOG) mfma_s<F>(dP, a, Vf[kk][X3_B[x]]);
            if constexpr (!NOG) gap(std::integral_constant<int, N0>{});
          } else {
            mfma_s<F>(At, a, Vf[kk][X3_B[x]]);
            gap(std::integral_constant<int, N0>{});
            mfma_s<F && NOG>(dP, a, Vtf[kk][X3_B[x]]);
            gap(std::integral_constant<int, N0 + 1>{});
          }
        });
      });
      if constexpr (DUAL) tiles_ready(dP, At);
      else if constexpr (TAN) tiles_ready(At);
      else tiles_ready(dP);
      // ---- dV^T += G^T P (+ gT^T P'), with dS; dK^T += Q^T dS (+ Q'^T dS'), with the rest of the staging -------
      static_for<4 * DB>([&](auto ic) {
        constexpr int i = decltype(ic)::value, G = i / (2 * DB), ii = i % (2 * DB), c = ii / DB, db = i % DB, sl = i % 2, MPS = DUAL && !(NOG && G == 0) ? 2 : 1;
        if constexpr (NOG && G == 0) x3_wait(cb[sl]);
        else if constexpr (DUAL) x3_wait(ca[sl], cb[sl]);
        else x3_wait(ca[sl]);
        if constexpr (i + 1 < 4 * DB) read_col(std::integral_constant<int, i + 1>{});
        __builtin_amdgcn_sched_barrier(0);
        static_for<6>([&](auto xc) {
          constexpr int x = decltype(xc)::value, n = (ii * 6 + x) * MPS, NG = 2 * DB * 6 * MPS;
          auto gap = [&](auto nc) {
            if constexpr (G == 0) x3_gap<decltype(nc)::value, NG, NU_DS, false>(unit_ds);
            else x3_gap<decltype(nc)::value, NG, NST4, false>([&](auto uc) { unit_st(std::integral_constant<int, NST1 + decltype(uc)::value>{}); });
          };
          if constexpr (G == 0) {
            if constexpr (!NOG) {
              mfma_acc(dV[db], x3_frag(ca[sl][X3_A[x]]), x3_frag(pf[c][X3_B[x]]));
              gap(std::integral_constant<int, n>{});
            }
            if constexpr (DUAL) {
              mfma_acc(dV[db], x3_frag(cb[sl][X3_A[x]]), x3_frag(tf[c][X3_B[x]]));
              gap(std::integral_constant<int, n + (NOG ? 0 : 1)>{});
            }
          } else {
            mfma_acc(dK[db], x3_frag(ca[sl][X3_A[x]]), x3_frag(ds[c][X3_B[x]]));
            gap(std::integral_constant<int, n>{});
            if constexpr (DUAL) {
              mfma_acc(dK[db], x3_frag(cb[sl][X3_A[x]]), x3_frag(dt[c][X3_B[x]]));
              gap(std::integral_constant<int, n + 1>{});
            }
          }
        });
      });
    };

    if (gi > 0) x3_barrier();  // every wave is done with the previous head's last tile
    int i0 = tile_at(0), i1 = tile_at(1), i2 = tile_at(2);
    if (ntiles > 0) {
      load_stat(i0);
      tiles.first(i0, i1, L, 1 < ntiles);
      store_stat(0);
      load_stat(i1);
    }
    auto step = [&](int t, auto LIMc) {
      tile(t, i0, i1, i2, LIMc);
      i0 = i1, i1 = i2, i2 = tile_at(t + 3);
    };
    int t = 0;
    if constexpr (MASK == MASK_NONE) {  // the tiles of the causal diagonal come first
      const int t_lim = pr.causal ? min(C::BLK / BT - walk.first, ntiles) : 0;
      for (; t < t_lim; ++t) step(t, std::true_type{});
    }
    for (; t < ntiles; ++t) step(t, std::false_type{});
  }
  accs_ready(dK, dV);
  float check = 0.f;  // not zero once an output is not finite
  if (krow < Lk) {
    const size_t elems = (size_t)pr.Z * pr.Hk * Lk * D;
    float *partk = split ? sp.part_k + share.index * 2 * elems : kv_part(pr, D, 2, 0, chunk), *partv = split ? partk + elems : kv_part(pr, D, 2, 1, chunk);
    const size_t off = kvhead + (size_t)krow * D;
    float *outk = (partk ? partk : reinterpret_cast<float *>(TAN ? p.dkt : p.dk)) + off;
    float *outv = (partv ? partv : reinterpret_cast<float *>(TAN ? p.dvt : p.dv)) + off;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        float k8[8], v8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          k8[e] = dK[db][8 * hf + e] * pr.scale;
          v8[e] = dV[db][8 * hf + e];
          check = __builtin_fmaf(k8[e], 0.f, check);
          check = __builtin_fmaf(v8[e], 0.f, check);
        }
        store8<float>(outk + 32 * db + 16 * hf + 8 * g, k8);
        store8<float>(outv + 32 * db + 16 * hf + 8 * g, v8);
      }
    }
  }
  return !x3_any(!(check == 0.f), lds0, wave, lane);
}
#endif

template <int D, int MODE> struct BwdX3Lds {
  static constexpr size_t DQ = 2 * (MODE == BWD_DUAL ? 4 : 2) * (size_t)X3Cfg<D>::OPB;  // (more than the fp32 tiles and statistics take)
  static constexpr size_t DKV = DQ + 2 * (MODE == BWD_DUAL ? 4 : 2) * X3Cfg<D>::BT * 4;
};
template <int D, int MODE, int MASK, bool GO, bool DROP = false, int WGS = MODE != BWD_DUAL && !DROP ? 2 : 1>
__global__ __launch_bounds__(256, WGS) void bwd_f32x3_dq_kernel(const BwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (!bwd_f32x3_dq_body<D, MODE, MASK, GO, DROP>(p, blockIdx.x)) bwd_f32_dq_body<D, MODE, MASK, GO, DROP>(p, blockIdx.x);
#endif
}
template <int D, int MODE, int MASK, bool GO, bool DROP = false>
__global__ __launch_bounds__(256, 1) void bwd_f32x3_dkdv_kernel(const BwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (!bwd_f32x3_dkdv_body<D, MODE, MASK, GO, DROP>(p, blockIdx.x)) bwd_f32_dkdv_body<D, MODE, MASK, GO, DROP>(p, blockIdx.x);
#endif
}

// Both roles in one launch (see bwd2_both_kernel): the first kv_blocks workgroups are dk/dv workgroups.  SPLIT: blocks' tiles split
// (split.hpp), compiled apart: what it needs takes 15 - 80 scalar registers that the others' loops have to spill (B2 H6 L777 D64 first
// order with a bias, whose rows are not aligned: 124 -> 159 us).
template <int D, int MODE, int MASK, bool GO, bool SPLIT>
__global__ __launch_bounds__(256, 1) void bwd_f32x3_both_kernel(const BwdParams p, const BwdSplit sp, const int kv_blocks) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int b = __builtin_amdgcn_readfirstlane(blockIdx.x);
  if (b < kv_blocks) {
    if (!bwd_f32x3_dkdv_body<D, MODE, MASK, GO, false, SPLIT>(p, b, sp, kv_blocks)) bwd_f32_dkdv_body<D, MODE, MASK, GO, false, SPLIT>(p, b, sp, kv_blocks);
  } else {
    if (!bwd_f32x3_dq_body<D, MODE, MASK, GO, false, SPLIT>(p, b - kv_blocks, sp, gridDim.x - kv_blocks)) bwd_f32_dq_body<D, MODE, MASK, GO, false, SPLIT>(p, b - kv_blocks, sp, gridDim.x - kv_blocks);
  }
#endif
}

}  // namespace jvpfa
