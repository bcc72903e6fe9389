// Fused dual forward for fp32, D in {32, 64}, on the 16-bit matrix instructions.
//
// An fp32 matrix instruction does 1/16 of the work of a bf16 one in the same time, and fwd_kernel_f32.hpp keeps the fp32
// ones busy for 80 - 85 % of its time: what is left to gain is the rate itself.  An fp32 value x is the sum of three bf16
// values, h = bf16(x), m = bf16(x - h), l = bf16(x - h - m) (both differences are exact; 27 bits with the signs; for |x| from 2^-108 on:
// below it l is subnormal and its last bits are lost), so
//     x y = l h' + h l' + m m' + m h' + h m' + h h'     (left out: m l' + l m' + l l', below 2^-26 of the product)
// is six bf16 products with fp32 accumulation: 6 x 32 cycles for 32x32x16 where the fp32 instructions take 8 x 64.
// How the sums are formed keeps the error below that of the fp32 instructions.  The matrix cores cut off what a product has
// below the last place of the accumulator, so the small products go first where the contraction is short (the scores), and
// into accumulators of their own where it runs over all keys; and parts are rounded to nearest, so that what is cut off has either
// sign.  Relative error (2-norm) of one product against 64 bits, normal operands, fp32 instructions / parts in one accumulator
// / in two: contraction 64: 1.4e-7 / 1.1e-7 / 5.0e-8; 8192: 1.6e-6 / 1.4e-6 / 5.6e-7, terms of one sign 1.2e-6 / 7.7e-7 / 4.3e-7.
//
// Infinities (inf = inf + nan + nan) and values that round to one are the exception: an output that is not finite makes
// its workgroup start over with the fp32 instructions, so that every result that is not finite is theirs.
//
// Work split and softmax as in fwd_kernel_f32.hpp (4 waves = 128 query rows, 32-key tiles, scores transposed, lane = query).
// Measured, dual forward at B4 H8 L1024 D64, kernel alone: key padding 201 -> 122 us, bias per head 206 -> 132 us (6 x 25.8
// GFLOP in 16 bits: 1.2 PFLOP/s).  What bounds it: one wave per SIMD, which pays for most of its 430 vector instructions
// beside 144 matrix instructions a tile.
// Q, Q' stay resident as parts.  K, V, K', V' tiles go global -> registers (a tile ahead) -> three bf16 planes each in LDS;
// splitting there costs a tile's share of every lane once, not every wave once.  A wave hides its vector work itself, one
// unit of it behind each matrix instruction, in two phases per tile t with one barrier:
//     A: scores of tile t + 1          with   exponentials, row sums and splitting of P, P S' of tile t
//     B: accumulation of tile t        with   logits and row maximum of tile t + 1, splitting of K (t + 2), V (t + 1)
#pragma once
#include "fwd_kernel_f32.hpp"
#include "fwd_kernel_v3.hpp"

namespace jvpfa {

template <int D> struct X3Cfg {
  static constexpr int NT = 4 * WAVE, BLK = 128, BT = 32;
  static constexpr int CH = D / 8, ROWB = 2 * D, PLANE = BT * ROWB, OPB = 3 * PLANE;  // a tile: three planes of bf16 rows
  static constexpr int TASKS = BT * CH;  // of staging a tile: eight consecutive elements each
};
// The two factors of product x (0 h, 1 m, 2 l), smallest products first.
constexpr int X3_A[6] = {2, 0, 1, 1, 0, 0}, X3_B[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ void anchor(const uint32_t &x) { asm volatile("" : : "v"(x)); }
// h and the exact rest of two values, packed (rest in place)
__device__ __forceinline__ uint32_t x3_take(float &a, float &b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  const uint32_t w = __builtin_bit_cast(uint32_t, v);
  a -= __uint_as_float(__builtin_amdgcn_perm(w, 0u, 0x05040c0cu));  // w << 16 (which the compiler would convert for again)
  b -= __uint_as_float(w & 0xffff0000u);
  return w;
}
__device__ __forceinline__ uint32_t x3_last(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
// Eight values of a lane as a fragment of each part.
__device__ __forceinline__ void x3_split8(const f32x4 &lo, const f32x4 &hi, u32x4 (&f)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = i < 2 ? lo[2 * i] : hi[2 * i - 4], b = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
    f[0][i] = x3_take(a, b);
    f[1][i] = x3_take(a, b);
    f[2][i] = x3_last(a, b);
  }
}

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ void x3_wait(u32x4 (&a)[3]) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])); }
__device__ __forceinline__ void x3_wait(u32x4 (&a)[3], u32x4 (&b)[3]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]));
}
__device__ __forceinline__ void x3_wait(u32x2 (&a)[3][2]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0][0]), "+v"(a[0][1]), "+v"(a[1][0]), "+v"(a[1][1]), "+v"(a[2][0]), "+v"(a[2][1]));
}
__device__ __forceinline__ void x3_wait(u32x2 (&a)[3][2], u32x2 (&b)[3][2]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0][0]), "+v"(a[0][1]), "+v"(a[1][0]), "+v"(a[1][1]), "+v"(a[2][0]), "+v"(a[2][1]),
               "+v"(b[0][0]), "+v"(b[0][1]), "+v"(b[1][0]), "+v"(b[1][1]), "+v"(b[2][0]), "+v"(b[2][1]));
}
__device__ __forceinline__ bf16x8 x3_frag(const u32x4 &a) { return __builtin_bit_cast(bf16x8, a); }
__device__ __forceinline__ bf16x8 x3_frag(const u32x2 (&a)[2]) {
  const u32x4 v = {a[0][0], a[0][1], a[1][0], a[1][1]};
  return __builtin_bit_cast(bf16x8, v);
}
// this wave's LDS writes have landed, and every wave's
__device__ __forceinline__ void x3_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }
// Some lane of the workgroup says so (uses the first words of the LDS, which nothing else may be using).
__device__ __forceinline__ bool x3_any(bool mine, uint32_t lds0, int wave, int lane) {
  x3_barrier();
  const bool any = __any(mine);
  JVPFA_LDS(uint32_t) w = (JVPFA_LDS(uint32_t))(uintptr_t)lds0;
  if (lane == 0) w[wave] = any ? 1u : 0u;
  x3_barrier();
  const bool all = (w[0] | w[1] | w[2] | w[3]) != 0;
  x3_barrier();
  return __builtin_amdgcn_readfirstlane(all ? 1 : 0) != 0;
}

// A bias is loaded as vectors from rows that start anywhere (an address that is a multiple of 4 is enough for one); element by element
// the plain kernel at D = 32 spent most of its time on it: B1 H24 L577 81 -> 27 us (fp32 instructions with such loads: 52).
template <int MASK> __device__ __forceinline__ bool x3_mask_rows(const Problem &pr) {
  if constexpr (MASK == MASK_ADD) return pr.ms[3] == 1 && (reinterpret_cast<uintptr_t>(pr.mask) & 3) == 0;
  else return mask_rows_aligned<float, MASK>(pr);
}
template <int MASK> __device__ __forceinline__ MaskAhead<float, MASK> x3_mask_fetch8(const Problem &pr, int64_t rowoff, int key0) {
  if constexpr (MASK == MASK_ADD) {
    typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
    const f32x4_any *src = reinterpret_cast<const f32x4_any *>(reinterpret_cast<const float *>(pr.mask) + rowoff + key0);
    const f32x4 lo = src[0], hi = src[1];
    MaskAhead<float, MASK> m;
#pragma unroll
    for (int e = 0; e < 4; ++e) m.f[e] = lo[e], m.f[e + 4] = hi[e];
    return m;
  } else {
    return mask_fetch8<float, MASK>(pr, rowoff, key0);
  }
}

// Returns whether every output is finite.
template <int D, bool DUAL, int MASK, bool DROP, bool SPLIT>
__device__ __forceinline__ bool fwd_f32x3_body(const FwdParams &p) {
  using C = X3Cfg<D>;
  constexpr int BT = C::BT, CH = C::CH, ROWB = C::ROWB, PLANE = C::PLANE, OPB = C::OPB;
  constexpr int KK = D / 16, DB = D / 32, NK = DUAL ? 2 : 1, STAGEB = NK * OPB;  // tiles of one kind (K, K' or V, V')
  constexpr float NEG_INF = -__builtin_inff(), TAU = 8.f;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;  // [K | K'] twice, then [V | V'] twice

  const Problem &pr = p.pr;
  const int L = pr.L, Lk = pr.Lk;
  const int nqb = (L + C::BLK - 1) / C::BLK;
  // SPLIT, small grids: the key tiles of query blocks are split over workgroups (see split.hpp)
  const Dealt share = SPLIT ? deal_query_block({pr.chunks, pr.chunk_tiles, 0, nqb}, blockIdx.x, gridDim.x, nqb, pr.Z * pr.H, pr.causal != 0, more_than_units(gridDim.x, pr.units))
                            : Dealt{xcd_remap(blockIdx.x, nqb, pr.Z * pr.H, pr.causal != 0), 1, 0};
  const bool split = SPLIT && share.count > 1;
  const int zh = share.id / nqb;
  const int qb = pr.causal ? nqb - 1 - share.id % nqb : share.id % nqb;  // causal: the longest key loops first
  const int z = zh / pr.H, h = zh % pr.H;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int r = lane % 32, g = lane / 32, pr32 = perm32(r);

  const size_t head = (size_t)zh * L * D;
  const size_t kvhead = ((size_t)z * pr.Hk + h / (pr.H / pr.Hk)) * Lk * D;  // grouped heads share K, V
  const float *Kg = reinterpret_cast<const float *>(p.k) + kvhead, *Vg = reinterpret_cast<const float *>(p.v) + kvhead;
  const float *Ktg = DUAL ? reinterpret_cast<const float *>(p.kt) + kvhead : nullptr;
  const float *Vtg = DUAL ? reinterpret_cast<const float *>(p.vt) + kvhead : nullptr;
  const int q0 = qb * C::BLK, qrow = q0 + wave * 32 + r, qld = qrow < L ? qrow : L - 1;

  // ---- Q, Q' as parts, resident in the accumulation file ---------------------------------------------------
  bf16x8 Qf[KK][3], Qtf[DUAL ? KK : 1][3];
  auto own_row = [&](bf16x8(&f)[3], const void *base, int kk) {
    const float *src = reinterpret_cast<const float *>(base) + head + (size_t)qld * D + 16 * kk + 8 * g;
    u32x4 x[3];
    x3_split8(*reinterpret_cast<const f32x4 *>(src), *reinterpret_cast<const f32x4 *>(src + 4), x);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      f[i] = x3_frag(x[i]);
      pin_acc(f[i]);
    }
  };
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    own_row(Qf[kk], p.q, kk);
    if constexpr (DUAL) own_row(Qtf[kk], p.qt, kk);
  }
  // accumulators: h h' products, and all others
  f32x16 Oacc[DB], Olow[DB], Tacc[DUAL ? DB : 1], Tlow[DUAL ? DB : 1];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      Oacc[db][e] = Olow[db][e] = 0.f;
      if constexpr (DUAL) Tacc[db][e] = Tlow[db][e] = 0.f;
    }
    pin_acc(Oacc[db]), pin_acc(Olow[db]);
    if constexpr (DUAL) pin_acc(Tacc[db]), pin_acc(Tlow[db]);
  }
  float m_i = NEG_INF, l_i = 0.f, mu_i = 0.f;  // l_i, mu_i: this lane's keys

  const float sl2 = pr.scale * LOG2E;
  const int64_t mrow = MASK != MASK_NONE ? z * pr.ms[0] + h * pr.ms[1] + (int64_t)qld * pr.ms[2] : 0;
  const uint32_t drop_row = DROP ? drop_row_word(pr, zh, qld) : 0u;
  bool mask_al = false;
  if constexpr (MASK != MASK_NONE) mask_al = x3_mask_rows<MASK>(pr);
  int kend = pr.causal ? min(Lk, q0 + C::BLK) : Lk;
  TileWalk<BT> walk;  // key tiles visited: up to kend, or the caller's list of those that hold an attended entry
  {
    const int *tl = nullptr;
    if constexpr (MASK != MASK_NONE) {
      if (pr.klimit) kend = min(kend, max(pr.klimit[z], 1));
      if (pr.tiles_q) tl = pr.tiles_q + tile_list_offset_q(pr, z, h, qb);
    }
    const int whole = ((pr.causal ? min(Lk, q0 + C::BLK) : Lk) + TILE_W - 1) / TILE_W;
    walk.init(tl, 0, kend, Lk);
    if (split) walk.take(share.index, share.count, whole);
  }
  const int ntiles = __builtin_amdgcn_readfirstlane(walk.n);
  // partial results of a share: [share][row][O | T][D], then [share][row][m, l, mu_acc, c]
  const size_t nrows = (size_t)pr.Z * pr.H * L, prow = (size_t)share.index * nrows + (size_t)zh * L + qrow;
  float *part_stat = pr.part + (size_t)pr.chunks * nrows * ((DUAL ? 2 : 1) * D) + prow * 4;
  if (split && ntiles <= 0) {  // none of its tiles is visited: it weighs nothing
    if (qrow < L && g == 0) *reinterpret_cast<f32x4 *>(part_stat) = f32x4{NEG_INF, -0.f, 0.f, 0.f};
    return true;
  }
  auto tile_at = [&](int it) { return __builtin_amdgcn_readfirstlane(walk.at(min(it, max(ntiles - 1, 0)))); };

  // ---- staging: task i of a lane is eight consecutive elements of a row of tensor op (K, K', V, V') --------
  constexpr int NTASK = 2 * NK * C::TASKS / C::NT;
  static_assert(C::TASKS == C::NT || 2 * C::TASKS == C::NT, "the tensor of a task is the same in every lane of a wave");
  const uint32_t st_src = (tid % C::TASKS) * 32;
  uint32_t st_dst[NTASK];
  const float *st_base[NTASK];
  bool st_v[NTASK];  // V or V'
#pragma unroll
  for (int i = 0; i < NTASK; ++i) {
    const int op = C::TASKS == C::NT ? i : 2 * i + wave / 2, row = (tid % C::TASKS) / CH, ch = tid % CH;
    st_v[i] = op >= NK;
    st_base[i] = op == 0 ? Kg : op == NK ? Vg : op == 1 ? Ktg : Vtg;
    st_dst[i] = lds0 + (st_v[i] ? 2 * STAGEB + (op - NK) * OPB : op * OPB) + row * ROWB + ((ch ^ (st_v[i] ? swz_v<CH>(row) : swz_k<CH>(row))) * 16);
  }
  f32x4 raw[NTASK][2];
  auto load_raw = [&](int i, int jk, bool k_on, int jv, bool v_on) {  // (rows past the end, and tiles that do not exist: zeros)
    const int j = st_v[i] ? jv : jk, rows = (st_v[i] ? v_on : k_on) ? Lk - j : 0;
    const int bytes = __builtin_amdgcn_readfirstlane(min(max(rows, 0), BT) * (D * 4));  // (the compiler clamps in the vector unit)
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)(st_base[i] + (size_t)j * D), 0, bytes, 0x00020000);
    raw[i][0] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, st_src, 0, 0));
    raw[i][1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, st_src + 16, 0, 0));
  };
  u32x4 sp[3];  // the task being split
  float sa = 0.f, sb = 0.f;
  auto store_parts = [&](int i, int kpar, int vpar) {
    const uint32_t a = st_dst[i] + (st_v[i] ? vpar : kpar) * STAGEB;
#pragma unroll
    for (int x = 0; x < 3; ++x) *(JVPFA_LDS(u32x4))(uintptr_t)(a + x * PLANE) = sp[x];
  };

  // ---- fragment reads (see fwd_kernel_v3.hpp) ----------------------------------------------------------------
  uint32_t koff[KK], voff[DB];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) koff[kk] = lds0 + pr32 * ROWB + (((2 * kk + g) ^ swz_k<CH>(pr32)) * 16);
  // (rows 4 further down, for the second read: CH = 8, 4 use only row bits 0 - 1 for the V-type swizzle)
  {
    const int a = (lane >> 4) & 1, j = lane & 15;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int row = 8 * g + (j >> 2);
      voff[db] = lds0 + 2 * STAGEB + row * ROWB + (((4 * db + 2 * a + (j & 1)) ^ swz_v<CH>(row)) * 16) + 8 * ((j >> 1) & 1);
    }
  }
  u32x4 ka[2][3], kb[2][3];
  auto issue_k = [&](auto kc, uint32_t stage) {
    constexpr int kk = decltype(kc)::value;
    const uint32_t a = koff[kk] + stage;
    static_for<3>([&](auto xc) { ka[kk % 2][decltype(xc)::value] = lds_b128<decltype(xc)::value * PLANE>(a); });
    if constexpr (DUAL) static_for<3>([&](auto xc) { kb[kk % 2][decltype(xc)::value] = lds_b128<OPB + decltype(xc)::value * PLANE>(a); });
  };
  u32x2 va[2][3][2], vb[2][3][2];
  auto issue_v = [&](auto ic, uint32_t stage) {
    constexpr int i = decltype(ic)::value, c = i / DB, db = i % DB, O = c * 16 * ROWB;
    const uint32_t a = voff[db] + stage;
    static_for<3>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      va[i % 2][x][0] = lds_tr64<O + x * PLANE>(a);
      va[i % 2][x][1] = lds_tr64<O + x * PLANE + 4 * ROWB>(a);
      if constexpr (DUAL) {
        vb[i % 2][x][0] = lds_tr64<O + OPB + x * PLANE>(a);
        vb[i % 2][x][1] = lds_tr64<O + OPB + x * PLANE + 4 * ROWB>(a);
      }
    });
  };

  // ---- vector work in units -------------------------------------------------------------------------------------
  f32x16 Sn, Spn;        // scores as the matrix instructions leave them
  float sc[16], spc[16];  // logits (log2 domain) and scaled S' of the tile whose softmax is next
  u32x4 pf[2][3], tf[2][3];  // P and P S' as parts: [keys 16 c + 8 g ..][part], entry e = 8 c + j
  MaskAhead<float, MASK> mk[2];
  auto fetch_masks = [&](int jn) {  // (keys past the end come masked)
    if constexpr (MASK != MASK_NONE) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
        mk[c] = (mask_al && jn + BT <= Lk) ? x3_mask_fetch8<MASK>(pr, mrow, jn + 16 * c + 8 * g) : mask_fetch8_lim<float, MASK>(pr, mrow, jn + 16 * c + 8 * g);
    }
  };
  const int klim = min(pr.causal ? qrow : 0x7fffffff, Lk - 1);
  const uint32_t vzero = 0u, vninf = 0xff800000u;
  float mx = NEG_INF, alpha = 1.f, m_use = 0.f, rs = 0.f, rmu = 0.f;
  bool any_up = false;
  // softmax of the tile at jh: per pair of entries 3 units, and 2 for each of the operands split
  constexpr int UPP = DUAL ? 7 : 5, NU_SM = 8 * UPP + 1;
  float pv0 = 0.f, pv1 = 0.f, ps0 = 0.f, ps1 = 0.f;
  auto unit_sm = [&](auto uc, int jh) {
    constexpr int u = decltype(uc)::value, q = u / UPP, s = u % UPP;
    if constexpr (q < 8) {
      constexpr int e = 2 * q, c = e / 8, w = (e % 8) / 2;
      if constexpr (s == 0) {
        pv0 = fast_exp2(sc[e] - m_use);
        ps1 = sc[e + 1] - m_use;
        anchor(pv0);
        anchor(ps1);
      } else if constexpr (s == 1) {
        pv1 = fast_exp2(ps1);
        if constexpr (DUAL) ps0 = pv0 * spc[e];
        rs += pv0;
        anchor(pv1);
        anchor(rs);
      } else if constexpr (s == 2) {
        if constexpr (DUAL) {
          rmu += ps0;
          ps1 = pv1 * spc[e + 1];
          rmu += ps1;
          anchor(rmu);
        }
        rs += pv1;
        anchor(rs);
        if constexpr (DROP) {  // the row sums are those of the full softmax
          const float k0 = drop_scale_of(pr, drop_row + (uint32_t)(jh + 16 * c + 8 * g + e % 8) * DROP_C_KEY);
          const float k1 = drop_scale_of(pr, drop_row + (uint32_t)(jh + 16 * c + 8 * g + e % 8 + 1) * DROP_C_KEY);
          pv0 *= k0, pv1 *= k1;
          if constexpr (DUAL) ps0 *= k0, ps1 *= k1;
          anchor(pv1);
        }
      } else if constexpr (s == 3) {
        pf[c][0][w] = x3_take(pv0, pv1);
        anchor(pv0), anchor(pv1);
      } else if constexpr (s == 4) {
        pf[c][1][w] = x3_take(pv0, pv1);
        pf[c][2][w] = x3_last(pv0, pv1);
        anchor(pf[c][2][w]);
      } else if constexpr (s == 5) {
        tf[c][0][w] = x3_take(ps0, ps1);
        anchor(ps0), anchor(ps1);
      } else {
        tf[c][1][w] = x3_take(ps0, ps1);
        tf[c][2][w] = x3_last(ps0, ps1);
        anchor(tf[c][2][w]);
      }
    } else {
      l_i += rs;
      if constexpr (DUAL) mu_i += rmu;
      rs = rmu = 0.f;
    }
  };
  // logits and reference point of the tile whose scores are in Sn, Spn: 8 units of two entries, and one
  constexpr int NU_FR = 9;
  auto unit_fr = [&](auto uc, auto LIMc, int jh) {
    constexpr int u = decltype(uc)::value;
    if constexpr (u < 8) {
      static_for<2>([&](auto ec) {
        constexpr int e = 2 * u + decltype(ec)::value;
        float s;
        if constexpr (MASK == MASK_ADD) s = __builtin_fmaf(Sn[e], sl2, mk[e / 8].f[e % 8] * LOG2E);
        else if constexpr (MASK == MASK_BOOL)
          s = __builtin_fmaf(Sn[e], sl2, mask_term_of_byte<e % 4>((e % 8) < 4 ? (uint32_t)mk[e / 8].w : (uint32_t)(mk[e / 8].w >> 32), vzero, vninf));
        else s = Sn[e] * sl2;
        if constexpr (decltype(LIMc)::value) s = (jh + 16 * (e / 8) + 8 * g + e % 8 <= klim) ? s : NEG_INF;
        sc[e] = s;
        mx = e == 0 ? s : fmaxf(mx, s);
        if constexpr (DUAL) {
          spc[e] = Spn[e] * pr.scale;
          anchor(spc[e]);
        }
      });
      anchor(mx);
    } else {
      mx = pair_max(mx);
      const bool up = mx > m_i + TAU;  // the reference point moves only when a row's maximum exceeds it by more than that
      any_up = __any(up);
      const float m_new = up ? mx : m_i;
      alpha = up ? fast_exp2(m_i - m_new) : 1.f;
      m_i = m_new;
      m_use = (m_new == NEG_INF) ? 0.f : m_new;
      anchor(m_use);
    }
  };
  auto follow = [&]() {  // rare: the accumulators follow the reference point
    if (any_up) {
      asm volatile("s_nop 15\n\ts_nop 15");  // the last accumulation has written its registers
      l_i *= alpha;
      if constexpr (DUAL) mu_i *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          acc_move_in_place(Olow[db][e], Oacc[db][e], alpha, 0.f);
          if constexpr (DUAL) acc_move_in_place(Tlow[db][e], Tacc[db][e], alpha, 0.f);
        }
      }
    }
  };
  // splitting of the staged tiles: per task 2 units for each pair of elements, one of writes, one of loads
  constexpr int UPT = 10, NU_ST = UPT * NTASK;
  auto unit_st = [&](auto uc, int t, int jk, int jv) {  // K (t + 2), V (t + 1) written, K (t + 3) at jk, V (t + 2) at jv requested
    constexpr int u = decltype(uc)::value, i = u / UPT, s = u % UPT, w = s / 2;
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
      store_parts(i, t & 1, (t + 1) & 1);
    } else {
      load_raw(i, jk, t + 3 < ntiles, jv, t + 2 < ntiles);
    }
  };

  using B0 = std::false_type;
  using B1 = std::true_type;
  // units [g NU / NG, (g + 1) NU / NG) follow matrix instruction g
  auto spread = [&](auto gc, auto NGc, auto NUc, auto &&unit) {
    constexpr int gi = decltype(gc)::value, NG = decltype(NGc)::value, NU = decltype(NUc)::value;
    constexpr int lo = gi * NU / NG, hi = (gi + 1) * NU / NG;
    static_for<hi - lo>([&](auto dc) { unit(std::integral_constant<int, lo + decltype(dc)::value>{}); });
    __builtin_amdgcn_sched_barrier(0);
  };
  // Phase A of tile t (softmax at jh), with the scores of the tile in K stage kst; ends with the first V reads of stage vst.
  auto phase_a = [&](auto QKc, auto SMc, uint32_t kst, uint32_t vst, int jh) {
    constexpr bool QK = decltype(QKc)::value, SM = decltype(SMc)::value;
    constexpr int NG = QK ? KK * 6 * (DUAL ? 3 : 1) : 1, AHEAD = QK && SM ? 4 : 0, NU = SM ? NU_SM - AHEAD : 0;
    auto unit = [&](auto uc) { unit_sm(std::integral_constant<int, AHEAD + decltype(uc)::value>{}, jh); };
    if constexpr (QK) {
      issue_k(std::integral_constant<int, 0>{}, kst);
      __builtin_amdgcn_sched_barrier(0);
      static_for<AHEAD>([&](auto uc) { unit_sm(uc, jh); });  // while the first fragments travel
      static_for<KK>([&](auto kc) {
        constexpr int kk = decltype(kc)::value, sl = kk % 2;
        if constexpr (DUAL) x3_wait(ka[sl], kb[sl]);
        else x3_wait(ka[sl]);
        if constexpr (kk + 1 < KK) issue_k(std::integral_constant<int, kk + 1>{}, kst);
        else if constexpr (SM) issue_v(std::integral_constant<int, 0>{}, vst);
        __builtin_amdgcn_sched_barrier(0);
        static_for<6>([&](auto xc) {
          constexpr int x = decltype(xc)::value, n = kk * 6 + x;
          constexpr bool F = n == 0;
          auto gap = [&](auto gc) { spread(gc, std::integral_constant<int, NG>{}, std::integral_constant<int, NU>{}, unit); };
          if constexpr (DUAL) {
            mfma_s<F>(Spn, x3_frag(ka[sl][X3_A[x]]), Qtf[kk][X3_B[x]]);
            gap(std::integral_constant<int, 3 * n>{});
            mfma_s<F>(Sn, x3_frag(ka[sl][X3_A[x]]), Qf[kk][X3_B[x]]);
            gap(std::integral_constant<int, 3 * n + 1>{});
            mfma_s<false>(Spn, x3_frag(kb[sl][X3_A[x]]), Qf[kk][X3_B[x]]);
            gap(std::integral_constant<int, 3 * n + 2>{});
          } else {
            mfma_s<F>(Sn, x3_frag(ka[sl][X3_A[x]]), Qf[kk][X3_B[x]]);
            gap(std::integral_constant<int, n>{});
          }
        });
      });
    } else {
      issue_v(std::integral_constant<int, 0>{}, vst);
      static_for<NU>([&](auto uc) { unit(uc); });
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Phase B of tile t: accumulation (PV), and (ST) the staging and the front of the next tile's softmax (first key jn).
  auto phase_b = [&](auto PVc, auto STc, auto LIMc, uint32_t vst, int t, int jn, int jk, int jv) {
    constexpr bool PV = decltype(PVc)::value, ST = decltype(STc)::value;
    constexpr int NPV = 2 * DB, MPS = DUAL ? 3 : 1, NG = PV ? NPV * 6 * MPS : 1, NU = ST ? NU_ST + NU_FR : 0;
    // the first task, then the logits (the scores' last matrix instructions are through by then), then the other tasks
    auto unit = [&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if constexpr (u < UPT) unit_st(uc, t, jk, jv);
      else if constexpr (u < UPT + NU_FR) unit_fr(std::integral_constant<int, u - UPT>{}, LIMc, jn);
      else unit_st(std::integral_constant<int, u - NU_FR>{}, t, jk, jv);
    };
    if constexpr (PV) {
      static_for<NPV>([&](auto ic) {
        constexpr int i = decltype(ic)::value, c = i / DB, db = i % DB, sl = i % 2;
        if constexpr (DUAL) x3_wait(va[sl], vb[sl]);
        else x3_wait(va[sl]);
        if constexpr (i + 1 < NPV) issue_v(std::integral_constant<int, i + 1>{}, vst);
        __builtin_amdgcn_sched_barrier(0);
        static_for<6>([&](auto xc) {
          constexpr int x = decltype(xc)::value, n = i * 6 + x;
          auto gap = [&](auto gc) { spread(gc, std::integral_constant<int, NG>{}, std::integral_constant<int, NU>{}, unit); };
          const bf16x8 fv = x3_frag(va[sl][X3_A[x]]), fp = x3_frag(pf[c][X3_B[x]]);
          if constexpr (DUAL) {
            f32x16 &T = x == 5 ? Tacc[db] : Tlow[db];
            mfma_acc(T, fv, x3_frag(tf[c][X3_B[x]]));
            gap(std::integral_constant<int, 3 * n>{});
            mfma_acc(x == 5 ? Oacc[db] : Olow[db], fv, fp);
            gap(std::integral_constant<int, 3 * n + 1>{});
            mfma_acc(T, x3_frag(vb[sl][X3_A[x]]), fp);
            gap(std::integral_constant<int, 3 * n + 2>{});
          } else {
            mfma_acc(x == 5 ? Oacc[db] : Olow[db], fv, fp);
            gap(std::integral_constant<int, n>{});
          }
        });
      });
    } else {
      if constexpr (DUAL) tiles_ready(Sn, Spn);
      else tiles_ready(Sn);
      static_for<NU>([&](auto uc) { unit(uc); });
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (ST) follow();
  };

  // tiles t + 1, t + 2, t + 3 of the iteration (their first keys)
  int j0 = tile_at(0), j1 = j0, j2 = tile_at(1), j3 = tile_at(2);
  // K (0), K' (0) at once; then the registers take K (1) and V (0)
#pragma unroll
  for (int i = 0; i < NTASK; ++i) load_raw(i, j1, true, j1, true);
#pragma unroll
  for (int i = 0; i < NTASK; ++i) {
    if (!st_v[i]) {
      x3_split8(raw[i][0], raw[i][1], sp);
      store_parts(i, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < NTASK; ++i) load_raw(i, j2, 1 < ntiles, j1, true);
  fetch_masks(j1);
  x3_barrier();
  // the limits of the causal diagonal and of the end: from tile t_lim on (no lists without a mask)
  int t_lim = Lk / BT;
  if (pr.causal) t_lim = min(t_lim, q0 / BT);
  t_lim -= walk.first;
  constexpr bool LIMITS = MASK == MASK_NONE;
  using LimB = std::integral_constant<bool, LIMITS>;
  phase_a(B1{}, B0{}, 0u, 0u, 0);
  phase_b(B0{}, B1{}, LimB{}, 0u, -1, j1, j3, j2);
  auto step = [&](int t, auto LIMc) {  // j0: first key of tile t
    j0 = j1, j1 = j2, j2 = j3, j3 = tile_at(t + 3);
    x3_barrier();
    fetch_masks(j1);
    const uint32_t vst = (t & 1) * STAGEB;
    phase_a(B1{}, B1{}, ((t + 1) & 1) * STAGEB, vst, j0);
    phase_b(B1{}, B1{}, LIMc, vst, t, j1, j3, j2);
  };
  int t = 0;
  if constexpr (LIMITS) {
    for (; t < min(t_lim, ntiles) - 1; ++t) step(t, B0{});
    for (; t < ntiles - 1; ++t) step(t, B1{});
  } else {
    for (; t < ntiles - 1; ++t) step(t, B0{});
  }
  x3_barrier();
  phase_a(B0{}, B1{}, 0u, (t & 1) * STAGEB, j1);
  phase_b(B1{}, B0{}, B0{}, (t & 1) * STAGEB, t, 0, 0, 0);
  accs_ready(Oacc, Olow);
  if constexpr (DUAL) accs_ready(Tacc, Tlow);

  // ---- epilogue ------------------------------------------------------------------------------------
  l_i += xor32(l_i);
  if constexpr (DUAL) mu_i += xor32(mu_i);
  const bool dead = !split && !(l_i > 0.f);
  const float inv = split ? 1.f : dead ? 0.f : 1.f / l_i, mu_n = split ? 0.f : mu_i * inv;  // a share is left as it stands for the merge kernel
  float check = l_i * 0.f;  // not zero once an output is not finite (a row sum that is not a number makes its row 0)
  if (qrow < L) {
    float *Og = split ? pr.part + prow * ((DUAL ? 2 : 1) * D) : reinterpret_cast<float *>(p.o) + head + (size_t)qrow * D;
    float *Otg = split ? Og + D : DUAL ? reinterpret_cast<float *>(p.ot) + head + (size_t)qrow * D : nullptr;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        float o8[8], t8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          o8[e] = (Oacc[db][8 * hf + e] + Olow[db][8 * hf + e]) * inv;
          check = __builtin_fmaf(o8[e], 0.f, check);
          if constexpr (DUAL) {
            t8[e] = (Tacc[db][8 * hf + e] + Tlow[db][8 * hf + e]) * inv - mu_n * o8[e];
            check = __builtin_fmaf(t8[e], 0.f, check);
          }
        }
        const int d0 = 32 * db + 16 * hf + 8 * g;
        store8<float>(Og + d0, o8);
        if constexpr (DUAL) store8<float>(Otg + d0, t8);
      }
    }
    if (split) {
      if (g == 0) *reinterpret_cast<f32x4 *>(part_stat) = f32x4{m_i, l_i, mu_i, 0.f};
    } else if (g == 0) {
      p.M[(size_t)zh * L + qrow] = dead ? __builtin_inff() : m_i + __builtin_amdgcn_logf(l_i);
      if constexpr (DUAL) p.mu[(size_t)zh * L + qrow] = mu_n;
    }
  }
  return !x3_any(qrow < L && !(check == 0.f), lds0, wave, lane);
}
#endif

template <int D, bool DUAL> struct X3Lds {
  static constexpr size_t FWD = 2 * (size_t)(DUAL ? 4 : 2) * X3Cfg<D>::OPB;  // (more than the fp32 tiles take)
};
template <int D, bool DUAL, int MASK, bool DROP, bool SPLIT, int WGS = DUAL ? 1 : 2>
__global__ __launch_bounds__(256, WGS) void fwd_f32x3_kernel(const FwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (!fwd_f32x3_body<D, DUAL, MASK, DROP, SPLIT>(p)) fwd_f32_body<D, DUAL, MASK, DROP, SPLIT>(p);
#endif
}

}  // namespace jvpfa
