// Fused dual forward for fp32, D in {32, 64, 128}, on the direct-to-LDS pipeline.  (Up to D = 64 it is what
// fwd_kernel_f32x3.hpp, faster there, falls back on for outputs that are not finite.)
//
// Mathematics and work split as in fwd_kernel.hpp (4 waves = 128 query rows, scores transposed, lane = query).  An fp32
// matrix instruction (32x32x2) takes 64 cycles for what is 4 of the bf16 one's 32, so a wave has time for everything else
// as long as it never waits: the register-staged kernel this replaces copied every tile through registers behind two
// barriers, wrote V transposed, fetched mask values where they were used and rescaled the accumulators on every tile,
// and kept the matrix cores busy 58 % of the time at B4 H8 L1024 D64 (one workgroup per compute unit, one wave per
// SIMD: nothing else runs while a wave waits).  Here:
//   * 32-key tiles of K, V (, K', V') go global -> LDS directly, two stages, one barrier per tile;
//   * every tile is row-major and read as it is.  The contraction index of a product may be dealt to the instructions in
//     any order as long as both operands agree: the scores take d = 8j + 4g + i (step j, lane half g), one ds_read_b128 per
//     four instructions, and the output rows of V^T P are d = DB * row + db, so that a lane reads the DB values it needs
//     of a key in one piece (ds_read_b32 / b64 / b128).  No transposed copy, no cross-lane move.
//   * 16-byte chunks are swizzled on the global side by the row, so the row-wise read (16 rows at one chunk) meets 64
//     different banks; the other read takes whole rows.
//   * reads run one step ahead of their products, mask values a tile ahead, and the reference point of the exponentials
//     moves only when a row's maximum exceeds it by 8 (log2 units).
// Measured, dual forward at that shape: additive bias per head 290 -> 200 us (84 % of the rate of a large fp32 matrix
// product on this card), key padding 276 -> 204 us; B4 H16 L2048 D128 without a mask 5.05 -> 2.91 ms (92 %).
#pragma once
#include "common.hpp"
#include "mask.hpp"
#include "params.hpp"
#include "pipeline.hpp"

namespace jvpfa {

template <int D> struct F32Cfg {
  static constexpr int NT = 4 * WAVE, BLK = 128, BT = 32;
  static constexpr int CH = D / 4, ROWB = D * 4, TILEB = BT * ROWB;
  static constexpr int IPW = TILEB / 1024 / 4;         // direct-load instructions per wave and tile
  static constexpr int NJ = D / 8, DB = D / 32;        // score steps; 32-row blocks of the output
};
// the chunk of a row is moved by this (CH = 8: two rows share the 256 bytes of all banks)
template <int CH> __device__ __forceinline__ int swz_f32(int row) { return CH == 8 ? (row >> 1) & 7 : row & 15; }

// N consecutive floats of a lane
template <int N> struct F32Row;
template <> struct F32Row<1> { using type = float; };
template <> struct F32Row<2> { using type = __attribute__((ext_vector_type(2))) float; };
template <> struct F32Row<4> { using type = f32x4; };
__device__ __forceinline__ float f32_at(const float &x, int) { return x; }
template <typename V> __device__ __forceinline__ float f32_at(const V &x, int i) { return x[i]; }
template <int OFF> __device__ __forceinline__ void lds_row(float &d, uint32_t a) { asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(d) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_row(F32Row<2>::type &d, uint32_t a) { asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(d) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_row(f32x4 &d, uint32_t a) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(d) : "v"(a), "n"(OFF)); }
// every LDS read of this wave has arrived; tied to the registers read
template <typename V> __device__ __forceinline__ void lds_done(V &a) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a)); }
template <typename V> __device__ __forceinline__ void lds_done(V &a, V &b) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a), "+v"(b)); }
template <typename V> __device__ __forceinline__ void lds_done(V &a, V &b, V &c, V &d) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d)); }
template <typename V> __device__ __forceinline__ void lds_done(V (&a)[4]) { lds_done(a[0], a[1], a[2], a[3]); }
template <typename V> __device__ __forceinline__ void lds_done(V (&a)[4], V (&b)[4]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
}

// Products in program order (see the 16-bit forms in pipeline.hpp and fwd_kernel_v3.hpp): a score tile in vector
// registers with a resident B operand in the accumulation file or (BV) in vector registers, and an accumulator in place.
// GUARD: two idle issue slots in front (nothing next to the 64 cycles of the product), for kernels that fill the
// accumulation file, where the allocator moves resident operands right before their use.
template <bool FIRST, bool BV = false, bool GUARD = false> __device__ __forceinline__ void mma_f32_s(f32x16 &c, float a, float b) {
  if constexpr (GUARD) {
    if constexpr (FIRST) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x2_f32 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
    else asm volatile("s_nop 1\n\tv_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
  } else if constexpr (BV) {
    if constexpr (FIRST) asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  } else {
    if constexpr (FIRST) asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
    else asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
  }
}
__device__ __forceinline__ void mma_f32_acc(f32x16 &c, float a, float b) {
  asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void pin_acc(f32x4 &f) { asm volatile("" : "+a"(f)); }
// A tile of zeros in the accumulation file by one product of zeros.  (Zeroed by element the compiler copies one register to
// all others; where this is the second body of a kernel the build's lint cannot tell those copies from a tile moved.)
__device__ __forceinline__ void zero_tile(f32x16 &c) { asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %1, 0" : "=a"(c) : "v"(0.f)); }

#if defined(__HIP_DEVICE_COMPILE__)
// Direct loads of the tiles of up to four tensors into stage `stage`, and the addresses of both reads.
template <int D, int NTILE> struct F32Tiles {
  using C = F32Cfg<D>;
  uint32_t ld_o[C::IPW], ld_dst = 0;
  __amdgpu_buffer_rsrc_t rs[NTILE];
  uint32_t row0;       // row-wise read: row perm32(r), chunk g, swizzled; step j is this xor 32 j
  uint32_t col[8];     // whole-row read: row 8g + e, this lane's DB floats
  __device__ __forceinline__ void init(int wave, int lane) {
    const int r = lane % 32, g = lane / 32, pr32 = perm32(r);
#pragma unroll
    for (int i = 0; i < C::IPW; ++i) {
      const int lc = 64 * (wave * C::IPW + i) + lane, row = lc / C::CH;
      ld_o[i] = row * C::ROWB + ((lc % C::CH) ^ swz_f32<C::CH>(row)) * 16;
    }
    row0 = pr32 * C::ROWB + ((g ^ swz_f32<C::CH>(pr32)) * 16);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int row = 8 * g + e, byte = r * C::DB * 4;
      col[e] = row * C::ROWB + (((byte / 16) ^ swz_f32<C::CH>(row)) * 16) + byte % 16;
    }
  }
  // rows: those that exist from this tile's first on (rows past them, and tiles that do not exist, read as zeros).  The
  // bytes of all that follow, 512 a row at D = 128, pass the descriptor's 32 bits at 2^23 rows: it then covers the next 2 GB.
  // (Cut to the tile instead, the compiler finds other schedules, which take a wave or 16 - 60 bytes of spill from 17 kernels.)
  __device__ __forceinline__ void aim(int t, const float *base, int first, int rows) {
    rs[t] = __builtin_amdgcn_make_buffer_rsrc((void *)(base + (size_t)first * D), 0, (int)min((long long)max(rows, 0) * C::ROWB, 0x7fffffffLL), 0x00020000);
  }
  template <int P> __device__ __forceinline__ void load() {
    constexpr int i = P / NTILE, t = P % NTILE;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs[t], (JVPFA_LDS(void))(uintptr_t)(ld_dst + i * 1024 + t * C::TILEB), 16, ld_o[i], 0, 0, 0);
  }
};

template <int D, bool DUAL, int MASK, bool DROP, bool SPLIT = false>
__device__ __forceinline__ void fwd_f32_body(const FwdParams &p) {
  using C = F32Cfg<D>;
  constexpr int BT = C::BT, NJ = C::NJ, DB = C::DB, NTILE = DUAL ? 4 : 2, STAGEB = NTILE * C::TILEB;
  constexpr float NEG_INF = -__builtin_inff(), TAU = 8.f;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem_raw;  // stage s: [K | V | K' | V']

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
  const int r = lane % 32, g = lane / 32;

  const size_t head = (size_t)zh * L * D;
  const size_t kvhead = ((size_t)z * pr.Hk + h / (pr.H / pr.Hk)) * Lk * D;  // grouped heads share K, V
  const float *Kg = reinterpret_cast<const float *>(p.k) + kvhead, *Vg = reinterpret_cast<const float *>(p.v) + kvhead;
  const float *Ktg = DUAL ? reinterpret_cast<const float *>(p.kt) + kvhead : nullptr;
  const float *Vtg = DUAL ? reinterpret_cast<const float *>(p.vt) + kvhead : nullptr;
  const int q0 = qb * C::BLK, qrow = q0 + wave * 32 + r, qld = qrow < L ? qrow : L - 1;

  f32x4 Qf[NJ], Qtf[DUAL ? NJ : 1];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    Qf[j] = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(p.q) + head + (size_t)qld * D + 8 * j + 4 * g);
    if constexpr (DUAL) Qtf[j] = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(p.qt) + head + (size_t)qld * D + 8 * j + 4 * g);
  }
  // resident in the accumulation file from here on (D = 128 with tangents: Q' does not fit next to Q, O and T)
  constexpr bool QT_V = DUAL && D == 128;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    pin_acc(Qf[j]);
    if constexpr (DUAL && !QT_V) pin_acc(Qtf[j]);
  }
  f32x16 Oacc[DB], Tacc[DUAL ? DB : 1];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    zero_tile(Oacc[db]);
    if constexpr (DUAL) zero_tile(Tacc[db]);
  }
  float m_i = NEG_INF, l_i = 0.f, mu_i = 0.f;  // l_i, mu_i: this lane's keys

  const float sl2 = pr.scale * LOG2E;
  const int64_t mrow = MASK != MASK_NONE ? z * pr.ms[0] + h * pr.ms[1] + (int64_t)qld * pr.ms[2] : 0;
  const uint32_t drop_row = DROP ? drop_row_word(pr, zh, qld) : 0u;
  bool mask_al = false;
  if constexpr (MASK != MASK_NONE) mask_al = mask_rows_aligned<float, MASK>(pr);
  int kend = pr.causal ? min(Lk, q0 + C::BLK) : Lk;
  // key tiles visited: up to kend, or the caller's list of those that hold an attended entry
  TileWalk<BT> walk;
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
    return;
  }
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
  MaskAhead<float, MASK> mcur[2], mnext[2];  // this tile's mask values and the next one's, 8 keys each
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
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's share of the tile and its mask values are there
    __syncthreads();                      // ... everyone's, and the other stage is no longer read
    if constexpr (MASK != MASK_NONE) {
      mcur[0] = mnext[0], mcur[1] = mnext[1];
      fetch_masks(jnext);
    }
    aim((t + 1) & 1, jnext, t + 1 < ntiles);
    const uint32_t sb = lds0 + (t & 1) * STAGEB;
    const uint32_t rowa = sb + tiles.row0;

    // ---- S^T = K Q^T, S'^T = K Q'^T + K' Q^T: step j takes d = 8j + 4g + 0..3 ---------------------------
    f32x16 S, Sp;
    f32x4 ka[2], kb[2];
    auto issue_k = [&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const uint32_t a = rowa ^ (32 * j);
      lds_row<0>(ka[j % 2], a);
      if constexpr (DUAL) lds_row<2 * C::TILEB>(kb[j % 2], a);
    };
    // V rows of 4 registers' keys (16 (i / 2) + 8g + 4 (i % 2) + 0..3)
    typename F32Row<DB>::type va[2][4], vb[2][4];
    auto issue_v = [&](auto ic) {
      constexpr int i = decltype(ic)::value;
      static_for<4>([&](auto ec) {
        constexpr int e = decltype(ec)::value;
        const uint32_t a = sb + tiles.col[4 * (i % 2) + e];
        lds_row<C::TILEB + (i / 2) * 16 * C::ROWB>(va[i % 2][e], a);
        if constexpr (DUAL) lds_row<3 * C::TILEB + (i / 2) * 16 * C::ROWB>(vb[i % 2][e], a);
      });
    };
    issue_k(std::integral_constant<int, 0>{});
    static_for<NJ>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (DUAL) lds_done(ka[j % 2], kb[j % 2]);
      else lds_done(ka[j % 2]);
      if constexpr (j + 1 < NJ) issue_k(std::integral_constant<int, j + 1>{});
      else issue_v(std::integral_constant<int, 0>{});
      static_for<(NLOAD + NJ - 1) / NJ>([&](auto pc) {
        constexpr int P = j * ((NLOAD + NJ - 1) / NJ) + decltype(pc)::value;
        if constexpr (P < NLOAD) tiles.template load<P>();
      });
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (no two consecutive products on the same tile)
        if constexpr (DUAL) {
          if (i == 0) mma_f32_s<j == 0, QT_V>(Sp, ka[j % 2][i], Qtf[j][i]);
          else mma_f32_s<false, QT_V>(Sp, ka[j % 2][i], Qtf[j][i]);
        }
        if (i == 0) mma_f32_s<j == 0>(S, ka[j % 2][i], Qf[j][i]);
        else mma_f32_s<false>(S, ka[j % 2][i], Qf[j][i]);
        if constexpr (DUAL) mma_f32_s<false>(Sp, kb[j % 2][i], Qf[j][i]);
      }
    });
    if constexpr (DUAL) tiles_ready(S, Sp);
    else tiles_ready(S);

    // ---- online softmax in the log2 domain (register e: key 16 (e / 8) + 8g + e % 8 of the tile) ---------
    const bool diag = pr.causal && (j0 + BT - 1 > q0 + wave * 32), ragged = j0 + BT > Lk;
    const int klim = min(pr.causal ? qrow : 0x7fffffff, Lk - 1);
    float mx = NEG_INF;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      float s = S[e] * sl2;
      if constexpr (MASK == MASK_ADD) s = __builtin_fmaf((float)mcur[e / 8].f[e % 8], LOG2E, s);
      if constexpr (MASK == MASK_BOOL) s = mask_keep_of<float, MASK>(mcur[e / 8], e % 8) ? s : NEG_INF;
      S[e] = s;
    }
    if (diag || ragged) {
#pragma unroll
      for (int e = 0; e < 16; ++e) S[e] = (j0 + 16 * (e / 8) + 8 * g + e % 8 <= klim) ? S[e] : NEG_INF;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, S[e]);
    mx = pair_max(mx);
    const bool up = mx > m_i + TAU;
    if (__any(up)) {
      const float m_new = up ? mx : m_i;
      const float alpha = up ? fast_exp2(m_i - m_new) : 1.f;
      m_i = m_new;
      l_i *= alpha;
      if constexpr (DUAL) mu_i *= alpha;
      asm volatile("s_nop 15\n\ts_nop 15");  // the accumulations of the previous tile, a phase of products ago, have landed
#pragma unroll
      for (int db = 0; db < DB; ++db) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          Oacc[db][e] = acc_scale(Oacc[db][e], alpha);
          if constexpr (DUAL) Tacc[db][e] = acc_scale(Tacc[db][e], alpha);
        }
      }
    }
    const float m_use = (m_i == NEG_INF) ? 0.f : m_i;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float pv = fast_exp2(S[e] - m_use);
      l_i += pv;
      float ks = 1.f;
      if constexpr (DROP) ks = drop_scale_of(pr, drop_row + (uint32_t)(j0 + 16 * (e / 8) + 8 * g + e % 8) * DROP_C_KEY);
      S[e] = DROP ? pv * ks : pv;
      if constexpr (DUAL) {
        const float ps = pv * (Sp[e] * pr.scale);
        mu_i += ps;
        Sp[e] = DROP ? ps * ks : ps;
      }
    }

    // the values are there, and two issue slots have passed, before the first product reads them
    if constexpr (DUAL) asm volatile("s_nop 1" : "+v"(S), "+v"(Sp));
    else asm volatile("s_nop 1" : "+v"(S));
    // ---- O^T += V^T P^T, T^T += V^T (P S')^T + V'^T P^T: row `row` of block db is d = DB row + db ----------
    static_for<4>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (DUAL) lds_done(va[i % 2], vb[i % 2]);
      else lds_done(va[i % 2]);
      if constexpr (i + 1 < 4) issue_v(std::integral_constant<int, i + 1>{});
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          mma_f32_acc(Oacc[db], f32_at(va[i % 2][e], db), S[4 * i + e]);
          if constexpr (DUAL) {
            mma_f32_acc(Tacc[db], f32_at(va[i % 2][e], db), Sp[4 * i + e]);
            mma_f32_acc(Tacc[db], f32_at(vb[i % 2][e], db), S[4 * i + e]);
          }
        }
      }
    });
    jcur = jnext;
    jnext = tile_at(t + 2);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);

  if constexpr (DUAL) accs_ready(Oacc, Tacc);
  else accs_ready(Oacc);
  // ---- epilogue ------------------------------------------------------------------------------------
  l_i += xor32(l_i);
  if constexpr (DUAL) mu_i += xor32(mu_i);
  const bool dead = !split && !(l_i > 0.f);
  const float inv = split ? 1.f : dead ? 0.f : 1.f / l_i, mu_n = split ? 0.f : mu_i * inv;  // a share is left as it stands for the merge kernel
  if (qrow < L) {
    float *Og = split ? pr.part + prow * ((DUAL ? 2 : 1) * D) : reinterpret_cast<float *>(p.o) + head + (size_t)qrow * D;
    float *Otg = split ? Og + D : DUAL ? reinterpret_cast<float *>(p.ot) + head + (size_t)qrow * D : nullptr;
    // registers 4q .. 4q + 3 are rows 8q + 4g + 0..3: 4 DB consecutive columns
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float o[4 * DB], ot[4 * DB];
#pragma unroll
      for (int x = 0; x < 4 * DB; ++x) {
        o[x] = Oacc[x % DB][4 * q + x / DB] * inv;
        if constexpr (DUAL) ot[x] = Tacc[x % DB][4 * q + x / DB] * inv - mu_n * o[x];
      }
      const int d0 = DB * (8 * q + 4 * g);
#pragma unroll
      for (int x = 0; x < 4 * DB; x += 4) {
        *reinterpret_cast<f32x4 *>(Og + d0 + x) = f32x4{o[x], o[x + 1], o[x + 2], o[x + 3]};
        if constexpr (DUAL) *reinterpret_cast<f32x4 *>(Otg + d0 + x) = f32x4{ot[x], ot[x + 1], ot[x + 2], ot[x + 3]};
      }
    }
    if (split) {
      if (g == 0) *reinterpret_cast<f32x4 *>(part_stat) = f32x4{m_i, l_i, mu_i, 0.f};
    } else if (g == 0) {
      p.M[(size_t)zh * L + qrow] = dead ? __builtin_inff() : m_i + __builtin_amdgcn_logf(l_i);
      if constexpr (DUAL) p.mu[(size_t)zh * L + qrow] = mu_n;
    }
  }
}
#endif

template <int D, bool DUAL, int MASK, bool DROP, bool SPLIT>
__global__ __launch_bounds__(256, 1) void fwd_f32_kernel(const FwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  fwd_f32_body<D, DUAL, MASK, DROP, SPLIT>(p);
#endif
}

}  // namespace jvpfa
