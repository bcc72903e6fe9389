// One translation unit per (element type, head dim): compiled with
//   -DJVPFA_T=<__bf16|_Float16|float> -DJVPFA_D=<32|64|128|256> -DJVPFA_NAME=<symbol>
// and exporting  int JVPFA_NAME(const BwdParams&, int mask_kind, bool dual, bool tangent_grads,
// hipStream_t): pre-pass, then the dq and dk/dv kernels of every requested mode.
#include "bwd_kernel.hpp"
#include "bwd_kernel_f32.hpp"
#include "bwd_kernel_f32x3.hpp"
#include "bwd_kernel_v2.hpp"
#include "bwd_kernel_wide.hpp"
#include "bwd_kernel_pair.hpp"
#include "launch.hpp"
#include "split.hpp"

namespace jvpfa {

// Which of the tangent-input gradients the dual kernels of the direct-to-LDS family produce on the way when
// all six gradients are asked for (dq' costs the dq kernel one more product per tile and dk', dv' the dk/dv
// kernel two, against a second pair of launches that forms the score tiles again): dq' wherever that family
// runs; dk', dv' where the two extra accumulators fit (D <= 64; at D = 64 that kernel then has a compute unit
// to itself instead of sharing it with a second workgroup and is still 4 - 9 % ahead; at D = 128 dK, dV, the
// resident K, V, K' and the tiles already take 452 of the 512 registers and dK', dV' would add 128).
template <typename T, int D> struct BwdFold {
  static constexpr bool DQ = sizeof(T) == 2;
  static constexpr bool KV = sizeof(T) == 2 && D <= 64;
};

// The dq kernel of the direct-to-LDS family for one launch.  MK is MASK, or MASK_BITS for a boolean mask whose packed copy
// the caller handed over.  six: the dual variant that also writes dq'.
template <typename T, int D, int MODE, int MK> static auto pick_dq(bool no_go, bool six) -> void (*)(const BwdParams) {
  constexpr bool NG = MODE != BWD_DUAL;  // the GO template argument of the kernels without gO
  if constexpr (MODE == BWD_DUAL) {
    if (six) {
      // (without gO the register cap of the two-workgroup twin makes the allocator copy LDS fragments out of
      // their registers before they have arrived, which the build's lint refuses: that variant runs uncapped)
      if constexpr (D == 64) return no_go ? bwd2_dq_kernel<T, D, MODE, MK, false, true> : bwd2_dq_kernel_2wg<T, D, MODE, MK, true, true>;
      else return no_go ? bwd2_dq_kernel<T, D, MODE, MK, false, true> : bwd2_dq_kernel<T, D, MODE, MK, true, true>;
    }
  }
  if constexpr (D == 128 && MODE == BWD_PLAIN) return bwd2_dq_kernel_2wg_plain<T, D, MODE, MK>;
  // D = 64: the register-capped twins, two workgroups per compute unit (D = 32 needs no cap for that)
  else if constexpr (D == 64) return no_go ? bwd2_dq_kernel_2wg<T, D, MODE, MK, NG> : bwd2_dq_kernel_2wg<T, D, MODE, MK, true>;
  else return no_go ? bwd2_dq_kernel<T, D, MODE, MK, NG> : bwd2_dq_kernel<T, D, MODE, MK, true>;
}

// The dk/dv kernel of the direct-to-LDS family for one launch.  MK is MASK, or MASK_BITS for a boolean mask
// whose bit-packed copy the caller handed over.  fold_kv: the dual variant that also writes dk', dv'.
template <typename T, int D, int MODE, int MK>
static auto pick_dkdv(bool no_go, bool grouped, bool fold_kv, bool drop) -> void (*)(const BwdParams) {
  constexpr bool NG = MODE != BWD_DUAL;  // the GO template argument of the kernels without gO
  if (drop) {
    if (grouped) return no_go ? bwd2_dkdv_kernel<T, D, MODE, MK, NG, true, false, true> : bwd2_dkdv_kernel<T, D, MODE, MK, true, true, false, true>;
    return no_go ? bwd2_dkdv_kernel<T, D, MODE, MK, NG, false, false, true> : bwd2_dkdv_kernel<T, D, MODE, MK, true, false, false, true>;
  }
  if constexpr (MODE == BWD_DUAL && BwdFold<T, D>::KV) {
    if (fold_kv) {
      if (grouped) return no_go ? bwd2_dkdv_kernel<T, D, MODE, MK, false, true, true> : bwd2_dkdv_kernel<T, D, MODE, MK, true, true, true>;
      return no_go ? bwd2_dkdv_kernel<T, D, MODE, MK, false, false, true> : bwd2_dkdv_kernel<T, D, MODE, MK, true, false, true>;
    }
  }
  // D = 64: the register-capped twins, two workgroups per compute unit (D = 32 needs no cap for that); the masked
  // dual kernel needs a few registers more than the cap leaves
  if constexpr (D == 64 && (MK == MASK_NONE || MODE != BWD_DUAL)) {
    if (grouped) return no_go ? bwd2_dkdv_kernel_2wg<T, D, MODE, MK, NG, true> : bwd2_dkdv_kernel_2wg<T, D, MODE, MK, true, true>;
    return no_go ? bwd2_dkdv_kernel_2wg<T, D, MODE, MK, NG> : bwd2_dkdv_kernel_2wg<T, D, MODE, MK, true>;
  }
  if (grouped) return no_go ? bwd2_dkdv_kernel<T, D, MODE, MK, NG, true> : bwd2_dkdv_kernel<T, D, MODE, MK, true, true>;
  return no_go ? bwd2_dkdv_kernel<T, D, MODE, MK, NG> : bwd2_dkdv_kernel<T, D, MODE, MK, true>;
}
// An additive mask can be streamed through LDS as tiles (MASK_TILE) when its rows are runs of contiguous keys
// that start on 16-byte boundaries wherever a tile starts, and 64 rows stay within a 32-bit offset.
template <typename T> static bool mask_rows_tileable(const Problem &pr) {
  const int64_t es = sizeof(T);
  if (pr.ms[3] != 1 || (reinterpret_cast<uintptr_t>(pr.mask) & 15u)) return false;
  for (int i = 0; i < 3; ++i)
    if (pr.ms[i] < 0 || (pr.ms[i] * es) % 16 != 0) return false;
  return 64 * pr.ms[2] * es < ((int64_t)1 << 31);
}
// *lds: the dynamic LDS bytes of the kernel returned
template <typename T, int D, int MODE, int MASK>
static auto pick_dkdv_for(const BwdParams &p, bool no_go, bool grouped, bool fold_kv, bool drop, size_t *lds) -> void (*)(const BwdParams) {
  using Cfg2 = Bwd2Cfg<T, D, MODE>;
  *lds = Cfg2::DKV_LDS;
  if constexpr (MASK == MASK_BOOL) {
    if (p.pr.bits_k) return pick_dkdv<T, D, MODE, MASK_BITS>(no_go, grouped, fold_kv, drop);
  }
  if constexpr (MASK == MASK_ADD) {
    if (mask_rows_tileable<T>(p.pr)) {
      *lds = Cfg2::DKV_LDS_MTILE;
      return pick_dkdv<T, D, MODE, MASK_TILE>(no_go, grouped, fold_kv, drop);
    }
  }
  return pick_dkdv<T, D, MODE, MASK>(no_go, grouped, fold_kv, drop);
}

// The dk/dv kernel for D = 256 without tangents in the launch: without masks one kernel whether the heads are split or not.
template <typename T, int D, int MODE, int MASK, bool DROP> static auto pick_wide_dkdv(const BwdParams &p) -> void (*)(const BwdParams) {
  if constexpr (MASK != MASK_NONE) {
    if (p.pr.chunks <= 1) return bwdw_dkdv_kernel<T, D, MODE, MASK, DROP>;
  }
  return bwdw_dkdv_kernel<T, D, MODE, MASK, DROP, true>;
}

// dk/dv and dq in one launch (launch_both in split.hpp says for which grids).
static int run_both(void (*kb)(const BwdParams, int), const BwdParams &p, long long kv_blocks, long long total, size_t lds, hipStream_t stream) {
  if (total > 0x7fffffffLL) return -2;
  const int rc = allow_lds(reinterpret_cast<const void *>(kb), lds);
  if (rc != 0) return rc;
  hipLaunchKernelGGL(kb, dim3((unsigned)total), dim3(256), lds, stream, p, (int)kv_blocks);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}
// The kernel for one launch of everything that is asked for (without dropout), or null where two are better or no such kernel
// exists: six gradients and grouped heads without a mask or (six gradients) with a packed one.
template <typename T, int D, int MODE, int MASK>
static auto pick_both(const BwdParams &p, bool no_go, bool grouped, bool six, long long blocks, long long kv_blocks) -> void (*)(const BwdParams, int) {
  constexpr bool NG = MODE != BWD_DUAL;
  const bool bits = MASK == MASK_BOOL && p.pr.bits_q && p.pr.bits_k;
  constexpr bool M = MASK != MASK_NONE;
  const int kind = bits ? MASK_BITS : MASK;  // as the kernels read it
  const bool causal = p.pr.causal != 0, twin = D == 64 && MODE == BWD_DUAL && !grouped && !six && (!M || bits);
  // (six: the dual and the tangent launch of a call decide alike)
  if (!(six ? launch_both<D, BWD_DUAL>(blocks, kv_blocks, causal, kind, false, true, grouped, false, no_go)
            : launch_both<D, MODE>(blocks, kv_blocks, causal, kind, false, false, grouped, twin, no_go)))
    return nullptr;
  if constexpr (MASK == MASK_ADD) {  // (read element by element here, and as tiles by the dk/dv kernel of its own launch)
    if (blocks >= device_cus() || kv_blocks >= device_cus()) return nullptr;
  }
  if (grouped) {
    if (six) return nullptr;
    if constexpr (MASK == MASK_NONE) return no_go ? bwd2_both_kernel<T, D, MODE, MASK, NG, true> : bwd2_both_kernel<T, D, MODE, MASK, true, true>;
    return nullptr;
  }
  if (six) {
    if (!(MASK == MASK_NONE || bits)) return nullptr;
    constexpr int MK = MASK == MASK_BOOL ? MASK_BITS : MASK_NONE;
    if constexpr (D == 128) return no_go ? bwd2_all_kernel<T, D, MK, false> : bwd2_all_kernel<T, D, MK, true>;
    else return no_go ? bwd2_both_kernel<T, D, BWD_DUAL, MK, false, false, true> : bwd2_both_kernel<T, D, BWD_DUAL, MK, true, false, true>;
  }
  if constexpr (D == 64 && MODE == BWD_DUAL && MASK != MASK_ADD) {
    constexpr int MK = MASK == MASK_BOOL ? MASK_BITS : MASK_NONE;
    if (twin && both_two_wgs(p.pr.L, p.pr.Lk, (long long)p.pr.Z * p.pr.H, causal))
      return no_go ? bwd2_both_kernel_2wg<T, D, MODE, MK, NG> : bwd2_both_kernel_2wg<T, D, MODE, MK, true>;
  }
  if constexpr (MASK == MASK_BOOL) {
    if (bits) return no_go ? bwd2_both_kernel<T, D, MODE, MASK_BITS, NG> : bwd2_both_kernel<T, D, MODE, MASK_BITS, true>;
  }
  return no_go ? bwd2_both_kernel<T, D, MODE, MASK, NG> : bwd2_both_kernel<T, D, MODE, MASK, true>;
}

// Adds up the shares of dk, dv (dk', dv' of the tangent mode; all four where the dual kernel folds them in) that a
// launch over pr.chunks query heads groups left, see split.hpp.
template <typename T, int D> static void launch_kv_merge(const BwdParams &p, bool tangent, bool four, hipStream_t stream) {
  if (p.pr.chunks <= 1) return;
  const size_t elems = (size_t)p.pr.Z * p.pr.Hk * p.pr.Lk * D;
  T *dk = reinterpret_cast<T *>(p.dk), *dv = reinterpret_cast<T *>(p.dv), *dkt = reinterpret_cast<T *>(p.dkt), *dvt = reinterpret_cast<T *>(p.dvt);
  hipLaunchKernelGGL((bwd_kv_merge_kernel<T>), dim3((unsigned)((elems / 8 + 255) / 256), four ? 4 : 2), dim3(256), 0, stream, p.pr.part,
                     p.pr.chunks, elems, tangent ? dkt : dk, tangent ? dvt : dv, dkt, dvt);
}

// The deal of a launch whose blocks' tiles are split (what jvpfa_bwd found worth it), and the workgroups of either role.
template <int D, bool F32> static BwdSplit split_of(const Problem &pr, bool dual, long long *kv_blocks, long long *blocks) {
  const BwdDeal d = bwd_deal(F32, D, pr.Z, pr.H, pr.L, pr.Lk, pr.causal != 0, dual);
  const long long heads = (long long)pr.Z * pr.H;
  const int bq = (pr.L + 127) / 128, bk = (pr.Lk + 127) / 128;
  *kv_blocks = heads * (d.k.step > 0 ? d.k.workgroups() + std::max(bk - bq, 0) : bk * d.k.most);
  *blocks = heads * (d.q.step > 0 ? d.q.workgroups() : bq * d.q.most);
  return {d.q, d.k, pr.part, pr.part + (d.q.most > 1 ? (size_t)d.q.most * heads * pr.L * D : 0)};
}
template <typename T, int D> static void launch_split_merge(const BwdParams &p, const BwdSplit &sp, bool tangent, hipStream_t stream) {
  constexpr int RPB = 2048 / D;
  hipLaunchKernelGGL((bwd_split_merge_kernel<T, D>), dim3((unsigned)((std::max(p.pr.L, p.pr.Lk) + RPB - 1) / RPB), p.pr.Z * p.pr.H, 3), dim3(256), 0,
                     stream, p, sp, tangent ? 1 : 0);
}

// The dq and dk/dv kernels for fp32 with D <= 128: up to D = 64 as three bf16 parts.
template <int D, int MODE, int MASK, bool GO, bool DROP> static auto pick_f32_dq() -> void (*)(const BwdParams) {
  if constexpr (D <= 64) return bwd_f32x3_dq_kernel<D, MODE, MASK, GO, DROP>;
  else return bwd_f32_dq_kernel<D, MODE, MASK, GO, DROP>;
}
template <int D, int MODE, int MASK, bool GO, bool DROP> static auto pick_f32_dkdv() -> void (*)(const BwdParams) {
  if constexpr (D <= 64) return bwd_f32x3_dkdv_kernel<D, MODE, MASK, GO, DROP>;
  else return bwd_f32_dkdv_kernel<D, MODE, MASK, GO, DROP>;
}
template <int D, int MODE, int MASK, bool GO> static auto pick_f32_both(bool split) -> void (*)(const BwdParams, const BwdSplit, int) {
  if constexpr (D <= 64) return split ? bwd_f32x3_both_kernel<D, MODE, MASK, GO, true> : bwd_f32x3_both_kernel<D, MODE, MASK, GO, false>;
  else return split ? bwd_f32_both_kernel<D, MODE, MASK, GO, true> : bwd_f32_both_kernel<D, MODE, MASK, GO, false>;
}
template <int D, int MODE, int MASK, bool DROP>
static int launch_bwd_f32(const BwdParams &p, long long blocks, long long kv_blocks, hipStream_t stream) {
  constexpr bool NG = MODE != BWD_DUAL;  // gO may be absent only in the dual mode
  const bool no_go = MODE == BWD_DUAL && p.go == nullptr;
  void (*kq)(const BwdParams) = no_go ? pick_f32_dq<D, MODE, MASK, NG, DROP>() : pick_f32_dq<D, MODE, MASK, true, DROP>();
  void (*kkv)(const BwdParams) = no_go ? pick_f32_dkdv<D, MODE, MASK, NG, DROP>() : pick_f32_dkdv<D, MODE, MASK, true, DROP>();
  using Lds = std::conditional_t<D <= 64, BwdX3Lds<D, MODE>, BwdF32Lds<D, MODE>>;
  int rc = allow_lds(reinterpret_cast<const void *>(kq), Lds::DQ);
  if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), Lds::DKV);
  if (rc != 0) return rc;
  if constexpr (!DROP) {
    const bool split = p.pr.chunk_tiles == -1;
    if (split || launch_both_f32<D, MODE>(blocks, kv_blocks, p.pr.causal != 0 || MASK == MASK_BOOL)) {
      void (*kb)(const BwdParams, const BwdSplit, int) = no_go ? pick_f32_both<D, MODE, MASK, NG>(split) : pick_f32_both<D, MODE, MASK, true>(split);
      const Problem &pr = p.pr;
      BwdSplit sp = {{1, 0, 0, 0}, {1, 0, 0, 0}, nullptr, nullptr};
      if (split) sp = split_of<D, true>(pr, MODE != BWD_PLAIN, &kv_blocks, &blocks);
      if (kv_blocks + blocks > 0x7fffffffLL) return -2;
      rc = allow_lds(reinterpret_cast<const void *>(kb), Lds::DKV);
      if (rc != 0) return rc;
      hipLaunchKernelGGL(kb, dim3((unsigned)(kv_blocks + blocks)), dim3(256), Lds::DKV, stream, p, sp, (int)kv_blocks);
      if (split) launch_split_merge<float, D>(p, sp, MODE == BWD_TANGENT, stream);
      else launch_kv_merge<float, D>(p, MODE == BWD_TANGENT, false, stream);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    }
  }
  hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(BWD_NT), Lds::DKV, stream, p);
  launch_kv_merge<float, D>(p, MODE == BWD_TANGENT, false, stream);
  hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(BWD_NT), Lds::DQ, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}

// Small grids: blocks' tiles split (split.hpp).
template <typename T, int D, int MODE> static int launch_split(const BwdParams &p, bool no_go, hipStream_t stream) {
  using Cfg = Bwd2Cfg<T, D, MODE>;
  long long kv_blocks, blocks;
  const BwdSplit sp = split_of<D, false>(p.pr, MODE == BWD_DUAL, &kv_blocks, &blocks);
  auto kern = no_go ? bwd2_split_kernel<T, D, MODE, MODE != BWD_DUAL> : bwd2_split_kernel<T, D, MODE, true>;
  constexpr size_t LDS = Cfg::DKV_LDS > Cfg::DQ_LDS ? Cfg::DKV_LDS : Cfg::DQ_LDS;
  const int rc = allow_lds(reinterpret_cast<const void *>(kern), LDS);
  if (rc != 0) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(kv_blocks + blocks)), dim3(Cfg::NT), LDS, stream, p, sp, (int)kv_blocks);
  launch_split_merge<T, D>(p, sp, false, stream);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}

// six: all six gradients were asked for.  The dual launch then also writes what BwdFold says, and the tangent
// launch skips the kernels whose outputs exist already.
template <typename T, int D, int MODE, int MASK>
static int launch_bwd_mode(const BwdParams &p, bool six, hipStream_t stream) {
  using Cfg = BwdCfg<T, D, MODE>;
  const int nb = (p.pr.L + BWD_BLK - 1) / BWD_BLK;
  const long long blocks = (long long)nb * p.pr.Z * p.pr.H;
  if (blocks > 0x7fffffffLL) return -2;
  // the dk/dv kernels run one workgroup per 128 keys of a key/value head (the same count as for dq
  // when k, v have q's shape)
  const long long kv_blocks = (long long)((p.pr.Lk + BWD_BLK - 1) / BWD_BLK) * p.pr.Z * p.pr.Hk * p.pr.chunks;
  if (kv_blocks > 0x7fffffffLL) return -2;
  if (p.pr.drop_thr != 0) {
    // dropout: the direct-to-LDS kernels carry it, the register-staged ones for fp32 at D = 256
    if constexpr (sizeof(T) == 2 && D <= 128) {
      using Cfg2 = Bwd2Cfg<T, D, MODE>;
      const bool no_go = MODE == BWD_DUAL && p.go == nullptr;
      constexpr bool NG = MODE != BWD_DUAL;
      const bool grouped = p.pr.Hk != p.pr.H;
      if constexpr (MASK == MASK_NONE) {
        if (launch_both<D, MODE>(blocks, kv_blocks, p.pr.causal != 0, MASK_NONE, true, false, grouped, false)) {
          void (*kb)(const BwdParams, int);
          if (grouped) kb = no_go ? bwd2_both_kernel<T, D, MODE, MASK, NG, true, false, true> : bwd2_both_kernel<T, D, MODE, MASK, true, true, false, true>;
          else kb = no_go ? bwd2_both_kernel<T, D, MODE, MASK, NG, false, false, true> : bwd2_both_kernel<T, D, MODE, MASK, true, false, false, true>;
          const int rc = run_both(kb, p, kv_blocks, kv_blocks + blocks, Cfg2::DKV_LDS > Cfg2::DQ_LDS ? Cfg2::DKV_LDS : Cfg2::DQ_LDS, stream);
          if (rc != 0) return rc;
          launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
          return hipGetLastError() == hipSuccess ? 0 : -6;
        }
      }
      void (*kq)(const BwdParams) = no_go ? bwd2_dq_kernel<T, D, MODE, MASK, NG, false, true> : bwd2_dq_kernel<T, D, MODE, MASK, true, false, true>;
      size_t kv_lds = 0;
      void (*kkv)(const BwdParams) = pick_dkdv_for<T, D, MODE, MASK>(p, no_go, grouped, false, true, &kv_lds);
      int rc = allow_lds(reinterpret_cast<const void *>(kq), Cfg2::DQ_LDS);
      if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), kv_lds);
      if (rc != 0) return rc;
      hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(Cfg2::NT), kv_lds, stream, p);
      launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
      hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(Cfg2::NT), Cfg2::DQ_LDS, stream, p);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    } else if constexpr (sizeof(T) == 2 && D == 256 && MODE == BWD_DUAL) {
      using CfgP = BwdPairCfg<T, D>;
      const bool no_go = p.go == nullptr;
      const long long qblocks = (long long)((p.pr.L + CfgP::BLK - 1) / CfgP::BLK) * p.pr.Z * p.pr.H;
      const long long kblocks = (long long)((p.pr.Lk + CfgP::BLK - 1) / CfgP::BLK) * p.pr.Z * p.pr.Hk * p.pr.chunks;
      if (qblocks > 0x7fffffffLL || kblocks > 0x7fffffffLL) return -2;
      void (*kq)(const BwdParams) = no_go ? bwdp_dq_kernel<T, D, MASK, false, false, true> : bwdp_dq_kernel<T, D, MASK, true, false, true>;
      void (*kkv)(const BwdParams) = no_go ? bwdp_dkdv_kernel<T, D, MASK, false, true> : bwdp_dkdv_kernel<T, D, MASK, true, true>;
      int rc = allow_lds(reinterpret_cast<const void *>(kq), CfgP::DQ_LDS);
      if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), CfgP::DKV_LDS);
      if (rc != 0) return rc;
      hipLaunchKernelGGL(kkv, dim3((unsigned)kblocks), dim3(CfgP::NT), CfgP::DKV_LDS, stream, p);
      launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
      hipLaunchKernelGGL(kq, dim3((unsigned)qblocks), dim3(CfgP::NT), CfgP::DQ_LDS, stream, p);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    } else if constexpr (sizeof(T) == 2 && D == 256) {
      using CfgW = BwdWideCfg<T, D, MODE>;
      using CfgK = BwdWideKvCfg<T, D, MODE>;
      auto kq = bwdw_dq_kernel<T, D, MODE, MASK, true>;
      auto kkv = pick_wide_dkdv<T, D, MODE, MASK, true>(p);
      int rc = allow_lds(reinterpret_cast<const void *>(kq), CfgW::DQ_LDS);
      if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), CfgK::DKV_LDS);
      if (rc != 0) return rc;
      hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(CfgK::NT), CfgK::DKV_LDS, stream, p);
      launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
      hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(CfgW::NT), CfgW::DQ_LDS, stream, p);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    } else if constexpr (D <= 128) {
      return launch_bwd_f32<D, MODE, MASK, true>(p, blocks, kv_blocks, stream);
    } else {
      auto kq = bwd_dq_kernel<T, D, MODE, MASK, true>;
      auto kkv = bwd_dkdv_kernel<T, D, MODE, MASK, true>;
      int rc = allow_lds(reinterpret_cast<const void *>(kq), Cfg::DQ_LDS);
      if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), Cfg::DKV_LDS);
      if (rc != 0) return rc;
      hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(BWD_NT), Cfg::DKV_LDS, stream, p);
      launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
      hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(BWD_NT), Cfg::DQ_LDS, stream, p);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    }
  }
  if constexpr (sizeof(T) == 2 && D <= 128) {  // direct-to-LDS, double-buffered kernels
   {
    using Cfg2 = Bwd2Cfg<T, D, MODE>;
    // gO may be absent only in the dual mode (loss depends on O' alone)
    const bool no_go = MODE == BWD_DUAL && p.go == nullptr;
    constexpr bool NG = MODE != BWD_DUAL;  // the GO template argument of the kernels without gO
    void (*kq)(const BwdParams), (*kkv)(const BwdParams);
    const bool grouped = p.pr.Hk != p.pr.H;  // a key/value head serves several query heads
    using Fold = BwdFold<T, D>;
    bool run_q = true, run_kv = true;
    if constexpr (MODE == BWD_TANGENT) {
      run_q = !(six && Fold::DQ);
      run_kv = !(six && Fold::KV);
    }
    kq = pick_dq<T, D, MODE, MASK>(no_go, MODE == BWD_DUAL && six);
    if constexpr (MASK == MASK_BOOL) {
      if (p.pr.bits_q) kq = pick_dq<T, D, MODE, MASK_BITS>(no_go, MODE == BWD_DUAL && six);
    }
    size_t kv_lds = 0;
    kkv = pick_dkdv_for<T, D, MODE, MASK>(p, no_go, grouped, MODE == BWD_DUAL && six, false, &kv_lds);
    if constexpr (MASK == MASK_NONE && MODE != BWD_TANGENT) {
      if (p.pr.chunk_tiles == -1) return launch_split<T, D, MODE>(p, no_go, stream);
    }
    if (auto kb = pick_both<T, D, MODE, MASK>(p, no_go, grouped, six, blocks, kv_blocks)) {
      if constexpr (MODE == BWD_TANGENT) {
        if (six) return 0;  // the dual launch has made all six
      }
      constexpr bool ALL = D == 128 && MODE == BWD_DUAL;  // then dk', dv' have workgroups of their own
      const int rcb = run_both(kb, p, kv_blocks, (ALL && six ? 2 : 1) * kv_blocks + blocks, Cfg2::DKV_LDS > Cfg2::DQ_LDS ? Cfg2::DKV_LDS : Cfg2::DQ_LDS, stream);
      if (rcb != 0) return rcb;
      launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    }
    int rc = allow_lds(reinterpret_cast<const void *>(kq), Cfg2::DQ_LDS);
    if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), kv_lds);
    if (rc != 0) return rc;
    if (run_kv) {
      hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(Cfg2::NT), kv_lds, stream, p);
      launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, MODE == BWD_DUAL && six && Fold::KV, stream);
    }
    if (run_q) hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(Cfg2::NT), Cfg2::DQ_LDS, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -6;
   }
  } else if constexpr (sizeof(T) == 2 && D == 256 && MODE == BWD_DUAL) {
    // pairs of waves that share 32 rows and split the resident operands: every product formed once
    using CfgP = BwdPairCfg<T, D>;
    const bool no_go = p.go == nullptr;
    const long long qblocks = (long long)((p.pr.L + CfgP::BLK - 1) / CfgP::BLK) * p.pr.Z * p.pr.H;
    const long long kblocks = (long long)((p.pr.Lk + CfgP::BLK - 1) / CfgP::BLK) * p.pr.Z * p.pr.Hk * p.pr.chunks;
    if (qblocks > 0x7fffffffLL || kblocks > 0x7fffffffLL) return -2;
    void (*kq)(const BwdParams) = no_go ? bwdp_dq_kernel<T, D, MASK, false> : bwdp_dq_kernel<T, D, MASK, true>;
    if (!six && launch_both<D, MODE>(qblocks, kblocks, p.pr.causal != 0, MASK, false, false, false, false)) {
      void (*kb)(const BwdParams, int) = no_go ? bwdp_both_kernel<T, D, MASK, false> : bwdp_both_kernel<T, D, MASK, true>;
      const int rcb = run_both(kb, p, kblocks, kblocks + qblocks, CfgP::DQ_LDS > CfgP::DKV_LDS ? CfgP::DQ_LDS : CfgP::DKV_LDS, stream);
      if (rcb != 0) return rcb;
      launch_kv_merge<T, D>(p, false, false, stream);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    }
    if (six) kq = no_go ? bwdp_dq_kernel<T, D, MASK, false, true> : bwdp_dq_kernel<T, D, MASK, true, true>;
    void (*kkv)(const BwdParams) = no_go ? bwdp_dkdv_kernel<T, D, MASK, false> : bwdp_dkdv_kernel<T, D, MASK, true>;
    int rc = allow_lds(reinterpret_cast<const void *>(kq), CfgP::DQ_LDS);
    if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), CfgP::DKV_LDS);
    if (rc != 0) return rc;
    hipLaunchKernelGGL(kkv, dim3((unsigned)kblocks), dim3(CfgP::NT), CfgP::DKV_LDS, stream, p);
    launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
    hipLaunchKernelGGL(kq, dim3((unsigned)qblocks), dim3(CfgP::NT), CfgP::DQ_LDS, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -6;
  } else if constexpr (sizeof(T) == 2 && D == 256) {
    // without tangents in the launch two operands stay resident and one workgroup holds all 256 columns
    using CfgW = BwdWideCfg<T, D, MODE>;
    using CfgK = BwdWideKvCfg<T, D, MODE>;
    if (MODE == BWD_PLAIN && launch_both<D, MODE>(blocks, kv_blocks, p.pr.causal != 0, MASK, false, false, false, false)) {
      void (*kb)(const BwdParams, int) = bwdw_both_kernel<T, D, BWD_PLAIN, MASK, true>;
      if constexpr (MASK != MASK_NONE) {
        if (p.pr.chunks <= 1) kb = bwdw_both_kernel<T, D, BWD_PLAIN, MASK, false>;
      }
      using CfgKP = BwdWideKvCfg<T, D, BWD_PLAIN>;
      const int rcb = run_both(kb, p, kv_blocks, kv_blocks + blocks, CfgKP::DKV_LDS > CfgKP::DQ_LDS ? CfgKP::DKV_LDS : CfgKP::DQ_LDS, stream);
      if (rcb != 0) return rcb;
      launch_kv_merge<T, D>(p, false, false, stream);
      return hipGetLastError() == hipSuccess ? 0 : -6;
    }
    auto kq = bwdw_dq_kernel<T, D, MODE, MASK>;
    auto kkv = pick_wide_dkdv<T, D, MODE, MASK, false>(p);
    int rc = allow_lds(reinterpret_cast<const void *>(kq), CfgW::DQ_LDS);
    if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), CfgK::DKV_LDS);
    if (rc != 0) return rc;
    hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(CfgK::NT), CfgK::DKV_LDS, stream, p);
    launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
    // (six: the tangent launch of a six-gradient call, whose dq' the dual launch has written already)
    if (!(MODE == BWD_TANGENT && six)) hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(CfgW::NT), CfgW::DQ_LDS, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -6;
  } else if constexpr (D <= 128) {
    return launch_bwd_f32<D, MODE, MASK, false>(p, blocks, kv_blocks, stream);
  } else {
    auto kq = bwd_dq_kernel<T, D, MODE, MASK>;
    auto kkv = bwd_dkdv_kernel<T, D, MODE, MASK>;
    int rc = allow_lds(reinterpret_cast<const void *>(kq), Cfg::DQ_LDS);
    if (rc == 0) rc = allow_lds(reinterpret_cast<const void *>(kkv), Cfg::DKV_LDS);
    if (rc != 0) return rc;
    hipLaunchKernelGGL(kkv, dim3((unsigned)kv_blocks), dim3(BWD_NT), Cfg::DKV_LDS, stream, p);
    launch_kv_merge<T, D>(p, MODE == BWD_TANGENT, false, stream);
    hipLaunchKernelGGL(kq, dim3((unsigned)blocks), dim3(BWD_NT), Cfg::DQ_LDS, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -6;
  }
}

template <typename T, int D, int MASK>
static int launch_bwd_mask(const BwdParams &p, bool dual, bool tangent_grads, hipStream_t stream) {
  const long long rows = (long long)p.pr.Z * p.pr.H * p.pr.L;
  constexpr int RPB = BWD_NT / (D / 8);
  hipLaunchKernelGGL((bwd_prepass_kernel<T, D>), dim3((unsigned)((rows + RPB - 1) / RPB)), dim3(BWD_NT), 0,
                     stream, p, rows, dual ? 1 : 0);
  if (hipGetLastError() != hipSuccess) return -6;
  if (!dual) return launch_bwd_mode<T, D, BWD_PLAIN, MASK>(p, false, stream);
  int rc = launch_bwd_mode<T, D, BWD_DUAL, MASK>(p, tangent_grads, stream);
  if (rc == 0 && tangent_grads) rc = launch_bwd_mode<T, D, BWD_TANGENT, MASK>(p, true, stream);
  return rc;
}

int JVPFA_NAME(const BwdParams &p, int mask, bool dual, bool tangent_grads, hipStream_t stream) {
  switch (mask) {
    case MASK_NONE: return launch_bwd_mask<JVPFA_T, JVPFA_D, MASK_NONE>(p, dual, tangent_grads, stream);
    case MASK_BOOL: return launch_bwd_mask<JVPFA_T, JVPFA_D, MASK_BOOL>(p, dual, tangent_grads, stream);
    case MASK_ADD: return launch_bwd_mask<JVPFA_T, JVPFA_D, MASK_ADD>(p, dual, tangent_grads, stream);
  }
  return -3;
}

}  // namespace jvpfa
