// Small grids: when a launch has fewer workgroups than the GPU has compute units (one sequence of a few thousand tokens, a
// handful of heads), or causal ones of very different length, the streamed tiles of blocks of owned rows are dealt to several
// workgroups ("shares", Deal).  Each leaves fp32 partial results in a workspace; the forward's merge kernel combines them with
// the online-softmax merge (every running quantity is linear in p once the reference points m and c are made common), the
// backward's adds them up.  The kernels that can: 16-bit element types without a mask (forward D = 64 or 128, backward D <= 128)
// and fp32 at D <= 128 with any mask, all without dropout.  Non-causal blocks get as many workgroups each, causal ones by their length.
// Where key/value heads are few (grouped heads), the backward deals the query heads of each to several workgroups (bwd_kv_chunks).
// And it runs its dk/dv and dq workgroups in one launch where that leaves fewer units idle (launch_both).  The reference has
// nothing like it (one program per 32 query rows, jvp_attention.py:2474).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <array>
#include <atomic>

#include "common.hpp"
#include "params.hpp"

namespace jvpfa {

// make() of these sizes, from the last ones that this thread asked for: a plan is a function of sizes alone, a call asks for it
// twice (its workspace and its launch), and making it takes 1 - 3 us.  As many as the attention shapes of a large model; looking
// through them takes 0.02 us, where eight, in turn over nine shapes, were made anew on every call.
template <typename Plan, int N, typename Make> inline Plan remembered(const std::array<int, N> &sizes, Make make) {
  constexpr int SLOTS = 32;
  struct Entry {
    std::array<int, N> sizes;
    Plan plan;
    bool used;
  };
  static thread_local Entry entries[SLOTS];
  static thread_local int next;  // (below SLOTS: a count of all plans would overflow in a long run)
  for (const Entry &e : entries)
    if (e.used && e.sizes == sizes) return e.plan;
  Entry &e = entries[next];
  next = (next + 1) % SLOTS;
  e = {sizes, make(), true};
  return e.plan;
}

struct SplitPlan {
  int chunks, chunk_tiles;  // as in Problem: Deal::most, Deal::step
};

// blocks: workgroups of the launch without a split; ntiles_max: streamed tiles of its longest block.
inline SplitPlan split_plan(long long blocks, int ntiles_max, int cus) {
  SplitPlan s = {1, 0};
  if (cus <= 0 || blocks <= 0 || 2 * blocks > cus) return s;
  // one workgroup per compute unit at most: a workgroup has a fixed cost of about three tiles (its first loads,
  // filling and draining the pipeline), so a second round of short chunks costs more than it saves
  long long want = cus / blocks;
  if (want > 8) want = 8;
  if (want > ntiles_max / 2) want = ntiles_max / 2;    // a chunk is at least two tiles
  if (want < 2) return s;
  const int tiles = (int)((ntiles_max + want - 1) / want);
  s.chunks = (ntiles_max + tiles - 1) / tiles;
  return s;
}

// What a launch takes whose blocks differ in length (causal) and are dealt as Deal says, in us, with the longest workgroups first:
// what the longest takes; where there are more workgroups than places for them also their sum dealt out and a share of the longest
// for the end, and two of the length at which the places run out.  The constants of a kernel fit what its shares of 1/2 ... 1/8 of the
// longest block took (17 shapes of 32 - 512 blocks for each of the backward's, within 7 %; what is picked by them is within 8 % of the
// best of those shares, 1 % on average).
struct DealCost {
  double tile;     // of 64 streamed rows
  double start;    // a workgroup's first loads, filling and draining its pipeline
  double merge;    // the launch that adds the shares up
  double traffic;  // a share of weight 1 for every unit, written and read again
  double end;      // of the longest, see above
  int places;      // workgroups that share a compute unit without taking longer
  double pair;     // of two workgroups in turn, see above
};
// A second launch and its workspace take 7 us on the host, and an eager step of forward and backward that takes the GPU less than
// some 110 us is bound by the host (B1 H2 L300 D64 fp32, both outputs' gradients, in shares: 57 -> 47 us on the GPU, 112 -> 127 us a
// step).  So a split that adds a launch is for forwards and backwards that take at least this long by the account, and a forward
// has to save what the launch costs; a backward of that length, which the host does not bound, has to be faster by its account
// alone.  A caller without that host time (a captured graph, the C ABI) has the same plans: that backward stays at 57 us there.
constexpr double SPLIT_LAUNCH_US = 7.0, SPLIT_FORWARD_US = 40.0, SPLIT_BACKWARD_US = 65.0;
class DealTime {
 public:
  DealTime(long long cus, const DealCost &cost) : cus_(cus), c_(cost) { std::fill(of_length_, of_length_ + TOP + 1, 0); }
  // scale: a tile of this role in tiles; weight: of its shares
  template <typename N> void add(const Deal &d, long long heads, double scale, double weight, N tiles_of) {
    for (int order = d.first; order < d.last; ++order) {
      const int n = tiles_of(order), count = d.shares(order);
      const double length = (n + count - 1) / count * scale;
      const long long w = count * heads;
      sum_ += length * c_.tile * w + w * c_.start, workgroups_ += w, longest_ = std::max(longest_, length * c_.tile);
      alike_ = alike_ && (workgroups_ == w || length == last_), last_ = length;
      of_length_[std::min((int)length, TOP)] += w;
      if (count > 1) parts_ += weight * w;
    }
  }
  double total() const {
    const long long places = cus_ * c_.places;
    double time = longest_ + c_.start;
    if (workgroups_ > places) {
      int length = TOP;
      for (long long n = of_length_[TOP]; n <= places && length > 0; n += of_length_[length]) --length;
      time = std::max({time, sum_ / places + c_.end * longest_, 2.0 * (c_.pair * length * c_.tile + c_.start)});
      if (alike_) time = std::max(time, (double)((workgroups_ + places - 1) / places) * (longest_ + c_.start));
    }
    return time + (parts_ > 0.0 ? c_.merge + c_.traffic * parts_ / cus_ : 0.0);
  }

 private:
  static constexpr int TOP = 512;
  long long cus_;
  DealCost c_;
  bool alike_ = true;  // one length: whole passes over the places
  double sum_ = 0.0, longest_ = 0.0, parts_ = 0.0, last_ = 0.0;
  long long workgroups_ = 0, of_length_[TOP + 1];
};

// Compute units of the current device (0 if it cannot be asked), looked up once per device.  Callable from any
// thread: the cache is atomic, and two threads that both find it empty store the same value.
inline int device_cus() {
  static std::atomic<int> cached[64];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 0;
    n = n > 0 ? n : -1;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n > 0 ? n : 0;
}

// Workspace of the forward: per chunk and query row 2 D accumulator values (O, T, not yet divided by l) and
// four statistics (m, l, mu_acc, c).
inline size_t fwd_part_floats(int chunks, long long rows, int D, bool dual) { return (size_t)chunks * rows * ((dual ? 2 : 1) * (size_t)D + 4); }
// The 16-bit kernels that can split: D = 64 or 128, no mask (the software-pipelined forward).  Tiles are 64 wide, blocks 128 rows.
template <typename P> inline bool split_capable(const P &p) {
  return p.dtype != 2 && (p.D == 128 || p.D == 64) && p.mask_kind == 0 && !(p.dropout_p > 0.f);
}
// fp32 at D <= 128 (without dropout): a tile takes three to nine times as long as in 16 bits, so that a split is worth it for
// any grid that leaves units idle, also by a second pass that is not full: 192 blocks in quarters are three passes of a quarter.
// Whole blocks -> this, us, dual / without tangents:
//   D64  B1 H8 L512 51 -> 33 / whole (24); H2 L4096 causal 342 -> 82 / 153 -> 49; B2 H6 L777 with a bias 79 -> 49 / whole (39)
//   D128 B1 H8 L512 186 -> 55 / 70 -> 33; H16 L1024 366 -> 208 / 135 -> 83; H40 L1000 732 -> 599 / 254 -> 214
//   D32  B1 H12 L1024 causal 58 -> 29 / whole (33)
template <typename P> inline SplitPlan fwd_split_plan_f32(const P &p, int Lk, bool dual, int cus) {
  SplitPlan best = {1, 0};
  const int nblk = (p.L + 127) / 128;
  const long long heads = (long long)p.Z * p.H, blocks = heads * nblk;
  if (p.D > 128 || p.dropout_p > 0.f || cus <= 0 || blocks >= 2 * cus) return best;
  const bool shared = !dual && p.D <= 64;  // two workgroups to a unit, so only as many as there are units
  const double tile = p.D == 128 ? (dual ? 22.4 : 8.1) : p.D == 64 ? (dual ? 5.6 : 2.4) : (dual ? 3.3 : 1.75);
  const DealCost cost = {tile, 6.0, 6.0, 8.4 * p.D / 64 * (dual ? 1.0 : 0.5), 0.25, 1, 1.0};
  auto n = [&](int order) { return ((p.causal ? std::min((order + 1) * 128, Lk) : Lk) + 63) / 64; };
  auto time = [&](const SplitPlan &s) {
    DealTime t(cus, cost);
    t.add({s.chunks, s.chunk_tiles, 0, nblk}, heads, 1.0, 1.0, n);
    return t.total();
  };
  const int longest = n(nblk - 1);
  if (time(best) < SPLIT_FORWARD_US) return best;
  double least = std::min(time(best) / 1.05, time(best) - SPLIT_LAUNCH_US);
  for (int most = 2; most <= 8 && most <= longest; ++most) {
    const SplitPlan s = {most, p.causal ? ((longest + 1) / 2 + most - 1) / most * 2 : 0};
    if (blocks * most > (shared ? 1 : 4) * cus) break;
    const double t = time(s);
    if (t < least) least = t, best = s;
  }
  return best;
}
template <typename P> inline SplitPlan fwd_split_plan_16(const P &p, int Lk, bool dual, int cus) {
  const SplitPlan none = {1, 0};
  if (!split_capable(p)) return none;
  const long long blocks = (long long)((p.L + 127) / 128) * p.Z * p.H;
  int keys = Lk;  // of the longest query block (causal: the last one sees keys up to its own last row)
  if (p.causal && ((p.L + 127) / 128) * 128 < keys) keys = ((p.L + 127) / 128) * 128;
  const int ntiles = (keys + 63) / 64;
  // D = 64: a tile takes half the time (1.8 us with tangents, 0.9 without), so what a split costs, 8 - 10 us with the merge, is
  // worth it from 16 or 32 tiles on (with fewer it is slower, L512 plain 10.8 -> 12.1).  Measured, bf16 B1, unsplit -> split, dual
  // and plain: H4 L1024 34 -> 28 and 18 -> unsplit (19); H4 L2048 62 -> 33 and 32 -> 21; H8 L2048 63 -> 42 and 33 -> 26;
  // H2 L4096 118 -> 44 and 61 -> 28; H4 L4096 119 -> 66 and 61 -> 40.
  if (p.D == 64 && ntiles < (dual ? 16 : 32)) return none;
  SplitPlan even = split_plan(blocks, ntiles, cus);
  // causal: shares of that length for the shorter blocks, too (all blocks in as many: H12 L693 D128 without tangents 18.8 -> 20.6 us)
  if (p.causal && even.chunks > 1) even.chunk_tiles = (ntiles + even.chunks - 1) / even.chunks;
  if (!p.causal || blocks >= cus || ntiles < 12) return even;
  // Causal: shares of one length for all blocks (Deal), where the account of DealTime says that it is worth a twentieth; fewer
  // blocks than there are units, whose longest ones alone set the time otherwise.  From as many blocks as units on every block
  // is one workgroup's (some launches of up to half as many again would gain as well, 1.1 - 1.3 times).
  // The costs fit what was measured of shares of 1/2 ... 1/8.  Causal, bf16, B1, us, before -> this, dual / without tangents:
  //   D128 H8 L2048 56 -> 49 / 34 -> 29; H12 L2048 80 -> 65 / whole (42); H6 L4096 146 -> 99 / 77 -> 50; H2 L8192 159 -> 123 / 84 -> 64
  //   D64  H12 L1500 43 -> 32 / whole (26); H6 L4096 103 -> 65 / 62 -> 38; H2 L8192 111 -> 80 / 66 -> 49; H1 L16384 207 -> 129 / 121 -> 67
  // Slower than equal shares of every block: a few of one to three heads, by 2 - 5 % and less than 1 us (D64 H1 L3128 19.9 -> 20.8).
  const bool wide = p.D == 128;
  const DealCost cost = {wide ? (dual ? 2.45 : 1.2) : (dual ? 1.6 : 0.85), wide && dual ? 6.0 : 5.0, 7.0, 11.0 * p.D / 128 * (dual ? 1.0 : 0.5), 0.25, 1, 1.0};
  const int nblk = (p.L + 127) / 128;
  auto time = [&](int most, int step) {
    // The merge reads a row's shares one after another.  Counted where three or more equal shares are the alternative and blocks
    // are short: H3 L1990 D64 without tangents in 4, 5, 8 shares 19.0, 19.2, 20.8 us; H6 L1111 D128 in 3, 5 shares 20.9, 22.6
    // (equal ones 21.5); over a hundred such launches 2.3 % less, 5 % more at worst.  In others the account is too coarse for it
    // (H1 L16384 D64, two equal shares: 67.5 us in 6, but 84 in the 3 that it would pick; H1 L8483, three: 32.6 in 7, 34.9 in 6).
    DealCost with_merge = cost;
    if (even.chunks > 2 && ntiles <= 64) with_merge.merge = 3.5 + 1.0 * most;
    DealTime t(cus, with_merge);
    t.add({most, step, 0, nblk}, (long long)p.Z * p.H, 1.0, 1.0, [&](int order) { return (std::min((order + 1) * 128, Lk) + 63) / 64; });
    return t.total();
  };
  SplitPlan best = none;
  if (even.chunks == 1 && time(1, 0) < SPLIT_FORWARD_US) return none;
  double least = std::min(time(1, 0) / 1.06, time(1, 0) - (even.chunks == 1 ? SPLIT_LAUNCH_US : 0.0));
  for (int most = 2; most <= 8; ++most) {
    const int step = ((ntiles + 1) / 2 + most - 1) / most * 2;  // the longest block, of ntiles, gets `most` shares
    if (step < 4 || blocks * most > 3 * cus) break;
    const double t = time(most, step);
    if (t < least) least = t, best = {most, step};
  }
  return best;
}

template <typename P> inline SplitPlan fwd_split_plan(const P &p, int Lk, bool dual) {
  const int cus = device_cus(), kind = (p.dtype == 2) | (p.causal != 0) << 1 | dual << 2 | (p.mask_kind != 0) << 3 | (p.dropout_p > 0.f) << 4;
  return remembered<SplitPlan, 7>({p.D, p.Z, p.H, p.L, Lk, kind, cus},
                                  [&] { return p.dtype == 2 ? fwd_split_plan_f32(p, Lk, dual, cus) : fwd_split_plan_16(p, Lk, dual, cus); });
}

// Backward with grouped heads.  A dk/dv workgroup owns 128 keys of a key/value head and works through the query heads
// of its group one after another: 4 key/value heads for 16 query heads make a quarter of the workgroups, each four
// times as long.  Where that leaves compute units idle, the group's query heads are dealt to `chunks` workgroups that
// leave fp32 shares of dk, dv (and dk', dv'), which bwd_kv_merge_kernel adds up (group_share: they may differ by a head).
// The number is the one with the least time by this account, in passes of one workgroup over one query head:
//   * a compute unit gets ceil(workgroups / units) of them, and waits for 5 % of one; causal, whose work falls from block to
//     block and is dealt longest first, half the work and a quarter of the longest share, but no less than that share;
//   * at 16 bits and D <= 64, where two or three workgroups share a unit, one alone runs at 0.6 of their joint rate (causal:
//     half of the longest share);
//   * a share costs about 4 tiles of 64 queries (its first loads, and 16 bytes per element written and read; in fp32, where
//     the products take 16 times as long, a sixteenth of that).
// At most 10 workgroups per unit, so that the shares take no more than 10 * units * 128 * D * 8 bytes (twice that with tangent
// gradients), whatever the group.  Measured, forward + backward, bf16, one share -> this rule (in brackets: with as many
// shares as the group has heads): B4 H16 over 4, L1500 D64, causal, dropout 363 -> 184 us; B8 H71 over 1, L2048 D64 5.51 ->
// 2.78 ms (2.79, and 595 MB of shares); B2 H28 over 4, D128, L4096 1.98 -> one share (2.02), L4800 3.57 -> 2.92, causal L4096
// 3.48 -> 2.64; fp16 B4 H16 over 8, L1024 D256 0.35 -> one share (0.40); fp32 B2 H16 over 4, L2048 D64 2.17 -> 1.15.
template <typename P> inline int bwd_kv_chunks(const P &p, int Lk, int Hk) {
  const int group = p.H / Hk, cus = device_cus();
  const long long blocks = (long long)((Lk + 127) / 128) * p.Z * Hk;
  if (cus <= 0 || group == 1) return 1;
  const bool shared = p.dtype != 2 && p.D <= 64;
  const double share_cost = (p.dtype == 2 ? 0.25 : 4.0) / ((p.L + 63) / 64);
  int best = 1;
  double least = 0.0;
  for (int c = 1; c <= group && (c == 1 || blocks * c <= 10LL * cus); ++c) {
    const double heads = (group + c - 1) / c, per_cu = (double)((blocks * c + cus - 1) / cus);
    double time = p.causal ? std::max(heads, 0.5 * group * blocks / cus + (shared ? 0.5 : 0.25) * heads) : (per_cu + 0.05) * heads;
    if (shared && per_cu < 2.0) time /= 0.6;
    if (c > 1) time += per_cu * share_cost;
    if (c == 1 || time < least) best = c, least = time;
  }
  return best;
}
// ... floats of the shares: dk, dv, and dk', dv' where one kernel makes all four (tangent_grads)
template <typename P> inline size_t bwd_part_floats(const P &p, int Lk, int Hk, int chunks, bool tangent_grads) {
  return (size_t)chunks * (tangent_grads ? 4 : 2) * ((size_t)p.Z * Hk * Lk * p.D);
}

// Backward of small grids (16-bit element types, D <= 128, no mask, no dropout, one query head per key/value head, not six
// gradients): the tiles that a block streams are dealt to several workgroups, dq's and dk/dv's in one launch, which leave fp32
// shares that bwd_split_merge_kernel adds up.
//   * As many workgroups as there are compute units; causal, whose blocks have half the tiles on average, up to three a block and
//     three a unit where that leaves 10 tiles to a share (with fewer the empty and the short ones cost more than they bring: H16
//     L1024 D128 60 -> 72 us, H6 L1024 42 -> 48; six for three at H2 L4096 98 -> 119).  Where a unit holds one of them (D = 128;
//     D = 64 with tangents) and both roles would be cut so, only if the blocks unsplit fit the units (D = 64: and an eighth), and
//     at D = 128 two a block only if they fit three quarters. Causal, unsplit / split, at 192, 240 - 256, 288 - 320, 384 blocks
//     of both roles: D128 dual 1.10, 0.93 (two), 1.17 (three), 0.83 - 0.94, 0.76 - 0.85, plain 0.99, 0.86, 1.00, 0.75 - 0.82,
//     0.67 - 0.79; D64 dual 1.21 - 1.46, 1.03 - 1.50, 0.85 - 1.02, 0.76 - 0.87, plain 1.27, 1.29, 1.27, 1.03 - 1.23; D32 1.44,
//     1.41, 1.35, 0.98 - 1.08.
//   * No share under 3 tiles at D = 128, where a tile takes 4 us, 4 at D = 64, 6 at D = 32; and without tangents none that saves
//     a block fewer than 7 tiles of 2 us at D = 128 (H8 L700 28 -> 31 us), the launch fewer than 6 of 1 us at D = 64 (H16 L512 19
//     -> 22 us): the merge takes 5 - 10 us.
//   * At D = 128 shares of up to 8 tiles only where they shorten the longest workgroup of the launch (a dk/dv tile takes 1.25 of
//     a dq tile) by 3 tiles, and then, as the merge grows with what it reads, only up to a number of them: unsplit / split, dual,
//     at 2, 8, 12, 16 heads and 512 rows 1.22, 1.06, 1.05, 0.94, causal 1.26, 1.16, 1.14, 1.09; 384 rows 1.15, 0.98, 1.01, 0.94,
//     causal 1.16, 1.06, 1.00, 1.00.
// Measured, bf16 B1, backward, unsplit -> split, dual / plain: D128 H1 L1024 65 -> 32 / 35 -> 23 us, H4 L1024 65 -> 38 / 36 ->
// 28, H2 L2048 120 -> 53 / 62 -> 35, H4 L2048 121 -> 85 / 62 -> 49, H2 L4096 231 -> 147 / 116 -> 77, causal H2 L4096 228 -> 98 /
// 115 -> 56, H4 L4096 237 -> 156 / 117 -> 96; D64 H4 L1024 49 -> 28 / 31 -> 23, H2 L2048 90 -> 38 / 55 -> 29, causal H4 L4096 173
// -> 116; D32 H4 L1024 34 -> 25 / 24 -> 19, H4 L2048 63 -> 41 / 44 -> 31, causal H4 L4096 121 -> 68.
struct BwdSplitPlan {
  int chunks_q, tiles_q, chunks_k, tiles_k;
  bool any() const { return chunks_q > 1 || chunks_k > 1; }
};
inline BwdSplitPlan bwd_split_plan(int D, int Z, int H, int L, int Lk, bool causal, bool dual, long long cus = device_cus()) {
  const long long bq = (long long)((L + 127) / 128) * Z * H, bk = (long long)((Lk + 127) / 128) * Z * H;
  const int reach = (L + 127) / 128 * 128, nq = ((causal && reach < Lk ? reach : Lk) + 63) / 64, nk = (L + 63) / 64;
  const int least = D == 128 ? 3 : D == 64 ? 4 : 6;
  BwdSplitPlan s = {1, nq, 1, nk};
  auto deal = [&](int n, int &chunks, int &tiles) {  // n: tiles of the longest block
    long long c = std::min<long long>(cus / (bq + bk), n / least);
    if (causal) {
      const long long more = std::min<long long>({3, 3 * cus / (bq + bk), n / 10});
      const bool alone = D == 128 || (D == 64 && dual), both = std::min(nq, nk) >= 20;
      const bool fits = D == 64 ? 8 * (bq + bk) <= 9 * cus : (more > 2 ? 1.0 : 0.75) * cus >= bq + bk;
      if (!alone || !both || fits) c = std::max(c, more);
    }
    c = std::min<long long>(c, 8);
    if (c < 2) return;
    const int per = (int)((n + c - 1) / c);
    if (D == 128 && !dual && n - per < 7) return;
    tiles = per, chunks = (n + per - 1) / per;
  };
  deal(nq, s.chunks_q, s.tiles_q);
  deal(nk, s.chunks_k, s.tiles_k);
  if (D == 64 && !dual && std::max(nq, nk) - std::max(s.tiles_q, s.tiles_k) < 6) return {1, nq, 1, nk};
  const bool short_q = s.chunks_q > 1 && nq <= 8, short_k = s.chunks_k > 1 && nk <= 8;
  if (D == 128 && (short_q || short_k)) {
    auto longest = [](int q, int k) { return std::max((double)q, 1.25 * k); };
    const double saved = longest(short_q ? nq : s.tiles_q, short_k ? nk : s.tiles_k) - longest(s.tiles_q, s.tiles_k);
    const double most = (saved >= 4.0 ? 0.75 : 0.3) + (causal ? 0.25 : 0.0);
    if (saved < 3.0 || (double)(s.chunks_q * bq + s.chunks_k * bk) > most * cus) {
      if (short_q) s.chunks_q = 1, s.tiles_q = nq;
      if (short_k) s.chunks_k = 1, s.tiles_k = nk;
    }
  }
  return s;
}
// The deal of either role's blocks that a launch goes by.  Causal, from 12 tiles on, where the account of DealTime says that it is
// shorter than with whole blocks: shares of one length for all blocks of both roles, so that the long ones get most of them.
// Causal, bf16, B1, us, before -> this, with tangents / without:
//   D128 H9 L2048 129 -> 109 / whole (65); H7 L2500 156 -> 124 / 78 -> 67; H2 L12000 717 -> 598 / 334 -> 265
//   D64  H6 L4096 174 -> 142 / 85 -> 70; H1 L30000 1218 -> 1109 / 712 -> 458; H3 L5000 136 -> 122 / 58 -> 60
//   D32  H6 L4096 118 -> 86 / 50 -> 44; H1 L8192 91 -> 60 / 63 -> 36
// H12 and H16 L1024 at any D stay whole, though shares would take D128 68 -> 57 and 69 -> 65, D64 50 -> 43 / 31 -> 29, D32 35 -> 24 / 24 -> 20:
// they are shorter than SPLIT_BACKWARD_US.  Slower: D64 H3 L4700 - L5100 without tangents, by 1 - 3 %.
// Otherwise shares of the length that bwd_split_plan says.
struct BwdDeal {
  Deal q, k;
  bool any() const { return q.most > 1 || k.most > 1; }
};
inline BwdDeal make_bwd_deal(int D, int Z, int H, int L, int Lk, bool causal, bool dual, long long cus = device_cus()) {
  const int bq = (L + 127) / 128, bk = (Lk + 127) / 128;
  const BwdSplitPlan even = bwd_split_plan(D, Z, H, L, Lk, causal, dual, cus);
  if (!causal) return {{even.chunks_q, 0, 0, bq}, {even.chunks_k, 0, 0, bk}};
  auto step_of = [](int chunks, int tiles) { return chunks > 1 ? tiles : 0; };
  // (in the account with shares of whole blocks, two tiles: what its pick was measured with)
  auto rounded = [](const BwdDeal &d) { return BwdDeal{{d.q.most, (d.q.step + 1) / 2 * 2, d.q.first, d.q.last}, {d.k.most, (d.k.step + 1) / 2 * 2, d.k.first, d.k.last}}; };
  const long long heads = (long long)Z * H;
  // tiles of the longest blocks; key blocks that a query sees
  const int nq = (std::min(bq * 128, Lk) + 63) / 64, nk = (L + 63) / 64, live = std::min(bk, bq);
  const BwdDeal alike = {{even.chunks_q, step_of(even.chunks_q, even.tiles_q), 0, bq}, {even.chunks_k, step_of(even.chunks_k, even.tiles_k), bq - live, bq}};
  if (cus <= 0 || std::max(nq, nk) < 12 || heads * (bq + bk) >= 2 * cus) return alike;
  const DealCost cost = D == 128 ? (dual ? DealCost{3.0, 2.9, 6.4, 9.9, 0.34, 1, 1.0} : DealCost{1.5, 3.9, 7.0, 6.1, 0.14, 1, 1.0})
                        : D == 64 ? (dual ? DealCost{2.0, 6.0, 4.2, 3.4, 0.2, 1, 1.0} : DealCost{1.2, 9.0, 3.6, 2.3, 0.4, 2, 0.7})
                                  : (dual ? DealCost{1.5, 5.5, 5.0, 2.1, 0.57, 2, 0.5} : DealCost{1.0, 4.5, 3.0, 1.8, 0.15, 2, 0.7});
  constexpr double KEYS = 1.25;  // a dk/dv tile in dq tiles
  auto time = [&](const BwdDeal &d) {
    DealTime t(cus, cost);
    t.add(d.q, heads, 1.0, 1.0, [&](int order) { return (std::min((order + 1) * 128, Lk) + 63) / 64; });
    t.add(d.k, heads, KEYS, 2.0, [&](int order) { return (L - 128 * (bq - 1 - order) + 63) / 64; });
    return t.total();
  };
  BwdDeal best = {{1, 0, 0, bq}, {1, 0, bq - live, bq}};
  double least = time(best) * (dual && D == 64 ? 1.07 : 1.0);  // (the account is fitted to shares; of whole blocks with tangents it makes 7 % too little at D = 64)
  if (!alike.any() && least < SPLIT_BACKWARD_US) return alike;
  if (alike.any()) least = std::min(least, 0.92 * time(rounded(alike)));  // (closer than that the account does not tell them apart)
  const double longest = std::max((double)nq, KEYS * nk);
  for (const int j : {4, 5, 6, 8, 12, 16}) {  // shares of 1/2 ... 1/8 of the longest block
    const double share = longest * 2 / j;
    auto deal = [&](int n, double t, int first, int last) {
      const int most = std::min(8, std::max(1, (int)(n * t / share + 0.99)));
      return Deal{most, most > 1 ? ((n + 1) / 2 + most - 1) / most * 2 : 0, first, last};
    };
    const BwdDeal d = {deal(nq, 1.0, 0, bq), deal(nk, KEYS, bq - live, bq)};
    if ((d.q.most > 1 && d.q.step < 4) || (d.k.most > 1 && d.k.step < 4) || heads * (d.q.most * bq + 2 * d.k.most * bk) > 6 * cus) break;
    const double t = time(d);
    if (t < least) least = t, best = d;
  }
  return best.any() ? best : alike;
}
// ... and in fp32 at D <= 128 (without dropout, one query head per key/value head; any mask, six gradients as well), by the same
// reasons as the forward.  Whole blocks -> this, us, with tangents / without:
//   D64  B1 H8 L512 82 -> 41 / whole (43); H12 L1024 causal 159 -> 104 / 78 -> 53; B3 H4 L640 padded 115 -> 72 / whole (65);
//        H2 L4096 causal 584 -> 249 / 278 -> 118; six gradients H4 L900 208 -> 93
//   D128 B1 H8 L512 336 -> 113 / 133 -> 55; H12 L1024 causal 670 -> 334 / 255 -> 146
//   D32  B1 H2 L4096 causal 361 -> 145 / 204 -> 63
inline BwdDeal make_bwd_deal_f32(int D, int Z, int H, int L, int Lk, bool causal, bool dual, long long cus = device_cus()) {
  const int bq = (L + 127) / 128, bk = (Lk + 127) / 128, live = causal ? std::min(bk, bq) : bk;
  const long long heads = (long long)Z * H;
  auto nq = [&](int order) { return ((causal ? std::min((order + 1) * 128, Lk) : Lk) + 63) / 64; };
  auto nk = [&](int order) { return (L - (causal ? 128 * (bq - 1 - order) : 0) + 63) / 64; };
  const int k0 = causal ? bq - live : 0, k1 = causal ? bq : bk;  // orders of the key blocks that a query sees
  BwdDeal best = {{1, 0, 0, bq}, {1, 0, k0, k1}};
  if (cus <= 0 || heads * (bq + bk) >= 4 * cus) return best;
  constexpr double KEYS = 1.3;  // a dk/dv tile in dq tiles
  const double tile = D == 128 ? (dual ? 32.0 : 12.5) : D == 64 ? (dual ? 7.5 : 3.4) : (dual ? 4.6 : 2.4);
  const DealCost cost = {tile, 6.0, 6.0, 4.2 * D / 64, 0.12, D == 32 && !dual ? 2 : 1, 1.0};
  auto time = [&](const BwdDeal &d) {
    DealTime t(cus, cost);
    t.add(d.k, heads, KEYS, 2.0, nk);
    t.add(d.q, heads, 1.0, 1.0, nq);
    return t.total();
  };
  const int longest_q = nq(bq - 1), longest_k = nk(k1 - 1);
  // whole blocks: in one launch, or in two that each end with units idle
  const double apart = (double)((heads * bq + cus - 1) / cus) * (longest_q * tile + cost.start) + (double)((heads * live + cus - 1) / cus) * (longest_k * KEYS * tile + cost.start);
  double least = std::min(time(best), apart) / 1.06;
  if (least < SPLIT_BACKWARD_US) return best;
  const double longest = std::max((double)longest_q, KEYS * longest_k);
  for (const int j : {3, 4, 5, 6, 8, 10, 12, 16}) {
    auto deal = [&](int n, double scale, int first, int last) {
      const int most = std::min({8, n, std::max(1, (int)(n * scale * j / (2 * longest) + 0.99))});
      return Deal{most, causal && most > 1 ? ((n + 1) / 2 + most - 1) / most * 2 : 0, first, last};
    };
    const BwdDeal d = {deal(longest_q, 1.0, 0, bq), deal(longest_k, KEYS, k0, k1)};
    if (heads * (d.q.most * bq + 2 * d.k.most * bk) > 8 * cus) break;
    const double t = time(d);
    if (d.any() && t < least) least = t, best = d;
  }
  return best;
}
inline BwdDeal bwd_deal(bool f32, int D, int Z, int H, int L, int Lk, bool causal, bool dual, long long cus = device_cus()) {
  return remembered<BwdDeal, 7>({D, Z, H, L, Lk, f32 | causal << 1 | dual << 2, (int)cus},
                                [&] { return f32 ? make_bwd_deal_f32(D, Z, H, L, Lk, causal, dual, cus) : make_bwd_deal(D, Z, H, L, Lk, causal, dual, cus); });
}
template <typename P> inline BwdDeal bwd_deal_of(const P &p, int Lk, int Hk, bool tangent_grads, bool dual) {
  if (p.dtype == 2 && p.D <= 128 && !(p.dropout_p > 0.f) && Hk == p.H) return bwd_deal(true, p.D, p.Z, p.H, p.L, Lk, p.causal != 0, dual);
  if (p.dtype == 2 || p.D > 128 || p.mask_kind != 0 || p.dropout_p > 0.f || Hk != p.H || tangent_grads) return {{1, 0, 0, 0}, {1, 0, 0, 0}};
  return bwd_deal(false, p.D, p.Z, p.H, p.L, Lk, p.causal != 0, dual);
}
template <typename P> inline size_t bwd_split_floats(const P &p, int Lk, const BwdDeal &d) {
  const size_t heads = (size_t)p.Z * p.H;
  return heads * p.D * ((d.q.most > 1 ? (size_t)d.q.most * p.L : 0) + (d.k.most > 1 ? (size_t)d.k.most * 2 * Lk : 0));
}

// Whether dk/dv and dq go into one launch (bwd2_both_kernel): it has one end with idle compute units instead of two, and where a
// kernel has to take both roles' registers fewer of its workgroups share a unit.  So: up to a number of blocks (in units of
// compute units) that depends on how many do.  mask: as the kernels read it.  twin: the launch has a capped kernel (both_two_wgs
// says which of the two runs it). D = 128 (one workgroup a unit either way, but for the dq kernel without tangents): causal and
// masked launches up to 2.5; others where the launches would round up to more passes over the units than the one does, 0.6 of a
// pass for its end. Measured, bf16, backward, two launches -> one, 288 / 544 / 704 / 1024 - 1152 blocks (dual unless said): D128
// 269 -> 205, 721 -> 607, 490 -> 492, 1236 -> 1135 us, causal 139 -> 111, 323 -> 316, 295 -> 290; plain 123 -> 100, 332 -> 285,
// 233 -> 237; D64 (2wg) causal 1024 blocks 314 -> 300, 1152 without a mask 731 -> 677, 1536 615 -> 602; D64 plain 69 -> 54, 164
// -> 147, 121 -> 118, 260 -> 245 us, 2048 blocks 471 -> 479; D32 88 -> 81, 253 -> 196, 171 -> 155, 462 -> 415, 2048 blocks 658 ->
// 644. The lines below those, each where the quotient two / one crosses 1 (L1000, 8 blocks a head, 256 units; at 256 / 288 / 384
// / 512 / 640 / 1024 blocks).  Packed masks, a dense one: D32 dual 0.99 / 0.97 / 0.90 / 0.77 / 0.88 / 0.74, D64 plain 1.04 / 0.94
// / 0.88 / 0.75 / 0.88 / 0.72 (the separate kernels keep three workgroups on a unit there).  D64 dual on the bytes of a key
// padding 1.00 / 1.30 / 1.16 / 0.95 / 1.08 / 0.97: past two units' worth the two launches begin a second, mostly empty pass.
// Dropout: D32 dual 1.02 / 1.03 / 0.92 / 0.76, causal 1.56 / 1.32 / 1.04 / 0.87; D64 plain 1.03 / 0.98 / 0.87 / 0.72, causal 1.50
// / 1.30 / 1.03 / 0.86 (and the tangent launch of six gradients there, which at D32 gains up to 2.5 units' worth).  Six
// gradients: D32 1.02 / 1.01 / 0.91 / 0.81 / 0.92, causal 1.50 / 1.29 / 1.05 / 0.95, packed mask 1.36 - 1.50 ... 1.07; D64 1.00 /
// 1.23 / 1.11 / 0.95 / 1.08, causal and packed 1.42 ... 1.01.  Grouped heads, D64 dual: 1.01 / 1.06 / 1.00 / 0.87 / 0.96 / 0.86,
// causal 1.40 / 1.32 / 1.09 / 0.99 / 0.88; plain (448, 512, 640, 1024, 1536) 0.94 - 0.99, 1.07, 1.10, 1.05, 1.07, causal (1024,
// 1536) 1.26, 1.13; gradients of O' alone, dual, at 448 / 512 / 640 1.02 / 1.04 / 1.18, causal 1.00 / 1.00 / 1.08. Documents in a
// packed mask differ with what is drawn: D32 dual 1.05 - 1.28 at 280 - 336 blocks, 0.9 - 1.4 at 384, 0.75 - 1.0 past that; D64
// plain 0.9 - 1.15 at 280 - 336.  Where they gain what a dense mask loses they have the line.  Padding by batch entry as bytes,
// D64 dual, at 392 1.12 - 1.16, with 512 blocks of one role and 64 - 96 of the other 1.10 - 1.27. D = 128 plain, masked, 448 /
// 512 blocks: padding 0.97 - 1.06 / 0.98, dense 0.94 / 0.96, documents 1.02 - 1.10 / 1.02 - 1.08. D = 256, whose blocks with
// tangents have 64 rows, by the same rule: dual 272 / 384 / 448 / 512 / 640 / 896 / 1024 blocks 1.32 / 1.21 / 0.98 / 1.01 / 1.14
// / 1.13 / 1.01, causal 1.39 / 1.04 / 1.01 / 1.00 / 1.08 / 1.03 / 1.03, masked 1.34 - 1.45 / 1.22 - 1.26 / 1.00 - 1.20 / 1.01 -
// 1.09 / 1.13 - 1.16; plain alike.
template <int D, int MODE>
inline bool launch_both(long long blocks, long long kv_blocks, bool causal, int mask, bool drop, bool six, bool grouped, bool twin,
                        bool no_go = false, long long cus = device_cus()) {
  if (cus <= 0) return false;  // the device cannot be asked: two launches
  const double most = (double)(blocks > kv_blocks ? blocks : kv_blocks) / cus;
  const bool bits = mask == MASK_BITS;
  if (D == 32) {
    if (MODE == BWD_PLAIN) return most <= (drop ? 2.5 : 8.0);
    if (drop) return most <= (MODE == BWD_TANGENT ? 2.5 : causal ? 1.5 : 1.25);
    if (six) return most <= (bits ? 2.2 : causal ? 1.5 : 1.35);
    return most <= (bits ? 1.35 : 8.0);
  }
  if (D == 64 && MODE == BWD_DUAL) {
    if (twin || drop) return most <= 8.0;
    if (six && (causal || bits)) return most <= 2.5;
    if (grouped) return most <= (no_go ? 2.75 : causal ? 2.0 : 1.5);
    const double least = (double)(blocks < kv_blocks ? blocks : kv_blocks) / cus;
    return (least <= 1.6 || most > 2.0) && most <= (six ? 2.5 : 2.75);
  }
  if (D == 64) return most <= (drop ? (causal ? 1.5 : 1.0) : bits ? 1.3 : grouped ? 6.0 : 4.5);
  if (most <= 1.0 || ((causal || mask != MASK_NONE) && most <= 2.5)) return true;
  const double apart = (double)((blocks + cus - 1) / cus + (kv_blocks + cus - 1) / cus);
  return apart > (MODE == BWD_DUAL ? 1.04 : 1.08) * ((double)(blocks + kv_blocks) / cus + 0.6);
}
// Whether bwd2_both_kernel_2wg runs a launch of D = 64, dual: two of its workgroups take longer for a pair of blocks than one
// uncapped for one, so it is for launches whose work, dealt evenly, keeps a unit busy for longer than its longest block takes
// (tiles, a dk/dv tile 1.25 of a dq tile).  Uncapped / capped with that quotient in brackets: causal, 140 - 250 blocks of either
// role, L777 - 2048 0.90 - 0.97 (0.59 - 0.95), L512 0.94 (0.70 - 0.84) and 1.04 (0.98), L340 - 640 1.04 - 1.13 (1.01 - 1.13); no
// mask 0.96 (0.90), 1.15 - 1.25 (0.98 on), 1500 queries over 700 keys 0.93 (0.81), but 512 over 1000 - 2000 1.15 - 1.3.
inline bool both_two_wgs(int L, int Lk, long long heads, bool causal, long long cus = device_cus()) {
  const double bq = (L + 127) / 128, bk = (Lk + 127) / 128, nq = (L + 63) / 64, nk = (Lk + 63) / 64;
  double of_q = bq * nk, of_k = bk * nq, longest = nk;  // tiles of all query blocks, of all key blocks, of the longest query block
  if (causal) {
    const double whole = std::min(bq, (double)((Lk + 63) / 64 / 2)), live = std::min(bk, (double)(((L + 63) / 64 + 1) / 2));
    of_q = whole * (whole + 1) + (bq - whole) * nk, of_k = live * nq - live * (live - 1);
    longest = std::min(nk, 2 * bq);
  }
  if (causal && heads * std::max(bq, bk) >= cus) return true;
  if (longest > 1.25 * nq) return heads * (bq + bk) > cus;  // long query blocks, which come last, must not wait for the key blocks
  return heads * (of_q + 1.25 * of_k) > 0.97 * cus * std::max(longest, 1.25 * nq);
}
// ... and in fp32 (one workgroup a compute unit but at D = 32 without tangents, and the separate dq kernel without tangents at D
// = 64). uneven: causal, or a boolean mask, which may leave blocks little to do.  Measured as above, two / one at 136 - 160, 168
// - 192, 224 - 256, 416, 448 - 512, 640 blocks (L1000): no mask, D64 dual 0.99 - 1.01, 0.90 - 0.94, 1.01, 1.00, 0.98 - 1.01,
// 1.10, plain 1.13 - 1.19, 0.96, 1.02, 1.03, 0.96 - 0.99, 1.09; D128 1.15, 0.99, 1.01, 1.08, 1.01, 1.16; a bias D64 dual 1.05,
// 0.93, 1.00, 1.01, 0.98 - 1.01, 1.10, plain at 448 0.96.  Padding by batch entry D64 1.10 - 1.28, 0.97 - 1.09, 1.02, 1.07, 0.98
// - 1.02, 1.10; documents 1.14 - 1.23, 1.34 - 1.41, 1.02 - 1.29, 1.13, 1.01 - 1.14, 1.08; a dense mask as a bias; causal 1.5 at
// 192, 1.02 at 640.  D32 plain, whatever the mask, 1.00 - 1.57, 1.01 - 1.04 at 2048 blocks (and the tangent launch of six
// gradients alike).
template <int D, int MODE>
inline bool launch_both_f32(long long blocks, long long kv_blocks, bool uneven, long long cus = device_cus()) {
  if (cus <= 0) return false;  // the device cannot be asked: two launches
  const double most = (double)(blocks > kv_blocks ? blocks : kv_blocks) / cus, together = (double)(blocks + kv_blocks) / cus;
  if (D == 32 && MODE != BWD_DUAL) return most <= 8.0;
  if (uneven && most <= 2.5) return true;
  if (most <= 1.0 && (D > 64 || MODE != BWD_DUAL || together <= 1.3 || most > 0.85)) return true;
  const double apart = (double)((blocks + cus - 1) / cus + (kv_blocks + cus - 1) / cus);
  return apart > together + 0.7;
}

// ---- merge kernels ------------------------------------------------------------------------------- Forward.  part =
// [chunk][row][O, with tangents T][D] accumulators, then [chunk][row][4] statistics.  One thread per (row, 8 columns), a grid of
// (rows of a head, heads).  With m the largest reference point of the row's chunks and w_c = 2^(m_c - m): l = sum w_c l_c,  O =
// sum w_c O_c,  and, with c the reference of S' of the heaviest chunk, T = sum w_c (T_c + (c_c - c) O_c),  mu_acc = sum w_c (mu_c
// + (c_c - c) l_c); then the epilogue of the forward kernels: O / l, O' = T / l - (mu_acc / l) O, M = m + log2 l, mu = mu_acc / l
// + c. A share that visited nothing says so by l = -0 (a sum is never that) and is left out.  All others are added up, however
// small their weight: that of a share whose scores are all NaN, which no reference point is taken from, or -inf is 0, and 0 times
// what it holds is what one workgroup's rescaling makes of it.  So the outputs that are not numbers are those of whole blocks.
template <typename T, int D, bool DUAL>
__global__ __launch_bounds__(256) void fwd_merge_kernel(const Problem pr, T *o, T *ot, float *M, float *mu) {
  constexpr int LPR = D / 8, RPB = 256 / LPR, ROW = DUAL ? 2 * D : D;
  const int in_head = blockIdx.x * RPB, chunks = Deal{pr.chunks, pr.chunk_tiles, 0, 0}.shares(in_head / 128);  // (uniform: RPB divides 128)
  if (chunks == 1 || in_head + (int)threadIdx.x / LPR >= pr.L) return;  // a block that one workgroup did is finished
  const size_t rows = (size_t)pr.Z * pr.H * pr.L, row = (size_t)blockIdx.y * pr.L + in_head + threadIdx.x / LPR;
  const int d0 = (threadIdx.x % LPR) * 8;
  const float *part = pr.part, *stat = part + (size_t)pr.chunks * rows * ROW;
  float m = -__builtin_inff();
  for (int c = 0; c < chunks; ++c) m = fmaxf(m, stat[((size_t)c * rows + row) * 4]);
  const float m_use = m == -__builtin_inff() ? 0.f : m;
  float l = 0.f, best = -1.f, cref = 0.f;
  for (int c = 0; c < chunks; ++c) {
    const float *st = stat + ((size_t)c * rows + row) * 4;
    const float w = __builtin_amdgcn_exp2f(st[0] - m_use);
    l += w * st[1];  // (no branch on what is loaded: it would put the shares' loads behind one another)
    if (w * st[1] > best) {
      best = w * st[1];
      cref = st[3];
    }
  }
  float O[8], Tt[8], mua = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) O[e] = Tt[e] = 0.f;
  for (int c = 0; c < chunks; ++c) {
    const float *st = stat + ((size_t)c * rows + row) * 4;
    if (__builtin_bit_cast(uint32_t, st[1]) == 0x80000000u) continue;
    const float w = __builtin_amdgcn_exp2f(st[0] - m_use);
    const float *acc = part + ((size_t)c * rows + row) * ROW + d0;
    const float dc = st[3] - cref;
    mua += w * (st[2] + dc * st[1]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float oc = acc[e];
      O[e] += w * oc;
      if constexpr (DUAL) Tt[e] += w * (acc[D + e] + dc * oc);
    }
  }
  const bool dead = !(l > 0.f);
  const float inv = dead ? 0.f : 1.f / l, mu_n = mua * inv;
  float o8[8], t8[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    o8[e] = O[e] * inv;
    t8[e] = Tt[e] * inv - mu_n * o8[e];
  }
  store8<T>(o + (size_t)row * D + d0, o8);
  if constexpr (DUAL) store8<T>(ot + (size_t)row * D + d0, t8);
  if (d0 == 0) {
    M[row] = dead ? __builtin_inff() : m + __builtin_amdgcn_logf(l);
    if constexpr (DUAL) mu[row] = !dead ? mu_n + cref : sizeof(T) == 4 ? mu_n : 0.f;  // (as the kernels of either type leave it)
  }
}

// Backward: gradient t = blockIdx.y out of gridDim.y is the sum of its shares part[chunk][t][elems].  One thread per 8
// elements; bound by HBM (the shares are read once, 16 bytes per lane and load).
template <typename T>
__global__ __launch_bounds__(256) void bwd_kv_merge_kernel(const float *part, int chunks, size_t elems, T *g0, T *g1, T *g2, T *g3) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= elems) return;
  const int t = blockIdx.y, nt = gridDim.y;
  float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < chunks; ++c) {
    const f32x8 x = ld8<float>(part + ((size_t)c * nt + t) * elems + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] += x[e];
  }
  store8<T>((t == 0 ? g0 : t == 1 ? g1 : t == 2 ? g2 : g3) + i, sum);
}

// Backward whose blocks' tiles are dealt to several workgroups: their partial results added up, in fp32 and in the order of the
// tiles: one thread per 8 elements of dq, dk, dv (blockIdx.z 0, 1, 2) of head blockIdx.y (tangent: dq', dk', dv').  Blocks that one
// workgroup did are complete.  Bound by memory: shares * 4 + sizeof(T) bytes an element.
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_split_merge_kernel(const BwdParams p, const BwdSplit sp, const int tangent) {
  const Problem &pr = p.pr;
  constexpr int RPB = 2048 / D;  // rows of a workgroup
  const int t = blockIdx.z, len = t == 0 ? pr.L : pr.Lk, other = t == 0 ? pr.Lk : pr.L;
  const int first = blockIdx.x * RPB, block = first / 128;  // (uniform: RPB divides 128)
  // streamed rows of the block: keys up to its last row, queries from its first 64-row tile on (causal), or all
  const int rows = !pr.causal ? other : t == 0 ? min(other, block * 128 + 128) : max(other - block * 128, 0);
  const Deal &d = t == 0 ? sp.q : sp.k;
  const int tiles = (rows + 63) / 64, dealt = d.step > 0 ? d.shares(t == 0 ? block : d.last - 1 - block) : d.most;
  if (dealt == 1 || first + (int)threadIdx.x / (D / 8) >= len) return;
  const int per = (tiles + dealt - 1) / dealt;
  const size_t elems = (size_t)pr.Z * pr.H * len * D, i = ((size_t)blockIdx.y * len + first) * D + threadIdx.x * 8;
  const float *src = t == 0 ? sp.part_q : sp.part_k + (size_t)(t - 1) * elems;
  const size_t step = t == 0 ? elems : 2 * elems;
  float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c == 0 || c * per < tiles; ++c) {
    const f32x8 x = ld8<float>(src + c * step + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] += x[e];
  }
  store8<T>(reinterpret_cast<T *>(t == 0 ? (tangent ? p.dqt : p.dq) : t == 1 ? (tangent ? p.dkt : p.dk) : (tangent ? p.dvt : p.dv)) + i, sum);
}

}  // namespace jvpfa
