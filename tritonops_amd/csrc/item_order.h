// Order of the work items of a causal launch whose sequences differ in length.
//
// The persistent kernels deal item ids to the workgroups by a fixed rule, so a
// launch is as long as its most loaded workgroup.  With ids numbered sequence
// by sequence the items of a round differ by the spread of the lengths, and
// ids that lie past the end of a short sequence leave their workgroup idle: on
// five sequences of 517 to 3400 tokens (32 heads) the busiest of 256 workgroups
// had 1.4 times the mean work with 8 kv-heads and twice the mean with 32 (queries).
//
// Here the items that exist are numbered LEVEL by level: level t holds the t-th
// tile of every sequence that has one, and the levels are walked from the last
// to the first.  A causal tile costs t + 1 tiles of keys whatever its sequence
// (counted from the sequence's start for queries, from its end for keys), so
// the numbering runs from the longest item to the shortest, and dealing it out
// in alternating directions leaves the busiest workgroup with 1.08 times the
// mean in both cases above without a shared counter and without the lengths
// being known on the host.  The keys of the backward pass (128 rows to an item):
// 1.61 -> 1.33 times the mean with 8 kv-heads, where 536 items make two rounds
// and a few items of a third and the longest one alone is 1.2 times the mean,
// 1.57 -> 1.09 with 32.  (Launches of fewer than four rounds of these deal their
// items, or halves of them, out at run time where they are given a place to count
// in: bwd.hip.)
//
// The window walk's items cost t + 1 tiles only until the local window is filled
// and a band each from there; numbered by level (always: what the unit order would
// cost it is not t + 1 either) it gains from the same balance: seven
// sequences of 500 to 7000 tokens, 16 heads, local window 2048: 296 -> 225 us
// with 4 kv-heads, 301 -> 234 with 16; six of 1024 to 12288, 32 heads: 964 -> 950
// and 1038 -> 994.
//
// What the order costs is sharing: items that run side by side on an XCD read
// the same K / V from its L2 only if they belong to one (sequence, kv-head).
// With one query head per kv-head and sixteen sequences of 2048 tokens every
// item of a level has K / V of its own, and the forward took 702 instead of
// 595 us, four sequences of 8192 (two sharers) 2085 instead of 1919.  So
//  - in launches of six rounds or more `block` adjacent levels of a sequence
//    stay together, as many as make four sharers with the query heads of the
//    group (eight from twelve rounds up: a level more or less weighs little),
//  - equal lengths, which the unit-by-unit order deals out evenly, keep that
//    order from four rounds up, and
//  - from six rounds up so do lengths that it deals out nearly evenly: many
//    sequences even out over a workgroup's rounds.  The kernel works out what the
//    busiest of 32 workgroups would get (about a microsecond) and takes the level
//    order above kLevelWorth of the mean.  Level -> unit order: 48 sequences of
//    490 to 700 tokens, 16 heads of their own (1.15 and 1.04 times the mean),
//    forward 153 -> 146 us, backward 522 -> 502; four of 8040 to 8192, 32 heads
//    (keys 1.00), backward 7059 -> 6616.  Where the level order stays, two
//    sequences of 5900 to 8192 (1.57 and more), it is 1.3 to 1.4 times as fast.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi {

// Sequences a walk can hold: one per lane of a wavefront.
constexpr int kLevelMaxBatch = 64;
// Rounds from which the unit-by-unit order is even enough for equal lengths
// (below: up to 1.8 times the level order's load on the busiest workgroup, for
// instance one sequence of 3000 tokens with 32 heads of its own, a round and a
// half of 256-row items: 121 against 83 us forward, 402 against 328 backward).
constexpr int kLevelEvenRounds = 4;
// From kLevelWorthRounds rounds on, the load of the busiest workgroup in the unit
// order, in hundredths of the mean, above which the level order pays for its
// sharing: measured on 63 batches of 1 to 64 sequences, it loses up to 12 % where
// that is 115 or less and gains 1 to 45 % from 123 on (launches of one workgroup
// or two per CU).  Three workgroups to a CU share what their CU has left when one
// of them is done: 124 to 130 still lost 2 to 3 %, 160 gained 22 (in fewer rounds).
constexpr int kLevelWorthRounds = 6, kLevelWorth = 120, kLevelWorthThree = 135, kLevelAlways = 0;

// Is a launch numbered by level?  (A single round of workgroups takes as long as
// its longest item in any order.  cu == null: a batched call, equal lengths.)
inline bool number_by_level(const int32_t* cu, bool causal, int batch, long long items, long long grid) {
  if (!causal || batch > kLevelMaxBatch || items <= grid) return false;
  return cu != nullptr || items < kLevelEvenRounds * grid;
}

// A workgroup's item of one round: sequence, head, its kv-head and tile (-1: none).
struct ItemId {
  int b, h, kvh, t;
};

// Rounds of one workgroup: one item per lane of a wavefront.
constexpr int kMaxRounds = 64;

// Workgroups of a persistent launch of `items` ids: `resident` run at once, and
// as many generations of them as leave each no more than kMaxRounds rounds.
inline long long persistent_grid(long long items, long long resident) {
  if (resident <= 0 || items <= resident) return items;
  const long long rounds = (items + resident - 1) / resident;
  return resident * ((rounds + kMaxRounds - 1) / kMaxRounds);
}

// All items of a workgroup, one per lane (round = lane): the searches and
// divisions of all of them at once, in vector code ahead of the item loop,
// instead of a chain of scalar code at every item boundary.  (The kv-head comes
// along: dividing by the group again at each boundary cost six registers at
// head_dim 128; in time no more than runs differ, 23.9 against 23.5 us on one
// prompt of 1000 tokens.)  Odd rounds are walked back to
// front within each XCD (id & 7 is kept), so that the workgroup that drew a
// long item in one round draws a short one in the next.
//
// Not by level: consecutive ids go round-robin to the 8 XCDs, each with a
// private L2; every XCD is given whole (sequence, kv-head) units, so that the
// K / V of a unit stay in one L2, and a unit's tiles run from the longest item
// to the shortest.  FROM_END: the first tile of a sequence costs most (keys,
// which every later query streams past), else the last.  heads_kv: heads per
// sequence that share nothing (units); heads / heads_kv items of a unit run
// side by side on each of its tiles.
//
// BY_LEVELS: where levels are taken one at a time a pair is found level by level, with
// the sequences of a level as bits of a mask, instead of pair by pair, 0.05 us each
// (64 sequences of 926 tokens, one head, dQ in two rounds of 128-row items with dK + dV
// 120 -> 89 us).  The other kernels' search is as it was.
template <int ROWS, bool FROM_END, int WORTH = kLevelWorth, bool BY_LEVELS = false>
__device__ __forceinline__ ItemId items_of_rounds(const int32_t* cu, const int batch, const int max_seqlen,
                                                  const int n_tiles, const int heads, const int heads_kv,
                                                  const bool level_order, const int n_items, const int grid) {
  const int lane = threadIdx.x & 63;
  const int round = lane;
  int w = blockIdx.x;
  if ((round & 1) && (grid & 7) == 0) w = (((grid >> 3) - 1 - (w >> 3)) << 3) | (w & 7);
  const long long id = (long long)round * grid + w;
  const bool any = id < n_items;
  const uint32_t bid = any ? (uint32_t)id : 0u;   // (unsigned: the shorter divisions)
  // x = q d + r.  All divisors are wave-uniform and ids below 2^22 need no more
  // than a float reciprocal: with x < 2^22 exact in fp32 and v_rcp_f32 within
  // 1 ulp the product is off by less than one, which one step either way mends.
  const bool small = n_items < (1 << 22);
  auto divmod = [&](uint32_t x, uint32_t d, uint32_t& q, uint32_t& r) __attribute__((always_inline)) {
    if (small) {
      q = (uint32_t)((float)x * __builtin_amdgcn_rcpf((float)d));
      r = x - q * d;
      if ((int)r < 0) {
        --q;
        r += d;
      } else if (r >= d) {
        ++q;
        r -= d;
      }
    } else {
      q = x / d;
      r = x % d;
    }
  };
  uint32_t group, rest;
  divmod((uint32_t)heads, (uint32_t)heads_kv, group, rest);
  // item `id` of the unit order: sequence, kv-head, member of its group and slot of the unit's tiles
  const uint32_t per_unit = (uint32_t)n_tiles * group;
  auto unit_item = [&](uint32_t id, uint32_t& b, uint32_t& kvh, uint32_t& member, int& t) __attribute__((always_inline)) {
    uint32_t unit, s, tile;
    if (((batch * heads_kv) & 7) == 0) {
      divmod(id >> 3, per_unit, unit, s);
      unit = unit * 8 + (id & 7);
    } else {
      divmod(id, per_unit, unit, s);
    }
    divmod(s, group, tile, member);
    divmod(unit, (uint32_t)heads_kv, b, kvh);
    t = FROM_END ? (int)tile : n_tiles - 1 - (int)tile;
  };
  ItemId it = {0, 0, 0, -1};
  if (level_order) {
    int tiles = 0;  // of sequence `lane`
    if (lane < batch) {
      const int len = cu ? min(cu[lane + 1] - cu[lane], max_seqlen) : max_seqlen;
      tiles = len > 0 ? (len + ROWS - 1) / ROWS : 0;
    }
    int total = tiles;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) total += __shfl_xor(total, m, 64);
    total = __builtin_amdgcn_readfirstlane(total);
    const int tiles0 = __builtin_amdgcn_readfirstlane(tiles);
    const bool even = __builtin_amdgcn_ballot_w64(lane < batch && tiles != tiles0) == 0;
    bool by_unit = cu && even && total * heads >= kLevelEvenRounds * grid;
    if (WORTH != kLevelAlways && !by_unit && total * heads >= kLevelWorthRounds * grid && (grid & 7) == 0) {
      // what the unit order would give 32 workgroups of the first XCD, one to a lane, rounds of one parity to a
      // half of the wavefront
      const int per_xcd = grid >> 3, half = lane >> 5;
      const int slot = (lane & 31) * max(per_xcd >> 5, 1);
      const int at = half ? per_xcd - 1 - slot : slot;
      int load = 0;
      for (int r = 0; r < kMaxRounds && (long long)r * grid < n_items; r += 2) {
        const long long id2 = (long long)(r + half) * grid + at * 8;
        const bool live = slot < per_xcd && id2 < n_items;
        uint32_t b2, kvh2, member2;
        int t2;
        unit_item(live ? (uint32_t)id2 : 0u, b2, kvh2, member2, t2);
        const int all = __shfl(tiles, (int)b2, 64);
        if (live && t2 < all) load += FROM_END ? all - t2 : t2 + 1;
      }
      load += __shfl_xor(load, 32, 64);
      float work = 0.5f * (float)tiles * (float)(tiles + 1);  // of one head of sequence `lane`
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) {
        load = max(load, __shfl_xor(load, m, 64));
        work += __shfl_xor(work, m, 64);
      }
      by_unit = (float)load * (float)grid * 100.f <= (float)WORTH * work * (float)heads;
      by_unit = __builtin_amdgcn_readfirstlane(by_unit);
    }
    if (!by_unit) {
      const int sharers = total * heads >= 12 * grid ? 8 : total * heads >= 6 * grid ? 4 : 1;
      int block = 1;  // adjacent levels of a sequence that stay together
      while (block * (int)group < sharers) block *= 2;
      uint32_t pair, r;
      divmod(bid, (uint32_t)heads, pair, r);
      const int n = any ? (int)pair : -1;  // (sequence, tile) pair in the order below
      int at = 0;                                             // pairs before the ones being looked at
      if (BY_LEVELS && block == 1) {
        uint32_t lo = 0, hi = 0;   // sequences of the level that the pair lies on
        int k = 0;                 // and which of them it is
        for (int t = n_tiles - 1; t >= 0; --t) {
          const uint64_t live = __builtin_amdgcn_ballot_w64(tiles > t);
          const int own = __builtin_popcountll(live);
          if (n >= at && n < at + own) {
            lo = (uint32_t)live;
            hi = (uint32_t)(live >> 32);
            k = n - at;
            it.t = t;
          }
          at += own;
          if (__builtin_amdgcn_ballot_w64(n >= at) == 0) break;
        }
        // the bit of the mask that has k set ones before it
        const int in_lo = __popc(lo);
        const bool upper = k >= in_lo;
        uint32_t m = upper ? hi : lo;
        k -= upper ? in_lo : 0;
        it.b = upper ? 32 : 0;
#pragma unroll
        for (int w = 16; w >= 1; w >>= 1) {
          const int c = __popc(m & ((1u << w) - 1));
          const bool above = k >= c;
          k -= above ? c : 0;
          it.b += above ? w : 0;
          m = above ? m >> w : m;
        }
        if (it.t < 0) it.b = 0;
        const int all = __shfl(tiles, it.b, 64);
        if (FROM_END && it.t >= 0) it.t = all - 1 - it.t;
      } else
      for (int first = (n_tiles - 1) / block * block; first >= 0; first -= block) {
        uint64_t live = __builtin_amdgcn_ballot_w64(tiles > first);
        while (live) {
          const int seq = __builtin_ctzll(live);
          live &= live - 1;
          const int all = __builtin_amdgcn_readlane(tiles, seq);
          const int own = min(all - first, block);
          const int k = n - at;
          if (k >= 0 && k < own) {
            it.b = seq;
            it.t = FROM_END ? all - first - own + k : first + own - 1 - k;
          }
          at += own;
        }
        if (__builtin_amdgcn_ballot_w64(n >= at) == 0) break;
      }
      // the kv-head runs fastest: ids eight apart, which share an XCD, then read
      // the same K / V whenever the head counts are multiples of eight
      uint32_t member, kvh;
      divmod(r, (uint32_t)heads_kv, member, kvh);
      it.h = (int)(kvh * group + member);
      it.kvh = (int)kvh;
      return it;
    }
  }
  uint32_t member, b, kvh;
  int t;
  unit_item(bid, b, kvh, member, t);
  it.b = (int)b;
  it.h = (int)(kvh * group + member);
  it.kvh = (int)kvh;
  const int len = cu ? min(cu[it.b + 1] - cu[it.b], max_seqlen) : max_seqlen;
  it.t = any && t * ROWS < len ? t : -1;
  return it;
}

}  // namespace mi
