// Single-query (decoding) attention for gfx950: split-KV pass + LSE merge pass,
// dense and block-sparse.
//
// Replaces flash_attn_decoding_kernel / flash_attn_decoding_correction_kernel
// of flash_attn_triton/flash_attn_decoding.py:9-122,:126-210 and their sparse
// twins in flash_attn_triton/flash_attn_decoding_sparse.py:10-127,:131-219.
//
// Pass 1: a work item is a (chunk, kv-head, sequence) triple and is handled
// by one workgroup of NW wavefronts.  A sequence's chunks follow from its own
// length and split_tokens (split_blocks) alone, and a chunk's tiles are worked on
// in order whatever NW is, so a row's bits depend neither on the other sequences
// of the batch nor on the launch.  The block-list form launches one workgroup
// per item; the dense form launches one resident round (8 wavefronts per CU)
// and deals the live chunks of a ragged batch to them round-robin.
// The G = hq/hkv query heads that share the kv-head sit in the first G of the 32
// query columns of the same S^T = K.Q^T / O^T = V^T.P^T MFMA pipeline the
// prefill kernel uses, so each K/V byte is fetched once for the whole group
// (the reference launches one program per q-head and re-reads KV G times,
// flash_attn_decoding.py:42-45,264-268) and the dot products cost no VALU
// work.  A group of more than 32 heads is split into slices of 32, each a work
// item of its own: KV is then fetched once per slice.  KV streams global -> registers -> wave-private LDS in 32-key tiles
// with fully coalesced 16-byte loads (non-temporal: every byte is used once);
// as soon as a tile has arrived, each register is written to LDS and refilled
// with its part of the tile after next.  With one wavefront no barriers are
// needed because a single wave's LDS operations execute in order; several take
// the tiles of a chunk in steps of NW, a tile each, between two barriers.
// Partials are fp32 (the reference rounds them to the input dtype, :249-251).
// Pass 2: per (sequence, q-head) merge  o = sum_c o_c 2^(lse_c - lse).
#include <atomic>
#include <type_traits>

#include "kernels.h"
#include "tile_core.h"

// Split-KV partials of mi_decode_noalloc: device memory the library holds from
// load time on, one copy per GPU.  Host code must not use this name as an
// address (it is a host-side stand-in); decode_static_scratch() below asks the
// runtime for the device address, per device, and everything else uses that.
static __device__ __align__(256) unsigned char scratch[mi::kDecodeScratchBytes];

namespace mi {
namespace {

constexpr int kDecTile = 32;

// The block list of the window form, which is arithmetic: the blocks of the
// first `wg` tokens (entries 0 .. n_sink-1), then the blocks from token
// max(len - wl, 0) to the last one (entries n_sink .. cnt-1, starting at block
// tail0), every block once.
struct WindowList {
  int n_sink, tail0, cnt;
  __device__ __forceinline__ int block(int e) const { return e < n_sink ? e : tail0 + (e - n_sink); }
};
__device__ __forceinline__ WindowList window_list(int len, int wg, int wl) {
  const int nblk = (len + 63) / 64;
  WindowList w;
  w.n_sink = min((wg + 63) / 64, nblk);
  w.tail0 = max(max(len - wl, 0) / 64, w.n_sink);
  w.cnt = w.n_sink + max(nblk - w.tail0, 0);
  return w;
}

// LDS of a workgroup: the K tiles of its wavefronts, then their V tiles.
template <int D>
constexpr int wave_lds() {
  using F = PaddedFrags<D>;
  return kDecTile * (F::KROWB + F::VROWB);
}

// Barrier between the wavefronts of a workgroup that orders LDS accesses only:
// the loads of the next tiles stay in flight across it.
template <int NW>
__device__ __forceinline__ void lds_barrier() {
  if constexpr (NW > 1) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
}

// A word at a wave-uniform address of memory that no kernel of the launch writes
// (lengths, block lists, page tables), through the scalar cache.  As an ordinary
// load it goes the way of the K/V tiles, whose loads retire in order: the wait for
// one page number or list entry then waits for every tile that is in flight: pass 1
// of 8 sequences of 4k to 8k tokens in pages of 64, 8 kv-heads of 128, 38.5 -> 35.2 us
// (32 of them 143 -> 135, contiguous 135), lists of 64 blocks, 4 sequences, 15.9 -> 14.4.
__device__ __forceinline__ int scalar_word(const int32_t* a) {
  typedef __attribute__((address_space(4))) const int32_t c_int32;
  const uint64_t u = (uint64_t)(uintptr_t)a;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)u);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return *(c_int32*)(((uint64_t)hi << 32) | lo);
}

// One work item: chunk `split` of (sequence b, kv-head kvh) for the 32 query
// heads of the group that start at head g0 of it (slice kvs % gslices; a group
// of up to 32 heads is one slice).
//
// NW > 1: the wavefronts fetch NW tiles at a time, one each, every wavefront
// works out all their scores and probabilities and 1 / NW of the output columns
// (blocks of 32, wave + NW j).  What is computed, and in which order, is what one wavefront computes,
// bit for bit; matrix and vector units have room for the repeated scores (memory
// is the bound), and the output needs no merge between wavefronts.
template <typename T, int D, int NW, bool LIST>
__device__ __forceinline__ void decode_item(const DecodeParams& p, unsigned char* smem, const int split, const int kvs,
                                            const int b, const int len) {
  const int kvh = kvs / p.gslices;
  const int g0 = (kvs % p.gslices) * 32;
  using G = RowGeom<D>;
  using F = PaddedFrags<D>;
  constexpr int KTILEB = kDecTile * F::KROWB;
  constexpr int NCHUNK = kDecTile * G::NCH;
  constexpr int VTILEB = kDecTile * F::VROWB;
  constexpr int LOADS = (NCHUNK + 63) / 64;
  constexpr int NB = (G::NDB + NW - 1) / NW;  // output blocks of a wavefront

  const int lane = threadIdx.x & 63;
  const int wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned char* sK = smem;
  unsigned char* sV = smem + NW * KTILEB;

  const int gqa_all = p.hq / p.hkv;
  const int gqa = min(32, gqa_all - g0);  // query heads of this slice
  constexpr bool sparse = LIST;
  const bool derived = p.list_mode == 2;

  int n_tiles, t_begin = 0;
  const int32_t* blist = nullptr;
  WindowList wlist = {0, 0, 0};
  int n_listed = 0;  // listed entries that fall into this chunk
  int b0 = 0;        // first entry of this chunk
  const int last_blk = (len - 1) / 64;
  if (sparse) {
    int cnt;
    if (derived) {
      wlist = window_list(len, p.win_global, p.win_local);
      cnt = min(wlist.cnt, p.max_blocks);
    } else {
      cnt = p.block_cnt ? min(scalar_word(p.block_cnt + b * p.hkv + kvh), p.max_blocks) : p.max_blocks;
    }
    const int total = cnt + p.add_last;  // the implicit last block sits behind the list
    b0 = split * p.split_blocks;
    if (b0 >= total || len <= 0) return;
    if (!derived) blist = p.block_idx + b * p.bi_sb + kvh * p.bi_sh + b0;
    n_tiles = 2 * min(total - b0, p.split_blocks);
    n_listed = max(0, min(cnt - b0, p.split_blocks));
  } else {
    t_begin = split * p.split_tokens;
    n_tiles = (min(len - t_begin, p.split_tokens) + kDecTile - 1) / kDecTile;
  }
  // sparse: entry i/2 of the chunk; entries behind the listed ones are the
  // implicit last block, and a LISTED last block is dropped when the implicit
  // one exists (base -1 => the whole tile is masked)
  auto tile_base = [&](int i) -> int {
    if (!sparse) return t_begin + i * kDecTile;
    const int e = i >> 1;
    const int blk = e < n_listed ? (derived ? wlist.block(b0 + e) : scalar_word(blist + e)) : last_blk;
    if (p.add_last && e < n_listed && blk == last_blk) return -1;
    return blk * 64 + (i & 1) * kDecTile;
  };

  // Start of this sequence's rows: batch stride, row offset cu[b] of a packed
  // buffer, or (paged) the pool itself with the page looked up per tile.
  const int64_t seq0 = p.kv_layout == 1 ? (int64_t)scalar_word(p.cu + b) : 0;
  const int64_t bsel = p.kv_layout == 0 ? b : 0;
  const T* kp = reinterpret_cast<const T*>(p.k) + bsel * p.k_sb + seq0 * p.k_ss + kvh * p.k_sh;
  const T* vp = reinterpret_cast<const T*>(p.v) + bsel * p.v_sb + seq0 * p.v_ss + kvh * p.v_sh;
  const bool paged = p.kv_layout == 2;
  const int32_t* ptab = paged ? p.page_table + b * p.pt_sb : nullptr;
  F lc;
  lc.init(lane);

  // Q^T operand: column lq is q-head kvh*gqa + lq, columns >= gqa are zero.
  i32x4 Qf[G::KSTEPS];
  {
    const T* qr = reinterpret_cast<const T*>(p.q) + b * p.q_sb +
                  (int64_t)(kvh * gqa_all + g0 + min(lc.lq, gqa - 1)) * p.q_sh + 8 * lc.lh;
#pragma unroll
    for (int c = 0; c < G::KSTEPS; ++c) {
      i32x4 t = *reinterpret_cast<const i32x4*>(qr + 16 * c);
      Qf[c] = lc.lq < gqa ? t : (i32x4){0, 0, 0, 0};
    }
  }

  f32x16 O[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) O[j] = (f32x16){0};
  float m = -INFINITY, l = 0.f;

  // The loads of tile t + 1 fly while tile t is worked on.  (Registers for a
  // second tile in flight do not exist: the occupancy of this kernel is bounded
  // by LDS, one private tile per wave, at 256 registers per wave, and O, Q and
  // one K/V set already take 240 of them at head_dim 128.)
  i32x4 kreg[LOADS], vreg[LOADS];
  // First token a tile is fetched from.  A tile that is masked as a whole (a
  // dropped duplicate, base -1, or the second half of the last block when the
  // sequence ends in its first half) is fetched from the tile of the last
  // token instead, so that no row outside [0, len) and no page beyond the
  // sequence is ever touched.
  const int last_tile = ((len - 1) / kDecTile) * kDecTile;
  auto addr_base = [&](int base) -> int { return min(max(base, 0), last_tile); };
  // Load i of a lane covers chunk lane % NCH of row lane / NCH + i * (64 / NCH)
  // when NCH divides 64 (head_dim 64 and 128): the address is then a uniform
  // base that advances by a fixed step per load plus one 32-bit lane offset.
  constexpr bool kUniformRows = 64 % G::NCH == 0;
  typedef __attribute__((address_space(1))) const i32x4 g_i32x4;  // global memory, not generic
  typedef __attribute__((address_space(1))) const char g_char;
  auto uniform64 = [](uint64_t x) __attribute__((always_inline)) -> uint64_t {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
  };
  // pins a uniform address in a scalar register pair, so that the load keeps
  // the form "scalar base + 32-bit lane offset" (the optimiser would otherwise
  // fold the lane offset into a 64-bit vector address per load)
  auto scalar_ptr = [](uint64_t a) __attribute__((always_inline)) -> g_char* {
    uint32_t lo = (uint32_t)a, hi = (uint32_t)(a >> 32);
    asm volatile("" : "+s"(lo), "+s"(hi));
    return (g_char*)(((uint64_t)hi << 32) | lo);
  };
  const uint32_t k_step = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)((64 / G::NCH) * p.k_ss * 2));
  const uint32_t v_step = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)((64 / G::NCH) * p.v_ss * 2));
  const uint32_t k_lane = (uint32_t)((lane / G::NCH) * p.k_ss * 2 + (lane % G::NCH) * 16);
  const uint32_t v_lane = (uint32_t)((lane / G::NCH) * p.v_ss * 2 + (lane % G::NCH) * 16);
  const uint32_t k_rowb = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p.k_ss * 2));
  const uint32_t v_rowb = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p.v_ss * 2));
  // reg <- chunk (lane + 64 i) of the tile at `tile` (uniform address of its
  // first row); rows beyond row_max re-read row row_max (the last token: same
  // tile, hence same page)
  auto load_one = [&](i32x4& reg, int i, uint64_t tile, int row_max, uint32_t rowb, uint32_t step,
                      uint32_t lane_off) __attribute__((always_inline)) {
    const int idx = lane + i * 64;
    if (NCHUNK % 64 != 0 && idx >= NCHUNK) return;
    if (kUniformRows && row_max >= kDecTile - 1) {
      reg = __builtin_nontemporal_load((g_i32x4*)(scalar_ptr(tile + (uint64_t)i * step) + lane_off));
    } else {
      const int row = idx / G::NCH, ch = idx % G::NCH;
      const uint32_t off = (uint32_t)min(row, row_max) * rowb + ch * 16;
      reg = __builtin_nontemporal_load((g_i32x4*)(scalar_ptr(tile) + off));
    }
  };
  auto store_one = [&](int i) __attribute__((always_inline)) {
    const int idx = lane + i * 64;
    if (NCHUNK % 64 != 0 && idx >= NCHUNK) return;
    const int row = idx / G::NCH, ch = idx % G::NCH;
    F::store_k(sK + wave * KTILEB, row, ch, kreg[i]);
    F::store_v(sV + wave * VTILEB, row, ch, vreg[i]);
  };
  // where a tile comes from: uniform addresses of its first K / V row and the
  // last row that may be read
  struct TileSrc {
    uint64_t k, v;
    int row_max;
  };
  auto tile_src = [&](int base) __attribute__((always_inline)) -> TileSrc {
    const int tb = addr_base(base);
    TileSrc t;
    int64_t page = 0;
    int row = tb;
    if (paged) {   // a 32-token tile never straddles a page (page_size % 32 == 0)
      const int lp = tb / p.page_size;
      page = scalar_word(ptab + lp);
      row = tb - lp * p.page_size;
    }
    t.k = uniform64((uint64_t)(uintptr_t)(kp + page * p.k_sb + (int64_t)row * p.k_ss));
    t.v = uniform64((uint64_t)(uintptr_t)(vp + page * p.v_sb + (int64_t)row * p.v_ss));
    t.row_max = len - 1 - tb;
    return t;
  };
  auto load_pair = [&](int i, const TileSrc& t) __attribute__((always_inline)) {
    load_one(kreg[i], i, t.k, t.row_max, k_rowb, k_step, k_lane);
    load_one(vreg[i], i, t.v, t.row_max, v_rowb, v_step, v_lane);
  };

  const int wl = LIST ? p.win_local : -1, wg = p.win_global;
  // A step is NW tiles, tile `wave` of each fetched by this wavefront.  Step t is
  // worked on from LDS while the tiles of step t + 1 are in flight into the
  // registers.  When they have arrived, every register is written to LDS and
  // refilled at once with its part of step t + 2, so that the next loads leave
  // as early as possible; the addresses of step t + 2 (block list and page
  // look-ups) are prepared before step t is worked on.
  auto step_bases = [&](int i0, int (&base)[NW]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NW; ++j) base[j] = i0 + j < n_tiles ? tile_base(i0 + j) : 0;
  };
  int cur[NW], nxt[NW];
  step_bases(0, cur);
  step_bases(NW, nxt);
  TileSrc src = tile_src(wave < n_tiles ? tile_base(wave) : 0);  // the first tile, the second, then the one two ahead of the compute
  if (wave < n_tiles) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_pair(i, src);
    if (NW + wave < n_tiles) src = tile_src(tile_base(NW + wave));
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      store_one(i);
      if (NW + wave < n_tiles) load_pair(i, src);
    }
  }
  for (int i0 = 0; i0 < n_tiles; i0 += NW) {
    lds_barrier<NW>();
    const bool refill = i0 + 2 * NW + wave < n_tiles;
    int nn[NW];
    step_bases(i0 + 2 * NW, nn);
    if (refill) src = tile_src(tile_base(i0 + 2 * NW + wave));
    if (NW == 1 || wave < G::NDB) {
      // (scores of tiles behind the chunk's last are computed and not used)
      f32x16 S[NW];
      qk_scores<T, D, NW>(sK, lc, Qf, S);
      auto tile = [&](auto tc) __attribute__((always_inline)) {
        constexpr int t = decltype(tc)::value;
        if (NW > 1 && i0 + t >= n_tiles) return;
        const int base = cur[t];
        bool need_mask = base + kDecTile > len || base < 0;
        if (wl >= 0) need_mask = need_mask || !((base + kDecTile - 1 < wg) || (base >= len - wl));
        auto allowed = [&](int key_in_tile) -> bool {
          const int key = base + key_in_tile;
          bool ok = key < len && base >= 0;
          if (wl >= 0) ok = ok && (key < wg || key >= len - wl);
          return ok;
        };
        f32x16 S1[1] = {S[t]};
        uint32_t P[1][8];
        softmax_tile<T, D, 1>(S1, lc.lh, O, m, l, p.scale, need_mask, allowed, P);
        pv_accumulate<T, D, 1, NW>(sV + t * VTILEB + wave * 64, lc, P, O);
      };
      using std::integral_constant;  // (a loop of this size is not unrolled, and S and cur went to scratch)
      tile(integral_constant<int, 0>{});
      if constexpr (NW > 1) tile(integral_constant<int, 1>{});
      if constexpr (NW > 2) tile(integral_constant<int, 2>{}), tile(integral_constant<int, 3>{});
    }
    lds_barrier<NW>();
    if (i0 + NW + wave < n_tiles) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        store_one(i);
        if (refill) load_pair(i, src);
      }
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      cur[j] = nxt[j];
      nxt[j] = nn[j];
    }
  }

  const float l_tot = sum_with_other_half(l);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (lc.lq < gqa) {
    const int h = kvh * gqa_all + g0 + lc.lq;
    const int64_t slot = ((int64_t)b * p.hq + h) * p.n_splits + split;
    // (a NaN sum stays NaN)
    if (lc.lh == 0 && wave == 0) p.part_lse[slot] = l_tot == 0.f ? -INFINITY : m + fast_log2(l_tot);
    float* po = p.part_o + slot * D;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int db = wave + NW * j;
      if (G::NDB % NW != 0 && db >= G::NDB) break;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float4 w = {O[j][4 * g] * inv, O[j][4 * g + 1] * inv, O[j][4 * g + 2] * inv, O[j][4 * g + 3] * inv};
        *reinterpret_cast<float4*>(po + 32 * db + 8 * g + 4 * lc.lh) = w;
      }
    }
  }
}

// Block-list form: one workgroup per (chunk, kv-head, sequence), grid
// (n_splits, hkv, batch).  Dense form: the live chunks of all sequences (a
// sequence of length L has ceil(L / split_tokens) of them) are numbered
// consecutively and dealt round-robin to gridDim.x workgroups, one resident
// round of the chip, so that ragged batches leave no tail of half-empty rounds:
// every workgroup gets the same number of chunks, give or take one.
// Bound by memory: 64 sequences of 16k to 32k tokens, 8 kv-heads of 128, take
// 1104 us (6.1 TB/s) in chunks of 2048 tokens, of which a wavefront has 3.2 on
// average and four at most.  (Ranges of equal length across the sequences take
// 1081, but then a row's bits change with the lengths of its neighbours.)
template <typename T, int D, int NW, bool LIST>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
decode_splitkv_kernel(const DecodeParams p) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[NW * wave_lds<D>()];
  if constexpr (LIST) {
    const int b = blockIdx.z;
    const int len = p.seq_lens ? scalar_word(p.seq_lens + b) : scalar_word(p.cu + b + 1) - scalar_word(p.cu + b);
    decode_item<T, D, NW, true>(p, smem, blockIdx.x, blockIdx.y, b, len);
    return;
  }
  const int lane = threadIdx.x & 63;
  auto len_of = [&](int b) -> int {
    return b >= p.batch ? 0 : p.seq_lens ? p.seq_lens[b] : p.cu[b + 1] - p.cu[b];
  };
  auto chunks_of = [&](int len) -> int { return len > 0 ? min((len - 1) / p.split_tokens + 1, p.n_splits) : 0; };
  auto chunks_up_to = [&](int n) __attribute__((always_inline)) -> int {  // inclusive scan over the lanes
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(n, d, 64);
      if (lane >= d) n += up;
    }
    return n;
  };
  // the first 64 sequences, which most batches end within: looked at once
  const int len_first = len_of(lane);
  const int n_first = chunks_of(len_first);
  const int incl_first = chunks_up_to(n_first);
  const uint32_t kv_slices = p.hkv * p.gslices;  // (kv-head, 32-head slice of its group) pairs
  // (every item has a slot of at least 64 floats in the workspace: ids stay far below 2^32)
  for (uint32_t g = blockIdx.x;; g += gridDim.x) {
    const int t = (int)(g / kv_slices), kvs = (int)(g % kv_slices);
    // the sequence that owns live chunk t, and the number of its first chunk
    int b = -1, first = 0, len = 0;
    for (int b0 = 0, seen = 0; b0 < p.batch; b0 += 64) {
      int n = n_first, incl = incl_first, own = len_first;
      if (b0 != 0) {
        own = len_of(b0 + lane);
        n = chunks_of(own);
        incl = chunks_up_to(n);
      }
      const int before = seen + incl - n;  // live chunks ahead of this lane's sequence
      const unsigned long long hit = __builtin_amdgcn_ballot_w64(n > 0 && t >= before && t < before + n);
      if (hit) {
        const int at = __builtin_ctzll(hit);
        b = b0 + at;
        first = __builtin_amdgcn_readlane(before, at);
        len = __builtin_amdgcn_readlane(own, at);
        break;
      }
      seen += __builtin_amdgcn_readlane(incl, 63);
    }
    if (b < 0) return;  // behind the last live chunk
    decode_item<T, D, NW, false>(p, smem, t - first, kvs, b, len);
  }
}

// Merge: a workgroup per (query head, sequence), a thread per output column.
// Bound by latency (a few KiB per workgroup), so the weights are formed by all
// lanes at once and the partial results requested kMergeBatch slots at a time;
// they are added slot by slot, in the order of the sequence.  (Eight slots side
// by side, then the sums of the eight: no faster, whole call 20.9 against 20.2 us
// for 2 sequences of 28 chunks, 35.8 against 34.3 for one of 64.)
// A NaN among a chunk's scores arrives as a NaN log-sum-exp and makes the
// result NaN; so does a NaN or infinity among its values, whatever the weight
// of the chunk.
//
// NE > 0 (at most 64 NE slots): every wavefront forms all weights, NE to a lane, which
// are read out of its lanes, and the log-sum-exps and the first kMergeAhead slots are
// requested before it is known how many of them pass 1 wrote (the length comes through
// the scalar cache meanwhile); the others as soon as it is, and a batch ahead.  No
// barrier, the same sums in the same order as the general form.  Merge alone, 32 heads
// of 128: two sequences of 32 slots 5.2 -> 4.3 us (a launch of nothing takes 4), 64 of 5
// 6.0 -> 4.6, one of 128 7.3 -> 6.0.
// Asking for a whole batch ahead, 0.2 us faster where all of it was written, reads up to
// 32 slots a row of what nobody wrote under a bound far above the lengths, and pass 1 of
// the call after it pays for the caches: both passes, four sequences of 250 to 1000
// tokens of 65536 49.7 us, with 4 ahead 45.2, 8 45.4, 16 47.2, none 45.8; 128 of 25 to
// 100 of 32768 23.4, 19.7, 20.4, 23.0, 20.6.  A list without counts of its own has as
// many slots as the launch says: all are asked for at once (64 blocks 19.4 -> 19.1).
constexpr int kMergeThreads = 128, kMergeBatch = 32, kMergeAhead = 4;
template <typename T, int NE>
__global__ void __launch_bounds__(kMergeThreads)
decode_merge_kernel(const DecodeParams p, int D) {
  __shared__ float weight[2][kMergeThreads];
  __shared__ float top[kMergeThreads / 64];
  const int h = blockIdx.x, b = blockIdx.y;
  const int d = threadIdx.x;
  const int64_t slot0 = ((int64_t)b * p.hq + h) * p.n_splits;
  const float* pl = p.part_lse + slot0;
  const float* po = p.part_o + slot0 * D + min(d, D - 1);
  float part[2][NE ? kMergeBatch : 1], e[NE ? NE : 1];
  // slots [first, kMergeBatch) of the batch at c0; those behind `last` read it once more
  auto request = [&](float (&x)[NE ? kMergeBatch : 1], int c0, auto first, int last) __attribute__((always_inline)) {
#pragma unroll
    for (int i = first; i < kMergeBatch; ++i) x[i] = po[(int64_t)min(c0 + i, last) * D];
  };
  const bool known = p.list_mode == 1 && !p.block_cnt;   // how many slots there are, without a look at memory
  if constexpr (NE > 0) {
#pragma unroll
    for (int k = 0; k < NE; ++k) e[k] = pl[min(64 * k + (d & 63), p.n_splits - 1)];
    if (known) {
      request(part[0], 0, std::integral_constant<int, 0>{}, p.n_splits - 1);
    } else {
#pragma unroll
      for (int i = 0; i < kMergeAhead; ++i) part[0][i] = po[(int64_t)min(i, p.n_splits - 1) * D];
    }
  }
  const int len = p.seq_lens ? scalar_word(p.seq_lens + b) : scalar_word(p.cu + b + 1) - scalar_word(p.cu + b);
  int nvalid;  // slots that pass 1 wrote
  if (p.list_mode != 0) {
    const int kvh = h / (p.hq / p.hkv);
    int cnt;
    if (p.list_mode == 2)
      cnt = min(window_list(len, p.win_global, p.win_local).cnt, p.max_blocks);
    else
      cnt = p.block_cnt ? min(scalar_word(p.block_cnt + b * p.hkv + kvh), p.max_blocks) : p.max_blocks;
    nvalid = (cnt + p.add_last + p.split_blocks - 1) / p.split_blocks;
  } else {
    nvalid = len > 0 ? (len - 1) / p.split_tokens + 1 : 0;
  }
  nvalid = len > 0 ? max(0, min(nvalid, p.n_splits)) : 0;

  float M = -INFINITY, den = 0.f, acc = 0.f;
  if constexpr (NE > 0) {
    if (!known && nvalid > kMergeAhead) request(part[0], 0, std::integral_constant<int, kMergeAhead>{}, nvalid - 1);
#pragma unroll
    for (int k = 0; k < NE; ++k) {
      e[k] = 64 * k + (d & 63) < nvalid ? e[k] : -INFINITY;
      M = fmaxf(M, e[k]);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) M = fmaxf(M, __shfl_xor(M, m, 64));
#pragma unroll
    for (int k = 0; k < NE; ++k) e[k] = e[k] == -INFINITY ? 0.f : fast_exp2(e[k] - M);
#pragma unroll
    for (int c0 = 0; c0 < 64 * NE; c0 += kMergeBatch) {
      if (c0 >= nvalid) break;
      float(&x)[kMergeBatch] = part[(c0 / kMergeBatch) & 1];
      if (c0 + kMergeBatch < nvalid) request(part[(c0 / kMergeBatch + 1) & 1], c0 + kMergeBatch, std::integral_constant<int, 0>{}, nvalid - 1);
#pragma unroll
      for (int i = 0; i < kMergeBatch; ++i) {
        const bool live = c0 + i < nvalid;
        const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e[c0 / 64]), c0 % 64 + i));
        den = live ? den + w : den;
        acc = live ? fmaf(w, x[i], acc) : acc;
      }
    }
  } else {
    for (int c = d; c < nvalid; c += kMergeThreads) M = fmaxf(M, pl[c]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) M = fmaxf(M, __shfl_xor(M, m, 64));
    if ((d & 63) == 0) top[d >> 6] = M;
    __syncthreads();
    M = fmaxf(top[0], top[1]);
    for (int c0 = 0, par = 0; c0 < nvalid; c0 += kMergeThreads, par ^= 1) {
      if (c0 + d < nvalid) {
        const float e = pl[c0 + d];
        weight[par][d] = e == -INFINITY ? 0.f : fast_exp2(e - M);
      }
      __syncthreads();  // (the other buffer is read until the next one)
      const int n = min(nvalid - c0, kMergeThreads);
      for (int c1 = 0; c1 < n; c1 += kMergeBatch) {
        float x[kMergeBatch];
#pragma unroll
        for (int i = 0; i < kMergeBatch; ++i)
          x[i] = po[(int64_t)(c0 + min(c1 + i, n - 1)) * D];
#pragma unroll
        for (int i = 0; i < kMergeBatch; ++i) {
          // (selects: a branch would pull the load down to it)
          const bool live = c1 + i < n;
          const float w = weight[par][min(c1 + i, n - 1)];
          den = live ? den + w : den;
          acc = live ? fmaf(w, x[i], acc) : acc;
        }
      }
    }
  }
  if (d < D) {
    T* op = reinterpret_cast<T*>(p.o) + b * p.o_sb + h * p.o_sh;
    op[d] = (T)(den == 0.f ? 0.f : acc / den);
  }
  if (d == 0 && p.lse) p.lse[(int64_t)b * p.hq + h] = den == 0.f ? -INFINITY : M + fast_log2(den);
}

template <typename T, int D, int NW>
int launch_waves(const DecodeParams& p, long long slots, long long resident, hipStream_t s) {
  if (p.list_mode != 0) {
    hipLaunchKernelGGL((decode_splitkv_kernel<T, D, NW, true>), dim3(p.n_splits, p.hkv * p.gslices, p.batch),
                       dim3(64 * NW), 0, s, p);
  } else {
    // one resident round, fewer workgroups when there are fewer chunks
    const unsigned grid = (unsigned)(slots * NW < resident ? slots : resident / NW);
    hipLaunchKernelGGL((decode_splitkv_kernel<T, D, NW, false>), dim3(grid), dim3(64 * NW), 0, s, p);
  }
  return (int)hipGetLastError();
}

// Wavefronts per chunk: as many as leave the launch within one resident round
// (8 wavefronts per CU), so that a call with few chunks still has eight streams
// in flight on every CU; where one wavefront to a chunk fills the round, the
// barriers of the others cost more than they give.  Whole call, one / two / four
// wavefronts, head_dim 128, 8 kv-heads: 8192 tokens 21.0 / 17.6 / 15.4 us, two
// sequences of 6k to 8k 22.6 / 20.5 / 20.5, one of 131072 99.7 / 96.8 / 110.9,
// 64 of 16k to 32k 1104 / 1157 / 1262.  (A list's chunk has two tiles per block.)
template <typename T, int D>
int launch_split(const DecodeParams& p, hipStream_t s) {
  const long long slots = (long long)p.n_splits * p.hkv * p.gslices * p.batch;
  const int cus = device_cu_count();
  const long long resident = 8LL * (cus > 0 ? cus : 256);
  const int tiles = p.list_mode != 0 ? 2 * p.split_blocks : p.split_tokens / kDecTile;
  if (4 * slots <= resident && tiles >= 4) return launch_waves<T, D, 4>(p, slots, resident, s);
  if (2 * slots <= resident && tiles >= 2) return launch_waves<T, D, 2>(p, slots, resident, s);
  return launch_waves<T, D, 1>(p, slots, resident, s);
}

}  // namespace

// Device address of `scratch` on the current device.  Looked up once per device
// with that device current (each GPU holds its own copy at its own address);
// the lookup allocates nothing.  Two threads racing on the first call both
// look it up and store the same value.
int decode_static_scratch(void** ptr) {
  constexpr int kMaxDev = 64;
  static std::atomic<void*> addr[kMaxDev];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDev) return (int)hipErrorInvalidDevice;
  void* a = addr[dev].load(std::memory_order_acquire);
  if (a == nullptr) {
    e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (a == nullptr) return (int)hipErrorInvalidSymbol;
    addr[dev].store(a, std::memory_order_release);
  }
  *ptr = a;
  return (int)hipSuccess;
}

int launch_decode_splitkv(const DecodeParams& p, int dtype, int head_dim, hipStream_t s) {
  if (dtype == 0) {
    switch (head_dim) {
      case 64: return launch_split<__bf16, 64>(p, s);
      case 96: return launch_split<__bf16, 96>(p, s);
      case 128: return launch_split<__bf16, 128>(p, s);
    }
  } else {
    switch (head_dim) {
      case 64: return launch_split<_Float16, 64>(p, s);
      case 96: return launch_split<_Float16, 96>(p, s);
      case 128: return launch_split<_Float16, 128>(p, s);
    }
  }
  return (int)hipErrorInvalidValue;
}

int launch_decode_merge(const DecodeParams& p, int dtype, int head_dim, hipStream_t s) {
  dim3 grid(p.hq, p.batch);
  auto pick = [&](auto zero) {
    using T = decltype(zero);
    return p.n_splits < 1 || p.n_splits > 256 ? decode_merge_kernel<T, 0>
           : p.n_splits <= 64                 ? decode_merge_kernel<T, 1> : decode_merge_kernel<T, 4>;
  };
  auto kern = dtype == 0 ? pick(__bf16()) : pick(_Float16());
  hipLaunchKernelGGL(kern, grid, dim3(kMergeThreads), 0, s, p, head_dim);
  return (int)hipGetLastError();
}

}  // namespace mi
