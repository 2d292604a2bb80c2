// Dense attention backward for gfx950: dq, dk, dv from q, k, v, o, do and the
// base-2 row log-sum-exp the forward pass returns.
//
// Replaces flash_attn_bwd_D_kernel, flash_attn_bwd_dq_kernel and
// flash_attn_bwd_dkdv_kernel (flash_attn_triton/flash_attn_triton.py:183-593)
// and their launcher flash_attn_triton_bwd (:661-813).  Math, with
// S2 = q.k * scale_log2, P = 2^(S2 - lse2), Delta_i = sum_d o_id do_id:
//   dV = P^T dO,   dP = dO V^T,   dS = P o (dP - Delta),
//   dQ = dS K * scale,   dK = dS^T Q * scale      (scale in the natural base).
// Delta is kept in fp32 (the reference rounds it to the input dtype, :677),
// P and dS are rounded to the input dtype before their second product as the
// reference does (in the dK + dV kernel dS is formed from the rounded P), the
// GQA members of a kv-head are accumulated in registers
// (the reference materialises one dk/dv per member and sums, :687-692,813).
//
// Two kernels on the forward pass's tile engine.  A wavefront keeps 32
// "resident" rows (their B operands) in registers and streams 64-row tiles of
// the other side through a three-stage LDS ring (direct-to-LDS loads).
//   dQ     : resident q, do rows; streams K, V.
//            S^T = K Q^T, dP^T = V dO^T, dQ^T += K^T dS^T
//            It also forms Delta of its resident rows (one pass over the o
//            rows) and stores it for the second kernel, which runs after it.
//   dK + dV: resident k, v rows; streams Q, dO (all query heads of the GQA
//            group in turn).  The work of a 32-row group is split between two
//            wavefronts that share a SIMD: one forms S, P and dV^T += dO^T P,
//            the other dP, dS and dK^T += Q^T dS (see bwd_dkdv_item).
// In every first product 16 streamed rows of ONE resident row land in each
// lane, and the rounded, pairwise packed result already is the B operand of
// the accumulating product; its A operand is a streamed tile read through the
// transposing LDS load.  Every streamed tile uses one layout that serves both
// the row-fragment read and the transposing read (UniFrags).
#include <algorithm>
#include <type_traits>

#include "item_order.h"
#include "kernels.h"
#include "tile_core.h"

namespace mi {
namespace {

template <int V>
using ic = std::integral_constant<int, V>;

// f(ic<B>{}), f(ic<B + 1>{}), ..., f(ic<E - 1>{})
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(ic<B>{});
    static_for<B + 1, E>(f);
  }
}

// vmcnt(N) expcnt(7) lgkmcnt(15) for s_waitcnt on gfx9-family encodings
constexpr int waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
// vmcnt(63) expcnt(7) lgkmcnt(N)
constexpr int waitcnt_lgkm(int n) { return 0xF | (3 << 14) | (7 << 4) | ((n & 0xF) << 8); }

// The lane id, computed here (no register has to carry it to this place).
__device__ __forceinline__ int opaque_lane() {
  int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  asm volatile("" : "+v"(lane));
  return lane;
}

// 256-byte rows (head_dim 64 and 96 leave the tail of a row unused), 16-byte
// chunks XOR-swizzled per row with a pattern
// that is free of bank conflicts for BOTH access patterns: a row-fragment read
// takes one chunk from 16 rows whose low four row bits are all different, a
// transposing read takes four consecutive chunks from four consecutive rows.
template <int D>
struct UniFrags {
  using G = RowGeom<D>;
  static constexpr int ROWB = 256;
  static constexpr int SLOTS = 16;
  static __device__ __forceinline__ int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
  int lq, lh;
  uint32_t r_a[G::KSTEPS];  // absolute LDS address of row fragment step c, block 0 of tile 0
  uint32_t t_a[G::NDB][2];  // same for the transposing read of (d block, first/second half)

  __device__ __forceinline__ void init(int lane, uint32_t lds_base) {
    lq = lane & 31;
    lh = lane >> 5;
    const int krow = key_perm(lq);
#pragma unroll
    for (int c = 0; c < G::KSTEPS; ++c) {
      r_a[c] = lds_base + krow * ROWB + (((2 * c + lh) ^ swz(krow)) << 4);
      asm volatile("" : "+v"(r_a[c]));
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int r = 8 * lh + 4 * e + ((lane & 15) >> 2);
#pragma unroll
      for (int db = 0; db < G::NDB; ++db) {
        const int ch = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
        t_a[db][e] = lds_base + r * ROWB + ((ch ^ swz(r)) << 4) + (lane & 1) * 8;
        asm volatile("" : "+v"(t_a[db][e]));
      }
    }
  }
  // swz is invariant under row += 16, so blocks are plain immediates
  __device__ __forceinline__ i32x4 rows(uint32_t tile_off, int blk, int c) const {
    typedef __attribute__((address_space(3))) const i32x4 lds_i32x4;
    return *(lds_i32x4*)(uintptr_t)(r_a[c] + tile_off + blk * 32 * ROWB);
  }
  __device__ __forceinline__ i32x4 tr(uint32_t tile_off, int kk, int db) const {
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(t_a[db][0] + tile_off + kk * 16 * ROWB));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(t_a[db][1] + tile_off + kk * 16 * ROWB));
    i32x2 l2 = __builtin_bit_cast(i32x2, lo);
    i32x2 h2 = __builtin_bit_cast(i32x2, hi);
    i32x4 out = {l2[0], l2[1], h2[0], h2[1]};
    return out;
  }
};

extern __shared__ __attribute__((aligned(1024))) unsigned char smem_bwd[];

constexpr int kBwdStages = 3;  // streamed tile pairs resident in LDS (4 measured the same)

// dQ: resident q, do rows; streams K, V.
//   S^T = K Q^T,  dP^T = V dO^T,  dS = P o (dP - Delta),  dQ^T += K^T dS^T
// NW wavefronts of 32 rows each: eight, two to a SIMD, or (launches of few items,
// see launch_all) four, while the other four send the loads.  A row meets its keys
// in the same order in both: the results are the same bits.
template <typename T, int D, int NW>
__device__ __forceinline__ void bwd_dq_item(const BwdParams& p, const int b, const int hr, const int rt, const int wave) {
  using G = RowGeom<D>;
  using F = UniFrags<D>;
  constexpr int BM = 32 * NW, TN = 64, NS = kBwdStages;
  constexpr bool kLoaders = NW == 4;              // wavefronts 4 to 7 send the loads and do nothing else
  constexpr int NL = kLoaders ? 4 : 8;            // wavefronts that send loads
  constexpr int TILEB = TN * F::ROWB;             // one streamed tile
  constexpr int STAGEB = 2 * TILEB + 1024;        // tile 0, tile 1, lse[64] and delta[64] (fp32)
  constexpr int RPI = 1024 / F::ROWB;             // tile rows per direct-to-LDS instruction
  constexpr int IPW = TN / RPI / NL;              // such instructions per tile and wave
  constexpr int IPT = 2 * IPW;                    // loads per streamed tile and wave
  constexpr int OROWB = D * 2 + 16;               // epilogue staging row

  // What is derived from the lane id (fragment addresses, load offsets) is
  // recomputed for every item instead of being held in registers across the
  // whole item loop, where it was spilled.
  const int lane = opaque_lane();

  const int gqa = p.hq / p.hkv;

  int len;
  int64_t start;  // first row of the sequence in packed tensors
  if (p.cu) {
    start = p.cu[b];
    // never beyond the bound the workspace and the grid were sized for
    len = min(p.cu[b + 1] - (int)start, p.max_seqlen);
  } else {
    start = 0;
    len = p.max_seqlen;
  }
  const int64_t bsel = p.cu ? 0 : b;
  const int r0 = rt * BM;
  if (rt < 0 || r0 >= len) return;

  F fr;
  const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem_bwd);
  fr.init(lane, lds0);
  const bool loader = kLoaders && wave >= NW;
  const int lw = wave & (NL - 1);               // which of the senders
  const int r0w = r0 + 32 * (wave & (NW - 1));
  const int rrow = r0w + fr.lq;                 // resident row of this lane
  const int rclamp = min(rrow, len - 1);

  // ---- resident B operands: lane (row lq, half lh) holds d = 16c + 8lh .. +7
  const T* xp = reinterpret_cast<const T*>(p.q) + bsel * p.q_sb + (start + rclamp) * p.q_ss + hr * p.q_sh;
  const T* yp = reinterpret_cast<const T*>(p.dout) + bsel * p.do_sb + (start + rclamp) * p.do_ss + hr * p.do_sh;
  const T* op = reinterpret_cast<const T*>(p.o) + bsel * p.o_sb + (start + rclamp) * p.o_ss + hr * p.o_sh;
  i32x4 Xf[G::KSTEPS], Yf[G::KSTEPS];
  // Delta[row] = sum_d o[row][d] * do[row][d] (fp32) is formed here, from the
  // resident do rows and one pass over the o rows, and stored for the dK + dV
  // kernel, which runs after this one.
  float delta_l = 0.f;
#pragma unroll
  for (int c = 0; c < G::KSTEPS; ++c) {
    Xf[c] = *reinterpret_cast<const i32x4*>(xp + 8 * fr.lh + 16 * c);
    Yf[c] = *reinterpret_cast<const i32x4*>(yp + 8 * fr.lh + 16 * c);
    const i32x4 Of = *reinterpret_cast<const i32x4*>(op + 8 * fr.lh + 16 * c);
    const T* oe = reinterpret_cast<const T*>(&Of);
    const T* de = reinterpret_cast<const T*>(&Yf[c]);
#pragma unroll
    for (int i = 0; i < 8; ++i) delta_l += (float)oe[i] * (float)de[i];
  }
  delta_l += __shfl_xor(delta_l, 32);
  if (fr.lh == 0 && rrow < len && !loader) p.delta[(int64_t)b * p.dl_sb + (int64_t)hr * p.dl_sh + rrow] = delta_l;
  const float lse_l = p.lse[bsel * p.lse_sb + (start + rclamp) * p.lse_ss + hr * p.lse_sh];

  f32x16 acc[G::NDB];
#pragma unroll
  for (int db = 0; db < G::NDB; ++db) acc[db] = (f32x16){0};

  // ---- streamed tiles: which rows, for which heads
  const int n_all = (len + TN - 1) / TN;
  const int n_stream = p.causal ? min(n_all, (r0 + BM + TN - 1) / TN) : n_all;  // key tiles 0 .. n_stream - 1

  // ---- direct-to-LDS loads (inline assembly: see the note in prefill.hip)
  const int drow = lane / F::SLOTS, dslot = lane % F::SLOTS;
  auto uniform64 = [](uint64_t x) __attribute__((always_inline)) -> uint64_t {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
  };
  // a load of the lanes in `mask` in straight-line code (all lanes are active
  // and control flow is wave-uniform here: exec is restored to all ones)
  auto dma_masked = [&](uint64_t mask, uint64_t base, uint32_t off, uint32_t slab) __attribute__((always_inline)) {
    if (kLoaders) {
      mask = uniform64(mask);
      base = uniform64(base);
      slab = (uint32_t)__builtin_amdgcn_readfirstlane(slab);
    }
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                 : : "s"(mask), "v"(off), "s"(base), "s"(slab) : "memory");
  };
  // Streamed tensors: K feeds the first product and, transposed, the last; V
  // the second.  Wave w sends slabs w and w + 8 (1 KiB = four rows) of either
  // tile; the swizzle of a lane's chunk depends on the slab only through
  // slab % 4, so one lane offset per tensor serves both and the slab moves the
  // scalar base.  The tile addresses are running, wave-uniform values.
  const int64_t pitch0 = p.k_ss * 2, pitch1 = p.v_ss * 2;
  const int hs = hr / gqa;
  const char* h0 = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.k) + bsel * p.k_sb + start * p.k_ss + hs * p.k_sh);
  const char* h1 = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.v) + bsel * p.v_sb + start * p.v_ss + hs * p.v_sh);
  uint64_t a0 = uniform64((uint64_t)(uintptr_t)h0), a1 = uniform64((uint64_t)(uintptr_t)h1);
  const uint64_t step0 = uniform64((uint64_t)(TN * pitch0)), step1 = uniform64((uint64_t)(TN * pitch1));
  const uint64_t slab0 = uniform64((uint64_t)(NL * RPI * pitch0)), slab1 = uniform64((uint64_t)(NL * RPI * pitch1));
  uint32_t off0, off1;
  uint64_t lane_mask;
  {
    const int r = RPI * lw + drow;
    const int c = dslot ^ F::swz(r);
    off0 = (uint32_t)r * (uint32_t)pitch0 + c * 16;
    off1 = (uint32_t)r * (uint32_t)pitch1 + c * 16;
    lane_mask = __builtin_amdgcn_ballot_w64(G::NCH == 16 || c < G::NCH);
  }
  static_assert(kLoaders || IPT == 4, "compute_fast() places four loads");
  int iss_s0 = 0;            // first row of the next request
  int iss_st = 0;            // its stage
  uint32_t iss_base = lds0;  // and the stage's LDS address
  uint64_t drip_on = 0;      // all ones while the loads of a request are still to be sent by a compute step
  // request(): a tile that reaches past the sequence end is loaded at once,
  // row by row with clamped row numbers (masked later); a whole tile only arms
  // drip(), and the compute step sends the four loads between its MFMAs.
  auto request = [&]() __attribute__((always_inline)) {
    if (iss_s0 + TN <= len) {
      drip_on = ~0ull;
    } else {
      drip_on = 0;
      const int last = len - 1 - iss_s0;  // >= 0
#pragma unroll
      for (int t = 0; t < IPW; ++t) {
        const int inst = lw + NL * t;
        const int r = RPI * inst + drow;
        const int c = dslot ^ F::swz(r);
        const int64_t rr = min(r, last);
        const uint32_t slab = (uint32_t)__builtin_amdgcn_readfirstlane(iss_base + inst * 1024);
        if (G::NCH == 16 || c < G::NCH) {
          asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                       : : "v"((const char*)a0 + rr * pitch0 + c * 16), "s"(slab) : "memory");
          asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                       : : "v"((const char*)a1 + rr * pitch1 + c * 16), "s"(slab + TILEB) : "memory");
        }
      }
    }
  };
  // load k of a request: k & 1 = tensor, k >> 1 = slab
  auto drip = [&](int k) __attribute__((always_inline)) {
    const int t = k >> 1;
    const int inst = lw + NL * t;
    if (k & 1)
      dma_masked(drip_on & lane_mask, a1 + t * slab1, off1, iss_base + TILEB + inst * 1024);
    else
      dma_masked(drip_on & lane_mask, a0 + t * slab0, off0, iss_base + inst * 1024);
  };
  auto drip_all = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < IPT; ++k) drip(k);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    drip_on = 0;
    iss_s0 += TN;
    a0 += step0;
    a1 += step1;
    const bool last_st = iss_st == NS - 1;
    iss_st = last_st ? 0 : iss_st + 1;
    iss_base = last_st ? lds0 : iss_base + STAGEB;
  };

  const float scale = p.scale;
  const int causal = p.causal;

  // ---- this wave's view of the tile it works on: LDS addresses that move
  // from stage to stage (one add per address register and step; every read is
  // then "register + immediate": absolute stage offsets exceed the 16-bit
  // immediate of an LDS instruction)
  int cmp_st = 0;
  auto rotate = [&]() __attribute__((always_inline)) {
    const bool last_st = cmp_st == NS - 1;
    const int d = last_st ? -(NS - 1) * STAGEB : STAGEB;
    cmp_st = last_st ? 0 : cmp_st + 1;
#pragma unroll
    for (int c = 0; c < G::KSTEPS; ++c) fr.r_a[c] += d;
#pragma unroll
    for (int db = 0; db < G::NDB; ++db) {
      fr.t_a[db][0] += d;
      fr.t_a[db][1] += d;
    }
  };

  constexpr int kPrefetch = 4;
  constexpr int K = G::KSTEPS;
  // slice of block 0's S chain behind which the n-th of a tile's four loads goes
  auto drip_slice = [](int n) constexpr { return K == 8 ? 2 * n + 1 : K == 6 ? n + 1 + (n >= 2) : n; };
  i32x4 f[kPrefetch];   // row fragments of the first two products, read ahead
  // One 32-row block of the streamed tile as one pinned instruction stream
  // (sched_barrier(0) after every slice): the S chain; the dP chain with the
  // exponentials of S behind its MFMAs; the first half of dS; the last product
  // with the second half of dS behind its first MFMAs.  Row fragments are read
  // four steps ahead, transposed fragments two.  Register r of this lane is
  // streamed row  sblk + 16*(r/8) + 8*lh + r%8.
  auto block = [&](auto sb_c, auto masked_c, const int sblk, const bool f_ready) __attribute__((always_inline)) {
    constexpr int sb = decltype(sb_c)::value;
    constexpr bool masked = decltype(masked_c)::value != 0;
    constexpr int NSTEP = 2 * K;
    f32x16 S = (f32x16){0}, dP = (f32x16){0};
    auto frag = [&](int st) __attribute__((always_inline)) -> i32x4 {
      return st < K ? fr.rows(0, sb, st) : fr.rows(TILEB, sb, st - K);
    };
    auto prob = [&](int r) __attribute__((always_inline)) {   // S[r] <- P[r]
      S[r] = fast_exp2(fmaf(S[r], scale, -lse_l));
    };
    auto dsv = [&](int r) __attribute__((always_inline)) -> float {
      return S[r] * (dP[r] - delta_l);
    };
    if (!f_ready) {
#pragma unroll
      for (int st = 0; st < kPrefetch; ++st) f[st] = frag(st);
    }
    // Issue priority: highest while the wave feeds the accumulators (the last
    // product, 2*NDB MFMAs over NDB independent chains), low during the two
    // serial chains S and dP; the two waves of a SIMD then fall out of step
    // instead of competing with the same kind of work (measured 3 %).
    __builtin_amdgcn_s_setprio(1);
    static_for<0, K>([&](auto st_c) __attribute__((always_inline)) {
      constexpr int st = decltype(st_c)::value;
      S = Elem<T>::mfma(f[st % kPrefetch], Xf[st], S);
      if (st + kPrefetch < NSTEP) f[st % kPrefetch] = frag(st + kPrefetch);
      if (sb == 0 && !masked && !kLoaders)
        static_for<0, IPT>([&](auto n_c) __attribute__((always_inline)) {
          if (st == drip_slice(decltype(n_c)::value)) drip(decltype(n_c)::value);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
    if (masked) {
      // rows / columns that do not exist or lie above the diagonal give P = 0
      bool need_mask = sblk + 32 > len;
      if (causal) need_mask = need_mask || sblk + 31 > r0w;
      if (need_mask) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int srow = sblk + 16 * (r >> 3) + 8 * fr.lh + (r & 7);
          const bool ok = srow < len && (!causal || srow <= rrow);
          S[r] = ok ? S[r] : -INFINITY;
        }
      }
    }
    i32x4 tf[2];
    uint32_t W[8];
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const int st = K + c;
      dP = Elem<T>::mfma(f[st % kPrefetch], Yf[c], dP);
      if (st + kPrefetch < NSTEP) f[st % kPrefetch] = frag(st + kPrefetch);
      if (c >= K - 2) tf[c - (K - 2)] = fr.tr(0, 2 * sb, c - (K - 2));
      // 16 exponentials spread over the K slices
#pragma unroll
      for (int r = 16 * c / K; r < 16 * (c + 1) / K; ++r) prob(r);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) W[i] = Elem<T>::pack2(dsv(2 * i), dsv(2 * i + 1));
    __builtin_amdgcn_sched_barrier(0);
    // last product: 2*NDB MFMAs, fragment (kk, db) = step kk*NDB + db
    constexpr int NACC = 2 * G::NDB;
    __builtin_amdgcn_s_setprio(3);
#pragma unroll
    for (int i = 0; i < NACC; ++i) {
      const int kk = i / G::NDB, db = i % G::NDB;
      const i32x4 wf = {(int)W[4 * kk], (int)W[4 * kk + 1], (int)W[4 * kk + 2], (int)W[4 * kk + 3]};
      acc[db] = Elem<T>::mfma(tf[i & 1], wf, acc[db]);
      if (i + 2 < NACC) tf[i & 1] = fr.tr(0, 2 * sb + (i + 2) / G::NDB, (i + 2) % G::NDB);
      // the ring is idle now: fetch the first fragments of the tile's second block
      if (sb == 0 && i >= NACC - kPrefetch) f[i - (NACC - kPrefetch)] = fr.rows(0, 1, i - (NACC - kPrefetch));
      if (i < G::NDB) {
        // second half of dS (8 values) spread over the first NDB slices
#pragma unroll
        for (int q = 4 * i / G::NDB; q < 4 * (i + 1) / G::NDB; ++q)
          W[4 + q] = Elem<T>::pack2(dsv(8 + 2 * q), dsv(9 + 2 * q));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // a tile whose 64 keys all exist and lie at or before this wave's first query
  auto compute_fast = [&](int s0) __attribute__((always_inline)) {
    block(ic<0>{}, ic<0>{}, s0, false);
    block(ic<1>{}, ic<0>{}, s0 + 32, true);
  };
  // a tile on the diagonal or at the sequence end
  auto compute_slow = [&](int s0) __attribute__((always_inline)) {
    if (!kLoaders) drip_all();
    bool f_ready = false;
    if (s0 < len && !(causal && s0 > r0w + 31)) {
      block(ic<0>{}, ic<1>{}, s0, false);
      f_ready = true;
    }
    if (s0 + 32 < len && !(causal && s0 + 32 > r0w + 31)) block(ic<1>{}, ic<1>{}, s0 + 32, f_ready);
  };

  // tiles 0 .. NS-2 are requested up front; step u requests tile u + NS - 1
  // into the stage that tile u - 1 has left
#pragma unroll
  for (int u = 0; u < NS - 1; ++u)
    if (u < n_stream && (!kLoaders || loader)) {
      request();
      drip_all();
      advance();
    }
  // resident operands and tile 0 are needed now; the full wait also tells the
  // compiler that no register load is pending inside the loop
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  __syncthreads();
  // Each loop below holds ONE kind of step (with the masked and the unmasked
  // path in one loop body the accumulators were copied between two register
  // sets on every trip); every step ends in the workgroup's barrier, so the
  // waves may split the tiles differently.
  int n_fast = min(n_stream, len / TN);
  if (causal) n_fast = min(n_fast, (r0w + 1) / TN);
  auto step = [&](auto fast_c, int u) __attribute__((always_inline)) {
    const bool refill = !kLoaders && u + NS - 1 < n_stream;
    if (refill) request();
    if (decltype(fast_c)::value)
      compute_fast(u * TN);
    else
      compute_slow(u * TN);
    rotate();
    if (refill) advance();
    // the next tile must have landed (this wave's loads retire in order: only
    // the tile requested in this step may still fly) and everyone is done with this one
    if (refill)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(IPT));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    __syncthreads();
  };
  if (loader) {
    for (int u = 0; u < n_stream; ++u) {
      const bool refill = u + NS - 1 < n_stream;
      if (refill) {
        request();
        drip_all();
        advance();
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(IPT));
      } else {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
      }
      __syncthreads();
    }
    __syncthreads();
    return;
  }
  for (int u = 0; u < n_fast; ++u) step(ic<1>{}, u);
  for (int u = n_fast; u < n_stream; ++u) step(ic<0>{}, u);
  __builtin_amdgcn_s_setprio(0);
  __syncthreads();

  // ---- epilogue: scale, transpose through LDS, coalesced 16-byte stores
  const float oscale = p.scale_nat;
  T* outp = reinterpret_cast<T*>(p.dq) + bsel * p.dq_sb + start * p.dq_ss + hr * p.dq_sh;
  const int64_t o_ss = p.dq_ss;
  unsigned char* stage = smem_bwd + wave * 32 * OROWB;
#pragma unroll
  for (int db = 0; db < G::NDB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * db + 8 * g + 4 * fr.lh;
      i32x2 w;
      w[0] = (int)Elem<T>::pack2(acc[db][4 * g] * oscale, acc[db][4 * g + 1] * oscale);
      w[1] = (int)Elem<T>::pack2(acc[db][4 * g + 2] * oscale, acc[db][4 * g + 3] * oscale);
      *reinterpret_cast<i32x2*>(stage + fr.lq * OROWB + d * 2) = w;
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wavefront reads only what it has staged itself)
#pragma unroll
  for (int i = 0; i < (32 * G::NCH + 63) / 64; ++i) {
    const int idx = lane + 64 * i;
    const int row = idx / G::NCH, ch = idx % G::NCH;
    if (((32 * G::NCH) % 64 == 0 || idx < 32 * G::NCH) && r0w + row < len) {
      const i32x4 val = *reinterpret_cast<const i32x4*>(stage + row * OROWB + ch * 16);
      *reinterpret_cast<i32x4*>(outp + (int64_t)(r0w + row) * o_ss + ch * 8) = val;
    }
  }
}

// ---------------------------------------------------------------------------
// dK and dV in one pass (replaces flash_attn_bwd_dkdv_kernel,
// flash_attn_triton/flash_attn_triton.py:413-592, which also forms both in one
// kernel).  Both accumulators of 32 resident k / v rows (2 x 64 registers at
// head_dim 128) plus the two resident B operands do not fit one wavefront at
// two wavefronts per SIMD, so the work of a 32-row group is split between TWO
// wavefronts that share a SIMD (waves w and w + 4):
//   score wave:  S = Q K^T -> P = 2^(S scale - lse),   dV^T += dO^T P
//   grad wave :  dP = dO V^T, dS = P o (dP - Delta),   dK^T += Q^T dS
// Each holds one resident operand (k or v), one accumulator, and runs half of
// the MFMAs; S and P are computed once for both gradients and Q / dO are
// streamed once.  P travels from the score wave to the grad wave through LDS,
// rounded to the storage dtype (the operand of dV; the reference forms dS from
// the fp32 P, :578): the score wave works one streamed tile AHEAD of the grad
// wave, so the barrier that ends a tile step is the only synchronisation.
template <typename T, int D, int NP, typename Next>
__device__ __forceinline__ void bwd_dkdv_item(const BwdParams& p, const int b, const int hr, const int rt, const int wave,
                                              Next&& take_next) {
  using G = RowGeom<D>;
  using F = UniFrags<D>;
  constexpr int BM = 32 * NP, TN = 64, NS = kBwdStages;
  static_assert(NS == 3, "stage reuse below assumes three stages");
  constexpr int TILEB = TN * F::ROWB;
  constexpr int STAGEB = 2 * TILEB + 1024;
  constexpr int RPI = 1024 / F::ROWB;
  constexpr int OROWB = D * 2 + 16;
  constexpr uint32_t PBUF = NS * STAGEB;       // P exchange: [2 tile slots][NP pairs][2 blocks][2 KiB]
  constexpr uint32_t PSLOT = NP * 2 * 2048;

  const int lane = opaque_lane();
  constexpr bool kLoaders = NP == 2;  // waves 4 to 7 send the loads and do nothing else
  const int pr = wave & (NP - 1);             // 32-row group of the item
  const bool grad = (wave & (2 * NP - 1)) >= NP;  // role of this wave
  const bool loader = kLoaders && wave >= 4;
  const bool sends = kLoaders ? loader : !grad;
  const int lw = wave & 3;            // which of the four senders
  // The wavefront that takes the workgroup's next unit, during the last step, in which it has nothing else to do
  // (at the start of an item the choice would be made before anyone knows who will be done first).
  constexpr int kTaker = kLoaders ? 7 : 3;

  const int gqa = p.hq / p.hkv;
  int len;
  int64_t start;
  if (p.cu) {
    start = p.cu[b];
    // never beyond the bound the workspace and the grid were sized for
    len = min(p.cu[b + 1] - (int)start, p.max_seqlen);
  } else {
    start = 0;
    len = p.max_seqlen;
  }
  const int64_t bsel = p.cu ? 0 : b;
  const int r0 = rt * BM;
  if (rt < 0 || r0 >= len) {
    if (wave == kTaker) take_next();
    return;
  }

  F fr;
  const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem_bwd);
  fr.init(lane, lds0);
  const int r0w = r0 + 32 * pr;
  const int rrow = r0w + fr.lq;
  const int rclamp = min(rrow, len - 1);

  // resident B operand: k rows (score wave) or v rows (grad wave)
  const T* xp = grad ? reinterpret_cast<const T*>(p.v) + bsel * p.v_sb + (start + rclamp) * p.v_ss + hr * p.v_sh
                     : reinterpret_cast<const T*>(p.k) + bsel * p.k_sb + (start + rclamp) * p.k_ss + hr * p.k_sh;
  i32x4 Xf[G::KSTEPS];
#pragma unroll
  for (int c = 0; c < G::KSTEPS; ++c) Xf[c] = *reinterpret_cast<const i32x4*>(xp + 8 * fr.lh + 16 * c);

  f32x16 acc[G::NDB];
#pragma unroll
  for (int db = 0; db < G::NDB; ++db) acc[db] = (f32x16){0};

  const int n_all = (len + TN - 1) / TN;
  const int j0 = p.causal ? r0 / TN : 0;
  const int nj = n_all - j0;
  const int n_stream = nj * gqa;

  const int drow = lane / F::SLOTS, dslot = lane % F::SLOTS;
  auto uniform64 = [](uint64_t x) __attribute__((always_inline)) -> uint64_t {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
  };
  // A direct-to-LDS load of the lanes in `mask` (all 64 lanes are active and
  // control flow is wave-uniform wherever this is called, so exec is restored
  // to all ones).  Switching a load off through the exec mask keeps it in
  // straight-line code: a branch around it would end the basic block and let
  // the compiler move the arithmetic that is meant to sit behind the MFMAs.
  auto dma_masked = [&](uint64_t mask, uint64_t base, uint32_t off, uint32_t slab, auto wide_c) __attribute__((always_inline)) {
    if (kLoaders) {
      mask = uniform64(mask);
      base = uniform64(base);
      slab = (uint32_t)__builtin_amdgcn_readfirstlane(slab);
    }
    if (decltype(wide_c)::value)
      asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                   : : "s"(mask), "v"(off), "s"(base), "s"(slab) : "memory");
    else
      asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b64 exec, -1"
                   : : "s"(mask), "v"(off), "s"(base), "s"(slab) : "memory");
  };

  // ---- streamed tiles.  Per tile and wavefront: four loads of 1 KiB (two of
  // Q, two of dO); wavefronts 0 and 1 also fetch the tile's 64 lse / Delta
  // values.  The addresses are running, wave-uniform values: they advance by
  // one tile per request and jump to the next query head of the group when a
  // head's tiles are through (one add each per step; the item's scalar
  // bookkeeping is issued by the same wavefronts that feed the MFMAs, one
  // instruction per four cycles, so every instruction saved per step counts).
  const int64_t pitch0 = p.q_ss * 2, pitch1 = p.do_ss * 2;
  const char* h0 = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.q) + bsel * p.q_sb + (start + j0 * TN) * p.q_ss + hr * gqa * p.q_sh);
  const char* h1 = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.dout) + bsel * p.do_sb + (start + j0 * TN) * p.do_ss + hr * gqa * p.do_sh);
  const char* hl = lw == 0
      ? reinterpret_cast<const char*>(p.lse + bsel * p.lse_sb + (start + j0 * TN) * p.lse_ss + hr * gqa * p.lse_sh)
      : reinterpret_cast<const char*>(p.delta + (int64_t)b * p.dl_sb + (int64_t)hr * gqa * p.dl_sh + j0 * TN);
  const int64_t pitchl = lw == 0 ? p.lse_ss * 4 : 4;
  uint64_t a0 = uniform64((uint64_t)(uintptr_t)h0), a1 = uniform64((uint64_t)(uintptr_t)h1), al = uniform64((uint64_t)(uintptr_t)hl);
  const uint64_t step0 = uniform64((uint64_t)(TN * pitch0)), step1 = uniform64((uint64_t)(TN * pitch1));
  const uint64_t stepl = uniform64((uint64_t)(TN * pitchl));
  const uint64_t wrap0 = uniform64((uint64_t)(p.q_sh * 2 - (int64_t)(nj - 1) * TN * pitch0));
  const uint64_t wrap1 = uniform64((uint64_t)(p.do_sh * 2 - (int64_t)(nj - 1) * TN * pitch1));
  const uint64_t wrapl = uniform64((uint64_t)((lw == 0 ? p.lse_sh * 4 : p.dl_sh * 4) - (int64_t)(nj - 1) * TN * pitchl));
  // The four score wavefronts send the loads (the grad wavefronts carry more
  // arithmetic per tile): wave pr sends slabs pr, pr + 4, pr + 8, pr + 12 of
  // the Q tile and of the dO tile (1 KiB = four rows each).  The swizzle of a
  // lane's chunk depends on the slab only through slab % 4, so one lane offset
  // per tensor serves all four slabs; the slab moves the scalar base.
  constexpr int kSlabs = TN / RPI / 4;      // slabs per tensor, tile and score wave
  constexpr int kDrips = 2 * kSlabs;
  static_assert(kDrips == 8, "compute_fast() places eight loads");
  uint32_t off0, off1;
  uint64_t lane_mask;
  {
    const int r = RPI * lw + drow;
    const int c = dslot ^ F::swz(r);
    off0 = (uint32_t)r * (uint32_t)pitch0 + c * 16;
    off1 = (uint32_t)r * (uint32_t)pitch1 + c * 16;
    lane_mask = __builtin_amdgcn_ballot_w64(G::NCH == 16 || c < G::NCH);
  }
  const uint64_t slab0 = uniform64((uint64_t)(4 * RPI * pitch0)), slab1 = uniform64((uint64_t)(4 * RPI * pitch1));
  const uint32_t lv_off = (uint32_t)lane * (uint32_t)pitchl;
  const uint64_t lv_mask = lw < 2 ? ~0ull : 0ull;
  int iss_left = nj;        // tiles of the current head still to request
  int iss_s0 = j0 * TN;     // first row of the next request
  int iss_st = 0;           // its stage
  uint32_t iss_base = lds0; // and the stage's LDS address
  uint64_t drip_on = 0;     // all ones while the loads of a request are still to be sent by compute_fast()
  // request(): a tile that reaches past the sequence end is loaded at once,
  // row by row with clamped row numbers (masked later); a full tile only arms
  // drip(), and compute_fast() sends the loads between its MFMAs: wavefronts
  // that send their loads together right after the barrier stand in the
  // memory pipeline's queue before any of them starts its arithmetic.
  auto request = [&]() __attribute__((always_inline)) {
    if (iss_s0 + TN <= len) {
      drip_on = ~0ull;
    } else {
      drip_on = 0;
      if (!sends) return;
      const int last = len - 1 - iss_s0;  // >= 0
      const int ln = opaque_lane();
#pragma unroll
      for (int t = 0; t < kSlabs; ++t) {
        const int inst = lw + 4 * t;
        const int r = RPI * inst + ln / F::SLOTS;
        const int c = (ln % F::SLOTS) ^ F::swz(r);
        const int64_t rr = min(r, last);
        const uint32_t slab = (uint32_t)__builtin_amdgcn_readfirstlane(iss_base + inst * 1024);
        if (G::NCH == 16 || c < G::NCH) {
          asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                       : : "v"((const char*)a0 + rr * pitch0 + c * 16), "s"(slab) : "memory");
          asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                       : : "v"((const char*)a1 + rr * pitch1 + c * 16), "s"(slab + TILEB) : "memory");
        }
      }
      if (lw < 2) {
        const int64_t rr = min(ln, last);
        const uint32_t slab = (uint32_t)__builtin_amdgcn_readfirstlane(iss_base + 2 * TILEB + (lw == 0 ? 0 : 256));
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
                     : : "v"((const char*)al + rr * pitchl), "s"(slab) : "memory");
      }
    }
  };
  // load k of a request (score waves): k & 1 = tensor, k >> 1 = slab
  auto drip = [&](int k) __attribute__((always_inline)) {
    const int t = k >> 1;
    const int inst = lw + 4 * t;
    if (k & 1)
      dma_masked(drip_on & lane_mask, a1 + t * slab1, off1, iss_base + TILEB + inst * 1024, ic<1>{});
    else
      dma_masked(drip_on & lane_mask, a0 + t * slab0, off0, iss_base + inst * 1024, ic<1>{});
    if (k == 0) dma_masked(drip_on & lv_mask, al, lv_off, iss_base + 2 * TILEB + (lw == 0 ? 0 : 256), ic<0>{});
  };
  auto drip_all = [&]() __attribute__((always_inline)) {
    if (!sends) return;
#pragma unroll
    for (int k = 0; k < kDrips; ++k) drip(k);
  };
  // after the loads of a request are out: the next request's addresses
  auto advance = [&]() __attribute__((always_inline)) {
    drip_on = 0;
    if (--iss_left == 0) {
      iss_left = nj;
      iss_s0 = j0 * TN;
      a0 += wrap0;
      a1 += wrap1;
      al += wrapl;
    } else {
      iss_s0 += TN;
      a0 += step0;
      a1 += step1;
      al += stepl;
    }
    const bool last_st = iss_st == NS - 1;
    iss_st = last_st ? 0 : iss_st + 1;
    iss_base = last_st ? lds0 : iss_base + STAGEB;
  };

  const float scale = p.scale;
  const int causal = p.causal;
  typedef __attribute__((address_space(3))) i32x4 lds_i32x4;
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) const f32x4 lds_f4;

  // ---- this wave's view of the tile it works on: LDS addresses that move
  // from stage to stage (one add per address register and step, every read
  // then is "register + immediate"; absolute stage offsets exceed the 16-bit
  // immediate of an LDS instruction)
  {
    const uint32_t tro = grad ? TILEB : 0;   // tile read as row fragments: dO (grad) / Q (score)
    const uint32_t tto = grad ? 0 : TILEB;   // tile read transposed for the accumulating product
#pragma unroll
    for (int c = 0; c < G::KSTEPS; ++c) fr.r_a[c] += tro;
#pragma unroll
    for (int db = 0; db < G::NDB; ++db) {
      fr.t_a[db][0] += tto;
      fr.t_a[db][1] += tto;
    }
  }
  uint32_t lva = lds0 + 2 * TILEB + (grad ? 256u : 0u) + 8 * fr.lh * 4;   // lse (score) / Delta (grad) of the tile's rows
  uint32_t pbv = lds0 + PBUF + (uint32_t)pr * 4096 + (uint32_t)lane * 16;   // P exchange slot of this 32-row group
  int pb_step = (int)PSLOT;
  int cmp_st = 0, cmp_left = nj, cmp_s0 = j0 * TN;
  const bool rows_full = r0w + 32 <= len;
  auto rotate = [&]() __attribute__((always_inline)) {
    const bool last_st = cmp_st == NS - 1;
    const int d = last_st ? -(NS - 1) * STAGEB : STAGEB;
    cmp_st = last_st ? 0 : cmp_st + 1;
#pragma unroll
    for (int c = 0; c < G::KSTEPS; ++c) fr.r_a[c] += d;
#pragma unroll
    for (int db = 0; db < G::NDB; ++db) {
      fr.t_a[db][0] += d;
      fr.t_a[db][1] += d;
    }
    lva += d;
    pbv += pb_step;
    pb_step = -pb_step;
    if (--cmp_left == 0) {
      cmp_left = nj;
      cmp_s0 = j0 * TN;
    } else {
      cmp_s0 += TN;
    }
  };

  constexpr int kPrefetch = 4;
  constexpr int NACC = 2 * G::NDB;
  // One streamed tile for this wave's role, common case: all 64 streamed rows
  // and all 32 resident rows exist and no pair is masked.  The two 32-row
  // blocks of the tile are worked on as one software pipeline, so that the
  // wave's vector arithmetic sits behind its own MFMAs:
  //   1. chain(0)                          3. accumulate(0)  + arithmetic(1)
  //   2. chain(1)  + arithmetic(0)         4. accumulate(1)
  auto compute_fast = [&](auto role_c) __attribute__((always_inline)) {
    constexpr bool grad = decltype(role_c)::value != 0;
    {
      // Slots of the pipeline: phase 1 is slots 0 .. K-1, phase 2 K .. 2K-1,
      // phase 3 2K .. 2K+NACC-1.  Pair i of block 0 is formed in phase 2,
      // pair j of block 1 in phase 3; the lse / Delta values (four per LDS
      // read) and the packed P a pair needs are read two slots earlier, so
      // that only a few of them are live at a time (registers).
      constexpr int K = G::KSTEPS;
      // slice of a chain phase behind which the n-th of its four loads goes
      auto drip_slice = [](int n) constexpr { return K == 8 ? 2 * n + 1 : K == 6 ? n + 1 + (n >= 2) : n; };
      auto slice_of = [](int i, int n) constexpr { int st = 0; while ((st + 1) * 8 / n <= i) ++st; return st; };
      auto use_slot = [&](int sb, int i) constexpr { return sb == 0 ? K + slice_of(i, K) : 2 * K + slice_of(i, NACC); };
      float lv[2][16];
      i32x4 pp[2][2];  // grad wave: packed P of the two blocks
      auto load_lv = [&](int sb, int q) __attribute__((always_inline)) {
        const f32x4 v4 = *(lds_f4*)(uintptr_t)(lva + (32 * sb + 16 * (q >> 1) + 4 * (q & 1)) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) lv[sb][4 * q + e] = v4[e];
      };
      // reads due at `slot` (or, for slot 0, everything due at or before it)
      auto side_reads = [&](auto slot_c) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_c)::value;
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int due = use_slot(sb, 2 * q) - 2;
            if (due == slot || (slot == 0 && due < 0)) load_lv(sb, q);
          }
          if (grad) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int due = use_slot(sb, 4 * h) - 2;
              if (due == slot || (slot == 0 && due < 0)) pp[sb][h] = *(lds_i32x4*)(uintptr_t)(pbv + sb * 2048 + h * 1024);
            }
          }
        }
      };
      f32x16 S0 = (f32x16){0}, S1 = (f32x16){0};
      uint32_t W0[8], W1[8];
      // pair i of a block: P (score wave) or dS (grad wave), rounded and packed
      auto pair = [&](const f32x16& S, const float* lvb, const i32x4* ppb, int i) __attribute__((always_inline)) -> uint32_t {
        if (!grad) {
          return Elem<T>::pack2(fast_exp2(fmaf(S[2 * i], scale, -lvb[2 * i])),
                                fast_exp2(fmaf(S[2 * i + 1], scale, -lvb[2 * i + 1])));
        } else {
          const uint32_t pk = (uint32_t)(i < 4 ? ppb[0][i] : ppb[1][i - 4]);
          float plo, phi;
          if (std::is_same<T, __bf16>::value) {
            plo = __builtin_bit_cast(float, pk << 16);
            phi = __builtin_bit_cast(float, pk & 0xffff0000u);
          } else {
            const f16x2 h2 = __builtin_bit_cast(f16x2, pk);
            plo = (float)h2[0];
            phi = (float)h2[1];
          }
          return Elem<T>::pack2(plo * (S[2 * i] - lvb[2 * i]), phi * (S[2 * i + 1] - lvb[2 * i + 1]));
        }
      };
      i32x4 f[kPrefetch];
#pragma unroll
      for (int st = 0; st < kPrefetch; ++st) f[st] = st < K ? fr.rows(0, 0, st) : fr.rows(0, 1, st - K);
      __builtin_amdgcn_s_setprio(1);
      // 1. chain of block 0
      static_for<0, K>([&](auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value;
        S0 = Elem<T>::mfma(f[st % kPrefetch], Xf[st], S0);
        constexpr int nx = st + kPrefetch;
        f[st % kPrefetch] = nx < K ? fr.rows(0, 0, nx) : fr.rows(0, 1, nx - K);
        side_reads(ic<st>{});
        if (!grad && !kLoaders)
          static_for<0, 4>([&](auto n_c) __attribute__((always_inline)) {
            if (st == drip_slice(decltype(n_c)::value)) drip(decltype(n_c)::value);
          });
        __builtin_amdgcn_sched_barrier(0);
      });
      // 2. chain of block 1, arithmetic of block 0
      i32x4 tf[2];
      tf[0] = fr.tr(0, 0, 0);
      tf[1] = fr.tr(0, 0, 1);
      static_for<0, K>([&](auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value;
        S1 = Elem<T>::mfma(f[(st + K) % kPrefetch], Xf[st], S1);
        constexpr int nx = st + kPrefetch;
        if (nx < K) f[(st + K) % kPrefetch] = fr.rows(0, 1, nx);
        side_reads(ic<K + st>{});
#pragma unroll
        for (int i = st * 8 / K; i < (st + 1) * 8 / K; ++i) {
          W0[i] = pair(S0, lv[0], pp[0], i);
          asm volatile("" : "+v"(W0[i]));  // computed here, behind this MFMA
        }
        if (!grad && !kLoaders)
          static_for<0, 4>([&](auto n_c) __attribute__((always_inline)) {
            if (st == drip_slice(decltype(n_c)::value)) drip(4 + decltype(n_c)::value);
          });
        __builtin_amdgcn_sched_barrier(0);
      });
      if (!grad) {
        *(lds_i32x4*)(uintptr_t)(pbv) = (i32x4){(int)W0[0], (int)W0[1], (int)W0[2], (int)W0[3]};
        *(lds_i32x4*)(uintptr_t)(pbv + 1024) = (i32x4){(int)W0[4], (int)W0[5], (int)W0[6], (int)W0[7]};
      }
      __builtin_amdgcn_s_setprio(3);
      // 3. accumulating product of block 0, arithmetic of block 1
      static_for<0, NACC>([&](auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        constexpr int kk = i / G::NDB, db = i % G::NDB;
        const i32x4 wf = {(int)W0[4 * kk], (int)W0[4 * kk + 1], (int)W0[4 * kk + 2], (int)W0[4 * kk + 3]};
        acc[db] = Elem<T>::mfma(tf[i & 1], wf, acc[db]);
        constexpr int nx = i + 2;
        tf[i & 1] = nx < NACC ? fr.tr(0, nx / G::NDB, nx % G::NDB) : fr.tr(0, 2 + (nx - NACC) / G::NDB, (nx - NACC) % G::NDB);
        side_reads(ic<2 * K + i>{});
#pragma unroll
        for (int j = i * 8 / NACC; j < (i + 1) * 8 / NACC; ++j) {
          W1[j] = pair(S1, lv[1], pp[1], j);
          asm volatile("" : "+v"(W1[j]));
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if (!grad) {
        *(lds_i32x4*)(uintptr_t)(pbv + 2048) = (i32x4){(int)W1[0], (int)W1[1], (int)W1[2], (int)W1[3]};
        *(lds_i32x4*)(uintptr_t)(pbv + 2048 + 1024) = (i32x4){(int)W1[4], (int)W1[5], (int)W1[6], (int)W1[7]};
      }
      // 4. accumulating product of block 1
#pragma unroll
      for (int i = 0; i < NACC; ++i) {
        const int kk = i / G::NDB, db = i % G::NDB;
        const i32x4 wf = {(int)W1[4 * kk], (int)W1[4 * kk + 1], (int)W1[4 * kk + 2], (int)W1[4 * kk + 3]};
        acc[db] = Elem<T>::mfma(tf[i & 1], wf, acc[db]);
        if (i + 2 < NACC) tf[i & 1] = fr.tr(0, 2 + (i + 2) / G::NDB, (i + 2) % G::NDB);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // Tiles on the diagonal or at the sequence end: block by block, with masks.
  auto compute_slow = [&](auto role_c) __attribute__((always_inline)) {
    constexpr bool grad = decltype(role_c)::value != 0;
    const int s0 = cmp_s0;
    if (!kLoaders) drip_all();
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      const int sblk = s0 + 32 * sb;
      if (sblk >= len) continue;
      if (causal && sblk + 31 < r0w) continue;  // queries before this group's first key
      // per streamed row: lse (score wave) or Delta (grad wave); register r of
      // this lane is streamed row  sblk + 16*(r/8) + 8*lh + r%8
      float vec_r[16];
#pragma unroll
      for (int g2 = 0; g2 < 2; ++g2)
#pragma unroll
        for (int q4 = 0; q4 < 2; ++q4) {
          const f32x4 v4 = *(lds_f4*)(uintptr_t)(lva + (32 * sb + 16 * g2 + 4 * q4) * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) vec_r[8 * g2 + 4 * q4 + e] = v4[e];
        }
      // first product: rows of Q (score) / dO (grad) against the resident operand
      f32x16 S = (f32x16){0};
      i32x4 f[kPrefetch];
#pragma unroll
      for (int st = 0; st < kPrefetch; ++st) f[st] = fr.rows(0, sb, st);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int st = 0; st < G::KSTEPS; ++st) {
        S = Elem<T>::mfma(f[st % kPrefetch], Xf[st], S);
        if (st + kPrefetch < G::KSTEPS) f[st % kPrefetch] = fr.rows(0, sb, st + kPrefetch);
        __builtin_amdgcn_sched_barrier(0);
      }
      i32x4 tf[2];
      tf[0] = fr.tr(0, 2 * sb, 0);
      tf[1] = fr.tr(0, 2 * sb, 1);
      uint32_t W[8];
      if (!grad) {
        // rows / columns that do not exist or lie above the diagonal give P = 0
        bool need_mask = sblk + 32 > len || !rows_full;
        if (causal) need_mask = need_mask || sblk < r0w + 31;
        if (need_mask) {
          const int ln = opaque_lane();
          const int rrow = r0w + (ln & 31);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int srow = sblk + 16 * (r >> 3) + 8 * (ln >> 5) + (r & 7);
            const bool ok = srow < len && rrow < len && (!causal || rrow <= srow);
            S[r] = ok ? S[r] : -INFINITY;
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
          W[i] = Elem<T>::pack2(fast_exp2(fmaf(S[2 * i], scale, -vec_r[2 * i])),
                                fast_exp2(fmaf(S[2 * i + 1], scale, -vec_r[2 * i + 1])));
        // P for the grad wave of this group (it reads it in the next tile step)
        *(lds_i32x4*)(uintptr_t)(pbv + sb * 2048) = (i32x4){(int)W[0], (int)W[1], (int)W[2], (int)W[3]};
        *(lds_i32x4*)(uintptr_t)(pbv + sb * 2048 + 1024) = (i32x4){(int)W[4], (int)W[5], (int)W[6], (int)W[7]};
      } else {
        const i32x4 p0 = *(lds_i32x4*)(uintptr_t)(pbv + sb * 2048);
        const i32x4 p1 = *(lds_i32x4*)(uintptr_t)(pbv + sb * 2048 + 1024);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t pk = (uint32_t)(i < 4 ? p0[i] : p1[i - 4]);
          float plo, phi;
          if (std::is_same<T, __bf16>::value) {
            plo = __builtin_bit_cast(float, pk << 16);
            phi = __builtin_bit_cast(float, pk & 0xffff0000u);
          } else {
            const f16x2 h2 = __builtin_bit_cast(f16x2, pk);
            plo = (float)h2[0];
            phi = (float)h2[1];
          }
          W[i] = Elem<T>::pack2(plo * (S[2 * i] - vec_r[2 * i]), phi * (S[2 * i + 1] - vec_r[2 * i + 1]));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      // accumulating product: dV^T += dO^T P  /  dK^T += Q^T dS
      __builtin_amdgcn_s_setprio(3);
#pragma unroll
      for (int i = 0; i < NACC; ++i) {
        const int kk = i / G::NDB, db = i % G::NDB;
        const i32x4 wf = {(int)W[4 * kk], (int)W[4 * kk + 1], (int)W[4 * kk + 2], (int)W[4 * kk + 3]};
        acc[db] = Elem<T>::mfma(tf[i & 1], wf, acc[db]);
        if (i + 2 < NACC) tf[i & 1] = fr.tr(0, 2 * sb + (i + 2) / G::NDB, (i + 2) % G::NDB);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // step i: the score waves work on tile i, the grad waves on tile i - 1, and
  // tile i + 1 is on its way into the stage that tile i - 2 has left
  if (n_stream > 0) {
    request();
    drip_all();
    advance();
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  __syncthreads();
  auto sync_step = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    __syncthreads();
  };
  // Tiles of a head that need masks: the first ones of a causal item (keys of
  // this group against queries at or before them) and a last, partial one.
  int n_pre = causal ? (32 * pr + 31 + TN - 1) / TN : 0;
  int n_post = (len % TN) != 0 ? 1 : 0;
  if (!rows_full) n_pre = nj;
  n_pre = min(n_pre, nj);
  n_post = min(n_post, nj - n_pre);
  int req_left = n_stream - 1;  // requests still to make (the first one is out)
  // Each loop below holds ONE kind of step: with the masked path and the
  // pipelined path in one loop body the accumulators were copied between two
  // register sets on every trip.
  auto run = [&](auto role_c) __attribute__((always_inline)) {
    constexpr bool gr = decltype(role_c)::value != 0;
    auto step = [&](auto fast_c) __attribute__((always_inline)) {
      const bool more = !kLoaders && req_left > 0;
      if (more) request();
      if (decltype(fast_c)::value)
        compute_fast(role_c);
      else
        compute_slow(role_c);
      rotate();
      if (more) advance();
      --req_left;
      sync_step();
    };
    if (gr) {  // step 0: nothing to work on yet
      if (!kLoaders && req_left > 0) {
        request();
        drip_all();
        advance();
      }
      --req_left;
      sync_step();
    }
    for (int g = 0; g < gqa; ++g) {
      for (int jj = 0; jj < n_pre; ++jj) step(ic<0>{});
      for (int jj = n_pre; jj < nj - n_post; ++jj) step(ic<1>{});
      for (int jj = nj - n_post; jj < nj; ++jj) step(ic<0>{});
    }
    if (!gr) {  // the grad waves' last tile
      if (wave == kTaker) take_next();
      sync_step();
    }
  };
  if (loader) {
    for (int i = 0; i <= n_stream; ++i) {
      if (i == n_stream && wave == kTaker) take_next();
      if (req_left > 0) {
        request();
        drip_all();
        advance();
      }
      --req_left;
      sync_step();
    }
  } else if (!grad) {
    run(ic<0>{});
  } else {
    run(ic<1>{});
  }

  // ---- epilogue: dV from the score waves, dK from the grad waves
  const float oscale = grad ? p.scale_nat : 1.f;
  T* outp = grad ? reinterpret_cast<T*>(p.dk) + bsel * p.dk_sb + start * p.dk_ss + hr * p.dk_sh
                 : reinterpret_cast<T*>(p.dv) + bsel * p.dv_sb + start * p.dv_ss + hr * p.dv_sh;
  const int64_t o_ss = grad ? p.dk_ss : p.dv_ss;
  const int ln = opaque_lane();
  unsigned char* stg = smem_bwd + wave * 32 * OROWB;
  if (loader) return;
#pragma unroll
  for (int db = 0; db < G::NDB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * db + 8 * g + 4 * (ln >> 5);
      i32x2 w;
      w[0] = (int)Elem<T>::pack2(acc[db][4 * g] * oscale, acc[db][4 * g + 1] * oscale);
      w[1] = (int)Elem<T>::pack2(acc[db][4 * g + 2] * oscale, acc[db][4 * g + 3] * oscale);
      *reinterpret_cast<i32x2*>(stg + (ln & 31) * OROWB + d * 2) = w;
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wavefront reads only what it has staged itself)
#pragma unroll
  for (int i = 0; i < (32 * G::NCH + 63) / 64; ++i) {
    const int idx = ln + 64 * i;
    const int row = idx / G::NCH, ch = idx % G::NCH;
    if (((32 * G::NCH) % 64 == 0 || idx < 32 * G::NCH) && r0w + row < len) {
      const i32x4 val = *reinterpret_cast<const i32x4*>(stg + row * OROWB + ch * 16);
      *reinterpret_cast<i32x4*>(outp + (int64_t)(r0w + row) * o_ss + ch * 8) = val;
    }
  }
}

// Persistent launch, as in the forward pass: at most one workgroup per CU, each
// walking the work items of its rounds (a fresh 512-thread workgroup with this
// much LDS starts several microseconds after its predecessor ends; order of the
// items: item_order.h).  The ids are kept in LDS behind the tiles (`LIST`): held
// in registers across the items they are spilled.
constexpr int kListBytes = 3 * kMaxRounds * 4;
template <int ROWS, uint32_t LIST, typename Item>
__device__ __forceinline__ void walk_items(const BwdParams& p, const int n_items, const int heads, const int heads_kv,
                                           const int n_rt, Item&& item) {
  typedef __attribute__((address_space(3))) int lds_int;
  lds_int* list = (lds_int*)(uintptr_t)((uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem_bwd) + LIST);
  const int grid = gridDim.x;
  if (threadIdx.x < kMaxRounds) {
    const ItemId ids = items_of_rounds<ROWS, false, kLevelWorth, true>(p.cu, p.batch, p.max_seqlen, n_rt, heads, heads_kv,
                                                       p.by_level, n_items, grid);
    list[threadIdx.x] = ids.t;
    list[kMaxRounds + threadIdx.x] = ids.b;
    list[2 * kMaxRounds + threadIdx.x] = ids.h;
  }
  __syncthreads();
  const int n_rounds = (n_items + grid - 1) / grid;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  for (int round = 0; round < n_rounds; ++round) {
    const int rt = __builtin_amdgcn_readfirstlane(list[round]);
    const int b = __builtin_amdgcn_readfirstlane(list[kMaxRounds + round]);
    const int h = __builtin_amdgcn_readfirstlane(list[2 * kMaxRounds + round]);
    item(b, h, rt, wave);
    if (round + 1 < n_rounds) __syncthreads();  // the next item's tiles overwrite the staging area
  }
}

constexpr uint32_t kDqLds = kBwdStages * (2 * 64 * 256 + 1024);
constexpr uint32_t kDkdvLds = kDqLds + 2 * 4 * 2 * 2048;  // tile ring + P exchange

// The units of work of the dK + dV launch, dealt out at run time.
//
// An item of 128 keys is worked on whole (eight wavefronts in their two roles, two
// to a SIMD), or as two halves of 64 keys (four wavefronts with a SIMD each, the
// other four send the loads).  What bounds a launch of few items is the chain of
// query tiles of its longest item: 1.23 us a tile, 0.80 in a half; with every CU
// at work a tile takes 1.9 to 2.0 us (matrix pipes at the power limit) and the two
// halves 1.18 times as long as the whole.  So the longest items are halved, as many
// as shorten the launch, and a workgroup takes the next unit, longest first, when
// it is done (in the fixed order two rounds of whole items left the busiest
// workgroup with 1.3 times the mean).  Rows meet their tiles in the same order
// either way: the results are the same bits.  dK + dV, fixed whole items -> this,
// head_dim 128: 1000 tokens, 4 kv-heads of 4 94 -> 68 us; 2048, 2 of 8 315 -> 216;
// 4096, 8 of 4 352 -> 292; 16384, 2 of 4 1362 -> 1137; five of 517 to 3400, 8 of 4
// 384 -> 332; 8192, 8 of 4 (two even rounds, none halved) 967 -> 954.
// Cost model, in hundredths of a microsecond, of n tiles:
constexpr int kFullTile = 175, kHalfTile = 100, kUnitFixed = 700;
static_assert(kFullTile * 4 == kHalfTile * 7, "key_units_before() orders the units by 4 : 7");
constexpr int kMaxLevels = 512;      // tiles of 128 keys of the longest sequence
static_assert(kMaxLevels < 1024, "plan_key_units() packs a level into ten bits");
// Items per workgroup from which the fixed order is even enough (one sequence of 8192, 16 heads of their own, two
// rounds: 128 us in either) and keeps neighbours together in an L2.
constexpr int kDealtRounds = 4;
// In one round: tiles of the longest chain, and how much of it has to be idle (plan_key_units()).
constexpr int kHalvedTiles = 7, kHalvedIdle = 160;

// In LDS, behind the tiles and the P exchange.
struct KeyPlan {
  int list[3 * kMaxRounds];          // fixed order: items of this workgroup
  int at_or_above[kMaxLevels + 1];  // (sequence, tile) pairs on level t and above; level: tiles counted from the sequence's end
  int weight[kMaxLevels + 1];       // the same, pairs weighted with their level + 1
  int tiles[kLevelMaxBatch];
  int top;                           // levels, rounded up to a wavefront's lanes; at_or_above[top] = 0
  int split_from, dealt;             // first of the levels that are halved; whether units are dealt at run time
  int next[2];                       // unit of the next round, by parity
};

typedef __attribute__((address_space(3))) KeyPlan LdsKeyPlan;

// Units run from the longest to the shortest: pairs that stand before level t's.
__device__ __forceinline__ int key_units_before(const LdsKeyPlan& k, const int t) {
  const int T = k.split_from;
  if (t >= T) {   // halves of level t: behind the whole items that cost more, 7 (t' + 1) > 4 (t + 1)
    const int first = min(4 * (t + 1) / 7, T);
    return 2 * k.at_or_above[t + 1] + k.at_or_above[first] - k.at_or_above[T];
  }
  const int first = max((7 * (t + 1) + 3) / 4 - 1, T);
  return k.at_or_above[t + 1] - k.at_or_above[T] + 2 * k.at_or_above[min(first, k.top)];
}

// By one wavefront: whether the units are dealt out, and then the levels and which of them are halved.  The
// estimate that is minimised is the longer of the longest unit and the mean load plus a quarter of a mean unit.  It
// is no schedule: against every level, or every twelfth of them, as the first that is halved, dQ with dK + dV took
// within 3 % of the best for ten of thirteen sizes, and 3.3 (six of 1500, 4 kv-heads of 8), 4.6 (4096, 8 of 4: 483 us,
// all halved 461) and 5.7 % more (40 of 700, one of 8) for the others; unhalved 4096 took 537.
//
// What this costs is 2.3 us of the launch whatever the number of sequences (looked through one after another they
// cost another 0.17 us each: 64 of 60 tokens, 2 heads, dK + dV 24.0 -> 12.9).  Where every whole item has a workgroup
// to itself only the halves can pay for it, and only where workgroups are idle for much of the longest item: from
// a chain of seven tiles on, where the mean load is 1.6 us less than six tenths of the longest item.  With dQ, whole
// items -> this: chains of four tiles 30.2 -> 30.4 us, of eight 40.2 -> 38.5, of sixteen 58.2 -> 53.0; with every CU at
// work, two of 1024, 16 heads (mean 0.65) 62.7 -> 64.7; eight of 77 to 512, 8 heads (0.53, a chain of eight)
// 43.8 -> 45.8; 40 of 700, one kv-head of 8 (0.56, of 96) 254.8 -> 253.8; one of 4096, 8 of 4 (0.52) 540 -> 483.
__device__ __forceinline__ void plan_key_units(LdsKeyPlan& k, const BwdParams& p, const int workers) {
  const int lane = threadIdx.x & 63;
  int tokens = 0;
  if (lane < p.batch) tokens = max(p.cu ? min(p.cu[lane + 1] - p.cu[lane], p.max_seqlen) : p.max_seqlen, 0);
  const int tiles = (tokens + 127) / 128;
  int most = tokens, all = tiles, all_w = tiles * (tiles + 1) / 2;   // tokens of the longest; pairs, and their weights
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    most = max(most, __shfl_xor(most, m, 64));
    all += __shfl_xor(all, m, 64);
    all_w += __shfl_xor(all_w, m, 64);
  }
  most = __builtin_amdgcn_readfirstlane(most);
  all = __builtin_amdgcn_readfirstlane(all);
  all_w = __builtin_amdgcn_readfirstlane(all_w);
  const int levels = (most + 127) / 128;   // of the longest sequence
  const float unit = 2.f * (p.hq / p.hkv);   // tiles of 64 queries of a level-0 item
  const bool one_round = all * p.hkv <= workers;
  const float whole_item = kFullTile * unit * levels + kUnitFixed;   // the longest
  bool dealt = all * p.hkv < kDealtRounds * workers;
  if (!p.causal) dealt = 2 * all * p.hkv <= workers;   // (every item of a sequence is as long as the next: all of them are halved or none)
  if (one_round) {
    const float mean = (float)p.hkv * (kFullTile * unit * all_w + kUnitFixed * all) / (float)workers;
    dealt = dealt && unit * levels >= kHalvedTiles && most > 64;   // (up to 64 tokens the second half has no keys)
    if (p.causal) dealt = dealt && mean + kHalvedIdle <= 0.6f * whole_item;
  }
  if (lane == 0) k.dealt = dealt;
  if (!dealt) return;

  // from the last level down: sequences that reach a level, and the sums over it and the levels above
  const int top = (levels + 63) / 64 * 64;
  for (int t = lane; t <= top; t += 64) k.weight[t] = 0;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // lanes read and add to what other lanes have written
  __hip_atomic_fetch_add(&k.weight[tiles], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  k.tiles[lane] = tiles;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  auto from_here_on = [&](int v) __attribute__((always_inline)) -> int {   // sum over this lane and those behind it
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_down(v, d, 64);
      v += lane + d < 64 ? o : 0;
    }
    return v;
  };
  int reach = __builtin_amdgcn_readfirstlane(k.weight[top]), above = 0, above_w = 0;
  if (lane == 0) k.at_or_above[top] = k.weight[top] = 0;
  for (int base = top - 64; base >= 0; base -= 64) {
    const int t = base + lane, ends = k.weight[t];
    const int at_least = reach + from_here_on(ends);        // sequences of t tiles and more
    const int n = above + from_here_on(at_least - ends), w = above_w + from_here_on((t + 1) * (at_least - ends));
    k.at_or_above[t] = n;
    k.weight[t] = w;
    reach = __builtin_amdgcn_readfirstlane(at_least);
    above = __builtin_amdgcn_readfirstlane(n);
    above_w = __builtin_amdgcn_readfirstlane(w);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  int T = 0;                         // halved from here on
  if (p.causal) {
    // (the estimate and the level in one word, the larger level among equals: one reduction)
    uint32_t best = ~0u;
    for (int base = 0; base <= levels; base += 64) {
      const int t = base + lane;     // candidate
      if (t <= levels) {
        const float a = (float)k.at_or_above[t], w = (float)k.weight[t];
        const float whole = (float)above - a, units = whole + 2.f * a;
        const float total = (float)p.hkv * (2.f * (kHalfTile * unit * w + kUnitFixed * a) +
                                            kFullTile * unit * ((float)above_w - w) + kUnitFixed * whole);
        float longest = t > 0 ? kFullTile * unit * t + kUnitFixed : 0.f;
        if (t < levels) longest = fmaxf(longest, kHalfTile * unit * levels + kUnitFixed);
        float est = total / (float)workers;
        if (units * (float)p.hkv > (float)workers) est += 0.25f * total / (units * (float)p.hkv);
        est = fmaxf(est, longest);
        best = min(best, (__builtin_bit_cast(uint32_t, est) & ~1023u) | (uint32_t)(1023 - t));
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) best = min(best, (uint32_t)__shfl_xor((int)best, m, 64));
    T = __builtin_amdgcn_readfirstlane(1023 - (int)(best & 1023u));
  }
  if (lane == 0) {
    k.top = top;
    k.split_from = T;
  }
}

// Unit u: sequence, kv-head, tile of 128 keys (-1: behind the last unit) and half (-1: a whole item).
struct KeyUnit {
  int b, kvh, rt, half;
};
__device__ __forceinline__ KeyUnit key_unit(const LdsKeyPlan& k, const int hkv, const int u) {
  KeyUnit it = {0, 0, -1, -1};
  const int pair = __builtin_amdgcn_readfirstlane((int)((uint32_t)u / (uint32_t)hkv));
  const int T = __builtin_amdgcn_readfirstlane(k.split_from), top = __builtin_amdgcn_readfirstlane(k.top);
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < top; base += 64) {
    const int t = base + lane;
    const int n = pair - key_units_before(k, t);
    const bool here = n >= 0 && n < (t >= T ? 2 : 1) * (k.at_or_above[t] - k.at_or_above[t + 1]);
    const uint64_t hit = __builtin_amdgcn_ballot_w64(here);
    if (hit) {
      const int at = __builtin_ctzll(hit);
      const int level = base + at;
      int seq = __builtin_amdgcn_readlane(n, at);
      if (level >= T) {
        it.half = seq & 1;
        seq >>= 1;
      }
      const int all = k.tiles[lane];
      const uint64_t live = __builtin_amdgcn_ballot_w64(all > level);
      const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0));
      it.b = __builtin_ctzll(__builtin_amdgcn_ballot_w64(all > level && rank == seq));
      it.kvh = u - pair * hkv;
      it.rt = __builtin_amdgcn_readlane(all, it.b) - 1 - level;
      break;
    }
  }
  return it;
}

// The kernel's parameters as its argument segment holds them, asked for again by
// every item.  Kept across the items they are spilled to vector registers, lane by
// lane (two forms of the item in one kernel: 168 of them, 73 this way), and come back
// by several hundred v_readlane at every item boundary: dK + dV in the fixed order,
// 40 sequences of 700 tokens, 8 heads of their own, 153.7 -> 145.6 us; eight of 512
// 22.0 -> 20.8; one item 11.4 -> 9.8.
__device__ __forceinline__ const BwdParams& fresh_params() {
  typedef __attribute__((address_space(4))) const BwdParams c_params;
  c_params* a = (c_params*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return *(const BwdParams*)a;
}

// Eight queues (workgroup ids go round-robin to the 8 XCDs): with the kv-head running
// fastest an XCD keeps to its kv-heads, whose queries and gradients its L2 then holds,
// whenever the head counts are multiples of eight.
template <typename T, int D>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
bwd_dkdv_kernel(const BwdParams p, const int n_items, const int n_rt, const int resident) {
  LdsKeyPlan& k = *(LdsKeyPlan*)(uintptr_t)((uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem_bwd) + kDkdvLds);
  const int grid = gridDim.x;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // Units are dealt to the workgroups that run at once.  Where the ids of a ragged batch make several generations of
  // them (persistent_grid()), the others would come to units that were meant to be first when the queues are empty.
  const int workers = min(grid, resident);
  const int queues = (workers & 7) == 0 ? 8 : 1;
  const int queue = queues == 8 ? blockIdx.x & 7 : 0;
  const int first = queues == 8 ? (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  bool dealt = false;
  if (p.queue) {
    if (wave == 0) plan_key_units(k, p, workers);
    __syncthreads();
    dealt = __builtin_amdgcn_readfirstlane(k.dealt);
    if (dealt && (int)blockIdx.x >= workers) return;
  }
  if (!dealt) {
    if (wave == 0) {
      const ItemId ids = items_of_rounds<128, true>(p.cu, p.batch, p.max_seqlen, n_rt, p.hkv, p.hkv, p.by_level, n_items, grid);
      k.list[threadIdx.x] = ids.t;
      k.list[kMaxRounds + threadIdx.x] = ids.b;
      k.list[2 * kMaxRounds + threadIdx.x] = ids.h;
    }
    __syncthreads();
  }
  const int n_rounds = (n_items + grid - 1) / grid;
  int unit = first * queues + queue;
  for (int round = 0;; ++round) {
    int b, h, rt, half = -1;
    if (dealt) {
      if (round > 0) unit = __builtin_amdgcn_readfirstlane(k.next[round & 1]);
      const KeyUnit it = key_unit(k, p.hkv, unit);   // (every wavefront by itself)
      if (it.rt < 0) break;
      b = it.b;
      h = it.kvh;
      rt = it.rt;
      half = it.half;
    } else {
      if (round == n_rounds) break;
      rt = __builtin_amdgcn_readfirstlane(k.list[round]);
      b = __builtin_amdgcn_readfirstlane(k.list[kMaxRounds + round]);
      h = __builtin_amdgcn_readfirstlane(k.list[2 * kMaxRounds + round]);
      if (rt < 0) continue;   // (a round without an item)
    }
    auto take_next = [&]() __attribute__((always_inline)) {
      if (dealt && (threadIdx.x & 63) == 0) {
        const int n = __hip_atomic_fetch_add(p.queue + 16 * queue, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        k.next[(round + 1) & 1] = (n + workers / queues) * queues + queue;
      }
    };
    if (half >= 0)
      bwd_dkdv_item<T, D, 2>(fresh_params(), b, h, 2 * rt + half, wave, take_next);
    else
      bwd_dkdv_item<T, D, 4>(fresh_params(), b, h, rt, wave, take_next);
    __syncthreads();  // the next item's tiles overwrite the staging area
  }
}

template <typename T, int D, int NW>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
bwd_dq_kernel(const BwdParams p, const int n_items, const int n_rt) {
  if (blockIdx.x == 0 && threadIdx.x < 8 && p.queue) p.queue[16 * threadIdx.x] = 0;  // for the dK + dV kernel, which runs after this one
  walk_items<32 * NW, kDqLds>(p, n_items, p.hq, p.hkv, n_rt, [&](int b, int hr, int rt, int wave) __attribute__((always_inline)) {
    bwd_dq_item<T, D, NW>(p, b, hr, rt, wave);
  });
}

template <typename T, int D, int NW>
int launch_dq(const BwdParams& p0, hipStream_t s) {
  BwdParams p = p0;
  constexpr size_t lds = kDqLds + kListBytes;
  static_assert(kDqLds >= 8 * 32 * (D * 2 + 16), "epilogue staging must fit the tile ring");
  auto kern = bwd_dq_kernel<T, D, NW>;
  static LdsLimitOnce lds_once;
  if (const int e = raise_lds_limit(lds_once, reinterpret_cast<const void*>(kern), (int)lds)) return e;
  const int n_rt = (p.max_seqlen + 32 * NW - 1) / (32 * NW);
  const long long items = (long long)n_rt * p.hq * p.batch;
  const long long grid = persistent_grid(items, device_cu_count());  // one workgroup per CU is resident (LDS)
  p.by_level = number_by_level(p.cu, p.causal, p.batch, items, grid);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(512), lds, s, p, (int)items, n_rt);
  return (int)hipGetLastError();
}

template <typename T, int D>
int launch_dkdv(const BwdParams& p0, hipStream_t s) {
  BwdParams p = p0;
  constexpr size_t lds = kDkdvLds + sizeof(KeyPlan);
  static_assert(kDqLds >= 8 * 32 * (D * 2 + 16), "epilogue staging must fit");
  auto kern = bwd_dkdv_kernel<T, D>;
  static LdsLimitOnce lds_once;
  if (const int e = raise_lds_limit(lds_once, reinterpret_cast<const void*>(kern), (int)lds)) return e;
  const int n_rt = (p.max_seqlen + 127) / 128;
  const long long items = (long long)n_rt * p.hkv * p.batch;
  const int cus = device_cu_count();
  long long grid = persistent_grid(items, cus);  // one workgroup per CU is resident (LDS)
  if (p.batch > kLevelMaxBatch || n_rt > kMaxLevels || (!p.cu && items >= kDealtRounds * (long long)cus)) p.queue = nullptr;
  if (items <= cus && (2 * (p.hq / p.hkv) * n_rt < kHalvedTiles || p.max_seqlen <= 64)) p.queue = nullptr;   // (as plan_key_units() would say)
  if (p.queue && items <= cus) grid = std::min((2 * items + 7) / 8 * 8, (long long)cus);  // each half a workgroup of its own
  p.by_level = number_by_level(p.cu, p.causal, p.batch, items, grid);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(512), lds, s, p, (int)items, n_rt, cus);
  return (int)hipGetLastError();
}

template <typename T, int D>
int launch_all(const BwdParams& p, hipStream_t s) {
  // dQ first: it also writes Delta, which the dK + dV kernel reads
  const bool short_items = bwd_dq_short_items(p.max_seqlen, p.batch, p.hq, p.causal, device_cu_count());
  if (const int rc = short_items ? launch_dq<T, D, 4>(p, s) : launch_dq<T, D, 8>(p, s)) return rc;
  return launch_dkdv<T, D>(p, s);
}

}  // namespace

// dQ's items of 128 queries, a wavefront to a SIMD, in place of 256, where a launch has few of them: a tile of 64
// keys then takes 1.5 instead of 2.1 us, and the longest chain bounds the launch.  In one round of workgroups they
// are never slower from 129 tokens on (1000 tokens, 16 heads 40 -> 29 us; 4096, 8 heads 135 -> 108); up to 128 both
// forms have the same items, which eight wavefronts load sooner than four (128 tokens, 16 to 256 items, 1.3 to 1.8
// us).  In the two rounds of a causal call, the second of short items, the gain of 0.53 us a tile of the longest
// chain has to pay for the second round's boundary, 3.5 us where both are full.  2048, 32 heads 82 -> 66; 4096, 16
// heads 135 -> 108; with dK + dV three of 1354, 8 heads 91 -> 79, but 64 of 256, 4 heads 59 -> 69, 24 of 384, 4 heads
// 48 -> 54.  Of 211 measured launches of two rounds this takes 106, 1.10 times as fast in the mean with dK + dV,
// three of them 1.5 to 2 % slower; 25 of those it leaves would gain 2 to 17 %.  Beyond two rounds: 4096, 32 heads (four)
// 191 -> 208.
bool bwd_dq_short_items(int max_seqlen, int batch, int heads_q, bool causal, int num_cus) {
  if (num_cus <= 0) num_cus = 256;
  const long long items = (long long)((max_seqlen + 127) / 128) * batch * heads_q;
  if (max_seqlen <= 128 || items > (causal ? 2 : 1) * (long long)num_cus) return false;
  return items <= num_cus || 53LL * ((max_seqlen + 63) / 64) >= 120 + 350 * items / num_cus;
}

int launch_attn_bwd(const BwdParams& p, int dtype, int head_dim, hipStream_t s) {
  if (dtype == 0) {
    if (head_dim == 64) return launch_all<__bf16, 64>(p, s);
    if (head_dim == 96) return launch_all<__bf16, 96>(p, s);
    if (head_dim == 128) return launch_all<__bf16, 128>(p, s);
  } else {
    if (head_dim == 64) return launch_all<_Float16, 64>(p, s);
    if (head_dim == 96) return launch_all<_Float16, 96>(p, s);
    if (head_dim == 128) return launch_all<_Float16, 128>(p, s);
  }
  return (int)hipErrorInvalidValue;
}

}  // namespace mi
