// Fused linear + cross-entropy for gfx950.
//
// Replaces cross_entropy_fused_fwd_lse_kernel and cross_entropy_fused_bwd_kernel
// of cross_entropy_triton/cross_entropy.py:43-183, :185-266 and the host
// combine in CrossEntropyFusedFunction.forward (:337-339):
//   logits[t, n] = sum_d x[t, d] w[n, d]        written to memory only by the keeping form
//   lse[t]  = log sum_n exp(logits[t, n])
//   loss[t] = lse[t] - logits[t, y[t]]
//   dlogits[t, n] = do[t] (exp(logits[t, n] - lse[t]) - [n == y[t]])   (:255-265)
//
// Forward (MFMA-bound).  A workgroup of 8 wavefronts owns 256 tokens and a
// range of 256-row vocabulary tiles; per tile it runs the D loop of
// logits^T = W X^T in 64-element steps (D is a multiple of 128): both 256 x 64 slabs are fetched with
// direct-to-LDS loads into a two-stage ring (rows of 128 bytes, 16-byte chunk c
// of row r stored in slot c ^ ((r >> 1) & 7), which makes the 16-byte fragment
// reads of 16 neighbouring rows conflict-free), one barrier per step.  A
// wavefront accumulates a 128 (vocabulary) x 64 (tokens) block in eight 32x32
// MFMA accumulators.  W is the A operand, so the 16 values a lane holds per
// accumulator belong to ONE token: the per-token maximum and exponential sum
// of a tile are in-lane arithmetic plus one exchange between the lane halves.
// The running (max, sum) pair and the target logit of every token stay in
// registers across the tiles; the two wavefronts that share tokens meet in LDS
// at the end and the workgroup writes one partial (lse, target logit) per token
// and vocabulary range.  A second kernel merges the ranges.
//
// Workgroup ids are dealt round-robin to the 8 XCDs.  Token tiles are taken in
// panels of up to eight, nearly equal in width; within a panel the tiles of a
// vocabulary range follow each other, and every XCD is given an eighth of this
// order: the 32 workgroups that run together on it form a block of tiles x ranges
// and share their slabs in its L2, and no XCD has more of them than another.
// (In whole blocks of 8 tiles x 4 ranges, a count of tiles that is no multiple of
// eight left some XCDs with two rounds of workgroups and others with half a one:
// 2876 tokens x 2560 x 64000 1769 -> 988 us, 6646 x 1024 x 64000 1893 -> 1260,
// 1292 x 1024 x 64000 364 -> 220, keeping the logits; 8192 x 4096 x 128256 as before.)
#include <type_traits>

#include "kernels.h"
#include "tile_core.h"

namespace mi {
namespace {

constexpr int waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

extern __shared__ __attribute__((aligned(1024))) unsigned char xsmem[];

constexpr int kXTileT = 256;   // tokens per workgroup
constexpr int kXTileN = 256;   // vocabulary rows per tile
constexpr int kXStepK = 64;    // elements of D per step
constexpr int kXSlabB = 256 * kXStepK * 2;  // one slab: 32 KiB
constexpr int kXLdsBytes = 4 * kXSlabB;     // W stage 0, W stage 1, X stage 0, X stage 1
typedef float xf32x4 __attribute__((ext_vector_type(4)));
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Kept logits: a unit is the 32 tokens x 128 vocabulary rows that one wavefront
// holds in four accumulators, 16 x 64 pieces of four floats in register order:
// piece (4 rb + g4, lane) holds the logits of token lane % 32 and vocabulary
// rows 32 rb + 8 g4 + 4 (lane / 32) + 0..3.  Units of a 256 x 256 tile follow
// each other as [wave][cb].  Returns the offset of a unit in floats.
constexpr int kXUnit = 32 * 128;
__device__ __forceinline__ int64_t kept_unit(int t_tile, int n_tile, int tiles_n, int wave, int cb) {
  return ((((int64_t)t_tile * tiles_n + n_tile) * 8 + wave) * 2 + cb) * kXUnit;
}

// GRAD = false: forward (partial lse and target logit per token and range).
// GRAD = true: the same product with the epilogue of the backward pass: every
// tile of logits is turned into dloss[t] (exp(logit - lse[t]) - [n == y[t]])
// straight from the fp32 accumulators and written to dlogits[t, n] in the
// storage dtype (the reference rounds the logits to the storage dtype first,
// cross_entropy.py:374,255-265, which costs accuracy when logits are large).
// KEEP (forward only): every tile's fp32 accumulators are also written out as
// they lie in the registers, one 1-KiB row of 64 lanes x 16 bytes per store
// (kept_unit above), for xent_kept_dlogits_kernel: the backward then reads 4
// bytes per logit instead of running the product again.  The stores of a tile
// drain before its next step's loads count as landed, and all workgroups reach
// the end of a tile together, so they cost what 4 bytes per logit cost at 5 to
// 6 TB/s: 6.49 -> 7.68 ms at 8192 x 4096 x 128256 (rows of 32 bytes per token
// would be row-major, and far slower: short pieces of many rows per store).  Without the non-temporal hint
// 7.74 ms there, but 1.40 instead of 1.15 ms at 4096 x 1024 x 128256, and at
// dim 512 it costs three times as much.
template <typename T, bool KEEP, bool GRAD>
__global__ void __launch_bounds__(512) xent_gemm_kernel(const XentParams p) {
  typedef __attribute__((address_space(3))) const i32x4 lds_i32x4;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;
  const int wv = wave >> 2;  // vocabulary half of the tile
  const int wt = wave & 3;   // 64-token quarter of the workgroup's tokens

  // ---- workgroup id -> (token tile, vocabulary range)
  int t_tile, split;
  {
    const int per_xcd = gridDim.x >> 3;
    const int at = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int panels = (p.tiles_t + 7) >> 3, base = p.tiles_t / panels, wider = p.tiles_t % panels;
    const int in_wider = wider * (base + 1) * p.n_split;   // workgroups of the panels that are a tile wider
    const bool w = at < in_wider;
    const int width = w ? base + 1 : base, rest = w ? at : at - in_wider;
    const int panel = rest / (width * p.n_split), in = rest % (width * p.n_split);
    t_tile = (w ? 0 : wider * (base + 1)) + panel * width + in % width;
    split = in / width;
    if (t_tile >= p.tiles_t) return;
  }
  const int t0 = t_tile * kXTileT;
  // vocabulary tiles of this range
  const int nt_all = (p.N + kXTileN - 1) / kXTileN;
  const int nt_base = nt_all / p.n_split, nt_rem = nt_all % p.n_split;
  const int tile_first = split * nt_base + min(split, nt_rem);
  const int tile_cnt = nt_base + (split < nt_rem ? 1 : 0);
  const int nk = p.D / kXStepK;
  const int total = tile_cnt * nk;

  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)xsmem);
  auto uniform64 = [](uint64_t v) __attribute__((always_inline)) -> uint64_t {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
  };
  const uint64_t w_base = uniform64((uint64_t)(uintptr_t)p.w);
  const uint64_t x_base = uniform64((uint64_t)(uintptr_t)p.x);
  const uint32_t w_pitch = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p.w_st * 2));
  const uint32_t x_pitch = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p.x_st * 2));

  // ---- loads: wavefront `wave` fills rows [32 wave, 32 wave + 32) of both
  // slabs with four instructions each; instruction q covers 8 rows, lane i
  // fills slot i % 8 of row 8 q + i / 8.
  const int ld_row = lane >> 3;   // row inside the instruction's 8 rows
  const int ld_slot = lane & 7;
  uint32_t xoff[4], woff[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 32 * wave + 8 * q + ld_row;
    const int c = ld_slot ^ ((r >> 1) & 7);
    const int tok = min(t0 + r, p.T - 1);  // rows past the end re-read the last token
    xoff[q] = (uint32_t)(tok - t0) * x_pitch + c * 16;
  }
  auto set_woff = [&](int n0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = 32 * wave + 8 * q + ld_row;
      const int c = ld_slot ^ ((r >> 1) & 7);
      const int rr = min(r, p.N - 1 - n0);  // rows past the vocabulary re-read its last row
      woff[q] = (uint32_t)rr * w_pitch + c * 16;
    }
  };
  int iss_k = 0, iss_n0 = tile_first * kXTileN;
  set_woff(iss_n0);
  // The eight loads of a step (four of W, four of X per wavefront) are sent one
  // at a time behind the first MFMAs of the step before: sent together right
  // after the barrier, 64 KiB of requests queue up in the memory pipeline and a
  // wavefront reaches its MFMAs only when its own requests have been accepted.
  // arm() fixes the wave-uniform slab addresses, drip(k) sends load k, next()
  // moves on; a load whose mask is 0 is a no-op (all 64 lanes are active and
  // control flow is wave-uniform here, so exec is restored to all ones).
  uint64_t drip_on = 0, drip_wb = 0, drip_xb = 0;
  uint32_t drip_sw = 0, drip_sx = 0;
  auto arm = [&](int stage, bool on) __attribute__((always_inline)) {
    drip_on = uniform64(on ? ~0ull : 0ull);
    drip_wb = uniform64(w_base + (uint64_t)iss_n0 * w_pitch + (uint32_t)(iss_k * kXStepK * 2));
    drip_xb = uniform64(x_base + (uint64_t)t0 * x_pitch + (uint32_t)(iss_k * kXStepK * 2));
    drip_sw = lds0 + stage * kXSlabB + wave * 4096;
    drip_sx = lds0 + (2 + stage) * kXSlabB + wave * 4096;
  };
  auto drip = [&](int k) __attribute__((always_inline)) {
    const int q = k >> 1;
    const uint64_t base = (k & 1) ? drip_xb : drip_wb;
    const uint32_t off = (k & 1) ? xoff[q] : woff[q];
    const uint32_t slab = (uint32_t)__builtin_amdgcn_readfirstlane(((k & 1) ? drip_sx : drip_sw) + q * 1024);
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                 :
                 : "s"(drip_on), "v"(off), "s"(base), "s"(slab)
                 : "memory");
  };
  auto next = [&]() __attribute__((always_inline)) {
    if (++iss_k == nk) {
      iss_k = 0;
      iss_n0 += kXTileN;
      if (iss_n0 < p.N) set_woff(iss_n0);
    }
  };

  // ---- fragment reads: row lq of a 32-row block, chunk 2 s + lh
  uint32_t a_addr[4], b_addr[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const uint32_t lo = lq * 128 + (((2 * s + lh) ^ ((lq >> 1) & 7)) << 4);
    a_addr[s] = lds0 + wv * 16384 + lo;
    b_addr[s] = lds0 + 2 * kXSlabB + wt * 8192 + lo;
    asm volatile("" : "+v"(a_addr[s]), "+v"(b_addr[s]));
  }

  f32x16 acc[4][2];
#pragma unroll
  for (int rb = 0; rb < 4; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) acc[rb][cb] = (f32x16){0};

  // One step = four 16-element sub-steps of 8 MFMAs.  The fragments of sub-step
  // s + 1 are read while the MFMAs of sub-step s issue; sched_barrier(0) pins
  // the slices (two reads, two MFMAs) so that the reads stay spread out.
  i32x4 af[2][4], bf[2][2];
  auto read_a = [&](int stage, int s, int rb) __attribute__((always_inline)) {
    af[s & 1][rb] = *(lds_i32x4*)(uintptr_t)(a_addr[s] + stage * kXSlabB + rb * 4096);
  };
  auto read_b = [&](int stage, int s, int cb) __attribute__((always_inline)) {
    bf[s & 1][cb] = *(lds_i32x4*)(uintptr_t)(b_addr[s] + stage * kXSlabB + cb * 4096);
  };
  auto read_first = [&](int stage) __attribute__((always_inline)) {
    read_b(stage, 0, 0);
    read_b(stage, 0, 1);
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) read_a(stage, 0, rb);
  };
  // sub-step s on the fragments in registers, those of sub-step sn of `stage` read along the way (sn < 0: none);
  // first_load >= 0: every slice carries one load of the step that drip() is armed for
  auto sub_step = [&](int s, int stage, int sn, int first_load) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      if (sn >= 0) {
        if (rb == 0) {
          read_b(stage, sn, 0);
          read_b(stage, sn, 1);
        } else if (rb == 1) {
          read_a(stage, sn, 0);
          read_a(stage, sn, 1);
        } else if (rb == 2) {
          read_a(stage, sn, 2);
          read_a(stage, sn, 3);
        }
      }
      acc[rb][0] = Elem<T>::mfma(af[s & 1][rb], bf[s & 1][0], acc[rb][0]);
      acc[rb][1] = Elem<T>::mfma(af[s & 1][rb], bf[s & 1][1], acc[rb][1]);
      if (first_load >= 0) drip(first_load + rb);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- per-token state: tokens t0 + 64 wt + 32 cb + lq
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f}, tgt[2] = {0.f, 0.f};
  long long yv[2] = {0, 0};
  if (!GRAD) {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const int tok = min(t0 + 64 * wt + 32 * cb + lq, p.T - 1);
      yv[cb] = p.y_is_i64 ? reinterpret_cast<const long long*>(p.y)[tok]
                          : (long long)reinterpret_cast<const int*>(p.y)[tok];
    }
  }

  // accumulators hold logits of vocabulary rows n0 + 128 wv + 32 rb + 8 (i / 4) + 4 lh + i % 4
  auto finish_tile = [&](int n0) __attribute__((always_inline)) {
    const int nw = n0 + 128 * wv;
    if (GRAD) {
      // The tile is transposed through LDS so that it leaves in 16-byte pieces
      // of whole 256-byte rows.  The slabs of the step just finished (stage 1:
      // a tile ends on an odd step) are free until the next step refills them;
      // each wavefront stages 32 tokens x 128 rows at a time in its own 8 KiB.
      __syncthreads();  // every wavefront is done reading stage 1
      typedef __attribute__((address_space(3))) i32x2 lds_w_i32x2;
      // (opaque copies: the row addresses below must be formed here, not hoisted
      // out of the main loop into registers that the loop cannot spare)
      int t0v = t0, ldv = (int)p.dl_ld;
      asm volatile("" : "+s"(t0v), "+s"(ldv));
      // per-token inputs are fetched here, once per tile, rather than kept in
      // registers through the main loop
      float lse2[2], gl[2];
      long long yt[2];
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        const int tok = min(t0v + 64 * wt + 32 * cb + lq, p.T - 1);
        lse2[cb] = p.lse[tok] * kLog2e;
        gl[cb] = p.dloss[tok];
        yt[cb] = p.y_is_i64 ? reinterpret_cast<const long long*>(p.y)[tok]
                            : (long long)reinterpret_cast<const int*>(p.y)[tok];
      }
      const uint32_t stg = lds0 + (wave < 4 ? 1 : 3) * kXSlabB + (wave & 3) * 8192;
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        // position of the label inside this wavefront's 128 rows, -1 if elsewhere
        const long long rel64 = yt[cb] - nw;
        const int rel = rel64 >= 0 && rel64 < 128 ? (int)rel64 : -1;
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) {
            const int nl = 32 * rb + 8 * g4 + 4 * lh;  // first of this lane's 4 consecutive rows
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float pr = exp2f(acc[rb][cb][4 * g4 + j] * kLog2e - lse2[cb]);
              v[j] = gl[cb] * (pr - (rel == nl + j ? 1.f : 0.f));
            }
            const i32x2 pk = {(int)Elem<T>::pack2(v[0], v[1]), (int)Elem<T>::pack2(v[2], v[3])};
            // 8-byte slot nl / 4 of token row lq, slot pairs swizzled by the row
            const uint32_t slot = (uint32_t)(nl >> 2) ^ ((lq & 15) << 1);
            *(lds_w_i32x2*)(uintptr_t)(stg + lq * 256 + slot * 8) = pk;
            __builtin_amdgcn_sched_barrier(0);  // keeps the register need of this rare block small
          }
        // read back: 16 lanes per row
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int r = 4 * i + (lane >> 4), ch = lane & 15;  // token row, 16-byte chunk (8 vocabulary rows)
          const uint32_t slot = (uint32_t)(2 * ch) ^ ((r & 15) << 1);
          const i32x4 val = *(lds_i32x4*)(uintptr_t)(stg + r * 256 + slot * 8);
          const int tok = t0v + 64 * wt + 32 * cb + r;
          const int n = nw + 8 * ch;
          if (tok < p.T && n < p.N) {
            T* dst = reinterpret_cast<T*>(p.dlogits) + (int64_t)tok * ldv + n;
            if (p.dl_vec && n + 8 <= p.N) {
              __builtin_nontemporal_store(val, reinterpret_cast<i32x4*>(dst));
            } else {
              const T* e = reinterpret_cast<const T*>(&val);
#pragma unroll
              for (int j = 0; j < 8; ++j)
                if (n + j < p.N) dst[j] = e[j];
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else if (nw < p.N) {
      if (KEEP) {
        // rows past the vocabulary are written too (their logits are never used), tokens past the end are not
        // (the lane's offset and the addresses are formed here, not carried through the main loop)
        const int nt = (p.N + kXTileN - 1) / kXTileN;
        int t0v = t0;
        uint32_t off = (uint32_t)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)) * 16;
        asm volatile("" : "+s"(t0v), "+v"(off));
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
          unsigned char* base = reinterpret_cast<unsigned char*>(p.kept + kept_unit(t_tile, n0 / kXTileN, nt, wave, cb));
          if (t0v + 64 * wt + 32 * cb + (int)((off >> 4) & 31) < p.T) {
#pragma unroll
            for (int rb = 0; rb < 4; ++rb)
#pragma unroll
              for (int g4 = 0; g4 < 4; ++g4) {
                const xf32x4 v = {acc[rb][cb][4 * g4], acc[rb][cb][4 * g4 + 1], acc[rb][cb][4 * g4 + 2],
                                  acc[rb][cb][4 * g4 + 3]};
                __builtin_nontemporal_store(v, reinterpret_cast<xf32x4*>(base + (4 * rb + g4) * 1024 + off));
                __builtin_amdgcn_sched_barrier(0);
              }
          }
        }
      }
      if (nw + 128 > p.N) {  // the tile that crosses the end of the vocabulary
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const bool dead = nw + 32 * rb + 8 * (i >> 2) + 4 * lh + (i & 3) >= p.N;
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
              if (dead) acc[rb][cb][i] = -INFINITY;
          }
      }
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        float mx = acc[0][cb][0];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int i = 0; i < 16; ++i) mx = fmaxf(mx, acc[rb][cb][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run[cb], mx);  // finite: row nw is alive
        const float mb = m_new * kLog2e;
        float sum = 0.f;
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int i = 0; i < 16; ++i) sum += exp2f(acc[rb][cb][i] * kLog2e - mb);
        l_run[cb] = l_run[cb] * exp2f((m_run[cb] - m_new) * kLog2e) + sum;
        m_run[cb] = m_new;
        const long long rel = yv[cb] - nw;
        const bool mine = rel >= 0 && rel < 128 && (((int)rel >> 2) & 1) == lh;
        if (__builtin_amdgcn_ballot_w64(mine)) {
          const int rl = (int)rel;
#pragma unroll
          for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (mine && rl == 32 * rb + 8 * (i >> 2) + 4 * lh + (i & 3)) tgt[cb] = acc[rb][cb][i];
        }
      }
    }
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) acc[rb][cb] = (f32x16){0};
  };

  // ---- main loop: one barrier per step.  D is a multiple of 128, so a tile is
  // a whole number of step pairs.
  arm(0, total > 0);
#pragma unroll
  for (int k = 0; k < 8; ++k) drip(k);
  next();
  if constexpr (GRAD) {
    int ck = 0, cn0 = tile_first * kXTileN;
    int it = 0;
    // The loads of step it + 1 fly during the products of step it, and the stage
    // that a tile's last step has left is the epilogue's staging area.
    auto step = [&](int stage) __attribute__((always_inline)) {
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
      __syncthreads();
      const bool more = ++it < total;
      arm(stage ^ 1, more);
      read_first(stage);
      sub_step(0, stage, 1, 0);
      sub_step(1, stage, 2, 4);
      sub_step(2, stage, 3, -1);
      sub_step(3, stage, -1, -1);
      if (more) next();
    };
    while (it < total) {
      step(0);
      step(1);
      ck += 2;
      if (ck == nk) {
        finish_tile(cn0);
        ck = 0;
        cn0 += kXTileN;
      }
    }
    return;
  }
  // The barrier of a step lies between its third and fourth sub-step: the step's
  // last fragments are in registers by then, so its stage is free for the loads
  // of step it + 2, and the fourth sub-step's MFMAs run while the first fragments
  // of step it + 1 are read.  With the barrier at the top of a step all eight
  // wavefronts wait for their first fragments together, with no MFMA in flight:
  // 6875 -> 6490 us at 8192 x 4096 x 128256 (keeping the logits 7845 -> 7680),
  // 937 -> 888 at 4096 x 2560 x 50257, 140 -> 134 at 1000 x 2048 x 32000, the
  // same bits.  (All eight loads of a step behind the fourth sub-step: 6465 / 7750
  // where 6412 / 7600 were measured for this split.)
  arm(1, total > 1);
#pragma unroll
  for (int k = 0; k < 8; ++k) drip(k);
  next();
  int sent = 2;              // steps whose loads have been sent, or are about to be
  bool half_sent = false;    // drip() is armed and its loads 4 to 7 are still to go
  arm(0, false);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(8));
  __syncthreads();
  // `more`: the next step is of the same tile, its first fragments are read along the way
  auto step = [&](int stage, bool more) __attribute__((always_inline)) {
    sub_step(0, stage, 1, 4);
    if (half_sent) next();
    sub_step(1, stage, 2, -1);
    sub_step(2, stage, 3, -1);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0) & ~(15 << 8));  // fragments read, the loads of step it + 1 landed
    __syncthreads();
    half_sent = sent < total;
    arm(stage, half_sent);
    ++sent;
    sub_step(3, stage ^ 1, more ? 0 : -1, 0);
  };
  for (int tile = 0; tile < tile_cnt; ++tile) {
    read_first(0);
    for (int k = 2; k < nk; k += 2) {
      step(0, true);
      step(1, true);
    }
    step(0, true);
    step(1, false);
    finish_tile((tile_first + tile) * kXTileN);
  }

  // ---- lane halves, then the two wavefronts that share tokens
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    l_run[cb] += __shfl_xor(l_run[cb], 32, 64);
    tgt[cb] += __shfl_xor(tgt[cb], 32, 64);
  }
  __syncthreads();  // every wavefront is done with the slabs
  float* ex = reinterpret_cast<float*>(xsmem);  // [2 halves][256 tokens][3]
  if (lh == 0) {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      float* e = ex + ((wv * 256) + 64 * wt + 32 * cb + lq) * 3;
      e[0] = m_run[cb];
      e[1] = l_run[cb];
      e[2] = tgt[cb];
    }
  }
  __syncthreads();
  if (tid < 256 && t0 + tid < p.T) {
    const float* e0 = ex + tid * 3;
    const float* e1 = ex + (256 + tid) * 3;
    const float M = fmaxf(e0[0], e1[0]);
    const float Lsum = e0[1] * exp2f((e0[0] - M) * kLog2e) + e1[1] * exp2f((e1[0] - M) * kLog2e);
    const int64_t o = (int64_t)(t0 + tid) * p.n_split + split;
    p.lse_part[o] = M + log2f(Lsum) * kLn2;
    p.tgt_part[o] = e0[2] + e1[2];
  }
}

// lse[t] = log sum over the ranges of exp(lse_part), loss[t] = lse[t] - target logit.
// A wavefront to a token (a thread that walks the ranges of its token by
// itself waits for memory at every one: 205 tokens, 256 ranges
// 77 -> 4.4 us, 500, 128 ranges 53 -> 4.6).
__global__ void __launch_bounds__(256) xent_combine_kernel(const XentParams p) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= p.T) return;
  const float* lp = p.lse_part + (int64_t)t * p.n_split;
  const float* tp = p.tgt_part + (int64_t)t * p.n_split;
  float M = -INFINITY, sum = 0.f, tg = 0.f;
  for (int s = lane; s < p.n_split; s += 64) {
    M = fmaxf(M, lp[s]);
    tg += tp[s];
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) M = fmaxf(M, __shfl_xor(M, m, 64));
  for (int s = lane; s < p.n_split; s += 64) sum += exp2f((lp[s] - M) * kLog2e);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    sum += __shfl_xor(sum, m, 64);
    tg += __shfl_xor(tg, m, 64);
  }
  const float lse = M + log2f(sum) * kLn2;
  if (lane == 0) {
    p.lse[t] = lse;
    p.loss[t] = lse - tg;
  }
}

// In place over a [rows, N] block of logits: g = do[t] (exp(logit - lse[t]) - [n == y[t]]).
// One workgroup per (row, 2048-column segment): blockIdx.x = row.
template <typename T>
__global__ void __launch_bounds__(256) xent_dlogits_kernel(const XentGradParams p) {
  const int64_t t = blockIdx.x;
  const int n0 = blockIdx.y * 2048 + threadIdx.x * 8;
  T* row = reinterpret_cast<T*>(p.logits) + t * p.ld;
  const float lse = p.lse[t] * kLog2e, g = p.dloss[t];
  const long long y = p.y_is_i64 ? reinterpret_cast<const long long*>(p.y)[t]
                                 : (long long)reinterpret_cast<const int*>(p.y)[t];
  if (p.vec && n0 + 8 <= p.N) {
    i32x4 raw = *reinterpret_cast<const i32x4*>(row + n0);
    T* e = reinterpret_cast<T*>(&raw);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      e[i] = (T)(g * (exp2f((float)e[i] * kLog2e - lse) - (n0 + i == y ? 1.f : 0.f)));
    *reinterpret_cast<i32x4*>(row + n0) = raw;
  } else {
    for (int i = 0; i < 8 && n0 + i < p.N; ++i)
      row[n0 + i] = (T)(g * (exp2f((float)row[n0 + i] * kLog2e - lse) - (n0 + i == y ? 1.f : 0.f)));
  }
}

// dlogits from the kept logits of the forward: a wavefront reads one unit
// (contiguous, 16 KiB), applies dloss[t] (exp(logit - lse[t]) - [n == y[t]]) to
// the same fp32 values and in the same order as the epilogue of the GRAD
// kernel, turns the unit through LDS and writes 32 pieces of 256-byte rows.
// A workgroup is the 64 tokens x 256 vocabulary rows of two wavefronts of the
// product.  HBM-bound: 4 bytes in and 2 out per logit: 1.12 ms (5.6 TB/s) at
// 8192 x 128256, where the GRAD kernel takes 7.12 at dim 4096.
//
// BOTH: the unit is also written the other way round, dlogits_t[n, t], for the
// product that sums over tokens (the library's kernels run 25 to 30 % faster on
// operands that are contiguous along the summed index).  A lane reads 8 tokens
// x 8 rows from the staged units of both 32-token halves, turns them with byte
// permutes in registers and writes eight pieces of 16 bytes; eight lanes make
// the 128 bytes of 64 tokens.  Columns of tokens past the end, up to the
// multiple of 64 that dlt_ld holds, are written as zeros.
template <typename T, bool BOTH>
__global__ void __launch_bounds__(256) xent_kept_dlogits_kernel(const XentParams p) {
  __shared__ __attribute__((aligned(16))) unsigned char stage[4][32 * 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lq = lane & 31, lh = lane >> 5;
  const int wv = wave & 1, cb = wave >> 1;
  const int nt = (p.N + kXTileN - 1) / kXTileN;
  const int n_tile = blockIdx.x % nt, q = blockIdx.x / nt;  // q: 64-token group
  const int t_tile = q >> 2, wt = q & 3;
  const int t0 = q * 64 + cb * 32;                          // first token of the unit
  const int nw = n_tile * kXTileN + 128 * wv;
  if (t0 < p.T && nw < p.N) {
    const xf32x4* src = reinterpret_cast<const xf32x4*>(p.kept + kept_unit(t_tile, n_tile, nt, 4 * wv + wt, cb)) + lane;
    const bool live = t0 + lq < p.T;
    const int tok = live ? t0 + lq : p.T - 1;
    xf32x4 in[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) in[i] = live ? __builtin_nontemporal_load(src + i * 64) : (xf32x4){0.f, 0.f, 0.f, 0.f};
    const float lse2 = p.lse[tok] * kLog2e, gl = p.dloss[tok];
    const long long y = p.y_is_i64 ? reinterpret_cast<const long long*>(p.y)[tok]
                                   : (long long)reinterpret_cast<const int*>(p.y)[tok];
    const long long rel64 = y - nw;
    const int rel = rel64 >= 0 && rel64 < 128 ? (int)rel64 : -1;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int nl = 8 * i + 4 * lh;
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float pr = exp2f(in[i][j] * kLog2e - lse2);
        v[j] = gl * (pr - (rel == nl + j ? 1.f : 0.f));
      }
      i32x2 pk = {(int)Elem<T>::pack2(v[0], v[1]), (int)Elem<T>::pack2(v[2], v[3])};
      if (BOTH && !live) pk = (i32x2){0, 0};
      const uint32_t slot = (uint32_t)(nl >> 2) ^ ((lq & 15) << 1);  // 8-byte slots, pairs swizzled by the row
      *reinterpret_cast<i32x2*>(&stage[wave][lq * 256 + slot * 8]) = pk;
    }
  } else if (BOTH) {
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<i32x4*>(&stage[wave][i * 1024 + lane * 16]) = (i32x4){0, 0, 0, 0};
  }
  __syncthreads();
  if (t0 < p.T && nw < p.N) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + (lane >> 4), ch = lane & 15;
      const uint32_t slot = (uint32_t)(2 * ch) ^ ((r & 15) << 1);
      const i32x4 val = *reinterpret_cast<const i32x4*>(&stage[wave][r * 256 + slot * 8]);
      const int n = nw + 8 * ch;
      if (t0 + r < p.T && n < p.N) {
        T* dst = reinterpret_cast<T*>(p.dlogits) + (int64_t)(t0 + r) * p.dl_ld + n;
        if (p.dl_vec && n + 8 <= p.N) {
          __builtin_nontemporal_store(val, reinterpret_cast<i32x4*>(dst));
        } else {
          const T* e = reinterpret_cast<const T*>(&val);
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (n + j < p.N) dst[j] = e[j];
        }
      }
    }
  }
  if (BOTH) {
    // wave (wv, cb): rows 64 cb .. +63 of the half wv, all 64 tokens; lane: token block lane / 8, row block lane % 8
    const int rb = lane >> 3, ch = 8 * cb + (lane & 7);
    i32x4 in[8], out[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 8 * (rb & 3) + i;
      const uint32_t slot = (uint32_t)(2 * ch) ^ ((r & 15) << 1);
      in[i] = *reinterpret_cast<const i32x4*>(&stage[wv + 2 * (rb >> 2)][r * 256 + slot * 8]);
    }
    transpose8x8(in, out);
    const int tq = q * 64 + 8 * rb;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int n = nw + 8 * ch + j;
      if (n < p.N)
        __builtin_nontemporal_store(out[j], reinterpret_cast<i32x4*>(reinterpret_cast<T*>(p.dlogits_t) + (int64_t)n * p.dlt_ld + tq));
    }
  }
}

}  // namespace

// Vocabulary ranges for `tokens` rows: as many as keep one round of workgroups
// (one per CU) busy, never more than there are 256-row vocabulary tiles.
int xent_choose_splits(long long tokens, int vocab, int num_cus) {
  const long long tiles_t = (tokens + kXTileT - 1) / kXTileT;
  const int tiles_n = (vocab + kXTileN - 1) / kXTileN;
  long long s = (num_cus > 0 ? num_cus : 256) / (tiles_t > 0 ? tiles_t : 1);
  if (s < 1) s = 1;
  if (s > tiles_n) s = tiles_n;
  return (int)s;
}

namespace {
template <typename T, bool KEEP, bool GRAD>
int launch_gemm(const XentParams& p, unsigned grid, hipStream_t s) {
  auto kern = xent_gemm_kernel<T, KEEP, GRAD>;
  static LdsLimitOnce lds_once;
  if (const int e = raise_lds_limit(lds_once, reinterpret_cast<const void*>(kern), kXLdsBytes)) return e;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), kXLdsBytes, s, p);
  return (int)hipGetLastError();
}
}  // namespace

// grad: the launch writes dlogits instead of the partial lse / target logit
int launch_xent_fwd(const XentParams& p0, int dtype, bool grad, hipStream_t s) {
  XentParams p = p0;
  p.tiles_t = (p.T + kXTileT - 1) / kXTileT;
  const unsigned grid = (unsigned)(((long long)p.tiles_t * p.n_split + 7) / 8 * 8);
  int rc;
  if (dtype == 0)
    rc = grad     ? launch_gemm<__bf16, false, true>(p, grid, s)
         : p.kept ? launch_gemm<__bf16, true, false>(p, grid, s)
                  : launch_gemm<__bf16, false, false>(p, grid, s);
  else
    rc = grad     ? launch_gemm<_Float16, false, true>(p, grid, s)
         : p.kept ? launch_gemm<_Float16, true, false>(p, grid, s)
                  : launch_gemm<_Float16, false, false>(p, grid, s);
  if (rc || grad) return rc;
  hipLaunchKernelGGL(xent_combine_kernel, dim3((unsigned)((p.T + 3) / 4)), dim3(256), 0, s, p);
  return (int)hipGetLastError();
}

size_t xent_kept_bytes(long long tokens, long long vocab) {
  const size_t tiles = (size_t)((tokens + kXTileT - 1) / kXTileT) * (size_t)((vocab + kXTileN - 1) / kXTileN);
  return tiles * kXTileT * kXTileN * sizeof(float);
}

int launch_xent_kept_dlogits(const XentParams& p, int dtype, hipStream_t s) {
  // the C entry bounds the grid
  const unsigned grid = (unsigned)(((p.T + 63) / 64) * (long long)((p.N + kXTileN - 1) / kXTileN));
  auto kern = p.dlogits_t ? (dtype == 0 ? xent_kept_dlogits_kernel<__bf16, true> : xent_kept_dlogits_kernel<_Float16, true>)
                          : (dtype == 0 ? xent_kept_dlogits_kernel<__bf16, false> : xent_kept_dlogits_kernel<_Float16, false>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, p);
  return (int)hipGetLastError();
}

int launch_xent_dlogits(const XentGradParams& p, int dtype, hipStream_t s) {
  const dim3 grid((unsigned)p.rows, (unsigned)((p.N + 2047) / 2048));
  if (dtype == 0)
    hipLaunchKernelGGL(xent_dlogits_kernel<__bf16>, grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL(xent_dlogits_kernel<_Float16>, grid, dim3(256), 0, s, p);
  return (int)hipGetLastError();
}

}  // namespace mi
