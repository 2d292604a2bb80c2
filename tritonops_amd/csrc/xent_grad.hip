// grad_x = dlogits w of the fused cross-entropy for gfx950, where the result is
// too small for its tiles to fill the chip, or fills it in uneven rounds: the
// vocabulary, which is summed over, is divided among workgroups.
//
// A result of T x D has T D / 65536 tiles of 256 x 256 for 256 CUs (1000 x 2560:
// 40), and the library's product, one workgroup to a tile, takes as long as one
// tile's whole vocabulary.  Here tiles x splits workgroups sum a range of the
// vocabulary each and write fp32 partial tiles, which a second kernel adds up in
// the order of the ranges (deterministic).  MFMA-bound at many tokens, bound by
// reading w at few.
//
// Workgroup = 8 wavefronts, 256 columns d x 256 tokens, steps of 64 vocabulary
// rows: w is the A operand (rows d), its slab kept as it lies in memory, rows n
// of 128 columns each, and read with the transposing LDS read; dlogits are the B
// operand, slabs of 256 tokens x 64 as in xent.hip.  The transposing read has half
// the rate of the plain one, so a wavefront takes 64 columns x 128 tokens.  Two
// stages; the barrier of a step lies between its third and fourth sub-step, as in
// xent.hip's forward.
#include "kernels.h"
#include "tile_core.h"

namespace mi {
namespace {

constexpr int waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
extern __shared__ __attribute__((aligned(1024))) unsigned char gsmem[];
typedef float gf32x4 __attribute__((ext_vector_type(4)));

constexpr int kStepN = 64;                   // vocabulary rows of a step
constexpr int kSlabB = 256 * kStepN * 2;     // one slab: 32 KiB
constexpr int kGradLdsBytes = 4 * kSlabB;    // W stage 0, W stage 1, dlogits stage 0, stage 1
constexpr int kUnitFloats = 64 * 128;        // a wavefront's part of a tile

template <typename T>
__global__ void __launch_bounds__(512) xent_gradx_kernel(const XentGradXParams p) {
  typedef __attribute__((address_space(3))) const i32x4 lds_i32x4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;
  const int wd = wave & 3, wt = wave >> 2;   // 64 columns and 128 tokens of the tile

  // ---- workgroup -> (range, tile): an XCD (ids eight apart) gets neighbouring ones, whose slabs are shared
  const int tiles = p.tiles_t * p.tiles_d;
  int L;
  {
    const int id = blockIdx.x, per = (gridDim.x + 7) >> 3;
    L = (id & 7) * per + (id >> 3);
    if (L >= tiles * p.n_split) return;      // (the grid is rounded up to whole XCDs)
  }
  const int split = L / tiles, tile = L % tiles;
  const int td = tile % p.tiles_d, tt = tile / p.tiles_d;
  const int t0 = tt * 256, d0 = td * 256;
  const int steps_all = (p.N + kStepN - 1) / kStepN, pairs = (steps_all + 1) / 2;
  const int base = pairs / p.n_split, rem = pairs % p.n_split;
  const int first = 2 * (split * base + min(split, rem));
  const int total = 2 * (base + (split < rem ? 1 : 0));   // steps; the last of all may lie behind the vocabulary

  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)gsmem);
  auto uniform64 = [](uint64_t v) __attribute__((always_inline)) -> uint64_t {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
  };
  const uint32_t w_pitch = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p.w_st * 2));
  const uint32_t g_pitch = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p.dl_ld * 2));
  const uint64_t w_base = uniform64((uint64_t)(uintptr_t)p.w + (uint64_t)d0 * 2);
  const uint64_t g_base = uniform64((uint64_t)(uintptr_t)p.dlogits + (uint64_t)t0 * g_pitch);

  // ---- loads: four of W and four of dlogits per wavefront and step.  Load q of
  // W fills four rows n of a 128-column half (256-byte rows, chunk c in slot
  // c ^ swz), of dlogits eight token rows of 128 bytes.  Columns, tokens and
  // vocabulary past the end re-read what is there.
  uint32_t woff[4], goff[4];
  auto set_off = [&](int n0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = 4 * wave + i, half = q >> 4;
      const int r = 4 * (q & 15) + (lane >> 4);
      const int c = (lane & 15) ^ (((r & 3) << 2) | ((r >> 2) & 3));
      const int d = 128 * half + 8 * c;
      woff[i] = (uint32_t)min(r, p.N - 1 - n0) * w_pitch + (uint32_t)(d0 + d < p.D ? d : 0) * 2;
      const int tr = 32 * wave + 8 * i + (lane >> 3);
      const int gc = (lane & 7) ^ ((tr >> 1) & 7);
      goff[i] = (uint32_t)min(tr, p.T - 1 - t0) * g_pitch + (uint32_t)(n0 + 8 * gc < p.N ? gc : 0) * 16;
    }
  };
  int sent = 0;              // steps whose loads have been sent, or are about to be
  uint64_t on = 0, wb = 0, gb = 0;
  uint32_t sw = 0, sg = 0;
  auto arm = [&](int stage, bool live) __attribute__((always_inline)) {
    const int step = min(first + sent, steps_all - 1);   // (a step behind the vocabulary re-reads the last one)
    const int n0 = step * kStepN;
    if (n0 + kStepN > p.N) set_off(n0);
    on = uniform64(live ? ~0ull : 0ull);
    wb = uniform64(w_base + (uint64_t)n0 * w_pitch);
    gb = uniform64(g_base + (uint64_t)n0 * 2);
    sw = lds0 + stage * kSlabB + wave * 4096;
    sg = lds0 + (2 + stage) * kSlabB + wave * 4096;
  };
  auto drip = [&](int k) __attribute__((always_inline)) {
    const int i = k >> 1;
    const uint64_t src = (k & 1) ? gb : wb;
    const uint32_t off = (k & 1) ? goff[i] : woff[i];
    const uint32_t slab = (uint32_t)__builtin_amdgcn_readfirstlane(((k & 1) ? sg : sw) + i * 1024);
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                 :
                 : "s"(on), "v"(off), "s"(src), "s"(slab)
                 : "memory");
  };

  // ---- fragments
  uint32_t a_addr[2][2], b_addr[4];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int r = 8 * lh + 4 * e + ((lane & 15) >> 2);
      const int ch = 4 * (2 * (wd & 1) + rb) + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
      a_addr[rb][e] = lds0 + (wd >> 1) * 16384 + r * 256 + ((ch ^ (((r & 3) << 2) | ((r >> 2) & 3))) << 4) + (lane & 1) * 8;
      asm volatile("" : "+v"(a_addr[rb][e]));
    }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    b_addr[s] = lds0 + 2 * kSlabB + wt * 16384 + lq * 128 + (((2 * s + lh) ^ ((lq >> 1) & 7)) << 4);
    asm volatile("" : "+v"(b_addr[s]));
  }
  f32x16 acc[2][4];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) acc[rb][cb] = (f32x16){0};
  i32x4 af[2][2], bf[2][4];
  auto read_a = [&](int stage, int s, int rb) __attribute__((always_inline)) {
    const uint32_t at = stage * kSlabB + s * 4096;
    af[s & 1][rb] = read_tr_at(a_addr[rb][0] + at, a_addr[rb][1] + at);
  };
  auto read_b = [&](int stage, int s, int cb) __attribute__((always_inline)) {
    bf[s & 1][cb] = *(lds_i32x4*)(uintptr_t)(b_addr[s] + stage * kSlabB + cb * 4096);
  };
  auto sub_step = [&](int s, int stage, int sn, int first_load) __attribute__((always_inline)) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      if (sn >= 0) {
        read_b(stage, sn, cb);
        if (cb < 2) read_a(stage, sn, cb);
      }
      acc[0][cb] = Elem<T>::mfma(af[s & 1][0], bf[s & 1][cb], acc[0][cb]);
      acc[1][cb] = Elem<T>::mfma(af[s & 1][1], bf[s & 1][cb], acc[1][cb]);
      if (first_load >= 0) drip(first_load + cb);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // rows of W and elements of dlogits behind the vocabulary in the slabs of step `it` of this range -> 0
  auto cut = [&](int stage, int it) {
    const int n0 = (first + it) * kStepN;
    if (n0 + kStepN <= p.N) return;
    const int live = max(p.N - n0, 0);
    unsigned char* w = gsmem + stage * kSlabB;
    for (int i = tid; i < (kStepN - live) * 32; i += 512) {
      const int r = live + (i >> 5), half = (i >> 4) & 1, slot = i & 15;
      *reinterpret_cast<i32x4*>(w + half * 16384 + r * 256 + slot * 16) = (i32x4){0, 0, 0, 0};
    }
    if (tid < 256) {
      unsigned char* row = gsmem + (2 + stage) * kSlabB + tid * 128;
      for (int e = live; e < kStepN; ++e)
        *reinterpret_cast<uint16_t*>(row + (((e >> 3) ^ ((tid >> 1) & 7)) << 4) + (e & 7) * 2) = 0;
    }
    __syncthreads();
  };

  set_off(0);   // (the vocabulary has a whole step at least: the C entry)
  arm(0, true);
#pragma unroll
  for (int k = 0; k < 8; ++k) drip(k);
  ++sent;
  arm(1, true);
#pragma unroll
  for (int k = 0; k < 8; ++k) drip(k);
  ++sent;
  bool half_sent = false;
  on = 0;
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(8));
  __syncthreads();
  cut(0, 0);
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) read_b(0, 0, cb);
  read_a(0, 0, 0);
  read_a(0, 0, 1);
  auto step = [&](int stage, int it) __attribute__((always_inline)) {
    sub_step(0, stage, 1, 4);
    if (half_sent) ++sent;
    sub_step(1, stage, 2, -1);
    sub_step(2, stage, 3, -1);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0) & ~(15 << 8));  // fragments read, the loads of step it + 1 landed
    __syncthreads();
    if (it + 1 < total) cut(stage ^ 1, it + 1);
    half_sent = sent < total;
    arm(stage, half_sent);
    sub_step(3, stage ^ 1, 0, 0);
  };
  for (int it = 0; it < total; it += 2) {
    step(0, it);
    step(1, it + 1);
  }

  // ---- the partial tile as it lies in the registers: 1 KiB to a store
  float* out = p.part + ((int64_t)(split * tiles + tile) * 8 + wave) * kUnitFloats + lane * 4;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const gf32x4 v = {acc[rb][cb][4 * g4], acc[rb][cb][4 * g4 + 1], acc[rb][cb][4 * g4 + 2], acc[rb][cb][4 * g4 + 3]};
        if (t0 + 128 * wt + 32 * cb < p.T) *reinterpret_cast<gf32x4*>(out + ((rb * 4 + cb) * 4 + g4) * 256) = v;
      }
}

// The partial tiles added up in the order of the ranges, rounded and written to
// grad_x: a thread takes four columns of a token, as the accumulators held them.
template <typename T>
__global__ void __launch_bounds__(256) xent_gradx_sum_kernel(const XentGradXParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;   // piece of four floats
  const int lane = (int)(i & 63), piece = (int)(i >> 6) & 31, wave = (int)(i >> 11) & 7;
  const int tile = (int)(i >> 14);
  const int tiles = p.tiles_t * p.tiles_d;
  const int rb = piece >> 4, cb = (piece >> 2) & 3, g4 = piece & 3;
  const int t = (tile / p.tiles_d) * 256 + 128 * (wave >> 2) + 32 * cb + (lane & 31);
  const int d = (tile % p.tiles_d) * 256 + 64 * (wave & 3) + 32 * rb + 8 * g4 + 4 * (lane >> 5);
  if (t >= p.T || d >= p.D) return;
  const gf32x4* src = reinterpret_cast<const gf32x4*>(p.part) + i;
  const int64_t step = (int64_t)tiles * 8 * kUnitFloats / 4;
  gf32x4 sum = src[0];
  for (int s = 1; s < p.n_split; ++s) sum += src[s * step];
  i32x2 out;
  out[0] = (int)Elem<T>::pack2(sum[0], sum[1]);
  out[1] = (int)Elem<T>::pack2(sum[2], sum[3]);
  *reinterpret_cast<i32x2*>(reinterpret_cast<T*>(p.gx) + (int64_t)t * p.gx_ld + d) = out;
}

template <typename T>
int launch_t(const XentGradXParams& p, hipStream_t s) {
  auto kern = xent_gradx_kernel<T>;
  static LdsLimitOnce lds_once;
  if (const int e = raise_lds_limit(lds_once, reinterpret_cast<const void*>(kern), kGradLdsBytes)) return e;
  const int tiles = p.tiles_t * p.tiles_d;
  const unsigned grid = (unsigned)((tiles * p.n_split + 7) / 8 * 8);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), kGradLdsBytes, s, p);
  const int e = (int)hipGetLastError();
  if (e) return e;
  hipLaunchKernelGGL(xent_gradx_sum_kernel<T>, dim3((unsigned)(tiles * 64)), dim3(256), 0, s, p);
  return (int)hipGetLastError();
}

}  // namespace

namespace {
// Ranges of the vocabulary that make the estimate of the time least, a round of
// workgroups being one per CU, a step 1.65 us and a partial result 8 bytes of
// traffic: the estimate in us and the ranges (at most `most`).
double best_splits(long long tokens, long long dim, long long vocab, int num_cus, long long most, int* splits) {
  const long long tiles = ((tokens + 255) / 256) * ((dim + 255) / 256);
  const long long pairs = ((vocab + kStepN - 1) / kStepN + 1) / 2;
  double least = 0.0;
  *splits = 1;
  for (long long s = 1; s <= pairs && s <= most && s * tiles <= 65536; ++s) {
    const double rounds = (double)((tiles * s + num_cus - 1) / num_cus);
    const double us = rounds * (double)((pairs + s - 1) / s) * 2 * 1.65 + (double)s * tokens * dim * 8 / 4.5e6;
    if (s == 1 || us < least) {
      least = us;
      *splits = (int)s;
    }
  }
  return least;
}
}  // namespace

// Ranges of the vocabulary for a result too small for its tiles to fill the chip;
// 0 where the vocabulary is less than a step.
int xent_gradx_splits(long long tokens, long long dim, long long vocab, int num_cus) {
  if (tokens <= 0 || dim <= 0 || vocab < kStepN) return 0;
  int s;
  best_splits(tokens, dim, vocab, num_cus > 0 ? num_cus : 256, 256, &s);
  return s;
}

// The same for a result with tiles enough, or 0 where the library's product is left
// to it.  The library has products at 1.0 to 1.2 times the time of the matrix rate
// where one of its tile shapes fills whole rounds of the chip (the large ones any
// number of rounds, those with a side of 192 or 160 a single one, 192 x 128 exactly)
// and for token counts that fill up a multiple of 512 to 3 %; elsewhere it mostly
// takes 1.3 to 1.9 times that time, and ranges of the vocabulary even the rounds
// out.  Library (with w the other way round where that is the rule) -> this, us, at
// 50257 / 128256 words: 1292 x 4096 741 -> 578 / 1905 -> 1380; 2876 x 2048 799 ->
// 563 / 2021 -> 1328; 2876 x 4096 1515 -> 1058 / 3891 -> 2599; 3700 x 3072 1520 ->
// 1039 / 3986 -> 2587; 4100 x 2560 1550 -> 936 / 4054 -> 2289; 4700 x 4096 3109 ->
// 1783 / 8188 -> 4290.  Of 757 sizes that the rule takes, drawn from 1000 to 8000
// tokens, 1024 to 5120 columns and ten vocabularies from 40000 to 128256 words, five
// lose (4, 4, 10, 12 and 12 %, the last 2394 x 2560 x 48000 519 -> 583) and all are
// 1.39 times as fast in the mean.  With the shapes 256 x 256 and half of it alone it
// took 50 of 406 sizes more, 35 of which lost up to 20 % (6430 x 2560 x 40000, 128 x
// 256 in two rounds, 1141, here 1365; 3900 x 3072 x 50257, 256 x 192 in one, 966,
// here 1077). Not taken either: 6200 x 2560 x 50257 (250 tiles) 1080, here 1280;
// vocabularies of 32000, where one in five loses (4700 x 2560 594, here 711; nothing
// was measured between 32000 and 40000).  All of it describes the library that this
// was measured with.  A step of 64 takes it 1.52 us a round of wide tiles and 0.80
// of narrow ones at best; the partial sums are at most as large as the dlogits.
int xent_gradx_uneven_splits(long long tokens, long long dim, long long vocab, int num_cus) {
  if (tokens <= 0 || dim <= 0 || vocab < 40000) return 0;
  if ((512 - tokens % 512) % 512 * 100 <= 3 * tokens) return 0;
  if (num_cus <= 0) num_cus = 256;
  const auto tiles_of = [&](long long rows, long long cols) { return ((tokens + rows - 1) / rows) * ((dim + cols - 1) / cols); };
  const long long tiles = tiles_of(256, 256);
  const long long wide_rounds = (tiles + num_cus - 1) / num_cus, narrow_rounds = (2 * tiles + num_cus - 1) / num_cus;
  // shapes of the library's tiles that fill whole rounds: any number of them, or the one (to hundredths of the CUs)
  constexpr struct { int rows, cols, rounds, fill; } shapes[] = {
      {256, 256, 1 << 30, 96}, {256, 128, 1 << 30, 96}, {128, 256, 1 << 30, 96}, {256, 192, 1, 96}, {192, 256, 1, 96},
      {256, 160, 1, 96}, {160, 256, 1, 96}, {192, 128, 1, 100}, {128, 192, 1, 100}};
  for (const auto& t : shapes) {
    const long long n = tiles_of(t.rows, t.cols), rounds = (n + num_cus - 1) / num_cus;
    if (rounds <= t.rounds && 100 * n >= t.fill * rounds * num_cus) return 0;
  }
  const double steps = (double)((vocab + kStepN - 1) / kStepN);
  const double wide = 1.52 * steps * (double)wide_rounds, narrow = 0.80 * steps * (double)narrow_rounds;
  int s;
  const long long most = 2 * tokens * vocab / (long long)xent_gradx_bytes(tokens, dim, 1);
  const double us = best_splits(tokens, dim, vocab, num_cus, most, &s);
  return most > 0 && us <= 1.2 * (wide < narrow ? wide : narrow) ? s : 0;
}

size_t xent_gradx_bytes(long long tokens, long long dim, int n_split) {
  const size_t tiles = (size_t)((tokens + 255) / 256) * (size_t)((dim + 255) / 256);
  return tiles * (size_t)n_split * 8 * kUnitFloats * sizeof(float);
}

int launch_xent_gradx(const XentGradXParams& p, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_t<__bf16>(p, s) : launch_t<_Float16>(p, s);
}

}  // namespace mi
