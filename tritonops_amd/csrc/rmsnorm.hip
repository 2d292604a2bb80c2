// RMSNorm forward and backward for gfx950 (HBM-bound).
//
// Replaces rmsnorm_fwd_kernel / rmsnorm_bwd_kernel of common/rms.py:8-88,
// :90-218 and their launchers in RMSNormTritonFunction (:221-355):
//   r_t  = 1 / sqrt(eps + mean_d x_td^2)          (saved, fp32, :67-68,88)
//   y_td = x_td * r_t * w_d                       (:81)
//   dx_td = dy_td w_d r_t - x_td r_t^3 (sum_d dy_td w_d x_td) / D   (:199-212)
//   dw_d  = sum_t dy_td x_td r_t                  (:213; the reference adds
//           per-tile sums with atomics, :215)
// A row is owned by part of a wavefront, by one, or by the four wavefronts of a
// workgroup and is read once, with 16-byte loads, into registers;
// the owners walk the rows with a fixed stride and request the next row before
// they work on the current one.  The backward pass keeps the dw sums of each
// thread's element positions in registers over all its rows; dw is reduced in
// two deterministic stages (every workgroup writes one fp32 partial row, a
// second kernel adds the partial rows).  Rows that cannot be read in 16-byte
// chunks (dim not a multiple of the chunk, unaligned rows) are read into
// registers element by element, each load 64 neighbouring elements: forward
// and backward of 134083 x 1001 bf16 took 469 and 661 us as two passes over
// the row with the dw sums in memory, 101 and 217 us (5.3 and 3.7 TB/s) now.
// Only rows of more than 8192 elements that are not chunks, or of more chunks
// than a workgroup's registers hold, still go that way, with one partial row
// per wavefront.  Rows of up to 32 chunks share a wavefront: with one row each,
// 8 of 64 lanes worked on a head of 64 (1048576 rows: 252 and 411 us, now 42
// and 75, 6.3 and 5.4 TB/s).
#include <type_traits>

#include "kernels.h"
#include "tile_core.h"

namespace mi {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// sum over aligned groups of LANES lanes
template <int LANES = 64>
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = LANES / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// element type tags: 0 bf16, 1 f16, 2 f32

// EPC elements per chunk: 16 bytes, or (WIDE = false) a single element, which
// rows of any width, alignment and stride can be read in.
template <typename T, bool WIDE>
struct Chunk {
  static constexpr int EPC = 16 / sizeof(T);
  typedef i32x4 Raw;
  Raw raw;
  __device__ __forceinline__ float at(int e) const { return (float)reinterpret_cast<const T*>(&raw)[e]; }
  __device__ __forceinline__ void set(int e, float v) { reinterpret_cast<T*>(&raw)[e] = (T)v; }
};
template <typename T>
struct Chunk<T, false> {
  static constexpr int EPC = 1;
  typedef T Raw;
  Raw raw;
  __device__ __forceinline__ float at(int) const { return (float)raw; }
  __device__ __forceinline__ void set(int, float v) { raw = (T)v; }
};

// One row's chunks of a thread: chunk j is row chunk t + GROUP*j, where
// GROUP threads (one wavefront, or the four of a workgroup) share the row.
template <typename T, int J, int GROUP, bool WIDE>
struct RowRegs {
  typedef Chunk<T, WIDE> C;
  static constexpr int EPC = C::EPC;
  C c[J];
  // STREAM: the row is not read again soon (non-temporal hint)
  template <bool STREAM = false>
  __device__ __forceinline__ void load(const T* row, int t, int nch) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int ch = t + GROUP * j;
      if (ch < nch) {
        const typename C::Raw* src = reinterpret_cast<const typename C::Raw*>(row + ch * EPC);
        c[j].raw = STREAM ? __builtin_nontemporal_load(src) : *src;
      }
    }
  }
};

// The weights of a thread's positions: kept for all rows where a chunk is one
// element (each would be a load of its own again), read from the cache with
// the row otherwise.
template <typename TW, int J, int GROUP, int EPC, bool KEPT>
struct WeightRegs {
  const TW* w;
  int t;
  __device__ __forceinline__ WeightRegs(const TW* w_, int t_, int) : w(w_), t(t_) {}
  __device__ __forceinline__ float at(int j, int e) const { return (float)w[(t + GROUP * j) * EPC + e]; }
};
template <typename TW, int J, int GROUP>
struct WeightRegs<TW, J, GROUP, 1, true> {
  float v[J];
  __device__ __forceinline__ WeightRegs(const TW* w, int t, int nch) {
#pragma unroll
    for (int j = 0; j < J; ++j) v[j] = t + GROUP * j < nch ? (float)w[t + GROUP * j] : 0.f;
  }
  __device__ __forceinline__ float at(int j, int) const { return v[j]; }
};

// Sum over the GROUP threads that share a row.  GROUP == 256: the wavefront sums
// meet in LDS; `xs` is double-buffered by row parity, so one barrier per row is
// enough (a wavefront can only overwrite a slot after every other wavefront
// has passed the barrier of the row in between).
template <int GROUP>
__device__ __forceinline__ float group_sum(float v, float (*xs)[4], int& par, int wave, int lane) {
  v = wave_sum<(GROUP < 64 ? GROUP : 64)>(v);
  if (GROUP > 64) {
    if (lane == 0) xs[par][wave] = v;
    __syncthreads();
    v = (xs[par][0] + xs[par][1]) + (xs[par][2] + xs[par][3]);
    par ^= 1;
  }
  return v;
}

// ---------------------------------------------------------------- forward
// GROUP threads (part of a wavefront, one, or a workgroup) own a row at a time
// and walk rows slot, slot + n_slots, ...; the next row is requested before the current one is reduced
// and scaled (J <= 8: two rows fit in registers).
template <typename T, typename TW, int J, int GROUP, bool WIDE>
__global__ void __launch_bounds__(256) rms_fwd_vec_kernel(const RmsParams p) {
  typedef Chunk<T, WIDE> C;
  constexpr int EPC = C::EPC;
  constexpr int ROWS = 256 / GROUP;  // rows a workgroup has in hand
  constexpr bool PF = J <= (WIDE ? 8 : 16);
  __shared__ float xs[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = (int)threadIdx.x % GROUP;
  const int slot = (int)blockIdx.x * ROWS + (int)threadIdx.x / GROUP;
  const int n_slots = (int)gridDim.x * ROWS;
  const int D = p.dim;
  const int nch = D / EPC;
  const WeightRegs<TW, J, GROUP, EPC, !WIDE> w(reinterpret_cast<const TW*>(p.w), t, nch);
  const T* xb = reinterpret_cast<const T*>(p.x);
  int par = 0;
  RowRegs<T, J, GROUP, WIDE> cur, nxt;
  if (PF && slot < p.rows) cur.load(xb + (int64_t)slot * p.x_st, t, nch);
  for (int64_t row = slot; row < p.rows; row += n_slots) {
    if (PF) {
      if (row + n_slots < p.rows) nxt.load(xb + (row + n_slots) * p.x_st, t, nch);
    } else {
      cur.load(xb + row * p.x_st, t, nch);
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (t + GROUP * j < nch) {
#pragma unroll
        for (int e = 0; e < EPC; ++e) ss += cur.c[j].at(e) * cur.c[j].at(e);
      }
    ss = group_sum<GROUP>(ss, xs, par, wave, lane);
    const float r = 1.0f / sqrtf(p.eps + ss / (float)D);
    T* y = reinterpret_cast<T*>(p.y) + row * p.y_st;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int ch = t + GROUP * j;
      if (ch < nch) {
        C o;
#pragma unroll
        for (int e = 0; e < EPC; ++e) o.set(e, cur.c[j].at(e) * r * w.at(j, e));
        __builtin_nontemporal_store(o.raw, reinterpret_cast<typename C::Raw*>(y + ch * EPC));
      }
    }
    if (t == 0) p.rsqrt[row] = r;
    if (PF) cur = nxt;
  }
}

// element-wise path: any dim, any alignment
template <typename T, typename TW>
__global__ void __launch_bounds__(256) rms_fwd_elem_kernel(const RmsParams p) {
  const int lane = threadIdx.x & 63;
  const int wid = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int n_waves = gridDim.x * 4;
  const TW* w = reinterpret_cast<const TW*>(p.w);
  const int D = p.dim;
  for (int64_t row = wid; row < p.rows; row += n_waves) {
    const T* x = reinterpret_cast<const T*>(p.x) + row * p.x_st;
    T* y = reinterpret_cast<T*>(p.y) + row * p.y_st;
    float ss = 0.f;
    for (int i = lane; i < D; i += 64) {
      const float v = (float)x[i];
      ss += v * v;
    }
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(p.eps + ss / (float)D);
    for (int i = lane; i < D; i += 64) y[i] = (T)((float)x[i] * r * (float)w[i]);
    if (lane == 0) p.rsqrt[row] = r;
  }
}

// --------------------------------------------------------------- backward
// GROUP threads (part of a wavefront, one, or a workgroup) own a row at a time
// and walk rows slot, slot + n_slots, ...; every thread keeps the dw contributions of its element
// positions in registers and the workgroup writes ONE fp32 partial row.
template <typename T, typename TW, int J, int GROUP, bool WIDE>
__global__ void __launch_bounds__(256) rms_bwd_vec_kernel(const RmsParams p) {
  typedef Chunk<T, WIDE> C;
  constexpr int EPC = C::EPC;
  constexpr int ROWS = 256 / GROUP;  // rows a workgroup has in hand
  constexpr bool PF = J <= (WIDE ? 4 : 16);  // two (x, dy) row pairs in registers
  __shared__ float xs[2][4];
  __shared__ float red[GROUP <= 64 ? 4 : 1][64][EPC + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = (int)threadIdx.x % GROUP;
  const int slot = (int)blockIdx.x * ROWS + (int)threadIdx.x / GROUP;
  const int n_slots = (int)gridDim.x * ROWS;
  const int D = p.dim;
  const int nch = D / EPC;
  const WeightRegs<TW, J, GROUP, EPC, !WIDE> w(reinterpret_cast<const TW*>(p.w), t, nch);
  const T* xb = reinterpret_cast<const T*>(p.x);
  const T* db = reinterpret_cast<const T*>(p.dy);
  int par = 0;
  float dwacc[J][EPC];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int e = 0; e < EPC; ++e) dwacc[j][e] = 0.f;
  // element by element an owner may walk many rows: their sums are folded away every eight rows, which keeps
  // the fp32 error at that of short sums (33563 x 3999 in fp32: 2.0e-7 without it, dw against 64 bits)
  float dwold[WIDE ? 1 : J];
  int walked = 0;
#pragma unroll
  for (int j = 0; j < (WIDE ? 1 : J); ++j) dwold[j] = 0.f;
  RowRegs<T, J, GROUP, WIDE> cx, cd, nx, nd;
  if (PF && slot < p.rows) {
    cx.template load<true>(xb + (int64_t)slot * p.x_st, t, nch);
    cd.template load<true>(db + (int64_t)slot * p.dy_st, t, nch);
  }
  for (int64_t row = slot; row < p.rows; row += n_slots) {
    if (PF) {
      if (row + n_slots < p.rows) {
        nx.template load<true>(xb + (row + n_slots) * p.x_st, t, nch);
        nd.template load<true>(db + (row + n_slots) * p.dy_st, t, nch);
      }
    } else {
      cx.template load<true>(xb + row * p.x_st, t, nch);
      cd.template load<true>(db + row * p.dy_st, t, nch);
    }
    T* dx = reinterpret_cast<T*>(p.dx) + row * p.dx_st;
    const float r = p.rsqrt[row];
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int ch = t + GROUP * j;
      if (ch < nch) {
#pragma unroll
        for (int e = 0; e < EPC; ++e) dot += cd.c[j].at(e) * w.at(j, e) * cx.c[j].at(e);
      }
    }
    dot = group_sum<GROUP>(dot, xs, par, wave, lane);
    const float k = r * r * r * dot / (float)D;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int ch = t + GROUP * j;
      if (ch < nch) {
        C o;
#pragma unroll
        for (int e = 0; e < EPC; ++e) {
          const float xv = cx.c[j].at(e), dv = cd.c[j].at(e);
          o.set(e, dv * w.at(j, e) * r - xv * k);
          dwacc[j][e] += dv * xv * r;
        }
        __builtin_nontemporal_store(o.raw, reinterpret_cast<typename C::Raw*>(dx + ch * EPC));
      }
    }
    if (PF) {
      cx = nx;
      cd = nd;
    }
    if (!WIDE && (++walked & 7) == 0) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        dwold[WIDE ? 0 : j] += dwacc[j][0];
        dwacc[j][0] = 0.f;
      }
    }
  }
  if (!WIDE) {
#pragma unroll
    for (int j = 0; j < J; ++j) dwacc[j][0] += dwold[WIDE ? 0 : j];
  }
  float* part = p.dw_part + (int64_t)blockIdx.x * D;
  if (GROUP > 64) {
    // every thread owns its positions of the workgroup's partial row
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int ch = t + GROUP * j;
      if (ch < nch) {
#pragma unroll
        for (int e = 0; e < EPC; ++e) part[ch * EPC + e] = dwacc[j][e];
      }
    }
  } else {
    // the groups of a wavefront and the four wavefronts cover the same positions: add by lane exchanges and
    // through LDS, one chunk position at a time
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
      for (int e = 0; e < EPC; ++e) {
        float v = dwacc[j][e];
#pragma unroll
        for (int m = 32; m >= GROUP; m >>= 1) v += __shfl_xor(v, m, 64);
        red[wave][lane][e] = v;
      }
      __syncthreads();
      if (wave == 0 && lane < GROUP) {
        const int ch = lane + GROUP * j;
        if (ch < nch) {
#pragma unroll
          for (int e = 0; e < EPC; ++e)
            part[ch * EPC + e] = red[0][lane][e] + red[1][lane][e] + red[2][lane][e] + red[3][lane][e];
        }
      }
      __syncthreads();
    }
  }
}

// element-wise path: any dim, any alignment
template <typename T, typename TW>
__global__ void __launch_bounds__(256) rms_bwd_elem_kernel(const RmsParams p) {
  const int lane = threadIdx.x & 63;
  const int wid = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int n_waves = gridDim.x * 4;
  const TW* w = reinterpret_cast<const TW*>(p.w);
  const int D = p.dim;
  float* part = p.dw_part + (int64_t)wid * D;
  for (int i = lane; i < D; i += 64) part[i] = 0.f;
  for (int64_t row = wid; row < p.rows; row += n_waves) {
    const T* x = reinterpret_cast<const T*>(p.x) + row * p.x_st;
    const T* dy = reinterpret_cast<const T*>(p.dy) + row * p.dy_st;
    T* dx = reinterpret_cast<T*>(p.dx) + row * p.dx_st;
    const float r = p.rsqrt[row];
    float dot = 0.f;
    for (int i = lane; i < D; i += 64) dot += (float)dy[i] * (float)w[i] * (float)x[i];
    dot = wave_sum(dot);
    const float k = r * r * r * dot / (float)D;
    for (int i = lane; i < D; i += 64) {
      const float xv = (float)x[i], dv = (float)dy[i];
      dx[i] = (T)(dv * (float)w[i] * r - xv * k);
      part[i] += dv * xv * r;  // element i of the partial row belongs to lane i % 64 alone
    }
  }
}

// dw[d] = sum of in[n_in][D] over the rows, in one launch: a workgroup covers
// CL x V columns with 256 / CL row slices, whose sums meet by lane exchanges and
// through LDS in a fixed order.  1024 rows of 4096: 5 us (two launches, 32 rows
// in between, took 5 + 4 and the gap between them).
template <typename TW, int V, int CL>
__global__ void __launch_bounds__(256) rms_dw_sum_kernel(const float* in, TW* dw, int n_in, int D) {
  __shared__ float red[4][CL][V];
  constexpr int NS = 256 / CL;
  const int c = threadIdx.x % CL, slice = threadIdx.x / CL;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = (blockIdx.x * CL + c) * V;
  float a4[4][V];  // four sums per column: short ones, whose loads do not wait for each other
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int e = 0; e < V; ++e) a4[u][e] = 0.f;
  if (col < D) {
    auto add = [&](int i, int u) __attribute__((always_inline)) {
      const float* src = in + (int64_t)i * D + col;
      if (V == 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
        for (int e = 0; e < V; ++e) a4[u][e] += v[e];
      } else {
        a4[u][0] += src[0];
      }
    };
    int i = slice;
    if (V == 4) {
      // few rows to a slice: the bound is looked at per row (1048576 x 64, whole backward: 75 against 82 us)
#pragma unroll 2
      for (; i < n_in; i += 4 * NS) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (i + u * NS >= n_in) break;
          add(i + u * NS, u);
        }
      }
    } else {
      // many: batches of sixteen loads (262144 x 511: 189 against 207 us)
#pragma unroll 4
      for (; i + 3 * NS < n_in; i += 4 * NS) {
#pragma unroll
        for (int u = 0; u < 4; ++u) add(i + u * NS, u);
      }
      for (; i < n_in; i += NS) add(i, 0);
    }
  }
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = (a4[0][e] + a4[1][e]) + (a4[2][e] + a4[3][e]);
#pragma unroll
  for (int e = 0; e < V; ++e) {
#pragma unroll
    for (int m = 32; m >= CL; m >>= 1) acc[e] += __shfl_xor(acc[e], m, 64);
    if (lane < CL) red[wave][c][e] = acc[e];
  }
  __syncthreads();
  if (threadIdx.x < CL * V) {
    const int cc = threadIdx.x / V, e = threadIdx.x % V;
    const int d = (blockIdx.x * CL + cc) * V + e;
    if (d < D) dw[d] = (TW)((red[0][cc][e] + red[1][cc][e]) + (red[2][cc][e] + red[3][cc][e]));
  }
}

// Adds the n_parts partial rows at p.dw_part into p.dw
template <typename TW>
int reduce_dw(const RmsParams& p, int n_parts, hipStream_t s) {
  const float* in = p.dw_part;
  TW* dw = reinterpret_cast<TW*>(p.dw);
  if (p.dim % 4 == 0 && reinterpret_cast<uintptr_t>(in) % 16 == 0)
    hipLaunchKernelGGL((rms_dw_sum_kernel<TW, 4, 4>), dim3((unsigned)((p.dim + 15) / 16)), dim3(256), 0, s, in, dw, n_parts,
                       p.dim);
  else
    hipLaunchKernelGGL((rms_dw_sum_kernel<TW, 1, 16>), dim3((unsigned)((p.dim + 15) / 16)), dim3(256), 0, s, in, dw, n_parts,
                       p.dim);
  return (int)hipGetLastError();
}

// Shapes of the chunked path: GROUP threads with J chunks each.  16-byte
// chunks: rows of up to 32 are owned by 8, 16 or 32 lanes, up to 128 by a
// wavefront, longer ones by a workgroup.  Single elements: a wavefront owns rows
// of up to 1024, a workgroup up to 8192.
constexpr int kWaveRowChunks = 128, kWaveRowElems = 1024, kMaxRowElems = 8192;
constexpr int kMaxRowWorkgroups = 1024, kMaxPartRowWorkgroups = 2048;

// MAX_J: 16-byte chunks that a thread holds at most (the C entry passes `wide` for no longer rows).
template <int MAX_J, typename F>
void by_shape(bool wide, int nch, F&& f) {
  using std::integral_constant;
  using std::true_type;
  using std::false_type;
  auto go = [&](auto j, auto group, auto w) { f(j, group, w); };
#define MI_RMS_SHAPE(J, GROUP, W) go(integral_constant<int, J>{}, integral_constant<int, GROUP>{}, W{})
  if (!wide) {
    if (nch <= 256) MI_RMS_SHAPE(4, 64, false_type);
    else if (nch <= 512) MI_RMS_SHAPE(8, 64, false_type);
    else if (nch <= kWaveRowElems) MI_RMS_SHAPE(16, 64, false_type);
    else if (nch <= 2048) MI_RMS_SHAPE(8, 256, false_type);
    else if (nch <= 4096) MI_RMS_SHAPE(16, 256, false_type);
    else MI_RMS_SHAPE(32, 256, false_type);
  } else {
    if (nch <= 8) MI_RMS_SHAPE(1, 8, true_type);
    else if (nch <= 16) MI_RMS_SHAPE(1, 16, true_type);
    else if (nch <= 32) MI_RMS_SHAPE(1, 32, true_type);
    else if (nch <= 64) MI_RMS_SHAPE(1, 64, true_type);
    else if (nch <= kWaveRowChunks) MI_RMS_SHAPE(2, 64, true_type);
    else if (nch <= 256) MI_RMS_SHAPE(1, 256, true_type);
    else if (nch <= 512) MI_RMS_SHAPE(2, 256, true_type);
    else if (nch <= 1024) MI_RMS_SHAPE(4, 256, true_type);
    else if (nch <= 2048) MI_RMS_SHAPE(8, 256, true_type);
    else if constexpr (MAX_J > 8) MI_RMS_SHAPE(MAX_J, 256, true_type);
  }
#undef MI_RMS_SHAPE
}

// Workgroups of the chunked path (= partial dw rows of the backward pass, so
// never more than n_waves, which is at least the number of rows up to 4096).
// Part-wavefront rows keep only 16 bytes per lane and row in flight: eight
// workgroups per CU instead of four.
inline unsigned vec_grid(const RmsParams& p, bool wide, int nch, int n_waves) {
  if (wide && nch <= 32) {
    const int rows_wg = 256 / (nch <= 8 ? 8 : nch <= 16 ? 16 : 32);
    const int64_t wgs = (p.rows + rows_wg - 1) / rows_wg;
    return (unsigned)(wgs < kMaxPartRowWorkgroups ? wgs : kMaxPartRowWorkgroups);
  }
  if (nch <= (wide ? kWaveRowChunks : kWaveRowElems)) return (unsigned)(n_waves / 4);
  return (unsigned)(p.rows < kMaxRowWorkgroups ? p.rows : kMaxRowWorkgroups);
}

template <typename T, typename TW>
int launch_fwd_t(const RmsParams& p, bool wide, int n_waves, hipStream_t s) {
  if (wide || p.dim <= kMaxRowElems) {
    const int nch = wide ? p.dim / (16 / (int)sizeof(T)) : p.dim;
    by_shape<kRmsMaxChunks>(wide, nch, [&](auto jc, auto wc, auto wide_c) {
      hipLaunchKernelGGL((rms_fwd_vec_kernel<T, TW, decltype(jc)::value, decltype(wc)::value, decltype(wide_c)::value>),
                         dim3(vec_grid(p, wide, nch, n_waves)), dim3(256), 0, s, p);
    });
  } else {
    hipLaunchKernelGGL((rms_fwd_elem_kernel<T, TW>), dim3((unsigned)(n_waves / 4)), dim3(256), 0, s, p);
  }
  return (int)hipGetLastError();
}

// Partial dw rows: one per workgroup (chunked path) or one per wavefront; never more than n_waves.
template <typename T, typename TW>
int launch_bwd_t(const RmsParams& p, bool wide, int n_waves, hipStream_t s) {
  int n_parts = n_waves;
  if (wide || p.dim <= kMaxRowElems) {
    const int nch = wide ? p.dim / (16 / (int)sizeof(T)) : p.dim;
    const unsigned grid = vec_grid(p, wide, nch, n_waves);
    n_parts = (int)grid;
    by_shape<kRmsMaxChunksBwd>(wide, nch, [&](auto jc, auto wc, auto wide_c) {
      hipLaunchKernelGGL((rms_bwd_vec_kernel<T, TW, decltype(jc)::value, decltype(wc)::value, decltype(wide_c)::value>),
                         dim3(grid), dim3(256), 0, s, p);
    });
  } else {
    hipLaunchKernelGGL((rms_bwd_elem_kernel<T, TW>), dim3((unsigned)(n_waves / 4)), dim3(256), 0, s, p);
  }
  int rc = (int)hipGetLastError();
  if (rc) return rc;
  return reduce_dw<TW>(p, n_parts, s);
}

template <typename F>
int dispatch2(int xt, int wt, F&& f) {
  // w is either of x's type or fp32 (an fp32 parameter under 16-bit activations)
  if (xt == 0) return wt == 0 ? f((__bf16*)nullptr, (__bf16*)nullptr) : f((__bf16*)nullptr, (float*)nullptr);
  if (xt == 1) return wt == 1 ? f((_Float16*)nullptr, (_Float16*)nullptr) : f((_Float16*)nullptr, (float*)nullptr);
  return f((float*)nullptr, (float*)nullptr);
}

}  // namespace

int rms_partial_rows(long long rows, int num_cus) {
  // wavefronts of a pass (and upper bound of the partial dw rows): enough to
  // fill the chip (16 wavefronts per CU), never more than one per row, a multiple of 4
  long long w = (long long)(num_cus > 0 ? num_cus : 256) * 16;
  if (w > rows) w = rows;
  w = (w + 3) / 4 * 4;
  return (int)(w < 4 ? 4 : w);
}

int launch_rms_fwd(const RmsParams& p, int x_dtype, int w_dtype, bool vec, int n_waves, hipStream_t s) {
  return dispatch2(x_dtype, w_dtype, [&](auto* tx, auto* tw) {
    using T = std::remove_pointer_t<decltype(tx)>;
    using TW = std::remove_pointer_t<decltype(tw)>;
    return launch_fwd_t<T, TW>(p, vec, n_waves, s);
  });
}

int launch_rms_bwd(const RmsParams& p, int x_dtype, int w_dtype, bool vec, int n_waves, hipStream_t s) {
  return dispatch2(x_dtype, w_dtype, [&](auto* tx, auto* tw) {
    using T = std::remove_pointer_t<decltype(tx)>;
    using TW = std::remove_pointer_t<decltype(tw)>;
    return launch_bwd_t<T, TW>(p, vec, n_waves, s);
  });
}

}  // namespace mi
