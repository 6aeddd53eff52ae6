// Row and query encoding for the int8 MFMA screen, tombstones and small fills (gfx950).
//
// Reference contracts: encode_int8_rows / encode_int8_queries (detail/int8.cuh:30-136) and
// remove_rows / remove_int8_rows (certex_kernels.cuh:391-415, detail/int8.cuh:139-147). For 8-bit
// integer vectors the code is the vector itself shifted into int8 (no projection, no scale), so
// the screen is exact; the row term folds the norm (l2) or the shift correction (inner product).

#include "../kernels.hpp"
#include "lanes.hpp"

#include <cmath>
#include <type_traits>

namespace certex_amd {
namespace {

inline unsigned blocks_for(int64_t n, int block = 256)
{
  return unsigned((n + block - 1) / block);
}

/**
 * Bytes [j0, j0 + 16) of a row of dim bytes as int8 codes (zero past dim) in four words. A whole
 * chunk is one 16-byte load whatever the row's alignment (memory accesses of any alignment are
 * enabled on these devices); only the chunk that crosses the row's end goes byte by byte.
 */
__device__ __forceinline__ void code_chunk(const uint8_t* row, int64_t dim, int64_t j0, uint8_t flip,
                                           int (&w)[4])
{
  if (j0 + 16 <= dim) {
    __builtin_memcpy(w, row + j0, 16);
    const uint32_t f = uint32_t(flip) * 0x01010101u;
#pragma unroll
    for (int i = 0; i < 4; ++i) { w[i] = int(uint32_t(w[i]) ^ f); }
    return;
  }
  uint8_t v[16];
#pragma unroll
  for (int b = 0; b < 16; ++b) { v[b] = j0 + b < dim ? uint8_t(row[j0 + b] ^ flip) : uint8_t(0); }
  __builtin_memcpy(w, v, 16);
}

/**
 * Stored rows of integer vectors: CPR consecutive lanes per row, lane c on the 16-byte chunks c,
 * c + CPR, ... of the row (CPR = 8 and 16: rows of 128 and 256 bytes, one chunk per lane; 16 also
 * for wider rows, whose rows are multiples of 256 bytes). The row's norm and sum meet by a
 * butterfly over its lanes. Memory-bound: 250,000 x 960 bytes (0.5 GB read and written) 290 -> 86
 * us, 5.8 TB/s (a wave per row and byte loads before).
 */
template <int CPR>
__global__ __launch_bounds__(256) void encode_rows_kernel(const uint8_t* x, int64_t n, int64_t dim, int row_bytes,
                                                          uint8_t flip, metric_kind metric, int8_t* codes,
                                                          int32_t* rowc)
{
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  const int64_t r = t / CPR;
  const int c     = int(t % CPR);
  int norm = 0, sum = 0;
  if (r < n) {
    for (int j = c; j < row_bytes / 16; j += CPR) {
      int w[4];
      code_chunk(x + r * dim, dim, int64_t(j) * 16, flip, w);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        norm = __builtin_amdgcn_sdot4(w[i], w[i], norm, false);
        sum  = __builtin_amdgcn_sdot4(w[i], 0x01010101, sum, false);
      }
      *reinterpret_cast<int4*>(codes + r * row_bytes + int64_t(j) * 16) = int4{w[0], w[1], w[2], w[3]};
    }
  }
  norm = lanes::sum<CPR>(norm);
  sum  = lanes::sum<CPR>(sum);
  if (r < n && c == 0) { rowc[r] = metric == metric_kind::l2 ? -(norm >> 1) : (flip ? 128 * sum : 0); }
}

__global__ void encode_queries_kernel(const uint8_t* q, const int32_t* rows, int64_t nq,
                                      int64_t nq_pad, int64_t dim, int row_bytes, uint8_t flip,
                                      int8_t* qcodes, int8_t* qpaired)
{
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= nq_pad * row_bytes) { return; }
  const int64_t i = t / row_bytes, j = t % row_bytes;
  const int64_t r = i < nq && rows != nullptr ? int64_t(rows[i]) : i;  // the caller's query row
  const int8_t c  = (i < nq && j < dim) ? int8_t(q[r * dim + j] ^ flip) : int8_t(0);
  qcodes[t]       = c;
  if (qpaired != nullptr) { qpaired[paired_offset(i, j, row_bytes)] = c; }
}

__device__ inline int64_t stored_row(const row_places& at, int64_t id)
{
  return id < at.n_listed ? int64_t(at.list_pos[id]) : id;
}

__global__ void remove_kernel(const int64_t* ids, int64_t n, int64_t size, int32_t* rowc,
                              unsigned long long* newly, row_places at)
{
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= n) { return; }
  const int64_t id = ids[t];
  if (id < 0 || id >= size) { return; }
  if (id < at.n_part) { static_cast<int32_t*>(at.part_rowc)[at.part_pos[id]] = kDeadRow; }
  if (at.anchor_stride > 0 && id % at.anchor_stride == 0 && id / at.anchor_stride < at.n_anchor) {
    static_cast<int32_t*>(at.anchor_rowc)[id / at.anchor_stride] = kDeadRow;
  }
  if (atomicExch(rowc + stored_row(at, id), kDeadRow) != kDeadRow) { atomicAdd(newly, 1ull); }
}

template <typename T>
__global__ void fill_kernel(T* p, int64_t n, T v)
{
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    p[i] = v;
  }
}

template <typename V>
__global__ __launch_bounds__(256) void mask_terms_kernel(const V* rowc, int64_t n, const V* anchor_rowc,
                                                         int64_t n_anchor, int64_t stride, filter_args f,
                                                         V dead, V* terms, V* anchor_terms)
{
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= n + n_anchor) { return; }
  const bool anchor = t >= n;
  const uint32_t id = anchor ? uint32_t((t - n) * stride) : listed_id(f, uint32_t(t));
  const V term      = anchor ? anchor_rowc[t - n] : rowc[t];
  const V v         = (f.words[id >> 5] >> (id & 31)) & 1u ? term : dead;
  if (anchor) {
    anchor_terms[t - n] = v;
  } else {
    terms[t] = v;
  }
}

/** Four boolean bytes as the bits 0 .. 3 (any non-zero byte counts): the bytes become 0 or 1, and
 *  one multiplication moves byte b to bit 24 + b. */
__device__ __forceinline__ uint32_t pack4(uint32_t w)
{
  const uint32_t ones = ((((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) >> 7) & 0x01010101u;
  return (ones * 0x01020408u) >> 24 & 0xfu;
}

/**
 * Boolean bytes to filter words: 16 bytes (one load, at any alignment) to 16 bits per thread.
 * Memory-bound: 60 million bytes took 790 us as tensor operations (a 32-bit copy of every byte, a
 * product and a sum), 14 us here.
 */
__global__ __launch_bounds__(256) void pack_bits_kernel(const uint8_t* mask, int64_t n, uint16_t* out, int64_t n_out)
{
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= n_out) { return; }
  const int64_t e0 = 16 * t;
  uint32_t w[4]    = {0, 0, 0, 0};
  if (e0 + 16 <= n) {
    __builtin_memcpy(w, mask + e0, 16);
  } else {
    uint8_t b[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) { b[i] = e0 + i < n ? mask[e0 + i] : uint8_t(0); }
    __builtin_memcpy(w, b, 16);
  }
  out[t] = uint16_t(pack4(w[0]) | pack4(w[1]) << 4 | pack4(w[2]) << 8 | pack4(w[3]) << 12);
}

__global__ void iota_kernel(int32_t* p, int64_t n, int32_t first)
{
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    p[i] = first + int32_t(i);
  }
}

// ---- float vectors ---------------------------------------------------------------------------

__device__ inline double coord(const void* p, elem t, int64_t i)
{
  if (t == elem::bf16) { return double(static_cast<const __bf16*>(p)[i]); }
  return t == elem::f32 ? double(static_cast<const float*>(p)[i])
                        : double(static_cast<const _Float16*>(p)[i]);
}

/** *p = max(*p, v) for non-negative doubles: a plain atomic on one word takes about 10 ns of every
 *  workgroup's turn, so a workgroup whose value cannot raise it only reads it. */
__device__ inline void atomic_max_pos(double* p, double v)
{
  if (!(v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) { return; }
  // non-negative doubles order like their bit patterns
  atomicMax(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v));
}

/** Upper bound of sqrt(s) for a non-negative fp64 sum s accumulated over `terms` terms. */
__device__ inline double sqrt_up(double s, int64_t terms)
{
  return sqrt(s * (1.0 + 4e-16 * double(terms + 4))) * (1.0 + 4e-16);
}

constexpr double kF16Safe = 4096.0;  // |Z| above this: the row is always a candidate

/** fp16 value of z (round to nearest), 0 for results below the smallest normal fp16. */
__device__ inline _Float16 to_f16(double z)
{
  const _Float16 h = _Float16(float(z));
  return fabs(double(h)) < 6.103515625e-05 ? _Float16(0.0f) : h;
}

/** to_f16 for queries, which may lie any distance from the rows: a finite value past the range of fp16
 *  becomes its largest one, and the difference goes into the query's |W - fp16(W)| (an infinite half
 *  made NaN screen values, which pass no threshold). */
__device__ inline _Float16 query_f16(double w)
{
  constexpr double most = 65504.0;
  return to_f16(fabs(w) > most && fabs(w) < INFINITY ? copysign(most, w) : w);
}

/** Sum of v over the 64 lanes of a wave (xor butterfly: every lane gets the sum). */
__device__ inline double wave_sum(double v) { return lanes::sum<64>(v); }

/** A lane's coordinates of one row loaded together: j = j0 + 64 u + lane, u < kLaneChunk. */
constexpr int kLaneChunk = 16;

template <typename T, int N>
__device__ inline void lane_coords_t(const T* row, int64_t dim, int64_t j0, int lane,
                                     double (&v)[N])
{
  T x[N];  // loads from clamped positions, unconditional: all issued before any use
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int64_t j = j0 + 64 * u + lane;
    x[u]            = row[j < dim ? j : dim - 1];
  }
#pragma unroll
  for (int u = 0; u < N; ++u) { v[u] = j0 + 64 * u + lane < dim ? double(x[u]) : 0.0; }
}

/** Coordinates j0 + 64 u + lane of row i (0 at and past dim), all loads issued before any use:
 *  a loop that used each coordinate as it arrived waited for one load at a time. */
template <int N = kLaneChunk>
__device__ inline void lane_coords(const void* x, elem t, int64_t i, int64_t dim, int64_t j0,
                                   int lane, double (&v)[N])
{
  if (t == elem::bf16) {
    lane_coords_t(static_cast<const __bf16*>(x) + i * dim, dim, j0, lane, v);
  } else if (t == elem::f32) {
    lane_coords_t(static_cast<const float*>(x) + i * dim, dim, j0, lane, v);
  } else {
    lane_coords_t(static_cast<const _Float16*>(x) + i * dim, dim, j0, lane, v);
  }
}

/** center[j0 + 64 u + lane], u < N (clamped positions past dim), loaded together. */
template <int N = kLaneChunk>
__device__ inline void lane_center(const double* center, int64_t dim, int64_t j0, int lane,
                                   double (&c)[N])
{
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int64_t j = j0 + 64 * u + lane;
    c[u]            = center[j < dim ? j : dim - 1];
  }
}

/** |x_i| (1 when zero) by a wave: per-lane fp64 partial sums in coordinate order, a butterfly. */
__device__ inline double wave_row_norm(const void* x, elem t, int64_t i, int64_t dim, int lane)
{
  double s2 = 0;
  for (int64_t j0 = 0; j0 < dim; j0 += 64 * kLaneChunk) {
    double v[kLaneChunk];
    lane_coords(x, t, i, dim, j0, lane, v);
#pragma unroll
    for (int u = 0; u < kLaneChunk; ++u) { s2 = fma(v[u], v[u], s2); }  // past dim: + 0, exact
  }
  s2 = wave_sum(s2);
  return s2 > 0 ? sqrt(s2) : 1.0;
}

/**
 * The kernels over the rows of a build or an addition (column_sums, max_norm, encode_rows_f16): G
 * lanes per row, 64 / G rows per wave, lane g of a row on the coordinates 4 (u G + g) .. + 3, u < N
 * (one vector load of 4 coordinates each, N of them in flight). (G, N) is sized so that one slice
 * of 4 G N coordinates covers the row (dim up to 1,024); wider rows (MULTI) take slice after slice.
 * Bound by memory, or for small builds by latency and the workgroups' atomics. A wave per row with
 * 16 coordinates per lane loaded 1,024 coordinates of a row of 64. 131,072 fp16 rows of 64: encoding
 * 229 -> 14 us, max_norm 117 -> 10 us; 60,000 x 300 float32, cosine: 163 -> 39 and 93 -> 24 us.
 */
constexpr int kRowThreads = 1024;  // of max_norm and encode_rows_f16: few workgroups, few atomics

template <typename T, int N>
struct row_slice {
  T v[N][4];
};

/** Coordinates of `row` from j0 on for lane g: a whole group of 4 is one load whatever the row's
 *  alignment, the group that crosses the row's end goes one by one; zero past dim. */
template <typename T, int G, int N>
__device__ __forceinline__ row_slice<T, N> load_slice(const T* row, int64_t dim, int64_t j0, int g)
{
  row_slice<T, N> s;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int64_t j = j0 + 4 * (u * G + g);
    if (j + 4 <= dim) {
      __builtin_memcpy(s.v[u], row + j, 4 * sizeof(T));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) { s.v[u][e] = j + e < dim ? row[j + e] : T(0); }
    }
  }
  return s;
}

/** The center's coordinates of a slice (any value past dim). */
template <int G, int N>
__device__ __forceinline__ void center_slice(const double* center, int64_t dim, int64_t j0, int g, double (&c)[N][4])
{
#pragma unroll
  for (int u = 0; u < N; ++u) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t j = j0 + 4 * (u * G + g) + e;
      c[u][e]         = center[j < dim ? j : dim - 1];
    }
  }
}

/** A row's norm and its reciprocal, for quotients. */
struct unit_scale {
  double nrm, inv;
};

/**
 * v / |x|: the product with the correctly rounded reciprocal, corrected once by its exact remainder
 * (Markstein's method), at a fifth of the division's instructions (an index of 240,000 x 300 cosine
 * halves built, searched and dropped: 660 us, 730 with the division). The corrected value is off the
 * quotient by at most 1.5 x 2^-53 ulp before its one rounding, so that it is the division's result
 * unless a quotient lies that close to the midpoint of two doubles: coordinates have at most 24 bits,
 * and of 4e8 quotients, and of the 102 closest to a midpoint found among 8.6e9 norms, every one is
 * the division's.
 */
__device__ __forceinline__ double unit_coord(double v, const unit_scale& s)
{
  const double q = v * s.inv;
  const double r = fma(-q, s.nrm, v);
  return fma(r, s.inv, q);
}

/** |x| of a row (1 when zero) over its G lanes, from its slice (or, MULTI, slice after slice). */
template <typename T, int G, int N, bool MULTI>
__device__ __forceinline__ unit_scale row_scale(const row_slice<T, N>& first, const T* row, int64_t dim, int g)
{
  double s2 = 0;
  row_slice<T, N> x = first;
  for (int64_t j0 = 0;;) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) { s2 = fma(double(x.v[u][e]), double(x.v[u][e]), s2); }
    }
    j0 += 4 * G * N;
    if (!MULTI || j0 >= dim) { break; }
    x = load_slice<T, G, N>(row, dim, j0, g);
  }
  s2 = lanes::sum<G>(s2);
  unit_scale k;
  k.nrm = s2 > 0 ? sqrt(s2) : 1.0;
  k.inv = 1.0 / k.nrm;
  return k;
}

/**
 * sums[j] += the column sums of the rows (of x / |x| when NORM): each wave keeps its lanes' columns
 * in registers over its rows; the block's waves meet in LDS and add each column with one atomic.
 * MULTI (dim above 1,024): the block's wave w takes the columns of slice w of every row of the block.
 * 60,000 x 300 float32 rows, cosine: 845 -> 35 us (a thread per column and serial row norms before).
 */
template <typename T, int G, int N, bool NORM, bool MULTI>
__global__ __launch_bounds__(256) void column_sums_kernel(const T* x, int64_t n, int64_t dim, double* sums)
{
  constexpr int RPW = 64 / G;
  constexpr int C   = 4 * G * N;  // columns of a slice
  __shared__ double part[MULTI ? 1 : 4 * C];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane % G, slot = lane / G;
  const int64_t col0  = MULTI ? int64_t(wave) * C : 0;
  const int64_t first = MULTI ? int64_t(blockIdx.x) : (blockIdx.x * int64_t(4) + wave) * RPW;
  const int64_t step  = MULTI ? int64_t(gridDim.x) : int64_t(gridDim.x) * 4 * RPW;
  double acc[N][4] = {};
  if (col0 < dim) {
    for (int64_t i0 = first; i0 < n; i0 += step) {
      const int64_t i = i0 + slot;
      const bool live = i < n;
      const T* row    = x + (live ? i : n - 1) * dim;
      const auto v    = load_slice<T, G, N>(row, dim, col0, g);
      unit_scale k{1.0, 1.0};
      if constexpr (NORM) {
        k = row_scale<T, G, N, MULTI>(MULTI ? load_slice<T, G, N>(row, dim, 0, g) : v, row, dim, g);
      }
#pragma unroll
      for (int u = 0; u < N; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double d = double(v.v[u][e]);
          acc[u][e] += live ? (NORM ? unit_coord(d, k) : d) : 0.0;
        }
      }
    }
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = 4 * (u * G + g) + e;
      if constexpr (MULTI) {
        if (col0 + j < dim) { atomicAdd(sums + col0 + j, acc[u][e]); }
      } else {
        double a = acc[u][e];
        if constexpr (G <= 16) { a += lanes::exchange<16>(a); }
        if constexpr (G <= 32) { a += lanes::exchange<32>(a); }
        if (slot == 0) { part[wave * C + j] = a; }
      }
    }
  }
  if constexpr (!MULTI) {
    __syncthreads();
    for (int j = threadIdx.x; j < C && j < dim; j += 256) {
      atomicAdd(sums + j, (part[j] + part[C + j]) + (part[2 * C + j] + part[3 * C + j]));
    }
  }
}

/**
 * out[0] raised to the largest |x / |x| - center| (|x - center| without NORM) over the n rows,
 * sqrt_up of the largest fp64 sum, one atomic per workgroup.
 */
template <typename T, int G, int N, bool NORM, bool MULTI>
__global__ __launch_bounds__(kRowThreads) void max_norm_kernel(const T* x, int64_t n, int64_t dim,
                                                       const double* center, double* out)
{
  constexpr int RPW = 64 / G;
  constexpr int C   = 4 * G * N;
  __shared__ double wmax[kRowThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane % G, slot = lane / G;
  double c[N][4];
  if constexpr (!MULTI) { center_slice<G, N>(center, dim, 0, g, c); }
  double m = 0;
  for (int64_t i0 = (blockIdx.x * int64_t(kRowThreads / 64) + wave) * RPW; i0 < n;
       i0 += int64_t(gridDim.x) * (kRowThreads / 64) * RPW) {
    const int64_t i = i0 + slot < n ? i0 + slot : n - 1;
    const T* row    = x + i * dim;
    auto v          = load_slice<T, G, N>(row, dim, 0, g);
    unit_scale k{1.0, 1.0};
    if constexpr (NORM) { k = row_scale<T, G, N, MULTI>(v, row, dim, g); }
    double s = 0;
    for (int64_t j0 = 0;;) {
      if constexpr (MULTI) { center_slice<G, N>(center, dim, j0, g, c); }
#pragma unroll
      for (int u = 0; u < N; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double d = double(v.v[u][e]);
          const double z = (NORM ? unit_coord(d, k) : d) - c[u][e];
          s              = j0 + 4 * (u * G + g) + e < dim ? fma(z, z, s) : s;
        }
      }
      j0 += C;
      if (!MULTI || j0 >= dim) { break; }
      v = load_slice<T, G, N>(row, dim, j0, g);
    }
    m = fmax(m, lanes::sum<G>(s));
  }
  m = lanes::max<64>(m);
  if (lane == 0) { wmax[wave] = m; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kRowThreads / 64; ++w) { m = fmax(m, wmax[w]); }
    atomic_max_pos(out, sqrt_up(m, dim));
  }
}

/**
 * rows[i] = fp16(Z) with Z = (x / |x| - center) / alpha (x / |x| with NORM), subnormals set to 0,
 * zero padded; rowc[i] = -|Z|^2 / 2, raised so that it bounds the term's fp32 accumulation (0 for
 * the inner product); a row with |Z| above kF16Safe is stored as zeros with rowc = +inf (always a
 * candidate). maxima[0] and maxima[1] are raised to the largest |fp16(Z)| and |Z - fp16(Z)|
 * (sqrt_up of the largest sums), one atomic each per workgroup. The fp64 sums are per-lane partials
 * and a butterfly; they only enter bounds that carry their rounding slack. A row that one slice
 * covers is read once and encoded from registers; wider rows (MULTI) are read again for the sums
 * before they are stored.
 */
template <typename T, int G, int N, bool NORM, bool MULTI>
__global__ __launch_bounds__(kRowThreads) void encode_rows_f16_kernel(const T* x, int64_t n, int64_t dim, int halves,
                                                              const double* center, double inv_alpha,
                                                              metric_kind metric, double gamma,
                                                              uint16_t* rows, float* rowc, double* maxima)
{
  constexpr int RPW = 64 / G;
  constexpr int C   = 4 * G * N;
  __shared__ double wmax[2][kRowThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane % G, slot = lane / G;
  double c[N][4];
  if constexpr (!MULTI) { center_slice<G, N>(center, dim, 0, g, c); }
  double mh = 0, me = 0;  // the largest sums of fp16(Z)^2 and (Z - fp16(Z))^2
  for (int64_t i0 = (blockIdx.x * int64_t(kRowThreads / 64) + wave) * RPW; i0 < n;
       i0 += int64_t(gridDim.x) * (kRowThreads / 64) * RPW) {
    const int64_t i = i0 + slot;
    const bool live = i < n;
    const T* row    = x + (live ? i : n - 1) * dim;
    auto v          = load_slice<T, G, N>(row, dim, 0, g);
    unit_scale k{1.0, 1.0};
    if constexpr (NORM) { k = row_scale<T, G, N, MULTI>(v, row, dim, g); }
    double a = 0, nz = 0, ez = 0;
    _Float16 h[N][4];
    for (int64_t j0 = 0;;) {
      if constexpr (MULTI) { center_slice<G, N>(center, dim, j0, g, c); }
#pragma unroll
      for (int u = 0; u < N; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in  = j0 + 4 * (u * G + g) + e < dim;
          const double d = double(v.v[u][e]);
          const double z = in ? ((NORM ? unit_coord(d, k) : d) - c[u][e]) * inv_alpha : 0.0;
          h[u][e]        = to_f16(z);
          const double r = z - double(h[u][e]);  // exact (Sterbenz, or h = 0)
          a  = fma(z, z, a);
          nz = fma(double(h[u][e]), double(h[u][e]), nz);
          ez = fma(r, r, ez);
        }
      }
      j0 += C;
      if (!MULTI || j0 >= dim) { break; }
      v = load_slice<T, G, N>(row, dim, j0, g);
    }
    a  = lanes::sum<G>(a);  // the same value in the lanes of a row
    nz = lanes::sum<G>(nz);
    ez = lanes::sum<G>(ez);
    const bool safe = a <= kF16Safe * kF16Safe;  // false for a NaN too
    if (safe) {
      mh = fmax(mh, nz);
      me = fmax(me, ez);
    }
    if (live) {
      _Float16* dst = reinterpret_cast<_Float16*>(rows + i * halves);
      for (int64_t j0 = 0;;) {
        if constexpr (MULTI) {  // this slice again
          v = load_slice<T, G, N>(row, dim, j0, g);
          center_slice<G, N>(center, dim, j0, g, c);
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int64_t j = j0 + 4 * (u * G + g);
          if constexpr (MULTI) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const double d = double(v.v[u][e]);
              h[u][e] = to_f16(j + e < dim ? ((NORM ? unit_coord(d, k) : d) - c[u][e]) * inv_alpha : 0.0);
            }
          }
          _Float16 o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) { o[e] = safe ? h[u][e] : _Float16(0.0f); }
          if (j < halves) { __builtin_memcpy(__builtin_assume_aligned(dst + j, 8), o, 8); }
        }
        j0 += C;
        if (!MULTI || j0 >= halves) { break; }
      }
      if (g == 0) {
        float f = INFINITY;
        if (safe && metric == metric_kind::inner) {
          f = 0.0f;
        } else if (safe) {
          // row term rounded up: the fp32 accumulation error of this term is folded in (factor
          // 1 - 2g)
          const double t = -(a * (1.0 - 1e-13) / 2.0) * (1.0 - 2.0 * gamma - 1e-10);
          f              = float(t);
          if (double(f) < t) { f = nextafterf(f, INFINITY); }
        }
        rowc[i] = f;
      }
    }
  }
  mh = lanes::max<64>(mh);
  me = lanes::max<64>(me);
  if (lane == 0) {
    wmax[0][wave] = mh;
    wmax[1][wave] = me;
  }
  __syncthreads();
  if (threadIdx.x < 2) {  // thread 0: the rows' norms, thread 1: their rounding errors
    double m = wmax[threadIdx.x][0];
    for (int w = 1; w < kRowThreads / 64; ++w) { m = fmax(m, wmax[threadIdx.x][w]); }
    atomic_max_pos(maxima + threadIdx.x, sqrt_up(m, dim));
  }
}

/**
 * One wave per query, its lanes over the coordinates j = lane, lane + 64, ... (coalesced loads):
 * qrows[i] = fp16(W) with W = (q / |q| - center) / alpha (q / |q| when normalizing), subnormals
 * set to 0, zero padded; qscal[3 i ..] = |W|^2 (lowered by 1e-13), |fp16(W)| and |W - fp16(W)|
 * (raised for the rounding of their sums, sqrt_up). Per-lane fp64 partial sums and a butterfly:
 * the sums only enter bounds that carry these slacks.
 */
template <int N>
__global__ __launch_bounds__(256) void encode_queries_f16_kernel(const void* q, const int32_t* rows,
                                                                 elem t, int64_t nq,
                                                                 int64_t nq_pad, int64_t dim,
                                                                 int halves, bool normalize,
                                                                 const double* center,
                                                                 double inv_alpha, uint16_t* qrows,
                                                                 double* qscal, uint16_t* qpaired)
{
  const int64_t i = blockIdx.x * int64_t(blockDim.x / 64) + (threadIdx.x >> 6);
  const int lane  = threadIdx.x & 63;
  if (i >= nq_pad) { return; }  // uniform over the wave
  _Float16* dst = reinterpret_cast<_Float16*>(qrows + i * halves);
  // half j of the query, and of its paired copy when there is one
  auto put = [&](int64_t j, _Float16 h) {
    dst[j] = h;
    if (qpaired != nullptr) {
      reinterpret_cast<_Float16*>(qpaired)[paired_offset(i, 2 * j, 2 * int64_t(halves)) / 2] = h;
    }
  };
  if (i >= nq) {
    for (int j = lane; j < halves; j += 64) { put(j, _Float16(0.0f)); }
    if (lane == 0) { qscal[3 * i] = qscal[3 * i + 1] = qscal[3 * i + 2] = 0.0; }
    return;
  }
  // a query of at most 64 N coordinates is loaded once, for its norm and its encoding (N, the
  // coordinates per lane and chunk, is sized to the dimension: fewer registers, more waves)
  const int64_t r      = rows != nullptr ? int64_t(rows[i]) : i;  // the caller's query row
  const bool one_chunk = dim <= 64 * N;
  double v[N], c[N];
  double nrm = 1.0;
  if (one_chunk) {
    lane_coords<N>(q, t, r, dim, 0, lane, v);
    lane_center<N>(center, dim, 0, lane, c);
    if (normalize) {
      double s2 = 0;
#pragma unroll
      for (int u = 0; u < N; ++u) { s2 = fma(v[u], v[u], s2); }  // past dim: + 0, exact
      s2  = wave_sum(s2);
      nrm = s2 > 0 ? sqrt(s2) : 1.0;
    }
  } else if (normalize) {
    nrm = wave_row_norm(q, t, r, dim, lane);
  }
  double a = 0, nw = 0, ew = 0;
  for (int64_t j0 = 0; j0 < dim; j0 += 64 * N) {
    if (!one_chunk) {
      lane_coords<N>(q, t, r, dim, j0, lane, v);
      lane_center<N>(center, dim, j0, lane, c);
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int64_t j = j0 + 64 * u + lane;
      if (j < dim) {
        const double w   = (v[u] / nrm - c[u]) * inv_alpha;
        const _Float16 h = query_f16(w);
        const double e   = w - double(h);
        put(j, h);
        a  = fma(w, w, a);
        nw = fma(double(h), double(h), nw);
        ew = fma(e, e, ew);
      }
    }
  }
  for (int64_t j = dim + lane; j < halves; j += 64) { put(j, _Float16(0.0f)); }
  a  = wave_sum(a);
  nw = wave_sum(nw);
  ew = wave_sum(ew);
  if (lane == 0) {
    qscal[3 * i]     = a * (1.0 - 1e-13);
    qscal[3 * i + 1] = sqrt_up(nw, dim);
    qscal[3 * i + 2] = sqrt_up(ew, dim);
  }
}

__global__ void remove_f_kernel(const int64_t* ids, int64_t n, int64_t size, float* rowc,
                                unsigned long long* newly, row_places at)
{
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= n) { return; }
  const int64_t id = ids[t];
  if (id < 0 || id >= size) { return; }
  if (id < at.n_part) { static_cast<float*>(at.part_rowc)[at.part_pos[id]] = -INFINITY; }
  if (at.anchor_stride > 0 && id % at.anchor_stride == 0 && id / at.anchor_stride < at.n_anchor) {
    static_cast<float*>(at.anchor_rowc)[id / at.anchor_stride] = -INFINITY;
  }
  const int old = atomicExch(reinterpret_cast<int*>(rowc + stored_row(at, id)),
                             __float_as_int(-INFINITY));
  if (old != __float_as_int(-INFINITY)) { atomicAdd(newly, 1ull); }
}

}  // namespace

namespace {

/**
 * f(T{}, integral G, integral N, bool_constant NORM, bool_constant MULTI, rows per wave) for the
 * row kernels: 16 lanes per row up to 64 coordinates, 32 up to 128, whole waves above, with as
 * many groups of 4 per lane as cover the row (at most 4: 1,024 coordinates per slice).
 */
template <typename T, bool NORM, typename F>
void with_shape(int64_t dim, F&& f)
{
  using std::integral_constant;
  const auto go = [&](auto g, auto nn, auto multi) {
    f(T{}, g, nn, std::bool_constant<NORM>{}, multi);
  };
  if (dim <= 64) {
    go(integral_constant<int, 16>{}, integral_constant<int, 1>{}, std::false_type{});
  } else if (dim <= 128) {
    go(integral_constant<int, 32>{}, integral_constant<int, 1>{}, std::false_type{});
  } else if (dim <= 256) {
    go(integral_constant<int, 64>{}, integral_constant<int, 1>{}, std::false_type{});
  } else if (dim <= 512) {
    go(integral_constant<int, 64>{}, integral_constant<int, 2>{}, std::false_type{});
  } else if (dim <= 768) {
    go(integral_constant<int, 64>{}, integral_constant<int, 3>{}, std::false_type{});
  } else if (dim <= 1024) {
    go(integral_constant<int, 64>{}, integral_constant<int, 4>{}, std::false_type{});
  } else {
    go(integral_constant<int, 64>{}, integral_constant<int, 4>{}, std::true_type{});
  }
}

template <typename F>
void with_rows(elem t, bool normalize, int64_t dim, F&& f)
{
  if (t == elem::f32) {
    normalize ? with_shape<float, true>(dim, f) : with_shape<float, false>(dim, f);
  } else if (t == elem::bf16) {
    normalize ? with_shape<__bf16, true>(dim, f) : with_shape<__bf16, false>(dim, f);
  } else {
    normalize ? with_shape<_Float16, true>(dim, f) : with_shape<_Float16, false>(dim, f);
  }
}

/**
 * Workgroups of a row kernel of `waves` waves with `rpw` rows each at a time: at most 512, which
 * stride over the rest. Each ends with atomics on the same words: with 2,048 workgroups those took
 * most of max_norm's 28 us over 131,072 rows of 64 fp16 (17 MB).
 */
unsigned row_blocks(int64_t n, int waves, int rpw)
{
  return unsigned(std::min<int64_t>((n + waves * rpw - 1) / (waves * rpw), 512));
}

}  // namespace

void column_sums(const void* x, elem t, int64_t n, int64_t dim, bool normalize, double* sums,
                 hipStream_t stream)
{
  if (n == 0) { return; }
  with_rows(t, normalize, dim, [&](auto v, auto g, auto nn, auto norm, auto multi) {
    using T          = decltype(v);
    constexpr int G  = decltype(g)::value, N = decltype(nn)::value;
    constexpr bool Z = decltype(norm)::value, M = decltype(multi)::value;
    const unsigned b = M ? unsigned(std::min<int64_t>(n, 512)) : row_blocks(n, 4, 64 / G);
    column_sums_kernel<T, G, N, Z, M><<<b, 256, 0, stream>>>(static_cast<const T*>(x), n, dim, sums);
  });
}

void max_norm(const void* x, elem t, int64_t n, int64_t dim, bool normalize, const double* center,
              double* out, hipStream_t stream)
{
  if (n == 0) { return; }
  with_rows(t, normalize, dim, [&](auto v, auto g, auto nn, auto norm, auto multi) {
    using T          = decltype(v);
    constexpr int G  = decltype(g)::value, N = decltype(nn)::value;
    constexpr bool Z = decltype(norm)::value, M = decltype(multi)::value;
    max_norm_kernel<T, G, N, Z, M><<<row_blocks(n, kRowThreads / 64, 64 / G), kRowThreads, 0, stream>>>(static_cast<const T*>(x), n, dim,
                                                                              center, out);
  });
}

void encode_rows_f16(const void* x, elem t, int64_t n, int64_t dim, int halves, bool normalize,
                     const double* center, double inv_alpha, metric_kind metric, double gamma,
                     uint16_t* rows, float* rowc, double* maxima, hipStream_t stream)
{
  if (n == 0) { return; }
  with_rows(t, normalize, dim, [&](auto v, auto g, auto nn, auto norm, auto multi) {
    using T          = decltype(v);
    constexpr int G  = decltype(g)::value, N = decltype(nn)::value;
    constexpr bool Z = decltype(norm)::value, M = decltype(multi)::value;
    encode_rows_f16_kernel<T, G, N, Z, M><<<row_blocks(n, kRowThreads / 64, 64 / G), kRowThreads, 0, stream>>>(
      static_cast<const T*>(x), n, dim, halves, center, inv_alpha, metric, gamma, rows, rowc, maxima);
  });
}

void encode_queries_f16(const void* q, elem t, int64_t nq, int64_t nq_pad, int64_t dim,
                        int halves, bool normalize, const double* center, double inv_alpha,
                        uint16_t* qrows, double* qscal, hipStream_t stream, uint16_t* qpaired,
                        const int32_t* rows)
{
  if (nq_pad == 0) { return; }
  // one wave per query, four per block; a lane's coordinates per chunk sized to the dimension
  const unsigned grid = unsigned((nq_pad + 3) / 4);
  auto go = [&](auto kernel) {
    kernel<<<grid, 256, 0, stream>>>(q, rows, t, nq, nq_pad, dim, halves, normalize, center,
                                     inv_alpha, qrows, qscal, qpaired);
  };
  if (dim <= 256) {
    go(encode_queries_f16_kernel<4>);
  } else if (dim <= 512) {
    go(encode_queries_f16_kernel<8>);
  } else if (dim <= 768) {
    go(encode_queries_f16_kernel<12>);
  } else {
    go(encode_queries_f16_kernel<kLaneChunk>);
  }
}

void remove_rows_f16(const int64_t* ids, int64_t n, int64_t size, float* rowc,
                     unsigned long long* newly_removed, const row_places& at, hipStream_t stream)
{
  if (n == 0) { return; }
  remove_f_kernel<<<blocks_for(n), 256, 0, stream>>>(ids, n, size, rowc, newly_removed, at);
}

void encode_rows_i8(const uint8_t* x, int64_t n, int64_t dim, int row_bytes, uint8_t flip,
                    metric_kind metric, int8_t* codes, int32_t* rowc, hipStream_t stream)
{
  if (n == 0) { return; }
  if (row_bytes == 128) {
    encode_rows_kernel<8><<<blocks_for(n * 8), 256, 0, stream>>>(x, n, dim, row_bytes, flip, metric, codes, rowc);
  } else {
    encode_rows_kernel<16><<<blocks_for(n * 16), 256, 0, stream>>>(x, n, dim, row_bytes, flip, metric, codes, rowc);
  }
}

void encode_queries_i8(const uint8_t* q, int64_t nq, int64_t nq_pad, int64_t dim, int row_bytes,
                       uint8_t flip, int8_t* qcodes, hipStream_t stream, int8_t* qpaired,
                       const int32_t* rows)
{
  const int64_t n = nq_pad * row_bytes;
  if (n == 0) { return; }
  encode_queries_kernel<<<blocks_for(n), 256, 0, stream>>>(q, rows, nq, nq_pad, dim, row_bytes,
                                                           flip, qcodes, qpaired);
}

void remove_rows_i8(const int64_t* ids, int64_t n, int64_t size, int32_t* rowc,
                    unsigned long long* newly_removed, const row_places& at, hipStream_t stream)
{
  if (n == 0) { return; }
  remove_kernel<<<blocks_for(n), 256, 0, stream>>>(ids, n, size, rowc, newly_removed, at);
}

void fill_u32(uint32_t* p, int64_t n, uint32_t v, hipStream_t stream)
{
  if (n == 0) { return; }
  const unsigned b = blocks_for(n) < 4096 ? blocks_for(n) : 4096;
  fill_kernel<uint32_t><<<b, 256, 0, stream>>>(p, n, v);
}

void fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t stream)
{
  if (n == 0) { return; }
  const unsigned b = blocks_for(n) < 4096 ? blocks_for(n) : 4096;
  fill_kernel<int32_t><<<b, 256, 0, stream>>>(p, n, v);
}

void mask_terms(const void* rowc, int64_t n, const void* anchor_rowc, int64_t n_anchor, int64_t stride,
                bool f16, const filter_args& f, void* terms, void* anchor_terms, hipStream_t stream)
{
  if (n + n_anchor == 0) { return; }
  const auto go = [&](auto dead) {
    using V = decltype(dead);
    mask_terms_kernel<V><<<blocks_for(n + n_anchor), 256, 0, stream>>>(
      static_cast<const V*>(rowc), n, static_cast<const V*>(anchor_rowc), n_anchor, stride, f, dead,
      static_cast<V*>(terms), static_cast<V*>(anchor_terms));
  };
  if (f16) {
    go(-float(INFINITY));
  } else {
    go(kDeadRow);
  }
}

void pack_bits(const uint8_t* mask, int64_t n, uint32_t* words, hipStream_t stream)
{
  const int64_t n_out = 2 * ((n + 31) / 32);  // 16-bit halves: the last word is written whole
  if (n_out == 0) { return; }
  pack_bits_kernel<<<blocks_for(n_out), 256, 0, stream>>>(mask, n, reinterpret_cast<uint16_t*>(words), n_out);
}

void iota_i32(int32_t* p, int64_t n, int32_t first, hipStream_t stream)
{
  if (n <= 0) { return; }
  const unsigned b = blocks_for(n) < 4096 ? blocks_for(n) : 4096;
  iota_kernel<<<b, 256, 0, stream>>>(p, n, first);
}

}  // namespace certex_amd
