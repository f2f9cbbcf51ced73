// Kernels of the sort-based aggregations (MEDIAN, QUANTILE) on gfx950.
//
// The reference sorts the keys, then sorts each group's values and reads the
// quantiles off the sorted segments (sort/sort_helper.cu, sort/
// group_quantiles.cu:30-80, quantiles/quantiles_util.hpp).  Here the rows are
// labelled with their group by the hash table and brought into group order by
// a stable LSD counting sort of the group numbers.  The values' order-
// preserving bits are then sorted group by group on the chip
// (k_sort_groups_wave, k_sort_groups_block) while every group has at most
// SORT_BLOCK_ROWS rows, else by more passes of the counting sort, over (group,
// null, value) with the bits written by k_quantile_keys.  k_group_quantiles
// reads every group's segment.
#include "device_ops.hpp"
#include "kernels.hpp"

namespace mig {

namespace {

constexpr int SBLOCK = 256;

__device__ __forceinline__ bool is_signed_st(int32_t st)
{
  return st == ST_I8 || st == ST_I16 || st == ST_I32 || st == ST_I64;
}

// Order-preserving bits of element `row` (32 bits for elements of up to 4
// bytes, 64 bits otherwise): signed integers with the sign bit flipped,
// unsigned integers unchanged, floats with NaN above +inf and -0.0 as 0.0.
__device__ __forceinline__ uint64_t order_bits(dcol const& c, int64_t row)
{
  auto const d = gp(c.data);
  switch (c.storage) {
    case ST_I8: return uint32_t(int32_t(reinterpret_cast<gmem<int8_t const>*>(d)[row])) ^ 0x80000000u;
    case ST_I16: return uint32_t(int32_t(reinterpret_cast<gmem<int16_t const>*>(d)[row])) ^ 0x80000000u;
    case ST_I32: return uint32_t(reinterpret_cast<gmem<int32_t const>*>(d)[row]) ^ 0x80000000u;
    case ST_I64: return uint64_t(reinterpret_cast<gmem<int64_t const>*>(d)[row]) ^ (1ull << 63);
    case ST_U8:
    case ST_BOOL: return d[row];
    case ST_U16: return reinterpret_cast<gmem<uint16_t const>*>(d)[row];
    case ST_U32: return reinterpret_cast<gmem<uint32_t const>*>(d)[row];
    case ST_U64: return reinterpret_cast<gmem<uint64_t const>*>(d)[row];
    case ST_F32: {
      float const x = reinterpret_cast<gmem<float const>*>(d)[row];
      if (isnan(x)) return 0xFFFFFFFFu;
      uint32_t const b = __float_as_uint(x == 0.0f ? 0.0f : x);
      return (b >> 31) ? ~b : (b | 0x80000000u);
    }
    default: {  // ST_F64
      double const x = reinterpret_cast<gmem<double const>*>(d)[row];
      if (isnan(x)) return ~0ull;
      uint64_t const b = uint64_t(__double_as_longlong(x == 0.0 ? 0.0 : x));
      return (b >> 63) ? ~b : (b | (1ull << 63));
    }
  }
}

__global__ void __launch_bounds__(SBLOCK)
  k_quantile_keys(dcol v, int64_t n, uint32_t* __restrict__ lo, uint32_t* __restrict__ hi,
                  uint32_t* __restrict__ null_flag)
{
  int64_t const r = int64_t(blockIdx.x) * SBLOCK + threadIdx.x;
  if (r >= n) return;
  bool const valid = dcol_valid(v, r);
  uint64_t const o = valid ? order_bits(v, r) : 0ull;
  gp(lo)[r]        = uint32_t(o);
  if (hi) gp(hi)[r] = uint32_t(o >> 32);
  if (null_flag) gp(null_flag)[r] = valid ? 0u : 1u;
}

// ---------------------------------------------------------------------------
// Sorting inside groups.  Nine counting passes (64-bit values, nulls, group)
// over 4M rows in 50,000 groups took 1.3 ms; gathering the order bits and
// sorting each group where it is held takes 0.07 ms (a call
// with MEDIAN, MAX and NUNIQUE 2.45 -> 1.43 ms).

// The value of lane (own lane ^ d), d a power of two.
__device__ __forceinline__ uint64_t lane_xor(uint64_t x, int d)
{
  uint32_t const lo = uint32_t(x), hi = uint32_t(x >> 32);
  switch (d) {  // constants after unrolling; DPP where it has the pattern
    case 1:
      return (uint64_t(uint32_t(__builtin_amdgcn_mov_dpp(int(hi), 0xB1, 0xF, 0xF, true))) << 32) |
             uint32_t(__builtin_amdgcn_mov_dpp(int(lo), 0xB1, 0xF, 0xF, true));
    case 2:
      return (uint64_t(uint32_t(__builtin_amdgcn_mov_dpp(int(hi), 0x4E, 0xF, 0xF, true))) << 32) |
             uint32_t(__builtin_amdgcn_mov_dpp(int(lo), 0x4E, 0xF, 0xF, true));
    case 8:
      return (uint64_t(uint32_t(__builtin_amdgcn_mov_dpp(int(hi), 0x128, 0xF, 0xF, true))) << 32) |
             uint32_t(__builtin_amdgcn_mov_dpp(int(lo), 0x128, 0xF, 0xF, true));
    default: return (uint64_t(uint32_t(__shfl_xor(int(hi), d, 64))) << 32) | uint32_t(__shfl_xor(int(lo), d, 64));
  }
}

// Bitonic sort of a wave's 64 * R values, element lane * R + r in v[r], so
// that steps of distance below R stay inside a lane; descending when `down`.
template <int R>
__device__ __forceinline__ void wave_sort(uint64_t (&v)[R], bool down)
{
  int const lane = int(threadIdx.x & 63u);
#pragma unroll
  for (int k = 2; k <= 64 * R; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        // the block of k elements is ascending (the last one: as asked)
        bool const up = k == 64 * R ? !down : (k < R ? (r & k) == 0 : (lane & (k / R)) == 0);
        if (j < R) {
          if (r & j) continue;
          uint64_t const a = v[r], b = v[r | j];
          bool const swap  = up ? b < a : a < b;
          v[r]             = swap ? b : a;
          v[r | j]         = swap ? a : b;
        } else {
          uint64_t const o    = lane_xor(v[r], j / R);
          bool const keep_min = ((lane & (j / R)) == 0) == up;
          v[r]                = (o < v[r]) == keep_min ? o : v[r];
        }
      }
    }
  }
}

// The last steps of a bitonic merge, inside 64 * R values with element
// r * 64 + lane in v[r].
template <int R>
__device__ __forceinline__ void wave_merge(uint64_t (&v)[R], bool down)
{
  int const lane = int(threadIdx.x & 63u);
#pragma unroll
  for (int j = 32 * R; j > 0; j >>= 1) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (j >= 64) {
        if (r & (j / 64)) continue;
        uint64_t const a = v[r], b = v[r | (j / 64)];
        bool const swap  = down ? a < b : b < a;
        v[r]             = swap ? b : a;
        v[r | (j / 64)]  = swap ? a : b;
      } else {
        uint64_t const o    = lane_xor(v[r], j);
        bool const keep_min = ((lane & j) == 0) != down;
        v[r]                = (o < v[r]) == keep_min ? o : v[r];
      }
    }
  }
}

// Order bits of the rows at places [b, e) of the group order; nulls and places
// past the end take the largest value, so that the first `valid` sorted places
// hold the valid values (equal bits are equal values).
struct group_sort {
  dcol v;
  uint32_t const* perm;
  uint32_t* lo;
  uint32_t* hi;   // 8-byte values
  uint32_t* nul;  // null flags, or nullptr when the column has no nulls
};

__device__ __forceinline__ uint64_t group_value(group_sort const& J, int64_t at, int64_t e, uint32_t& valid)
{
  bool ok    = at < e;
  uint64_t o = ~0ull;
  if (ok) {
    int64_t const row = gp(J.perm)[at];
    ok                = dcol_valid(J.v, row);
    if (ok) o = order_bits(J.v, row);
  }
  valid += uint32_t(__popcll(__builtin_amdgcn_ballot_w64(ok)));
  return o;
}

__device__ __forceinline__ void group_store(group_sort const& J, int64_t at, int64_t e, uint64_t o, bool null)
{
  if (at >= e) return;
  gp(J.lo)[at] = uint32_t(o);
  if (J.hi) gp(J.hi)[at] = uint32_t(o >> 32);
  if (J.nul) gp(J.nul)[at] = null ? 1u : 0u;
}

constexpr int SORT_WAVE_ROWS = 512;  // a wave's registers hold 8 values per lane

template <int R>
__device__ __forceinline__ void sort_group(group_sort const& J, int64_t b, int64_t e)
{
  int const lane = int(threadIdx.x & 63u);
  uint64_t v[R];
  uint32_t valid = 0;
#pragma unroll
  for (int r = 0; r < R; r++) v[r] = group_value(J, b + r * 64 + lane, e, valid);
  wave_sort<R>(v, false);
#pragma unroll
  for (int r = 0; r < R; r++) group_store(J, b + lane * R + r, e, v[r], uint32_t(lane * R + r) >= valid);
}

// One wave per group of at most SORT_WAVE_ROWS rows.
__global__ void __launch_bounds__(SBLOCK) k_sort_groups_wave(group_sort J, int32_t const* __restrict__ off, int64_t G)
{
  int64_t const g = int64_t(blockIdx.x) * (SBLOCK / 64) + (threadIdx.x >> 6);
  if (g >= G) return;
  int64_t const b = gp(off)[g], e = gp(off)[g + 1];
  int64_t const n = e - b;
  if (n <= 64) sort_group<1>(J, b, e);
  else if (n <= 128) sort_group<2>(J, b, e);
  else if (n <= 256) sort_group<4>(J, b, e);
  else if (n <= SORT_WAVE_ROWS) sort_group<8>(J, b, e);
}

// One workgroup per listed group (up to SORT_BLOCK_ROWS rows): chunks of
// SORT_WAVE_ROWS sorted in registers, alternately up and down, then merged;
// only the steps across chunks go through LDS.
constexpr int SORT_BLOCK = 512;

__global__ void __launch_bounds__(SORT_BLOCK)
  k_sort_groups_block(group_sort J, int32_t const* __restrict__ off, uint32_t const* __restrict__ list)
{
  __shared__ uint64_t x[SORT_BLOCK_ROWS];
  __shared__ uint32_t valid_sh;
  constexpr int R = SORT_WAVE_ROWS / 64;
  int64_t const g = gp(list)[blockIdx.x];
  int64_t const b = gp(off)[g], e = gp(off)[g + 1];
  int size = 2 * SORT_WAVE_ROWS;
  while (size < int(e - b)) size *= 2;
  int const chunks = size / SORT_WAVE_ROWS, wave = int(threadIdx.x >> 6), lane = int(threadIdx.x & 63u);
  if (threadIdx.x == 0) valid_sh = 0;
  __syncthreads();
  uint32_t valid = 0;
  for (int c = wave; c < chunks; c += SORT_BLOCK / 64) {
    uint64_t v[R];
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = group_value(J, b + c * SORT_WAVE_ROWS + r * 64 + lane, e, valid);
    wave_sort<R>(v, (c & 1) != 0);
#pragma unroll
    for (int r = 0; r < R; r++) x[c * SORT_WAVE_ROWS + lane * R + r] = v[r];
  }
  if (lane == 0) __hip_atomic_fetch_add(&valid_sh, valid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  __syncthreads();
  valid = valid_sh;
  for (int k = 2 * SORT_WAVE_ROWS; k <= size; k *= 2) {
    for (int j = k / 2; j >= SORT_WAVE_ROWS; j /= 2) {
      for (int i = threadIdx.x; i < size / 2; i += SORT_BLOCK) {
        int const at     = ((i & ~(j - 1)) << 1) | (i & (j - 1));
        uint64_t const p = x[at], q = x[at + j];
        if (((at & k) == 0) == (q < p)) {
          x[at]     = q;
          x[at + j] = p;
        }
      }
      __syncthreads();
    }
    for (int c = wave; c < chunks; c += SORT_BLOCK / 64) {
      uint64_t v[R];
      int const c0 = c * SORT_WAVE_ROWS;
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = x[c0 + r * 64 + lane];
      wave_merge<R>(v, (c0 & k) != 0);
      if (k < size) {
#pragma unroll
        for (int r = 0; r < R; r++) x[c0 + r * 64 + lane] = v[r];
      } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
          int const i = c0 + r * 64 + lane;
          group_store(J, b + i, e, v[r], uint32_t(i) >= valid);
        }
      }
    }
    __syncthreads();
  }
}

// Groups by how they are sorted: counts[0] listed ones (more than
// SORT_WAVE_ROWS rows), counts[1] those past SORT_BLOCK_ROWS.
__global__ void __launch_bounds__(SBLOCK)
  k_list_groups(int32_t const* __restrict__ off, int64_t G, uint32_t* __restrict__ list, uint32_t* counts)
{
  int64_t const g = int64_t(blockIdx.x) * SBLOCK + threadIdx.x;
  if (g >= G) return;
  int32_t const n = gp(off)[g + 1] - gp(off)[g];
  if (n <= SORT_WAVE_ROWS) return;
  if (n > SORT_BLOCK_ROWS) astore(counts + 1, 1u);
  gp(list)[__hip_atomic_fetch_add(gp(counts), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)] = uint32_t(g);
}

// The element of storage `st` whose order bits are (lo, hi), as double.
__device__ __forceinline__ double order_value(int32_t st, uint32_t lo, uint32_t hi)
{
  switch (st) {
    case ST_I8:
    case ST_I16:
    case ST_I32: return double(int32_t(lo ^ 0x80000000u));
    case ST_I64: return double(int64_t(((uint64_t(hi) << 32) | lo) ^ (1ull << 63)));
    case ST_U64: return double((uint64_t(hi) << 32) | lo);
    case ST_F32: {
      uint32_t const b = (lo >> 31) ? (lo & 0x7FFFFFFFu) : ~lo;
      return double(__uint_as_float(b));
    }
    case ST_F64: {
      uint64_t const o = (uint64_t(hi) << 32) | lo;
      uint64_t const b = (o >> 63) ? (o & ~(1ull << 63)) : ~o;
      return __longlong_as_double(int64_t(b));
    }
    default: return double(lo);  // unsigned up to 32 bits, bool
  }
}

__device__ __forceinline__ int64_t order_int64(uint32_t lo, uint32_t hi)
{
  return int64_t(((uint64_t(hi) << 32) | lo) ^ (1ull << 63));
}

// quantile_index and select_quantile_data of quantiles/quantiles_util.hpp:
// v = q * (n - 1) with q clamped to [0, 1]; LINEAR and MIDPOINT in double,
// MIDPOINT of int64 values by halves (no overflow); the arithmetic is not
// contracted into fused multiply-adds.
__global__ void __launch_bounds__(SBLOCK)
  k_group_quantiles(uint32_t const* __restrict__ ord_lo, uint32_t const* __restrict__ ord_hi,
                    uint32_t const* __restrict__ null_flag, int32_t const* __restrict__ off, int64_t G,
                    int32_t storage, double const* __restrict__ q, int32_t nq, int32_t interp,
                    double* __restrict__ out, uint32_t* __restrict__ out_mask)
{
#pragma clang fp contract(off)
  int64_t const g = int64_t(blockIdx.x) * SBLOCK + threadIdx.x;
  if (g >= G) return;
  int64_t const b = gp(off)[g], e = gp(off)[g + 1];
  // valid values come first in the segment (the null flag sorts above them)
  int64_t m = e - b;
  if (null_flag) {
    int64_t lo = b, hi = e;
    while (lo < hi) {
      int64_t const mid = (lo + hi) >> 1;
      if (gp(null_flag)[mid]) hi = mid;
      else lo = mid + 1;
    }
    m = lo - b;
  }
  auto elem = [&](int64_t i) {
    return order_value(storage, gp(ord_lo)[b + i], ord_hi ? gp(ord_hi)[b + i] : 0u);
  };
  for (int32_t j = 0; j < nq; j++) {
    int64_t const o = g * nq + j;
    double r        = 0.0;
    if (m > 0) {
      double qq = gp(q)[j];
      qq        = qq < 0.0 ? 0.0 : (qq > 1.0 ? 1.0 : qq);
      double const v   = qq * double(m - 1);
      int64_t const lo = int64_t(floor(v)), hi = int64_t(ceil(v)), ne = int64_t(rint(v));
      double const f   = v - double(lo);
      switch (interp) {
        case MIG_INTERP_LINEAR: {
          double const a = elem(lo), c = elem(hi);
          double const x = (1.0 - f) * a;
          double const y = f * c;
          r              = x + y;
          break;
        }
        case MIG_INTERP_LOWER: r = elem(lo); break;
        case MIG_INTERP_HIGHER: r = elem(hi); break;
        case MIG_INTERP_NEAREST: r = elem(ne); break;
        default: {  // MIDPOINT
          if (storage == ST_I64) {
            int64_t const a = order_int64(gp(ord_lo)[b + lo], gp(ord_hi)[b + lo]);
            int64_t const c = order_int64(gp(ord_lo)[b + hi], gp(ord_hi)[b + hi]);
            int64_t const half = a / 2 + c / 2, rest = a % 2 + c % 2;
            r = double(half) + double(rest) * 0.5;
          } else {
            r = elem(lo) / 2 + elem(hi) / 2;
          }
          break;
        }
      }
      __hip_atomic_fetch_or(out_mask + (o >> 5), 1u << (o & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    gp(out)[o] = r;
  }
}

__global__ void __launch_bounds__(SBLOCK)
  k_first_rows(uint32_t const* __restrict__ map, int32_t const* __restrict__ off, int64_t G, uint32_t* __restrict__ rep)
{
  int64_t const g = int64_t(blockIdx.x) * SBLOCK + threadIdx.x;
  if (g < G) gp(rep)[g] = gp(map)[gp(off)[g]];
}

// Rows the null policy dropped (NO_GROUP) take group number G.
__global__ void __launch_bounds__(SBLOCK) k_clamp_groups(uint32_t* __restrict__ gid, int64_t n, uint32_t G)
{
  int64_t const r = int64_t(blockIdx.x) * SBLOCK + threadIdx.x;
  if (r < n && gp(gid)[r] > G) gp(gid)[r] = G;
}

int64_t sgrid(int64_t n) { return (n + SBLOCK - 1) / SBLOCK; }

}  // namespace

void launch_quantile_keys(dcol const& v, int64_t n, uint32_t* lo, uint32_t* hi, uint32_t* null_flag, hipStream_t s)
{
  if (n > 0) hipLaunchKernelGGL(k_quantile_keys, dim3(sgrid(n)), dim3(SBLOCK), 0, s, v, n, lo, hi, null_flag);
}

void launch_list_groups(int32_t const* off, int64_t G, uint32_t* list, uint32_t* counts, hipStream_t s)
{
  if (G > 0) hipLaunchKernelGGL(k_list_groups, dim3(sgrid(G)), dim3(SBLOCK), 0, s, off, G, list, counts);
}

void launch_sort_groups(dcol const& v, uint32_t const* perm, int32_t const* off, int64_t G, uint32_t const* list,
                        int64_t listed, uint32_t* lo, uint32_t* hi, uint32_t* nul, hipStream_t s)
{
  if (G <= 0) return;
  group_sort const J{v, perm, lo, hi, nul};
  hipLaunchKernelGGL(k_sort_groups_wave, dim3((G + SBLOCK / 64 - 1) / (SBLOCK / 64)), dim3(SBLOCK), 0, s, J, off, G);
  if (listed > 0) hipLaunchKernelGGL(k_sort_groups_block, dim3(listed), dim3(SORT_BLOCK), 0, s, J, off, list);
}

void launch_group_quantiles(uint32_t const* ord_lo, uint32_t const* ord_hi, uint32_t const* null_flag,
                            int32_t const* off, int64_t G, int32_t storage, double const* q, int32_t nq,
                            int32_t interp, double* out, uint32_t* out_mask, hipStream_t s)
{
  if (G > 0)
    hipLaunchKernelGGL(k_group_quantiles, dim3(sgrid(G)), dim3(SBLOCK), 0, s, ord_lo, ord_hi, null_flag, off, G,
                       storage, q, nq, interp, out, out_mask);
}

void launch_clamp_groups(uint32_t* gid, int64_t n, uint32_t G, hipStream_t s)
{
  if (n > 0) hipLaunchKernelGGL(k_clamp_groups, dim3(sgrid(n)), dim3(SBLOCK), 0, s, gid, n, G);
}

void launch_first_rows(uint32_t const* map, int32_t const* off, int64_t G, uint32_t* rep, hipStream_t s)
{
  if (G > 0) hipLaunchKernelGGL(k_first_rows, dim3(sgrid(G)), dim3(SBLOCK), 0, s, map, off, G, rep);
}

}  // namespace mig
