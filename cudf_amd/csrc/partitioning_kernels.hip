// Kernels of hash partitioning and table concatenation (partitioning.cpp).
//
// hash_partition (cpp/src/partitioning/partitioning.cu:469-711) assigns each
// row the partition `row_hash % num_partitions` and regroups the rows so that
// each partition is contiguous.  Here the regrouping is a stable LSD counting
// sort of the partition numbers, HP_DIGIT_BITS bits per pass, over ranges of
// whole tiles (one workgroup per range):
//   k_hp_ids_count / k_hp_count  digit histogram of every range, written
//                 digit-major so that one exclusive scan of the whole array
//                 gives every range's first output position for every digit;
//   k_hp_scatter  replays its range tile by tile in order; a tile's rows are
//                 ranked stably (ballots inside a wave, per-wave counters
//                 across waves), staged in LDS in output order and written
//                 in runs, so the order inside a partition is the input row
//                 order (deterministic output).
// One pass covers up to 2048 partitions.
#include "partition_common.hpp"
#include "partitioning.hpp"

namespace mig {

namespace {

constexpr int HP_BLOCK = 256;
constexpr int HP_WAVES = HP_BLOCK / 64;
constexpr int HP_TILE_BLOCK = 512;  // counting and scatter kernels
constexpr int HP_TILE_WAVES = HP_TILE_BLOCK / 64;
constexpr int HP_MAX_RPT    = 8;    // rows per thread of a scatter tile (at most)

__device__ __forceinline__ uint64_t lanes_below()
{
  return (1ull << (threadIdx.x & 63)) - 1ull;
}

// IdentityHash of one element (partitioning.cu:738-758): the value converted
// to uint32.  Integers wrap modulo 2^32; floats convert with truncation and
// saturation (NaN and negatives give 0), as the hardware conversion does.
__device__ __forceinline__ uint32_t identity_elem(dcol const& c, int64_t row)
{
  if (!dcol_valid(c, row)) return NULL_HASH;
  auto d = gp(c.data);
  switch (c.storage) {
    case ST_I8: return uint32_t(int32_t(reinterpret_cast<gmem<int8_t const>*>(d)[row]));
    case ST_I16: return uint32_t(int32_t(reinterpret_cast<gmem<int16_t const>*>(d)[row]));
    case ST_I32: return uint32_t(reinterpret_cast<gmem<int32_t const>*>(d)[row]);
    case ST_I64: return uint32_t(uint64_t(reinterpret_cast<gmem<int64_t const>*>(d)[row]));
    case ST_U8:
    case ST_BOOL: return uint32_t(reinterpret_cast<gmem<uint8_t const>*>(d)[row]);
    case ST_U16: return uint32_t(reinterpret_cast<gmem<uint16_t const>*>(d)[row]);
    case ST_U32: return reinterpret_cast<gmem<uint32_t const>*>(d)[row];
    case ST_U64: return uint32_t(reinterpret_cast<gmem<uint64_t const>*>(d)[row]);
    case ST_F32:
    case ST_F64: {
      double const x = c.storage == ST_F32 ? double(reinterpret_cast<gmem<float const>*>(d)[row])
                                           : reinterpret_cast<gmem<double const>*>(d)[row];
      if (!(x > 0.0)) return 0u;
      if (x >= 4294967295.0) return 0xFFFFFFFFu;
      return uint32_t(x);
    }
    default: return 0u;
  }
}

// Rows [r * per, min((r + 1) * per, n)) belong to range r.
__device__ __forceinline__ void range_rows(int64_t n, int64_t per, int64_t r, int64_t& b, int64_t& e)
{
  b = r * per;
  e = b + per < n ? b + per : n;
}

// Digit histogram of a range from LDS, digit-major.
__device__ __forceinline__ void store_hist(uint32_t const* cnt, uint32_t nd, int64_t W, uint32_t* hist)
{
  for (uint32_t d = threadIdx.x; d < nd; d += HP_TILE_BLOCK) gp(hist)[int64_t(d) * W + blockIdx.x] = cnt[d];
}

// Partition numbers of a range's rows and the histogram of their first digit
// (one pass over the hashed columns; a separate counting pass read the
// numbers back, 82 us at 50M rows).  ST is the storage of a single MurmurHash3
// column, or ST_NONE for any columns and either hash: with the storage read
// per row the pass is bound by its scalar and vector instructions (193 us at
// 50M int64 rows, against 157 us with the storage fixed).
template <int ST>
__global__ void __launch_bounds__(HP_TILE_BLOCK)
  k_hp_ids_count(dcol const* __restrict__ cols, int ncols, int64_t n, uint32_t seed, int identity,
                 uint32_t num_partitions, uint32_t* __restrict__ pid, int64_t per, int64_t W, uint32_t dmask,
                 uint32_t* __restrict__ hist)
{
  extern __shared__ uint32_t hp_lds[];
  uint32_t const nd = dmask + 1;
  for (uint32_t d = threadIdx.x; d < nd; d += HP_TILE_BLOCK) hp_lds[d] = 0;
  lds_barrier();
  int64_t b, e;
  range_rows(n, per, blockIdx.x, b, e);
  bool const pow2 = (num_partitions & (num_partitions - 1)) == 0;
  constexpr int U = 4;  // rows in flight per thread
  for (int64_t i0 = b + threadIdx.x; i0 < e; i0 += U * HP_TILE_BLOCK) {
    uint32_t h[U];
#pragma unroll
    for (int u = 0; u < U; u++) h[u] = seed;
    if constexpr (ST != ST_NONE) {
      dcol col    = cols[0];
      col.storage = ST;
#pragma unroll
      for (int u = 0; u < U; u++) {
        int64_t const i = i0 + u * HP_TILE_BLOCK;
        if (i < e) h[u] = hash_combine(seed, elem_hash(col, i, seed));
      }
    }
    for (int c = 0; ST == ST_NONE && c < ncols; c++) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        int64_t const i = i0 + u * HP_TILE_BLOCK;
        if (i >= e) continue;
        h[u] = hash_combine(h[u], identity ? identity_elem(cols[c], i) : elem_hash(cols[c], i, seed));
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      int64_t const i = i0 + u * HP_TILE_BLOCK;
      if (i >= e) continue;
      uint32_t const p = pow2 ? (h[u] & (num_partitions - 1)) : h[u] % num_partitions;
      gp(pid)[i]       = p;
      __hip_atomic_fetch_add(&hp_lds[p & dmask], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  lds_barrier();
  store_hist(hp_lds, nd, W, hist);
}

__global__ void __launch_bounds__(HP_BLOCK)
  k_map_partition_ids(void const* __restrict__ map, int32_t map_storage, int64_t n, uint32_t num_partitions,
                      uint32_t* __restrict__ pid, uint32_t* __restrict__ bad)
{
  int64_t const i = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (i >= n) return;
  int64_t v;
  switch (map_storage) {
    case ST_I8: v = reinterpret_cast<gmem<int8_t const>*>(gp(map))[i]; break;
    case ST_I16: v = reinterpret_cast<gmem<int16_t const>*>(gp(map))[i]; break;
    case ST_I32: v = reinterpret_cast<gmem<int32_t const>*>(gp(map))[i]; break;
    case ST_U8: v = reinterpret_cast<gmem<uint8_t const>*>(gp(map))[i]; break;
    case ST_U16: v = reinterpret_cast<gmem<uint16_t const>*>(gp(map))[i]; break;
    case ST_U32: v = reinterpret_cast<gmem<uint32_t const>*>(gp(map))[i]; break;
    case ST_U64: {
      uint64_t const u = reinterpret_cast<gmem<uint64_t const>*>(gp(map))[i];
      v = u > uint64_t(INT64_MAX) ? -1 : int64_t(u);
      break;
    }
    default: v = reinterpret_cast<gmem<int64_t const>*>(gp(map))[i]; break;
  }
  bool const ok = v >= 0 && v < int64_t(num_partitions);
  if (!ok) atomicOr(bad, 1u);
  gp(pid)[i] = ok ? uint32_t(v) : 0u;
}

__global__ void __launch_bounds__(HP_TILE_BLOCK)
  k_hp_count(uint32_t const* __restrict__ pid, int64_t n, int64_t per, int64_t W, int shift, uint32_t dmask,
             uint32_t* __restrict__ hist)
{
  extern __shared__ uint32_t hp_lds[];
  uint32_t const nd = dmask + 1;
  for (uint32_t d = threadIdx.x; d < nd; d += HP_TILE_BLOCK) hp_lds[d] = 0;
  lds_barrier();
  int64_t b, e;
  range_rows(n, per, blockIdx.x, b, e);
  for (int64_t i = b + threadIdx.x; i < e; i += HP_TILE_BLOCK)
    __hip_atomic_fetch_add(&hp_lds[(gp(pid)[i] >> shift) & dmask], 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
  lds_barrier();
  store_hist(hp_lds, nd, W, hist);
}

// Values of one moved column for the thread's rows of a tile, zero-extended
// (the low half of 16-byte elements when `half` is 0, else the high half).
// Without a row map the tile's rows are t0 + (the thread's places), so the
// offsets fit 32 bits and the base is uniform.
template <int RPT, bool MAPPED>
__device__ __forceinline__ void load_moved(hp_move_col const& mc, int half, int64_t t0, uint32_t live,
                                           uint32_t const (&row)[RPT], uint64_t (&raw)[RPT])
{
  auto from = [&](auto* src, int stride) {
    auto const s = gp(src) + (MAPPED ? 0 : t0 * stride) + half;
#pragma unroll
    for (int k = 0; k < RPT; k++)
      if ((live >> k) & 1u) raw[k] = MAPPED ? s[int64_t(row[k]) * stride] : s[row[k] * uint32_t(stride)];
  };
  switch (mc.width) {
    case 1: from(static_cast<uint8_t const*>(mc.src), 1); break;
    case 2: from(static_cast<uint16_t const*>(mc.src), 1); break;
    case 4: from(static_cast<uint32_t const*>(mc.src), 1); break;
    case 8: from(static_cast<uint64_t const*>(mc.src), 1); break;
    default: from(static_cast<uint64_t const*>(mc.src), 2); break;
  }
}

// The thread's elements into the stage, at their output-order positions.
template <typename T, int RPT, typename V>
__device__ __forceinline__ void stage_tile(uint8_t* stage, uint32_t live, uint32_t const (&lp)[RPT], V const (&v)[RPT])
{
#pragma unroll
  for (int k = 0; k < RPT; k++)
    if ((live >> k) & 1u) reinterpret_cast<T*>(stage)[lp[k]] = T(v[k]);
}

// The staged tile to its place: consecutive threads store consecutive
// elements of a run (`dst` is the output index of position k * block + thread).
template <typename T, int RPT>
__device__ __forceinline__ void store_tile(uint8_t const* stage, int tid, uint32_t const (&dst)[RPT], int total,
                                           void* out, int64_t stride, int64_t off)
{
  auto const o = gp(static_cast<T*>(out)) + off;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    int const j = k * HP_TILE_BLOCK + tid;
    if (j < total) o[int64_t(dst[k]) * stride] = reinterpret_cast<T const*>(stage)[j];
  }
}

// One counting pass over a range.  Bound by memory: every value is read and
// written once.  Storing each element from its own lane (runs of 64 /
// partitions elements) moved 50M 20-byte rows into 256 partitions in 2.9 ms;
// a tile of RPT x 512 rows staged in LDS gives runs of RPT * 512 / partitions
// rows, and since a workgroup owns a contiguous range, consecutive tiles
// continue its runs: 0.83 ms (2.7 TB/s), 0.44 ms into 2 partitions
// (5 TB/s: what is left is the partial lines at the runs' ends).  Tiles of
// 4,096 rows beat 2,048 from 64 partitions on (1.10 against 1.28 ms a call at
// 256, 1.30 against 1.47 at 500) and tie below.  56 KB of LDS at 2048 digits,
// 42 KB at 256, and 102 registers: two workgroups per CU.
template <int RPT, bool MAPPED>
__global__ void __launch_bounds__(HP_TILE_BLOCK)
  k_hp_scatter(uint32_t const* __restrict__ pid_in, uint32_t const* __restrict__ rows_in, int64_t n, int64_t per,
               int64_t W, int shift, int bits, uint32_t const* __restrict__ start, uint32_t* __restrict__ pid_out,
               uint32_t* __restrict__ rows_out, hp_move_col const* __restrict__ move, int nmove)
{
  constexpr int T = RPT * HP_TILE_BLOCK;
  extern __shared__ __attribute__((aligned(16))) uint8_t hp_tile_lds[];
  __shared__ uint32_t wave_sum[HP_TILE_WAVES];
  uint32_t const dmask = (1u << bits) - 1u;
  int const nd         = int(dmask) + 1;
  // the per-wave counters are dead once every row has its position; the
  // value stage takes their place
  int const stage_bytes = T * 8 > HP_TILE_WAVES * nd * 2 ? T * 8 : HP_TILE_WAVES * nd * 2;
  uint8_t* const stage  = hp_tile_lds;
  auto* const next      = reinterpret_cast<uint32_t*>(hp_tile_lds + stage_bytes);  // next output index per digit
  auto* const delta     = next + nd;  // output index minus position, of a digit's rows in this tile
  auto* const sdig      = reinterpret_cast<uint16_t*>(delta + nd);
  volatile uint16_t* const wcnt = reinterpret_cast<uint16_t*>(hp_tile_lds) + (threadIdx.x >> 6) * nd;
  auto* const cnt16             = reinterpret_cast<uint16_t*>(hp_tile_lds);
  for (int d = threadIdx.x; d < nd; d += HP_TILE_BLOCK) next[d] = gp(start)[int64_t(d) * W + blockIdx.x];
  int64_t b, e;
  range_rows(n, per, blockIdx.x, b, e);
  uint64_t const below = lanes_below();
  int const per_t      = (nd + HP_TILE_BLOCK - 1) / HP_TILE_BLOCK;  // digits per thread of the scan
  for (int64_t t0 = b; t0 < e; t0 += T) {
    int const total = e - t0 < T ? int(e - t0) : T;
    // opaque per tile: otherwise the offsets of every row, element width and
    // column are computed once and kept (180 registers instead of 102)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    int const wave = tid >> 6, lane = tid & 63;
    for (int d = lane; d < nd; d += 64) wcnt[d] = 0;
    // wave w takes the rows [w * 64 * RPT, (w + 1) * 64 * RPT) of the tile
    uint32_t p[RPT], row[RPT], lp[RPT];
    uint64_t raw[RPT];
    uint32_t live = 0;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      int const j = (wave * RPT + k) * 64 + lane;
      p[k]        = 0;
      row[k]      = 0;
      if (j < total) {
        live |= 1u << k;
        p[k]   = gp(pid_in)[t0 + j];
        row[k] = MAPPED ? gp(rows_in)[t0 + j] : uint32_t(j);
      }
    }
    // the first column's loads overlap the ranking
    if (nmove > 0) load_moved<RPT, MAPPED>(move[0], 0, t0, live, row, raw);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < RPT; k++) {  // stable rank among the wave's rows of the digit
      bool const valid = (live >> k) & 1u;
      uint32_t const d = (p[k] >> shift) & dmask;
      uint64_t peers   = __ballot(valid);
#pragma unroll
      for (int q = 0; q < HP_DIGIT_BITS; q++) {
        if (q >= bits) break;
        int32_t const bit  = int32_t(d << (31 - q)) >> 31;  // all ones when bit q is set
        uint64_t const set = __ballot(bit != 0);
        peers &= ~(set ^ uint64_t(int64_t(bit)));
      }
      uint32_t first = 0;
      if (valid) first = wcnt[d];
      __builtin_amdgcn_wave_barrier();
      uint32_t const ahead = uint32_t(__popcll(peers & below));
      lp[k]                = first + ahead;
      if (valid && ahead == 0) wcnt[d] = uint16_t(first + uint32_t(__popcll(peers)));
      __builtin_amdgcn_wave_barrier();
    }
    lds_barrier();
    // rows per digit over the waves, then each wave's first position per digit
    uint32_t sum = 0;
    for (int q = 0; q < per_t; q++) {
      int const d = tid * per_t + q;
      if (d < nd)
        for (int w = 0; w < HP_TILE_WAVES; w++) sum += cnt16[w * nd + d];
    }
    uint32_t incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
      uint32_t const y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wave_sum[wave] = incl;
    lds_barrier();
    uint32_t run = incl - sum;
    for (int w = 0; w < wave; w++) run += wave_sum[w];
    for (int q = 0; q < per_t; q++) {
      int const d = tid * per_t + q;
      if (d >= nd) break;
      uint32_t const first = run;
      for (int w = 0; w < HP_TILE_WAVES; w++) {
        uint32_t const c  = cnt16[w * nd + d];
        cnt16[w * nd + d] = uint16_t(run);
        run += c;
      }
      delta[d] = next[d] - first;
      next[d] += run - first;
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      if (!((live >> k) & 1u)) continue;
      uint32_t const d = (p[k] >> shift) & dmask;
      lp[k] += wcnt[d];
      sdig[lp[k]] = uint16_t(d);
    }
    lds_barrier();  // the counters become the stage
    uint32_t dst[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      int const j = k * HP_TILE_BLOCK + tid;
      dst[k]      = j < total ? delta[sdig[j]] + uint32_t(j) : 0u;
    }
    if (pid_out) {  // needed by a later pass or the offsets kernel only
      stage_tile<uint32_t, RPT>(stage, live, lp, p);
      lds_barrier();
      store_tile<uint32_t, RPT>(stage, tid, dst, total, pid_out, 1, 0);
      lds_barrier();
    }
    if (rows_out) {
      if (!MAPPED) {
#pragma unroll
        for (int k = 0; k < RPT; k++) p[k] = uint32_t(t0) + row[k];
      }
      stage_tile<uint32_t, RPT>(stage, live, lp, MAPPED ? row : p);
      lds_barrier();
      store_tile<uint32_t, RPT>(stage, tid, dst, total, rows_out, 1, 0);
      lds_barrier();
    }
    // the last pass moves fixed-width values straight to their place, 16-byte
    // elements as two halves; the next loads are in flight while one is written
    for (int c = 0, half = 0; c < nmove;) {
      hp_move_col const mc = move[c];
#pragma unroll
      for (int k = 0; k < RPT; k++)  // opaque per column, as `tid`
        asm volatile("" : "+v"(lp[k]), "+v"(dst[k]), "+v"(row[k]));
      switch (mc.width) {
        case 1: stage_tile<uint8_t, RPT>(stage, live, lp, raw); break;
        case 2: stage_tile<uint16_t, RPT>(stage, live, lp, raw); break;
        case 4: stage_tile<uint32_t, RPT>(stage, live, lp, raw); break;
        default: stage_tile<uint64_t, RPT>(stage, live, lp, raw); break;
      }
      int const done = half;
      half           = (mc.width == 16) & (half == 0);
      c += half == 0;
      if (c < nmove) load_moved<RPT, MAPPED>(move[c], half, t0, live, row, raw);
      lds_barrier();
      switch (mc.width) {
        case 1: store_tile<uint8_t, RPT>(stage, tid, dst, total, mc.dst, 1, 0); break;
        case 2: store_tile<uint16_t, RPT>(stage, tid, dst, total, mc.dst, 1, 0); break;
        case 4: store_tile<uint32_t, RPT>(stage, tid, dst, total, mc.dst, 1, 0); break;
        case 8: store_tile<uint64_t, RPT>(stage, tid, dst, total, mc.dst, 1, 0); break;
        default: store_tile<uint64_t, RPT>(stage, tid, dst, total, mc.dst, 2, done); break;
      }
      lds_barrier();
    }
    if (!pid_out && !rows_out && nmove == 0) lds_barrier();  // the stage's last barrier otherwise
  }
}

// offsets[q] = first output row of partition q (pid_sorted is non-decreasing).
__global__ void __launch_bounds__(HP_BLOCK)
  k_hp_offsets(uint32_t const* __restrict__ pid_sorted, int64_t n, uint32_t num_partitions,
               int32_t* __restrict__ offsets)
{
  int64_t const i = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (i > n) return;
  int64_t const prev = i == 0 ? -1 : int64_t(gp(pid_sorted)[i - 1]);
  int64_t const cur  = i == n ? int64_t(num_partitions) - 1 : int64_t(gp(pid_sorted)[i]);
  for (int64_t q = prev + 1; q <= cur; q++) gp(offsets)[q] = int32_t(i);
}

// One counting pass: the first row of partition q is the scanned histogram
// entry of digit q for wave 0.
__global__ void __launch_bounds__(HP_BLOCK)
  k_hp_offsets_from_hist(uint32_t const* __restrict__ start, int64_t W, uint32_t num_partitions,
                         int32_t* __restrict__ offsets)
{
  int64_t const q = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (q < num_partitions) gp(offsets)[q] = int32_t(gp(start)[q * W]);
}

template <typename T>
__global__ void __launch_bounds__(HP_BLOCK)
  k_gather_fixed(T const* __restrict__ src, uint32_t const* __restrict__ map, int64_t n, T* __restrict__ dst)
{
  int64_t const i = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (i < n) gp(dst)[i] = gp(src)[gp(map)[i]];
}

// 16-byte elements (DECIMAL128) as two 8-byte halves.
__global__ void __launch_bounds__(HP_BLOCK)
  k_gather_16(uint64_t const* __restrict__ src, uint32_t const* __restrict__ map, int64_t n,
              uint64_t* __restrict__ dst)
{
  int64_t const i = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (i >= n) return;
  int64_t const r = gp(map)[i];
  uint64_t const lo = gp(src)[2 * r], hi = gp(src)[2 * r + 1];
  gp(dst)[2 * i]     = lo;
  gp(dst)[2 * i + 1] = hi;
}

// Null count of a workgroup added once: the per-wave counts are summed in
// LDS first (one atomic per row would serialise on a single address).
__device__ __forceinline__ void add_block_nulls(uint32_t wave_nulls, uint32_t* null_count)
{
  __shared__ uint32_t part[HP_WAVES];
  int const wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) part[wave] = wave_nulls;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < HP_WAVES; w++) t += part[w];
    if (t) atomicAdd(null_count, t);
  }
}

// Output validity: each wave builds two mask words per 64 rows (grid-stride
// over the rows), nulls counted per workgroup.
__global__ void __launch_bounds__(HP_BLOCK)
  k_gather_mask(uint32_t const* __restrict__ mask, int64_t mask_offset, uint32_t const* __restrict__ map,
                int64_t n, uint32_t* __restrict__ out, uint32_t* __restrict__ null_count)
{
  uint32_t nulls = 0;
  for (int64_t base = int64_t(blockIdx.x) * HP_BLOCK; base < n; base += int64_t(gridDim.x) * HP_BLOCK) {
    int64_t const i = base + threadIdx.x;
    bool v = false;
    if (i < n) {
      int64_t const r = int64_t(gp(map)[i]) + mask_offset;
      v               = (gp(mask)[r >> 5] >> (r & 31)) & 1u;
    }
    uint64_t const bal = __ballot(v);
    uint64_t const in  = __ballot(i < n);
    if ((threadIdx.x & 63) == 0 && in) {
      int64_t const word = (i >> 5);
      gp(out)[word]      = uint32_t(bal);
      gp(out)[word + 1]  = uint32_t(bal >> 32);
      nulls += uint32_t(__popcll(in & ~bal));
    }
  }
  add_block_nulls(nulls, null_count);
}

__global__ void __launch_bounds__(HP_BLOCK)
  k_gather_str_sizes(dcol src, uint32_t const* __restrict__ map, int64_t n, int32_t* __restrict__ sizes)
{
  int64_t const i = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (i >= n) return;
  int64_t b, e;
  str_span(src, int64_t(gp(map)[i]), b, e);
  gp(sizes)[i] = int32_t(e - b);
}

// ---- concatenation -----------------------------------------------------------
__device__ __forceinline__ int find_piece(concat_piece const* __restrict__ pieces, int np, int64_t r)
{
  int lo = 0, hi = np - 1;  // last piece with row_start <= r
  while (lo < hi) {
    int const mid = (lo + hi + 1) >> 1;
    if (pieces[mid].row_start <= r) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ void __launch_bounds__(HP_BLOCK)
  k_concat_mask(concat_piece const* __restrict__ pieces, int np, int64_t n, uint32_t* __restrict__ out,
                uint32_t* __restrict__ null_count)
{
  uint32_t nulls = 0;
  for (int64_t base = int64_t(blockIdx.x) * HP_BLOCK; base < n; base += int64_t(gridDim.x) * HP_BLOCK) {
    int64_t const i = base + threadIdx.x;
    bool v = false;
    if (i < n) {
      concat_piece const& P = pieces[find_piece(pieces, np, i)];
      if (P.mask == nullptr) v = true;
      else {
        int64_t const r = i - P.row_start + P.offset;
        v               = (gp(P.mask)[r >> 5] >> (r & 31)) & 1u;
      }
    }
    uint64_t const bal = __ballot(v);
    uint64_t const in  = __ballot(i < n);
    if ((threadIdx.x & 63) == 0 && in) {
      int64_t const word = (i >> 5);
      gp(out)[word]      = uint32_t(bal);
      gp(out)[word + 1]  = uint32_t(bal >> 32);
      nulls += uint32_t(__popcll(in & ~bal));
    }
  }
  add_block_nulls(nulls, null_count);
}

// String offsets of the concatenation: each piece's offsets rebased to where
// its chars land.  offsets[n] = total chars.
__global__ void __launch_bounds__(HP_BLOCK)
  k_concat_str_offsets(concat_piece const* __restrict__ pieces, int np, int64_t n, int64_t total_chars,
                       int32_t* __restrict__ out)
{
  int64_t const i = int64_t(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (i > n) return;
  if (i == n) {
    gp(out)[n] = int32_t(total_chars);
    return;
  }
  concat_piece const& P = pieces[find_piece(pieces, np, i)];
  int64_t const r       = i - P.row_start + P.offset;
  int64_t o;
  if (P.offsets64) o = reinterpret_cast<gmem<int64_t const>*>(gp(P.offsets))[r];
  else o = reinterpret_cast<gmem<int32_t const>*>(gp(P.offsets))[r];
  gp(out)[i] = int32_t(o - P.chars_begin + P.chars_start);
}

// First and last offset of each string piece (its chars range).
__global__ void k_concat_char_ranges(concat_piece const* __restrict__ pieces, int np, int64_t* __restrict__ ranges)
{
  int const k = int(blockIdx.x) * HP_BLOCK + threadIdx.x;
  if (k >= np) return;
  concat_piece const& P = pieces[k];
  int64_t b, e;
  if (P.rows == 0 || P.offsets == nullptr) {  // an empty strings column may have no offsets
    b = 0;
    e = 0;
  } else if (P.offsets64) {
    auto o = reinterpret_cast<gmem<int64_t const>*>(gp(P.offsets));
    b = o[P.offset];
    e = o[P.offset + P.rows];
  } else {
    auto o = reinterpret_cast<gmem<int32_t const>*>(gp(P.offsets));
    b = o[P.offset];
    e = o[P.offset + P.rows];
  }
  gp(ranges)[2 * k]     = b;
  gp(ranges)[2 * k + 1] = e;
}

inline unsigned grid_of(int64_t n) { return unsigned((n + HP_BLOCK - 1) / HP_BLOCK); }
// mask kernels: enough workgroups to fill the device, each looping over rows
inline unsigned mask_grid(int64_t n) { return unsigned(std::min<int64_t>(grid_of(n), 4096)); }

}  // namespace

hp_ranges hp_plan(int64_t n, int bits, int num_cus)
{
  hp_ranges r;
  // two tiles per CU at least: fewer rows take shorter tiles
  r.rpt = HP_MAX_RPT;
  while (r.rpt > 1 && n < int64_t(HP_TILE_BLOCK) * r.rpt * 2 * num_cus) r.rpt /= 2;
  int64_t const tile  = int64_t(HP_TILE_BLOCK) * r.rpt;
  int64_t const tiles = (n + tile - 1) / tile;
  // ranges: six rounds of the two workgroups a CU holds, and a digit-major
  // histogram of at most 2^22 counters
  int64_t const most = std::max<int64_t>(64, std::min<int64_t>(int64_t(num_cus) * 12, (int64_t(1) << 22) >> bits));
  r.per = (tiles + most - 1) / most * tile;
  r.W   = (n + r.per - 1) / r.per;
  return r;
}

void launch_hp_ids_count(dcol const* d_cols, int ncols, int32_t storage, int64_t n, uint32_t seed, bool identity,
                         uint32_t num_partitions, uint32_t* pid, hp_ranges const& R, int bits, uint32_t* hist,
                         hipStream_t s)
{
  if (n == 0) return;
  auto kernel = k_hp_ids_count<ST_NONE>;
  if (ncols == 1 && !identity) switch (storage) {
      case ST_I32:
      case ST_U32: kernel = k_hp_ids_count<ST_U32>; break;
      case ST_I64:
      case ST_U64: kernel = k_hp_ids_count<ST_U64>; break;
      case ST_F32: kernel = k_hp_ids_count<ST_F32>; break;
      case ST_F64: kernel = k_hp_ids_count<ST_F64>; break;
      default: break;
    }
  hipLaunchKernelGGL(kernel, dim3(unsigned(R.W)), dim3(HP_TILE_BLOCK), sizeof(uint32_t) << bits, s, d_cols, ncols, n,
                     seed, identity ? 1 : 0, num_partitions, pid, R.per, R.W, (1u << bits) - 1u, hist);
}

void launch_map_partition_ids(void const* map, int32_t map_storage, int64_t n, uint32_t num_partitions,
                              uint32_t* pid, uint32_t* bad, hipStream_t s)
{
  if (n == 0) return;
  hipLaunchKernelGGL(k_map_partition_ids, dim3(grid_of(n)), dim3(HP_BLOCK), 0, s, map, map_storage, n,
                     num_partitions, pid, bad);
}

void launch_hp_count(uint32_t const* pid, int64_t n, hp_ranges const& R, int shift, int bits, uint32_t* hist,
                     hipStream_t s)
{
  hipLaunchKernelGGL(k_hp_count, dim3(unsigned(R.W)), dim3(HP_TILE_BLOCK), sizeof(uint32_t) << bits, s, pid, n,
                     R.per, R.W, shift, (1u << bits) - 1u, hist);
}

template <int RPT>
static void launch_scatter_form(uint32_t const* pid_in, uint32_t const* rows_in, int64_t n, hp_ranges const& R,
                                int shift, int bits, uint32_t const* start, uint32_t* pid_out, uint32_t* rows_out,
                                hp_move_col const* move, int nmove, hipStream_t s)
{
  constexpr size_t T = size_t(RPT) * HP_TILE_BLOCK;
  size_t const nd    = size_t(1) << bits;
  size_t const lds   = std::max(T * 8, HP_TILE_WAVES * nd * 2) + nd * 8 + T * 2;
  auto const kernel  = rows_in ? k_hp_scatter<RPT, true> : k_hp_scatter<RPT, false>;
  hipLaunchKernelGGL(kernel, dim3(unsigned(R.W)), dim3(HP_TILE_BLOCK), lds, s, pid_in, rows_in, n, R.per, R.W, shift,
                     bits, start, pid_out, rows_out, move, nmove);
}

void launch_hp_scatter(uint32_t const* pid_in, uint32_t const* rows_in, int64_t n, hp_ranges const& R, int shift,
                       int bits, uint32_t const* start, uint32_t* pid_out, uint32_t* rows_out,
                       hp_move_col const* move, int nmove, hipStream_t s)
{
  auto const form = R.rpt == 8 ? launch_scatter_form<8>
                    : R.rpt == 4 ? launch_scatter_form<4>
                    : R.rpt == 2 ? launch_scatter_form<2>
                                 : launch_scatter_form<1>;
  form(pid_in, rows_in, n, R, shift, bits, start, pid_out, rows_out, move, nmove, s);
}

void launch_hp_offsets(uint32_t const* pid_sorted, int64_t n, uint32_t num_partitions, int32_t* offsets,
                       hipStream_t s)
{
  hipLaunchKernelGGL(k_hp_offsets, dim3(grid_of(n + 1)), dim3(HP_BLOCK), 0, s, pid_sorted, n, num_partitions,
                     offsets);
}

void launch_hp_offsets_from_hist(uint32_t const* start, int64_t W, uint32_t num_partitions, int32_t* offsets,
                                 hipStream_t s)
{
  hipLaunchKernelGGL(k_hp_offsets_from_hist, dim3(grid_of(num_partitions)), dim3(HP_BLOCK), 0, s, start, W,
                     num_partitions, offsets);
}

void launch_gather_fixed(void const* src, int width, uint32_t const* map, int64_t n, void* dst, hipStream_t s)
{
  if (n == 0) return;
  dim3 const g(grid_of(n)), b(HP_BLOCK);
  switch (width) {
    case 1: hipLaunchKernelGGL(k_gather_fixed<uint8_t>, g, b, 0, s, static_cast<uint8_t const*>(src), map, n, static_cast<uint8_t*>(dst)); break;
    case 2: hipLaunchKernelGGL(k_gather_fixed<uint16_t>, g, b, 0, s, static_cast<uint16_t const*>(src), map, n, static_cast<uint16_t*>(dst)); break;
    case 4: hipLaunchKernelGGL(k_gather_fixed<uint32_t>, g, b, 0, s, static_cast<uint32_t const*>(src), map, n, static_cast<uint32_t*>(dst)); break;
    case 8: hipLaunchKernelGGL(k_gather_fixed<uint64_t>, g, b, 0, s, static_cast<uint64_t const*>(src), map, n, static_cast<uint64_t*>(dst)); break;
    default: hipLaunchKernelGGL(k_gather_16, g, b, 0, s, static_cast<uint64_t const*>(src), map, n, static_cast<uint64_t*>(dst)); break;
  }
}

void launch_gather_mask(uint32_t const* mask, int64_t mask_offset, uint32_t const* map, int64_t n, uint32_t* out,
                        uint32_t* null_count, hipStream_t s)
{
  if (n == 0) return;
  hipLaunchKernelGGL(k_gather_mask, dim3(mask_grid(n)), dim3(HP_BLOCK), 0, s, mask, mask_offset, map, n, out,
                     null_count);
}

void launch_gather_str_sizes(dcol const& src, uint32_t const* map, int64_t n, int32_t* sizes, hipStream_t s)
{
  if (n == 0) return;
  hipLaunchKernelGGL(k_gather_str_sizes, dim3(grid_of(n)), dim3(HP_BLOCK), 0, s, src, map, n, sizes);
}

void launch_concat_mask(concat_piece const* pieces, int np, int64_t n, uint32_t* out, uint32_t* null_count,
                        hipStream_t s)
{
  if (n == 0) return;
  hipLaunchKernelGGL(k_concat_mask, dim3(mask_grid(n)), dim3(HP_BLOCK), 0, s, pieces, np, n, out, null_count);
}

void launch_concat_char_ranges(concat_piece const* pieces, int np, int64_t* ranges, hipStream_t s)
{
  hipLaunchKernelGGL(k_concat_char_ranges, dim3(grid_of(np)), dim3(HP_BLOCK), 0, s, pieces, np, ranges);
}

void launch_concat_str_offsets(concat_piece const* pieces, int np, int64_t n, int64_t total_chars, int32_t* out,
                               hipStream_t s)
{
  hipLaunchKernelGGL(k_concat_str_offsets, dim3(grid_of(n + 1)), dim3(HP_BLOCK), 0, s, pieces, np, n,
                     total_chars, out);
}

}  // namespace mig
