// gfx950 kernels of the hash group-by.
//
// Row hashing follows cudf/table/experimental/row_operators.cuh:1858-1883 and
// the MurmurHash3_x86_32 element hash; equality follows row_operators.cuh:
// 1352-1364, 1429-1448 (nulls equal, NaN equal NaN, -0.0 equal 0.0).  The
// accumulate step replaces compute_single_pass_aggs_fn
// (groupby/hash/groupby_kernels.cuh:98-105) and the variance pass replaces
// var_hash_functor (groupby/hash/multi_pass_kernels.cuh:74-111).
#include "device_ops.hpp"
#include "lds_accumulate.hpp"

#include <map>
#include <mutex>
#include <type_traits>

namespace mig {

constexpr int BLOCK = 256;

// ---------------------------------------------------------------------------
// public row hash: cudf::hashing::murmurhash3_x86_32 (src/hash/murmurhash3_x86_32.cu:34-57)
__global__ void __launch_bounds__(BLOCK)
  k_hash_rows(dcol const* __restrict__ cols, int ncols, int64_t n, uint32_t seed, uint32_t* out)
{
  for (int64_t r = int64_t(blockIdx.x) * BLOCK + threadIdx.x; r < n; r += int64_t(gridDim.x) * BLOCK)
    out[r] = row_hash(cols, ncols, r, seed);
}

void launch_hash_rows(dcol const* d_cols, int ncols, int64_t n, uint32_t seed, uint32_t* out,
                      hipStream_t s)
{
  if (n <= 0) return;
  int64_t blocks = (n + BLOCK - 1) / BLOCK;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_hash_rows, dim3(blocks), dim3(BLOCK), 0, s, d_cols, ncols, n, seed, out);
}

// ---------------------------------------------------------------------------
// cardinality sample: row hashes of `nsample` evenly strided rows
// A pseudo-random permutation of [0, n): a 4-round Feistel network on the
// smallest even number of bits covering n (round function: MurmurHash3's
// finaliser), walking the cycle until the value falls below n.
__device__ __forceinline__ int64_t sample_row(int64_t i, int64_t n)
{
  int bits = 2;
  while ((int64_t(1) << bits) < n) bits += 2;
  int const half      = bits / 2;
  uint64_t const mask = (uint64_t(1) << half) - 1;
  uint64_t x          = uint64_t(i);
  for (int walk = 0; walk < 256; walk++) {
    uint64_t l = x >> half, r = x & mask;
    for (uint32_t round = 0; round < 4; round++) {
      uint64_t const f = mm_fmix32(uint32_t(r) * 0x9E3779B9u + round * 0x85EBCA6Bu + uint32_t(r >> 32));
      uint64_t const t = l ^ (f & mask);
      l                = r;
      r                = t;
    }
    x = (l << half) | r;
    if (x < uint64_t(n)) return int64_t(x);
  }
  return (i * 7919) % n;  // not reached in practice: the cycle through i < n returns below n
}

// Distinct hashes of the sampled rows.  A workgroup first counts its rows'
// hashes in LDS, so a hot hash costs one global atomic per workgroup instead
// of one per row, and everything that used to be counted with atomics on one
// address (rows, distinct hashes, the highest multiplicity) is read off the
// finished table by k_sample_freqs.  65,536 rows: 28-52 us with uniform keys
// and 151 us with Zipf(1.1) keys before, 16-25 us now.
constexpr int SAMPLE_LDS   = 2 * SAMPLE_BLOCK;  // at most half filled

// Add `count` rows of hash `h` to the table of (rows << 32) | hash slots
// (0 = empty, mask + 1 slots, never full).
template <int SCOPE, typename P>
__device__ __forceinline__ void sample_add(P table, uint32_t mask, uint32_t h, uint32_t count)
{
  uint32_t s = mm_fmix32(h) & mask;
  for (uint32_t k = 0; k <= mask; k++) {
    uint64_t cur = __hip_atomic_load(table + s, __ATOMIC_RELAXED, SCOPE);
    if (cur == 0 &&
        __hip_atomic_compare_exchange_strong(table + s, &cur, (uint64_t(count) << 32) | h, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, SCOPE))
      return;
    if (uint32_t(cur) == h) {
      __hip_atomic_fetch_add(table + s, uint64_t(count) << 32, __ATOMIC_RELAXED, SCOPE);
      return;
    }
    s = (s + 1) & mask;
  }
}

__global__ void __launch_bounds__(SAMPLE_BLOCK)
  k_sample_hash(gb_params const* __restrict__ Pp, int64_t n, int64_t nsample, uint64_t* table, uint32_t table_mask,
                int64_t* __restrict__ range)
{
  __shared__ uint64_t part[SAMPLE_LDS];
  __shared__ int64_t low[SAMPLE_BLOCK / 64], high[SAMPLE_BLOCK / 64];
  int64_t lo = INT64_MAX, hi = INT64_MIN;
  gb_params const& P = *Pp;
  for (int i = threadIdx.x; i < SAMPLE_LDS; i += SAMPLE_BLOCK) part[i] = 0;
  __syncthreads();
  int64_t const i = int64_t(blockIdx.x) * SAMPLE_BLOCK + threadIdx.x;
  if (i < nsample) {
    // every row when the sample covers the input; otherwise a uniformly random
    // subset (sample index -> row through a pseudo-random permutation of
    // [0, n)): evenly strided rows would all fall in different runs of sorted
    // or clustered keys and look like all-distinct keys, and rows drawn with
    // replacement would repeat rows and look like repeated keys
    int64_t const row = nsample < n ? sample_row(i, n) : i;
    // rows the group-by drops (null keys under EXCLUDE) are not part of the
    // population whose distinct keys are estimated
    if (!(P.skip_null_keys && any_key_null(P, row)))
      sample_add<__HIP_MEMORY_SCOPE_WORKGROUP>(part, SAMPLE_LDS - 1u, row_hash(P.keys, P.num_keys, row, 0), 1u);
    if (range && dcol_valid(P.keys[0], row)) {
      uint64_t c[1] = {load_fixed_bits(P.keys[0], row)};
      canon_rows(P.key_storage, c);
      lo = hi = int64_t(c[0]);
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, int64_t(__shfl_down(lo, o, 64)));
    hi = max(hi, int64_t(__shfl_down(hi, o, 64)));
  }
  if ((threadIdx.x & 63) == 0) {
    low[threadIdx.x >> 6]  = lo;
    high[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  if (range && threadIdx.x == 0) {
    for (int w = 1; w < SAMPLE_BLOCK / 64; w++) {
      lo = min(lo, low[w]);
      hi = max(hi, high[w]);
    }
    gp(range)[2 * blockIdx.x]     = lo;
    gp(range)[2 * blockIdx.x + 1] = hi;
  }
  for (int s = threadIdx.x; s < SAMPLE_LDS; s += SAMPLE_BLOCK) {
    uint64_t const e = part[s];
    if (e != 0) sample_add<__HIP_MEMORY_SCOPE_AGENT>(gp(table), table_mask, uint32_t(e), uint32_t(e >> 32));
  }
}

// What the finished table says, per workgroup b at out[b * SAMPLE_STATS]: rows
// sampled, distinct hashes, the highest multiplicity, the hashes seen once and
// twice, and those seen at least SAMPLE_HOT_MIN << j times.
__global__ void __launch_bounds__(SAMPLE_BLOCK)
  k_sample_freqs(uint64_t const* __restrict__ table, uint32_t slots, uint32_t* __restrict__ out)
{
  __shared__ uint32_t red[SAMPLE_STATS][SAMPLE_BLOCK / 64];
  uint32_t v[SAMPLE_STATS] = {0};
  for (uint32_t i = blockIdx.x * SAMPLE_BLOCK + threadIdx.x; i < slots; i += gridDim.x * SAMPLE_BLOCK) {
    uint32_t const c = uint32_t(gp(table)[i] >> 32);
    v[0] += c;
    v[1] += c != 0u;
    v[2] = max(v[2], c);
    v[3] += c == 1u;
    v[4] += c == 2u;
#pragma unroll
    for (int j = 0; j < SAMPLE_HOT_LEVELS; j++) v[5 + j] += c >= uint32_t(SAMPLE_HOT_MIN << j);
  }
  for (int o = 32; o > 0; o >>= 1)
    for (int j = 0; j < SAMPLE_STATS; j++) {
      uint32_t const y = __shfl_down(v[j], o, 64);
      v[j]             = j == 2 ? max(v[j], y) : v[j] + y;
    }
  if ((threadIdx.x & 63) == 0)
    for (int j = 0; j < SAMPLE_STATS; j++) red[j][threadIdx.x >> 6] = v[j];
  __syncthreads();
  if (threadIdx.x < SAMPLE_STATS) {
    int const j = threadIdx.x;
    uint32_t t  = 0;
    for (int w = 0; w < SAMPLE_BLOCK / 64; w++) t = j == 2 ? max(t, red[j][w]) : t + red[j][w];
    gp(out)[blockIdx.x * SAMPLE_STATS + j] = t;
  }
}

void launch_sample_hash(gb_params const* dP, int64_t n, int64_t nsample, uint64_t* table, uint32_t table_mask,
                        uint32_t* stats, int64_t* range, hipStream_t s)
{
  int64_t const blocks = sample_blocks(nsample);
  hipLaunchKernelGGL(k_sample_hash, dim3(blocks), dim3(SAMPLE_BLOCK), 0, s, dP, n, nsample, table, table_mask, range);
  hipLaunchKernelGGL(k_sample_freqs, dim3(SAMPLE_STAT_BLOCKS), dim3(SAMPLE_BLOCK), 0, s, table, table_mask + 1u, stats);
}

// ---------------------------------------------------------------------------
// state initialisation: table, row counts, special flags and accumulator identities

__global__ void __launch_bounds__(BLOCK) k_init_state(gb_params const* __restrict__ Pp)
{
  gb_params const& P = *Pp;
  int64_t const total = int64_t(P.cap) + 2;
  int const which = blockIdx.y;  // 0 = table, 1 = row counts, 2.. = fields
  int64_t const stride = int64_t(gridDim.x) * BLOCK;
  int64_t i = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (which == 0) {
    if (P.key_mode == KM_INLINE) {
      for (int64_t j = i; j < int64_t(P.cap); j += stride) P.slot_keys[j] = EMPTY_KEY;
    } else {
      for (int64_t j = i; j < int64_t(P.cap); j += stride) P.slot_rows[j] = EMPTY_ROW;
    }
    if (i == 0) {
      P.special[0] = 0;
      P.special[1] = 0;
      *P.overflow  = 0;
    }
  } else if (which == 1) {
    if (P.slot_count)
      for (int64_t j = i; j < total; j += stride) *count_at(P, j) = 0;
  } else {
    field_desc const& F = P.fields[which - 2];
    uint64_t const id = field_identity(F.kind);
    if (F.width == 8) {
      for (int64_t j = i; j < total; j += stride) *reinterpret_cast<uint64_t*>(field_at(F, j)) = id;
    } else {
      for (int64_t j = i; j < total; j += stride) *reinterpret_cast<uint32_t*>(field_at(F, j)) = uint32_t(id);
    }
  }
}

void launch_init_state(gb_params const* dP, gb_params const& hP, hipStream_t s)
{
  int64_t total = int64_t(hP.cap) + 2;
  int64_t blocks = (total + BLOCK - 1) / BLOCK;
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(k_init_state, dim3(blocks, 2 + hP.num_fields), dim3(BLOCK), 0, s, dP);
}

// ---------------------------------------------------------------------------
// hash table probing
__device__ __forceinline__ void mark_special(gb_params const& P, int which)
{
  if (aload(&P.special[which]) == 0u) astore(&P.special[which], 1u);
}

// Insert-or-find of an inline key; returns the slot, or -1 on overflow.
__device__ __forceinline__ int64_t insert_inline(gb_params const& P, uint64_t key, uint32_t h)
{
  if (key == EMPTY_KEY) {
    mark_special(P, 0);
    return int64_t(P.cap);
  }
  uint64_t s = h & P.cap_mask;
  for (uint32_t i = 0; i < P.probe_limit; i++) {
    if ((i & 63u) == 63u && aload(P.overflow) != 0) return -1;  // the table is being rebuilt
    uint64_t cur = aload(&P.slot_keys[s]);
    if (cur == key) return int64_t(s);
    if (cur == EMPTY_KEY) {
      uint64_t old = acas64(&P.slot_keys[s], EMPTY_KEY, key);
      if (old == EMPTY_KEY || old == key) return int64_t(s);
    }
    s = (s + 1) & P.cap_mask;
  }
  astore(P.overflow, 1);
  return -1;
}

__device__ __forceinline__ int64_t find_inline(gb_params const& P, uint64_t key, uint32_t h)
{
  if (key == EMPTY_KEY) return int64_t(P.cap);
  uint64_t s = h & P.cap_mask;
  for (uint32_t i = 0; i < P.probe_limit; i++) {
    uint64_t cur = P.slot_keys[s];
    if (cur == key) return int64_t(s);
    if (cur == EMPTY_KEY) return -1;
    s = (s + 1) & P.cap_mask;
  }
  return -1;
}

__device__ __forceinline__ int64_t insert_general(gb_params const& P, int64_t row, uint32_t h)
{
  uint64_t const mine = (uint64_t(h) << 32) | uint32_t(row);
  uint64_t s = h & P.cap_mask;
  for (uint32_t i = 0; i < P.probe_limit; i++) {
    if ((i & 63u) == 63u && aload(P.overflow) != 0) return -1;  // the table is being rebuilt
    uint64_t cur = aload(&P.slot_rows[s]);
    if (cur == EMPTY_ROW) {
      uint64_t old = acas64(&P.slot_rows[s], EMPTY_ROW, mine);
      if (old == EMPTY_ROW) return int64_t(s);
      cur = old;
    }
    if (uint32_t(cur >> 32) == h && rows_equal(P, int64_t(uint32_t(cur)), row)) return int64_t(s);
    s = (s + 1) & P.cap_mask;
  }
  astore(P.overflow, 1);
  return -1;
}

__device__ __forceinline__ int64_t find_general(gb_params const& P, int64_t row, uint32_t h)
{
  uint64_t s = h & P.cap_mask;
  for (uint32_t i = 0; i < P.probe_limit; i++) {
    uint64_t cur = P.slot_rows[s];
    if (cur == EMPTY_ROW) return -1;
    if (uint32_t(cur >> 32) == h && rows_equal(P, int64_t(uint32_t(cur)), row)) return int64_t(s);
    s = (s + 1) & P.cap_mask;
  }
  return -1;
}

// One row per hash and workgroup inserts its key (thousands of rows share a hot
// key, and atomics on one address queue up: 50 us with every row inserting).
// Of two keys with one hash, either may be left out.
__global__ void __launch_bounds__(SAMPLE_BLOCK)
  k_insert_hot(gb_params const* __restrict__ Pp, int64_t n, int64_t nsample, uint64_t const* __restrict__ table,
               uint32_t table_mask, uint32_t at_least)
{
  __shared__ uint64_t seen[SAMPLE_LDS];  // (1 << 32) | hash, 0 = empty
  gb_params const& P = *Pp;
  for (int i = threadIdx.x; i < SAMPLE_LDS; i += SAMPLE_BLOCK) seen[i] = 0;
  __syncthreads();
  int64_t const i = int64_t(blockIdx.x) * SAMPLE_BLOCK + threadIdx.x;
  if (i >= nsample) return;
  int64_t const row = nsample < n ? sample_row(i, n) : i;
  dcol const& kc    = P.keys[0];
  if (!dcol_valid(kc, row)) return;
  uint64_t const bits = load_fixed_bits(kc, row);
  uint32_t const h    = hash_combine(0u, hash_fixed_bits(kc.storage, bits, 0u));
  uint64_t const mine = (1ull << 32) | h;
  uint32_t s          = mm_fmix32(h) & uint32_t(SAMPLE_LDS - 1);
  for (;;) {  // at most half filled
    uint64_t cur = 0;
    if (__hip_atomic_compare_exchange_strong(seen + s, &cur, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED, WG_SCOPE)) break;
    if (cur == mine) return;
    s = (s + 1) & uint32_t(SAMPLE_LDS - 1);
  }
  s = mm_fmix32(h) & table_mask;
  for (uint32_t k = 0; k <= table_mask; k++) {
    uint64_t const cur = gp(table)[s];
    if (cur == 0) return;
    if (uint32_t(cur) == h) {
      if (uint32_t(cur >> 32) >= at_least && bits != EMPTY_KEY) (void)insert_inline(P, bits, h);
      return;
    }
    s = (s + 1) & table_mask;
  }
}

void launch_insert_hot(gb_params const* dP, int64_t n, int64_t nsample, uint64_t const* table, uint32_t table_mask,
                       uint32_t at_least, hipStream_t s)
{
  hipLaunchKernelGGL(k_insert_hot, dim3(sample_blocks(nsample)), dim3(SAMPLE_BLOCK), 0, s, dP, n, nsample, table,
                     table_mask, at_least);
}

__global__ void __launch_bounds__(BLOCK) k_pack_valid(uint8_t const* __restrict__ bytes, int64_t n, uint32_t* words)
{
  int64_t const i    = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  uint64_t const bal = __ballot(i < n && gp(bytes)[i] != 0);
  int const lane     = threadIdx.x & 63;
  if (i < n && (lane & 31) == 0) gp(words)[i >> 5] = lane ? uint32_t(bal >> 32) : uint32_t(bal);
}

void launch_pack_valid(uint8_t const* bytes, int64_t n, uint32_t* words, hipStream_t s)
{
  if (n > 0) hipLaunchKernelGGL(k_pack_valid, dim3((n + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, bytes, n, words);
}

// Slot of `row`'s group (inserting it when INSERT), or -1 when the row is
// skipped (null key under EXCLUDE) or the table overflowed.
template <int KM, bool INSERT>
__device__ __forceinline__ int64_t locate(gb_params const& P, int64_t row)
{
  if constexpr (KM == KM_INLINE) {
    dcol const& kc = P.keys[0];
    if (!dcol_valid(kc, row)) {
      if (P.skip_null_keys) return -1;
      if (INSERT) mark_special(P, 1);
      return int64_t(P.cap) + 1;
    }
    uint64_t const bits = load_fixed_bits(kc, row);
    uint32_t const h    = hash_combine(0u, hash_fixed_bits(kc.storage, bits, 0u));
    return INSERT ? insert_inline(P, bits, h) : find_inline(P, bits, h);
  } else {
    if (P.skip_null_keys && any_key_null(P, row)) return -1;
    uint32_t const h = row_hash(P.keys, P.num_keys, row, 0u);
    return INSERT ? insert_general(P, row, h) : find_general(P, row, h);
  }
}

// ---------------------------------------------------------------------------
// accumulate one row into the group's accumulators (apply_field: device_ops.hpp)

// ARGMIN / ARGMAX: is row r's value a better choice than row o's?  The
// reference keeps the first of equal values to reach the target
// (aggregation.cuh:440-490); here equal values take the smaller row, and a
// NaN only wins when both are NaN (NaN compares false in the reference, so a
// number there is never replaced by a NaN), which makes the result
// deterministic.
__device__ __forceinline__ bool arg_better(dcol const& c, int32_t kind, int64_t r, int64_t o)
{
  int cmp = 0;
  if (c.storage == ST_STRING) {  // bytewise, then by length (string_view::compare)
    int64_t rb, re, ob, oe;
    str_span(c, r, rb, re);
    str_span(c, o, ob, oe);
    int64_t const lr = re - rb, lo = oe - ob, m = lr < lo ? lr : lo;
    auto const d     = gp(c.data);
    for (int64_t i = 0; i < m && cmp == 0; i++) {
      uint8_t const x = d[rb + i], y = d[ob + i];
      cmp             = x < y ? -1 : (x > y ? 1 : 0);
    }
    if (cmp == 0) cmp = lr < lo ? -1 : (lr > lo ? 1 : 0);
    if (cmp != 0) return kind == FK_ARGMIN ? cmp < 0 : cmp > 0;
    return r < o;
  }
  loaded_value const a = load_value(c, r), b = load_value(c, o);
  if (c.storage == ST_F32 || c.storage == ST_F64) {
    bool const an = isnan(a.d), bn = isnan(b.d);
    if (an != bn) return bn;  // a number beats a NaN
    if (!an) cmp = a.d < b.d ? -1 : (a.d > b.d ? 1 : 0);
  } else if (is_unsigned_storage_dev(c.storage)) {
    cmp = uint64_t(a.i) < uint64_t(b.i) ? -1 : (uint64_t(a.i) > uint64_t(b.i) ? 1 : 0);
  } else {
    cmp = a.i < b.i ? -1 : (a.i > b.i ? 1 : 0);
  }
  if (cmp != 0) return kind == FK_ARGMIN ? cmp < 0 : cmp > 0;
  return r < o;
}

// Compare-and-swap loop on the group's row index (aggregation.cuh:440-490).
__device__ __forceinline__ void arg_update(field_desc const& F, int64_t slot, dcol const& c, int64_t row)
{
  auto* a      = reinterpret_cast<unsigned int*>(field_at(F, slot));
  uint32_t cur = __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (cur == 0xFFFFFFFFu || arg_better(c, F.kind, row, int64_t(cur))) {
    uint32_t const prev = atomicCAS(a, cur, uint32_t(row));
    if (prev == cur) break;
    cur = prev;
  }
}

__device__ __forceinline__ void update_row(gb_params const& P, int64_t slot, int64_t row)
{
  if (P.need_count_all) aadd(count_at(P, slot), 1u);
  for (int vc = 0; vc < P.num_vals; vc++) {
    int const fb = P.val_field_begin[vc], fe = P.val_field_begin[vc + 1];
    if (fb == fe) continue;
    dcol const& c = P.vals[vc];
    if (!dcol_valid(c, row)) continue;
    loaded_value const v = load_value(c, row);
    for (int f = fb; f < fe; f++) {
      field_desc const& F = P.fields[f];
      if (F.kind == FK_ARGMIN || F.kind == FK_ARGMAX) arg_update(F, slot, c, row);
      else apply_field(F, slot, v);
    }
  }
}

template <int KM>
__global__ void __launch_bounds__(BLOCK) k_aggregate_global(gb_params const* __restrict__ Pp)
{
  gb_params const& P = *Pp;
  int64_t const n = P.num_rows;
  for (int64_t row = int64_t(blockIdx.x) * BLOCK + threadIdx.x; row < n;
       row += int64_t(gridDim.x) * BLOCK) {
    if (aload(P.overflow) != 0) break;  // the call rebuilds a larger table: stop early
    int64_t const slot = locate<KM, true>(P, row);
    if (slot < 0) continue;
    update_row(P, slot, row);
  }
}

static int64_t row_grid(int64_t n, int num_cus, int per_cu)
{
  int64_t blocks = (n + BLOCK - 1) / BLOCK;
  int64_t cap = int64_t(num_cus) * per_cu;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  return blocks;
}

template <int KM>
__global__ void __launch_bounds__(BLOCK) k_aggregate_global_combined(gb_params const* __restrict__ Pp);

// Whether every accumulator of the plan combines partials (the wave-combined
// form of k_aggregate_global) and slot numbers fit its 26-bit sort keys.
static bool combinable(gb_params const& hP)
{
  if (hP.cap + 2 >= (uint64_t(1) << 26)) return false;
  for (int f = 0; f < hP.num_fields; f++) {
    switch (hP.fields[f].kind) {
      case FK_ARGMIN:
      case FK_ARGMAX:
      case FK_NUNIQUE:
      case FK_NUNIQUE_NULLS:
      case FK_NTH: return false;
      default: break;
    }
  }
  return true;
}

void launch_aggregate(gb_params const* dP, gb_params const& hP, int num_cus, hipStream_t s)
{
  if (hP.num_rows <= 0) return;
  int64_t blocks = row_grid(hP.num_rows, num_cus, 16);
  if (combinable(hP)) {
    if (hP.key_mode == KM_INLINE)
      hipLaunchKernelGGL(k_aggregate_global_combined<KM_INLINE>, dim3(blocks), dim3(BLOCK), 0, s, dP);
    else
      hipLaunchKernelGGL(k_aggregate_global_combined<KM_GENERAL>, dim3(blocks), dim3(BLOCK), 0, s, dP);
    return;
  }
  if (hP.key_mode == KM_INLINE)
    hipLaunchKernelGGL(k_aggregate_global<KM_INLINE>, dim3(blocks), dim3(BLOCK), 0, s, dP);
  else
    hipLaunchKernelGGL(k_aggregate_global<KM_GENERAL>, dim3(blocks), dim3(BLOCK), 0, s, dP);
}

// ---------------------------------------------------------------------------
// Group labels for the sort-based path: every row's slot in the device-wide
// table (UINT32_MAX for a dropped row), then each slot's rank among the
// occupied slots (the compaction order), then every row's group number.
template <int KM>
__global__ void __launch_bounds__(BLOCK) k_label_rows(gb_params const* __restrict__ Pp, uint32_t* __restrict__ slot_of_row)
{
  gb_params const& P = *Pp;
  int64_t const n    = P.num_rows;
  for (int64_t row = int64_t(blockIdx.x) * BLOCK + threadIdx.x; row < n; row += int64_t(gridDim.x) * BLOCK) {
    int64_t const slot = locate<KM, true>(P, row);
    gp(slot_of_row)[row] = slot < 0 ? 0xFFFFFFFFu : uint32_t(slot);
  }
}

void launch_label_rows(gb_params const* dP, gb_params const& hP, int num_cus, uint32_t* slot_of_row, hipStream_t s)
{
  if (hP.num_rows <= 0) return;
  int64_t blocks = row_grid(hP.num_rows, num_cus, 16);
  if (hP.key_mode == KM_INLINE)
    hipLaunchKernelGGL(k_label_rows<KM_INLINE>, dim3(blocks), dim3(BLOCK), 0, s, dP, slot_of_row);
  else
    hipLaunchKernelGGL(k_label_rows<KM_GENERAL>, dim3(blocks), dim3(BLOCK), 0, s, dP, slot_of_row);
}

__global__ void __launch_bounds__(BLOCK)
  k_rank_slots(uint32_t const* __restrict__ map, int64_t G, uint32_t* __restrict__ rank_of_slot)
{
  int64_t const j = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (j < G) gp(rank_of_slot)[gp(map)[j]] = uint32_t(j);
}

__global__ void __launch_bounds__(BLOCK)
  k_gid_of_rows(uint32_t const* __restrict__ slot_of_row, uint32_t const* __restrict__ rank_of_slot, int64_t n,
                uint32_t dropped, uint32_t* __restrict__ gid)
{
  int64_t const r = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (r >= n) return;
  uint32_t const s = gp(slot_of_row)[r];
  gp(gid)[r]       = s == 0xFFFFFFFFu ? dropped : gp(rank_of_slot)[s];
}

void launch_group_numbers(uint32_t const* map, int64_t G, uint32_t const* slot_of_row, int64_t n,
                          uint32_t* rank_of_slot, uint32_t* gid, hipStream_t s)
{
  if (G > 0) hipLaunchKernelGGL(k_rank_slots, dim3((G + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, map, G, rank_of_slot);
  if (n > 0)
    hipLaunchKernelGGL(k_gid_of_rows, dim3((n + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, slot_of_row, rank_of_slot, n,
                       uint32_t(G), gid);
}

// ---------------------------------------------------------------------------
// second pass: sum of squared deviations from the group mean (VARIANCE / STD)
__device__ __forceinline__ double field_as_double(field_desc const& F, int64_t slot)
{
  switch (F.kind) {
    case FK_PROD_I64: return double(*reinterpret_cast<int64_t const*>(field_at(F, slot)));
    case FK_PROD_F32: return double(*reinterpret_cast<float const*>(field_at(F, slot)));
    case FK_PROD_F64: return *reinterpret_cast<double const*>(field_at(F, slot));
    case FK_SUM_I64: return double(*reinterpret_cast<int64_t const*>(field_at(F, slot)));
    case FK_SUM_F32: return double(*reinterpret_cast<float const*>(field_at(F, slot)));
    case FK_SUM_F64: return *reinterpret_cast<double const*>(field_at(F, slot));
    case FK_COUNT: return double(*reinterpret_cast<uint32_t const*>(field_at(F, slot)));
    default: return 0.0;
  }
}

// Count accumulator `f`, or the group row count when f == -2 (columns
// without nulls count their values with the row count).
__device__ __forceinline__ uint32_t count_of(gb_params const& P, int32_t f, int64_t slot)
{
  return f == -2 ? *count_at(P, slot) : *reinterpret_cast<uint32_t const*>(field_at(P.fields[f], slot));
}

template <int KM>
__global__ void __launch_bounds__(BLOCK) k_second_pass(gb_params const* __restrict__ Pp)
{
  gb_params const& P = *Pp;
  int64_t const n = P.num_rows;
  for (int64_t row = int64_t(blockIdx.x) * BLOCK + threadIdx.x; row < n;
       row += int64_t(gridDim.x) * BLOCK) {
    int64_t slot = -2;
    for (int vc = 0; vc < P.num_vals; vc++) {
      int const fb = P.val_field_begin[vc], fe = P.val_field_begin[vc + 1];
      bool has_m2 = false;
      for (int f = fb; f < fe; f++) has_m2 |= (P.fields[f].kind == FK_M2);
      if (!has_m2) continue;
      dcol const& c = P.vals[vc];
      if (!dcol_valid(c, row)) continue;
      if (slot == -2) slot = locate<KM, false>(P, row);
      if (slot < 0) break;
      loaded_value const v = load_value(c, row);
      for (int f = fb; f < fe; f++) {
        field_desc const& F = P.fields[f];
        if (F.kind != FK_M2) continue;
        double const cnt  = double(count_of(P, F.aux_count, slot));
        double const mean = field_as_double(P.fields[F.aux_sum], slot) / cnt;
        double const d    = v.d - mean;
        gadd_f64(reinterpret_cast<double*>(field_at(F, slot)), d * d);
      }
    }
  }
}

void launch_second_pass(gb_params const* dP, gb_params const& hP, int num_cus, hipStream_t s)
{
  if (hP.num_rows <= 0) return;
  int64_t blocks = row_grid(hP.num_rows, num_cus, 16);
  if (hP.key_mode == KM_INLINE)
    hipLaunchKernelGGL(k_second_pass<KM_INLINE>, dim3(blocks), dim3(BLOCK), 0, s, dP);
  else
    hipLaunchKernelGGL(k_second_pass<KM_GENERAL>, dim3(blocks), dim3(BLOCK), 0, s, dP);
}

// ---------------------------------------------------------------------------
// Few groups (one fixed-width key): per-workgroup partial tables in LDS, merged
// once per workgroup.  A global atomic per row and field would run at 24 G/s on
// this device (7 G/s on a thousand addresses); LDS atomics take 5-12 ns per
// wave and CU.  Rows whose key finds no room go to the device-wide table.
//
// Bound by instruction issue and LDS operations, so: descriptors come from the
// lanes of a register (lds_plan); rows that don't count go to a spare slot of
// their lane instead of a branch; integer keys of a range that fits take the
// slot of their value (no hash, no probe); the other tables are a third full and
// a thread's rows probe together; float32 sums are kept in float64 (an LDS
// float32 add takes 80 ns, a float64 one 12).  One workgroup of 1024 threads
// per CU: 40M rows, 1,000 keys, 6 accumulators over 2 nullable columns 917 us
// before, 200 us now (500 us by probing); 1M rows 67 us before, 13 us now.
constexpr int LBLOCK   = 1024;
constexpr int LDS_ROWS = 4;  // rows per thread in flight in k_aggregate_lds

// First slot of hash `h` in an LDS table of S slots (any S: the high word of
// the product, so the table is sized by its groups, not to a power of two).
__device__ __forceinline__ uint32_t lds_first_slot(uint32_t h, int S) { return __umulhi(h, uint32_t(S)); }

// Hash of key bits for the LDS tables, whose places nobody else sees: a third
// of the row hash's (quarter-rate) multiplications.
__device__ __forceinline__ uint32_t lds_key_hash(uint64_t bits)
{
  uint32_t h = uint32_t(bits) * 0x9E3779B1u + uint32_t(bits >> 32) * 0x85EBCA77u;
  h ^= h >> 15;
  return h * 0xC2B2AE3Du;
}

// Insert `key` into an LDS open-addressing table of S u64 slots whose free
// slots hold `empty`, with at most `limit` keys (`fill` counts them); returns
// its slot, or -1 when the table is full.
__device__ __forceinline__ int lds_insert_any(uint64_t* tkeys, uint32_t* fill, uint64_t key, uint32_t h,
                                              uint64_t empty, int S, uint32_t limit)
{
  uint32_t s = lds_first_slot(h, S);
  for (int p = 0; p < S; p++) {
    uint64_t const cur = __hip_atomic_load(tkeys + s, __ATOMIC_RELAXED, WG_SCOPE);
    if (cur == key) return int(s);
    if (cur == empty) {
      if (__hip_atomic_load(fill, __ATOMIC_RELAXED, WG_SCOPE) >= limit) return -1;
      uint64_t expected = empty;
      if (__hip_atomic_compare_exchange_strong(tkeys + s, &expected, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               WG_SCOPE)) {
        __hip_atomic_fetch_add(fill, 1u, __ATOMIC_RELAXED, WG_SCOPE);
        return int(s);
      }
      if (expected == key) return int(s);
    }
    s = s + 1 == uint32_t(S) ? 0u : s + 1;
  }
  return -1;
}

// lds_insert_any for the rows of `pending` (bit u: keys[u], hash h[u]), their
// probes interleaved so that every round has all of them in flight; a row
// whose key finds no room gets -1, the others their slot.
template <int N>
__device__ __forceinline__ void lds_insert_rows(uint64_t* tkeys, uint32_t* fill, uint64_t const (&keys)[N],
                                                uint32_t const (&h)[N], uint32_t pending, int S, uint32_t limit,
                                                int (&id)[N])
{
  uint32_t pos[N];
#pragma unroll
  for (int u = 0; u < N; u++) pos[u] = lds_first_slot(h[u], S);
  // S rounds pass every slot.  `limit` is soft (threads that read the count
  // together all insert), so a small table can fill up: a key that is in it is
  // found, any other row leaves after the S rounds with -1.
  for (int p = 0; p < S && pending != 0; p++) {
    uint64_t cur[N];
#pragma unroll
    for (int u = 0; u < N; u++)
      if ((pending >> u) & 1u) cur[u] = __hip_atomic_load(tkeys + pos[u], __ATOMIC_RELAXED, WG_SCOPE);
#pragma unroll
    for (int u = 0; u < N; u++) {
      if (!((pending >> u) & 1u)) continue;
      bool done = cur[u] == keys[u];
      if (cur[u] == EMPTY_KEY) {
        if (__hip_atomic_load(fill, __ATOMIC_RELAXED, WG_SCOPE) >= limit) {
          pos[u] = 0xffffffffu;
          done   = true;
        } else {
          uint64_t expected = EMPTY_KEY;
          if (__hip_atomic_compare_exchange_strong(tkeys + pos[u], &expected, keys[u], __ATOMIC_RELAXED,
                                                   __ATOMIC_RELAXED, WG_SCOPE)) {
            __hip_atomic_fetch_add(fill, 1u, __ATOMIC_RELAXED, WG_SCOPE);
            done = true;
          } else {
            done = expected == keys[u];
          }
        }
      }
      if (done) {
        id[u] = int(pos[u]);
        pending &= ~(1u << u);
      } else {
        pos[u] = pos[u] + 1 == uint32_t(S) ? 0u : pos[u] + 1;
      }
    }
  }
#pragma unroll
  for (int u = 0; u < N; u++)
    if ((pending >> u) & 1u) id[u] = -1;
}

// Validity words of the rows r0 + u * LBLOCK (row e - 1 past the end); bit
// (r0 + offset) & 31 of word u is row u's (LBLOCK is a multiple of 32).
template <int N>
__device__ __forceinline__ void load_valid_words(gmem<uint32_t const>* mask, uint32_t offset, uint32_t r0, uint32_t e,
                                                 uint32_t (&w)[N])
{
#pragma unroll
  for (int u = 0; u < N; u++) {
    w[u] = mask[(min(r0 + uint32_t(u) * LBLOCK, e - 1u) + offset) >> 5];  // rows and offsets below 2^31
  }
}

// A column's element values and validity words of one chunk, as loaded.
struct lds_column {
  uint64_t c[LDS_ROWS];
  uint32_t w[LDS_ROWS];
};

// The value columns of the request, one per lane (see lane_value), and the
// accumulators, field f in lane f: kind | LDS offset << 8.
struct lds_plan {
  int32_t ncols;
  uint32_t cd;  // storage | has validity << 7 | first field << 8 | end << 16
  uint32_t data_lo, data_hi, mask_lo, mask_hi, mask_offset;
  uint32_t fd;
};

__device__ __forceinline__ lds_plan load_lds_plan(gb_params const& P)
{
  lds_plan A;
  int const lane = int(threadIdx.x & 63);
  int const v    = lane < P.num_vals ? lane : 0;
  A.ncols        = P.num_vals;
  dcol const& c  = P.vals[v];
  uint64_t const d = reinterpret_cast<uint64_t>(c.data), m = reinterpret_cast<uint64_t>(c.mask);
  A.cd          = uint32_t(c.storage) | (m ? 0x80u : 0u) | (uint32_t(P.val_field_begin[v]) << 8) |
         (uint32_t(P.val_field_begin[v + 1]) << 16);
  A.data_lo     = uint32_t(d);
  A.data_hi     = uint32_t(d >> 32);
  A.mask_lo     = uint32_t(m);
  A.mask_hi     = uint32_t(m >> 32);
  A.mask_offset = uint32_t(c.mask_offset);
  int const f   = lane < P.num_fields ? lane : 0;
  A.fd          = uint32_t(P.fields[f].kind) | (uint32_t(P.fields[f].lds_off) << 8);
  return A;
}

__device__ __forceinline__ void load_lds_column(lds_plan const& A, int i, uint32_t r0, uint32_t n, lds_column& col)
{
  uint32_t const cd = lane_value(A.cd, i);
  if (((cd >> 8) & 0xffu) == ((cd >> 16) & 0xffu)) return;  // no accumulators (COUNT_ALL alone)
  if (cd & 0x80u)
    load_valid_words(reinterpret_cast<gmem<uint32_t const>*>(lane_value64(A.mask_lo, A.mask_hi, i)),
                     lane_value(A.mask_offset, i), r0, n, col.w);
  int const st = int(cd & 0x7fu);
  if (st != ST_STRING)  // a string column takes part by its validity alone (COUNT_VALID)
    load_chunk<LBLOCK>(reinterpret_cast<gmem<uint8_t const>*>(lane_value64(A.data_lo, A.data_hi, i)),
                       storage_width(st), r0, n, col.c);
}

// Orders a wave's LDS writes before its other lanes' reads.
__device__ __forceinline__ void wave_lds_order()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Key bits (zero-extended, as load_fixed_bits gives them) of slot i of a table
// indexed by the key itself.
__device__ __forceinline__ uint64_t lds_direct_key(gb_params const& P, uint64_t i)
{
  uint64_t const k = uint64_t(P.lds_key_min) + i;
  int const w      = storage_width(P.key_storage);
  return w == 8 ? k : k & ((1ull << (8 * w)) - 1ull);
}

// Slot of the group of the keys equal to EMPTY_KEY (0) or of the null keys (1).
__device__ __forceinline__ int64_t insert_special(gb_params const& P, int which)
{
  mark_special(P, which);
  return int64_t(P.cap) + which;
}

// Add an LDS partial of field F (float32 sums held in float64) to its
// accumulator in the device-wide table.
__device__ __forceinline__ void combine_partial(field_desc const& F, int64_t slot, uint64_t part)
{
  if (rpa_wide_sum(F.kind, true)) part = __float_as_uint(float(__longlong_as_double(int64_t(part))));
  // an identity partial changes nothing (float sums start at +0.0)
  if (part != field_identity(F.kind)) acc_combine(F.kind, field_at(F, slot), part);
}

// One wave's rows whose keys found no room in the LDS table, processed 64 at
// a time: a wave keeps at most 63 between rows and adds at most 64.
constexpr int LDS_SPILL = 128;

// How a row finds its LDS slot: by probing a table filled as keys come (rows
// that find no room update the device-wide table), by the key itself, or by
// probing a table of given keys (the rows of all others become the input of
// the partitioned path).
enum lds_mode : int { LDS_FILLED = 0, LDS_DIRECT, LDS_FIXED };

template <int MODE>
__global__ void __launch_bounds__(LBLOCK) k_aggregate_lds(gb_params const* __restrict__ Pp)
{
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ uint32_t fill_sh, present_sh[2];
  __shared__ uint32_t spill_sh[LBLOCK / 64][LDS_SPILL];
  __shared__ uint32_t rows_sh[2][LBLOCK / 64], base_sh[2];
  gb_params const& P  = *Pp;
  int const S         = P.lds_slots;
  uint32_t const limit = MODE == LDS_FIXED ? 0u : uint32_t(P.lds_fill);
  int32_t const count_off = P.lds_count_off;
  lds_plan const A    = load_lds_plan(P);
  int const nfields   = P.num_fields;
  auto* tkeys         = reinterpret_cast<uint64_t*>(lds);
  for (int i = threadIdx.x; i < S; i += LBLOCK) tkeys[i] = EMPTY_KEY;
  int64_t const key_min = P.lds_key_min;
  for (int f = 0; f < nfields; f++) {
    uint32_t const d   = lane_value(A.fd, f);
    int32_t const kind = int32_t(d & 0xffu), off = int32_t(d >> 8);
    if (kind == FK_M2) continue;
    uint64_t const idv = field_identity(kind);
    if (rpa_lds_width(kind, true) == 8)
      for (int i = threadIdx.x; i < S + 2; i += LBLOCK) *lds_at<uint64_t>(lds, off, i) = idv;
    else
      for (int i = threadIdx.x; i < S + 2; i += LBLOCK) *lds_at<uint32_t>(lds, off, i) = uint32_t(idv);
  }
  if (count_off >= 0)
    for (int i = threadIdx.x; i < S + 2; i += LBLOCK) *lds_at<uint32_t>(lds, count_off, i) = 0;
  if (threadIdx.x == 0) {
    fill_sh       = 0;
    present_sh[0] = 0;
    present_sh[1] = 0;
  }
  __syncthreads();
  if constexpr (MODE == LDS_FIXED) {
    for (int i = threadIdx.x; i < int(P.cap); i += LBLOCK) {
      uint64_t const k = gp(P.slot_keys)[i];
      if (k != EMPTY_KEY && lds_insert_any(tkeys, &fill_sh, k, lds_key_hash(k), EMPTY_KEY, S, uint32_t(S)) < 0)
        astore(P.overflow, 1);  // not expected: the call takes another path
    }
    __syncthreads();
  }
  dcol const kc         = P.keys[0];
  int32_t const kst     = kc.storage;
  int const kw          = storage_width(kst);
  bool const skip_nulls = P.skip_null_keys != 0;
  auto const kdata      = gp(kc.data);
  auto const kmask      = gp(kc.mask);
  uint32_t const koff   = uint32_t(kc.mask_offset);
  uint32_t const n      = uint32_t(P.num_rows);  // a size_type
  auto hash             = [&](uint64_t b) { return hash_combine(0u, hash_fixed_bits(kst, b, 0u)); };
  constexpr int U       = LDS_ROWS;
  uint32_t* const spill = spill_sh[threadIdx.x >> 6];
  int turn              = 0;
  uint32_t nspill       = 0;  // the same in every lane of the wave
  // rows spill[0, count): the device-wide table, one row per lane
  auto drain = [&](uint32_t count) {
    uint32_t const lane = threadIdx.x & 63u;
    wave_lds_order();
    if (lane < count) {
      int64_t const row   = int64_t(spill[lane]);
      uint64_t const bits = load_fixed_bits(kc, row);
      int64_t const slot  = insert_inline(P, bits, hash(bits));
      if (slot >= 0) update_row(P, slot, row);
    }
    wave_lds_order();
  };
  int const spare       = S + 2 + int(threadIdx.x & 63u);  // accumulators nobody reads
  uint32_t const stride = gridDim.x * (LBLOCK * U);
  uint64_t key[U];
  uint32_t kwv[U];
  auto load_keys = [&](uint32_t r0) {
    if (kmask) load_valid_words(kmask, koff, r0, n, kwv);
    load_chunk<LBLOCK>(kdata, kw, r0, n, key);
  };
  // a wave's rows run out together except in the last chunk, where the loop
  // bound is the workgroup's, so that every lane takes part in the ballots
  uint32_t const wg0 = blockIdx.x * (LBLOCK * U);
  if (wg0 < n) load_keys(wg0 + threadIdx.x);
  for (uint32_t w0 = wg0; w0 < n; w0 += stride) {
    uint32_t const r0 = w0 + threadIdx.x;
    lds_column cur;
    if (A.ncols > 0) load_lds_column(A, 0, r0, n, cur);
    int id[U];  // LDS slot; rows that do not count there: this lane's spare slot
    uint32_t full = 0;
    if constexpr (MODE == LDS_DIRECT) {
      canon_rows(kst, key);
#pragma unroll
      for (int u = 0; u < U; u++) {
        bool const in    = r0 + uint32_t(u) * LBLOCK < n;
        bool const null  = kmask && !((kwv[u] >> ((r0 + koff) & 31u)) & 1u);
        uint64_t const i = key[u] - uint64_t(key_min);
        bool const hit   = in && !null && i < uint64_t(S);
        id[u]            = hit ? int(i) : spare;
        tkeys[id[u]]     = i;  // marks the group (any value but EMPTY_KEY)
        if (in && null && !skip_nulls) {
          id[u]         = S + 1;
          present_sh[1] = 1;
        }
        full |= uint32_t(in && !null && !hit) << u;
      }
    } else {
      uint32_t probe = 0, h[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        id[u] = spare;
        if (kst == ST_F32) key[u] = normalize_f32_bits(uint32_t(key[u]));
        else if (kst == ST_F64) key[u] = normalize_f64_bits(key[u]);
        else if (kst == ST_BOOL) key[u] = key[u] != 0;
        h[u]            = lds_key_hash(key[u]);
        bool const in   = r0 + uint32_t(u) * LBLOCK < n;
        bool const null = kmask && !((kwv[u] >> ((r0 + koff) & 31u)) & 1u);
        if (in && null && !skip_nulls) {
          id[u]         = S + 1;
          present_sh[1] = 1;
        } else if (in && !null && key[u] == EMPTY_KEY) {
          id[u]         = S;
          present_sh[0] = 1;
        }
        probe |= uint32_t(in && !null && key[u] != EMPTY_KEY) << u;
      }
      int found[U];
      lds_insert_rows(tkeys, &fill_sh, key, h, probe, S, limit, found);
#pragma unroll
      for (int u = 0; u < U; u++) {
        bool const mine = (probe >> u) & 1u;
        if (mine && found[u] >= 0) id[u] = found[u];
        full |= uint32_t(mine && found[u] < 0) << u;
      }
    }
    if (w0 + uint64_t(stride) < n) load_keys(r0 + stride);  // in flight during the accumulation
    constexpr uint32_t ALL = (1u << U) - 1u;
    if (count_off >= 0)
      for_rows<U>(ALL, [&](int u) {
        __hip_atomic_fetch_add(lds_at<uint32_t>(lds, count_off, id[u]), 1u, __ATOMIC_RELAXED, WG_SCOPE);
      });
    for (int i = 0; i < A.ncols; i++) {
      lds_column next;
      if (i + 1 < A.ncols) load_lds_column(A, i + 1, r0, n, next);
      uint32_t const cd = lane_value(A.cd, i);
      int const st = int(cd & 0x7fu), fb = int((cd >> 8) & 0xffu), fe = int((cd >> 16) & 0xffu);
      if (fb < fe) {
        int at[U];
#pragma unroll
        for (int u = 0; u < U; u++) at[u] = id[u];
        if (cd & 0x80u) {
          uint32_t const sh = (r0 + lane_value(A.mask_offset, i)) & 31u;
#pragma unroll
          for (int u = 0; u < U; u++) at[u] = (cur.w[u] >> sh) & 1u ? at[u] : spare;
        }
        canon_rows(st, cur.c);
        for (int f = fb; f < fe; f++) {
          uint32_t const d = lane_value(A.fd, f);
          opaque_rows(at, cur.c);
          if ((d & 0xffu) != FK_M2) acc_rows_lds(int32_t(d & 0xffu), int32_t(d >> 8), st, lds, at, ALL, cur.c, true);
        }
      }
      cur = next;
    }
    if constexpr (MODE == LDS_FIXED) {
      // append the rows of other keys to the spill columns: one reservation
      // per chunk (`turn` alternates the buffers, so that the next chunk's
      // counts don't meet this one's readers)
      uint64_t bal[U];
      uint32_t wave_rows = 0;
#pragma unroll
      for (int u = 0; u < U; u++) {
        bal[u] = __builtin_amdgcn_ballot_w64((full >> u) & 1u);
        wave_rows += uint32_t(__popcll(bal[u]));
      }
      int const wave = int(threadIdx.x >> 6);
      if ((threadIdx.x & 63u) == 0) rows_sh[turn][wave] = wave_rows;
      lds_barrier();
      if (threadIdx.x == 0) {
        uint32_t all = 0;
        for (int w = 0; w < LBLOCK / 64; w++) all += rows_sh[turn][w];
        base_sh[turn] = all ? __hip_atomic_fetch_add(gp(P.spill_count), all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                            : 0u;
      }
      lds_barrier();
      uint32_t at = base_sh[turn];
      for (int w = 0; w < wave; w++) at += rows_sh[turn][w];
      turn ^= 1;
      uint32_t dst[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        dst[u] = at + uint32_t(__popcll(bal[u] & ((1ull << (threadIdx.x & 63u)) - 1ull)));
        at += uint32_t(__popcll(bal[u]));
      }
      auto copy = [&](int w, uint8_t* to, uint8_t const* from) {
        for_rows<U>(full, [&](int u) {
          uint32_t const r = r0 + uint32_t(u) * LBLOCK;
          switch (w) {
            case 1: gp(to)[dst[u]] = gp(from)[r]; break;
            case 2: gp(reinterpret_cast<uint16_t*>(to))[dst[u]] = gp(reinterpret_cast<uint16_t const*>(from))[r]; break;
            case 4: gp(reinterpret_cast<uint32_t*>(to))[dst[u]] = gp(reinterpret_cast<uint32_t const*>(from))[r]; break;
            default: gp(reinterpret_cast<uint64_t*>(to))[dst[u]] = gp(reinterpret_cast<uint64_t const*>(from))[r]; break;
          }
        });
      };
      if (wave_rows) {
        copy(kw, P.spill_key, kc.data);
        for (int v = 0; v < A.ncols; v++) {
          if (!P.spill_val[v]) continue;  // no accumulators
          dcol const c = P.vals[v];
          copy(storage_width(c.storage), P.spill_val[v], c.data);
          if (c.mask)
            for_rows<U>(full, [&](int u) {
              gp(P.spill_valid[v])[dst[u]] = dcol_valid(c, int64_t(r0 + uint32_t(u) * LBLOCK)) ? 1 : 0;
            });
        }
      }
      continue;
    }
    // keys that found no room in the LDS table update the device-wide table
    if (__builtin_amdgcn_ballot_w64(full != 0) != 0) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        bool const mine      = (full >> u) & 1u;
        uint64_t const bal   = __builtin_amdgcn_ballot_w64(mine);
        uint64_t const below = (1ull << (threadIdx.x & 63u)) - 1ull;
        if (mine) spill[nspill + uint32_t(__popcll(bal & below))] = r0 + uint32_t(u) * LBLOCK;
        nspill += uint32_t(__popcll(bal));
        if (nspill >= 64u) {
          drain(64u);
          uint32_t const rest = nspill - 64u;
          uint32_t const keep = (threadIdx.x & 63u) < rest ? spill[64u + (threadIdx.x & 63u)] : 0u;
          wave_lds_order();
          if ((threadIdx.x & 63u) < rest) spill[threadIdx.x & 63u] = keep;
          nspill = rest;
        }
      }
      // the call rebuilds a larger table: stop early (one load per wave, so
      // the whole wave leaves together)
      if (__builtin_amdgcn_readfirstlane(int(aload(P.overflow))) != 0) break;
    }
  }
  if (nspill) drain(nspill);
  __syncthreads();
  if (aload(P.overflow) != 0) return;  // this table is discarded
  if (P.lds_dump) {  // many workgroups: k_merge_lds combines their tables
    auto const out  = gp(reinterpret_cast<uint64_t*>(P.lds_dump + int64_t(blockIdx.x) * P.lds_dump_stride));
    int const words = P.lds_dump_stride / 8 - 1;
    for (int i = threadIdx.x; i < words; i += LBLOCK) out[i] = reinterpret_cast<uint64_t const*>(lds)[i];
    if (threadIdx.x == 0) out[words] = (uint64_t(present_sh[1]) << 32) | present_sh[0];
    return;
  }
  // merge the partials into the global table
  for (int i = threadIdx.x; i < S + 2; i += LBLOCK) {
    int64_t slot;
    if (i < S) {
      if (tkeys[i] == EMPTY_KEY) continue;
      uint64_t const k = MODE == LDS_DIRECT ? lds_direct_key(P, uint64_t(i)) : tkeys[i];
      slot = insert_inline(P, k, hash(k));
    } else {
      if (!present_sh[i - S]) continue;
      slot = insert_special(P, i - S);
    }
    if (slot < 0) continue;
    if (count_off >= 0) aadd(count_at(P, slot), *lds_at<uint32_t>(lds, count_off, i));
    for (int f = 0; f < nfields; f++) {
      field_desc const& F = P.fields[f];
      if (F.kind == FK_M2) continue;
      combine_partial(F, slot, rpa_lds_width(F.kind, true) == 8 ? *lds_at<uint64_t>(lds, F.lds_off, i)
                                                                : uint64_t(*lds_at<uint32_t>(lds, F.lds_off, i)));
    }
  }
}

// Combine two LDS partials (float32 sums held in float64).
__device__ __forceinline__ void lds_combine(int32_t kind, uint64_t* a, uint64_t part)
{
  constexpr int R = __ATOMIC_RELAXED;
  auto* u32       = reinterpret_cast<uint32_t*>(a);
  switch (kind) {
    case FK_SUM_I64:
    case FK_SUMSQ_I64: __hip_atomic_fetch_add(a, part, R, WG_SCOPE); break;
    case FK_SUM_F32:
    case FK_SUMSQ_F32:
    case FK_SUM_F64:
    case FK_SUMSQ_F64:
      __hip_atomic_fetch_add(reinterpret_cast<double*>(a), __longlong_as_double(int64_t(part)), R, WG_SCOPE);
      break;
    case FK_MIN_S32: __hip_atomic_fetch_min(reinterpret_cast<int32_t*>(a), int32_t(part), R, WG_SCOPE); break;
    case FK_MAX_S32: __hip_atomic_fetch_max(reinterpret_cast<int32_t*>(a), int32_t(part), R, WG_SCOPE); break;
    case FK_MIN_S64: __hip_atomic_fetch_min(reinterpret_cast<int64_t*>(a), int64_t(part), R, WG_SCOPE); break;
    case FK_MAX_S64: __hip_atomic_fetch_max(reinterpret_cast<int64_t*>(a), int64_t(part), R, WG_SCOPE); break;
    case FK_MIN_U32:
    case FK_MIN_F32: __hip_atomic_fetch_min(u32, uint32_t(part), R, WG_SCOPE); break;
    case FK_MAX_U32:
    case FK_MAX_F32: __hip_atomic_fetch_max(u32, uint32_t(part), R, WG_SCOPE); break;
    case FK_MIN_U64:
    case FK_MIN_F64: __hip_atomic_fetch_min(a, part, R, WG_SCOPE); break;
    case FK_MAX_U64:
    case FK_MAX_F64: __hip_atomic_fetch_max(a, part, R, WG_SCOPE); break;
    case FK_COUNT: __hip_atomic_fetch_add(u32, uint32_t(part), R, WG_SCOPE); break;
    default: break;
  }
}

// Combines the tables that the workgroups of k_aggregate_lds stored: a
// workgroup takes LDS_MERGE_RANGE slots of every table (one more takes the two
// special groups), adds up equal keys in LDS and updates the device-wide table
// once per key.  Equal keys sit at nearly the same slot of every table; where
// they don't, two workgroups update the group.  Atomics on few addresses run
// at 7 G/s on this device (24 G/s on many), so merging 256 tables of 1,000
// groups and 7 accumulators straight into the device-wide table took 245 us;
// this kernel takes 22 us (16 us
// for 245 tables); 8 slots a workgroup: with 32, too few workgroups, 45 us.
constexpr int LDS_MERGE_RANGE = 8;
constexpr int LDS_MERGE_SLOTS = 64;
constexpr int LDS_MERGE_TABLES = 2;

__global__ void __launch_bounds__(LBLOCK) k_merge_lds(gb_params const* __restrict__ Pp, int tables)
{
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ uint32_t fill_sh, present_sh[2];
  gb_params const& P = *Pp;
  if (aload(P.overflow) != 0) return;  // the tables are discarded
  constexpr int MS   = LDS_MERGE_SLOTS;
  int const S        = P.lds_slots;
  int const nfields  = P.num_fields;
  int32_t const kst  = P.key_storage;
  int32_t const count_off = P.lds_count_off;
  auto* tkeys        = reinterpret_cast<uint64_t*>(lds);
  // accumulator f of slot i (f == nfields: the row count)
  auto acc = [&](int f, int i) { return tkeys + MS + f * (MS + 2) + i; };
  for (int i = threadIdx.x; i < MS; i += LBLOCK) tkeys[i] = EMPTY_KEY;
  for (int f = 0; f <= nfields; f++) {
    uint64_t const idv = f < nfields ? field_identity(P.fields[f].kind) : 0;
    for (int i = threadIdx.x; i < MS + 2; i += LBLOCK) *acc(f, i) = idv;
  }
  if (threadIdx.x == 0) {
    fill_sh       = 0;
    present_sh[0] = 0;
    present_sh[1] = 0;
  }
  __syncthreads();
  int const first    = int(blockIdx.x) * LDS_MERGE_RANGE;
  bool const special = first >= S;
  int const width    = special ? 2 : LDS_MERGE_RANGE;
  auto hash          = [&](uint64_t b) { return hash_combine(0u, hash_fixed_bits(kst, b, 0u)); };
  // LDS_MERGE_TABLES tables per thread at a time: their keys, then one accumulator
  // of all of them, are in flight together
  constexpr int V    = LDS_MERGE_TABLES;
  int const which    = int(threadIdx.x) % width, group = int(threadIdx.x) / width, groups = LBLOCK / width;
  int const s        = special ? S + which : first + which;
  bool const direct  = P.lds_direct != 0;
  uint32_t const fd  = load_lds_plan(P).fd;
  auto const dump    = gp(static_cast<uint8_t const*>(P.lds_dump));
  int64_t const step = P.lds_dump_stride;
  int const sc       = special ? s : min(s, S - 1);  // in bounds; unused past the last slot
  // every lane stays in the loop: the plan is read from lanes of its own
  for (int tb = 0; tb < tables; tb += V * groups) {
    int const t0 = tb + group;
    uint64_t key[V];
    int id[V];
    auto table = [&](int v) { return dump + int64_t(min(t0 + v * groups, tables - 1)) * step; };
#pragma unroll
    for (int v = 0; v < V; v++)
      key[v] = special ? uint64_t(reinterpret_cast<gmem<uint32_t const>*>(table(v) + (step - 8))[which])
                       : reinterpret_cast<gmem<uint64_t const>*>(table(v))[sc];
    uint32_t mine = 0;
#pragma unroll
    for (int v = 0; v < V; v++) {
      id[v] = -2;
      if (t0 + v * groups >= tables || s != sc) continue;
      if (special) {
        if (!key[v]) continue;
        present_sh[which] = 1;
        id[v]             = MS + which;
      } else {
        if (key[v] == EMPTY_KEY) continue;
        if (direct) key[v] = lds_direct_key(P, uint64_t(s));
        id[v] = lds_insert_any(tkeys, &fill_sh, key[v], mm_fmix32(lds_key_hash(key[v])), EMPTY_KEY, MS, MS * 7 / 8);
      }
      mine |= 1u << v;
    }
    for (int f = 0; f <= nfields; f++) {
      uint32_t const d   = lane_value(fd, f < nfields ? f : 0);
      int32_t const kind = f < nfields ? int32_t(d & 0xffu) : int32_t(FK_COUNT);
      int32_t const off  = f < nfields ? int32_t(d >> 8) : count_off;
      if (kind == FK_M2 || off < 0) continue;
      bool const w8 = rpa_lds_width(kind, true) == 8;
      uint64_t part[V];
#pragma unroll
      for (int v = 0; v < V; v++) {
        if (w8) part[v] = reinterpret_cast<gmem<uint64_t const>*>(table(v) + off)[sc];
        else part[v] = reinterpret_cast<gmem<uint32_t const>*>(table(v) + off)[sc];
      }
#pragma unroll
      for (int v = 0; v < V; v++)
        if (((mine >> v) & 1u) && id[v] >= 0) lds_combine(kind, acc(f, id[v]), part[v]);
    }
#pragma unroll
    for (int v = 0; v < V; v++) {  // no room in LDS: straight to the table
      if (!((mine >> v) & 1u) || id[v] >= 0) continue;
      int64_t const slot = insert_inline(P, key[v], hash(key[v]));
      if (slot < 0) continue;
      if (count_off >= 0) aadd(count_at(P, slot), reinterpret_cast<gmem<uint32_t const>*>(table(v) + count_off)[s]);
      for (int f = 0; f < nfields; f++) {
        field_desc const& F = P.fields[f];
        if (F.kind == FK_M2) continue;
        combine_partial(F, slot, rpa_lds_width(F.kind, true) == 8
                                   ? reinterpret_cast<gmem<uint64_t const>*>(table(v) + F.lds_off)[s]
                                   : uint64_t(reinterpret_cast<gmem<uint32_t const>*>(table(v) + F.lds_off)[s]));
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < MS + 2; i += LBLOCK) {
    int64_t slot;
    if (i < MS) {
      if (tkeys[i] == EMPTY_KEY) continue;
      slot = insert_inline(P, tkeys[i], hash(tkeys[i]));
    } else {
      if (!present_sh[i - MS]) continue;
      slot = insert_special(P, i - MS);
    }
    if (slot < 0) continue;
    if (count_off >= 0) aadd(count_at(P, slot), uint32_t(*acc(nfields, i)));
    for (int f = 0; f < nfields; f++)
      if (P.fields[f].kind != FK_M2) combine_partial(P.fields[f], slot, *acc(f, i));
  }
}

// The variance pass over the groups of the finished device-wide table: their
// means are loaded into LDS once, so a row costs its probe (or none: DIRECT, as
// in k_aggregate_lds), one read and one add per column.  Rows whose group found
// no room update the device-wide table.  Accumulators: mean, then Σ(x - mean)²,
// per FK_M2 field at lds_m2_off.
template <bool DIRECT>
__global__ void __launch_bounds__(LBLOCK) k_second_pass_lds(gb_params const* __restrict__ Pp)
{
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ uint32_t fill_sh;
  gb_params const& P  = *Pp;
  int const S         = P.lds_slots;
  int const NS        = S + LDS_EXTRA_SLOTS;
  lds_plan const A    = load_lds_plan(P);
  int const nfields   = P.num_fields;
  int const lane      = int(threadIdx.x & 63u);
  uint32_t const m2_l = uint32_t(P.lds_m2_off[lane < nfields ? lane : 0]);
  auto* tkeys         = reinterpret_cast<uint64_t*>(lds);
  auto* tslots        = reinterpret_cast<uint32_t*>(tkeys + NS);  // device-wide slots
  auto mean           = [&](int32_t off, int i) { return reinterpret_cast<double*>(lds + off) + i; };
  auto m2             = [&](int32_t off, int i) { return reinterpret_cast<double*>(lds + off) + NS + i; };
  for (int i = threadIdx.x; i < NS; i += LBLOCK) {
    tkeys[i]  = EMPTY_KEY;
    tslots[i] = 0xffffffffu;
  }
  for (int f = 0; f < nfields; f++) {
    if ((lane_value(A.fd, f) & 0xffu) != FK_M2) continue;
    int32_t const off = int32_t(lane_value(m2_l, f));
    for (int i = threadIdx.x; i < 2 * NS; i += LBLOCK) *mean(off, i) = 0.0;
  }
  if (threadIdx.x == 0) fill_sh = 0;
  __syncthreads();
  dcol const kc         = P.keys[0];
  int32_t const kst     = kc.storage;
  int64_t const key_min = P.lds_key_min;
  for (int64_t g = threadIdx.x; g < int64_t(P.cap) + 2; g += LBLOCK) {
    int id = -1;
    if (g < int64_t(P.cap)) {
      uint64_t c[1] = {gp(P.slot_keys)[g]};
      if (c[0] == EMPTY_KEY) continue;
      if constexpr (DIRECT) {
        canon_rows(kst, c);
        uint64_t const i = c[0] - uint64_t(key_min);
        if (i < uint64_t(S)) id = int(i);
      } else {
        id = lds_insert_any(tkeys, &fill_sh, c[0], lds_key_hash(c[0]), EMPTY_KEY, S, uint32_t(P.lds_fill));
      }
    } else if (P.special[g - int64_t(P.cap)]) {
      id = S + int(g - int64_t(P.cap));
    }
    if (id < 0) continue;
    tslots[id] = uint32_t(g);  // the table of few groups is small
    for (int f = 0; f < nfields; f++) {
      field_desc const& F = P.fields[f];
      if (F.kind == FK_M2)
        *mean(P.lds_m2_off[f], id) = field_as_double(P.fields[F.aux_sum], g) / double(count_of(P, F.aux_count, g));
    }
  }
  __syncthreads();
  int const kw          = storage_width(kst);
  bool const skip_nulls = P.skip_null_keys != 0;
  auto const kdata      = gp(kc.data);
  auto const kmask      = gp(kc.mask);
  uint32_t const koff   = uint32_t(kc.mask_offset);
  uint32_t const n      = uint32_t(P.num_rows);
  constexpr int U       = LDS_ROWS;
  int const spare       = S + 2 + lane;
  uint32_t const stride = gridDim.x * (LBLOCK * U);
  for (uint32_t w0 = blockIdx.x * (LBLOCK * U); w0 < n; w0 += stride) {
    uint32_t const r0 = w0 + threadIdx.x;
    uint64_t key[U];
    uint32_t kwv[U];
    if (kmask) load_valid_words(kmask, koff, r0, n, kwv);
    load_chunk<LBLOCK>(kdata, kw, r0, n, key);
    int id[U];
    uint32_t full = 0, probe = 0, h[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      id[u]           = spare;
      bool const in   = r0 + uint32_t(u) * LBLOCK < n;
      bool const null = kmask && !((kwv[u] >> ((r0 + koff) & 31u)) & 1u);
      if (in && null && !skip_nulls) id[u] = S + 1;
      if (kst == ST_F32) key[u] = normalize_f32_bits(uint32_t(key[u]));
      else if (kst == ST_F64) key[u] = normalize_f64_bits(key[u]);
      else if (kst == ST_BOOL) key[u] = key[u] != 0;
      if (in && !null && key[u] == EMPTY_KEY) id[u] = S;
      h[u] = lds_key_hash(key[u]);
      probe |= uint32_t(in && !null && key[u] != EMPTY_KEY) << u;
    }
    int found[U];
    if constexpr (DIRECT) {
      uint64_t c[U];
#pragma unroll
      for (int u = 0; u < U; u++) c[u] = key[u];
      canon_rows(kst, c);
#pragma unroll
      for (int u = 0; u < U; u++) {
        uint64_t const i = c[u] - uint64_t(key_min);
        found[u]         = i < uint64_t(S) ? int(i) : -1;
      }
    } else {
      lds_insert_rows(tkeys, &fill_sh, key, h, probe, S, 0u, found);  // finds only
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      bool const mine = (probe >> u) & 1u;
      if (mine && found[u] >= 0) id[u] = found[u];
      full |= uint32_t(mine && found[u] < 0) << u;
    }
    for (int i = 0; i < A.ncols; i++) {
      uint32_t const cd = lane_value(A.cd, i);
      int const fb = int((cd >> 8) & 0xffu), fe = int((cd >> 16) & 0xffu), st = int(cd & 0x7fu);
      int m2f = -1;
      for (int f = fb; f < fe; f++)
        if ((lane_value(A.fd, f) & 0xffu) == FK_M2) m2f = f;
      if (m2f < 0) continue;
      int32_t const off = int32_t(lane_value(m2_l, m2f));
      lds_column col;
      load_lds_column(A, i, r0, n, col);
      canon_rows(st, col.c);
      int at[U];
#pragma unroll
      for (int u = 0; u < U; u++) at[u] = id[u];
      if (cd & 0x80u) {
        uint32_t const sh = (r0 + lane_value(A.mask_offset, i)) & 31u;
#pragma unroll
        for (int u = 0; u < U; u++) at[u] = (col.w[u] >> sh) & 1u ? at[u] : spare;
      }
      double mu[U];
#pragma unroll
      for (int u = 0; u < U; u++) mu[u] = *mean(off, at[u]);
#pragma unroll
      for (int u = 0; u < U; u++) {
        double const d = canon_double(st, col.c[u]) - mu[u];
        __hip_atomic_fetch_add(m2(off, at[u]), d * d, __ATOMIC_RELAXED, WG_SCOPE);
      }
    }
    if (__builtin_amdgcn_ballot_w64(full != 0) == 0) continue;
    for (int u = 0; u < U; u++) {  // groups without room in LDS
      if (!((full >> u) & 1u)) continue;
      int64_t const row  = int64_t(r0 + uint32_t(u) * LBLOCK);
      int64_t const slot = locate<KM_INLINE, false>(P, row);
      if (slot < 0) continue;
      for (int f = 0; f < nfields; f++) {
        field_desc const& F = P.fields[f];
        if (F.kind != FK_M2 || !dcol_valid(P.vals[F.vcol], row)) continue;
        double const mu = field_as_double(P.fields[F.aux_sum], slot) / double(count_of(P, F.aux_count, slot));
        double const d  = load_value(P.vals[F.vcol], row).d - mu;
        gadd_f64(reinterpret_cast<double*>(field_at(F, slot)), d * d);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < S + 2; i += LBLOCK) {
    uint32_t const slot = tslots[i];
    if (slot == 0xffffffffu) continue;
    for (int f = 0; f < nfields; f++) {
      if (P.fields[f].kind != FK_M2) continue;
      double const part = *m2(P.lds_m2_off[f], i);
      if (part != 0.0) gadd_f64(reinterpret_cast<double*>(field_at(P.fields[f], int64_t(slot))), part);
    }
  }
}

// The same for hot keys among many groups, and where LDS does not hold every
// group (the estimate was low): a table of group slots filled as the rows come,
// so that it holds the hot ones.  Means loaded in the order of the device-wide
// table may leave out the hottest key, whose rows then queue up on one address:
// 5M rows, Zipf(2), 36.6 ms against 0.06 ms.
__global__ void __launch_bounds__(LBLOCK) k_second_pass_hot(gb_params const* __restrict__ Pp)
{
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ uint32_t fill_sh;
  gb_params const& P = *Pp;
  constexpr int WG   = __HIP_MEMORY_SCOPE_WORKGROUP;
  constexpr uint64_t NO = ~0ull;  // free slot of the LDS table of group slots
  int const S        = P.lds_slots;
  auto* tslots       = reinterpret_cast<uint64_t*>(lds);
  for (int i = threadIdx.x; i < S; i += LBLOCK) tslots[i] = NO;
  // partials of M2 field f
  auto m2 = [&](int f, int i) { return lds_at<double>(lds, P.lds_m2_off[f], i); };
  for (int f = 0; f < P.num_fields; f++) {
    if (P.fields[f].kind != FK_M2) continue;
    for (int i = threadIdx.x; i < S; i += LBLOCK) *m2(f, i) = 0.0;
  }
  if (threadIdx.x == 0) fill_sh = 0;
  __syncthreads();
  for (int64_t row = int64_t(blockIdx.x) * LBLOCK + threadIdx.x; row < P.num_rows;
       row += int64_t(gridDim.x) * LBLOCK) {
    int64_t slot = -2;
    int id       = -1;
    for (int vc = 0; vc < P.num_vals; vc++) {
      int const fb = P.val_field_begin[vc], fe = P.val_field_begin[vc + 1];
      bool has_m2  = false;
      for (int f = fb; f < fe; f++) has_m2 |= (P.fields[f].kind == FK_M2);
      if (!has_m2) continue;
      dcol const& c = P.vals[vc];
      if (!dcol_valid(c, row)) continue;
      if (slot == -2) {
        slot = locate<KM_INLINE, false>(P, row);
        if (slot >= 0) id = lds_insert_any(tslots, &fill_sh, uint64_t(slot), mm_fmix32(uint32_t(slot)), NO, S,
                                           uint32_t(P.lds_fill));
      }
      if (slot < 0) break;
      loaded_value const v = load_value(c, row);
      for (int f = fb; f < fe; f++) {
        field_desc const& F = P.fields[f];
        if (F.kind != FK_M2) continue;
        double const cnt  = double(count_of(P, F.aux_count, slot));
        double const mean = field_as_double(P.fields[F.aux_sum], slot) / cnt;
        double const d    = v.d - mean;
        if (id >= 0) __hip_atomic_fetch_add(m2(f, id), d * d, __ATOMIC_RELAXED, WG);
        else gadd_f64(reinterpret_cast<double*>(field_at(F, slot)), d * d);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < S; i += LBLOCK) {
    uint64_t const slot = tslots[i];
    if (slot == NO) continue;
    for (int f = 0; f < P.num_fields; f++) {
      if (P.fields[f].kind != FK_M2) continue;
      double const part = *m2(f, i);
      if (part != 0.0) gadd_f64(reinterpret_cast<double*>(field_at(P.fields[f], int64_t(slot))), part);
    }
  }
}

void allow_dynamic_lds(void const* fn, int bytes)
{
  if (bytes <= 64 * 1024) return;
  // Raised once per kernel and device (and only upwards): setting a function
  // attribute is not a stream operation, but other threads may be capturing
  // graphs, so it is kept off the per-call path.
  static std::mutex mu;
  static std::map<std::pair<void const*, int>, int> done;
  int dev = 0;
  MIG_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  int& cur = done[{fn, dev}];
  if (bytes <= cur) return;
  MIG_HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  cur = bytes;
}

void launch_aggregate_lds(gb_params const* dP, gb_params const& hP, int64_t blocks, hipStream_t s)
{
  if (hP.num_rows <= 0) return;
  auto run = [&](auto* kernel) {
    allow_dynamic_lds(reinterpret_cast<void const*>(kernel), hP.lds_bytes);
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(LBLOCK), hP.lds_bytes, s, dP);
  };
  if (hP.lds_fixed) run(&k_aggregate_lds<LDS_FIXED>);
  else if (hP.lds_direct) run(&k_aggregate_lds<LDS_DIRECT>);
  else run(&k_aggregate_lds<LDS_FILLED>);
  if (!hP.lds_dump) return;
  int const lds = 8 * (LDS_MERGE_SLOTS + (hP.num_fields + 1) * (LDS_MERGE_SLOTS + 2));
  allow_dynamic_lds(reinterpret_cast<void const*>(&k_merge_lds), lds);
  int const ranges = (hP.lds_slots + LDS_MERGE_RANGE - 1) / LDS_MERGE_RANGE;
  hipLaunchKernelGGL(k_merge_lds, dim3(ranges + 1), dim3(LBLOCK), lds, s, dP, int(blocks));
}

void launch_second_pass_lds(gb_params const* dP, gb_params const& hP, int64_t blocks, bool all_fit, hipStream_t s)
{
  if (hP.num_rows <= 0) return;
  auto run = [&](auto* kernel) {
    allow_dynamic_lds(reinterpret_cast<void const*>(kernel), hP.lds_m2_bytes);
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(LBLOCK), hP.lds_m2_bytes, s, dP);
  };
  if (hP.lds_hot || !all_fit) run(&k_second_pass_hot);
  else if (hP.lds_direct) run(&k_second_pass_lds<true>);
  else run(&k_second_pass_lds<false>);
}

// ---------------------------------------------------------------------------
// compaction of occupied slots -> dense group ids
__device__ __forceinline__ bool slot_occupied(gb_params const& P, uint64_t slot)
{
  if (slot < P.cap) {
    return P.key_mode == KM_INLINE ? (P.slot_keys[slot] != EMPTY_KEY)
                                   : (P.slot_rows[slot] != EMPTY_ROW);
  }
  return P.special[slot - P.cap] != 0u;
}


__global__ void __launch_bounds__(BLOCK)
  k_count_occupied(gb_params const* __restrict__ Pp, uint32_t* block_counts)
{
  __shared__ uint32_t red[BLOCK / 64];
  gb_params const& P = *Pp;
  uint64_t const total = P.cap + 2;
  uint64_t const base  = uint64_t(blockIdx.x) * SCAN_TILE;
  uint32_t c = 0;
  for (int k = threadIdx.x; k < SCAN_TILE; k += BLOCK) {
    uint64_t slot = base + k;
    if (slot < total && slot_occupied(P, slot)) c++;
  }
  c = block_sum_u32(c, red);
  if (threadIdx.x == 0) block_counts[blockIdx.x] = c;
}

void launch_count_occupied(gb_params const* dP, gb_params const& hP, uint32_t* block_counts,
                           hipStream_t s)
{
  int64_t nb = (int64_t(hP.cap) + 2 + SCAN_TILE - 1) / SCAN_TILE;
  hipLaunchKernelGGL(k_count_occupied, dim3(nb), dim3(BLOCK), 0, s, dP, block_counts);
}

// Exclusive scan of `n` u32 values in place by one block of 1024 threads.
__global__ void __launch_bounds__(1024) k_scan_small(uint32_t* data, int64_t n, uint32_t* total)
{
  __shared__ uint32_t part[1024];
  int64_t const per = (n + 1023) / 1024;
  int64_t const b   = int64_t(threadIdx.x) * per;
  int64_t const e   = (b + per < n) ? b + per : n;
  uint32_t s = 0;
  for (int64_t i = b; i < e; i++) s += data[i];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    uint32_t v = threadIdx.x >= o ? part[threadIdx.x - o] : 0;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = threadIdx.x ? part[threadIdx.x - 1] : 0;
  for (int64_t i = b; i < e; i++) {
    uint32_t v = data[i];
    data[i]    = run;
    run += v;
  }
  if (threadIdx.x == 1023 && total) *total = part[1023];
}

void launch_scan_blocks(uint32_t* block_counts, int64_t nblocks, uint32_t* total, hipStream_t s)
{
  hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, block_counts, nblocks, total);
}

// Writes the gather map: rep_rows[g] = slot of dense group g (slot order).
__global__ void __launch_bounds__(BLOCK)
  k_compact(gb_params const* __restrict__ Pp, uint32_t const* block_offsets, uint32_t* map)
{
  __shared__ uint32_t wave_tot[BLOCK / 64];
  gb_params const& P = *Pp;
  uint64_t const total = P.cap + 2;
  uint64_t const base  = uint64_t(blockIdx.x) * SCAN_TILE;
  uint32_t running     = block_offsets[blockIdx.x];
  int const wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int k = 0; k < SCAN_TILE; k += BLOCK) {
    uint64_t const slot = base + k + threadIdx.x;
    bool const occ     = slot < total && slot_occupied(P, slot);
    uint64_t const bal = __ballot(occ);
    uint32_t const below = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[wave] = __popcll(bal);
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int w = 0; w < BLOCK / 64; w++) {
      if (w < wave) before += wave_tot[w];
      all += wave_tot[w];
    }
    if (occ) map[running + before + below] = uint32_t(slot);
    running += all;
    __syncthreads();
  }
}

void launch_compact(gb_params const* dP, gb_params const& hP, uint32_t const* block_offsets,
                    uint32_t* map, hipStream_t s)
{
  int64_t nb = (int64_t(hP.cap) + 2 + SCAN_TILE - 1) / SCAN_TILE;
  hipLaunchKernelGGL(k_compact, dim3(nb), dim3(BLOCK), 0, s, dP, block_offsets, map);
}

// Both steps and the scan between them for a small table, by one workgroup:
// map[g] = slot of dense group g, *total = groups.
__global__ void __launch_bounds__(1024) k_compact_small(gb_params const* __restrict__ Pp, uint32_t* map, uint32_t* total)
{
  __shared__ uint32_t wave_tot[1024 / 64];
  gb_params const& P   = *Pp;
  uint32_t const slots = uint32_t(P.cap) + 2u;
  uint32_t const per   = (slots + 1023u) / 1024u;  // at most COMPACT_SMALL / 1024 + 1
  uint32_t const b     = threadIdx.x * per;
  int const wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint32_t occ = 0;  // bit j: slot b + j
  for (uint32_t j = 0; j < per; j++)
    if (b + j < slots && slot_occupied(P, b + j)) occ |= 1u << j;
  uint32_t const mine = uint32_t(__popc(occ));
  uint32_t incl       = mine;
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t const y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) wave_tot[wave] = incl;
  __syncthreads();
  uint32_t at = incl - mine;
  for (int w = 0; w < wave; w++) at += wave_tot[w];
  for (uint32_t j = 0; j < per; j++)
    if ((occ >> j) & 1u) map[at++] = b + j;
  if (threadIdx.x == 1023) *total = at;
}

void launch_compact_small(gb_params const* dP, uint32_t* map, uint32_t* total, hipStream_t s)
{
  hipLaunchKernelGGL(k_compact_small, dim3(1), dim3(1024), 0, s, dP, map, total);
}

// ---------------------------------------------------------------------------
// dense outputs: keys and aggregation results for group g = blockIdx*BLOCK+tid
__device__ __forceinline__ uint64_t field_bits(field_desc const& F, int64_t slot)
{
  return F.width == 8 ? *reinterpret_cast<uint64_t const*>(field_at(F, slot))
                      : *reinterpret_cast<uint32_t const*>(field_at(F, slot));
}


// Writes the validity bit of group g for the whole wave with one ballot.
__device__ __forceinline__ void store_valid_bits(uint32_t* mask, int64_t g, int64_t G, bool valid)
{
  uint64_t const bal = __ballot(g < G && valid);
  int const lane     = threadIdx.x & 63;
  int64_t const g0   = g - lane;  // multiple of 64
  if (lane == 0 && g0 < G) mask[g0 >> 5] = uint32_t(bal);
  if (lane == 32 && g0 + 32 < G) mask[(g0 >> 5) + 1] = uint32_t(bal >> 32);
}

template <int KM>
__global__ void __launch_bounds__(BLOCK)
  k_outputs(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ map, int64_t G,
            uint32_t* rep_rows)
{
  gb_params const& P = *Pp;
  int64_t const g    = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  bool const live    = g < G;
  int64_t const slot = live ? int64_t(map[g]) : 0;

  // keys
  if constexpr (KM == KM_INLINE) {
    uint64_t bits = 0;
    bool kvalid   = true;
    if (live) {
      if (slot < int64_t(P.cap)) bits = P.slot_keys[slot];
      else if (slot == int64_t(P.cap)) bits = EMPTY_KEY;
      else kvalid = false;
      store_width(P.out_keys[0], g, storage_width(P.key_storage), kvalid ? bits : 0);
    }
    if (P.out_key_mask[0]) store_valid_bits(P.out_key_mask[0], g, G, kvalid);
  } else {
    if (live) rep_rows[g] = uint32_t(P.slot_rows[slot]);
  }

  // aggregation results
  for (int o = 0; o < P.num_outs; o++) {
    out_desc const& O = P.outs[o];
    bool valid        = true;
    if (live) {
      uint32_t cnt = 0;
      if (O.count_field != -1) {
        cnt   = count_of(P, O.count_field, slot);
        valid = cnt > 0;
      }
      switch (O.kind) {
        case OK_COPY_I64:
        case OK_COPY_F64: reinterpret_cast<uint64_t*>(O.data)[g] = field_bits(P.fields[O.field], slot); break;
        case OK_COPY_F32: reinterpret_cast<uint32_t*>(O.data)[g] = uint32_t(field_bits(P.fields[O.field], slot)); break;
        case OK_COUNT:
          reinterpret_cast<int32_t*>(O.data)[g] =
            int32_t(*reinterpret_cast<uint32_t const*>(field_at(P.fields[O.field], slot)));
          valid = true;
          break;
        case OK_COUNT_ALL:
          reinterpret_cast<int32_t*>(O.data)[g] = int32_t(*count_at(P, slot));
          valid = true;
          break;
        case OK_MINMAX: {
          field_desc const& F = P.fields[O.field];
          uint64_t b          = field_bits(F, slot);
          if (F.kind == FK_MIN_F32 || F.kind == FK_MAX_F32) b = unord32(uint32_t(b));
          else if (F.kind == FK_MIN_F64 || F.kind == FK_MAX_F64) b = unord64(b);
          store_width(O.data, g, O.out_width, b);
          break;
        }
        case OK_MEAN: {
          double const sum = field_as_double(P.fields[O.field], slot);
          reinterpret_cast<double*>(O.data)[g] = valid ? sum / double(cnt) : 0.0;
          break;
        }
        case OK_SUM_I32:
          reinterpret_cast<int32_t*>(O.data)[g] = int32_t(uint32_t(field_bits(P.fields[O.field], slot)));
          break;
        case OK_MEAN_INT: {  // fixed-point mean: the representation's sum / count, truncated
          int64_t sum = int64_t(field_bits(P.fields[O.field], slot));
          if (O.out_width == 4) sum = int64_t(int32_t(uint32_t(sum)));
          store_width(O.data, g, O.out_width, uint64_t(valid ? sum / int64_t(cnt) : 0));
          break;
        }
        case OK_ARG: {
          uint32_t const r = *reinterpret_cast<uint32_t const*>(field_at(P.fields[O.field], slot));
          valid            = r != 0xFFFFFFFFu;
          reinterpret_cast<int32_t*>(O.data)[g] = valid ? int32_t(r) : -1;
          break;
        }
        case OK_NTH: {  // gather of the value at the group's n-th row
          field_desc const& F = P.fields[O.field];
          dcol const& c       = P.vals[F.vcol];
          uint32_t const r    = *reinterpret_cast<uint32_t const*>(field_at(F, slot));
          valid               = r != 0xFFFFFFFFu && dcol_valid(c, r);
          uint64_t b          = 0;
          if (valid) {
            auto const d = gp(c.data);
            switch (O.out_width) {
              case 1: b = d[r]; break;
              case 2: b = reinterpret_cast<gmem<uint16_t const>*>(d)[r]; break;
              case 4: b = reinterpret_cast<gmem<uint32_t const>*>(d)[r]; break;
              default: b = reinterpret_cast<gmem<uint64_t const>*>(d)[r]; break;
            }
          }
          store_width(O.data, g, O.out_width, b);
          break;
        }
        case OK_VAR:
        case OK_STD: {
          int64_t const dn = int64_t(cnt) - O.ddof;
          valid            = cnt > 0 && dn > 0;
          double var       = 0.0;
          if (valid) var = *reinterpret_cast<double const*>(field_at(P.fields[O.field], slot)) / double(dn);
          reinterpret_cast<double*>(O.data)[g] = (O.kind == OK_STD) ? sqrt(var) : var;
          break;
        }
        default: break;
      }
    }
    if (O.mask) store_valid_bits(O.mask, g, G, valid);
  }
}

void launch_outputs(gb_params const* dP, gb_params const& hP, uint32_t const* map, int64_t G,
                    uint32_t* rep_rows, hipStream_t s)
{
  if (G <= 0) return;
  int64_t blocks = (G + BLOCK - 1) / BLOCK;
  if (hP.key_mode == KM_INLINE)
    hipLaunchKernelGGL(k_outputs<KM_INLINE>, dim3(blocks), dim3(BLOCK), 0, s, dP, map, G, rep_rows);
  else
    hipLaunchKernelGGL(k_outputs<KM_GENERAL>, dim3(blocks), dim3(BLOCK), 0, s, dP, map, G, rep_rows);
}

// ---------------------------------------------------------------------------
// key gather for the general table (fixed-width keys and string lengths).
// With up to GATHER_KEYS_AT_ONCE key columns every column's validity word
// and value (or string offsets) is loaded before the first store, so a
// group costs one round of random reads instead of one or two per column.
constexpr int GATHER_KEYS_AT_ONCE = 4;

__device__ __forceinline__ void gather_key_column(gb_params const& P, int c, int64_t g, int64_t G, bool live,
                                                  bool v, uint64_t x, uint64_t e, int32_t* str_sizes,
                                                  int64_t* str_begin, int& nstr)
{
  dcol const& kc = P.keys[c];
  if (kc.storage == ST_STRING) {
    if (live) {
      str_sizes[int64_t(nstr) * G + g] = v ? int32_t(e - x) : 0;
      str_begin[int64_t(nstr) * G + g] = int64_t(x);
    }
    nstr++;
  } else if (live) {
    store_width(P.out_keys[c], g, storage_width(kc.storage), x);
  }
  if (P.out_key_mask[c]) store_valid_bits(P.out_key_mask[c], g, G, live && v);
}

__device__ __forceinline__ uint64_t raw_key(dcol const& kc, int64_t r)
{
  auto const d = gp(kc.data);
  switch (storage_width(kc.storage)) {
    case 1: return d[r];
    case 2: return reinterpret_cast<gmem<uint16_t const>*>(d)[r];
    case 4: return reinterpret_cast<gmem<uint32_t const>*>(d)[r];
    default: return reinterpret_cast<gmem<uint64_t const>*>(d)[r];
  }
}

__global__ void __launch_bounds__(BLOCK)
  k_gather_keys(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ rep_rows, int64_t G,
                int32_t* str_sizes, int64_t* str_begin)
{
  gb_params const& P = *Pp;
  int64_t const g    = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  bool const live    = g < G;
  int64_t const r    = live ? int64_t(rep_rows[g]) : 0;
  int nstr           = 0;
  if (P.num_keys <= GATHER_KEYS_AT_ONCE) {
    bool v[GATHER_KEYS_AT_ONCE];
    uint64_t x[GATHER_KEYS_AT_ONCE], e[GATHER_KEYS_AT_ONCE];  // value, or string begin / end
#pragma unroll
    for (int c = 0; c < GATHER_KEYS_AT_ONCE; c++) {
      v[c] = false;
      x[c] = e[c] = 0;
      if (c >= P.num_keys) continue;
      dcol const& kc = P.keys[c];
      v[c]           = live && dcol_valid(kc, r);
      if (!live) continue;
      if (kc.storage == ST_STRING) {
        int64_t b0, e0;
        str_span(kc, r, b0, e0);
        x[c] = uint64_t(b0);
        e[c] = uint64_t(e0);
      } else {
        x[c] = raw_key(kc, r);
      }
    }
#pragma unroll
    for (int c = 0; c < GATHER_KEYS_AT_ONCE; c++)
      if (c < P.num_keys) gather_key_column(P, c, g, G, live, v[c], x[c], e[c], str_sizes, str_begin, nstr);
    return;
  }
  for (int c = 0; c < P.num_keys; c++) {
    dcol const& kc = P.keys[c];
    bool const v   = live && dcol_valid(kc, r);
    uint64_t x = 0, e = 0;
    if (live) {
      if (kc.storage == ST_STRING) {
        int64_t b0, e0;
        str_span(kc, r, b0, e0);
        x = uint64_t(b0);
        e = uint64_t(e0);
      } else {
        x = raw_key(kc, r);
      }
    }
    gather_key_column(P, c, g, G, live, v, x, e, str_sizes, str_begin, nstr);
  }
}

void launch_gather_keys(gb_params const* dP, gb_params const& hP, uint32_t const* rep_rows,
                        int64_t G, int32_t* str_sizes, int64_t* str_begin, hipStream_t s)
{
  if (G <= 0) return;
  int64_t blocks = (G + BLOCK - 1) / BLOCK;
  hipLaunchKernelGGL(k_gather_keys, dim3(blocks), dim3(BLOCK), 0, s, dP, rep_rows, G, str_sizes, str_begin);
}

// Exclusive scan of int32 values (three phases: tile sums, scan of sums, apply).
constexpr int I32_TILE = 4096;
__global__ void __launch_bounds__(BLOCK) k_tile_sums_i32(int32_t const* data, int64_t n, uint32_t* sums)
{
  __shared__ uint32_t red[BLOCK / 64];
  int64_t const base = int64_t(blockIdx.x) * I32_TILE;
  uint32_t s = 0;
  for (int k = threadIdx.x; k < I32_TILE; k += BLOCK)
    if (base + k < n) s += uint32_t(data[base + k]);
  s = block_sum_u32(s, red);
  if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

__global__ void __launch_bounds__(BLOCK)
  k_apply_scan_i32(int32_t* data, int64_t n, uint32_t const* tile_offsets)
{
  __shared__ uint32_t wave_tot[BLOCK / 64];
  int64_t const base = int64_t(blockIdx.x) * I32_TILE;
  uint32_t running   = tile_offsets[blockIdx.x];
  int const wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int k = 0; k < I32_TILE; k += BLOCK) {
    int64_t const i = base + k + threadIdx.x;
    uint32_t v      = i < n ? uint32_t(data[i]) : 0u;
    // inclusive scan within the wave
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
      uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wave_tot[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int w = 0; w < BLOCK / 64; w++) {
      if (w < wave) before += wave_tot[w];
      all += wave_tot[w];
    }
    if (i < n) data[i] = int32_t(running + before + x - v);
    running += all;
    __syncthreads();
  }
}

void launch_exclusive_scan_i32(int32_t* data, int64_t n, int32_t* total, hipStream_t s)
{
  // `total` must point at data[n] (one extra element) or be a separate slot.
  int64_t const nt = (n + I32_TILE - 1) / I32_TILE;
  uint32_t* sums   = nullptr;
  MIG_HIP_TRY(hipMallocAsync(reinterpret_cast<void**>(&sums), sizeof(uint32_t) * (nt + 1), s));
  hipLaunchKernelGGL(k_tile_sums_i32, dim3(nt), dim3(BLOCK), 0, s, data, n, sums);
  hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, sums, nt, reinterpret_cast<uint32_t*>(total));
  hipLaunchKernelGGL(k_apply_scan_i32, dim3(nt), dim3(BLOCK), 0, s, data, n, sums);
  MIG_HIP_TRY(hipFreeAsync(sums, s));
}

// Chars of each group's representative string: GATHER_LANES lanes per group
// (strings are short; a wave serves 64 / GATHER_LANES groups).
constexpr int GATHER_LANES = 4;

__global__ void __launch_bounds__(BLOCK)
  k_gather_chars(dcol src, uint32_t const* __restrict__ rep_rows, int64_t G,
                 int32_t const* __restrict__ out_offsets, uint8_t* out_chars)
{
  int64_t const t = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  int64_t const g = t / GATHER_LANES;
  int const lane  = int(t % GATHER_LANES);
  if (g >= G) return;
  int64_t const o   = out_offsets[g];
  int64_t const len = int64_t(out_offsets[g + 1]) - o;
  if (len == 0) return;
  int64_t b, e;
  str_span(src, int64_t(rep_rows[g]), b, e);
  for (int64_t i = lane; i < len; i += GATHER_LANES) gp(out_chars)[o + i] = gp(src.data)[b + i];
}

// The same copy from source offsets k_gather_keys recorded (sequential reads
// instead of a second random read of the string offsets).
__global__ void __launch_bounds__(BLOCK)
  k_gather_chars_from(uint8_t const* __restrict__ src_chars, int64_t const* __restrict__ src_begin, int64_t G,
                      int32_t const* __restrict__ out_offsets, uint8_t* out_chars)
{
  int64_t const t = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  int64_t const g = t / GATHER_LANES;
  int const lane  = int(t % GATHER_LANES);
  if (g >= G) return;
  int64_t const o   = out_offsets[g];
  int64_t const len = int64_t(out_offsets[g + 1]) - o;
  if (len == 0) return;
  int64_t const b = src_begin[g];
  for (int64_t i = lane; i < len; i += GATHER_LANES) gp(out_chars)[o + i] = gp(src_chars)[b + i];
}

void launch_gather_chars_from(uint8_t const* src_chars, int64_t const* src_begin, int64_t G,
                              int32_t const* out_offsets, uint8_t* out_chars, hipStream_t s)
{
  if (G <= 0) return;
  int64_t blocks = (G * GATHER_LANES + BLOCK - 1) / BLOCK;
  hipLaunchKernelGGL(k_gather_chars_from, dim3(blocks), dim3(BLOCK), 0, s, src_chars, src_begin, G, out_offsets,
                     out_chars);
}

void launch_gather_string_chars(dcol const& src, uint32_t const* rep_rows, int64_t G,
                                int32_t const* out_offsets, uint8_t* out_chars, hipStream_t s)
{
  if (G <= 0) return;
  int64_t blocks = (G * GATHER_LANES + BLOCK - 1) / BLOCK;
  hipLaunchKernelGGL(k_gather_chars, dim3(blocks), dim3(BLOCK), 0, s, src, rep_rows, G, out_offsets,
                     out_chars);
}

// Number of valid rows among [0, n) of a column view: popcount of the mask
// words covering bits [mask_offset, mask_offset + n), the partial first and
// last words masked.
__global__ void __launch_bounds__(BLOCK) k_count_valid(dcol c, int64_t n, uint32_t* out)
{
  __shared__ uint32_t red[BLOCK / 64];
  if (c.mask == nullptr) {  // no mask: every row is valid
    if (blockIdx.x == 0 && threadIdx.x == 0) aadd(out, uint32_t(n));
    return;
  }
  int64_t const b0 = c.mask_offset, b1 = int64_t(c.mask_offset) + n;
  int64_t const w0 = b0 >> 5, w1 = (b1 + 31) >> 5;
  uint32_t cnt = 0;
  for (int64_t w = w0 + int64_t(blockIdx.x) * BLOCK + threadIdx.x; w < w1; w += int64_t(gridDim.x) * BLOCK) {
    uint32_t bits = c.mask[w];
    if (w == w0) bits &= ~0u << (b0 & 31);
    if (w == w1 - 1 && (b1 & 31) != 0) bits &= (1u << (b1 & 31)) - 1u;
    cnt += __popc(bits);
  }
  cnt = block_sum_u32(cnt, red);
  if (threadIdx.x == 0 && cnt != 0) aadd(out, cnt);
}

// Set bits among the first n bits of each of up to MASK_LIST masks (word
// aligned, as result masks are): blockIdx.y picks the mask.
constexpr int MASK_LIST = 32;
struct mask_list {
  uint32_t const* mask[MASK_LIST];
};

__global__ void __launch_bounds__(BLOCK) k_count_valid_list(mask_list L, int64_t n, uint32_t* out)
{
  __shared__ uint32_t red[BLOCK / 64];
  auto const mask    = gp(L.mask[blockIdx.y]);
  int64_t const w1   = (n + 31) >> 5;
  uint32_t cnt       = 0;
  for (int64_t w = int64_t(blockIdx.x) * BLOCK + threadIdx.x; w < w1; w += int64_t(gridDim.x) * BLOCK) {
    uint32_t bits = mask[w];
    if (w == w1 - 1 && (n & 31) != 0) bits &= (1u << (n & 31)) - 1u;
    cnt += __popc(bits);
  }
  cnt = block_sum_u32(cnt, red);
  if (threadIdx.x == 0 && cnt != 0) aadd(out + blockIdx.y, cnt);
}

void launch_count_valid_list(uint32_t const* const* masks, int count, int64_t n, uint32_t* d_counts, hipStream_t s)
{
  if (n <= 0) return;
  int64_t blocks = ((n + 31) / 32 + BLOCK - 1) / BLOCK;
  if (blocks > 256) blocks = 256;
  for (int i0 = 0; i0 < count; i0 += MASK_LIST) {
    int const k = count - i0 < MASK_LIST ? count - i0 : MASK_LIST;
    mask_list L{};
    for (int i = 0; i < k; i++) L.mask[i] = masks[i0 + i];
    hipLaunchKernelGGL(k_count_valid_list, dim3(blocks, k), dim3(BLOCK), 0, s, L, n, d_counts + i0);
  }
}

void launch_count_nulls(dcol const& c, int64_t n, uint32_t* d_count, hipStream_t s)
{
  if (n <= 0) return;
  int64_t const words = (int64_t(c.mask_offset & 31) + n + 31) / 32;
  int64_t blocks      = c.mask == nullptr ? 1 : (words + BLOCK - 1) / BLOCK;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(k_count_valid, dim3(blocks), dim3(BLOCK), 0, s, c, n, d_count);
}

// ---------------------------------------------------------------------------
// Pre-sorted keys (groupby(keys, null_policy, sorted::YES)): the groups are
// the runs of equal adjacent key rows, numbered in input order, as the
// reference's sort path finds them with keys_pre_sorted (sort/sort_helper.cu:
// 55-72, 133-181).  k_sorted_count counts run heads per tile, a scan gives
// each tile its first group number, k_sorted_assign writes every row's group
// (NO_GROUP for rows the null policy drops) and each group's first row, and
// the aggregation kernels reduce each 64-row chunk with a segmented scan
// across the wave, so a run costs one atomic per wave and field.
constexpr int SORTED_ROWS = 16;                    // rows per thread per tile
constexpr int SORTED_TILE = BLOCK * SORTED_ROWS;   // rows per tile
constexpr uint32_t NO_GROUP = 0xFFFFFFFFu;

__device__ __forceinline__ bool sorted_included(gb_params const& P, int64_t row)
{
  return !(P.skip_null_keys && any_key_null(P, row));
}

__device__ __forceinline__ bool sorted_head(gb_params const& P, int64_t row)
{
  if (!sorted_included(P, row)) return false;
  if (row == 0 || !sorted_included(P, row - 1)) return true;
  return !rows_equal(P, row, row - 1);
}

// Inclusion and run-head flags of a row (sorted_included, sorted_head).  With
// one fixed-width key column, the common case, the row's and its
// predecessor's validity and key bits are read once each.
__device__ __forceinline__ bool sorted_one_key(gb_params const& P)
{
  return P.num_keys == 1 && P.keys[0].storage != ST_STRING;
}

__device__ __forceinline__ void sorted_flags(gb_params const& P, bool one_key, int64_t row, bool& incl, bool& head)
{
  if (!one_key) {
    incl = sorted_included(P, row);
    head = incl && sorted_head(P, row);
    return;
  }
  dcol const& k = P.keys[0];
  bool const v  = dcol_valid(k, row);
  incl          = v || !P.skip_null_keys;
  head          = incl;
  if (incl && row > 0) {
    bool const pv = dcol_valid(k, row - 1);
    if (pv || !P.skip_null_keys)  // the predecessor is kept: a head when the keys differ (nulls equal)
      head = v != pv || (v && load_fixed_bits(k, row) != load_fixed_bits(k, row - 1));
  }
}

__global__ void __launch_bounds__(BLOCK) k_sorted_count(gb_params const* __restrict__ Pp, uint32_t* block_counts)
{
  __shared__ uint32_t red[BLOCK / 64];
  gb_params const& P = *Pp;
  bool const one_key = sorted_one_key(P);
  int64_t const base = int64_t(blockIdx.x) * SORTED_TILE;
  uint32_t heads = 0;
  for (int j = 0; j < SORTED_ROWS; j++) {
    int64_t const row = base + int64_t(j) * BLOCK + threadIdx.x;
    if (row < P.num_rows) {
      bool incl, head;
      sorted_flags(P, one_key, row, incl, head);
      heads += head ? 1u : 0u;
    }
  }
  uint32_t const t = block_sum_u32<BLOCK>(heads, red);
  if (threadIdx.x == 0) block_counts[blockIdx.x] = t;
}

__global__ void __launch_bounds__(BLOCK)
  k_sorted_assign(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ block_offsets,
                  uint32_t* __restrict__ gid, uint32_t* __restrict__ group_last)
{
  constexpr int NW = BLOCK / 64;
  __shared__ uint32_t wave_tot[NW];
  __shared__ uint64_t head_bal[NW], incl_bal[NW];
  gb_params const& P = *Pp;
  int const wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint64_t const below = (1ull << lane) - 1ull;
  int64_t const base   = int64_t(blockIdx.x) * SORTED_TILE;
  uint32_t running     = block_offsets[blockIdx.x];  // heads before this iteration's rows
  // the block's last thread: its row's group when that row is included and
  // whether the group ends there is decided by the next iteration's first row
  uint32_t pending_g = NO_GROUP;
  uint32_t pending_row = 0;
  bool const one_key   = sorted_one_key(P);
  for (int j = 0; j < SORTED_ROWS; j++) {
    int64_t const row = base + int64_t(j) * BLOCK + threadIdx.x;
    bool const live   = row < P.num_rows;
    bool incl = false, head = false;
    if (live) sorted_flags(P, one_key, row, incl, head);
    uint64_t const bal  = __ballot(head);
    uint64_t const ibal = __ballot(incl);
    if (lane == 0) {
      wave_tot[wave] = uint32_t(__popcll(bal));
      head_bal[wave] = bal;
      incl_bal[wave] = ibal;
    }
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int w = 0; w < NW; w++) {
      if (w < wave) before += wave_tot[w];
      all += wave_tot[w];
    }
    uint32_t const heads_before = running + before + uint32_t(__popcll(bal & below));
    uint32_t const g            = !incl ? NO_GROUP : (head ? heads_before : heads_before - 1u);
    // A group's rows are one run with no dropped row inside (a dropped row
    // ends a run), so its last row is the included row whose successor is
    // dropped, a head or past the end.  The successor's flags come from the
    // wave's ballots, the next wave's (LDS), or for the block's last row the
    // next iteration's first row.
    if (group_last != nullptr) {
      if (pending_g != NO_GROUP && ((incl_bal[0] & 1u) == 0 || (head_bal[0] & 1u) != 0))
        group_last[pending_g] = pending_row;  // the previous iteration's last row (block's last thread only)
      pending_g = NO_GROUP;
      if (incl) {
        bool ends = false;
        if (lane < 63) ends = ((ibal >> (lane + 1)) & 1u) == 0 || ((bal >> (lane + 1)) & 1u) != 0;
        else if (wave < NW - 1) ends = (incl_bal[wave + 1] & 1u) == 0 || (head_bal[wave + 1] & 1u) != 0;
        else if (j + 1 < SORTED_ROWS && row + 1 < P.num_rows) {
          pending_g   = g;
          pending_row = uint32_t(row);
        } else {  // the tile's last row: its successor starts the next tile
          int64_t const nr = row + 1;
          bool ni = false, nh = false;
          if (nr < P.num_rows) sorted_flags(P, one_key, nr, ni, nh);
          ends = !ni || nh;
        }
        if (ends) group_last[g] = uint32_t(row);
      }
    }
    if (live) {
      gid[row] = g;
      if (head) P.slot_rows[g] = uint64_t(row);
    }
    running += all;
    __syncthreads();
  }
}

// Value of one row in the accumulator encoding of field kind `kind`.
__device__ __forceinline__ uint64_t sorted_part(int32_t kind, loaded_value const& v)
{
  switch (kind) {
    case FK_SUM_I64: return uint64_t(v.i);
    case FK_SUM_F32: return __float_as_uint(v.f);
    case FK_SUM_F64: return uint64_t(__double_as_longlong(v.d));
    case FK_SUMSQ_I64: return uint64_t(v.i) * uint64_t(v.i);
    case FK_SUMSQ_F32: return __float_as_uint(v.f * v.f);
    case FK_SUMSQ_F64: return uint64_t(__double_as_longlong(v.d * v.d));
    case FK_MIN_S32:
    case FK_MAX_S32: return uint32_t(int32_t(v.i));
    case FK_MIN_S64:
    case FK_MAX_S64:
    case FK_MIN_U64:
    case FK_MAX_U64: return uint64_t(v.i);
    case FK_MIN_U32:
    case FK_MAX_U32: return uint32_t(v.i);
    case FK_MIN_F32:
    case FK_MAX_F32: return isnan(v.f) ? field_identity(kind) : ord32(uint32_t(v.b));
    case FK_MIN_F64:
    case FK_MAX_F64: return isnan(v.d) ? field_identity(kind) : ord64(v.b);
    case FK_COUNT: return 1;
    case FK_PROD_I64: return uint64_t(v.i);
    case FK_PROD_F32: return __float_as_uint(v.f);
    case FK_PROD_F64: return uint64_t(__double_as_longlong(v.d));
    default: return 0;
  }
}

// Combine two partials in the accumulator encoding.
__device__ __forceinline__ uint64_t sorted_combine(int32_t kind, uint64_t a, uint64_t b)
{
  switch (kind) {
    case FK_SUM_I64:
    case FK_SUMSQ_I64:
    case FK_COUNT: return a + b;
    case FK_SUM_F32:
    case FK_SUMSQ_F32: return __float_as_uint(__uint_as_float(uint32_t(a)) + __uint_as_float(uint32_t(b)));
    case FK_SUM_F64:
    case FK_SUMSQ_F64:
    case FK_M2:
      return uint64_t(__double_as_longlong(__longlong_as_double(int64_t(a)) + __longlong_as_double(int64_t(b))));
    case FK_MIN_S32: return uint32_t(min(int32_t(uint32_t(a)), int32_t(uint32_t(b))));
    case FK_MAX_S32: return uint32_t(max(int32_t(uint32_t(a)), int32_t(uint32_t(b))));
    case FK_MIN_S64: return uint64_t(min(int64_t(a), int64_t(b)));
    case FK_MAX_S64: return uint64_t(max(int64_t(a), int64_t(b)));
    case FK_MIN_U32:
    case FK_MIN_F32: return min(uint32_t(a), uint32_t(b));
    case FK_MAX_U32:
    case FK_MAX_F32: return max(uint32_t(a), uint32_t(b));
    case FK_MIN_U64:
    case FK_MIN_F64: return min(a, b);
    case FK_MAX_U64:
    case FK_MAX_F64: return max(a, b);
    case FK_PROD_I64: return a * b;
    case FK_PROD_F32: return __float_as_uint(__uint_as_float(uint32_t(a)) * __uint_as_float(uint32_t(b)));
    case FK_PROD_F64:
      return uint64_t(__double_as_longlong(__longlong_as_double(int64_t(a)) * __longlong_as_double(int64_t(b))));
    default: return a;
  }
}

// Combining operations of the accumulator kinds (sums and counts add in their
// type; min / max compare signed or unsigned: float min / max accumulators
// hold order-preserving unsigned encodings).
enum seg_op : int32_t {
  OP_ADD_I64 = 0, OP_ADD_F32, OP_ADD_F64, OP_MIN_S32, OP_MAX_S32, OP_MIN_S64, OP_MAX_S64,
  OP_MIN_U32, OP_MAX_U32, OP_MIN_U64, OP_MAX_U64, OP_MUL_I64, OP_MUL_F32, OP_MUL_F64
};

__host__ __device__ inline int32_t seg_op_of(int32_t kind)
{
  switch (kind) {
    case FK_SUM_F32:
    case FK_SUMSQ_F32: return OP_ADD_F32;
    case FK_SUM_F64:
    case FK_SUMSQ_F64:
    case FK_M2: return OP_ADD_F64;
    case FK_MIN_S32: return OP_MIN_S32;
    case FK_MAX_S32: return OP_MAX_S32;
    case FK_MIN_S64: return OP_MIN_S64;
    case FK_MAX_S64: return OP_MAX_S64;
    case FK_MIN_U32:
    case FK_MIN_F32: return OP_MIN_U32;
    case FK_MAX_U32:
    case FK_MAX_F32: return OP_MAX_U32;
    case FK_MIN_U64:
    case FK_MIN_F64: return OP_MIN_U64;
    case FK_MAX_U64:
    case FK_MAX_F64: return OP_MAX_U64;
    case FK_PROD_I64: return OP_MUL_I64;
    case FK_PROD_F32: return OP_MUL_F32;
    case FK_PROD_F64: return OP_MUL_F64;
    default: return OP_ADD_I64;  // integer sums, sums of squares, counts
  }
}

template <int OP>
__device__ __forceinline__ uint64_t op_combine(uint64_t a, uint64_t b)
{
  if constexpr (OP == OP_ADD_I64) return a + b;
  if constexpr (OP == OP_ADD_F32) return __float_as_uint(__uint_as_float(uint32_t(a)) + __uint_as_float(uint32_t(b)));
  if constexpr (OP == OP_ADD_F64)
    return uint64_t(__double_as_longlong(__longlong_as_double(int64_t(a)) + __longlong_as_double(int64_t(b))));
  if constexpr (OP == OP_MIN_S32) return uint32_t(min(int32_t(uint32_t(a)), int32_t(uint32_t(b))));
  if constexpr (OP == OP_MAX_S32) return uint32_t(max(int32_t(uint32_t(a)), int32_t(uint32_t(b))));
  if constexpr (OP == OP_MIN_S64) return uint64_t(min(int64_t(a), int64_t(b)));
  if constexpr (OP == OP_MAX_S64) return uint64_t(max(int64_t(a), int64_t(b)));
  if constexpr (OP == OP_MIN_U32) return min(uint32_t(a), uint32_t(b));
  if constexpr (OP == OP_MAX_U32) return max(uint32_t(a), uint32_t(b));
  if constexpr (OP == OP_MIN_U64) return min(a, b);
  if constexpr (OP == OP_MAX_U64) return max(a, b);
  if constexpr (OP == OP_MUL_I64) return a * b;
  if constexpr (OP == OP_MUL_F32) return __float_as_uint(__uint_as_float(uint32_t(a)) * __uint_as_float(uint32_t(b)));
  if constexpr (OP == OP_MUL_F64)
    return uint64_t(__double_as_longlong(__longlong_as_double(int64_t(a)) * __longlong_as_double(int64_t(b))));
  return a;
}

// One step of the segmented scan: lanes take the partial of the lane the DPP
// control names (row shift within 16-lane rows, or a broadcast of a row's last
// lane to the next rows) and combine it when that lane holds the same group.
// Lanes without a source keep `old`, whose group value matches no group.
template <int OP, int CTRL, int ROW_MASK>
__device__ __forceinline__ void seg_step(uint64_t& part, uint32_t g)
{
  constexpr int NOT_A_GROUP = int(0xFFFFFFFEu);
  uint32_t const olo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(part)), CTRL, ROW_MASK, 0xF, false));
  uint32_t const ohi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(part >> 32)), CTRL, ROW_MASK, 0xF, false));
  uint32_t const og  = uint32_t(__builtin_amdgcn_update_dpp(NOT_A_GROUP, int(g), CTRL, ROW_MASK, 0xF, false));
  if (og == g) part = op_combine<OP>(part, (uint64_t(ohi) << 32) | olo);
}

// Inclusive scan of `part` over the lanes of each run of equal `g` (runs
// are contiguous lanes because group numbers never decrease along rows):
// row shifts by 1, 2, 4, 8 inside each 16-lane row, then row 0's and row 2's
// last lanes into rows 1 and 3, then lane 31 into rows 2 and 3.  A lane only
// combines a partial of its own group, and groups are contiguous, so every
// lane between the source and the lane belongs to the same group.
template <int OP>
__device__ __forceinline__ uint64_t seg_scan(uint64_t part, uint32_t g)
{
  seg_step<OP, 0x111, 0xF>(part, g);  // row_shr:1
  seg_step<OP, 0x112, 0xF>(part, g);  // row_shr:2
  seg_step<OP, 0x114, 0xF>(part, g);  // row_shr:4
  seg_step<OP, 0x118, 0xF>(part, g);  // row_shr:8
  seg_step<OP, 0x142, 0xA>(part, g);  // row_bcast:15
  seg_step<OP, 0x143, 0xC>(part, g);  // row_bcast:31
  return part;
}

// One dispatch on the combining operation per scan.
__device__ __forceinline__ uint64_t segmented_scan(int32_t kind, uint64_t part, uint32_t g, int)
{
  switch (seg_op_of(kind)) {
    case OP_ADD_F32: return seg_scan<OP_ADD_F32>(part, g);
    case OP_ADD_F64: return seg_scan<OP_ADD_F64>(part, g);
    case OP_MIN_S32: return seg_scan<OP_MIN_S32>(part, g);
    case OP_MAX_S32: return seg_scan<OP_MAX_S32>(part, g);
    case OP_MIN_S64: return seg_scan<OP_MIN_S64>(part, g);
    case OP_MAX_S64: return seg_scan<OP_MAX_S64>(part, g);
    case OP_MIN_U32: return seg_scan<OP_MIN_U32>(part, g);
    case OP_MAX_U32: return seg_scan<OP_MAX_U32>(part, g);
    case OP_MIN_U64: return seg_scan<OP_MIN_U64>(part, g);
    case OP_MAX_U64: return seg_scan<OP_MAX_U64>(part, g);
    case OP_MUL_I64: return seg_scan<OP_MUL_I64>(part, g);
    case OP_MUL_F32: return seg_scan<OP_MUL_F32>(part, g);
    case OP_MUL_F64: return seg_scan<OP_MUL_F64>(part, g);
    default: return seg_scan<OP_ADD_I64>(part, g);
  }
}

// Ascending bitonic sort of one 32-bit key per lane across the wave.
__device__ __forceinline__ uint32_t wave_sort_u32(uint32_t key)
{
  int const lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 2; k <= 64; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      uint32_t const other = uint32_t(__shfl_xor(int(key), j));
      bool const keep_min  = ((lane & j) == 0) == ((lane & k) == 0);
      key                  = keep_min ? min(key, other) : max(key, other);
    }
  }
  return key;
}

// The device-wide table with equal groups of a wave combined before the
// atomics: each wave sorts its rows' (slot, lane) pairs, so rows of one group
// sit in adjacent lanes; every accumulator's row contributions are reduced
// over each run by the segmented scan, and the run's last lane applies the
// total with one atomic.  Hot keys then cost one atomic per wave and field
// instead of one per row.
template <int KM>
__global__ void __launch_bounds__(BLOCK) k_aggregate_global_combined(gb_params const* __restrict__ Pp)
{
  constexpr uint32_t NONE = (1u << 26) - 1u;  // sort key of a lane without a group
  gb_params const& P = *Pp;
  int64_t const n    = P.num_rows;
  int const lane     = threadIdx.x & 63;
  for (int64_t base = int64_t(blockIdx.x) * BLOCK; base < n; base += int64_t(gridDim.x) * BLOCK) {
    // the call rebuilds a larger table: stop early (one load of the flag per
    // wave, so the whole wave leaves together)
    if (__builtin_amdgcn_readfirstlane(int(aload(P.overflow))) != 0) break;
    int64_t const row  = base + threadIdx.x;
    int64_t const slot = row < n ? locate<KM, true>(P, row) : -1;
    uint32_t const key = wave_sort_u32(((slot < 0 ? NONE : uint32_t(slot)) << 6) | uint32_t(lane));
    uint32_t const g   = key >> 6;
    int64_t const srow = base + (threadIdx.x & ~63) + int64_t(key & 63u);  // the row this lane now holds
    bool const has     = g != NONE;
    uint32_t const gn  = uint32_t(__shfl_down(int(g), 1));
    bool const tail    = has && (lane == 63 || gn != g);
    if (P.need_count_all) {
      uint64_t const part = seg_scan<OP_ADD_I64>(has ? 1u : 0u, g);
      if (tail) aadd(count_at(P, g), uint32_t(part));
    }
    for (int vc = 0; vc < P.num_vals; vc++) {
      int const fb = P.val_field_begin[vc], fe = P.val_field_begin[vc + 1];
      if (fb == fe) continue;
      dcol const& c    = P.vals[vc];
      bool const valid = has && dcol_valid(c, srow);
      loaded_value v{0, 0.0, 0.0f, 0};
      if (valid) v = load_value(c, srow);
      for (int f = fb; f < fe; f++) {
        field_desc const& F = P.fields[f];
        if (F.kind == FK_M2) continue;  // the second pass
        uint64_t const ident = field_identity(F.kind);
        uint64_t const part  = segmented_scan(F.kind, valid ? sorted_part(F.kind, v) : ident, g, 0);
        if (tail && part != ident) acc_combine(F.kind, field_at(F, g), part);
      }
    }
  }
}

// Accumulators one pass over the rows reduces: up to SORTED_FPP fields
// (index -1: the group row count) reading up to SORTED_COLS value columns.
constexpr int SORTED_FPP  = 8;
constexpr int SORTED_COLS = 4;
struct sorted_pass {
  int32_t n;
  int32_t ncols;
  int32_t field[SORTED_FPP];
  int32_t col_of[SORTED_FPP];   // loaded column slot of each field (-1: the row count)
  int32_t kind[SORTED_FPP];     // accumulator kind (FK_COUNT for the row count)
  int32_t op[SORTED_FPP];       // combining operation (seg_op)
  uint64_t ident[SORTED_FPP];   // identity, in the scan domain (see scan_domain)
  int32_t xf[SORTED_FPP];       // accumulator encoding -> scan domain (scan_domain)
  int32_t col[SORTED_COLS];     // value column (index into P.vals) of each slot
};

// Element bits of a fixed-width column as stored (no float normalisation).
// A string column (width 0) is in a pass only for its validity (COUNT_VALID):
// its chars buffer is not indexed by row, so nothing is loaded.
__device__ __forceinline__ uint64_t raw_bits(dcol const& c, int64_t row)
{
  auto const d = gp(c.data);
  switch (storage_width(c.storage)) {
    case 1: return d[row];
    case 2: return reinterpret_cast<gmem<uint16_t const>*>(d)[row];
    case 4: return reinterpret_cast<gmem<uint32_t const>*>(d)[row];
    case 8: return reinterpret_cast<gmem<uint64_t const>*>(d)[row];
    default: return 0;
  }
}

// The loaded_value of element bits (as load_value builds it from memory).
__device__ __forceinline__ loaded_value value_of_bits(int32_t st, uint64_t u)
{
  loaded_value v{0, 0.0, 0.0f, 0};
  switch (st) {
    case ST_I8: v.i = int8_t(u); break;
    case ST_I16: v.i = int16_t(u); break;
    case ST_I32: v.i = int32_t(u); break;
    case ST_I64: v.i = int64_t(u); break;
    case ST_BOOL: v.i = (u & 0xff) != 0; break;
    case ST_U8: v.i = uint8_t(u); break;
    case ST_U16: v.i = uint16_t(u); break;
    case ST_U32: v.i = uint32_t(u); break;
    case ST_U64: v.i = int64_t(u); v.d = double(u); return v;
    case ST_F32: v.b = uint32_t(u); v.f = __uint_as_float(uint32_t(u)); v.d = double(v.f); return v;
    case ST_F64: v.b = u; v.d = __longlong_as_double(int64_t(u)); return v;
    default: return v;
  }
  v.d = double(v.i);
  return v;
}

__device__ __forceinline__ void sorted_item(gb_params const& P, int32_t f, int64_t g, int32_t& kind, int32_t& width,
                                            void*& ptr)
{
  if (f < 0) {
    kind  = FK_COUNT;
    width = 4;
    ptr   = count_at(P, g);
  } else {
    field_desc const& F = P.fields[f];
    kind  = F.kind;
    width = F.width;
    ptr   = field_at(F, g);
  }
}

// A finished group total: stored when no other wave holds rows of the group,
// combined atomically otherwise (the accumulators start at the identity).
__device__ __forceinline__ void sorted_flush(gb_params const& P, int32_t f, uint32_t g, uint64_t part, bool shared)
{
  int32_t kind, width;
  void* ptr;
  sorted_item(P, f, g, kind, width, ptr);
  if (shared) {
    if (kind == FK_M2) gadd_f64(static_cast<double*>(ptr), __longlong_as_double(int64_t(part)));
    else acc_combine(kind, ptr, part);
  } else if (width == 8) {
    *gp(static_cast<uint64_t*>(ptr)) = part;
  } else {
    *gp(static_cast<uint32_t*>(ptr)) = uint32_t(part);
  }
}

// Row contribution of accumulator `f` (kind `kind`, identity `ident`) from
// the row's loaded value (the value's square deviation from the group mean
// for FK_M2).
__device__ __forceinline__ uint64_t sorted_row_part(gb_params const& P, int32_t f, int32_t kind, uint64_t ident,
                                                    uint32_t g, bool valid, loaded_value const& v)
{
  if (f < 0) return g != NO_GROUP ? 1u : 0u;
  if (g == NO_GROUP || !valid) return ident;
  if (kind != FK_M2) return sorted_part(kind, v);
  field_desc const& F = P.fields[f];
  double const cnt    = double(count_of(P, F.aux_count, g));
  double const mean   = field_as_double(P.fields[F.aux_sum], g) / cnt;
  double const d      = v.d - mean;
  return uint64_t(__double_as_longlong(d * d));
}

// The runs reduction works in a "scan domain" with few combining operations:
// every MIN / MAX accumulator becomes a signed 64-bit MIN / MAX (32-bit
// signed values sign-extended, 32-bit unsigned values and float order codes
// zero-extended, 64-bit unsigned values and float order codes with the sign
// bit flipped, which maps unsigned order onto signed order).  Sums, counts
// and products keep their operation.  Fewer operations, fewer instantiated
// scans: the kernel's hot loop stays small for the instruction cache.
enum scan_xf : int32_t { XF_NONE = 0, XF_SEXT32 = 1, XF_ZEXT32 = 2, XF_FLIP64 = 3 };

__host__ __device__ inline void scan_domain(int32_t kind, int32_t& op, int32_t& xf)
{
  xf = XF_NONE;
  switch (kind) {
    case FK_MIN_S32: op = OP_MIN_S64; xf = XF_SEXT32; return;
    case FK_MAX_S32: op = OP_MAX_S64; xf = XF_SEXT32; return;
    case FK_MIN_U32:
    case FK_MIN_F32: op = OP_MIN_S64; xf = XF_ZEXT32; return;
    case FK_MAX_U32:
    case FK_MAX_F32: op = OP_MAX_S64; xf = XF_ZEXT32; return;
    case FK_MIN_U64:
    case FK_MIN_F64: op = OP_MIN_S64; xf = XF_FLIP64; return;
    case FK_MAX_U64:
    case FK_MAX_F64: op = OP_MAX_S64; xf = XF_FLIP64; return;
    default: op = seg_op_of(kind); return;
  }
}

__host__ __device__ inline uint64_t xf_fwd(int32_t xf, uint64_t u)
{
  switch (xf) {
    case XF_SEXT32: return uint64_t(int64_t(int32_t(uint32_t(u))));
    case XF_ZEXT32: return uint64_t(uint32_t(u));
    case XF_FLIP64: return u ^ 0x8000000000000000ull;
    default: return u;
  }
}

__host__ __device__ inline uint64_t xf_inv(int32_t xf, uint64_t t)
{
  switch (xf) {
    case XF_SEXT32:
    case XF_ZEXT32: return uint64_t(uint32_t(t));
    case XF_FLIP64: return t ^ 0x8000000000000000ull;
    default: return t;
  }
}

// Combine two partials of the scan domain.
__device__ __forceinline__ uint64_t domain_combine(int32_t op, uint64_t a, uint64_t b)
{
  switch (op) {
    case OP_ADD_F32: return op_combine<OP_ADD_F32>(a, b);
    case OP_ADD_F64: return op_combine<OP_ADD_F64>(a, b);
    case OP_MIN_S64: return op_combine<OP_MIN_S64>(a, b);
    case OP_MAX_S64: return op_combine<OP_MAX_S64>(a, b);
    case OP_MUL_I64: return op_combine<OP_MUL_I64>(a, b);
    case OP_MUL_F32: return op_combine<OP_MUL_F32>(a, b);
    case OP_MUL_F64: return op_combine<OP_MUL_F64>(a, b);
    default: return op_combine<OP_ADD_I64>(a, b);
  }
}

// Segmented scan of the scan domain, the operation chosen once per call.
__device__ __forceinline__ uint64_t segmented_scan_op(int32_t op, uint64_t part, uint32_t g)
{
  switch (op) {
    case OP_ADD_F32: return seg_scan<OP_ADD_F32>(part, g);
    case OP_ADD_F64: return seg_scan<OP_ADD_F64>(part, g);
    case OP_MIN_S64: return seg_scan<OP_MIN_S64>(part, g);
    case OP_MAX_S64: return seg_scan<OP_MAX_S64>(part, g);
    case OP_MUL_I64: return seg_scan<OP_MUL_I64>(part, g);
    case OP_MUL_F32: return seg_scan<OP_MUL_F32>(part, g);
    case OP_MUL_F64: return seg_scan<OP_MUL_F64>(part, g);
    default: return seg_scan<OP_ADD_I64>(part, g);
  }
}

// ARGMIN / ARGMAX on runs: a row's partial is (order key of its value, row),
// reduced lexicographically (smallest / largest key, then the smallest row),
// which is the device-wide path's rule (first row among equal values, NaN
// only in an all-NaN group; -0.0 equals 0.0).  Rows without a valid value
// carry the identity key and row 0xFFFFFFFF.
template <bool IS_MIN>
__device__ __forceinline__ void arg_pick(uint64_t& key, uint32_t& row, uint64_t okey, uint32_t orow)
{
  bool const take = IS_MIN ? (okey < key || (okey == key && orow < row)) : (okey > key || (okey == key && orow < row));
  if (take) {
    key = okey;
    row = orow;
  }
}

__device__ __forceinline__ uint64_t arg_order_key(bool is_min, int32_t st, loaded_value const& v)
{
  if (st == ST_F32 || st == ST_F64) {
    if (isnan(v.d)) return is_min ? ~0ull : 0ull;  // a NaN never beats a number
    double const d = v.d == 0.0 ? 0.0 : v.d;        // -0.0 equals 0.0
    return ord64(uint64_t(__double_as_longlong(d)));
  }
  if (is_unsigned_storage_dev(st)) return uint64_t(v.i);
  return uint64_t(v.i) ^ 0x8000000000000000ull;
}

template <bool IS_MIN, int CTRL, int ROW_MASK>
__device__ __forceinline__ void arg_step(uint64_t& key, uint32_t& row, uint32_t g)
{
  constexpr int NOT_A_GROUP = int(0xFFFFFFFEu);
  constexpr int ID_WORD     = IS_MIN ? -1 : 0;
  uint32_t const klo = uint32_t(__builtin_amdgcn_update_dpp(ID_WORD, int(uint32_t(key)), CTRL, ROW_MASK, 0xF, false));
  uint32_t const khi = uint32_t(__builtin_amdgcn_update_dpp(ID_WORD, int(uint32_t(key >> 32)), CTRL, ROW_MASK, 0xF, false));
  uint32_t const orow = uint32_t(__builtin_amdgcn_update_dpp(-1, int(row), CTRL, ROW_MASK, 0xF, false));
  uint32_t const og   = uint32_t(__builtin_amdgcn_update_dpp(NOT_A_GROUP, int(g), CTRL, ROW_MASK, 0xF, false));
  if (og == g) arg_pick<IS_MIN>(key, row, (uint64_t(khi) << 32) | klo, orow);
}

template <bool IS_MIN>
__device__ __forceinline__ void arg_scan(uint64_t& key, uint32_t& row, uint32_t g)
{
  arg_step<IS_MIN, 0x111, 0xF>(key, row, g);  // row_shr:1
  arg_step<IS_MIN, 0x112, 0xF>(key, row, g);  // row_shr:2
  arg_step<IS_MIN, 0x114, 0xF>(key, row, g);  // row_shr:4
  arg_step<IS_MIN, 0x118, 0xF>(key, row, g);  // row_shr:8
  arg_step<IS_MIN, 0x142, 0xA>(key, row, g);  // row_bcast:15
  arg_step<IS_MIN, 0x143, 0xC>(key, row, g);  // row_bcast:31
}

// A finished group's row: stored when no other wave holds rows of the group,
// otherwise merged by the device-wide path's compare-and-swap on the values.
__device__ __forceinline__ void arg_flush(gb_params const& P, int32_t f, uint32_t g, uint32_t row, bool shared)
{
  if (row == 0xFFFFFFFFu) return;  // no valid value: the accumulator keeps "none"
  field_desc const& F = P.fields[f];
  if (shared) arg_update(F, g, P.vals[F.vcol], int64_t(row));
  else *gp(reinterpret_cast<uint32_t*>(field_at(F, g))) = row;
}

// Each wave reduces a contiguous range of rows in 64-row chunks; the group
// still open at a chunk's last lane is carried into the next chunk.  Groups
// that start and end inside the range are stored once; the range's first and
// last groups may have rows in the neighbouring ranges and are combined
// atomically.  HAS_ARG: the pass holds ARGMIN / ARGMAX accumulators (their
// branch is compiled only into that variant, which keeps the common one lean).
template <bool HAS_ARG>
__global__ void __launch_bounds__(BLOCK)
  k_sorted_reduce(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ gid, int64_t per, int64_t W,
                  sorted_pass pass)
{
  // the partials carried between chunks live in LDS (one row per wave): the
  // field loop stays rolled, which keeps the kernel small enough for the
  // instruction cache
  __shared__ uint64_t carry[BLOCK / 64][SORTED_FPP];
  __shared__ uint32_t carry_row[HAS_ARG ? BLOCK / 64 : 1][SORTED_FPP];  // ARGMIN / ARGMAX partials
  gb_params const& P = *Pp;
  int const lane     = threadIdx.x & 63;
  int const wave     = threadIdx.x >> 6;
  int64_t const w    = int64_t(blockIdx.x) * (BLOCK / 64) + wave;
  if (w >= W) return;
  int64_t const b = w * per;
  int64_t const e = b + per < P.num_rows ? b + per : P.num_rows;
  uint32_t const first_g = gid[b];  // may continue from the previous range
  uint32_t carry_g       = NO_GROUP;
  for (int64_t i0 = b; i0 < e; i0 += 64) {
    int64_t const row = i0 + lane;
    bool const live   = row < e;
    int64_t const rc  = live ? row : e - 1;  // every load of the chunk issues before any use
    uint32_t const gl = gid[rc];
    uint64_t bits[SORTED_COLS];
    bool vld[SORTED_COLS];
#pragma unroll
    for (int c = 0; c < SORTED_COLS; c++) {
      bits[c] = 0;
      vld[c]  = false;
      if (c < pass.ncols) {
        dcol const& d = P.vals[pass.col[c]];
        bits[c]       = raw_bits(d, rc);
        vld[c]        = dcol_valid(d, rc);
      }
    }
    // each column's value decoded once per chunk
    loaded_value lv[SORTED_COLS];
#pragma unroll
    for (int c = 0; c < SORTED_COLS; c++)
      lv[c] = c < pass.ncols ? value_of_bits(P.vals[pass.col[c]].storage, bits[c]) : loaded_value{0, 0.0, 0.0f, 0};
    uint32_t const g  = live ? gl : NO_GROUP;
    // group of the next lane (wave_shl:1; the last lane gets no group)
    uint32_t const gn = uint32_t(__builtin_amdgcn_update_dpp(int(NO_GROUP), int(g), 0x130, 0xF, 0xF, false));
    uint32_t const g0 = uint32_t(__builtin_amdgcn_readlane(int(g), 0));
    bool const carry_ends = carry_g != NO_GROUP && g0 != carry_g;
    bool const ends_here  = g != NO_GROUP && lane < 63 && gn != g;
#pragma unroll 1
    for (int k = 0; k < pass.n; k++) {
      int32_t const f    = pass.field[k];
      int32_t const cs   = pass.col_of[k];
      int32_t const kind = pass.kind[k];
      uint64_t const c   = carry[wave][k];
      // the field's column among the loaded ones (uniform select, no indexing)
      loaded_value const v  = cs <= 0 ? lv[0] : cs == 1 ? lv[1] : cs == 2 ? lv[2] : lv[3];
      bool const vv         = cs <= 0 ? vld[0] : cs == 1 ? vld[1] : cs == 2 ? vld[2] : vld[3];
      if (HAS_ARG && (kind == FK_ARGMIN || kind == FK_ARGMAX)) {
        bool const is_min  = kind == FK_ARGMIN;
        uint32_t const crow = carry_row[wave][k];
        if (carry_ends && lane == 0) arg_flush(P, f, carry_g, crow, carry_g == first_g);
        bool const valid = g != NO_GROUP && vv;
        uint64_t key     = valid ? arg_order_key(is_min, P.vals[pass.col[cs]].storage, v) : (is_min ? ~0ull : 0ull);
        uint32_t r       = valid ? uint32_t(row) : 0xFFFFFFFFu;
        if (lane == 0 && carry_g != NO_GROUP && g == carry_g) {
          if (is_min) arg_pick<true>(key, r, c, crow);
          else arg_pick<false>(key, r, c, crow);
        }
        if (is_min) arg_scan<true>(key, r, g);
        else arg_scan<false>(key, r, g);
        if (ends_here) arg_flush(P, f, g, r, g == first_g);
        uint64_t const klast = (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(key >> 32)), 63))) << 32) |
                               uint32_t(__builtin_amdgcn_readlane(int(uint32_t(key)), 63));
        uint32_t const rlast = uint32_t(__builtin_amdgcn_readlane(int(r), 63));
        if (lane == 0) {
          carry[wave][k]     = klast;
          carry_row[wave][k] = rlast;
        }
        continue;
      }
      int32_t const op = pass.op[k], xf = pass.xf[k];
      if (carry_ends && lane == 0) sorted_flush(P, f, carry_g, xf_inv(xf, c), carry_g == first_g);
      uint64_t part = sorted_row_part(P, f, kind, pass.ident[k], g, vv, v);
      if (f >= 0 && g != NO_GROUP && vv) part = xf_fwd(xf, part);  // the identity is already in the domain
      if (lane == 0 && carry_g != NO_GROUP && g == carry_g) part = domain_combine(op, part, c);
      part = segmented_scan_op(op, part, g);
      if (ends_here) sorted_flush(P, f, g, xf_inv(xf, part), g == first_g);
      uint64_t const last = (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(part >> 32)), 63))) << 32) |
                            uint32_t(__builtin_amdgcn_readlane(int(uint32_t(part)), 63));
      if (lane == 0) carry[wave][k] = last;
    }
    carry_g = uint32_t(__builtin_amdgcn_readlane(int(g), 63));
  }
  if (carry_g != NO_GROUP && lane == 0) {
    for (int k = 0; k < pass.n; k++) {  // may continue in the next range
      if (HAS_ARG && (pass.kind[k] == FK_ARGMIN || pass.kind[k] == FK_ARGMAX))
        arg_flush(P, pass.field[k], carry_g, carry_row[wave][k], true);
      else
        sorted_flush(P, pass.field[k], carry_g, xf_inv(pass.xf[k], carry[wave][k]), true);
    }
  }
}

__global__ void __launch_bounds__(BLOCK) k_iota_u32(uint32_t* out, int64_t n)
{
  int64_t const i = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (i < n) out[i] = uint32_t(i);
}

void launch_sorted_count(gb_params const* dP, int64_t n, uint32_t* block_counts, hipStream_t s)
{
  int64_t const nb = (n + SORTED_TILE - 1) / SORTED_TILE;
  hipLaunchKernelGGL(k_sorted_count, dim3(nb), dim3(BLOCK), 0, s, dP, block_counts);
}

void launch_sorted_assign(gb_params const* dP, int64_t n, uint32_t const* block_offsets, uint32_t* gid,
                          uint32_t* group_last, hipStream_t s)
{
  int64_t const nb = (n + SORTED_TILE - 1) / SORTED_TILE;
  hipLaunchKernelGGL(k_sorted_assign, dim3(nb), dim3(BLOCK), 0, s, dP, block_offsets, gid, group_last);
}

int64_t sorted_tiles(int64_t n) { return (n + SORTED_TILE - 1) / SORTED_TILE; }

// Wave ranges: enough waves to fill the device, at least 64 rows each.
static void sorted_ranges(int64_t n, int num_cus, int64_t& per, int64_t& W)
{
  int64_t const target = int64_t(num_cus) * 64;
  per = ((n + target - 1) / target + 63) / 64 * 64;
  if (per < 64) per = 64;
  W = (n + per - 1) / per;
}

// ---------------------------------------------------------------------------
// Column statistics on runs.  A value column whose accumulators are all among
// SUM, SUM_OF_SQUARES, COUNT, MIN, MAX and M2 (VARIANCE / STD), stored as int32, int64,
// float32 or float64, is reduced by a kernel compiled for its type: the combining
// operations are fixed at compile time, the segment masks of the six scan
// steps are computed once per chunk for all accumulators, and the partials
// carried between chunks stay in registers.  M2 comes from the sums in the
// same pass where that is exact or within the bound below; the groups where
// it is not (and the groups a wave shares with its neighbours) get the exact
// two-pass M2 (the reference's mean, then squared deviations:
// sort/group_std.cu:60-69 through sort/aggregate.cpp:286-306): groups of at most
// M2_WAVE_ROWS rows are listed and reduced by one wave each
// (k_sorted_stats_m2_list), longer ones are flagged for the row-parallel
// k_sorted_stats_m2, which returns at once when none is.
template <int ST>
struct stats_traits;
template <>
struct stats_traits<ST_I32> {
  using T   = int32_t;
  using Sum = int64_t;
  using Ord = int32_t;  // MIN / MAX domain
};
template <>
struct stats_traits<ST_I64> {
  using T   = int64_t;
  using Sum = int64_t;
  using Ord = int64_t;
};
template <>
struct stats_traits<ST_F64> {
  using T   = double;
  using Sum = double;
  using Ord = int64_t;
};
template <>
struct stats_traits<ST_F32> {
  using T   = float;
  using Sum = double;  // float32 sums and sums of squares accumulate in double, rounded once when stored
  using Ord = int32_t;
};

// Value of a row in the signed MIN / MAX domain (floats: the order code with
// the sign bit flipped, as scan_domain maps them; integers: themselves).
template <int ST>
__device__ __forceinline__ typename stats_traits<ST>::Ord stats_order(typename stats_traits<ST>::T x)
{
  if constexpr (ST == ST_F64) return int64_t(ord64(uint64_t(__double_as_longlong(x))) ^ 0x8000000000000000ull);
  else if constexpr (ST == ST_F32) return int32_t(ord32(__float_as_uint(x)) ^ 0x80000000u);
  else return x;
}

// The accumulator value of a MIN / MAX domain value.
template <int ST>
__device__ __forceinline__ typename stats_traits<ST>::Ord stats_order_inv(typename stats_traits<ST>::Ord t)
{
  if constexpr (ST == ST_F64) return int64_t(uint64_t(t) ^ 0x8000000000000000ull);
  else if constexpr (ST == ST_F32) return int32_t(uint32_t(t) ^ 0x80000000u);
  else return t;
}

// Same-group masks of the six scan steps (see seg_scan): lane l combines the
// partial the step's DPP control brings when that lane holds l's group.
struct seg_masks {
  bool s[6];
};

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ bool seg_same(uint32_t g)
{
  constexpr int NOT_A_GROUP = int(0xFFFFFFFEu);
  return uint32_t(__builtin_amdgcn_update_dpp(NOT_A_GROUP, int(g), CTRL, ROW_MASK, 0xF, false)) == g;
}

__device__ __forceinline__ seg_masks seg_masks_of(uint32_t g)
{
  return seg_masks{{seg_same<0x111, 0xF>(g), seg_same<0x112, 0xF>(g), seg_same<0x114, 0xF>(g),
                    seg_same<0x118, 0xF>(g), seg_same<0x142, 0xA>(g), seg_same<0x143, 0xC>(g)}};
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp64(uint64_t x)
{
  uint32_t const lo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(x)), CTRL, ROW_MASK, 0xF, false));
  uint32_t const hi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(x >> 32)), CTRL, ROW_MASK, 0xF, false));
  return (uint64_t(hi) << 32) | lo;
}

// Segmented inclusive scan with precomputed masks; `F` combines two partials.
template <typename V, typename F>
__device__ __forceinline__ V mscan(V x, seg_masks const& m, F&& f)
{
  auto step = [&](auto ctrl, auto rmask, bool same) {
    constexpr int C = decltype(ctrl)::value, R = decltype(rmask)::value;
    V o;
    if constexpr (sizeof(V) == 8) {
      uint64_t const u = dpp64<C, R>(__builtin_bit_cast(uint64_t, x));
      o                = __builtin_bit_cast(V, u);
    } else {
      o = __builtin_bit_cast(V, uint32_t(__builtin_amdgcn_update_dpp(0, int(__builtin_bit_cast(uint32_t, x)), C, R,
                                                                     0xF, false)));
    }
    if (same) x = f(x, o);
  };
  step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xF>{}, m.s[0]);
  step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xF>{}, m.s[1]);
  step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xF>{}, m.s[2]);
  step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xF>{}, m.s[3]);
  step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{}, m.s[4]);
  step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{}, m.s[5]);
  return x;
}

template <typename V>
__device__ __forceinline__ V lane63(V x)
{
  if constexpr (sizeof(V) == 8) {
    uint64_t const u = __builtin_bit_cast(uint64_t, x);
    uint64_t const r = (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u >> 32)), 63))) << 32) |
                       uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u)), 63));
    return __builtin_bit_cast(V, r);
  } else {
    return __builtin_bit_cast(V, uint32_t(__builtin_amdgcn_readlane(int(__builtin_bit_cast(uint32_t, x)), 63)));
  }
}

// M2 of a whole group from its count n, sum s1 and sum of squares s2 (the
// rule of the partitioned path's m2_from_sums): integer sources while s2 <
// 2^53 (every partial then exact in double) through n·M2 = n·s2 − s1² in 128
// bits; float64 sources with at most 256 values when the rounding error of
// s2 − s1²/n, at most ~3·n·ε·s2, is below 1e-11 of the result.  False: the
// group goes to the exact pass.
template <int ST>
__device__ __forceinline__ bool stats_m2(uint32_t n, typename stats_traits<ST>::Sum s1, double s2, double& m2)
{
  if (n <= 1 && isfinite(s2)) {  // one finite value (or none): no deviation; NaN / inf give NaN below
    m2 = 0.0;
    return true;
  }
  if constexpr (ST == ST_F64 || ST == ST_F32) {  // float32 values: exact squares, sums in double
    if (n > 256) return false;
    double const v = s2 - s1 * (s1 / double(n));
    if (!(v > 0.0) || 3.0 * double(n) * 1.1102230246251565e-16 * s2 > 1e-11 * v) {
      m2 = 0.0;
      return v == 0.0 && s2 == 0.0;
    }
    m2 = v;
    return true;
  } else {
    if (!(s2 < 9007199254740992.0)) return false;
    if (double(n) * s2 < 9.2e18) {  // n·s2 < 2^63, and s1² <= n·s2: 64 bits hold both
      int64_t const num = int64_t(n) * int64_t(s2) - s1 * s1;
      m2                = double(num) / double(n);
      return true;
    }
    __int128 const num = __int128(n) * __int128(uint64_t(s2)) - __int128(s1) * __int128(s1);
    m2                 = double(num) / double(n);
    return true;
  }
}

struct sorted_stats_job {
  int32_t vcol;
  int32_t f_sum, f_count, f_min, f_max, f_m2;  // field index, -1 when not requested
  int32_t f_sumsq;
  int32_t count_rows;                          // also the group row count
  int64_t min_ident, max_ident;                // identities in the MIN / MAX domain
  // the accumulators of the fields above (arrays of G entries)
  uint32_t* p_rows;
  uint32_t* p_count;
  void* p_sum;
  void* p_min;
  void* p_max;
  void* p_sumsq;
  double* p_m2;
  uint8_t* m2_flag;                            // per group: 1 = M2 by the row-parallel exact pass
  uint32_t* m2_list;                           // groups whose M2 one wave each recomputes
  uint32_t* m2_counts;                         // [0] listed groups, [1] flagged groups
};

// Longest group whose exact M2 one wave recomputes; longer groups take the
// row-parallel pass.
constexpr int64_t M2_WAVE_ROWS = 4096;

template <int ST>
struct stats_part {
  uint32_t rows, cnt;
  typename stats_traits<ST>::Sum sum;
  typename stats_traits<ST>::Ord mn, mx;
  double sq;     // Σx² in double (M2; SUM_OF_SQUARES of float64)
  uint64_t isq;  // Σx² of integers, wrapping (SUM_OF_SQUARES of int32 / int64)
};

// A group's partials: stored when the group lies inside one wave's range,
// combined atomically when neighbouring ranges hold rows of it.
// `ends`: no later row of the group follows (this is the group's last flush),
// and `last_row` is then its last row.
template <int ST>
__device__ __forceinline__ void stats_flush(gb_params const& P, sorted_stats_job const& J, uint32_t g,
                                            stats_part<ST> const& a, bool shared, bool ends, int64_t last_row)
{
  using Sum = typename stats_traits<ST>::Sum;
  using Ord = typename stats_traits<ST>::Ord;
  if (J.count_rows) {
    if (shared) aadd(J.p_rows + g, a.rows);
    else *gp(J.p_rows + g) = a.rows;
  }
  if (J.f_count >= 0) {
    if (shared) aadd(J.p_count + g, a.cnt);
    else *gp(J.p_count + g) = a.cnt;
  }
  if (J.f_sum >= 0) {
    if constexpr (ST == ST_F32) {
      float* p = static_cast<float*>(J.p_sum) + g;
      if (shared) gadd_f32(p, float(a.sum));
      else *gp(p) = float(a.sum);
    } else if constexpr (ST == ST_F64) {
      Sum* p = static_cast<Sum*>(J.p_sum) + g;
      if (shared) gadd_f64(p, a.sum);
      else *gp(p) = a.sum;
    } else {
      Sum* p = static_cast<Sum*>(J.p_sum) + g;
      if (shared) aadd(reinterpret_cast<uint64_t*>(p), uint64_t(a.sum));
      else *gp(p) = a.sum;
    }
  }
  // MIN / MAX accumulators: int32 / int64 values, float order codes (unsigned)
  if (J.f_min >= 0) {
    Ord const u = stats_order_inv<ST>(a.mn);
    Ord* p      = static_cast<Ord*>(J.p_min) + g;
    if (!shared) *gp(p) = u;
    else if constexpr (ST == ST_F64) amin(reinterpret_cast<uint64_t*>(p), uint64_t(u));
    else if constexpr (ST == ST_F32) amin(reinterpret_cast<uint32_t*>(p), uint32_t(u));
    else amin(p, u);
  }
  if (J.f_max >= 0) {
    Ord const u = stats_order_inv<ST>(a.mx);
    Ord* p      = static_cast<Ord*>(J.p_max) + g;
    if (!shared) *gp(p) = u;
    else if constexpr (ST == ST_F64) amax(reinterpret_cast<uint64_t*>(p), uint64_t(u));
    else if constexpr (ST == ST_F32) amax(reinterpret_cast<uint32_t*>(p), uint32_t(u));
    else amax(p, u);
  }
  if (J.f_sumsq >= 0) {
    if constexpr (ST == ST_F32) {
      float* p = static_cast<float*>(J.p_sumsq) + g;
      if (shared) gadd_f32(p, float(a.sq));
      else *gp(p) = float(a.sq);
    } else if constexpr (ST == ST_F64) {
      double* p = static_cast<double*>(J.p_sumsq) + g;
      if (shared) gadd_f64(p, a.sq);
      else *gp(p) = a.sq;
    } else {
      uint64_t* p = static_cast<uint64_t*>(J.p_sumsq) + g;
      if (shared) aadd(p, a.isq);
      else *gp(p) = a.isq;
    }
  }
  if (J.f_m2 >= 0) {
    double m2        = 0.0;
    bool const exact = !shared && stats_m2<ST>(a.cnt, a.sum, a.sq, m2);  // a group not shared ends here
    if (exact) {
      if (m2 != 0.0) *gp(J.p_m2 + g) = m2;
      *gp(J.m2_flag + g) = 0;
    } else if (ends) {  // once per group: its last flush
      bool const large   = last_row - int64_t(gp(P.slot_rows)[g]) + 1 > M2_WAVE_ROWS;
      *gp(J.m2_flag + g) = large ? 1 : 0;
      if (large) aadd(J.m2_counts + 1, 1u);
      else *gp(J.m2_list + __hip_atomic_fetch_add(J.m2_counts, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) = g;
    }
  }
}

// Rows per lane in k_sorted_stats: a lane first combines its consecutive rows
// serially, so one cross-lane scan covers 64 * STATS_ROWS rows.
constexpr int STATS_ROWS = 4;

// Two partials of one group combined.
template <int ST>
__device__ __forceinline__ stats_part<ST> stats_combine(stats_part<ST> a, stats_part<ST> const& b)
{
  a.rows += b.rows;
  a.cnt += b.cnt;
  a.sum += b.sum;
  a.sq += b.sq;
  a.isq += b.isq;
  a.mn = a.mn < b.mn ? a.mn : b.mn;
  a.mx = a.mx > b.mx ? a.mx : b.mx;
  return a;
}

// One wave per contiguous row range (the range layout and the carry between
// chunks of k_sorted_reduce), chunks of 64 * STATS_ROWS rows with
// STATS_ROWS consecutive rows per lane.  A lane's rows are combined serially;
// a group that ends inside the lane (before its last row) is finished there
// with the scan total of the lanes before it, and the partial of the lane's
// last group takes part in the segmented scan across the wave.
template <int ST>
__global__ void __launch_bounds__(BLOCK)
  k_sorted_stats(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ gid, int64_t per, int64_t W,
                 sorted_stats_job J)
{
  using T            = typename stats_traits<ST>::T;
  using Sum          = typename stats_traits<ST>::Sum;
  using Ord          = typename stats_traits<ST>::Ord;
  constexpr int K    = STATS_ROWS;
  gb_params const& P = *Pp;
  int const lane     = threadIdx.x & 63;
  int64_t const w    = int64_t(blockIdx.x) * (BLOCK / 64) + (threadIdx.x >> 6);
  if (w >= W) return;
  int64_t const b = w * per;
  int64_t const e = b + per < P.num_rows ? b + per : P.num_rows;
  dcol const c    = P.vals[J.vcol];
  auto const* data = reinterpret_cast<gmem<T const>*>(gp(c.data));
  constexpr bool FLOAT = ST == ST_F64 || ST == ST_F32;
  bool const want_sq  = J.f_m2 >= 0 || (FLOAT && J.f_sumsq >= 0);
  bool const want_isq = !FLOAT && J.f_sumsq >= 0;
  uint32_t const first_g = gid[b];  // may continue from the previous range
  uint32_t carry_g       = NO_GROUP;
  Ord const min_ident    = Ord(J.min_ident);
  Ord const max_ident    = Ord(J.max_ident);
  stats_part<ST> const none{0, 0, Sum(0), min_ident, max_ident, 0.0, 0};
  stats_part<ST> cy = none;
  for (int64_t i0 = b; i0 < e; i0 += 64 * K) {
    int64_t const r0 = i0 + int64_t(K) * lane;  // the lane's first row
    uint32_t gg[K];
    stats_part<ST> a[K];
#pragma unroll
    for (int u = 0; u < K; u++) {
      int64_t const row = r0 + u;
      bool const live   = row < e;
      int64_t const rc  = live ? row : e - 1;
      uint32_t const gl = gid[rc];
      T const x         = data[rc];
      bool const vv     = dcol_valid(c, rc);
      gg[u]             = live ? gl : NO_GROUP;
      bool const has    = gg[u] != NO_GROUP && vv;
      a[u].rows         = gg[u] != NO_GROUP ? 1u : 0u;
      a[u].cnt          = has ? 1u : 0u;
      a[u].sum          = has ? Sum(x) : Sum(0);
      a[u].sq           = has && want_sq ? double(x) * double(x) : 0.0;
      a[u].isq          = has && want_isq ? uint64_t(int64_t(x)) * uint64_t(int64_t(x)) : 0;
      bool ordered      = has;
      if constexpr (FLOAT) ordered = has && !isnan(x);  // NaN takes no part in MIN / MAX
      Ord const t = stats_order<ST>(x);
      a[u].mn     = ordered ? t : min_ident;
      a[u].mx     = ordered ? t : max_ident;
    }
    uint32_t const g0 = uint32_t(__builtin_amdgcn_readlane(int(gg[0]), 0));
    if (carry_g != NO_GROUP && g0 != carry_g) {
      if (lane == 0) stats_flush<ST>(P, J, carry_g, cy, carry_g == first_g, true, i0 - 1);
    } else if (carry_g != NO_GROUP && lane == 0) {  // the carried group continues at lane 0
      a[0] = stats_combine<ST>(a[0], cy);
    }
    // the lane's rows, serially: `first` holds the lane's first group when
    // that group ends inside the lane
    uint32_t cur = gg[0];
    stats_part<ST> R = a[0], first = none;
    bool split = false;
#pragma unroll
    for (int u = 1; u < K; u++) {
      if (gg[u] == cur) {
        R = stats_combine<ST>(R, a[u]);
      } else {
        if (!split) {
          first = R;
          split = true;
        } else if (cur != NO_GROUP) {  // a group wholly inside the lane (more than two rows per lane)
          stats_flush<ST>(P, J, cur, R, cur == first_g, true, r0 + u - 1);
        }
        cur = gg[u];
        R   = a[u];
      }
    }
    seg_masks const m = seg_masks_of(cur);
    auto add32        = [](uint32_t p, uint32_t q) { return p + q; };
    if (J.count_rows) R.rows = mscan(R.rows, m, add32);
    R.cnt = mscan(R.cnt, m, add32);
    R.sum = mscan(R.sum, m, [](Sum p, Sum q) { return p + q; });
    if (J.f_min >= 0) R.mn = mscan(R.mn, m, [](Ord p, Ord q) { return p < q ? p : q; });
    if (J.f_max >= 0) R.mx = mscan(R.mx, m, [](Ord p, Ord q) { return p > q ? p : q; });
    if (want_sq) R.sq = mscan(R.sq, m, [](double p, double q) { return p + q; });
    if (want_isq) R.isq = mscan(R.isq, m, [](uint64_t p, uint64_t q) { return p + q; });
    // a first group that ended inside the lane: its rows in the lanes before
    // (the previous lane's scan total when that lane's last group is the same)
    uint32_t const cprev = uint32_t(__builtin_amdgcn_update_dpp(int(NO_GROUP), int(cur), 0x138, 0xF, 0xF, false));
    stats_part<ST> prev;
    prev.rows = uint32_t(__builtin_amdgcn_update_dpp(0, int(R.rows), 0x138, 0xF, 0xF, false));
    prev.cnt  = uint32_t(__builtin_amdgcn_update_dpp(0, int(R.cnt), 0x138, 0xF, 0xF, false));
    prev.sum  = __builtin_bit_cast(Sum, dpp64<0x138, 0xF>(__builtin_bit_cast(uint64_t, R.sum)));
    if constexpr (sizeof(Ord) == 8) {
      prev.mn = __builtin_bit_cast(Ord, dpp64<0x138, 0xF>(__builtin_bit_cast(uint64_t, R.mn)));
      prev.mx = __builtin_bit_cast(Ord, dpp64<0x138, 0xF>(__builtin_bit_cast(uint64_t, R.mx)));
    } else {
      prev.mn = Ord(__builtin_amdgcn_update_dpp(0, int(R.mn), 0x138, 0xF, 0xF, false));
      prev.mx = Ord(__builtin_amdgcn_update_dpp(0, int(R.mx), 0x138, 0xF, 0xF, false));
    }
    prev.sq  = __builtin_bit_cast(double, dpp64<0x138, 0xF>(__builtin_bit_cast(uint64_t, R.sq)));
    prev.isq = dpp64<0x138, 0xF>(R.isq);
    if (split && gg[0] != NO_GROUP) {
      stats_part<ST> const tot = lane > 0 && cprev == gg[0] ? stats_combine<ST>(first, prev) : first;
      stats_flush<ST>(P, J, gg[0], tot, gg[0] == first_g, true, r0);
    }
    // the lane's last group ends at the lane's last row when the next lane
    // starts another group
    uint32_t const gnext = uint32_t(__builtin_amdgcn_update_dpp(int(NO_GROUP), int(gg[0]), 0x130, 0xF, 0xF, false));
    if (cur != NO_GROUP && lane < 63 && gnext != cur) stats_flush<ST>(P, J, cur, R, cur == first_g, true, r0 + K - 1);
    cy.rows = lane63(R.rows);
    cy.cnt  = lane63(R.cnt);
    cy.sum  = lane63(R.sum);
    cy.mn   = lane63(R.mn);
    cy.mx   = lane63(R.mx);
    cy.sq   = lane63(R.sq);
    cy.isq  = lane63(R.isq);
    carry_g = uint32_t(__builtin_amdgcn_readlane(int(cur), 63));
  }
  if (carry_g != NO_GROUP && lane == 0) {  // may continue in the next range
    bool const ends = e == P.num_rows || gid[e] != carry_g;
    stats_flush<ST>(P, J, carry_g, cy, true, ends, e - 1);
  }
}

// The exact M2 of the flagged (long) groups: Σ(x − mean)² with the mean from
// the finished sum and count, summed over each run of a chunk and added to
// the group's M2 once per chunk.  Chunks without a flagged row only read
// their group numbers and flags; with no flagged group every wave returns
// after reading the count.
template <int ST>
__global__ void __launch_bounds__(BLOCK)
  k_sorted_stats_m2(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ gid, sorted_stats_job J)
{
  using T            = typename stats_traits<ST>::T;
  gb_params const& P = *Pp;
  if (aload(J.m2_counts + 1) == 0) return;
  int64_t const n    = P.num_rows;
  int const lane     = threadIdx.x & 63;
  dcol const c       = P.vals[J.vcol];
  auto const* data   = reinterpret_cast<gmem<T const>*>(gp(c.data));
  field_desc const& F = P.fields[J.f_m2];
  for (int64_t base = int64_t(blockIdx.x) * BLOCK + (threadIdx.x & ~63); base < n;
       base += int64_t(gridDim.x) * BLOCK) {
    int64_t const row = base + lane;
    uint32_t const g  = row < n ? gid[row] : NO_GROUP;
    bool const fl     = g != NO_GROUP && gp(J.m2_flag)[g] != 0;
    if (__builtin_amdgcn_ballot_w64(fl) == 0) continue;
    double d2 = 0.0;
    if (fl && dcol_valid(c, row)) {
      double const cnt  = double(count_of(P, F.aux_count, g));
      double const mean = field_as_double(P.fields[F.aux_sum], g) / cnt;
      double const d    = double(data[row]) - mean;
      d2                = d * d;
    }
    uint32_t const gk  = fl ? g : NO_GROUP;
    seg_masks const m  = seg_masks_of(gk);
    d2                 = mscan(d2, m, [](double p, double q) { return p + q; });
    uint32_t const gn  = uint32_t(__builtin_amdgcn_update_dpp(int(NO_GROUP), int(gk), 0x130, 0xF, 0xF, false));
    if (fl && (lane == 63 || gn != gk) && d2 != 0.0) gadd_f64(reinterpret_cast<double*>(field_at(F, g)), d2);
  }
}

// The exact M2 of the listed groups (at most M2_WAVE_ROWS rows each): one
// wave per group walks its rows from the first (the runs are contiguous),
// sums the squared deviations in its lanes, reduces them across the wave and
// stores the group's M2 (the only writer).
template <int ST>
__global__ void __launch_bounds__(BLOCK)
  k_sorted_stats_m2_list(gb_params const* __restrict__ Pp, uint32_t const* __restrict__ gid, sorted_stats_job J)
{
  using T             = typename stats_traits<ST>::T;
  gb_params const& P  = *Pp;
  int64_t const n     = P.num_rows;
  int const lane      = threadIdx.x & 63;
  dcol const c        = P.vals[J.vcol];
  auto const* data    = reinterpret_cast<gmem<T const>*>(gp(c.data));
  field_desc const& F = P.fields[J.f_m2];
  uint32_t const listed = aload(J.m2_counts);
  for (uint32_t i = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6); i < listed; i += gridDim.x * (BLOCK / 64)) {
    uint32_t const g    = gp(J.m2_list)[i];
    int64_t const first = int64_t(gp(P.slot_rows)[g]);
    double const cnt    = double(count_of(P, F.aux_count, g));
    double const mean   = field_as_double(P.fields[F.aux_sum], g) / cnt;
    double acc          = 0.0;
    for (int64_t r0 = first; r0 < n; r0 += 64) {
      int64_t const row = r0 + lane;
      bool const in     = row < n && gid[row] == g;
      if (in && dcol_valid(c, row)) {
        double const d = double(data[row]) - mean;
        acc += d * d;
      }
      if (__builtin_amdgcn_ballot_w64(in) != ~0ull) break;  // the run ended in this chunk
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) *gp(reinterpret_cast<double*>(field_at(F, g))) = acc;
  }
}

__global__ void k_zero_u32(uint32_t* p, int n)
{
  if (int(threadIdx.x) < n) p[threadIdx.x] = 0;
}

template <int ST>
static void launch_stats_job(gb_params const* dP, sorted_stats_job const& J, int64_t n, uint32_t const* gid,
                             int num_cus, hipStream_t s)
{
  int64_t per, W;
  sorted_ranges(n, num_cus, per, W);
  // ranges of whole chunks: a range then ends at a chunk's last lane, so a
  // group at a range's end is always carried (and combined atomically)
  constexpr int64_t CH = 64 * STATS_ROWS;
  per = (per + CH - 1) / CH * CH;
  W   = (n + per - 1) / per;
  unsigned const blocks = unsigned((W + BLOCK / 64 - 1) / (BLOCK / 64));
  hipLaunchKernelGGL(k_sorted_stats<ST>, dim3(blocks), dim3(BLOCK), 0, s, dP, gid, per, W, J);
}

template <int ST>
static void launch_stats_m2(gb_params const* dP, sorted_stats_job const& J, int64_t n, uint32_t const* gid,
                            int num_cus, hipStream_t s)
{
  hipLaunchKernelGGL(k_sorted_stats_m2_list<ST>, dim3(unsigned(num_cus * 8)), dim3(BLOCK), 0, s, dP, gid, J);
  hipLaunchKernelGGL(k_sorted_stats_m2<ST>, dim3(unsigned(row_grid(n, num_cus, 8))), dim3(BLOCK), 0, s, dP, gid, J);
}

static bool stats_kind_ok(int32_t st, int32_t kind)
{
  switch (kind) {
    case FK_COUNT:
    case FK_M2: return true;
    case FK_SUM_I64: return st == ST_I32 || st == ST_I64;
    case FK_SUM_F64: return st == ST_F64;
    case FK_SUMSQ_I64: return st == ST_I32 || st == ST_I64;
    case FK_SUMSQ_F64: return st == ST_F64;
    case FK_SUM_F32:
    case FK_SUMSQ_F32:
    case FK_MIN_F32:
    case FK_MAX_F32: return st == ST_F32;
    case FK_MIN_S32:
    case FK_MAX_S32: return st == ST_I32;
    case FK_MIN_S64:
    case FK_MAX_S64: return st == ST_I64;
    case FK_MIN_F64:
    case FK_MAX_F64: return st == ST_F64;
    default: return false;
  }
}

// The column jobs of a request: every value column whose fields all have a
// specialised form.  The first job also counts the group rows when the
// request needs them.
// Device scratch of one column with M2: per-group flags, the list of groups
// and two counters.
static size_t m2_column_bytes(int64_t G)
{
  size_t const g = size_t(G > 0 ? G : 1);
  return ((g + 255) & ~size_t(255)) + ((4 * g + 255) & ~size_t(255)) + 256;
}

size_t sorted_stats_scratch_bytes(int64_t G, int m2_columns) { return m2_column_bytes(G) * size_t(m2_columns); }

static std::vector<std::pair<int32_t, sorted_stats_job>> stats_jobs(gb_params const& hP, uint8_t* m2_scratch,
                                                                   int64_t G)
{
  std::vector<std::pair<int32_t, sorted_stats_job>> jobs;
  int64_t m2_jobs = 0;
  for (int j = 0; j < hP.num_vals; j++) {
    int32_t const st = hP.vals[j].storage;
    int const fb = hP.val_field_begin[j], fe = hP.val_field_begin[j + 1];
    if (fb == fe || (st != ST_I32 && st != ST_I64 && st != ST_F64 && st != ST_F32)) continue;
    sorted_stats_job J{};
    J.vcol = j;
    J.f_sum = J.f_count = J.f_min = J.f_max = J.f_m2 = J.f_sumsq = -1;
    bool ok = true;
    // the kernels index accumulators as dense arrays
    if (hP.need_count_all && hP.count_stride != 4) continue;
    for (int f = fb; f < fe && ok; f++) {
      int32_t const k = hP.fields[f].kind;
      ok              = stats_kind_ok(st, k) && hP.fields[f].stride == hP.fields[f].width;
      int32_t* slot   = k == FK_COUNT ? &J.f_count
                        : k == FK_M2  ? &J.f_m2
                        : (k == FK_SUMSQ_I64 || k == FK_SUMSQ_F64 || k == FK_SUMSQ_F32) ? &J.f_sumsq
                        : (k == FK_SUM_I64 || k == FK_SUM_F64 || k == FK_SUM_F32)       ? &J.f_sum
                        : (k == FK_MIN_S32 || k == FK_MIN_S64 || k == FK_MIN_F64 || k == FK_MIN_F32) ? &J.f_min
                                                                                   : &J.f_max;
      if (ok) {
        ok    = *slot < 0;
        *slot = f;
      }
    }
    if (!ok || (J.f_m2 >= 0 && (J.f_sum < 0 || hP.fields[J.f_m2].aux_sum != J.f_sum))) continue;
    auto ptr = [&](int32_t f) { return f >= 0 ? hP.fields[f].ptr : nullptr; };
    J.p_rows  = hP.slot_count;
    J.p_count = static_cast<uint32_t*>(ptr(J.f_count));
    J.p_sum   = ptr(J.f_sum);
    J.p_min   = ptr(J.f_min);
    J.p_max   = ptr(J.f_max);
    J.p_sumsq = ptr(J.f_sumsq);
    J.p_m2    = static_cast<double*>(ptr(J.f_m2));
    if (st == ST_F32) {  // float32 order codes with the sign bit flipped: a signed 32-bit domain
      J.min_ident = int64_t(int32_t(uint32_t(field_identity(FK_MIN_F32)) ^ 0x80000000u));
      J.max_ident = int64_t(int32_t(uint32_t(field_identity(FK_MAX_F32)) ^ 0x80000000u));
    } else {
      int32_t const kmin = st == ST_I32 ? FK_MIN_S32 : st == ST_I64 ? FK_MIN_S64 : FK_MIN_F64;
      int32_t const kmax = st == ST_I32 ? FK_MAX_S32 : st == ST_I64 ? FK_MAX_S64 : FK_MAX_F64;
      int32_t op, xf;
      scan_domain(kmin, op, xf);
      J.min_ident = int64_t(xf_fwd(xf, field_identity(kmin)));
      scan_domain(kmax, op, xf);
      J.max_ident = int64_t(xf_fwd(xf, field_identity(kmax)));
    }
    if (J.f_m2 >= 0 && m2_scratch != nullptr) {  // scratch of its own per column
      size_t const g  = size_t(G > 0 ? G : 1);
      uint8_t* base   = m2_scratch + m2_column_bytes(G) * size_t(m2_jobs++);
      J.m2_flag       = base;
      J.m2_list       = reinterpret_cast<uint32_t*>(base + ((g + 255) & ~size_t(255)));
      J.m2_counts     = reinterpret_cast<uint32_t*>(base + ((g + 255) & ~size_t(255)) + ((4 * g + 255) & ~size_t(255)));
    }
    jobs.push_back({st, J});
  }
  if (!jobs.empty() && hP.need_count_all) jobs.front().second.count_rows = 1;
  return jobs;
}

sorted_stats_cover sorted_stats_plan(gb_params const& hP)
{
  sorted_stats_cover cover;
  cover.field.assign(size_t(hP.num_fields), 0);
  for (auto const& [st, J] : stats_jobs(hP, nullptr, 0)) {
    for (int f = hP.val_field_begin[J.vcol]; f < hP.val_field_begin[J.vcol + 1]; f++) cover.field[size_t(f)] = 1;
    cover.rows |= J.count_rows != 0;
    cover.m2_columns += J.f_m2 >= 0 ? 1 : 0;
  }
  return cover;
}

void launch_sorted_stats(gb_params const* dP, gb_params const& hP, int64_t n, int64_t G, uint32_t const* gid,
                         int num_cus, uint8_t* m2_scratch, hipStream_t s)
{
  if (n <= 0) return;
  for (auto const& [st, J] : stats_jobs(hP, m2_scratch, G)) {
    if (J.f_m2 >= 0) hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, J.m2_counts, 2);
    if (st == ST_I32) launch_stats_job<ST_I32>(dP, J, n, gid, num_cus, s);
    else if (st == ST_I64) launch_stats_job<ST_I64>(dP, J, n, gid, num_cus, s);
    else if (st == ST_F32) launch_stats_job<ST_F32>(dP, J, n, gid, num_cus, s);
    else launch_stats_job<ST_F64>(dP, J, n, gid, num_cus, s);
  }
}

void launch_sorted_stats_m2(gb_params const* dP, gb_params const& hP, int64_t n, int64_t G, uint32_t const* gid,
                            int num_cus, uint8_t* m2_scratch, hipStream_t s)
{
  if (n <= 0) return;
  for (auto const& [st, J] : stats_jobs(hP, m2_scratch, G)) {
    if (J.f_m2 < 0) continue;
    if (st == ST_I32) launch_stats_m2<ST_I32>(dP, J, n, gid, num_cus, s);
    else if (st == ST_I64) launch_stats_m2<ST_I64>(dP, J, n, gid, num_cus, s);
    else if (st == ST_F32) launch_stats_m2<ST_F32>(dP, J, n, gid, num_cus, s);
    else launch_stats_m2<ST_F64>(dP, J, n, gid, num_cus, s);
  }
}

static void launch_sorted_passes(gb_params const* dP, gb_params const& hP, int64_t n, uint32_t const* gid,
                                 int num_cus, bool m2, sorted_stats_cover const* cover, hipStream_t s)
{
  std::vector<int32_t> items;
  if (!m2 && hP.need_count_all && !(cover && cover->rows)) items.push_back(-1);
  for (int f = 0; f < hP.num_fields; f++) {
    int32_t const k = hP.fields[f].kind;
    if (cover && cover->field[size_t(f)]) continue;  // launch_sorted_stats
    if (k == FK_NUNIQUE || k == FK_NUNIQUE_NULLS || k == FK_NTH) continue;  // kernels of their own
    if ((k == FK_ARGMIN || k == FK_ARGMAX) && hP.vals[hP.fields[f].vcol].storage == ST_STRING)
      continue;  // launch_sorted_string_arg
    if ((hP.fields[f].kind == FK_M2) == m2) items.push_back(f);
  }
  int64_t per, W;
  sorted_ranges(n, num_cus, per, W);
  unsigned const blocks = unsigned((W + BLOCK / 64 - 1) / (BLOCK / 64));
  size_t i = 0;
  while (i < items.size()) {
    sorted_pass pass{};
    while (i < items.size() && pass.n < SORTED_FPP) {
      int32_t const f = items[i];
      int32_t slot    = -1;
      if (f >= 0) {
        int32_t const vc = hP.fields[f].vcol;
        for (int c = 0; c < pass.ncols; c++)
          if (pass.col[c] == vc) slot = c;
        if (slot < 0) {
          if (pass.ncols == SORTED_COLS) break;  // next pass
          slot                  = pass.ncols;
          pass.col[pass.ncols++] = vc;
        }
      }
      int32_t const kind  = f < 0 ? int32_t(FK_COUNT) : hP.fields[f].kind;
      pass.field[pass.n]  = f;
      pass.col_of[pass.n] = slot;
      pass.kind[pass.n]   = kind;
      scan_domain(kind, pass.op[pass.n], pass.xf[pass.n]);
      pass.ident[pass.n]  = kind == FK_M2 ? 0ull : xf_fwd(pass.xf[pass.n], field_identity(kind));
      pass.n++;
      i++;
    }
    bool has_arg = false;
    for (int k = 0; k < pass.n; k++) has_arg |= pass.kind[k] == FK_ARGMIN || pass.kind[k] == FK_ARGMAX;
    if (has_arg) hipLaunchKernelGGL(k_sorted_reduce<true>, dim3(blocks), dim3(BLOCK), 0, s, dP, gid, per, W, pass);
    else hipLaunchKernelGGL(k_sorted_reduce<false>, dim3(blocks), dim3(BLOCK), 0, s, dP, gid, per, W, pass);
  }
}

// ARGMIN / ARGMAX of a string column on runs (and through them string MIN /
// MAX): each wave reduces its rows of every run to the run's best row with
// string comparisons (segmented over lanes of equal group numbers, which are
// contiguous), and the run's first lane folds that row into the group's
// accumulator with the compare-and-swap of the device-wide path.  Equal
// strings keep the smaller row, so the result does not depend on the order
// of the updates.
__global__ void __launch_bounds__(BLOCK)
  k_sorted_string_arg(gb_params const* __restrict__ Pp, int32_t f, int64_t n, uint32_t const* __restrict__ gid)
{
  constexpr uint32_t NONE = 0xFFFFFFFFu;
  gb_params const& P  = *Pp;
  field_desc const& F = P.fields[f];
  dcol const& c       = P.vals[F.vcol];
  int const lane      = threadIdx.x & 63;
  for (int64_t base = int64_t(blockIdx.x) * BLOCK + (threadIdx.x & ~63); base < n;
       base += int64_t(gridDim.x) * BLOCK) {
    int64_t const row = base + lane;
    uint32_t const g  = row < n ? gid[row] : NO_GROUP;
    uint32_t best     = (g != NO_GROUP && dcol_valid(c, row)) ? uint32_t(row) : NONE;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      uint32_t const other = uint32_t(__shfl_down(int(best), d));
      uint32_t const og    = uint32_t(__shfl_down(int(g), d));
      if (lane + d < 64 && og == g && other != NONE &&
          (best == NONE || arg_better(c, F.kind, int64_t(other), int64_t(best))))
        best = other;
    }
    uint32_t const gprev = uint32_t(__shfl_up(int(g), 1));
    bool const head      = lane == 0 || gprev != g;
    if (head && g != NO_GROUP && best != NONE) arg_update(F, int64_t(g), c, int64_t(best));
  }
}

void launch_sorted_string_arg(gb_params const* dP, gb_params const& hP, int64_t n, uint32_t const* gid,
                              hipStream_t s)
{
  if (n <= 0) return;
  unsigned const blocks = unsigned(std::min<int64_t>((n + BLOCK - 1) / BLOCK, int64_t(1) << 20));
  for (int f = 0; f < hP.num_fields; f++) {
    int32_t const k = hP.fields[f].kind;
    if ((k == FK_ARGMIN || k == FK_ARGMAX) && hP.vals[hP.fields[f].vcol].storage == ST_STRING)
      hipLaunchKernelGGL(k_sorted_string_arg, dim3(blocks), dim3(BLOCK), 0, s, dP, f, n, gid);
  }
}

// Group rows of the gathered (group-ordered) columns back to input rows:
// rows[g] = perm[rows[g]] where the row is set (-1 stays).
__global__ void __launch_bounds__(BLOCK)
  k_map_rows(int32_t* __restrict__ rows, int64_t G, uint32_t const* __restrict__ perm)
{
  int64_t const g = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (g < G && rows[g] >= 0) rows[g] = int32_t(perm[rows[g]]);
}

void launch_map_rows(int32_t* rows, int64_t G, uint32_t const* perm, hipStream_t s)
{
  if (G > 0) hipLaunchKernelGGL(k_map_rows, dim3(unsigned((G + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, s, rows, G, perm);
}

void launch_sorted_aggregate(gb_params const* dP, gb_params const& hP, int64_t n, uint32_t const* gid, int num_cus,
                             sorted_stats_cover const* cover, hipStream_t s)
{
  launch_sorted_passes(dP, hP, n, gid, num_cus, false, cover, s);
}

void launch_sorted_second_pass(gb_params const* dP, gb_params const& hP, int64_t n, uint32_t const* gid,
                               int num_cus, sorted_stats_cover const* cover, hipStream_t s)
{
  launch_sorted_passes(dP, hP, n, gid, num_cus, true, cover, s);
}

// NUNIQUE on runs.  The reference sorts each group's values and counts the
// heads of equal runs (sort/group_nunique.cu:44-64).  Here a group whose rows
// all lie in one 64-row chunk of a wave is counted inside the wave: a counted
// row is a new value when no earlier row of its group holds an equal one
// (shuffles over at most the group's length).  Every other counted row (longer
// or chunk-crossing groups, and strings) inserts (group, value) into an
// open-addressing set of row indices, and the row that claims an empty slot
// adds one distinct value to its group.  Rows
// are equal when they share the group and both are null (counted only with
// nulls included) or hold the same value, -0.0 equal to 0.0 and NaN equal to
// NaN (the row comparator's defaults).  Group g probes only its own region
// of the set, slots [2 * first, 2 * end) where [first, end) are the rows from
// its first row to the next group's: the region has at least twice as many
// slots as the group has rows, so every probe sequence reaches an empty slot
// or a match, and a group's probes stay within a few cache lines (the groups
// of sorted keys are contiguous rows).
__device__ __forceinline__ uint64_t nunique_bits(dcol const& c, int64_t row)
{
  uint64_t b = raw_bits(c, row);
  if (c.storage == ST_F32) {
    float const x = __uint_as_float(uint32_t(b));
    b             = isnan(x) ? 0x7fc00000ull : (x == 0.0f ? 0ull : b);
  } else if (c.storage == ST_F64) {
    double const x = __longlong_as_double(int64_t(b));
    b              = isnan(x) ? 0x7ff8000000000000ull : (x == 0.0 ? 0ull : b);
  } else if (c.storage == ST_BOOL) {
    b = b != 0;
  }
  return b;
}

__global__ void __launch_bounds__(BLOCK) k_fill_empty(uint32_t* __restrict__ out, int64_t n)
{
  for (int64_t i = int64_t(blockIdx.x) * BLOCK + threadIdx.x; i < n; i += int64_t(gridDim.x) * BLOCK)
    out[i] = 0xFFFFFFFFu;
}

__global__ void __launch_bounds__(BLOCK)
  k_sorted_nunique(gb_params const* __restrict__ Pp, int32_t f, int64_t n, int64_t G,
                   uint32_t const* __restrict__ gid, uint32_t* __restrict__ table)
{
  constexpr uint32_t EMPTY = 0xFFFFFFFFu;
  gb_params const& P   = *Pp;
  field_desc const& F  = P.fields[f];
  dcol const& c        = P.vals[F.vcol];
  bool const with_null = F.kind == FK_NUNIQUE_NULLS;
  bool const str       = c.storage == ST_STRING;  // strings: hashed, then compared byte-wise
  int const lane       = threadIdx.x & 63;
  // each wave takes 64 consecutive rows per step (the loop bound is uniform
  // across the wave, so every lane reaches the ballots below)
  for (int64_t base0 = int64_t(blockIdx.x) * BLOCK + (threadIdx.x & ~63); base0 < n;
       base0 += int64_t(gridDim.x) * BLOCK) {
    int64_t const row = base0 + lane;
    uint32_t const g  = row < n ? gid[row] : NO_GROUP;
    bool const valid  = g != NO_GROUP && dcol_valid(c, row);
    bool const counts = g != NO_GROUP && (valid || with_null);
    bool inserted     = false;
    uint64_t const b  = !valid ? 0ull : (str ? uint64_t(elem_hash(c, row, 0u)) : nunique_bits(c, row));
    uint64_t first = 0, end = 0;
    if (g != NO_GROUP) {
      first = P.slot_rows[g];
      end   = int64_t(g) + 1 < G ? P.slot_rows[g + 1] : uint64_t(n);
    }
    // A group whose rows all lie in this chunk is counted here: a counted
    // lane is a new value when no lower lane of its group holds an equal one
    // (the group's lanes are contiguous, from lane first - base0).
    bool const local    = counts && !str && first >= uint64_t(base0) && end <= uint64_t(base0 + 64);
    uint64_t const lmask = __ballot(local);
    if (lmask != 0) {
      uint64_t const cmask = __ballot(counts);
      uint64_t const vmask = __ballot(valid);
      int dist             = local ? lane - int(first - uint64_t(base0)) : 0;
      int maxd             = dist;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) maxd = max(maxd, __shfl_xor(maxd, off));
      bool dup = false;
      for (int d = 1; d <= maxd; d++) {
        uint64_t const ob = __shfl_up(b, d);
        int const o       = lane - d;  // the other lane, in the group when d <= dist
        if (d <= dist && ((cmask >> o) & 1u) && (((vmask >> o) & 1u) != 0) == valid && (!valid || ob == b))
          dup = true;
      }
      inserted = local && !dup;
    }
    if (counts && !local) {
      uint32_t const h     = mm_fmix32(uint32_t(b) ^ mm_fmix32(uint32_t(b >> 32) ^ uint32_t(valid)));
      uint64_t const hbase = 2 * first, len = 2 * (end - first);
      uint64_t off         = (uint64_t(h) * len) >> 32;  // in [0, len)
      for (;;) {
        uint64_t const slot = hbase + off;
        uint32_t cur = __hip_atomic_load(&table[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cur == EMPTY) {
          uint32_t const prev = atomicCAS(&table[slot], EMPTY, uint32_t(row));
          if (prev == EMPTY) {
            inserted = true;
            break;
          }
          cur = prev;
        }
        // the region holds rows of group g only
        bool const cv = dcol_valid(c, cur);
        if (cv == valid && (!valid || (str ? elem_equal(c, cur, row) : nunique_bits(c, cur) == b)))
          break;  // already counted
        off = off + 1 == len ? 0 : off + 1;
      }
    }
    // one add per run of equal groups in the wave (group numbers do not
    // decrease along the rows): the run's first lane adds the run's insertions
    uint32_t const gp_  = uint32_t(__shfl(int(g), lane == 0 ? 0 : lane - 1));
    bool const head     = lane == 0 || gp_ != g;
    uint64_t const heads = __ballot(head);
    uint64_t const ins   = __ballot(inserted);
    if (head && g != NO_GROUP) {
      uint64_t const later = lane == 63 ? 0ull : heads & ~((2ull << lane) - 1ull);  // heads above this lane
      uint64_t const upto  = later ? ((later & (~later + 1ull)) - 1ull) : ~0ull;     // lanes below the next head
      uint32_t const cnt   = uint32_t(__popcll(ins & upto & ~((1ull << lane) - 1ull)));
      if (cnt) atomicAdd(reinterpret_cast<unsigned int*>(field_at(F, g)), cnt);
    }
  }
}

// NTH_ELEMENT on runs (sort/group_nth_element.cu:50-140): the group's n-th
// row in row order (from the end for n < 0), counting every row under
// INCLUDE and rows with a valid value under EXCLUDE; none when the group has
// too few.  Group g holds rows first..last (slot_rows[g],
// group_last[g]) with no dropped row among them, so when every row counts
// (nulls included, or a value column without nulls) the n-th row is found by
// index arithmetic, one thread per group.
__global__ void __launch_bounds__(BLOCK)
  k_sorted_nth_direct(gb_params const* __restrict__ Pp, int32_t f, int64_t G, uint32_t const* __restrict__ group_last)
{
  int64_t const g = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (g >= G) return;
  gb_params const& P  = *Pp;
  field_desc const& F = P.fields[f];
  int64_t const nth   = F.aux_sum;
  int64_t const first = int64_t(P.slot_rows[g]);
  int64_t const last  = min(int64_t(group_last[g]), P.num_rows - 1);
  int64_t const size  = last - first + 1;
  uint32_t found      = 0xFFFFFFFFu;
  if (nth >= 0 ? nth < size : -nth <= size) found = uint32_t(nth >= 0 ? first + nth : last + 1 + nth);
  *reinterpret_cast<uint32_t*>(field_at(F, g)) = found;
}

// The r-th (0-based) set bit of `bits`, counted from the low end or, when
// `high`, from the high end; r < popcount(bits).
__device__ __forceinline__ int select_bit(uint32_t bits, int r, bool high)
{
  if (high) {
    for (int i = 0; i < r; i++) bits &= ~(0x80000000u >> __clz(bits));
    return 31 - __clz(bits);
  }
  for (int i = 0; i < r; i++) bits &= bits - 1u;
  return __ffs(bits) - 1;
}

// NTH_ELEMENT on runs with null values excluded.  The group's rows are bits
// b0..b1 of the value column's mask; the n-th valid row (from the front for
// n >= 0, from the back for n < 0) is found by counting set bits word by
// word.  Groups of at most NTH_THREAD_WORDS mask words are counted by one
// thread each; larger groups are listed (large[0] = count, large[1..] =
// groups) for k_sorted_nth_scan, where a wave counts 64 words per step.
constexpr int NTH_THREAD_WORDS = 8;

struct nth_bits {
  int64_t b0, b1, w0, w1;
};

__device__ __forceinline__ nth_bits nth_group_bits(gb_params const& P, dcol const& c, uint32_t const* group_last,
                                                   int64_t g)
{
  nth_bits r;
  r.b0 = int64_t(P.slot_rows[g]) + c.mask_offset;
  r.b1 = min(int64_t(group_last[g]), P.num_rows - 1) + c.mask_offset;
  r.w0 = r.b0 >> 5;
  r.w1 = r.b1 >> 5;
  return r;
}

// Mask word w restricted to the group's bits.
__device__ __forceinline__ uint32_t nth_word(gmem<uint32_t const>* mask, nth_bits const& q, int64_t w)
{
  uint32_t bits = mask[w];
  if (w == q.w0) bits &= ~0u << (q.b0 & 31);
  if (w == q.w1 && (q.b1 & 31) != 31) bits &= (2u << (q.b1 & 31)) - 1u;
  return bits;
}

__global__ void __launch_bounds__(BLOCK)
  k_sorted_nth_small(gb_params const* __restrict__ Pp, int32_t f, int64_t G, uint32_t const* __restrict__ group_last,
                     uint32_t* __restrict__ large)
{
  int64_t const g = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (g >= G) return;
  gb_params const& P  = *Pp;
  field_desc const& F = P.fields[f];
  dcol const& c       = P.vals[F.vcol];
  nth_bits const q    = nth_group_bits(P, c, group_last, g);
  if (q.w1 - q.w0 >= NTH_THREAD_WORDS) {
    uint32_t const i = atomicAdd(&large[0], 1u);
    large[1 + i]     = uint32_t(g);
    return;
  }
  auto const mask    = gp(c.mask);
  int64_t const nth  = F.aux_sum;
  bool const back    = nth < 0;
  int64_t const want = back ? -nth - 1 : nth;
  int64_t seen       = 0;
  uint32_t found     = 0xFFFFFFFFu;
  for (int64_t k = 0; k <= q.w1 - q.w0; k++) {
    int64_t const w     = back ? q.w1 - k : q.w0 + k;
    uint32_t const bits = nth_word(mask, q, w);
    int const cnt       = __popc(bits);
    if (seen + cnt > want) {
      found = uint32_t((w << 5) + select_bit(bits, int(want - seen), back) - c.mask_offset);
      break;
    }
    seen += cnt;
  }
  *reinterpret_cast<uint32_t*>(field_at(F, g)) = found;
}

__global__ void __launch_bounds__(BLOCK)
  k_sorted_nth_scan(gb_params const* __restrict__ Pp, int32_t f, uint32_t const* __restrict__ group_last,
                    uint32_t const* __restrict__ large)
{
  gb_params const& P  = *Pp;
  field_desc const& F = P.fields[f];
  dcol const& c       = P.vals[F.vcol];
  auto const mask     = gp(c.mask);
  int64_t const nth   = F.aux_sum;
  bool const back     = nth < 0;
  int64_t const want  = back ? -nth - 1 : nth;  // 0-based among the valid rows, from the chosen end
  int const lane      = threadIdx.x & 63;
  int64_t const waves = int64_t(gridDim.x) * (BLOCK / 64);
  int64_t const count = int64_t(large[0]);
  for (int64_t i = (int64_t(blockIdx.x) * BLOCK + threadIdx.x) >> 6; i < count; i += waves) {
    int64_t const g  = int64_t(large[1 + i]);
    nth_bits const q = nth_group_bits(P, c, group_last, g);
    int64_t seen     = 0;
    uint32_t found   = 0xFFFFFFFFu;
    for (int64_t k = 0; k <= q.w1 - q.w0; k += 64) {
      int64_t const w = back ? q.w1 - k - lane : q.w0 + k + lane;
      uint32_t bits   = 0;
      if (w >= q.w0 && w <= q.w1) bits = nth_word(mask, q, w);
      int const cnt = __popc(bits);
      int upto      = cnt;  // inclusive prefix over the lanes
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        int const t = __shfl_up(upto, d);
        if (lane >= d) upto += t;
      }
      int const total = __shfl(upto, 63);
      if (seen + total > want) {
        int64_t const r = want - seen;  // < total
        bool const mine = upto - cnt <= r && r < upto;
        uint32_t row    = 0;
        if (mine) row = uint32_t((w << 5) + select_bit(bits, int(r - (upto - cnt)), back) - c.mask_offset);
        int const src = __ffsll(static_cast<unsigned long long>(__ballot(mine))) - 1;
        found         = uint32_t(__shfl(int(row), src));
        break;
      }
      seen += total;
    }
    if (lane == 0) *reinterpret_cast<uint32_t*>(field_at(F, g)) = found;
  }
}

void launch_sorted_nth(gb_params const* dP, gb_params const& hP, int32_t f, int64_t G, uint32_t const* group_last,
                       uint32_t* large, hipStream_t s)
{
  if (G <= 0) return;
  field_desc const& F = hP.fields[f];
  unsigned const per_group = unsigned((G + BLOCK - 1) / BLOCK);
  if (F.aux_count != 0 || hP.vals[F.vcol].mask == nullptr) {
    hipLaunchKernelGGL(k_sorted_nth_direct, dim3(per_group), dim3(BLOCK), 0, s, dP, f, G, group_last);
    return;
  }
  MIG_HIP_TRY(hipMemsetAsync(large, 0, sizeof(uint32_t), s));
  hipLaunchKernelGGL(k_sorted_nth_small, dim3(per_group), dim3(BLOCK), 0, s, dP, f, G, group_last, large);
  int64_t const blocks = std::min<int64_t>((G + BLOCK / 64 - 1) / (BLOCK / 64), 4096);
  hipLaunchKernelGGL(k_sorted_nth_scan, dim3(unsigned(blocks)), dim3(BLOCK), 0, s, dP, f, group_last, large);
}

void launch_sorted_nunique(gb_params const* dP, int32_t f, int64_t n, int64_t G, uint32_t const* gid,
                           uint32_t* table, hipStream_t s)
{
  if (n <= 0 || G <= 0) return;
  auto const grid = [](int64_t m) { return dim3(unsigned(std::min<int64_t>((m + BLOCK - 1) / BLOCK, 1 << 20))); };
  hipLaunchKernelGGL(k_fill_empty, grid(2 * n), dim3(BLOCK), 0, s, table, 2 * n);
  hipLaunchKernelGGL(k_sorted_nunique, grid(n), dim3(BLOCK), 0, s, dP, f, n, G, gid, table);
}

// String MIN / MAX from the groups' ARGMIN / ARGMAX rows: lengths (0 for
// groups without a valid value) and validity words.
__global__ void __launch_bounds__(BLOCK)
  k_str_arg_sizes(dcol src, int32_t const* __restrict__ rows, int64_t G, int32_t* __restrict__ sizes,
                  uint32_t* __restrict__ mask)
{
  int64_t const g = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  bool valid      = false;
  if (g < G) {
    int32_t const r = rows[g];
    valid           = r != -1 && dcol_valid(src, r);  // NTH_ELEMENT's row may hold a null
    int64_t b = 0, e = 0;
    if (valid) str_span(src, r, b, e);
    sizes[g] = int32_t(e - b);
  }
  if (mask) store_valid_bits(mask, g, G, valid);
}

void launch_str_arg_sizes(dcol const& src, int32_t const* rows, int64_t G, int32_t* sizes, uint32_t* mask,
                          hipStream_t s)
{
  if (G > 0)
    hipLaunchKernelGGL(k_str_arg_sizes, dim3((G + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, src, rows, G, sizes, mask);
}

void launch_iota_u32(uint32_t* out, int64_t n, hipStream_t s)
{
  if (n > 0) hipLaunchKernelGGL(k_iota_u32, dim3((n + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, out, n);
}

}  // namespace mig
