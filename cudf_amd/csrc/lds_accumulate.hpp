// LDS accumulation shared by the aggregating kernels: a chunk of N rows per
// thread is loaded column by column, and each accumulator is applied to all
// of the chunk's rows at once with LDS atomics.
#pragma once

#include "device_ops.hpp"

namespace mig {

constexpr int WG_SCOPE = __HIP_MEMORY_SCOPE_WORKGROUP;

// Element i of a per-lane plan (descriptors sit one per lane of a VGPR: a
// scalar load inside a row loop would wait for every LDS operation in flight,
// and a uniform index into a register array would go to memory).
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int i)
{
  return uint32_t(__builtin_amdgcn_readlane(int(v), i));
}
__device__ __forceinline__ uint64_t lane_value64(uint32_t lo, uint32_t hi, int i)
{
  return (uint64_t(lane_value(hi, i)) << 32) | lane_value(lo, i);
}

// Apply `f(k)` to the rows k of a chunk whose bit is set in `ok` (the loop is
// unrolled; the caller's switch on the accumulator kind stays outside it).
template <int N, typename F>
__device__ __forceinline__ void for_rows(uint32_t ok, F&& f)
{
#pragma unroll
  for (int k = 0; k < N; k++)
    if ((ok >> k) & 1u) f(k);
}

// Raw elements of a column for the rows r0 + k * BLK of a chunk, zero-extended
// to 64 bits (canon_rows gives the canonical form).  Rows at or past `e` read
// row e - 1; their lanes take no part.
template <int BLK, typename T, typename I, int N>
__device__ __forceinline__ void load_rows(gmem<T const>* p, I r0, I e, uint64_t (&c)[N])
{
#pragma unroll
  for (int k = 0; k < N; k++) {
    I const r = r0 + I(k) * I(BLK);
    c[k]      = uint64_t(p[r < e ? r : e - 1]);
  }
}

template <int BLK, typename I, int N>
__device__ __forceinline__ void load_chunk(gmem<uint8_t const>* src, int w, I r0, I e, uint64_t (&c)[N])
{
  switch (w) {
    case 1: load_rows<BLK>(src, r0, e, c); break;
    case 2: load_rows<BLK>(reinterpret_cast<gmem<uint16_t const>*>(src), r0, e, c); break;
    case 4: load_rows<BLK>(reinterpret_cast<gmem<uint32_t const>*>(src), r0, e, c); break;
    default: load_rows<BLK>(reinterpret_cast<gmem<uint64_t const>*>(src), r0, e, c); break;
  }
}

// Canonical form of a chunk's raw elements of storage `st`: integers sign-
// or zero-extended to 64 bits (bool as 0/1), float bits unchanged.
template <int N>
__device__ __forceinline__ void canon_rows(int32_t st, uint64_t (&c)[N])
{
  switch (st) {
    case ST_I8:
#pragma unroll
      for (int k = 0; k < N; k++) c[k] = uint64_t(int64_t(int8_t(c[k])));
      break;
    case ST_I16:
#pragma unroll
      for (int k = 0; k < N; k++) c[k] = uint64_t(int64_t(int16_t(c[k])));
      break;
    case ST_I32:
#pragma unroll
      for (int k = 0; k < N; k++) c[k] = uint64_t(int64_t(int32_t(c[k])));
      break;
    case ST_BOOL:
#pragma unroll
      for (int k = 0; k < N; k++) c[k] = c[k] != 0;
      break;
    default: break;
  }
}

// A canonical element as double.
__device__ __forceinline__ double canon_double(int32_t st, uint64_t c)
{
  if (st == ST_F64) return __longlong_as_double(int64_t(c));
  if (st == ST_F32) return double(__uint_as_float(uint32_t(c)));
  if (st == ST_U64) return double(c);
  return double(int64_t(c));
}

// Keeps a chunk's slots and values opaque to the optimiser: in a loop over the
// accumulators it would otherwise compute the addresses and conversions of
// every accumulator kind once before the loop, whichever kinds there are, and
// hold them all in registers.
template <int N>
__device__ __forceinline__ void opaque_rows(int (&slot)[N], uint64_t (&c)[N])
{
#pragma unroll
  for (int k = 0; k < N; k++) asm volatile("" : "+v"(slot[k]), "+v"(c[k]));
}

// One accumulator over the rows of a chunk: `c[k]` holds row k's value in
// canonical form (integers sign- or zero-extended to 64 bits, float bits
// unchanged), `slot[k]` its group slot, bit k of `ok` whether it counts.  With
// every bit of `ok` set at compile time there are no branches: a caller whose
// rows may not count points those at a slot of their lane's that nobody reads.
template <int N>
__device__ __forceinline__ void acc_rows_lds(int32_t kind, int32_t lds_off, int32_t st, uint8_t* lds,
                                             int const (&slot)[N], uint32_t ok,
                                             uint64_t const (&c)[N], bool wide_f32)
{
  uint8_t* const base = lds + lds_off;
  auto u64 = [&](int k) { return reinterpret_cast<uint64_t*>(base) + slot[k]; };
  auto u32 = [&](int k) { return reinterpret_cast<uint32_t*>(base) + slot[k]; };
  auto fl  = [&](int k) { return __uint_as_float(uint32_t(c[k])); };
  auto db  = [&](int k) { return __longlong_as_double(int64_t(c[k])); };
  constexpr int R = __ATOMIC_RELAXED;
  switch (kind) {
    case FK_SUM_I64: for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_add(u64(k), c[k], R, WG_SCOPE); }); break;
    case FK_SUM_F32:  // in float64 when wide (rounded to float32 at output)
      if (wide_f32)
        for_rows<N>(ok, [&](int k) {
          __hip_atomic_fetch_add(reinterpret_cast<double*>(u64(k)), double(fl(k)), R, WG_SCOPE);
        });
      else
        for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_add(reinterpret_cast<float*>(u32(k)), fl(k), R, WG_SCOPE); });
      break;
    case FK_SUM_F64:
      for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_add(reinterpret_cast<double*>(u64(k)), db(k), R, WG_SCOPE); });
      break;
    case FK_SUMSQ_I64:
      for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_add(u64(k), c[k] * c[k], R, WG_SCOPE); });
      break;
    case FK_SUMSQ_F32:
      if (wide_f32)
        for_rows<N>(ok, [&](int k) {
          double const x = double(fl(k));
          __hip_atomic_fetch_add(reinterpret_cast<double*>(u64(k)), x * x, R, WG_SCOPE);
        });
      else
        for_rows<N>(ok, [&](int k) {
          __hip_atomic_fetch_add(reinterpret_cast<float*>(u32(k)), fl(k) * fl(k), R, WG_SCOPE);
        });
      break;
    case FK_SUMSQ_F64:
      for_rows<N>(ok, [&](int k) {
        __hip_atomic_fetch_add(reinterpret_cast<double*>(u64(k)), db(k) * db(k), R, WG_SCOPE);
      });
      break;
    case FK_MIN_S32:
      for_rows<N>(ok, [&](int k) {
        __hip_atomic_fetch_min(reinterpret_cast<int32_t*>(u32(k)), int32_t(c[k]), R, WG_SCOPE);
      });
      break;
    case FK_MAX_S32:
      for_rows<N>(ok, [&](int k) {
        __hip_atomic_fetch_max(reinterpret_cast<int32_t*>(u32(k)), int32_t(c[k]), R, WG_SCOPE);
      });
      break;
    case FK_MIN_S64:
      for_rows<N>(ok, [&](int k) {
        __hip_atomic_fetch_min(reinterpret_cast<int64_t*>(u64(k)), int64_t(c[k]), R, WG_SCOPE);
      });
      break;
    case FK_MAX_S64:
      for_rows<N>(ok, [&](int k) {
        __hip_atomic_fetch_max(reinterpret_cast<int64_t*>(u64(k)), int64_t(c[k]), R, WG_SCOPE);
      });
      break;
    case FK_MIN_U32: for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_min(u32(k), uint32_t(c[k]), R, WG_SCOPE); }); break;
    case FK_MAX_U32: for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_max(u32(k), uint32_t(c[k]), R, WG_SCOPE); }); break;
    case FK_MIN_U64: for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_min(u64(k), c[k], R, WG_SCOPE); }); break;
    case FK_MAX_U64: for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_max(u64(k), c[k], R, WG_SCOPE); }); break;
    case FK_MIN_F32:
      for_rows<N>(ok, [&](int k) {
        uint32_t const id = uint32_t(field_identity(FK_MIN_F32));
        __hip_atomic_fetch_min(u32(k), isnan(fl(k)) ? id : ord32(uint32_t(c[k])), R, WG_SCOPE);
      });
      break;
    case FK_MAX_F32:
      for_rows<N>(ok, [&](int k) {
        uint32_t const id = uint32_t(field_identity(FK_MAX_F32));
        __hip_atomic_fetch_max(u32(k), isnan(fl(k)) ? id : ord32(uint32_t(c[k])), R, WG_SCOPE);
      });
      break;
    case FK_MIN_F64:
      for_rows<N>(ok, [&](int k) {
        uint64_t const id = field_identity(FK_MIN_F64);
        __hip_atomic_fetch_min(u64(k), isnan(db(k)) ? id : ord64(c[k]), R, WG_SCOPE);
      });
      break;
    case FK_MAX_F64:
      for_rows<N>(ok, [&](int k) {
        uint64_t const id = field_identity(FK_MAX_F64);
        __hip_atomic_fetch_max(u64(k), isnan(db(k)) ? id : ord64(c[k]), R, WG_SCOPE);
      });
      break;
    case FK_COUNT: for_rows<N>(ok, [&](int k) { __hip_atomic_fetch_add(u32(k), 1u, R, WG_SCOPE); }); break;
    case FK_M2:  // pass A: sum of squares in double (finalised into M2 after the pass)
      for_rows<N>(ok, [&](int k) {
        double const x = canon_double(st, c[k]);
        __hip_atomic_fetch_add(reinterpret_cast<double*>(u64(k)), x * x, R, WG_SCOPE);
      });
      break;
    default: break;
  }
}

}  // namespace mig
