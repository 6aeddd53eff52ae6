// Exchanges between the lanes of a 64-lane wave on the VALU (gfx950).
//
// __shfl_xor and __shfl_up are ds_bpermute: they go through the LDS pipe (one per CU, shared by
// its four SIMDs) and wait for its latency. The reductions and scans here use DPP moves within
// rows of 16 lanes and the row swaps v_permlane16_swap / v_permlane32_swap across them, which are
// ordinary vector instructions.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

namespace certex_amd::lanes {

constexpr int kQuadXor1    = 0xB1;   // quad_perm [1, 0, 3, 2]
constexpr int kQuadXor2    = 0x4E;   // quad_perm [2, 3, 0, 1]
constexpr int kQuadReverse = 0x1B;   // quad_perm [3, 2, 1, 0]
constexpr int kHalfMirror  = 0x141;  // lane i of each 8 reads 7 - i
constexpr int kRowRor      = 0x120;  // + n: row rotated right by n lanes
constexpr int kRowShr      = 0x110;  // + n: row shifted right by n lanes
constexpr int kRowBcast15  = 0x142;  // lane 15 of a row to the next row
constexpr int kRowBcast31  = 0x143;  // lane 31 to rows 2 and 3

/** v through a DPP move of its 32-bit words. */
template <int CTRL, typename V>
__device__ __forceinline__ V dpp(V v)
{
  static_assert(sizeof(V) % 4 == 0, "words of 32 bits");
  int w[sizeof(V) / 4];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (int i = 0; i < int(sizeof(V) / 4); ++i) {
    w[i] = __builtin_amdgcn_update_dpp(0, w[i], CTRL, 0xf, 0xf, true);
  }
  __builtin_memcpy(&v, w, sizeof(V));
  return v;
}

/** op(v, v of the lane 32 away), the lower lane's value first. */
template <typename V, typename F>
__device__ __forceinline__ V fold32(V v, F op)
{
  int w[sizeof(V) / 4], lo[sizeof(V) / 4], hi[sizeof(V) / 4];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (int i = 0; i < int(sizeof(V) / 4); ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(w[i], w[i], false, false);
    lo[i]        = int(r[0]);
    hi[i]        = int(r[1]);
  }
  V a, b;
  __builtin_memcpy(&a, lo, sizeof(V));
  __builtin_memcpy(&b, hi, sizeof(V));
  return op(a, b);
}

/** op(v, v of the lane 16 away), the lower lane's value first. */
template <typename V, typename F>
__device__ __forceinline__ V fold16(V v, F op)
{
  int w[sizeof(V) / 4], lo[sizeof(V) / 4], hi[sizeof(V) / 4];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (int i = 0; i < int(sizeof(V) / 4); ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(w[i], w[i], false, false);
    lo[i]        = int(r[0]);
    hi[i]        = int(r[1]);
  }
  V a, b;
  __builtin_memcpy(&a, lo, sizeof(V));
  __builtin_memcpy(&b, hi, sizeof(V));
  return op(a, b);
}

/**
 * The xor butterfly (distances L / 2, ..., 2, 1) of a commutative op over groups of L lanes:
 * every lane of a group gets the same result, op(v[i], v[i ^ d]) level by level, so that the bits
 * of a floating-point sum are those of a __shfl_xor butterfly. L = 16, 32 or 64: after the level
 * of distance 8 a row's values repeat every 8 lanes, so that the rotation by 4 reads lane i ^ 4,
 * and so on down. L = 8 and below: distances 1, 2, then the half-row mirror (the values of a quad
 * are equal by then), for ops whose order does not matter.
 */
template <int L, typename V, typename F>
__device__ __forceinline__ V butterfly(V v, F op)
{
  static_assert(L == 1 || L == 2 || L == 4 || L == 8 || L == 16 || L == 32 || L == 64, "lanes");
  if constexpr (L >= 16) {
    if constexpr (L == 64) { v = fold32(v, op); }
    if constexpr (L >= 32) { v = fold16(v, op); }
    v = op(v, dpp<kRowRor + 8>(v));
    v = op(v, dpp<kRowRor + 4>(v));
    v = op(v, dpp<kRowRor + 2>(v));
    v = op(v, dpp<kRowRor + 1>(v));
  } else {
    if constexpr (L >= 2) { v = op(v, dpp<kQuadXor1>(v)); }
    if constexpr (L >= 4) { v = op(v, dpp<kQuadXor2>(v)); }
    if constexpr (L >= 8) { v = op(v, dpp<kHalfMirror>(v)); }
  }
  return v;
}

/** v of lane i ^ D (D a power of two below 64). */
template <int D, typename V>
__device__ __forceinline__ V exchange(V v)
{
  if constexpr (D == 1) {
    return dpp<kQuadXor1>(v);
  } else if constexpr (D == 2) {
    return dpp<kQuadXor2>(v);
  } else if constexpr (D == 4) {
    return dpp<kQuadReverse>(dpp<kHalfMirror>(v));  // i ^ 7, then i ^ 3
  } else if constexpr (D == 8) {
    return dpp<kRowRor + 8>(v);
  } else {
    static_assert(D == 16 || D == 32, "distances within a wave");
    const bool upper = (threadIdx.x & D) != 0;
    const auto pick  = [&](V lo, V hi) { return upper ? lo : hi; };
    if constexpr (D == 16) { return fold16(v, pick); }
    return fold32(v, pick);
  }
}

/**
 * One level (distance D) of N butterfly sums at once, the sums split over the lanes: lanes whose
 * bit D is clear go on with the sums [0, N / 2), the others with [N / 2, N). The kept sums are the
 * butterfly's own, w[i] + w[i] of lane ^ D, at half of its exchanges and additions.
 */
template <int D, int N, typename V>
__device__ __forceinline__ void split_level(V* w)
{
  static_assert(N >= 2 && N % 2 == 0, "pairs of sums");
  if constexpr (D >= 16) {
    // the row swap is the split: (a, b) -> (a lower, b lower), (a upper, b upper)
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      int a[sizeof(V) / 4], b[sizeof(V) / 4];
      __builtin_memcpy(a, &w[i], sizeof(V));
      __builtin_memcpy(b, &w[i + N / 2], sizeof(V));
#pragma unroll
      for (int j = 0; j < int(sizeof(V) / 4); ++j) {
        if constexpr (D == 32) {
          const auto r = __builtin_amdgcn_permlane32_swap(a[j], b[j], false, false);
          a[j] = int(r[0]), b[j] = int(r[1]);
        } else {
          const auto r = __builtin_amdgcn_permlane16_swap(a[j], b[j], false, false);
          a[j] = int(r[0]), b[j] = int(r[1]);
        }
      }
      V x, y;
      __builtin_memcpy(&x, a, sizeof(V));
      __builtin_memcpy(&y, b, sizeof(V));
      w[i] = x + y;
    }
  } else {
    const bool upper = (threadIdx.x & D) != 0;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const V keep = upper ? w[i + N / 2] : w[i];
      const V send = upper ? w[i] : w[i + N / 2];
      w[i]         = keep + exchange<D>(send);
    }
  }
}

/**
 * N butterfly sums (N a power of two, at most L) over groups of L lanes, split over the lanes from
 * the widest distance down (split_level): sum i ends in w[0] of the lanes whose bits L / 2, L / 4,
 * ... spell i from its highest bit down (a sum is held by L / N lanes of the group).
 */
template <int L, int N, typename V>
__device__ __forceinline__ void split_sums(V* w)
{
  constexpr int D = L / 2;
  if constexpr (D >= 1) {
    if constexpr (N > 1) {
      split_level<D, N>(w);
      split_sums<D, N / 2>(w);
    } else {
      w[0] += exchange<D>(w[0]);
      split_sums<D, 1>(w);
    }
  }
}

template <int L, typename V>
__device__ __forceinline__ V sum(V v)
{
  return butterfly<L>(v, [](V a, V b) { return a + b; });
}
template <int L, typename V>
__device__ __forceinline__ V min(V v)
{
  return butterfly<L>(v, [](V a, V b) { return b < a ? b : a; });
}
template <int L, typename V>
__device__ __forceinline__ V max(V v)
{
  return butterfly<L>(v, [](V a, V b) { return a < b ? b : a; });
}

/** Inclusive prefix sum of v over the 64 lanes: shifts within the rows, then the row totals. */
__device__ __forceinline__ int scan_incl(int v)
{
  v += __builtin_amdgcn_update_dpp(0, v, kRowShr + 1, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kRowShr + 2, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kRowShr + 4, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kRowShr + 8, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kRowBcast15, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kRowBcast31, 0xc, 0xf, false);
  return v;
}

}  // namespace certex_amd::lanes
