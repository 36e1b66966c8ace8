// Pieces shared by the 2-D tiled q8_0 / q4_0 GEMMs (qgemm_wide.hip,
// qgemm_mx.hip): grids of 32 x 32 MFMA tiles per wave, operands streamed
// through an LDS ring with explicit waits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qc_lds_dma.h"

namespace qc {
namespace wide {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

// Exponent slot of an activation row holding NaN or +-inf.
constexpr int kRowNonfinite = 0x40000000;

__device__ __forceinline__ void wait_lgkmcnt0() {
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
}

// Barrier that neither drains outstanding global->LDS loads (the waits are
// explicit) nor lets the compiler move memory accesses across it.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

// A wave-uniform pointer, in scalar registers.
__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const uint8_t*>(static_cast<uint64_t>(hi) << 32 | lo);
}

// Tile (mb, nbk) and K range ks of workgroup blockIdx.x in an XCD-aware
// order: workgroup ids are dealt to the 8 XCDs in turn; each XCD takes a
// contiguous range of tiles, m fastest, so that it reads few weight panels.
// (Integer divisions run on the vector unit: back to scalar registers.)
__device__ __forceinline__ void tile_of_workgroup(int mblocks, int nblocks, int ks_count, int& mb,
                                                  int& nbk, int& ks) {
  const int tiles = mblocks * nblocks * ks_count;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int per = tiles >> 3, rem = tiles & 7;
  const int t = xcd * per + min(xcd, rem) + idx;
  const int tq = __builtin_amdgcn_readfirstlane(t / mblocks);
  ks = __builtin_amdgcn_readfirstlane(tq / nblocks);
  mb = t - tq * mblocks;
  nbk = tq - ks * nblocks;
}

// Stores a wave's accumulators: acc[tm][tn][e] of lane l is row m0 + 32 tm +
// 8 (e >> 2) + 4 (l >> 5) + (e & 3), column n0 + 32 tn + (l & 31), times
// 2^rexp[row], to out (rows ld floats apart), or added to it.  Rows marked
// kRowNonfinite take nonfinite(row, column) instead.  rexp is readable (and
// 16-byte aligned) for whole tiles.  Row pointers are scalar; waves whose rows
// and columns are all in range and finite -- nearly all -- store without
// checks.  (With per-lane 64-bit addresses and checks on every element the
// stores of a 256 x 256 tile took about 10 us, as long as ten K steps.)
template <int TM, int TN, class Nonfinite>
__device__ __forceinline__ void store_tiles(const f32x16 (&acc)[TM][TN], const int* rexp,
                                            float* out, long long ld, bool add, int m0, int n0,
                                            int M, int N, Nonfinite nonfinite) {
  const int lane = threadIdx.x & 63;
  const int col = lane & 31, half = lane >> 5;
  i32x4 rx[TM][4];
  bool special = false;
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      rx[tm][g] = *reinterpret_cast<const i32x4*>(rexp + m0 + 32 * tm + 8 * g + 4 * half);
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int e = 0; e < 16; ++e)
      special = special || (rx[tm][e >> 2][e & 3] == kRowNonfinite &&
                            m0 + 32 * tm + 8 * (e >> 2) + 4 * half + (e & 3) < M);
  special = __any(special);
  float* const base = out + m0 * ld + n0;
  const long long lo = 4 * half * ld + col;
  const bool whole = m0 + 32 * TM <= M && n0 + 32 * TN <= N && !special;
  bool ok[TN];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) ok[tn] = n0 + 32 * tn + col < N;
  auto all = [&](auto checked, auto put) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = rx[tm][e >> 2][e & 3];
        const int up = 32 * tm + 8 * (e >> 2) + (e & 3);
        float* const row = base + up * ld;
        const bool in = !decltype(checked)::value ||
                        (m0 + up + 4 * half < M && (r != kRowNonfinite));
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          if (!decltype(checked)::value || (in && ok[tn])) put(row + 32 * tn, ldexpf(acc[tm][tn][e], r));
      }
  };
  const auto store = [&](float* p, float v) { p[lo] = v; };
  const auto atomic = [&](float* p, float v) { atomicAdd(p + lo, v); };
  if (whole) {
    if (add) all(std::false_type(), atomic);
    else all(std::false_type(), store);
    return;
  }
  if (add) all(std::true_type(), atomic);
  else all(std::true_type(), store);
  if (!special) return;
#pragma unroll 1
  for (int q = 0; q < TM * TN * 16; ++q) {
    const int tn = q % TN, tm = q / TN / 16, e = q / TN % 16;
    const int n = n0 + 32 * tn + col;
    const int m = m0 + 32 * tm + 8 * (e >> 2) + 4 * half + (e & 3);
    if (n >= N || m >= M || rexp[m] != kRowNonfinite) continue;
    const float v = nonfinite(m, n);
    if (add) atomicAdd(out + m * ld + n, v);
    else out[m * ld + n] = v;
  }
}

// Host side: the tile and K split of a call by modelled time.
//
// A workgroup's K unit takes at least `alone_us` (its waves' own work and
// latency) and, with a full chip of `slots` workgroups per CU, `full_us` per
// round of all slots: the clock drops under MFMA power, so time then follows
// the total work and a partial round costs its share.
struct Tile {
  int bm, bn, slots;
  double alone_us, full_us;
};
struct TilePlan {
  int tile = 0, ks = 1, per = 1;   // K ranges of `per` units
  double us = 1e30;
};
// ranges: the K ranges wanted, 0 = any up to max_ks.  Two ranges add into a
// cleared y (2048 x 4096 outputs: about 45 us more than stores); more are
// summed from partial outputs, of at most max_partial bytes, by a second launch
// (4 bytes / ps).
inline TilePlan plan_tiles(const Tile* tiles, int count, int m, int n, int units, int cus,
                           int ranges, int max_ks, double max_partial = 256e6) {
  TilePlan best;
  const double bytes = 4.0 * m * n;
  for (int i = 0; i < count; ++i) {
    const Tile& c = tiles[i];
    const double wgs = static_cast<double>((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
    for (int want : {1, 2, 3, 4, 6, 8, 12, 16, 24}) {
      if (ranges > 0 ? want != std::min(ranges, units) : want > max_ks) continue;
      const int per = (units + want - 1) / want;
      const int ks = (units + per - 1) / per;
      if (ks != want || (ks > 2 && ks * bytes > max_partial)) continue;
      const double rounds = wgs * ks / (static_cast<double>(cus) * c.slots);
      const double us = std::max(std::ceil(rounds) * (per * c.alone_us + 2.0),
                                 rounds * per * c.full_us + 2.0) +
                        (ks == 2  ? 1.0 + bytes * 1.2e-6
                         : ks > 2 ? 2.5 + 2.0 * ks * bytes * 1e-6 / 4.0
                                  : 0.0);
      if (us < best.us) best = TilePlan{i, ks, per, us};
    }
  }
  return best;
}

}  // namespace wide
}  // namespace qc
