// Canonical int8 projections of more than a few activation rows on f16 MFMA
// (qc_cint8.h has the limits and the entry): y = x . dequant(W)^T over int8
// codes with row or group scales and optional zero points, the epilogue fused
// (kernels/quantization/qgemm_canonical.cpp:125-176,2550-2581).
//
// Numerics.  Activation rows are scaled by a power of two so that their
// largest element lies in [2^14, 2^15).  f16 and bf16 activations are then f16
// values (exactly, down to 2^-28 of the row's largest), f32 ones a pair hi + lo
// of them within 2^-22 of each element plus 2^-25.  Codes minus the integer of [-1152, 896]
// next to their zero point (at most 1280 in magnitude) are exact in f16,
// products and sums are f32.  What of the zero point that leaves (up to 0.5 of a
// fractional one) times the sum of x is subtracted in f32, so nothing is summed
// that is larger than the codes' distances from their zero point.  An f32 row
// holding 16-bit values has lo = 0 throughout and gives the bits of the 16-bit
// call.
//
// What bounds it: with few workgroups the chain of a step (one barrier, the
// LDS reads' latency, eight MFMAs: about 0.4 us per 64 columns); with a full
// chip VALU issue (the codes' conversion, five VALU per four codes of a lane,
// shared by the wave's m-tiles, and with groups the fold, one FMA per output and
// 64 columns) and the operands' way into LDS.  K = 4096, groups of 32, N =
// 14336, M = 512: 586 us on the row planes -> 151; groups of 128 257 -> 120; row
// scales N = 4096 63 -> 41 (16-bit activations).  Fractional zero points: groups
// of 128, M = 512 257 on the planes, 200 with MFMAs over all of x against ones,
// 146 with the sums that the prep writes.  Small tiles with rings of 6-8
// stages while the larger leave CUs idle; 128 x 256 above that.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "qc_cint8.h"
#include "qc_device.h"
#include "qc_internal.h"
#include "qc_lds_dma.h"
#include "qc_wide.h"

namespace qc {
namespace {

using namespace wide;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Activation fragments of one 32-row m-tile and 64-column step: slots of
// [64 lanes][16 B], lane l holding row l & 31.  Slot 2 b + s (P = 1) holds
// elements 32 b + 16 (l >> 5) + 8 s + i; with P = 2 slots 2 (2 b + s) and
// + 1 hold their hi and lo.
constexpr int kSlotBytes = 1024;

// Eight activation rows per workgroup, K in gridDim.y slices of whole steps:
// the rows' scales (over whole rows, in every slice), then the fragments, and
// (sums = 1, 2) each row's scaled sum over every 64 or 32 columns, as
// xs[32-row m-tile][K / 64 * sums][32].
// Each 128-byte line is eight rows' 16-byte pieces, stored at once.
template <int P>
__global__ __launch_bounds__(512) void f16_prep(const void* __restrict__ x, int xtype,
                                                long long ldx, bool vec, int M, int K,
                                                int steps_per_slice, uint8_t* __restrict__ xf,
                                                int* __restrict__ rexp, float* __restrict__ xs,
                                                int sums) {
  __shared__ int sexp[8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = 8 * blockIdx.x;
  const int steps = K / 64;
  auto load8 = [&](long long at, float (&v)[8]) {
    if (!vec) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = load_x(x, at + i, xtype);
    } else if constexpr (P == 2) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(static_cast<const float*>(x) + at);
      const f32x4 b = *reinterpret_cast<const f32x4*>(static_cast<const float*>(x) + at + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = a[i];
        v[4 + i] = b[i];
      }
    } else {
      const u32x4 a = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(x) + at);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t b = (a[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
        v[i] = xtype == QC_STORAGE_F16 ? half_bits_to_float(b) : __uint_as_float(b << 16);
      }
    }
  };
  if (m0 + wave < M) {                             // wave w: the maximum of row m0 + w
    const long long xr = static_cast<long long>(m0 + wave) * ldx;
    float mx = 0.f, z = 0.f;
    for (int c = 8 * lane; c < K; c += 512) {
      float v[8];
      load8(xr + c, v);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        mx = fmaxf(mx, fabsf(v[i]));
        z = fmaf(0.0f, v[i], z);                   // NaN once an element is not finite
      }
    }
    mx = wave_max_nonneg(mx);
    const bool bad = __any(z != 0.0f);
    int e = 0;
    if (mx > 0.f && mx <= 3.402823466e38f) (void)frexpf(mx, &e);
    e -= 15;
    if (lane == 0) {
      sexp[wave] = bad ? 0 : e;
      if (blockIdx.y == 0) rexp[m0 + wave] = bad ? kRowNonfinite : e;
    }
  }
  __syncthreads();
  // lane: row m0 + (lane & 7), block (lane >> 4) & 1, half lane >> 5, operand
  // s = (lane >> 3) & 1 of one step
  const int row = lane & 7, s = (lane >> 3) & 1, b = (lane >> 4) & 1, half = lane >> 5;
  const int m = m0 + row;
  if (m >= M) return;
  const int e = -sexp[row];
  const long long src = static_cast<long long>(m) * ldx + 32 * b + 16 * half + 8 * s;
  uint8_t* dst = xf + static_cast<long long>(m >> 5) * steps * (4 * P * kSlotBytes) +
                 16 * ((m & 31) + 32 * half) + P * (2 * b + s) * kSlotBytes;
  const int t0 = blockIdx.y * steps_per_slice, t1 = min(t0 + steps_per_slice, steps);
  for (int t = t0 + wave; t < t1; t += 8) {
    float v[8];
    load8(src + 64LL * t, v);
    f16x8 hi, lo;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float w = ldexpf(v[i], e);
      sum += w;
      hi[i] = static_cast<_Float16>(w);
      if constexpr (P == 2) lo[i] = static_cast<_Float16>(w - static_cast<float>(hi[i]));
    }
    uint8_t* d = dst + static_cast<long long>(t) * (4 * P * kSlotBytes);
    *reinterpret_cast<f16x8*>(d) = hi;
    if constexpr (P == 2) *reinterpret_cast<f16x8*>(d + kSlotBytes) = lo;
    if (sums > 0) {
      sum += dpp_f32<0x128>(sum);                  // lane ^ 8 (a rotation of 16 lanes)
      const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum),
                                                      false, false);
      sum = __uint_as_float(h[0]) + __uint_as_float(h[1]);
      if (sums == 1) {
        const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum),
                                                        false, false);
        sum = __uint_as_float(q[0]) + __uint_as_float(q[1]);
      }
      if (lane < 16 * sums && s == 0)
        xs[(static_cast<long long>(m >> 5) * steps * sums + t * sums + (sums == 2 ? b : 0)) * 32 +
           (m & 31)] = sum;
    }
  }
}

struct F16Out {
  const int8_t* w[2];          // SwiGLU: gate, up
  const float* scale[2];
  const float* zero[2];
  void* y;
  long long ld;
  int ytype, rows;
  const float* bias;
  int act, epi;
  int groups, gsize;
};

// a pointer out of two without an indexed (private memory) array
template <class T>
__device__ __forceinline__ T* pick(T* a, T* b, bool second) {
  const uint64_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return reinterpret_cast<T*>(x ^ ((x ^ y) & (0 - static_cast<uint64_t>(second))));
}

// The part of a zero point that codes can be reduced by exactly in f16.
__device__ __forceinline__ float code_zero(float z) {
  return __builtin_amdgcn_fmed3f(rintf(z), -1152.0f, 896.0f);
}

// The projection of activation row xr (elements) on weight row n in the
// reference's f32 form: for rows of x that hold NaN or +-inf.
__device__ __noinline__ float f16_row_f32(const int8_t* w, const float* scale, const float* zp,
                                          long long n, int groups, int gsize, const void* x,
                                          int xtype, long long xr, int k) {
  float acc = 0.0f;
  for (int b = 0; b < k; b += 32) {
    const long long si = n * groups + b / gsize;
    const float z = zp != nullptr ? zp[si] : 0.0f;
    acc += scale[si] * cint8_block_f32(w + n * k + b, x, xr + b, xtype, z);
  }
  return acc;
}

// Tile of TM x TN 32 x 32 MFMA tiles per wave, WGM x WGN waves, S stages.
// GPS: scale groups per 64-column step (0: one scale per row, 1: groups of 64
// or more, 2: groups of 32).
template <int P, int TM, int TN, int WGM, int WGN, int S, int GPS>
struct F16Tile {
  static constexpr int NW = WGM * WGN;
  static constexpr int BM = 32 * TM * WGM, BN = 32 * TN * WGN;   // x rows, weight rows
  static constexpr int XS = BM / 32 * 4 * P * kSlotBytes;     // x bytes per step
  static constexpr int XL = XS / 1024 / NW;                   // x loads per wave per step
  static constexpr int WC = BN / 16 / NW;                     // code loads (16 rows x 64 B)
  static constexpr int SW = GPS == 0 ? 0 : (BN / 32 * GPS + NW - 1) / NW;   // scale / zero gathers
  static constexpr int G = XL + WC + SW;
  static constexpr int SD = GPS * BN * 8;                     // scale and zero bytes
  static constexpr int stage = XS + BN * 64 + SD;
  static constexpr int lds = S * stage;
  static_assert(XS % (1024 * NW) == 0 && BN % (16 * NW) == 0, "whole loads");
  static_assert(lds <= 160 * 1024 && S >= 3 && (S - 2) * G < 64, "ring");
};

template <int P, int TM, int TN, int WGM, int WGN, int S, int GPS, bool SWIGLU>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void f16_gemm(
    const uint8_t* __restrict__ xf, const F16Out o, const int* __restrict__ rexp,
    const float* __restrict__ xs, const void* __restrict__ x, int xtype, long long ldx, int M, int K, int mblocks,
    int nblocks) {
  using C = F16Tile<P, TM, TN, WGM, WGN, S, GPS>;
  static_assert(!SWIGLU || TN == 2, "gate and up tiles side by side");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[C::lds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WGM, wn = wave / WGM;
  const int col = lane & 31, half = lane >> 5;
  int mb, nbk, ks;
  tile_of_workgroup(mblocks, nblocks, 1, mb, nbk, ks);
  const int mt0 = mb * (C::BM / 32);
  const int n0 = nbk * (SWIGLU ? C::BN / 2 : C::BN);          // first output column
  const int steps = K / 64;
  const bool zeros = o.zero[0] != nullptr;

  // Weight row r of the tile: SwiGLU alternates 32 gate and 32 up rows.
  auto row_of = [&](int r, bool& second) {
    second = SWIGLU && ((r >> 5) & 1);
    const int n = SWIGLU ? n0 + 32 * (r >> 6) + (r & 31) : n0 + r;
    return min(n, o.rows - 1);
  };
  auto key = [](int r) { return (r >> 2) & 3; };
  // x: 1 KB chunk q = wave * XL + i of a step (m-tile q / (4 P), slot q % (4 P))
  constexpr int XT = 4 * P;
  static_assert(C::XL <= XT ? XT % C::XL == 0 : C::XL % XT == 0, "x loads");
  const long long xtile = static_cast<long long>(steps) * XT * kSlotBytes;
  const uint8_t* xsrc = uniform_ptr(xf + (mt0 + wave * C::XL / XT) * xtile +
                                    (wave * C::XL % XT) * kSlotBytes);
  // codes: load i covers rows 16 (wave WC + i) .. + 15, four lanes a row, chunk
  // c stored at c ^ key(row); 16 rows share a matrix
  const uint8_t* wsrc[C::WC];
  uint32_t woff[C::WC];
#pragma unroll
  for (int i = 0; i < C::WC; ++i) {
    const int r0 = 16 * (wave * C::WC + i), r = r0 + lane / 4;
    bool second;
    const int n = row_of(r, second), nf = row_of(r0, second);
    wsrc[i] = uniform_ptr(reinterpret_cast<const uint8_t*>(pick(o.w[0], o.w[1], second)) +
                          static_cast<long long>(nf) * K);
    woff[i] = static_cast<uint32_t>(n - nf) * static_cast<uint32_t>(K) + 16 * ((lane % 4) ^ key(r));
  }
  // scales and zero points: gather j covers 32 rows of group half j / (BN / 32)
  // of the step, {scale, zero} per row (the scale twice without zero points)
  const float* ssrc[C::SW > 0 ? C::SW : 1];
  int sgrp[C::SW > 0 ? C::SW : 1];
  auto sq = [&](int i) {
    return __builtin_amdgcn_readfirstlane(min(wave * C::SW + i, C::BN / 32 * (GPS > 0 ? GPS : 1) - 1));
  };
  if constexpr (GPS > 0) {
#pragma unroll
    for (int i = 0; i < C::SW; ++i) {
      const int j = sq(i);
      bool second;
      const int n = row_of(32 * (j % (C::BN / 32)) + (lane >> 1), second);
      const float* sc = pick(o.scale[0], o.scale[1], second);
      const float* zp = zeros ? pick(o.zero[0], o.zero[1], second) : sc;
      ssrc[i] = pick(sc, zp, lane & 1) + static_cast<long long>(n) * o.groups;
      sgrp[i] = j / (C::BN / 32);
    }
  }
  // x of step t + S - 1 and the weights of step t + S go out at step t
  int xstep = 0, wstep = 0;                        // next steps to issue
  auto issue_x = [&](int slot) {
#pragma unroll
    for (int i = 0; i < C::XL; ++i)
      dma16(xsrc + (i / XT) * xtile + (i % XT) * kSlotBytes, 16 * lane,
            lds + slot * C::stage + (wave * C::XL + i) * 1024);
    xsrc += xstep + 1 < steps ? XT * kSlotBytes : 0;
    ++xstep;
  };
  auto issue_w = [&](int slot) {
    uint8_t* base = lds + slot * C::stage + C::XS;
#pragma unroll
    for (int i = 0; i < C::WC; ++i) {
      dma16(wsrc[i], woff[i], base + 1024 * (wave * C::WC + i));
      wsrc[i] += wstep + 1 < steps ? 64 : 0;
    }
    if constexpr (GPS > 0) {
      const int st = min(wstep, steps - 1);
#pragma unroll
      for (int i = 0; i < C::SW; ++i) {
        const int g = GPS == 2 ? 2 * st + sgrp[i] : 64 * st / o.gsize;
        dma4_addr(ssrc[i] + g, base + C::BN * 64 + 256 * sq(i));
      }
    }
    ++wstep;
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  // One step's weight operands: f16 codes less their zero points' code_zero
  // (`rest` notes any that leave something), and each group's scale.
  constexpr int NG = GPS > 0 ? GPS : 1;
  struct Weights {
    f16x8 w[TN][4];
    float s[TN][NG];
  };
  float rz[TN];                                    // row zero points (GPS = 0)
  bool rest = false;
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) {
    rz[tn] = 0.f;
    if (GPS == 0 && zeros) {
      bool second;
      const int n = row_of((wn * TN + tn) * 32 + col, second);
      const float z = pick(o.zero[0], o.zero[1], second)[n];
      rz[tn] = code_zero(z);
      rest = rest || rz[tn] != z;
    }
  }
  struct Raw {
    u32x4 q[TN][2];
    float2 sz[TN][NG];
  };
  auto read_w = [&](int slot, Raw& r) {
    const uint8_t* base = lds + slot * C::stage + C::XS;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int at = (wn * TN + tn) * 32 + col;
#pragma unroll
      for (int b = 0; b < 2; ++b)
        r.q[tn][b] = *reinterpret_cast<const u32x4*>(base + 64 * at + 16 * ((2 * b + half) ^ key(at)));
      if constexpr (GPS > 0) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
          r.sz[tn][g] = *reinterpret_cast<const float2*>(base + C::BN * 64 + 8 * (g * C::BN + at));
      }
    }
  };
  auto decode = [&](const Raw& r, Weights& o2) {
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      float z[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if constexpr (GPS > 0) {
          o2.s[tn][g] = r.sz[tn][g].x;
          z[g] = zeros ? code_zero(r.sz[tn][g].y) : 0.f;
          rest = rest || (zeros && z[g] != r.sz[tn][g].y);
        } else {
          z[g] = rz[tn];
        }
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        // byte u = q + 128 under the high byte 0x64 of f16(1024) is
        // f16(1024 + u); less 1152 + z that is q - z
        const _Float16 off = static_cast<_Float16>(1152.0f + z[GPS == 2 ? b : 0]);
        const f16x2 k2 = f16x2{off, off};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t c = r.q[tn][b][i] ^ 0x80808080u;
          const f16x2 a = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c, 0x04010400u)) - k2;
          const f16x2 d = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c, 0x04030402u)) - k2;
          f16x8& v = o2.w[tn][2 * b + (i >> 1)];
          const int e = 4 * (i & 1);
          v[e] = a[0];
          v[e + 1] = a[1];
          v[e + 2] = d[0];
          v[e + 3] = d[1];
        }
      }
    }
  };

  issue_w(0);
#pragma unroll
  for (int r = 0; r < S - 1; ++r) {
    issue_x(r);
    issue_w(r + 1);
  }
  wait_vmcnt<(S - 1) * C::G - C::XL>();            // W(0)
  ring_barrier();
  Weights w0, w1;
  Raw raw;
  read_w(0, raw);
  decode(raw, w0);
  int cur = 0;
  auto step = [&](const Weights& w, Weights& nw) {
    const int nxt = cur + 1 < S ? cur + 1 : 0, prv = cur > 0 ? cur - 1 : S - 1;
    wait_vmcnt<(S - 2) * C::G>();                  // x of this step, weights of the next
    wait_lgkmcnt0();
    ring_barrier();
    // every LDS read of the step first: their latency is paid once
    const uint8_t* xb = lds + cur * C::stage + wm * TM * XT * kSlotBytes + 16 * lane;
    f16x8 av[TM][XT];
#pragma unroll
    for (int q = 0; q < XT; ++q) av[0][q] = *reinterpret_cast<const f16x8*>(xb + q * kSlotBytes);
    read_w(nxt, raw);
#pragma unroll
    for (int tm = 1; tm < TM; ++tm)
#pragma unroll
      for (int q = 0; q < XT; ++q)
        av[tm][q] = *reinterpret_cast<const f16x8*>(xb + (tm * XT + q) * kSlotBytes);
    issue_x(prv);
    issue_w(cur);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const f16x8(&a)[XT] = av[tm];
      const auto products = [&](int b0, int b1, const f16x8 (&v)[4], f32x16 c) {
#pragma unroll
        for (int q = P * b0; q < P * b1; ++q)
          c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[q], v[q / P], c, 0, 0, 0);
        return c;
      };
      if constexpr (GPS == 0) {
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = products(0, 4, w.w[tn], acc[tm][tn]);
      } else {
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) {
            const f32x16 c = products(4 / NG * g, 4 / NG * (g + 1), w.w[tn], f32x16{});
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[tm][tn][e] = fmaf(c[e], w.s[tn][g], acc[tm][tn][e]);
          }
      }
      if (tm == 0) decode(raw, nw);
    }
    cur = nxt;
  };
  for (int t = 0; t < steps; t += 2) {
    step(w0, w1);
    if (t + 1 < steps) step(w1, w0);
  }
  wait_vmcnt<0>();   // no global->LDS load may outlive the workgroup's LDS

  // What the codes left of the zero points: the product of the rows' sums of x
  // over a group (row scales: a step) with it and the scale, two of them an f32
  // MFMA.
  if (__any(rest)) {
    const int per = GPS == 1 ? o.gsize / 64 : 1;   // sums to a group
    const int cols = GPS == 1 ? o.groups : NG * steps;
    constexpr int U = 4;                           // MFMAs whose operands load together
    for (int c0 = 0; c0 < cols; c0 += 2 * U) {
      float f[U][TN], a[U][TM];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = min(c0 + 2 * u + half, cols - 1);
        const bool in = c0 + 2 * u + half < cols;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          bool second;
          const long long n = row_of((wn * TN + tn) * 32 + col, second);
          const long long si = n * o.groups + (GPS == 0 ? 0 : c);
          const float z = pick(o.zero[0], o.zero[1], second)[si];
          const float sc = GPS == 0 ? 1.0f : pick(o.scale[0], o.scale[1], second)[si];
          f[u][tn] = in ? (code_zero(z) - z) * sc : 0.f;
        }
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) a[u][tm] = 0.f;
      }
      for (int j = 0; j < per; ++j)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int tm = 0; tm < TM; ++tm) {
            const long long c = static_cast<long long>(mt0 + wm * TM + tm) * cols + c0 + 2 * u + half;
            const float v = xs[(min(c, (mt0 + wm * TM + tm + 1LL) * cols - 1) * per + j) * 32 + col];
            a[u][tm] += c0 + 2 * u + half < cols ? v : 0.f;
          }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn)
            acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][tm], f[u][tn], acc[tm][tn], 0, 0, 0);
    }
  }

  // acc[tm][tn][e]: row 32 (mt0 + wm TM + tm) + 8 (e >> 2) + 4 half + (e & 3)
  const int mrow = 32 * (mt0 + wm * TM) + 4 * half;
  constexpr int JS = SWIGLU ? 2 : 1;
#pragma unroll
  for (int tn = 0; tn < TN; tn += JS) {
    const int n = SWIGLU ? n0 + 32 * wn + col : n0 + 32 * (wn * TN + tn) + col;
    if (n >= o.rows) continue;
    float sc[JS];
#pragma unroll
    for (int j = 0; j < JS; ++j) sc[j] = GPS == 0 ? (j == 0 ? o.scale[0] : o.scale[1])[n] : 1.0f;
    const float bias = o.epi && o.bias != nullptr ? o.bias[n] : 0.0f;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const i32x4 rx = *reinterpret_cast<const i32x4*>(rexp + mrow + 32 * tm + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = mrow + 32 * tm + 8 * g + i;
          if (m >= M) continue;
          auto value = [&](int j) {
            if (rx[i] == kRowNonfinite)
              return f16_row_f32(j == 0 ? o.w[0] : o.w[1], j == 0 ? o.scale[0] : o.scale[1],
                                 j == 0 ? o.zero[0] : o.zero[1], n, o.groups, o.gsize, x, xtype,
                                 m * ldx, K);
            const float v = acc[tm][tn + j][4 * g + i];
            return ldexpf(GPS == 0 ? v * sc[j] : v, rx[i]);
          };
          float v = value(0);
          if constexpr (SWIGLU) {
            v = (v / (1.0f + expf(-v))) * value(1);
          } else if (o.epi) {
            if (o.bias != nullptr) v += bias;
            v = linear_activation(v, o.act);
          }
          store_y(o.y, m * o.ld + n, o.ytype, v);
        }
      }
  }
}

template <int P, int TM, int TN, int WGM, int WGN, int S, int GPS, bool SWIGLU>
hipError_t launch_tile(const uint8_t* xf, const F16Out& o, const int* rexp, const float* xs,
                       const void* x, int xtype, long long ldx, int m, int k, hipStream_t s) {
  using C = F16Tile<P, TM, TN, WGM, WGN, S, GPS>;
  const int mblocks = (m + C::BM - 1) / C::BM;
  const int bn = SWIGLU ? C::BN / 2 : C::BN;
  const int nblocks = (o.rows + bn - 1) / bn;
  f16_gemm<P, TM, TN, WGM, WGN, S, GPS, SWIGLU>
      <<<static_cast<unsigned>(mblocks) * nblocks, 64 * C::NW, 0, s>>>(xf, o, rexp, xs, x, xtype, ldx,
                                                                      m, k, mblocks, nblocks);
  return hipGetLastError();
}

// Tile by workgroups: the small one while the larger would leave CUs idle.
template <int P, int GPS, bool SWIGLU>
hipError_t launch_f16(const uint8_t* xf, const F16Out& o, const int* rexp, const float* xs,
                      const void* x, int xtype, long long ldx, int m, int k, hipStream_t s) {
  const long long cols = SWIGLU ? 2LL * o.rows : o.rows;
  const long long big = ((m + 127) / 128) * ((cols + 127) / 128);
#define QC_F16(TM_, TN_, A_, B_, S_) \
  launch_tile<P, TM_, TN_, A_, B_, S_, GPS, SWIGLU>(xf, o, rexp, xs, x, xtype, ldx, m, k, s)
  if (big >= 5 * device_cu_count() / 4) return QC_F16(2, 2, 2, 4, P == 2 ? 3 : GPS == 0 ? 5 : 4);
  if constexpr (SWIGLU) return QC_F16(1, 2, 2, 2, P == 1 ? 8 : 6);
  else return QC_F16(2, 1, 1, 4, P == 1 ? 8 : 6);
#undef QC_F16
}

size_t up256(size_t b) { return (b + 255) / 256 * 256; }

}  // namespace

namespace {

// A call's scratch: the fragments of `rows` activation rows (chunks of at most
// 256 MB), their exponents, and with zero points their sums over 32 (groups of
// 32) or 64 columns.
struct F16Scratch {
  int p, gps, sums, chunk, rows;
  size_t xf_bytes, bytes;
};
F16Scratch f16_scratch(const CSegs& sg, const CInt8Launch& L, int m, int k) {
  F16Scratch f;
  f.p = L.xtype == QC_STORAGE_F32 ? 2 : 1;
  f.gps = sg.groups == 1 ? 0 : sg.gsize == 32 ? 2 : 1;
  bool zeros = false;
  for (int i = 0; i < L.nw; ++i) zeros = zeros || sg.zero[i] != nullptr;
  f.sums = !zeros ? 0 : f.gps == 2 ? 2 : 1;
  const long long fit = (256LL << 20) / (2LL * f.p * k) / 256 * 256;
  f.chunk = static_cast<int>(std::max<long long>(256, std::min<long long>(fit, 1 << 20)));
  f.rows = std::min(f.chunk, (m + 255) / 256 * 256);
  f.xf_bytes = up256(2ull * f.p * f.rows * k);
  f.bytes = f.xf_bytes + 4ull * f.rows + 4ull * f.rows * (k / 64) * f.sums;
  return f;
}

}  // namespace

size_t cint8_f16_scratch(const CSegs& sg, const CInt8Launch& L, int m, int k) {
  return f16_scratch(sg, L, m, k).bytes;
}

hipError_t launch_cint8_f16(const CSegs& sg, const CInt8Launch& L, int m, int k, hipStream_t s) {
  const F16Scratch f = f16_scratch(sg, L, m, k);
  const int p = f.p, gps = f.gps, sums = f.sums, chunk = f.chunk, rows = f.rows;
  const int nmat = L.mode == 1 ? 1 : L.nw;
  const size_t es = p == 2 ? 4 : 2;
  const bool vec = reinterpret_cast<uintptr_t>(L.x) % 16 == 0 && L.ldx % (16 / es) == 0;
  std::unique_lock<std::mutex> hold;
  uint8_t* base = nullptr;
  hipError_t e = call_scratch(s, f.bytes, hold, reinterpret_cast<void**>(&base));
  if (e != hipSuccess) return e;
  int* rexp = reinterpret_cast<int*>(base + f.xf_bytes);
  float* xs = reinterpret_cast<float*>(rexp + rows);
  for (int m0 = 0; m0 < m; m0 += chunk) {
    const int mc = std::min(chunk, m - m0);
    const void* xc = static_cast<const uint8_t*>(L.x) + es * static_cast<size_t>(m0) * L.ldx;
    const int groups = (mc + 7) / 8, steps = k / 64;
    const int want = std::max(1, std::min((steps + 7) / 8, 512 / groups));
    const int per = (steps + want - 1) / want;
    const dim3 grid(groups, (steps + per - 1) / per);
    if (p == 2) f16_prep<2><<<grid, 512, 0, s>>>(xc, L.xtype, L.ldx, vec, mc, k, per, base, rexp, xs, sums);
    else f16_prep<1><<<grid, 512, 0, s>>>(xc, L.xtype, L.ldx, vec, mc, k, per, base, rexp, xs, sums);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    for (int i = 0; i < nmat; ++i) {
      const bool pair = L.mode == 1;
      const int j = pair ? 1 : i;
      const size_t ys = sg.ytype[i] == QC_STORAGE_F32 ? 4 : 2;
      const F16Out o{{sg.w[i], sg.w[j]}, {sg.scale[i], sg.scale[j]}, {sg.zero[i], sg.zero[j]},
                     static_cast<uint8_t*>(sg.y[i]) + ys * static_cast<size_t>(m0) * sg.ld[i],
                     sg.ld[i], sg.ytype[i], static_cast<int>(L.w[i].rows), sg.bias, sg.act,
                     !pair && i == 0 && (sg.bias != nullptr || sg.act != 0) ? 1 : 0, sg.groups,
                     sg.gsize};
#define QC_F16(P_, G_, W_) launch_f16<P_, G_, W_>(base, o, rexp, xs, xc, L.xtype, L.ldx, mc, k, s)
#define QC_F16_G(P_, W_) \
  gps == 0 ? QC_F16(P_, 0, W_) : gps == 1 ? QC_F16(P_, 1, W_) : QC_F16(P_, 2, W_)
      e = p == 2 ? (pair ? QC_F16_G(2, true) : QC_F16_G(2, false))
                 : (pair ? QC_F16_G(1, true) : QC_F16_G(1, false));
#undef QC_F16_G
#undef QC_F16
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

}  // namespace qc
