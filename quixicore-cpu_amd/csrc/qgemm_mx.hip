// 2-D tiled q4_0 GEMM on gfx950's block-scaled 6-bit MFMA, for calls with
// enough activation rows to pay for re-encoding the weights.
//
// Semantics as the reference's qgemm (kernels/quantization/qgemm_ref.cpp:
// 156-162; its row-panel GEMM is kernels/quantization/qgemm_panel.cpp:234-286):
// y[m][n] = sum_b d[n][b] * sum_{k in b} q[n][k] * x[m][k].
//
// Numerics.  q4_0 codes (-8..7) are exact in E2M3.  Each activation of a
// 32-element block becomes four E2M3 digits, each under its own scale for the
// block: the power of two that takes the largest of what the digits before it
// left to at most 7.5.  x - sum of digits is then within 2^-20 of the power of
// two above the block's largest element (2^-19 of that element), and 2^-22 of
// the element in the root mean square of normal activations.  The scales are the
// instruction's own block scales.
// v_mfma_scale_f32_32x32x64_f8f6f4 with E2M3 operands multiplies two digits of
// 32 elements at once (the digits are its two K halves, against the same codes
// twice), so a block of a 32 x 32 tile is two MFMAs, half of the f16 form's
// four, folded into the f32 accumulators by one FMA per output with the
// block's scale.
//
// That step is absolute within a block: beside an element much larger than the
// rest, the rest lose bits, which shows in the outputs whose codes are small
// there (a channel large in every row, with small weights).  So a row whose
// blocks' squared maxima average kSpread times its mean magnitude squared (both as
// exponents) gets four more digits in the blocks kFar binades above that
// mean; the GEMM adds those blocks' products after its main loop.  Relative to
// the result, K = 4096, against 64 bits: N(0, 1) 5.3e-7, with 0.1% of the elements 20
// times larger 6.7e-7 (hi / lo bf16: 2.4e-6 both); two channels at 1000 and
// codes of zero there 5.2e-7 (bf16 2.5e-6, four digits alone 1.5e-5); the worst
// of some forty sets, with outliers just below the limits, 1.7e-6.  (Elements
// 2^-23 of their block's largest and below keep 15 bits or more, as an f32
// largest takes up to five of the eight digits.)
//
// What bounds it: VALU issue and MFMA power (16 fold FMAs and two MFMAs of 32
// cycles per tile and block).  Weights are re-encoded once per call (0.875
// bytes a weight, most of 20 us for 14336 x 4096, in the launch that encodes the
// activations), which decoding in the GEMM would repeat for every 128 or 256
// rows of x.  q4_0, N = 14336, K = 4096: M = 512 139 -> 102 us, M = 2048
// 552 -> 328 us (with blocks of eight digits: a third of them 116 and 440 us,
// all 205 and 713).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "qc_device.h"
#include "qc_internal.h"
#include "qc_lds_dma.h"
#include "qc_wide.h"

namespace qc {
namespace {

using namespace wide;

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x6 __attribute__((ext_vector_type(6)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

// Activations of one 32-row m-tile and block: operands j = 0, 1 as
// [64 lanes][16 B] then [64 lanes][8 B] (lane l: row l & 31, digit
// 2 j + (l >> 5): 32 6-bit codes), then the block's scale bytes [64 lanes]
// {operand 0, operand 1, 0, 0}.  A second array of the same layout holds the
// further digits of the blocks that have them, with a byte per eight rows and
// block that says so, and one per eight rows (any block).
constexpr int kXOp = 1536;
constexpr int kXFrag = 2 * kXOp;
constexpr int kXBlock = kXFrag + 256;
// Weights of one 32-row n-tile and block: [32 rows][16 B], [32 rows][8 B]
// codes, [32 rows] f32 scales.
constexpr int kWBlock = 32 * 28;
constexpr int kWSlot = 1024;                // its bytes in LDS (one load; the last 128 unused)
// Rows and blocks with further digits (modelled over forty distributions:
// silu(a) b and relu(a)^2 of normal a, b, whose ratio is 340-410, stay below;
// with up to 800 the four digits' error is at most 1.7e-6 of any outputs).
constexpr float kSpread = 800.0f;
constexpr float kFar = 5.0f;

// Codes 2 i and 2 i + 1 of a block's 32 are elements i and i + 16: the order
// of the q4_0 bytes' nibbles, and of v_cvt_scalef32_2xpk16_fp6_f32.

// Four nibbles u (bytes 0..15) as the E2M3 codes of (u - 8) / 8: sign, and a
// magnitude 0..8 whose code is the integer itself (E2M3 is linear in eighths
// up to 15 / 8).
__device__ __forceinline__ uint32_t nibble_codes(uint32_t u) {
  const uint32_t s = ((u >> 3) & 0x01010101u) ^ 0x01010101u;      // u < 8
  const uint32_t mag = ((u ^ ((s << 3) - s)) & 0x07070707u) + s;  // u < 8: 7 - u + 1
  return mag | (s << 5);
}
// The eight codes of four q4_0 bytes: 24 bits each of bytes 0, 1 and 2, 3.
__device__ __forceinline__ void byte_codes(uint32_t c, uint32_t& lo, uint32_t& hi) {
  const uint32_t l = nibble_codes(c & 0x0F0F0F0Fu), h = nibble_codes((c >> 4) & 0x0F0F0F0Fu);
  const uint32_t even = (l & 0x00FF00FFu) | ((h & 0x00FF00FFu) << 6);
  const uint32_t odd = ((l >> 8) & 0x00FF00FFu) | ((h >> 2) & 0x3FC03FC0u);
  lo = (even & 0xFFFu) | ((odd & 0xFFFu) << 12);
  hi = (even >> 16) | ((odd >> 16) << 12);
}

// One launch prepares both operands.  Workgroups [0, xwgs): eight activation
// rows each and one of `slices` slices of K: the rows' power-of-two scales
// (largest element in [0.5, 1)) and spreads, then the digits of the slice's
// blocks, one lane per row and block.  The next wwgs: weights, a wave per n-tile
// and two block pairs, one lane per row and pair (with eight pairs a wave the
// last workgroups run on after the others: 14336 x 4096, M = 512 104 -> 99 us for
// the whole call).  Any beyond clear y.
__global__ __launch_bounds__(512) void mx_prep(const float* __restrict__ x, int M, int K,
                                               int slices, int blocks_per_slice, int xwgs,
                                               uint8_t* __restrict__ xf, uint8_t* __restrict__ xr,
                                               uint8_t* __restrict__ xflag,
                                               uint8_t* __restrict__ xspread, int* __restrict__ rexp,
                                               const uint8_t* __restrict__ W, int N,
                                               uint8_t* __restrict__ wf, int wwgs,
                                               float* zero_y, long long ldy) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nb = K / 32, npairs = K / 64;
  if (static_cast<int>(blockIdx.x) >= xwgs + wwgs) {
    const int first = blockIdx.x - xwgs - wwgs, stride = gridDim.x - xwgs - wwgs;
    for (int m = first; m < M; m += stride)
      for (int n = tid; n < N; n += 512) zero_y[m * ldy + n] = 0.0f;
    return;
  }
  if (static_cast<int>(blockIdx.x) >= xwgs) {
    const int groups = (npairs + 1) / 2;
    const int ntiles = (N + 31) / 32;
    const long long item = static_cast<long long>(blockIdx.x - xwgs) * 8 + wave;
    const int nt = static_cast<int>(item / groups);
    const int p = 2 * static_cast<int>(item % groups) + (lane >> 5);
    if (nt >= ntiles || p >= npairs) return;
    const int col = lane & 31;
    const long long r = min(32 * nt + col, N - 1);
    const uint8_t* src = W + r * npairs * 36;
    uint8_t* dst = wf + static_cast<long long>(nt) * nb * kWBlock;
    const uint32_t* s = reinterpret_cast<const uint32_t*>(src + 36LL * p);
    uint32_t q[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) q[i] = s[i];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        c[i] = h == 0 ? __builtin_amdgcn_alignbyte(q[i + 1], q[i], 2) : q[5 + i];
      uint32_t o[6];
#pragma unroll
      for (int i = 0; i < 4; i += 2) {           // two dwords: 96 bits
        uint32_t a, b, e, f;
        byte_codes(c[i], a, b);
        byte_codes(c[i + 1], e, f);
        o[3 * (i / 2)] = a | (b << 24);
        o[3 * (i / 2) + 1] = (b >> 8) | (e << 16);
        o[3 * (i / 2) + 2] = (e >> 16) | (f << 8);
      }
      uint8_t* t = dst + static_cast<long long>(2 * p + h) * kWBlock;
      *reinterpret_cast<u32x4*>(t + 16 * col) = u32x4{o[0], o[1], o[2], o[3]};
      *reinterpret_cast<u32x2*>(t + 512 + 8 * col) = u32x2{o[4], o[5]};
      *reinterpret_cast<float*>(t + 768 + 4 * col) =
          half_bits_to_float(h == 0 ? q[0] & 0xFFFFu : q[4] >> 16);
    }
    return;
  }

  __shared__ int sexp[8], sfar[8];
  const int group = blockIdx.x / slices, slice = blockIdx.x % slices;
  const int m0 = 8 * group;
  const bool aligned = reinterpret_cast<uintptr_t>(x) % 16 == 0;
  if (m0 + wave < M) {                             // wave w: row m0 + w
    const float* xr0 = x + static_cast<long long>(m0 + wave) * K;
    float mx = 0.f, z = 0.f;
    // exponents of the row's nonzero elements (sum and count); sum of 4^exponent
    // of its nonzero blocks' maxima, as bs * 4^be, and their count
    int esum = 0, count = 0, blocks = 0, be = -1000;
    float bs = 0.f;
    // v: this lane's elements of a block of 8 lanes (wide: of 32)
    auto see = [&](const f32x4& v, bool wide) {
      float bm = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = fabsf(v[e]);
        esum += __builtin_amdgcn_frexp_expf(a);   // 0 for 0
        count += a > 0.f ? 1 : 0;
        bm = fmaxf(bm, a);
        z = fmaf(0.0f, v[e], z);                   // NaN once an element is not finite
      }
      bm = group8_max(bm);
      if (wide) {
        bm = fmaxf(bm, __shfl_xor(bm, 8));
        bm = fmaxf(bm, __shfl_xor(bm, 16));
      }
      mx = fmaxf(mx, bm);
      if (bm > 0.f) {
        const int ex = __builtin_amdgcn_frexp_expf(bm);
        const int ne = max(be, ex);
        bs = ldexpf(bs, 2 * (be - ne)) + ldexpf(1.0f, 2 * (ex - ne));
        be = ne;
        ++blocks;
      }
    };
    if (aligned) {
      const f32x4* x4 = reinterpret_cast<const f32x4*>(xr0);
      const int n4 = K / 4;
      int i = lane;
      for (; i + 448 < n4; i += 512) {
        f32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = x4[i + 64 * u];
#pragma unroll
        for (int u = 0; u < 8; ++u) see(v[u], false);
      }
      for (; i < n4; i += 64) see(x4[i], false);
    } else {
      for (int i = lane; i < K; i += 64) see(f32x4{xr0[i], 0.f, 0.f, 0.f}, true);
    }
    mx = wave_max_nonneg(mx);
    const bool bad = __any(z != 0.0f);
    int e = 0;
    if (mx > 0.f && mx <= 3.402823466e38f) (void)frexpf(mx, &e);
    // every lane of a block carries its term: the copies cancel in the ratio
    const float sum = wave_sum(ldexpf(bs, max(2 * (be - e), -400)));
    const float mean = wave_sum(static_cast<float>(esum)) / wave_sum(static_cast<float>(count));
    const bool far = !bad && sum > kSpread * wave_sum(static_cast<float>(blocks)) *
                                          exp2f(2.0f * (mean - static_cast<float>(e)));
    if (lane == 0) {
      sexp[wave] = bad ? 0 : e;
      sfar[wave] = far ? static_cast<int>(ceilf(mean + kFar)) - e : INT_MAX;
      if (slice == 0) rexp[m0 + wave] = bad ? kRowNonfinite : e;
    }
  }
  __syncthreads();
  const int row = lane & 7;
  const int m = m0 + row;
  if (m >= M) return;
  const bool spread = __any(sfar[row] != INT_MAX);
  if (slice == 0 && tid == 0) xspread[group] = spread ? 1 : 0;
  const int e = -sexp[row], farex = sfar[row];
  const int b0 = slice * blocks_per_slice, b1 = min(b0 + blocks_per_slice, nb);
  for (int b = b0 + 8 * wave + (lane >> 3); b < b1; b += 64) {
    const float* src = x + static_cast<long long>(m) * K + 32 * b;
    f32x16 lo, hi;                                 // elements 0..15 and 16..31
    if (aligned) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 a = reinterpret_cast<const f32x4*>(src)[i];
        const f32x4 c = reinterpret_cast<const f32x4*>(src)[4 + i];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          lo[4 * i + u] = a[u];
          hi[4 * i + u] = c[u];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        lo[i] = src[i];
        hi[i] = src[16 + i];
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      lo[i] = ldexpf(lo[i], e);
      hi[i] = ldexpf(hi[i], e);
    }
    // Four digits of what lo, hi hold (which keep what the digits leave,
    // exactly) to a block's fragments at d; the exponent of the largest.
    const int r = m & 31;
    auto digits = [&](uint8_t* d) {
      int first = INT_MIN;
      uint32_t sb[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fmaxf(fabsf(lo[i]), fabsf(hi[i])));
        int ex = -123;
        float f = 0.f;
        if (mx > 0.f && mx <= 3.402823466e38f) {
          f = frexpf(mx, &ex);
          if (t == 0) first = ex;
        }
        // 2^s: the largest at most 7.5 of it
        const int s = max(ex - (f > 0.9375f ? 2 : 3), -126);
        const float scale = __int_as_float((s + 127) << 23);
        const u32x6 o = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(lo, hi, scale);
        const f32x32 v = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(o, scale);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          lo[i] -= v[2 * i];
          hi[i] -= v[2 * i + 1];
        }
        uint8_t* op = d + (t >> 1) * kXOp;
        const int l = r + 32 * (t & 1);
        *reinterpret_cast<u32x4*>(op + 16 * l) = u32x4{o[0], o[1], o[2], o[3]};
        *reinterpret_cast<u32x2*>(op + 1024 + 8 * l) = u32x2{o[4], o[5]};
        sb[t] = static_cast<uint32_t>(s + 127);
      }
      // scale bytes (exponent + 127) of digits h and 2 + h, h = 0, 1
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<uint32_t*>(d + kXFrag + 4 * (r + 32 * h)) = sb[h] | (sb[2 + h] << 8);
      return first;
    };
    const long long at = static_cast<long long>(m >> 5) * nb + b;
    const bool more = digits(xf + at * kXBlock) >= farex;
    // further digits for all eight rows once one of them needs them
    const bool any = (__ballot(more) >> (lane & 56) & 0xFFu) != 0;
    if (row == 0) xflag[4 * at + (r >> 3)] = any ? 1 : 0;
    if (any) (void)digits(xr + at * kXBlock);
  }
}

// Tile of TM x TN 32 x 32 MFMA tiles per wave, WGM x WGN waves, S block
// stages in LDS.
template <int TM, int TN, int WGM, int WGN, int S>
struct Mx {
  static constexpr int NW = WGM * WGN;
  static constexpr int MT = TM * WGM, NT = TN * WGN;          // m-tiles, n-tiles
  static constexpr int BM = 32 * MT, BN = 32 * NT;
  static constexpr int FL = (MT * 3 + NW - 1) / NW;           // 1 KB operand loads per wave
  static constexpr int SL = (MT + NW - 1) / NW;               // scale loads
  static constexpr int WL = (NT + NW - 1) / NW;               // n-tile loads
  static constexpr int G = FL + SL + WL;
  static constexpr int XS = MT * kXFrag, SS = MT * 256, WS = NT * kWSlot;
  static constexpr int stage = XS + SS + WS;
  static constexpr int lds = S * stage;
  static_assert(lds <= 160 * 1024 && G * (S - 2) < 64 && S >= 3, "ring");
};

template <int TM, int TN, int WGM, int WGN, int S>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void mx_gemm(
    const uint8_t* __restrict__ wf, const uint8_t* __restrict__ xf, const uint8_t* __restrict__ xr,
    const uint8_t* __restrict__ xflag, const uint8_t* __restrict__ xspread, float* __restrict__ y,
    const int* __restrict__ rexp, const uint8_t* __restrict__ W, const float* __restrict__ x, int M, int N, long long ldy,
    int K, int mblocks, int nblocks, int blocks_per_split, int ks_count) {
  using C = Mx<TM, TN, WGM, WGN, S>;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[C::lds];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WGM, wn = wave / WGM;
  const int col = lane & 31;

  int mb, nbk, ks;
  tile_of_workgroup(mblocks, nblocks, ks_count, mb, nbk, ks);
  const int mt0 = mb * C::MT, nt0 = nbk * C::NT;
  const int nb = K / 32;
  const int ntiles = (N + 31) / 32;
  const int b0 = ks * blocks_per_split, b1 = min(b0 + blocks_per_split, nb);
  const int steps = b1 - b0;

  // Sources, advanced by one block per issue and stopped at the last one.
  // Loads past the tile's share (a count that does not divide by the waves)
  // repeat its last one: the same bytes to the same place.
  const uint8_t* xsrc = uniform_ptr(xf + (static_cast<long long>(mt0) * nb + b0) * kXBlock);
  const uint8_t* wsrc = uniform_ptr(wf + static_cast<long long>(b0) * kWBlock);
  int left = __builtin_amdgcn_readfirstlane(steps - 1);
  const long long xtile = static_cast<long long>(nb) * kXBlock, wtile = static_cast<long long>(nb) * kWBlock;
  auto fq = [&](int i) { return __builtin_amdgcn_readfirstlane(min(wave * C::FL + i, 3 * C::MT - 1)); };
  auto sq = [&](int i) { return __builtin_amdgcn_readfirstlane(min(wave * C::SL + i, C::MT - 1)); };
  auto wq = [&](int i) { return __builtin_amdgcn_readfirstlane(min(wave * C::WL + i, C::NT - 1)); };
  const uint8_t* fsrc[C::FL];
  const uint8_t* ssrc[C::SL];
  const uint8_t* nsrc[C::WL];
#pragma unroll
  for (int i = 0; i < C::FL; ++i) {
    const int q = fq(i);
    fsrc[i] = uniform_ptr(xsrc + (q / 3) * xtile + (q % 3) * 1024);
  }
#pragma unroll
  for (int i = 0; i < C::SL; ++i)
    ssrc[i] = uniform_ptr(xsrc + sq(i) * xtile + kXFrag);
#pragma unroll
  for (int i = 0; i < C::WL; ++i)
    nsrc[i] = uniform_ptr(wsrc + min(nt0 + wq(i), ntiles - 1) * wtile);
  auto issue = [&](int slot, int l) {
    uint8_t* base = lds + slot * C::stage;
    if (l < C::FL) {
      dma16(fsrc[l < C::FL ? l : 0], 16 * lane, base + fq(l) * 1024);
    } else if (l < C::FL + C::SL) {
      const int i = l - C::FL;
      dma4(ssrc[i < C::SL ? i : 0], 4 * lane, base + C::XS + sq(i) * 256);
    } else {
      const int i = l - C::FL - C::SL;
      dma16(nsrc[i < C::WL ? i : 0], 16 * lane, base + C::XS + C::SS + wq(i) * kWSlot);
    }
  };
  auto advance = [&]() {
    const int dx = left > 0 ? kXBlock : 0, dw = left > 0 ? kWBlock : 0;
    --left;
#pragma unroll
    for (int i = 0; i < C::FL; ++i) fsrc[i] += dx;
#pragma unroll
    for (int i = 0; i < C::SL; ++i) ssrc[i] += dx;
#pragma unroll
    for (int i = 0; i < C::WL; ++i) nsrc[i] += dw;
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  auto read6 = [&](const uint8_t* p16, const uint8_t* p8, i32x8& o) {
    const i32x4 a = *reinterpret_cast<const i32x4*>(p16);
    const u32x2 b = *reinterpret_cast<const u32x2*>(p8);
    o[0] = a[0];
    o[1] = a[1];
    o[2] = a[2];
    o[3] = a[3];
    o[4] = static_cast<int>(b[0]);
    o[5] = static_cast<int>(b[1]);
  };
  // operand j and scales of m-tile tm, n-tile tn's codes and scale
  auto read_a = [&](int slot, int tm, int j, i32x8& o) {
    const uint8_t* p = lds + slot * C::stage + (wm * TM + tm) * kXFrag + j * kXOp;
    read6(p + 16 * lane, p + 1024 + 8 * lane, o);
  };
  auto read_s = [&](int slot, int tm) {
    return *reinterpret_cast<const int*>(lds + slot * C::stage + C::XS + (wm * TM + tm) * 256 + 4 * lane);
  };
  auto read_w = [&](int slot, int tn, i32x8& o, float& d) {
    const uint8_t* p = lds + slot * C::stage + C::XS + C::SS + (wn * TN + tn) * kWSlot;
    read6(p + 16 * col, p + 512 + 8 * col, o);
    d = *reinterpret_cast<const float*>(p + 768 + 4 * col);
  };

  // Per m-tile a byte for each eight rows: any of them with further digits at
  // all, and (per block) in block b.  Bytes past M are not set.
  auto in_rows = [&](int tm, uint32_t f) {
    const int groups = (M - 32 * (mt0 + wm * TM + tm) + 7) / 8;
    return groups >= 4 ? f : groups <= 0 ? 0u : f & ((1u << (8 * groups)) - 1);
  };
  uint32_t further = 0;

  if (steps > 0) {
    // Barrier B_s stands before the last m-tile of step s.  Step s issues,
    // before B_s, stage s + S - 1 into the slot of stage s - 1; at B_s the
    // loads of the last S - 2 steps may be outstanding, so stage s + 1 is in.
#pragma unroll
    for (int r = 0; r < S - 1; ++r) {
#pragma unroll
      for (int l = 0; l < C::G; ++l) issue(r, l);
      advance();
    }
    typedef uint32_t Words __attribute__((ext_vector_type(TM)));   // (while those are in flight)
    const Words spread = *reinterpret_cast<const Words*>(xspread + 4 * (mt0 + wm * TM));
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) further |= in_rows(tm, spread[tm]);
    wait_vmcnt<(S - 2) * C::G>();
    ring_barrier();
    i32x8 a[2][2], w[2][TN];                       // two buffers each
    int sc[2];
    float d[2][TN];
#pragma unroll
    for (int j = 0; j < 2; ++j) read_a(0, 0, j, a[0][j]);
    sc[0] = read_s(0, 0);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) read_w(0, tn, w[0][tn], d[0][tn]);
    f32x16 c[2];
    float dprev = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) c[1][e] = 0.f;
    int cur = 0;
    auto step = [&](auto par) {
      constexpr int P = decltype(par)::value;      // weight buffer of this step
      constexpr int T = TM * TN, B = (TM - 1) * TN;
      static_assert(TM % 2 == 0 && T % 2 == 0 && TN <= 2, "buffers alternate within a step");
      const int nxt = cur + 1 < S ? cur + 1 : 0, free = cur > 0 ? cur - 1 : S - 1;
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const int tm = i / TN, tn = i % TN, ab = tm & 1;
        const int pi = i == 0 ? T - 1 : i - 1, pm = pi / TN, pn = pi % TN;
        if (i == B) {
          wait_vmcnt<(S - 2) * C::G>();
          wait_lgkmcnt0();
          ring_barrier();
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const f32x16 z = {};
          // E2M3 operands; A scale: byte q; B scale 2^3 (codes are eighths)
          c[i & 1] = q == 0 ? __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                                  a[ab][0], w[P][tn], z, 2, 2, 0, sc[ab], 0, 130)
                            : __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                                  a[ab][1], w[P][tn], c[i & 1], 2, 2, 1, sc[ab], 0, 130);
          __builtin_amdgcn_sched_barrier(0);
          const int slot = 2 * i + q;
          // the next m-tile's operands, one per n-tile pair of slots
          const int rs = tm + 1 < TM ? cur : nxt, rm = tm + 1 < TM ? tm + 1 : 0;
          const int ms = 2 * tn + q;
          if (ms == 0) sc[ab ^ 1] = read_s(rs, rm);
          if (ms == TN - 1) read_a(rs, rm, 0, a[ab ^ 1][0]);
          if (ms == 2 * TN - 1 - (TN > 1 ? 1 : 0)) read_a(rs, rm, 1, a[ab ^ 1][1]);
          // the next block's weights, right after B_s
          if (i == B && q < TN) read_w(nxt, q, w[P ^ 1][q], d[P ^ 1][q]);
          if (i < B) {
#pragma unroll
            for (int l = slot * C::G / (2 * B); l < (slot + 1) * C::G / (2 * B); ++l) issue(free, l);
          }
          // the previous tile: its last MFMA runs into slot 0
#pragma unroll
          for (int e = q == 0 ? 0 : 5; e < (q == 0 ? 5 : 16); ++e)
            acc[pm][pn][e] = fmaf(c[(i & 1) ^ 1][e], dprev, acc[pm][pn][e]);
          if (q == 1) dprev = d[P][tn];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      cur = nxt;
      advance();
    };
    int s = 0;
    for (; s + 1 < steps; s += 2) {
      step(std::integral_constant<int, 0>());
      step(std::integral_constant<int, 1>());
    }
    if (s < steps) step(std::integral_constant<int, 0>());
#pragma unroll
    for (int e = 0; e < 16; ++e)
      acc[TM - 1][TN - 1][e] = fmaf(c[1][e], dprev, acc[TM - 1][TN - 1][e]);
  }
  wait_vmcnt<0>();   // no global->LDS load may outlive the workgroup's LDS

  // The further digits, from memory: few blocks, each wave its own m-tiles'.
  if (further != 0) {
    for (int c0 = b0; c0 < b1; c0 += 64) {
      uint32_t f[TM];
      uint64_t todo = 0;
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        const int b = min(c0 + lane, b1 - 1);
        const long long at = static_cast<long long>(mt0 + wm * TM + tm) * nb + b;
        f[tm] = c0 + lane < b1 ? in_rows(tm, reinterpret_cast<const uint32_t*>(xflag)[at]) : 0;
        todo |= __ballot(f[tm] != 0);
      }
      while (todo != 0) {
        const int i = __builtin_ctzll(todo);
        todo &= todo - 1;
        i32x8 w[TN], a[TM][2];
        int sc[TM];
        float d[TN];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const uint8_t* p = wf + min(nt0 + wn * TN + tn, ntiles - 1) * wtile + (c0 + i) * kWBlock;
          read6(p + 16 * col, p + 512 + 8 * col, w[tn]);
          d[tn] = *reinterpret_cast<const float*>(p + 768 + 4 * col);
        }
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
          const uint32_t g = __builtin_amdgcn_readlane(f[tm], i);
          const i32x8 zero = {};
          a[tm][0] = a[tm][1] = zero;
          sc[tm] = 0;
          if (g >> (8 * (col >> 3)) & 0xFF) {
            const uint8_t* p = xr + (mt0 + wm * TM + tm) * xtile + (c0 + i) * kXBlock;
#pragma unroll
            for (int j = 0; j < 2; ++j)
              read6(p + j * kXOp + 16 * lane, p + j * kXOp + 1024 + 8 * lane, a[tm][j]);
            sc[tm] = *reinterpret_cast<const int*>(p + kXFrag + 4 * lane);
          }
        }
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) {
            const f32x16 z = {};
            f32x16 v = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[tm][0], w[tn], z, 2, 2, 0,
                                                                       sc[tm], 0, 130);
            v = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[tm][1], w[tn], v, 2, 2, 1, sc[tm],
                                                                0, 130);
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[tm][tn][e] = fmaf(v[e], d[tn], acc[tm][tn][e]);
          }
      }
    }
  }

  store_tiles<TM, TN>(acc, rexp, y, ldy, ks_count > 1, 32 * (mt0 + wm * TM), 32 * (nt0 + wn * TN), M, N,
                      [&](int m, int n) {
                        return nonfinite_blocks_f32<kQ4_0>(W + static_cast<long long>(n) * nb * 18,
                                                           x + static_cast<long long>(m) * K, b0, b1);
                      });
}

// Times per block, measured on MI355X at K = 4096: 256 x 256 tiles 118 us
// for 112 workgroups, 298 for 448; 128 x 256 85 us for 224, 326 for 896;
// 128 x 128 48 us for 64, 92 for 448, 339 for 1792.
constexpr int kTiles = 3;
constexpr Tile kTile[kTiles] = {
    {256, 256, 1, 0.88, 1.30}, {128, 256, 1, 0.42, 0.74}, {128, 128, 2, 0.35, 0.80}};

// A call's operands: activation fragments, their further digits and which blocks
// have them, row exponents, re-encoded weights.
struct Operands {
  uint8_t *xf, *xr, *xflag, *xspread, *wf;
  int* rexp;
};

template <int TM, int TN, int WGM, int WGN, int S>
hipError_t launch_tile(const Operands& o, float* y, const uint8_t* W, const float* x, int m, int n,
                       long long ldy, int k, const TilePlan& p, hipStream_t s) {
  using C = Mx<TM, TN, WGM, WGN, S>;
  const int mblocks = (m + C::BM - 1) / C::BM, nblocks = (n + C::BN - 1) / C::BN;
  mx_gemm<TM, TN, WGM, WGN, S><<<static_cast<unsigned>(mblocks) * nblocks * p.ks, 64 * C::NW, 0, s>>>(
      o.wf, o.xf, o.xr, o.xflag, o.xspread, y, o.rexp, W, x, m, n, ldy, k, mblocks, nblocks, p.per, p.ks);
  return hipGetLastError();
}

// One chunk of rows and one of weight rows, each encoded here unless a call
// before did.
hipError_t run_mx(const Operands& o, bool encode_x, bool encode_w, const uint8_t* W, const float* x,
                  float* y, int m, int n, long long ldy, int k, hipStream_t s) {
  const int nb = k / 32;
  const TilePlan p = plan_tiles(kTile, kTiles, m, n, nb, device_cu_count(), 0, 2);
  // activations: eight rows a workgroup, K in as many slices as give ~512
  // workgroups of at least 64 blocks (one per eight lanes)
  const int groups = (m + 7) / 8;
  const int want = std::max(1, std::min((nb + 63) / 64, 512 / groups));
  const int per_slice = (nb + want - 1) / want;
  const int slices = (nb + per_slice - 1) / per_slice;
  const int xwgs = encode_x ? groups * slices : 0;
  const long long items = static_cast<long long>((n + 31) / 32) * ((k / 64 + 1) / 2);
  const int wwgs = encode_w ? static_cast<int>((items + 7) / 8) : 0;
  const int clear = p.ks == 2 ? 512 : 0;
  if (xwgs + wwgs + clear > 0) {
    mx_prep<<<static_cast<unsigned>(xwgs) + wwgs + clear, 512, 0, s>>>(
        x, m, k, slices, per_slice, xwgs, o.xf, o.xr, o.xflag, o.xspread, o.rexp, W, n, o.wf, wwgs, y, ldy);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  switch (p.tile) {
    case 0: return launch_tile<4, 2, 2, 4, 4>(o, y, W, x, m, n, ldy, k, p, s);
    case 1: return launch_tile<2, 2, 2, 4, 6>(o, y, W, x, m, n, ldy, k, p, s);
    default: return launch_tile<2, 2, 2, 2, 4>(o, y, W, x, m, n, ldy, k, p, s);
  }
}

// Chunks of at most `most` (at least 256) as even as multiples of 256 allow.
int even_chunk(int count, long long most) {
  const int cap = static_cast<int>(std::max<long long>(256, std::min<long long>(most / 256 * 256, INT_MAX / 2)));
  const int chunks = (count + cap - 1) / cap;
  return ((count + chunks - 1) / chunks + 255) / 256 * 256;
}

}  // namespace

// The 6-bit form saves about a quarter of the f16 form's time where it fills
// the chip, against about 8 us of encoding and of a second prep's latency (so
// from 4.8e9 products), and its larger tiles leave CUs idle below some 2.3e6
// outputs, more with long K, which the f16 form cuts into up to eight ranges.
// Measured over 280 shapes, f16 / 6-bit form in us: K = 512 N = 6144 M = 768 24.5
// / 23.5, N = 14336 M = 512 / 2048 26.0 / 28.3 and 79.3 / 70.4; K = 1024 N = 4096
// M = 512 / 1024 / 2048 20.1 / 27.0, 30.9 / 31.2 and 47.1 / 42.1; K = 4096 N = 2048
// M = 384 / 1024 / 2048 34.8 / 41.8, 54.2 / 56.0 and 92.9 / 79.1, N = 4096 M = 512 /
// 768 49.8 / 51.1 and 75.1 / 66.2, N = 14336 M = 384 / 512 118 / 88 and 123 / 101;
// K = 14336 N = 2048 M = 512 / 2048 90 / 132 and 290 / 251, N = 4096 M = 512 / 1024
// 143 / 151 and 250 / 236.  The worst pick is 5% off the faster form.
bool mx_pays(int m, int n, int k) {
  const double outs = static_cast<double>(m) * n;
  return m >= 384 && n >= 2048 && outs * k >= 4.8e9 && outs >= 2.3e6 + 40.0 * std::max(0, k - 4096);
}

hipError_t launch_qgemm_mx(const void* W, const float* x, float* y, int m, int n, int k,
                           hipStream_t s, StreamWorkspace* ws) {
  const auto* w = static_cast<const uint8_t*>(W);
  const int nb = k / 32;
  // Activation rows in chunks whose digits (3.25 bytes an element) take at most
  // 256 MB, and as much for their further digits; weight rows in chunks of at most 256 MB (0.875 bytes a weight).
  const int mchunk = even_chunk(m, (256LL << 20) / (4LL * k));
  const int nchunk = even_chunk(n, (256LL << 20) / k);
  const size_t mpad = (std::min(m, mchunk) + 255) / 256 * 256;   // read in whole tiles
  const size_t xf_bytes = mpad / 32 * nb * kXBlock, flag_bytes = mpad / 8 * (nb + 1);
  const size_t wf_bytes = static_cast<size_t>((std::min(n, nchunk) + 31) / 32) * nb * kWBlock + 128;   // kWSlot reads
  void* buf = nullptr;
  hipError_t e = stream_buffer(ws, s, 2 * xf_bytes + flag_bytes + wf_bytes, 0, &buf);
  if (e != hipSuccess) return e;
  Operands o;
  o.xf = static_cast<uint8_t*>(buf);
  o.xr = o.xf + xf_bytes;
  o.xflag = o.xr + xf_bytes;
  o.xspread = o.xflag + mpad / 8 * nb;
  o.wf = o.xflag + flag_bytes;
  e = stream_buffer(ws, s, sizeof(int) * mpad, 1, &buf);
  if (e != hipSuccess) return e;
  o.rexp = static_cast<int*>(buf);
  // each chunk of weights encoded once, its rows inside; the rows once where
  // they are one chunk
  for (int n0 = 0; n0 < n; n0 += nchunk)
    for (int m0 = 0; m0 < m; m0 += mchunk) {
      e = run_mx(o, m > mchunk || n0 == 0, m0 == 0, w + static_cast<long long>(n0) * nb * 18,
                 x + static_cast<long long>(m0) * k, y + static_cast<long long>(m0) * n + n0,
                 std::min(mchunk, m - m0), std::min(nchunk, n - n0), n, k, s);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

}  // namespace qc
