// 2-D tiled q8_0 / q4_0 GEMM on gfx950 f16 MFMA, for more activation rows
// than one small-batch pass takes.
//
// Semantics as the reference's qgemm (kernels/quantization/qgemm_ref.cpp:
// 156-162; its own row-panel GEMM is kernels/quantization/qgemm_panel.cpp:
// 234-286): y[m][n] = sum_b d[n][b] * sum_{k in b} q[n][k] * x[m][k].
//
// Numerics.  Each activation row is scaled by a power of two and split into
// hi = f16(x) and lo = f16(x - hi), so x - hi - lo is within 2^-22 |x| + 2^-25
// at that scale (largest element in [2^14, 2^15)); codes (-128..127) are exact
// in f16.  A 32-element block of a 32 x 32 tile is four
// v_mfma_f32_32x32x16_f16 (two K halves, hi and lo) into a zeroed tile, folded
// into the f32 accumulators by one FMA per output with the block's scale.
//
// What bounds it: MFMA power and VALU issue.  Per tile and block a wave has
// four MFMAs (32 cycles each) and 16 fold FMAs; with 32 x 32 tiles these
// overlap, where the 16 x 16 x 32 form of the same work spends its time
// issuing.  A wave takes 4 x 2 tiles (128 x 64 outputs), so that a weight
// fragment's decode (12 VALU per four codes of a lane) is shared by four tiles
// and an activation fragment's LDS read by two.  Every slot of the main loop is
// one MFMA with its share of the previous tile's fold, the next operands' LDS
// reads, the next block's decode and the ring's loads, in fixed order.
// q8_0, N = 14336, K = 4096, M = 2048: 602 -> 467 us (515 TFLOP/s; a plain f16
// GEMM of this chip reaches 1430, and this is two products); M = 77, N = 5461,
// K = 2752: 51.7 -> 24.5 us (three passes of 32 rows before).  For 17-32 rows
// (q4_0) a 32 x 128 tile of four waves: what bounds it there is the activation
// fragments, which every workgroup reads whole (57 MB from L2 at N = 14336,
// K = 4096, beside 33 MB of weights): 28.0 -> 24.4 us; N = 28672, K = 14336
// 172 -> 111 us.
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

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Activation fragments: [32-row m-tile][block][hi s0 | lo s0 | hi s1 | lo s1]
// [64 lanes][16 B]; lane l of slot s holds row l & 31, elements 16 (l >> 5) +
// 8 s + i (i = 0..7) of the 32-element block.
constexpr int kStepBytes = 4096;

// Eight activation rows per workgroup (blockIdx.x), K in gridDim.y slices of
// whole blocks: each row's power-of-two scale (its largest element goes into
// [2^14, 2^15), so that no element that matters is subnormal in f16 and no
// product overflows), found over the whole row by every slice, then the
// slice's fragments.  A 128-byte line of a fragment is eight rows' 16-byte
// pieces, so each line is written whole by one store of eight lanes.
// Workgroups blockIdx.x >= ceil(M / 8) only clear y.
__global__ __launch_bounds__(512) void wide_prep(const float* __restrict__ x, int M, int K,
                                                 int blocks_per_slice, uint8_t* __restrict__ xf,
                                                 int* __restrict__ rexp, float* zero_y,
                                                 long long zero_count) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row_groups = (M + 7) / 8;
  if (static_cast<int>(blockIdx.x) >= row_groups) {
    const long long w = (blockIdx.x - row_groups) * gridDim.y + blockIdx.y;
    const long long first = w * 512 + tid;
    const long long stride = static_cast<long long>(gridDim.x - row_groups) * gridDim.y * 512;
    long long done = 0;
    if (reinterpret_cast<uintptr_t>(zero_y) % 16 == 0) {
      const long long n4 = zero_count / 4;
      for (long long i = first; i < n4; i += stride)
        reinterpret_cast<f32x4*>(zero_y)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      done = 4 * n4;
    }
    for (long long i = done + first; i < zero_count; i += stride) zero_y[i] = 0.0f;
    return;
  }
  __shared__ int sexp[8];
  const int m0 = 8 * blockIdx.x;
  const int nb = K / 32;
  const bool aligned = reinterpret_cast<uintptr_t>(x) % 16 == 0;   // rows are K % 64 floats

  // wave w: the maximum of row m0 + w
  if (m0 + wave < M) {
    const float* xr = x + static_cast<long long>(m0 + wave) * K;
    float mx = 0.f, z = 0.f;
    auto see = [&](const f32x4& v) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        mx = fmaxf(mx, fabsf(v[e]));
        z = fmaf(0.0f, v[e], z);                   // NaN once an element is not finite
      }
    };
    if (aligned) {
      const f32x4* x4 = reinterpret_cast<const f32x4*>(xr);
      const int n4 = K / 4;
      int i = lane;
      for (; i + 448 < n4; i += 512) {
        f32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = x4[i + 64 * u];
#pragma unroll
        for (int u = 0; u < 8; ++u) see(v[u]);
      }
      for (; i < n4; i += 64) see(x4[i]);
    } else {
      for (int i = lane; i < K; i += 64) see(f32x4{xr[i], 0.f, 0.f, 0.f});
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

  // lane: row m0 + (lane & 7), eight elements (operand s of half) of one block
  const int row = lane & 7, s = (lane >> 3) & 1, half = (lane >> 4) & 1;
  const int m = m0 + row;
  if (m >= M) return;
  const int e = -sexp[row];
  const float* src = x + static_cast<long long>(m) * K + 16 * half + 8 * s;
  uint8_t* dst = xf + static_cast<long long>(m >> 5) * nb * kStepBytes + 16 * (m & 31) + 512 * half +
                 2048 * s;
  const int b0 = blockIdx.y * blocks_per_slice;
  const int b1 = min(b0 + blocks_per_slice, nb);
  for (int b = b0 + 2 * wave + (lane >> 5); b < b1; b += 16) {
    float v[8];
    if (aligned) {
      *reinterpret_cast<f32x4*>(&v[0]) = *reinterpret_cast<const f32x4*>(src + 32 * b);
      *reinterpret_cast<f32x4*>(&v[4]) = *reinterpret_cast<const f32x4*>(src + 32 * b + 4);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = src[32 * b + i];
    }
    f16x8 hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float w = ldexpf(v[i], e);
      hi[i] = static_cast<_Float16>(w);
      lo[i] = static_cast<_Float16>(w - static_cast<float>(hi[i]));
    }
    uint8_t* d = dst + static_cast<long long>(b) * kStepBytes;
    *reinterpret_cast<f16x8*>(d) = hi;
    *reinterpret_cast<f16x8*>(d + 1024) = lo;
  }
}

// y[o] = sum over the K ranges of partial, in index order.
__global__ __launch_bounds__(256) void wide_reduce(const float* __restrict__ partial,
                                                   float* __restrict__ y, long long count, int ks) {
  for (long long o = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; o < count;
       o += static_cast<long long>(gridDim.x) * 256) {
    float sum = 0.0f;
    for (int q0 = 0; q0 < ks; q0 += 4) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = partial[static_cast<long long>(min(q0 + j, ks - 1)) * count + o];
      sum = q0 == 0 ? v[0] : sum + v[0];
#pragma unroll
      for (int j = 1; j < 4; ++j)
        if (q0 + j < ks) sum += v[j];
    }
    y[o] = sum;
  }
}

// Tile of TM x TN 32 x 32 MFMA tiles per wave, WGM x WGN waves.
template <int FMT, int TM, int TN, int WGM, int WGN, int XR>
struct Wide {
  static constexpr int NW = WGM * WGN;
  static constexpr int BM = 32 * TM * WGM, BN = 32 * TN * WGN;
  static constexpr int PB = FMT == kQ8_0 ? 68 : 36;           // bytes of a row's block pair
  static constexpr int CH = PB / 16;                          // its whole 16-byte chunks
  static constexpr int XS = BM / 32 * kStepBytes;             // x bytes per block step
  static constexpr int XL = XS / 1024 / NW;                   // x loads per wave per step
  static constexpr int RPL = 64 / CH;                         // weight rows per chunk load
  static constexpr int WC = BN / RPL / NW;                    // chunk loads per wave per pair
  static constexpr int WL = WC + 1;                           // and one of last dwords
  static constexpr int WX = BN * CH * 16;                     // byte offset of the last dwords
  static constexpr int WS = WX + 4 * BN;                      // weight bytes per pair
  static_assert(BN % (RPL * NW) == 0 && BN % 64 == 0, "whole weight loads");
  static constexpr int WR = (XR + 1) / 2;                     // weight pairs in the ring
  static constexpr int lds = XR * XS + WR * WS;
  static_assert(XR % 2 == 1 && XR >= 3, "x steps in the ring");
  static_assert((XR - 2) * XL + WR * WL < 64, "vmcnt range");
  static_assert(XS % (1024 * NW) == 0, "whole x loads");
  static_assert(lds <= 160 * 1024, "LDS");
};

template <int FMT, int TM, int TN, int WGM, int WGN, int XR>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void wide_gemm(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ xf, float* __restrict__ y,
    float* __restrict__ partial, const int* __restrict__ rexp, const float* __restrict__ x, int M,
    int N, int K, int mblocks, int nblocks, int pairs_per_split, int ks_count) {
  using C = Wide<FMT, TM, TN, WGM, WGN, XR>;
  constexpr int WR = C::WR;
  constexpr int PB = C::PB, CH = C::CH, RPL = C::RPL;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[C::lds];
  uint8_t* const xring = lds;
  uint8_t* const wring = lds + XR * C::XS;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WGM, wn = wave / WGM;
  const int col = lane & 31, half = lane >> 5;

  int mb, nbk, ks;
  tile_of_workgroup(mblocks, nblocks, ks_count, mb, nbk, ks);
  const int n0 = nbk * C::BN;
  const int mt0 = mb * (C::BM / 32);
  const int nb = K / 32, npairs = K / 64;
  const int p0 = ks * pairs_per_split;
  const int p1 = min(p0 + pairs_per_split, npairs);
  const long long row_bytes = static_cast<long long>(npairs) * PB;

  // Sources advance by one step / pair per issue and stop at the last one.
  // x chunk q = wave * XL + i (1 KB) of a step: m-tile q / 4, slot q % 4.
  const int steps = 2 * (p1 - p0);
  static_assert(C::XL <= 4 ? 4 % C::XL == 0 : C::XL % 4 == 0, "x loads");
  const uint8_t* xsrc =
      uniform_ptr(xf + (static_cast<long long>(mt0 + (wave * C::XL >> 2)) * nb + 2 * p0) * kStepBytes +
                  (wave * C::XL & 3) * 1024);
  int xleft = __builtin_amdgcn_readfirstlane(steps - 1);
  auto issue_x1 = [&](int slot, int i) {
    dma16(xsrc + (i >> 2) * static_cast<long long>(nb) * kStepBytes + (i & 3) * 1024,
          16 * lane, xring + slot * C::XS + (wave * C::XL + i) * 1024);
  };
  auto next_x = [&]() {
    xsrc += xleft > 0 ? kStepBytes : 0;
    --xleft;
  };
  // Weights: load i of a wave covers RPL rows, CH lanes a row; the chunk c of
  // row r is stored at position c ^ key(r), so that eight consecutive rows'
  // 16-byte reads fall on distinct banks.  The dword past the whole chunks
  // is gathered for 64 rows at once, behind all chunks (workgroups with more
  // waves than that takes write some of them twice, the same bytes).
  const uint8_t* wsrc = uniform_ptr(W + static_cast<long long>(n0) * row_bytes +
                                    static_cast<long long>(p0) * PB);
  int wleft = __builtin_amdgcn_readfirstlane(p1 - p0 - 1);
  auto key = [](int r) { return CH == 4 ? (r >> 2) & 3 : (r >> 3) & 1; };
  uint32_t woff[C::WC], xoff;
#pragma unroll
  for (int i = 0; i < C::WC; ++i) {
    const int r = RPL * (wave * C::WC + i) + lane / CH;
    woff[i] = static_cast<uint32_t>(min(n0 + r, N - 1) - n0) * static_cast<uint32_t>(row_bytes) +
              16 * ((lane % CH) ^ key(r));
  }
  constexpr int XG = C::BN / 64;                   // gathers of last dwords
  xoff = static_cast<uint32_t>(min(n0 + 64 * (wave % XG) + lane, N - 1) - n0) *
             static_cast<uint32_t>(row_bytes) + 16 * CH;
  auto issue_w1 = [&](int slot, int i) {
    uint8_t* base = wring + slot * C::WS;
    if (i < C::WC) dma16(wsrc, woff[i < C::WC ? i : 0], base + 1024 * (wave * C::WC + i));
    else dma4(wsrc, xoff, base + C::WX + 256 * (wave % XG));
  };
  auto next_w = [&]() {
    wsrc += wleft > 0 ? PB : 0;
    --wleft;
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  // The operands of one block and n-tile: codes as f16 and the block scale;
  // and the dwords they are decoded from.
  struct Weights {
    f16x8 w[2];
    float d;
  };
  struct Raw {
    u32x4 c;
    uint32_t x, d;
  };
  // This lane's bytes of a row (n-tile 0; n-tiles and waves are whole
  // multiples of 32 rows, which keep the key): chunk c is at chunk0 ^ 16 c.
  // Block 0 is chunk (q8_0: half; q4_0: 0) and the next one's first dword;
  // block 1 q8_0 chunk 2 + half from its second dword on and the first dword
  // of chunk 3 or the last dword, q4_0 chunk 1 and the last dword.  The offsets
  // are formed at each read: held, they would cost registers that spill.
  const int row0 = wn * 32 * TN + col;
  const int chunk0 = 16 * (CH * row0 + key(row0)), last0 = C::WX + 4 * row0;
  auto read_raw = [&](int slot, int h, int tn, Raw& o) {
    const uint8_t* sw = wring + slot * C::WS;
    const int t0 = tn * 16 * CH * 32;
    int at = chunk0;
    asm volatile("" : "+v"(at));
    const int hs = FMT == kQ8_0 ? 16 * half : 0;
    const int c = (at ^ hs) ^ (h == 0 ? 0 : FMT == kQ8_0 ? 32 : 16);
    const int d = at ^ (h == 0 ? 0 : FMT == kQ8_0 ? 32 : 16);
    int x = at ^ (16 + hs);
    int xt = t0;
    if (h == 1) {
      const bool last = FMT != kQ8_0 || half == 1;
      x = last ? last0 + 128 * tn : (at ^ 48) + t0;
      xt = 0;
    }
    o.c = *reinterpret_cast<const u32x4*>(sw + c + t0);
    o.x = *reinterpret_cast<const uint32_t*>(sw + x + xt);
    if constexpr (FMT == kQ8_0) o.d = *reinterpret_cast<const uint32_t*>(sw + d + t0);
    else o.d = o.c[0];
  };
  // dword i (four codes)
  auto decode1 = [&](const Raw& o, int h, int i, Weights& w) {
    const uint32_t nx = i < 3 ? o.c[i < 3 ? i + 1 : 0] : o.x;
    uint32_t c = h == 0 ? __builtin_amdgcn_alignbyte(nx, o.c[i], 2) : nx;
    if constexpr (FMT == kQ8_0) c ^= 0x80808080u;
    else c = (c >> (4 * half)) & 0x0F0F0F0Fu;
    constexpr float off = FMT == kQ8_0 ? 1152.0f : 1032.0f;
    const f16x2 k = f16x2{static_cast<_Float16>(off), static_cast<_Float16>(off)};
    const f16x2 a = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c, 0x04010400u)) - k;
    const f16x2 b = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c, 0x04030402u)) - k;
    f16x8& v = w.w[i >> 1];
    const int e = 4 * (i & 1);
    v[e] = a[0];
    v[e + 1] = a[1];
    v[e + 2] = b[0];
    v[e + 3] = b[1];
    if (i == 3) {
      float f = half_bits_to_float(h == 0 ? o.d & 0xFFFFu : o.d >> 16);
      asm("" : "+v"(f));                           // keep the fold a plain f32 FMA
      w.d = f;
    }
  };

  if (steps > 0) {
    // Barrier B_s stands before the last m-tile of step s.  Step s issues,
    // before B_s, x step s + XR - 1 and (s odd) weight pair (s - 1) / 2 + WR;
    // at B_s only the loads of the last XR - 2 steps may be outstanding, so x
    // step s + 1 and the weights of block s + 2 are in.  With one m-tile B_s
    // opens step s, whose loads follow it (into x slot s - 1, last read before
    // B_{s-1}): the loads of the last XR - 3 steps may then be outstanding.
    auto load_w = [&](int slot) {
#pragma unroll
      for (int i = 0; i < C::WL; ++i) issue_w1(slot, i);
      next_w();
    };
    load_w(0);
#pragma unroll
    for (int r = 0; r < XR - 1; ++r) {
#pragma unroll
      for (int i = 0; i < C::XL; ++i) issue_x1(r, i);
      next_x();
      if (r % 2 == 1) load_w((r + 1) / 2);
    }
    wait_vmcnt<(XR - 2) * C::XL + (WR - 1) * C::WL>();   // W(0), x(0)
    ring_barrier();
    // The operands of n-tiles 0 .. NE - 1 are decoded a step ahead (two
    // buffers); with TN > 1 those of the last n-tile at the start of their
    // own step, while n-tile 0 is multiplied (one buffer).
    constexpr int NE = TN > 1 ? TN - 1 : 1;
    Weights we[2][NE], wl;
    constexpr int RL = TN > 1 && TM * TN < 8 ? 1 : 0;   // raw dwords of the last n-tile
    static_assert(TN <= 2, "one early n-tile per set of raw dwords");
    Raw raw[RL + 1];
#pragma unroll
    for (int tn = 0; tn < NE; ++tn) {
      read_raw(0, 0, tn, raw[0]);
#pragma unroll
      for (int i = 0; i < 4; ++i) decode1(raw[0], 0, i, we[0][tn]);
    }
    if (TN > 1) read_raw(0, 0, TN - 1, raw[RL]);
    f16x8 ae[2][2], al[2];                         // operands 0, 1 (two buffers) and 2, 3
    const uint8_t* const xw = xring + wm * TM * kStepBytes + 16 * lane;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      ae[0][q] = *reinterpret_cast<const f16x8*>(xw + q * 1024);
      al[q] = *reinterpret_cast<const f16x8*>(xw + 2048 + q * 1024);
    }
    wait_lgkmcnt0();
    f32x16 c[2];
    float dprev = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) c[1][e] = 0.f;
    int xs = 0, ws = 0;                            // slots of the current step and pair

    auto step = [&](auto odd) {
      constexpr bool kOdd = decltype(odd)::value;
      constexpr int T = TM * TN, B = (TM - 1) * TN;   // tiles; the one B_s comes before
      constexpr int kGap = TN > 1 ? TN - 1 : 1;
      // loads of window s - 1 issued in this step, before B_s (the first
      // ones went out after B_{s-1})
      constexpr int NL = C::XL + (kOdd ? C::WL : 0);
      const int xn = xs + 1 < XR ? xs + 1 : 0, xp = xs > 0 ? xs - 1 : XR - 1;
      const int wn1 = ws + 1 < WR ? ws + 1 : 0;
      auto issue = [&](int l) {
        if (l < C::XL) issue_x1(xp, l);
        else issue_w1(ws, l - C::XL);
      };
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const int tm = i / TN, tn = i % TN;
        const Weights& cur = tn < NE ? we[kOdd ? 1 : 0][tn < NE ? tn : 0] : wl;
        const int ab = ((kOdd ? TM : 0) + tm) & 1;     // operand buffer of this m-tile
        const int pi = i == 0 ? T - 1 : i - 1, pm = pi / TN, pn = pi % TN;
        const int cb = ((kOdd ? T : 0) + i) & 1;       // result buffer
        if (i == B) {
          if constexpr (B > 0)
            wait_vmcnt<(XR - 2) * C::XL + (kOdd ? XR - 1 : XR - 3) / 2 * C::WL>();
          else                                     // this step's loads go out after B_s
            wait_vmcnt<(XR - 3) * C::XL + (XR - 3) / 2 * C::WL>();
          wait_lgkmcnt0();
          ring_barrier();
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16 z = {};
          // the last n-tile takes operands 2, 3 first: they are then free
          // for the next m-tile's
          const int o = TN > 1 && tn == TN - 1 ? q ^ 2 : q;
          c[cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o < 2 ? ae[ab][o & 1] : al[o & 1],
                                                         cur.w[o >> 1], q == 0 ? z : c[cb], 0, 0, 0);
          // the previous tile's last MFMA is still running in slot 0
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int e = q == 0 ? 0 : 16 * (q - 1) / 3; e < 16 * q / 3; ++e)
            acc[pm][pn][e] = fmaf(c[cb ^ 1][e], dprev, acc[pm][pn][e]);
          const int ms = 4 * tn + q, slot = 4 * i + q;
          // the next m-tile's operands: 0 and 1 early, 2 and 3 after their last use
          const uint8_t* nx = tm + 1 < TM ? xw + xs * C::XS + (tm + 1) * kStepBytes
                                          : xw + xn * C::XS;
          if (ms == TN - 1 || ms == 2 * TN - 1)
            ae[ab ^ 1][ms / TN] = *reinterpret_cast<const f16x8*>(nx + ms / TN * 1024);
          if (tn == TN - 1 && o >= 2)
            al[o & 1] = *reinterpret_cast<const f16x8*>(nx + o * 1024);
          constexpr int kIssue = 4 * (B > 0 ? B : T);    // slots that issue loads
          if (slot < kIssue) {
#pragma unroll
            for (int l = slot * NL / kIssue; l < (slot + 1) * NL / kIssue; ++l) issue(l);
          }
          // weights: read n-tile by n-tile (well before B_s, which waits for
          // LDS reads), decoded a dword at a time
          if (TN > 1 && i == 0) decode1(raw[RL], kOdd ? 1 : 0, q, wl);
#pragma unroll
          for (int u = 0; u < TN; ++u) {
            // two sets of raw dwords: both reads early; one: in turn
            const int at = TN == 1 ? 0 : RL == 1 ? (u < NE ? u : 4) : 4 + u * (2 * B - 1) / kGap;
            const int len = TN == 1 ? 4 * T - 1 : RL == 1 ? 8 : (2 * B - 1) / kGap;
            if (slot == at) read_raw(kOdd ? wn1 : ws, kOdd ? 0 : 1, u, raw[u < NE ? 0 : RL]);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (u < NE && slot == at + 3 + j * (len - 3) / 4)
                decode1(raw[0], kOdd ? 0 : 1, j, we[kOdd ? 0 : 1][u < NE ? u : 0]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        dprev = cur.d;
      }
      xs = xn;
      next_x();
      if constexpr (kOdd) {
        next_w();
        ws = wn1;
      }
    };
    for (int s = 0; s < steps; s += 2) {
      step(std::integral_constant<bool, false>());
      step(std::integral_constant<bool, true>());
    }
#pragma unroll
    for (int e = 0; e < 16; ++e)
      acc[TM - 1][TN - 1][e] = fmaf(c[1][e], dprev, acc[TM - 1][TN - 1][e]);
  }
  wait_vmcnt<0>();   // no global->LDS load may outlive the workgroup's LDS

  store_tiles<TM, TN>(acc, rexp, ks_count > 2 ? partial + static_cast<long long>(ks) * M * N : y, N,
                      ks_count == 2, 32 * (mt0 + wm * TM), n0 + 32 * wn * TN, M, N, [&](int m, int n) {
                        return nonfinite_blocks_f32<FMT>(W + static_cast<long long>(n) * row_bytes,
                                                         x + static_cast<long long>(m) * K, 2 * p0, 2 * p1);
                      });
}

// Times per block pair, measured on MI355X with q8_0 at K = 4096 (q4_0 within
// 10%): 256 x 256 tiles 182 us for 112 workgroups, 467 for 448; 128 x 256
// 129 us for 224, 538 for 896; 128 x 128 145 us for 448; 64 x 128 30 us for
// 128 half-K workgroups.  Up to 32 rows take the last tile alone (q4_0,
// K = 14336: 98 us for 16 workgroups, 111 for 224): a workgroup more than there
// are CUs costs a round (two share a CU's operand feed), and its ring is nine
// steps deep, because a step is only one MFMA tile (N = 14336, K = 4096, two K
// ranges: 25.7 us with seven steps, 24.4 with nine, 25.5 with fifteen).  It may
// take up to 24 K ranges: with few columns and long K eight leave most CUs
// idle (M = 17, K = 14336, N = 64 / 256 / 2048 23.2 / 23.6 / 24.9 us with eight,
// 18.7 / 19.3 / 21.5 with more; bf16 passes 19.5 / 20.5 / 24.4).
constexpr int kTiles = 4;   // for more than 32 rows
constexpr Tile kTile[kTiles + 1] = {{256, 256, 1, 2.84, 4.10},
                                {128, 256, 1, 1.70, 2.30},
                                    {128, 128, 2, 1.10, 2.44},
                                    {64, 128, 1, 0.48, 0.68},
                                    {32, 128, 1, 0.42, 0.48}};

template <int FMT, int TM, int TN, int WGM, int WGN, int XR>
hipError_t launch_tile(const uint8_t* W, const uint8_t* xf, float* y, float* partial,
                       const int* rexp, const float* x, int m, int n, int k, const TilePlan& p,
                       hipStream_t s) {
  using C = Wide<FMT, TM, TN, WGM, WGN, XR>;
  const int mblocks = (m + C::BM - 1) / C::BM, nblocks = (n + C::BN - 1) / C::BN;
  wide_gemm<FMT, TM, TN, WGM, WGN, XR><<<static_cast<unsigned>(mblocks) * nblocks * p.ks, 64 * C::NW, 0, s>>>(
      W, xf, y, partial, rexp, x, m, n, k, mblocks, nblocks, p.per, p.ks);
  return hipGetLastError();
}

template <int FMT>
hipError_t run_wide(const uint8_t* W, const float* x, float* y, int m, int n, int k, int ranges,
                    hipStream_t s, Scratch& scratch) {
  const int nb = k / 32;
  const int mtiles = m <= 32 ? 1 : (m + 255) / 256 * 8;
  const size_t xf_bytes = static_cast<size_t>(mtiles) * nb * kStepBytes;
  const double left = scratch.w != nullptr ? 256e6
                                           : static_cast<double>(scratch.fixed_bytes) -
                                                 static_cast<double>(scratch.fixed_split + xf_bytes);
  const int cus = device_cu_count();
  TilePlan p = m <= 32 ? plan_tiles(&kTile[kTiles], 1, m, n, k / 64, cus, ranges, 24, left)
                       : plan_tiles(kTile, kTiles, m, n, k / 64, cus, ranges, 8, left);
  if (m <= 32) p.tile = kTiles;
  const long long outs = static_cast<long long>(m) * n;
  const size_t part_bytes = p.ks > 2 ? static_cast<size_t>(p.ks) * outs * sizeof(float) : 0;
  void* buf = nullptr;
  hipError_t e = scratch.get(s, xf_bytes + part_bytes, &buf);
  if (e != hipSuccess) return e;
  uint8_t* xf = static_cast<uint8_t*>(buf);
  float* partial = reinterpret_cast<float*>(xf + xf_bytes);
  // read in whole tiles: padded to the largest
  e = scratch.get(s, sizeof(int) * 32 * static_cast<size_t>(mtiles), &buf, 1);
  if (e != hipSuccess) return e;
  int* rexp = static_cast<int*>(buf);

  // eight rows a workgroup, K in as many slices as give ~512 workgroups of
  // at least 16 blocks (one per lane pair of a workgroup's waves)
  const int groups = (m + 7) / 8;
  const int want = std::max(1, std::min((nb + 15) / 16, 512 / groups));
  const int per_slice = (nb + want - 1) / want;
  const int slices = (nb + per_slice - 1) / per_slice;
  const int clear = p.ks == 2 ? static_cast<int>(std::max<long long>(
                                    1, std::min<long long>(512, outs / 8192) / slices))
                              : 0;
  wide_prep<<<dim3(groups + clear, slices), 512, 0, s>>>(x, m, k, per_slice, xf, rexp, y,
                                                         p.ks == 2 ? outs : 0);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  switch (p.tile) {
    case 0: e = launch_tile<FMT, 4, 2, 2, 4, 3>(W, xf, y, partial, rexp, x, m, n, k, p, s); break;
    case 1: e = launch_tile<FMT, 2, 2, 2, 4, 3>(W, xf, y, partial, rexp, x, m, n, k, p, s); break;
    case 2: e = launch_tile<FMT, 2, 2, 2, 2, 3>(W, xf, y, partial, rexp, x, m, n, k, p, s); break;
    case 3: e = launch_tile<FMT, 2, 1, 1, 4, 5>(W, xf, y, partial, rexp, x, m, n, k, p, s); break;
    default: e = launch_tile<FMT, 1, 1, 1, 4, 9>(W, xf, y, partial, rexp, x, m, n, k, p, s); break;
  }
  if (e != hipSuccess || p.ks <= 2) return e;
  wide_reduce<<<static_cast<unsigned>(std::min<long long>(4096, (outs + 255) / 256)), 256, 0, s>>>(
      partial, y, outs, p.ks);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_qgemm_wide(int fmt, const void* W, const float* x, float* y, int m, int n, int k,
                             int ranges, hipStream_t s, Scratch& scratch) {
  const auto* w = static_cast<const uint8_t*>(W);
  if (fmt == kQ4_0 && ranges == 0 && mx_pays(m, n, k)) return launch_qgemm_mx(W, x, y, m, n, k, s, scratch.w);
  // Rows in chunks whose fragments (4 bytes an element) take at most 256 MB.
  const long long fit = (256LL << 20) / (4LL * k) / 256 * 256;
  const int chunk = static_cast<int>(std::max<long long>(256, std::min<long long>(fit, INT_MAX / 2)));
  for (int m0 = 0; m0 < m; m0 += chunk) {
    const int mc = std::min(chunk, m - m0);
    const float* xm = x + static_cast<long long>(m0) * k;
    float* ym = y + static_cast<long long>(m0) * n;
    const hipError_t e = fmt == kQ8_0 ? run_wide<kQ8_0>(w, xm, ym, mc, n, k, ranges, s, scratch)
                                      : run_wide<kQ4_0>(w, xm, ym, mc, n, k, ranges, s, scratch);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace qc
