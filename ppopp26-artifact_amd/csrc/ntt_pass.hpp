// NTT pass kernel template (included by the per-radix translation units).
// NTT / iNTT passes for gfx950.
//
// Algorithm: four-step (Bailey) decimation in frequency, applied recursively.
// A size-N transform, N = 2^lg, is split into passes of M' = 2^m points
// (3 <= m <= 6).  With N = N1*N2, j = j1 + N1*j2, k = k2 + N2*k1:
//
//   X[k2 + N2 k1] = sum_j1 w_N1^(j1 k1) * ( w_N^(j1 k2) * sum_j2 x[j1 + N1 j2] w_N2^(j2 k2) )
//
// Pass 1 does the inner column DFTs (size N2 = 2^m, stride N1) and the twiddle
// w_N^(j1 k2), in place; the rows of length N1 that remain are contiguous and
// are split the same way by the next pass.  The last pass transforms
// contiguous sub-rows and writes each result straight to its digit-reversed
// (natural-order) position, so no separate permutation pass exists.  This
// replaces the reference's host bit-reversal plus sppark-style CT passes
// (ntt.cu:979-1037; ntt_kernel/algorithm.cuh:8-59; ct_mixed_radix_wide.cuh:47-189)
// with the same mathematical result.
//
// Workgroup: A waves own a tile of 64 adjacent columns of M' = 8 A points,
// one column per lane, 8 elements of it in VGPRs (about 110-128 VGPRs per
// lane, so four waves share each SIMD: one wave alone cannot issue
// multiply-adds back to back, and four reach ~15 % more than two).  A column
// is computed as DFT_8 over rho2 (wave rho1), an inner twiddle
// w_M'^(rho1 k2), one exchange through LDS (48 KiB per workgroup for A = 8,
// in three rounds), then DFT_A over rho1 (wave k2).  With one column per lane
// everything that varies inside a column is the same for the whole wave: the
// factors inside the DFTs and the inner twiddles come as pre-reduced rows in
// SGPRs (rows29, fr29.hpp), 107-117 VALU instructions per product instead of
// 196 and an unpack (13 x iNTT 2^15: 67.6 -> 56.5 us; proof batch of 2^12 ..
// 2^20: 2.98 -> 2.64 ms; the per-lane twiddles of a 16-column tile of two
// waves before).  Longer tiles leave two workgroups of eight waves on a CU,
// so loads and stores hide less behind the other's products than with eight
// of two: 2^24, a middle pass, 0.42 -> 0.32 ms with 757 -> 519 VALU
// instructions per element (plain digits, below, included).  Loading the next tile's words into the registers
// that the results leave (a workgroup looping over 2 .. 16 tiles) was slower
// (2^24: 1.32 -> 1.42 ms): the passes wait for VALU issue and for memory, not
// for single loads.
// Global accesses move 64 * 32 contiguous bytes, the last pass's loads whole
// sub-rows.  Between passes the data is held as 256-bit words of the class
// mod r, not reduced; the last pass writes canonical values in [0, r).
//
// Elements are plain digits in [0, 2^29) (a signed top) from load to
// exchange to store, factors balanced ones: a digit taken plain is a
// two-operand and (1.1 ns per wave and SIMD at four waves), taken balanced a
// three-operand bit-field extract (1.9) and a multiply-add that rounds its
// column (2.0).  2^24: 1.317 -> 1.281 ms, 2^22: 0.340 -> 0.327, 2^20: 102.6 ->
// 97.2 us with balanced digits before.
#pragma once
#include <type_traits>

#include "fr29.hpp"
#include "pl_internal.hpp"

namespace pl {

// w_16^e and w_16^-e, e = 0..7, as w R' mod r (R' = 2^261) in balanced
// digits (b_i in [-2^28, 2^28), sum b_i 2^(29 i)); domain_build derives the
// in-register DFTs' factors (PassArgs::rows) from e = 2, 4, 6
static __constant__ const uint32_t kW16b[2][8][9] = {
    {{0xffffffbau, 0x00000230u, 0xfcb61180u, 0x0a4e5c01u, 0x0ee8b1a2u, 0xf6e6aedfu, 0xf907f8bcu, 0x0853ddf8u, 0x004d043fu},
     {0x04056c96u, 0x0f64e4d8u, 0xfc1c7b56u, 0xfcbda468u, 0xf4e761dbu, 0xf28ae057u, 0xfd2f3145u, 0x0f463b6eu, 0x006dc1feu},
     {0x085dfee9u, 0x0f4995e4u, 0xf941c136u, 0x0b284958u, 0xfc313523u, 0xff28f6a6u, 0x07ad921eu, 0x0d72d344u, 0x002ca644u},
     {0xf81392abu, 0xf40c77eeu, 0x0175e03eu, 0x09f5a4e3u, 0x0f090202u, 0x0c6252cbu, 0xfc504ed8u, 0x038e921cu, 0x00408014u},
     {0xf139f60bu, 0xf0567553u, 0xfe6cfcdeu, 0x03679a02u, 0x08c51075u, 0xff9df144u, 0xfeb67e0cu, 0xfa6828a5u, 0x00231dc7u},
     {0x0142510bu, 0x02a002b3u, 0x09a9466eu, 0xff776142u, 0x002a3050u, 0xf0591c89u, 0x04f2cdf4u, 0x0d6e4f9eu, 0x006990bbu},
     {0xf6551b88u, 0xff9842ffu, 0x0f9a0689u, 0xfb208bceu, 0xfe704152u, 0x09d87034u, 0xfd460dfbu, 0x063990acu, 0x0050578fu},
     {0xf7ddaa4du, 0xfd2e4775u, 0x06b5ad2fu, 0xf9075af7u, 0x06ef6bbeu, 0xf25fb8efu, 0x07ff9caeu, 0xf5571281u, 0x00687c14u}},
    {{0xffffffbau, 0x00000230u, 0xfcb61180u, 0x0a4e5c01u, 0x0ee8b1a2u, 0xf6e6aedfu, 0xf907f8bcu, 0x0853ddf8u, 0x004d043fu},
     {0x082255b4u, 0x02d1b883u, 0xf8e15291u, 0x0240ab09u, 0xf690e97eu, 0xf9a44be2u, 0x0d21303au, 0xf50e212eu, 0x000b7194u},
     {0x09aae479u, 0x0067bcf9u, 0x0ffcf937u, 0x00277a31u, 0xff1013eau, 0x022b949du, 0xf7dabeecu, 0x042ba304u, 0x00239618u},
     {0xfebdaef6u, 0xfd5ffd45u, 0xf5edb952u, 0xfbd0a4beu, 0xfd5624ecu, 0xfbaae848u, 0xf02dfef4u, 0xfcf6e412u, 0x000a5cecu},
     {0x0ec609f6u, 0x0fa98aa5u, 0x012a02e2u, 0xf7e06bfeu, 0xf4bb44c7u, 0x0c66138du, 0xf66a4edbu, 0x0ffd0b0bu, 0x0050cfe0u},
     {0x07ec6d56u, 0x0bf3880au, 0xfe211f82u, 0xf152611du, 0x0e77533au, 0xffa1b205u, 0xf8d07e0fu, 0x06d6a194u, 0x00336d93u},
     {0xf7a20118u, 0xf0b66a14u, 0x06553e8au, 0xf01fbca8u, 0x014f2019u, 0x0cdb0e2bu, 0x0d733ac9u, 0xfcf2606bu, 0x00474763u},
     {0xfbfa936bu, 0xf09b1b20u, 0x037a846au, 0xfe8a6198u, 0x0898f361u, 0xf979247au, 0xf7f19ba3u, 0xfb1ef842u, 0x00062ba9u}}};

// an ordering point for the eight limbs of v (no instruction)
__device__ __forceinline__ void pin(fr& v) {
  asm volatile("" : "+v"(v.l[0]), "+v"(v.l[1]), "+v"(v.l[2]), "+v"(v.l[3]), "+v"(v.l[4]), "+v"(v.l[5]),
               "+v"(v.l[6]), "+v"(v.l[7]));
}

// global memory operations stay on their side of this point, as do asm blocks
__device__ __forceinline__ void mem_here() { __builtin_amdgcn_sched_barrier(0x0002 | 0x0004 | 0x0080); }

__host__ __device__ constexpr int brev(int v, int bits) {
  int r = 0;
  for (int i = 0; i < bits; i++) r |= ((v >> i) & 1) << (bits - 1 - i);
  return r;
}

// The pass kernels' wave-uniform factors, as rows29 tables of 81 words each
// (PassArgs::rows): i = w_8^2, (w_8 + w_8^3) / 2 and (w_8 - w_8^3) / 2 for the
// in-register DFTs (D = 1), then w_64^e, e < 64, for the inner twiddles
// (D = 2); inverse transforms: of w_8^-1 and w_64^-1.
enum { kDftI = 0, kDftC1 = 1, kDftC2 = 2, kInner = 3, kRowFactors = 3 + 64 };
constexpr int kRowWords = 81;

// DFT of size 2^LOGB (at most 8) on x[OFF + i], natural order in, bit-reversed
// order out: afterwards x[OFF + brev(k)] = X[k].  The odd outputs of the DFT_8
// need w d1 + w^3 d3 and w^3 d1 + w d3 (w = w_8): as A + B and A - B with
// A = (w + w^3)/2 (d1 + d3), B = (w - w^3)/2 (d1 - d3) they take two products
// where the radix-2 network takes three, four in all instead of five.  Every
// factor is wave-uniform, so the products are rows29 (fr29.hpp) with one
// Montgomery digit: about 107 VALU instructions against mont29's 196.
// NTT 2^24: 1.64 -> 1.43 ms; 2^16: 46 -> 43.7 us (a lone wave per SIMD).
//
// Bounds, with input limbs plain digits in [0, 2^29) (the top one signed and
// small) of values within V: sums of four lie in [0, 2^31) and differences of
// such within 2^31, so only y0, a sum of eight, leaves 32 bits (zero_bias
// brings it back); d = x_i - x_(i+4) has |l| < 2^29, e0, e1, d1 +- d3 < 2^30,
// the products' inputs; the products' limbs lie in [0, 2^29).  e0 +- i e1
// within 2^30 + 2^29; f = d0 +- i d2 within (-2^30, 2^30), so y1 = f + A + B
// within [-2^30, 2^31) and the others smaller.  Values: i d2 within 5.6 r,
// i e1, A, B within 10.2 r, so every output is within max(8 V, 2 V + 26 r).
template <int LOGB, int OFF, int NX>
__device__ __forceinline__ void dft_dif(v9 (&x)[NX], uwords f) {
  static_assert(LOGB <= 3, "limb growth: at most three butterfly levels");
  // one butterfly at a time: the empty asm statements order them, so the live
  // set stays at the lane's elements plus one butterfly's temporaries
  auto bfly = [](v9& a, v9& b) {
    pin9(a);
    pin9(b);
    const v9 s = v9_add(a, b);
    b = v9_sub(a, b);
    a = s;
    pin9(a);
    pin9(b);
  };
  // y0 back into signed limbs: a sum of eight plain digits lies in [0, 2^32),
  // and adding -2^31 to limb 0, 4 - 2^31 to the middle ones and 4 to limb 8
  // adds nothing (2^31 at limb i is 4 at limb i + 1)
  auto zero_bias = [](v9& a) {
    a.l[0] ^= 1u << 31;
#pragma unroll
    for (int i = 1; i < 8; i++) a.l[i] += 4u - (1u << 31);
    a.l[8] += 4;
    pin9(a);
  };
  // x times factor e; n is the next product's
  rows_cols g;
  if constexpr (LOGB >= 2) g = rows29_open(f + kRowWords * kDftI);
  auto mul = [&](v9& a, int e, int n) {
    a = v9_mul_rows<1, false>(a, f + kRowWords * e, g, f + kRowWords * n);
    pin9(a);
  };
  if constexpr (LOGB == 1) {
    bfly(x[OFF], x[OFF + 1]);
  } else if constexpr (LOGB == 2) {
    bfly(x[OFF], x[OFF + 2]);      // a0, d0
    bfly(x[OFF + 1], x[OFF + 3]);  // a1, d1
    mul(x[OFF + 3], kDftI, kDftI);  // i d1
    bfly(x[OFF], x[OFF + 1]);      // y0, y2
    bfly(x[OFF + 2], x[OFF + 3]);  // y1, y3
  } else if constexpr (LOGB == 3) {
    static_for<0, 4>([&](auto i_) { bfly(x[OFF + decltype(i_)::value], x[OFF + decltype(i_)::value + 4]); });
    bfly(x[OFF], x[OFF + 2]);      // b0, e0
    bfly(x[OFF + 1], x[OFF + 3]);  // b1, e1
    bfly(x[OFF], x[OFF + 1]);      // y0, y4
    zero_bias(x[OFF]);
    mul(x[OFF + 3], kDftI, kDftI);  // i e1
    bfly(x[OFF + 2], x[OFF + 3]);  // y2, y6
    mul(x[OFF + 6], kDftI, kDftC1);  // i d2
    bfly(x[OFF + 4], x[OFF + 6]);  // f+, f-
    bfly(x[OFF + 5], x[OFF + 7]);  // d1 + d3, d1 - d3
    mul(x[OFF + 5], kDftC1, kDftC2);  // A
    mul(x[OFF + 7], kDftC2, kDftI);   // B
    bfly(x[OFF + 5], x[OFF + 7]);  // A + B, A - B
    bfly(x[OFF + 4], x[OFF + 5]);  // y1, y5
    bfly(x[OFF + 6], x[OFF + 7]);  // y3, y7
  }
}

struct PassArgs {
  const fr* in;
  fr* out;
  const fr* premul;     // !LAST: optional factor per input element [(poly & pm_mask) << lgN | pos], pbd words of c R''
  const fr* tw;         // !LAST: pass twiddles (pbd words of w R' mod r), index j + S*k within the sub-problem
  const fr* inner;      // w_256^e (or w_256^-e), e < 256, stored form (small-size kernel)
  const uint32_t* rows; // rows29 tables of the wave-uniform factors (pass kernels)
  uint64_t in_pstride;  // element stride between input polys (0: shared input)
  uint64_t nlines;      // lines (columns) in this launch
  uint32_t pm_mask;
  uint32_t lgN;         // log2 poly size
  uint32_t lgMp;        // log2 sub-problem size of this pass
  uint32_t lgS;         // log2 column stride (0 in the last pass)
  uint32_t lgI;         // LAST: output interleave
  uint32_t ndig;        // LAST: number of earlier passes
  uint32_t do_scale;    // multiply every output by `scale` (single-pass transforms)
  uint32_t lgrad[PL_MAX_PASSES];  // LAST: log2 radices of the earlier passes, pass 1 first
  fr scale;             // stored form (small-size kernel)
  fr scale29;           // pbd word of scale R' mod r (pass kernels)
};

// Tile geometry (see the file header): passes have 2^m-point columns,
// m = kLgPerT + LA, LA <= kLgPerT.
constexpr int kLgPerT = 3;           // log2 elements per lane
constexpr int kPerT = 1 << kLgPerT;
constexpr int kLgLines = 6;          // log2 columns per workgroup, one per lane
constexpr int kLines = 1 << kLgLines;
constexpr int kWavesPerSimd = 4;     // that the register allocation must allow
constexpr int kPhases = 3;           // LDS exchange rounds
constexpr int kW = 9 / kPhases;      // limbs per exchange round
static_assert(kW == 3 && kW * kPhases == 9, "rounds of one uint3 cover the nine limbs");

// the limbs of one round
__device__ __forceinline__ uint3 pack_limbs(const uint32_t* v) { return make_uint3(v[0], v[1], v[2]); }
__device__ __forceinline__ void unpack_limbs(uint32_t* v, const uint3& q) {
  v[0] = q.x; v[1] = q.y; v[2] = q.z;
}

// One pass over columns of M' = 8*A points, A = 2^LA; blk = tile index.
//
// Arithmetic: the lane's elements are signed-limb values (v9).  The input,
// any 256-bit words (below 2.21 r), is split into plain digits, so each
// in-register DFT starts from such digits and its limbs stay within 32 bits;
// every product takes such limbs.  Value bounds: the first DFT's outputs are
// within 2 * 2.21 r + 26 r = 30.4 r; an inner-twiddle product lies in
// (-1.001 r, 0.001 r), and elements k2 = 0 and rho1 = 0, which have no inner
// twiddle, are reduced into [0, 1.01 r); so DFT_A's outputs are within
// 28.1 r, or 30.4 r without one.  The pass twiddle multiplies by at most
// r / 2^261 < 0.0142, so that mont29_word's product is a word in
// (0.06 r, 1.94 r).  The last pass reduces its outputs to [0, r).
// SCALE: multiply every output by a.scale29 (single-pass inverse transforms;
// a separate instance, so the other last-pass kernels keep no registers for it)
template <int LA, bool INV, bool LAST, bool SCALE>
__device__ __forceinline__ void ntt_pass_body(const PassArgs& a, const uint64_t blk) {
  static_assert(!SCALE || LAST, "the scale factor is applied by the last pass");
  constexpr int A = 1 << LA;
  constexpr int m = LA + kLgPerT;
  constexpr int F2 = kPerT / A;   // DFT_A groups per lane in sub-step 2
  typedef uint3 vec;
  // kW limbs of every tile element (the exchange), and in the last pass first
  // 16 bytes of every element (the loads)
  constexpr size_t kLdsBytes = LAST ? (size_t)16 << (kLgLines + m) : LA > 0 ? sizeof(vec) << (kLgLines + m) : 16;
  __shared__ uint4 lds_raw[kLdsBytes / 16];
  vec* const lds = (vec*)lds_raw;

  const int lc = threadIdx.x & (kLines - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> kLgLines);
  const uint64_t line_of = (blk << kLgLines) + lc;
  const uint32_t lgL = a.lgN - m;  // log2 lines per polynomial = log2(N / M')
  const uwords rows = (uwords)a.rows;

  // ---- sub-step 1: kPerT points of one (line, rho1), DFT over rho2 ----------
  // rho = rho1 + A*rho2
  const int rho1 = wv;
  v9 x[kPerT];
  // lanes beyond the launch's lines load its last line and store nothing
  const uint64_t line = line_of < a.nlines ? line_of : a.nlines - 1;
  if constexpr (LAST) {
    uint64_t poly, lp;
    if (a.lgI) {
      poly = line & ((1ull << a.lgI) - 1);
      lp = line >> a.lgI;
    } else {
      poly = line >> lgL;
      lp = line & ((1ull << lgL) - 1);
    }
    // the sub-problem whose outputs land at lp + (N/M')*k: undo the digit
    // reversal lp = d1 + M1*(d2 + M2*(...)) -> r = (((d1)*M2 + d2)*M3 + ...)
    uint64_t r = 0, q = lp;
    for (uint32_t p = 0; p < a.ndig; p++) {
      uint32_t lr = a.lgrad[p];
      r = (r << lr) | (q & ((1ull << lr) - 1));
      q >>= lr;
    }
    const uint64_t base = (uint64_t)(a.in + poly * a.in_pstride + (r << m));
    // Adjacent lines are far-apart sub-rows (their first digit differs), so a
    // lane reading its own line would touch 64 pages with every load.  The
    // waves read whole sub-rows instead (lane = element, line uniform for
    // A = 8) and the raw words change hands through LDS, one 16-byte half at a
    // time (64 KiB for A = 8); the XOR keeps both sides free of bank
    // conflicts.  Last pass of 2^24:
    // 0.333 -> 0.291 ms.
    uint4 raw[kPerT][2];
    const int i1 = lc & ((1 << m) - 1);
    static_for<0, kPerT>([&](auto q_) {
      constexpr int q = decltype(q_)::value;
      const int ll = LA == 3 ? wv * kPerT + q : (((wv * kPerT + q) << kLgLines) + lc) >> m;
      uint32_t lo, hi;
      if constexpr (LA == 3) {
        lo = __builtin_amdgcn_readlane((uint32_t)base, ll);
        hi = __builtin_amdgcn_readlane((uint32_t)(base >> 32), ll);
      } else {
        lo = __builtin_amdgcn_ds_bpermute(4 * ll, (uint32_t)base);
        hi = __builtin_amdgcn_ds_bpermute(4 * ll, (uint32_t)(base >> 32));
      }
      const uint4* src = (const uint4*)(((uint64_t)hi << 32) | lo) + 2 * i1;
      raw[q][0] = src[0];
      raw[q][1] = src[1];
    });
    static_for<0, 2>([&](auto h_) {
      constexpr int h = decltype(h_)::value;
      if constexpr (h > 0) __syncthreads();
      static_for<0, kPerT>([&](auto q_) {
        constexpr int q = decltype(q_)::value;
        const int ll = (((wv * kPerT + q) << kLgLines) + lc) >> m;
        lds_raw[(i1 << kLgLines) + (ll ^ (i1 & (kLines - 1)))] = raw[q][h];
      });
      __syncthreads();
      static_for<0, kPerT>([&](auto r2_) {
        constexpr int r2 = decltype(r2_)::value;
        const int i = rho1 + A * r2;
        raw[r2][h] = lds_raw[(i << kLgLines) + (lc ^ (i & (kLines - 1)))];
      });
    });
    if constexpr (LA > 0) __syncthreads();  // before the exchange below reuses the buffer
    static_for<0, kPerT>([&](auto r2_) {
      constexpr int r2 = decltype(r2_)::value;
      const uint4 l = raw[r2][0], u = raw[r2][1];
      const uint32_t w[8] = {l.x, l.y, l.z, l.w, u.x, u.y, u.z, u.w};
      split29(w, x[r2].l);
    });
  } else {
    const uint64_t poly = line >> lgL;
    const uint64_t lp = line & ((1ull << lgL) - 1);
    const uint64_t j = lp & ((1ull << a.lgS) - 1);
    const uint64_t rr = lp >> a.lgS;
    const uint64_t pos0 = (rr << a.lgMp) + j;
    const uint64_t estride = 1ull << a.lgS;
    const fr* src = a.in + poly * a.in_pstride;
    // plain digits of any 256-bit words: caller data (optionally times a
    // premultiplication factor) or a previous pass's
    if (a.premul) {
      const fr* pm = a.premul + ((uint64_t)(poly & a.pm_mask) << a.lgN) + pos0 + (uint64_t)rho1 * estride;
      const fr* sp = src + pos0 + (uint64_t)rho1 * estride;
      // factors are pbd words of c R' (the coset powers); the product with
      // plain output digits lies in (-r, 0.03 r) and leaves such
      // digits, as the DFT wants.  Elements and factors are asked for two
      // products ahead, one once half the lane's results are held: their
      // loads hide behind those products; addresses are opaque bases plus
      // wave-uniform offsets
      fr f[kPerT], v[kPerT];
      auto load = [&](auto k_) {
        constexpr int k = decltype(k_)::value;
        const fr* q = pm;
        const fr* d = sp;
        asm volatile("" : "+v"(q), "+v"(d));
        v[k] = fr_load(d + (uint64_t)(A * k) * estride);
        f[k] = fr_load(q + (uint64_t)(A * k) * estride);
        mem_here();
      };
      static_for<0, 2>(load);
      static_for<0, kPerT>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        constexpr int n = k < kPerT / 2 - 1 ? k + 2 : k + 1;
        if constexpr (n < kPerT && k != kPerT / 2 - 1) load(std::integral_constant<int, n>());
        v9 xx;
        split29(v[k].l, xx.l);
        uint32_t w[9];
        pbd_unpack(f[k].l, w);
        x[k] = v9_mul<false, false, false>(xx, w);
        pin9(x[k]);
      });
    } else {
      fr raw[kPerT];
      static_for<0, kPerT>([&](auto r2_) {
        constexpr int r2 = decltype(r2_)::value;
        raw[r2] = fr_load(src + pos0 + (uint64_t)(rho1 + A * r2) * estride);
      });
      static_for<0, kPerT>([&](auto r2_) {
        constexpr int r2 = decltype(r2_)::value;
        split29(raw[r2].l, x[r2].l);
      });
    }
  }
  dft_dif<kLgPerT, 0>(x, rows);  // x[brev3(k2)] = sum_rho2 z[rho1 + A rho2] w8^(rho2 k2)
  v9 (&y)[kPerT] = x;
  if constexpr (LA > 0) {
    // back to plain digits of small values, so that DFT_A again starts from
    // such: k2 = 0 and wave rho1 = 0 take no twiddle and are reduced (about 45
    // instructions)
    auto reduce = [&](v9& v) {
      v9 t0;
      reduce_below_2r(v.l, t0.l);
      v = t0;
      pin9(v);
    };
    reduce(x[0]);
    const uwords tw = rows + kRowWords * kInner;
    const int step = (kRowWords * rho1) << (6 - m);  // w_M'^rho1
    rows_cols g = rows29_open(tw + step);
    static_for<1, kPerT>([&](auto k2_) {
      constexpr int k2 = decltype(k2_)::value;
      v9& v = x[brev(k2, kLgPerT)];
      pin9(v);
      if (rho1 == 0) {
        reduce(v);
      } else {
        v = v9_mul_rows<2, false>(v, tw + step * k2, g, tw + step * (k2 < kPerT - 1 ? k2 + 1 : k2));
        pin9(v);
      }
    });
    // Exchange through LDS in kPhases rounds of kW limbs (3 rounds of 12 bytes,
    // 48 KiB for A = 8, so two workgroups = four waves per SIMD fit a CU).  A
    // lane only meets its own column's elements; consecutive lanes hit
    // consecutive slots.  Each round's gathered limbs go back into the
    // registers that round vacated: y lives in x (x[f*A + r1] afterwards).
    static_for<0, kPhases>([&](auto h_) {
      constexpr int h = decltype(h_)::value;
      uint32_t hv[kPerT][kW];
      static_for<0, kPerT>([&](auto k2_) {
        constexpr int k2 = decltype(k2_)::value;
#pragma unroll
        for (int w = 0; w < kW; w++) hv[k2][w] = x[brev(k2, kLgPerT)].l[kW * h + w];
      });
      if constexpr (h > 0) __syncthreads();  // previous round's reads done before overwrite
      static_for<0, kPerT>([&](auto k2_) {
        constexpr int k2 = decltype(k2_)::value;
        lds[((k2 * A + rho1) << kLgLines) + lc] = pack_limbs(hv[k2]);
      });
      __syncthreads();
      // sub-step 2 gathers: DFT_A over rho1 for F2 values of k2 of one line
      static_for<0, F2>([&](auto f_) {
        constexpr int f = decltype(f_)::value;
        static_for<0, A>([&](auto r1_) {
          constexpr int r1 = decltype(r1_)::value;
          unpack_limbs(&y[f * A + r1].l[kW * h], lds[(((wv * F2 + f) * A + r1) << kLgLines) + lc]);
        });
      });
    });
  }
  // no barrier follows: lanes of lines beyond the launch leave here
  if (line_of >= a.nlines) return;
  // fresh copies of the lane's position, so that sub-step 2's indices are not
  // shared with sub-step 1's and kept live across it
  uint64_t line2 = line_of;
  asm volatile("" : "+v"(line2));
  // last pass: the lane's output base, computed before DFT_A so that its
  // 64-bit temporaries are not live beside the eight results
  fr* base = nullptr;
  const uint32_t lgI = a.lgI;
  if constexpr (LAST) {
    uint64_t poly, lp;
    if (lgI) {
      poly = line2 & ((1ull << lgI) - 1);
      lp = line2 >> lgI;
    } else {
      poly = line2 >> lgL;
      lp = line2 & ((1ull << lgL) - 1);
    }
    fr* dst = a.out + ((poly >> lgI) << (a.lgN + lgI)) + (poly & ((1ull << lgI) - 1));
    base = dst + (lp << lgI);
    asm volatile("" : "+v"(base));
  }
  if constexpr (LA > 0) {
    static_for<0, F2>([&](auto f_) { dft_dif<LA, decltype(f_)::value * A>(y, rows); });
  }
  // y[f*A + brev_LA(k1)] = Z[k2 + kPerT*k1], k2 = wv*F2 + f (A = 1: y[brev(f)])

  if (LAST) {
    if constexpr (SCALE) {
      // single-pass inverse transforms: the factor 2^-lg, once per element
      uint32_t w[9];
      pbd_unpack(a.scale29.l, w);
      static_for<0, kPerT>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        pin9(y[i]);
        y[i] = v9_mul<false, false, false>(y[i], w);
      });
    }
    static_for<0, F2>([&](auto f_) {
      constexpr int f = decltype(f_)::value;
      const int k2 = wv * F2 + f;
      static_for<0, A>([&](auto k1_) {
        constexpr int k1 = decltype(k1_)::value;
        const uint64_t k = (uint64_t)(k2 + kPerT * k1);
        v9 v = y[LA > 0 ? f * A + brev(k1, LA) : brev(f, kLgPerT)];
        pin9(v);
        uint32_t tt[9];
        reduce_below_2r(v.l, tt);
        fr o;
        join29(tt, o.l);
        // the address from an opaque copy of the lane's base, so that the
        // eight addresses are not all computed ahead and held
        fr* d = base;
        asm volatile("" : "+v"(d));
        fr c = fr_reduce_once(o);
        pin(c);  // one element's reduction at a time
        fr_store(d + (k << (lgL + lgI)), c);
      });
    });
  } else {
    const uint64_t poly = line2 >> lgL;
    const uint64_t lp = line2 & ((1ull << lgL) - 1);
    const uint64_t j = lp & ((1ull << a.lgS) - 1);
    const uint64_t rr = lp >> a.lgS;
    fr* dst = a.out + (poly << a.lgN) + (rr << a.lgMp) + j;
    const fr* tw = a.tw + j;
    // Each twiddle is asked for one product ahead, before the result in
    // between is stored: memory operations complete in order, so a load issued
    // after a store would wait for it too (NTT 2^24 1.38 -> 1.33 ms by turns).
    // VALU instructions per busy cycle of the sequencers, where the multiply-add
    // probe reaches 7.65: the middle passes 7.0 and 7.2, pass 0 and the last,
    // nearer the memory rate, 6.1 and 5.8.
    auto row = [&](int i) { return (uint64_t)((wv * F2 + i / A) + kPerT * (i % A)) << a.lgS; };
    fr next = fr_load(tw + row(0));
    mem_here();
    static_for<0, kPerT>([&](auto i_) {
      constexpr int i = decltype(i_)::value, f = i / A, k1 = i % A;
      const fr cur = next;
      if constexpr (i + 1 < kPerT) {
        next = fr_load(tw + row(i + 1));
        mem_here();
      }
      v9 v = y[LA > 0 ? f * A + brev(k1, LA) : brev(f, kLgPerT)];
      pin9(v);
      uint32_t w[9];
      pbd_unpack(cur.l, w);
      fr_store(dst + row(i), v9_mul_word(v, w));
    });
  }
}


template <int LA, bool INV, bool LAST, bool SCALE>
__global__ void __launch_bounds__(kLines << LA, kWavesPerSimd) ntt_pass_kernel(PassArgs a) {
  ntt_pass_body<LA, INV, LAST, SCALE>(a, blockIdx.x);
}

// Ragged form: one launch runs the tiles of many polynomials of different
// sizes (one PassArgs per segment).  seg_block0[s] is segment s's first
// block, ascending; a block finds its segment by binary search (uniform
// scalar loads, a few steps for the tens of segments of a batch).
template <int LA, bool INV, bool LAST, bool SCALE>
__global__ void __launch_bounds__(kLines << LA, kWavesPerSimd)
    ntt_pass_ragged_kernel(const PassArgs* __restrict__ segs, const uint32_t* __restrict__ seg_block0,
                           uint32_t nsegs) {
  const uint32_t b = blockIdx.x;
  uint32_t lo = 0, hi = nsegs - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (seg_block0[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  // read the arguments in place; a private copy would put the dynamically
  // indexed lgrad[] in scratch
  const PassArgs& a = segs[lo];
  ntt_pass_body<LA, INV, LAST, SCALE>(a, b - seg_block0[lo]);
}

// Host launcher for one radix: LA = log2(column size) - kLgPerT.
template <int LA, bool INV, bool LAST, bool SCALE = false>
static void launch_pass(const PassArgs& a, hipStream_t s) {
  const uint64_t tiles = (a.nlines + kLines - 1) >> kLgLines;
  hipLaunchKernelGGL((ntt_pass_kernel<LA, INV, LAST, SCALE>), dim3((unsigned)tiles), dim3(kLines << LA), 0, s, a);
}

template <int LA, bool INV, bool LAST, bool SCALE = false>
static void launch_pass_ragged(const PassArgs* segs, const uint32_t* seg_block0, uint32_t nsegs, uint32_t nblocks,
                               hipStream_t s) {
  hipLaunchKernelGGL((ntt_pass_ragged_kernel<LA, INV, LAST, SCALE>), dim3(nblocks), dim3(kLines << LA), 0, s, segs,
                     seg_block0, nsegs);
}

// scale (a.do_scale) only with inv && last
#define PL_DEFINE_PASS_LAUNCHER(LA)                                                            \
  void launch_pass_la##LA(bool inv, bool last, const PassArgs& a, hipStream_t s) {             \
    if (inv) {                                                                                 \
      if (last) {                                                                              \
        if (a.do_scale) launch_pass<LA, true, true, true>(a, s);                               \
        else launch_pass<LA, true, true>(a, s);                                                \
      } else {                                                                                 \
        launch_pass<LA, true, false>(a, s);                                                    \
      }                                                                                        \
    } else {                                                                                   \
      if (last) launch_pass<LA, false, true>(a, s);                                            \
      else launch_pass<LA, false, false>(a, s);                                                \
    }                                                                                          \
  }                                                                                            \
  void launch_pass_ragged_la##LA(bool inv, bool last, bool scale, const PassArgs* segs, const uint32_t* sb, \
                                 uint32_t ns, uint32_t nb, hipStream_t s) {                    \
    if (inv) {                                                                                 \
      if (last) {                                                                              \
        if (scale) launch_pass_ragged<LA, true, true, true>(segs, sb, ns, nb, s);              \
        else launch_pass_ragged<LA, true, true>(segs, sb, ns, nb, s);                          \
      } else {                                                                                 \
        launch_pass_ragged<LA, true, false>(segs, sb, ns, nb, s);                              \
      }                                                                                        \
    } else {                                                                                   \
      if (last) launch_pass_ragged<LA, false, true>(segs, sb, ns, nb, s);                      \
      else launch_pass_ragged<LA, false, false>(segs, sb, ns, nb, s);                          \
    }                                                                                          \
  }

#define PL_DECLARE_RAGGED(LA)                                                                  \
  void launch_pass_ragged_la##LA(bool inv, bool last, bool scale, const PassArgs* segs, const uint32_t* sb, \
                                 uint32_t ns, uint32_t nb, hipStream_t s);
// Kernel arguments of pass p of the call c when every pass is a regular
// tile pass (false for the tiny and single-pass premultiplied forms, which
// ntt_launch handles with extra kernels).
bool pass_args_regular(const Domain& d, const NttCall& c, int p, PassArgs& a);
PL_DECLARE_RAGGED(0)
PL_DECLARE_RAGGED(1)
PL_DECLARE_RAGGED(2)
PL_DECLARE_RAGGED(3)
void launch_pass_la0(bool inv, bool last, const PassArgs& a, hipStream_t s);
void launch_pass_la1(bool inv, bool last, const PassArgs& a, hipStream_t s);
void launch_pass_la2(bool inv, bool last, const PassArgs& a, hipStream_t s);
void launch_pass_la3(bool inv, bool last, const PassArgs& a, hipStream_t s);

}  // namespace pl
