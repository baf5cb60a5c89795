// Scans over Fr: grand product, division by (X + c), evaluation.
//
//  grand product  z[0] = 1, z[i+1] = z[i] * p[i]     (exclusive prefix product)
//                 [accumulate_mul_poly, mont_arithmetic.cu:181-201, 333-361]
//  division       s_i = a_i + z * s_{i+1}, s_n = 0, z = -c; q[i] = s_{i+1},
//                 q[n-1] = 0, remainder a(z) = s_0     (affine suffix scan)
//                 [poly_div_poly, mont_arithmetic.cu:165-179, 203-212, 304-331]
//  evaluation     y = sum c_i x^i = s_0 of the same scan with z = x
//                 [evaluate, mont_arithmetic.cu:104-163, 283-302]
//
// The reference runs log2(n) Hillis-Steele passes over the whole array (one
// mulmod per element per pass).  Here every scan is work-efficient: a block
// owns 4096 consecutive elements (256 threads x 16), a reduce kernel folds
// each block to one value, the block values are scanned by the same code one
// level up (recursively), and a downsweep kernel rescans each block from its
// carry.  About 3 mulmods per element in total, three memory sweeps.
#include "fr29.hpp"
#include "pl_internal.hpp"
#include "run_stage.hpp"

namespace pl {

constexpr int kScanThreads = 256;
#ifndef PL_SCAN_LGPER
#define PL_SCAN_LGPER 4
#endif
constexpr int kLgPer = PL_SCAN_LGPER;        // elements per thread: 2^kLgPer
constexpr int kPer = 1 << kLgPer;
constexpr int kSeg = kScanThreads * kPer;    // elements per block
constexpr int kLgSeg = 8 + kLgPer;

// the bulk kernels move their runs in chunks of four elements (run_stage.hpp)
constexpr int kChunk = 4;
typedef RunStage<kChunk> Stage;

static inline unsigned sgrid(uint64_t n) { return (unsigned)((n + kSeg - 1) / kSeg); }

__device__ __forceinline__ void lds_put(uint4 (*l)[kScanThreads], int t, const fr& v) {
  l[0][t] = make_uint4(v.l[0], v.l[1], v.l[2], v.l[3]);
  l[1][t] = make_uint4(v.l[4], v.l[5], v.l[6], v.l[7]);
}
__device__ __forceinline__ fr lds_get(uint4 (*l)[kScanThreads], int t) {
  uint4 a = l[0][t], b = l[1][t];
  fr v;
  v.l[0] = a.x; v.l[1] = a.y; v.l[2] = a.z; v.l[3] = a.w;
  v.l[4] = b.x; v.l[5] = b.y; v.l[6] = b.z; v.l[7] = b.w;
  return v;
}

// R' mod r: the R'-form of one (R' = 2^261)
__host__ __device__ constexpr uint32_t rp_one_limb(int i) {
  return i == 0 ? 0xffffffbau : i == 1 ? 0x00000045u : i == 2 ? 0x0072d846u : i == 3 ? 0x1a25272eu
       : i == 4 ? 0x5dbeee8bu : i == 5 ? 0xfe2eedcdu : i == 6 ? 0x9eefbe41u : 0x4d043f42u;
}
__device__ __forceinline__ fr rp_one_fr() {
  fr o;
#pragma unroll
  for (int i = 0; i < 8; i++) o.l[i] = rp_one_limb(i);
  return o;
}

// Block geometry of a scan kernel: 256 threads x 2^LG elements.  LG = kLgPer
// for the bulk; a single-block level takes the smallest that covers it, where
// the latency of the per-thread chains (2^LG dependent products) dominates.
template <int LG>
struct ScanGeom {
  static constexpr int kPer = 1 << LG;
  static constexpr int kLgSeg = 8 + LG;
};

// ---------------------------------------------------------------------------
// multiplicative prefix scan
// ---------------------------------------------------------------------------
// The products run in signed radix-2^29 limbs (fr29.hpp): P(a, b) = a b / R',
// R' = 2^261, about 205 VALU instructions against the saturated product's 290.
// A stored word S(x) = x R shifted left by five bits is the integer 32 x R =
// x R', the R'-form that P is closed under, and it fits nine 29-bit digits; so
// P(S(a), 32 S(b)) = S(a b) with the shift taken in the digit split.  Level 0
// (RF false) reads stored words: its running products stay in stored form,
// its block products and everything a level above reads are in R'-form
// (RF true).  At 2^21 the only block of the upper level took 37-54 us on
// chains of 16 products and eight barrier-separated scan steps; with two
// elements per thread and the scan inside the wave, 9-12 us.  Bounds: a word of
// at most r enters as w = 32 x R <= 32 r, so a step maps |h| to at most
// 0.453 |h| + r / 2 with centred Montgomery digits (BM), and |h| < 0.96 r from
// h = S(x_0) <= r; in R'-form a step of values within 1.1 r lies in (-1.02 r,
// 0.02 r).  Both fit a pbd word (1.104 r).  pfx_reduce_kernel packs nothing, so
// it takes any 256-bit words (16 steps stay within 9 r).

// nine 29-bit digits of 32 x (x any 256-bit word)
__device__ __forceinline__ void split29_x32(const uint32_t* x, uint32_t* a) {
  a[0] = (x[0] << 5) & kMask29;
#pragma unroll
  for (int i = 1; i < 8; i++) {
    const int b = 29 * i - 5;
    a[i] = funnel_r(x[(b >> 5) + 1], x[b >> 5], b & 31) & kMask29;
  }
  a[8] = x[7] >> 3;
}

// a word of x's class below (1 + 2^-30) r: what the running products' bounds
// above ask of a caller's word.  Canonical words fail the one comparison; any
// other 256-bit word (below 2.21 r) is at most two subtractions away.
__device__ __forceinline__ void fr_near_canonical(fr& x) {
  while (x.l[7] > r_limb(7)) {
    uint32_t b = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) x.l[i] = __builtin_subc(x.l[i], r_limb(i), b, &b);
  }
}

// 32 v for balanced digits of a value within 1.1 r, again balanced
__device__ __forceinline__ v9 v9_x32(const v9& v) {
  v9 o;
  int64_t acc = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    acc += (int64_t)(int32_t)v.l[i] * 32;
    o.l[i] = sext29((uint32_t)acc);
    acc = (acc - (int64_t)(int32_t)o.l[i]) >> 29;
  }
  o.l[8] = (uint32_t)(acc + (int64_t)(int32_t)v.l[8] * 32);
  return o;
}

__device__ __forceinline__ v9 shfl_up9(const v9& v, int s) {
  v9 o;
#pragma unroll
  for (int i = 0; i < 9; i++) o.l[i] = (uint32_t)__shfl_up((int)v.l[i], s);
  return o;
}

// P closed in R'-form, balanced digits
__device__ __forceinline__ v9 mul_r(const v9& a, const v9& b) { return v9_mul<false, false, true>(a, b.l); }

// partial[b] = product of block b's elements (R'-form word).  The product is
// order-free, so thread t takes elements b*kSeg + 256 k + t: every load is
// coalesced.  Across the wave six exchange steps, then the four wave products.
template <bool RF>
__global__ void __launch_bounds__(kScanThreads) pfx_reduce_kernel(const fr* in, uint64_t n, fr* partial) {
  __shared__ uint32_t wt[4][9];
  const int t = threadIdx.x;
  const uint64_t b0 = (uint64_t)blockIdx.x << kLgSeg;
  const uint32_t rem = (uint32_t)(n - b0 < kSeg ? n - b0 : kSeg);
  fr v[kPer];
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    if ((uint32_t)(k * kScanThreads + t) < rem) v[k] = fr_load(in + b0 + k * kScanThreads + t);
  });
  v9 h;
  unpack_ext(rp_one_fr().l, h.l);
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    // one element at a time, as its load arrives
    if ((uint32_t)(k * kScanThreads + t) < rem) {
      uint32_t w[9];
      if constexpr (RF) split29(v[k].l, w);
      else split29_x32(v[k].l, w);
      h = v9_mul<false, !RF, true>(h, w);
    }
  });
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    v9 o;
#pragma unroll
    for (int i = 0; i < 9; i++) o.l[i] = (uint32_t)__shfl_xor((int)h.l[i], m);
    h = mul_r(h, o);
  }
  if ((t & 63) == 0) {
#pragma unroll
    for (int i = 0; i < 9; i++) wt[t >> 6][i] = h.l[i];
  }
  __syncthreads();
  if (t >= 64) return;
#pragma unroll
  for (int w = 1; w < 4; w++) h = v9_mul<false, false, true>(h, wt[w]);
  if (t == 0) fr_store(partial + blockIdx.x, v9_canonical(h));
}

// out_excl[i] = carry_b * prod_{block start <= j < i} in[j]; optional inclusive
// output.  carry (R'-form words) == nullptr means one.  in may equal out_excl.
template <int LG, bool RF>
__global__ void __launch_bounds__(kScanThreads) __attribute__((amdgpu_waves_per_eu(2)))
pfx_down_kernel(const fr* in, fr* out_excl, fr* out_incl, uint64_t n, const fr* carry) {
  constexpr int kPer = ScanGeom<LG>::kPer, kLgSeg = ScanGeom<LG>::kLgSeg;
  __shared__ uint32_t wt[4][9];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint64_t b0 = (uint64_t)blockIdx.x << kLgSeg;
  const int rem = (int)(n - b0 < kScanThreads * kPer ? n - b0 : kScanThreads * kPer) - t * kPer;
  const fr* src = in + b0 + t * kPer;
  fr e[kPer];
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    e[k] = fr_zero();
    if (k < rem) e[k] = fr_load(src + k);
  });
  v9 one;
  unpack_ext(rp_one_fr().l, one.l);
  // local inclusive products: e[k] = in[base] * ... * in[base+k], pbd words
  // (level 0: stored form; an element beyond n counts as one)
  v9 h;
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    if constexpr (!RF) fr_near_canonical(e[k]);
    if constexpr (k == 0) {
      h = one;  // no element of this thread: R'-form one (never stored)
      if (rem > 0) unpack_ext(e[0].l, h.l);
    } else if (k < rem) {
      uint32_t w[9];
      if constexpr (RF) split29(e[k].l, w);
      else split29_x32(e[k].l, w);
      h = v9_mul<false, !RF, true>(h, w);
    }
    pbd_pack(h.l, e[k].l);  // words below 1.1 r and products fit
  });
  // thread products in R'-form, their exclusive prefix across the block
  v9 p = RF || rem <= 0 ? h : v9_x32(h);
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const v9 o = shfl_up9(p, s);
    const v9 q = mul_r(p, o);
    if (lane >= s) p = q;
  }
  if (lane == 63) {
#pragma unroll
    for (int i = 0; i < 9; i++) wt[wave][i] = p.l[i];
  }
  __syncthreads();
  v9 pre = shfl_up9(p, 1);
  if (lane == 0) pre = one;
#pragma unroll
  for (int w = 0; w < 3; w++)
    if (w < wave) pre = v9_mul<false, false, true>(pre, wt[w]);
  if (carry) {
    uint32_t c[9];
    split29(fr_load(carry + blockIdx.x).l, c);
    pre = v9_mul<false, false, true>(pre, c);
  }
  fr* dst = out_excl + b0 + t * kPer;
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    if (k < rem) {
      fr ex;
      if constexpr (k == 0) {
        if constexpr (RF) {
          ex = v9_canonical(pre);
        } else {
          uint32_t w[9];
          split29(fr_one().l, w);
          ex = v9_canonical(v9_mul<false, false, false>(pre, w));
        }
      } else {
        uint32_t w[9];
        pbd_unpack(e[k > 0 ? k - 1 : 0].l, w);
        ex = v9_canonical(v9_mul<false, false, false>(pre, w));
      }
      fr_store(dst + k, ex);
      if constexpr (!RF) {
        // an inclusive output is the next element's exclusive one
        if (out_incl) {
          if constexpr (k > 0) fr_store(out_incl + b0 + t * kPer + k - 1, ex);
          if (k == kPer - 1 || k == rem - 1) {
            uint32_t w[9];
            pbd_unpack(e[k].l, w);
            fr_store(out_incl + b0 + t * kPer + k, v9_canonical(v9_mul<false, false, false>(pre, w)));
          }
        }
      }
    }
  });
}

// Exclusive prefix product of n elements; scratch needs pfx_scratch_elems(n).
static uint64_t pfx_scratch_elems(uint64_t n) {
  uint64_t tot = 0;
  while (n > (uint64_t)kSeg) {
    n = (n + kSeg - 1) / kSeg;
    tot += 2 * n;
  }
  return tot + 1;
}

// the only block of a level: the smallest geometry that covers it
template <bool RF>
static void pfx_one_block(const fr* in, fr* out_excl, fr* out_incl, uint64_t n, hipStream_t s) {
  const dim3 g(1), b(kScanThreads);
  const fr* none = nullptr;
  if (n <= 256) hipLaunchKernelGGL((pfx_down_kernel<0, RF>), g, b, 0, s, in, out_excl, out_incl, n, none);
  else if (n <= 512) hipLaunchKernelGGL((pfx_down_kernel<1, RF>), g, b, 0, s, in, out_excl, out_incl, n, none);
  else if (n <= 1024) hipLaunchKernelGGL((pfx_down_kernel<2, RF>), g, b, 0, s, in, out_excl, out_incl, n, none);
  else if (n <= 2048) hipLaunchKernelGGL((pfx_down_kernel<3, RF>), g, b, 0, s, in, out_excl, out_incl, n, none);
  else hipLaunchKernelGGL((pfx_down_kernel<kLgPer, RF>), g, b, 0, s, in, out_excl, out_incl, n, none);
}

template <bool RF>
static hipError_t prefix_product(const fr* in, fr* out_excl, fr* out_incl, uint64_t n, fr* scratch, hipStream_t s) {
  if (n <= (uint64_t)kSeg) {
    pfx_one_block<RF>(in, out_excl, out_incl, n, s);
    return hipGetLastError();
  }
  const uint64_t nb = (n + kSeg - 1) / kSeg;
  fr* part = scratch;
  fr* part_excl = scratch + nb;
  hipLaunchKernelGGL(pfx_reduce_kernel<RF>, dim3(sgrid(n)), dim3(kScanThreads), 0, s, in, n, part);
  hipError_t e = prefix_product<true>(part, part_excl, nullptr, nb, scratch + 2 * nb, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((pfx_down_kernel<kLgPer, RF>), dim3(sgrid(n)), dim3(kScanThreads), 0, s, in, out_excl, out_incl,
                     n, (const fr*)part_excl);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// affine suffix scan  s_i = a_i + m * s_{i+1}
// pw: device table of m^(2^j) R' mod r, j = 0..kLgSeg (m^kSeg last), R' = 2^261:
// every product of the scan multiplies a value by a power of m, so it runs as
// the radix-2^29 product (fr29.hpp) with the power in that form: the Horner
// steps in signed limbs (horner29), the block combines on canonical values.
// ---------------------------------------------------------------------------

// a * w R' / R' = a w (stored form), canonical
__device__ __forceinline__ fr mulp(const fr& a, const fr& w) { return fr_reduce_once(fr_mul29(a, w)); }
// block suffix combine: V_t <- V_t + m^(2^LG * 2^s) V_{t+2^s}; returns the
// suffix value starting at thread t (the block's carry folded in by the caller)
template <int LG>
__device__ fr block_suffix(fr v, uint4 (*l)[kScanThreads], const fr* pw) {
  constexpr int kLgPer = LG;
  const int t = threadIdx.x;
  lds_put(l, t, v);
  __syncthreads();
  for (int s = 0; (1 << s) < kScanThreads; s++) {
    const int o = 1 << s;
    fr other = t + o < kScanThreads ? lds_get(l, t + o) : fr_zero();
    __syncthreads();
    if (t + o < kScanThreads) v = fr_add(v, mulp(other, fr_load(pw + kLgPer + s)));  // m^(kPer * 2^s)
    lds_put(l, t, v);
    __syncthreads();
  }
  return v;
}

// Run suffixes of a block, S_t = sum_(t' >= t) v_t' mu^(t' - t): six exchange
// steps inside the wave, then the sum over the waves after: with D_w = s at the
// end of wave w, S_t += mu^(64 - lane) D_w (f: that power's digits).  The
// running value is signed limbs: products with balanced digits (2^28) summed
// seven times.  pw(s, p): the balanced digits of mu^(2^s) R', s < 7.
template <class Pw>
__device__ __forceinline__ fr run_suffix(v9 v, const uint32_t (&f)[9], uint32_t (*wt)[9], Pw pw) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int s = 0; s < 6; s++) {
    v9 o;
#pragma unroll
    for (int i = 0; i < 9; i++) o.l[i] = (uint32_t)__shfl_down((int)v.l[i], 1 << s);
    uint32_t p[9];
    pw(s, p);
    o = v9_mul<false, false, true>(o, p);
    if (lane + (1 << s) < 64) v = v9_add(v, o);
  }
  if (lane == 0) {
    const fr c = v9_canonical(v);
    v9 b;
    unpack_ext(c.l, b.l);
#pragma unroll
    for (int i = 0; i < 9; i++) wt[w][i] = b.l[i];
  }
  __syncthreads();
  if (w < 3) {
    v9 d;  // D_w: the later waves' values by Horner in mu^64
    uint32_t p[9];
    pw(6, p);
#pragma unroll
    for (int i = 0; i < 9; i++) d.l[i] = wt[3][i];
    for (int k = 2; k > w; k--) {
      d = v9_mul<false, false, true>(d, p);
#pragma unroll
      for (int i = 0; i < 9; i++) d.l[i] += wt[k][i];
    }
    v = v9_add(v, v9_mul<false, false, true>(d, f));
  }
  return v9_canonical(v);
}

// the factor of the word w R' for a whole kernel's Horner steps
__device__ __forceinline__ rows_all rp_rows(const fr* w) { return rows29_spread(rows29_make<true>(fr_load(w))); }

// sum_k v_k w^k by Horner in signed limbs (fr29.hpp): h <- h w + v_k with the
// wave-uniform w held as rows in SGPRs (about 150 VALU instructions per step,
// 225 with w per lane; evaluation of 2^24 176 -> 154 us, of 2^20 24.9 -> 22.3,
// division 598 -> 565 and 52.7 -> 48.7), limb-wise sums of a product and a word
// (digits in [0, 2^29) both), so every limb stays below 2^30 and the product within
// (-1.001 r, 0.001 r); canonical once at the end.
template <int K>
__device__ __forceinline__ fr horner29(const fr (&v)[K], const rows_all& w) {
  v9 h;
  split29(v[K - 1].l, h.l);
  static_for<0, K - 1>([&](auto k_) {
    constexpr int k = K - 2 - decltype(k_)::value;
    v9 x;
    split29(v[k].l, x.l);
    h = v9_add(v9_mul_all<false>(h, w), x);
  });
  return v9_canonical(h);
}

// The powers table beyond level 0: pw[from + j] = pw[from + j - 1]^2 for
// j < count - from.  A multi-level scan's first reduce launch runs it in one
// extra block (block 0, dispatched first) beside the reduction; only the
// levels above read those entries.
struct PwExt {
  fr* pw;
  int from, count;  // count == 0: no extension
};
__device__ void pw_extend(const PwExt& e) {
  fr m = fr_load(e.pw + e.from - 1);
  for (int j = e.from; j < e.count; j++) {
    m = mulp(m, m);
    fr_store(e.pw + j, m);
  }
}

// partial[b] = sum over block b of a_k m^(k - start).  The sum is
// order-free: thread t takes elements start + 256 j + t (coalesced loads),
// H_t = sum_j a m^(256 j) by Horner in m^256, then m^t H_t; a plain sum over
// the block finishes it.
template <int LG>
__global__ void __launch_bounds__(kScanThreads) sfx_reduce_kernel(const fr* a, uint64_t n, const fr* pw, fr* partial,
                                                                   PwExt ext, const fr* mtab) {
  constexpr int kPer = ScanGeom<LG>::kPer, kLgSeg = ScanGeom<LG>::kLgSeg;
  __shared__ uint4 l[2][kScanThreads];
  const int t = threadIdx.x;
  uint32_t blk = blockIdx.x;
  if (ext.count) {
    if (blk == 0) {
      if (t == 0) pw_extend(ext);
      return;
    }
    blk--;
  }
  const uint64_t b0 = (uint64_t)blk << kLgSeg;
  const rows_all M = rp_rows(pw + 8);  // m^256
  fr v[kPer];
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const uint64_t i = b0 + (uint64_t)k * kScanThreads + t;
    v[k] = i < n ? fr_load(a + i) : fr_zero();
  });
  fr h = horner29<kPer>(v, M);
  // m^t R': from the table when the caller built one (sfx_powers_kernel),
  // else from the powers m^(2^bit) R'
  fr mt;
  if (mtab) {
    mt = fr_load(mtab + t);
  } else {
#pragma unroll
    for (int i = 0; i < 8; i++) mt.l[i] = rp_one_limb(i);
    static_for<0, 8>([&](auto b_) {
      constexpr int b = decltype(b_)::value;
      if ((t >> b) & 1) mt = mulp(mt, fr_load(pw + b));
    });
  }
  h = mulp(h, mt);
  lds_put(l, t, h);
  __syncthreads();
  for (int s = kScanThreads / 2; s > 0; s >>= 1) {
    if (t < s) {
      h = fr_add(h, lds_get(l, t + s));
      lds_put(l, t, h);
    }
    __syncthreads();
  }
  if (t == 0) fr_store(partial + blk, h);
}

// partial[b] as sfx_reduce_kernel computes it, from contiguous runs (thread t
// owns the kPer elements the down-sweep gives it).  lt takes what the
// down-sweep needs of each run, so that it starts at its rescan.  TAB, the
// level that holds the data: the suffix S_t of the block's runs (run_suffix,
// with mu = m^kPer and its powers in mutab), and the block's value is S_0.
// Otherwise the run's Horner value L_t, scanned again below with the carry.
// The runs come as 128-byte chunks through LDS (run_stage.hpp).
// Division of 2^24: this kernel 230 -> 200 us, bound by its products; the
// down-sweep 331 -> 195, a copy's time; with the chunks alone, the scans as
// before, 200 and 266.  (After half a second of the same load this kernel takes
// 177, the down-sweep 191.)  Opening of 2^24 + 5 coefficients 845 us, of 2^22 + 5
// 262; 1010 and 340 with the scans before these and the factor per lane.
template <bool TAB>
__global__ void __launch_bounds__(kScanThreads) sfx_run_reduce_kernel(const fr* a, uint64_t n, const fr* pw,
                                                                      fr* partial, fr* lt, PwExt ext,
                                                                      const fr* mutab) {
  __shared__ uint4 l[2][TAB ? 1 : kScanThreads];
  __shared__ uint32_t wt[4][9];
  __shared__ uint4 stage[Stage::kSlots * kScanThreads / 64];
  const int t = threadIdx.x;
  uint32_t blk = blockIdx.x;
  if (ext.count) {
    if (blk == 0) {
      if (t == 0) pw_extend(ext);
      return;
    }
    blk--;
  }
  const uint64_t tid = (uint64_t)blk * kScanThreads + t;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint64_t w0 = ((uint64_t)blk * kScanThreads + 64 * wave) * kPer;  // the wave's first element
  const bool all = w0 + 64 * kPer <= n;
  const int64_t lim = (int64_t)(n - w0);
  const Stage st{stage + Stage::kSlots * wave, t & 63};
  uint4 raw[Stage::P];
  st.fetch(a + w0 + kPer - kChunk, kPer, lim - (kPer - kChunk), all, raw);
  const rows_all m = rp_rows(pw);
  // Horner over the run in signed limbs (horner29), top chunk first; the next
  // chunk is asked for before the chain over this one
  v9 hv;
  static_for<0, kPer / kChunk>([&](auto c_) {
    constexpr int k0 = kPer - kChunk * (decltype(c_)::value + 1);
    st.put(raw);
    if constexpr (k0 > 0) st.fetch(a + w0 + (k0 - kChunk), kPer, lim - (k0 - kChunk), all, raw);
    static_for<0, kChunk>([&](auto j_) {
      constexpr int j = kChunk - 1 - decltype(j_)::value;
      v9 x;
      split29(st.get(j).l, x.l);
      if constexpr (k0 + j == kPer - 1) hv = x;
      else hv = v9_add(v9_mul_all<false>(hv, m), x);
    });
  });
  const fr h = v9_canonical(hv);
  if constexpr (TAB) {
    v9 v;
    unpack_ext(h.l, v.l);
    uint32_t f[9];
    unpack_ext(fr_load(mutab + 64 - (t & 63)).l, f);
    const fr S = run_suffix(v, f, wt, [&](int s, uint32_t* p) { unpack_ext(fr_load(pw + kLgPer + s).l, p); });
    fr_store(lt + tid, S);
    if (t == 0) fr_store(partial + blk, S);
  } else {
    fr_store(lt + tid, h);
    const fr v = block_suffix<kLgPer>(h, l, pw);
    if (t == 0) fr_store(partial + blk, v);
  }
}

// out[i] = s_{i+1} within each block given carry[b] = s at the block's end
// (nullptr: zero); total (block 0) = s_0.  out may equal a.
// LT: lt comes from sfx_run_reduce_kernel; the elements are then read only for
// the rescan, in chunks through LDS (run_stage.hpp).  With TAB lt holds the run
// suffixes and the carry at the end of run t is S_(t+1) + mu^(255 - t) K, one
// product where the block suffix takes eight behind 16 barriers.  Otherwise
// the local Horner values are scanned here.
template <int LG, bool LT, bool TAB>
__global__ void __launch_bounds__(kScanThreads) __attribute__((amdgpu_waves_per_eu(LT ? 4 : 1)))
sfx_down_kernel(const fr* a, fr* out, uint64_t n, const fr* pw,
                                                                 const fr* carry, fr* total, const fr* lt,
                                                                 const fr* mutab) {
  static_assert(!TAB || LT, "run suffixes come from the reduce");
  constexpr int kPer = ScanGeom<LG>::kPer, kLgSeg = ScanGeom<LG>::kLgSeg, kLgPer = LG;
  __shared__ uint4 stage[LT ? Stage::kSlots * kScanThreads / 64 : 1];
  const int t = threadIdx.x;
  const uint64_t base = ((uint64_t)blockIdx.x << kLgSeg) + (uint64_t)t * kPer;
  [[maybe_unused]] uint4 raw[Stage::P];
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint64_t w0 = ((uint64_t)blockIdx.x << kLgSeg) + (uint64_t)(64 * wave) * kPer;  // the wave's first element
  const bool all = w0 + 64 * kPer <= n;
  const int64_t lim = (int64_t)(n - w0);
  [[maybe_unused]] const Stage st{stage + (LT ? Stage::kSlots * wave : 0), t & 63};
  if constexpr (LT) st.fetch(a + w0 + (kPer - kChunk), kPer, lim - (kPer - kChunk), all, raw);
  const v9 row = rows29_make<true>(fr_load(pw));  // m's rows, spread where they are used
  fr K = carry ? fr_load(carry + blockIdx.x) : fr_zero();
  fr cin;  // s at the start of thread t+1
  if constexpr (TAB) {
    cin = mulp(K, fr_load(mutab + (kScanThreads - 1 - t)));
    if (t + 1 < kScanThreads) cin = fr_add(cin, fr_load(lt + ((uint64_t)blockIdx.x * kScanThreads + t + 1)));
  } else {
    // local Horner: L = sum_k e_k m^k
    fr h;
    if constexpr (LT) {
      h = fr_load(lt + ((uint64_t)blockIdx.x * kScanThreads + t));
    } else {
      fr e[kPer];
      static_for<0, kPer>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        e[k] = base + k < n ? fr_load(a + base + k) : fr_zero();
      });
      h = horner29<kPer>(e, rows29_spread(row));
    }
    // fold the block carry into the last thread: s(start of thread 255) = L + m^kPer K
    if (t == kScanThreads - 1) h = fr_add(h, mulp(K, fr_load(pw + kLgPer)));
    __shared__ uint4 l[2][kScanThreads];
    const fr v = block_suffix<LG>(h, l, pw);  // s at the start of this thread's run
    cin = t + 1 < kScanThreads ? lds_get(l, t + 1) : K;
    if (total && blockIdx.x == 0 && t == 0) fr_store(total, v);
  }
  // rescan: s_k = e_k + m s_{k+1}, out[base + k] = s_{k+1} (signed limbs,
  // canonical where stored); out may equal a: each half's elements are read
  // before its outputs are written, and the low half's outputs only overwrite
  // elements already read
  const rows_all m = rows29_spread(row);
  v9 sn;
  split29(cin.l, sn.l);
  if constexpr (LT) {
    // the next chunk is asked for before the chain over this one
    static_for<0, kPer / kChunk>([&](auto c_) {
      constexpr int k0 = kPer - kChunk * (decltype(c_)::value + 1);
      st.put(raw);
      if constexpr (k0 > 0) st.fetch(a + w0 + (k0 - kChunk), kPer, lim - (k0 - kChunk), all, raw);
      static_for<0, kChunk>([&](auto j_) {
        constexpr int j = kChunk - 1 - decltype(j_)::value, k = k0 + j;
        v9 x;
        split29(st.get(j).l, x.l);
        st.set(j, k == kPer - 1 ? cin : v9_canonical(sn));
        if constexpr (k > 0) sn = v9_add(v9_mul_all<false>(sn, m), x);
      });
      st.store(out + w0 + k0, kPer, lim - k0, all);
    });
  } else {
    constexpr int G = kPer > 1 ? 2 : 1, Q = kPer / G;
    static_for<0, G>([&](auto g_) {
      constexpr int top = kPer - 1 - decltype(g_)::value * Q;  // highest index of this half
      fr e[Q];
      static_for<0, Q>([&](auto j_) {
        constexpr int k = top - decltype(j_)::value;
        e[top - k] = k > 0 && base + k < n ? fr_load(a + base + k) : fr_zero();
      });
      static_for<0, Q>([&](auto j_) {
        constexpr int k = top - decltype(j_)::value;
        if (base + k < n) fr_store(out + base + k, k == kPer - 1 ? cin : v9_canonical(sn));
        if constexpr (k > 0) {
          v9 x;
          split29(e[top - k].l, x.l);
          sn = v9_add(v9_mul_all<false>(sn, m), x);
        }
      });
    });
  }
}

__global__ void zero_kernel(fr* p, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) fr_store(p + i, fr_zero());
}

hipError_t fill_zero(fr* p, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

// pw[j] = m^(2^j) R' mod r, j < count; m = neg ? -(*src) : *src.  32 m (five
// doublings) is m R' in the stored form; squares stay in that form.  Level L
// of a scan (values combined 4096^L at a time) uses pw + 12 L: its multiplier
// is m^(4096^L), whose powers of two continue the same squaring chain.
// tab (128 threads): also tab[t] = m^(t 2^sh) R' for t < 256: sh = 0 for the
// evaluation's reduce, which multiplies each thread's value by m^t, kLgPer for
// the run suffixes.  The second wave extends it by doubling (step j fills
// [2^j, 2^(j+1)) from pw[sh + j]) while thread 0 raises the next square.
__global__ void sfx_powers_kernel(const fr* src, int neg, fr* pw, int count, fr* tab, int sh) {
  const int t = threadIdx.x;
  fr m;
  if (t == 0) {
    m = fr_load(src);
    if (neg) m = fr_neg(m);
    for (int d = 0; d < 5; d++) m = fr_add(m, m);
  }
  if (tab && t == 64) {
    fr one;
#pragma unroll
    for (int i = 0; i < 8; i++) one.l[i] = rp_one_limb(i);
    fr_store(tab, one);
  }
  for (int j = 0; j < count; j++) {
    if (t == 0) fr_store(pw + j, m);
    if (tab) __syncthreads();  // pw[j] and the table's entries below 2^j visible
    if (t == 0 && j + 1 < count) m = mulp(m, m);
    if (tab && j >= sh && j < sh + 8 && t >= 64) {
      const int h = 1 << (j - sh);
      for (int i = t - 64; i < h; i += 64) fr_store(tab + h + i, mulp(fr_load(tab + i), fr_load(pw + j)));
    }
  }
}

constexpr int kPw = kLgSeg + 1;

// levels of a suffix scan over n values, and the power-table entries they use
static int sfx_levels(uint64_t n) {
  int L = 1;
  while (n > (uint64_t)kSeg) {
    n = (n + kSeg - 1) / kSeg;
    L++;
  }
  return L;
}
static int sfx_pw_count(uint64_t n) { return kPw + kLgSeg * (sfx_levels(n) - 1); }
// the entries that the powers kernel raises: level 0's, for a single block those
// that its geometry reads (sfx_one_block: m^256, or mu^(2^s) up to s = 7)
static int sfx_pw_first(uint64_t n) {
  return n <= 512 ? 9 : n <= 1024 ? 10 : kPw;
}
// the entries beyond level 0's, for the first reduce launch (none for one level)
static PwExt pw_ext(fr* pw, int np) { return np > kPw ? PwExt{pw, kPw, np} : PwExt{nullptr, 0, 0}; }

static uint64_t sfx_scratch_elems(uint64_t n) {
  uint64_t tot = (uint64_t)sfx_pw_count(n);
  while (n > (uint64_t)kSeg) {
    n = (n + kSeg - 1) / kSeg;
    tot += 2 * n + n * kScanThreads;  // block values, carries, local Horner values
  }
  return tot;
}

// the only block of a level: the smallest geometry that covers it, as the
// chains of 2^LG dependent steps are what it takes (2001
// coefficients: reduce 9.5 -> 6.9 us, sweep 25.4 -> 20.2 with 8 per thread
// for 16; opening of 1001 63.6 -> 40.4 us)
template <int LG>
static void sfx_one_block(const fr* a, fr* out, uint64_t n, const fr* pw, fr* total, const fr* mt, hipStream_t s) {
  const fr* none = nullptr;
  if (out)
    hipLaunchKernelGGL((sfx_down_kernel<LG, false, false>), dim3(1), dim3(kScanThreads), 0, s, a, out, n, pw, none, total, none,
                       none);
  else  // the reduce kernel's tree value is s_0
    hipLaunchKernelGGL(sfx_reduce_kernel<LG>, dim3(1), dim3(kScanThreads), 0, s, a, n, pw, total,
                       PwExt{nullptr, 0, 0}, mt);
}

// suffix scan with powers table pw (this level's m): out[i] = s_{i+1} (if out),
// *total = s_0 (if total).  out == nullptr: reduction only.  mt (the level
// that holds the data): the powers kernel's table, of m^t for a reduction, of
// m^(kPer t) with a down-sweep.
static hipError_t suffix_scan(const fr* a, fr* out, uint64_t n, const fr* pw, fr* total, fr* scratch, hipStream_t s,
                              PwExt ext = PwExt{nullptr, 0, 0}, const fr* mt = nullptr) {
  if (n <= (uint64_t)kSeg) {
    if (n <= 256) sfx_one_block<0>(a, out, n, pw, total, mt, s);
    else if (n <= 512) sfx_one_block<1>(a, out, n, pw, total, mt, s);
    else if (n <= 1024) sfx_one_block<2>(a, out, n, pw, total, mt, s);
    else if (n <= 2048) sfx_one_block<3>(a, out, n, pw, total, mt, s);
    else sfx_one_block<kLgPer>(a, out, n, pw, total, mt, s);
    return hipGetLastError();
  }
  const uint64_t nb = (n + kSeg - 1) / kSeg;
  fr* part = scratch;
  fr* carry = scratch + nb;
  fr* lt = scratch + 2 * nb;
  // with a down-sweep, the reduce runs over the down-sweep's runs and keeps
  // their local Horner values; a reduction alone reads strided (coalesced)
  const unsigned grid = sgrid(n) + (ext.count ? 1 : 0);
  const dim3 th(kScanThreads);
  if (!out)
    hipLaunchKernelGGL(sfx_reduce_kernel<kLgPer>, dim3(grid), th, 0, s, a, n, pw, part, ext, mt);
  else if (mt)
    hipLaunchKernelGGL(sfx_run_reduce_kernel<true>, dim3(grid), th, 0, s, a, n, pw, part, lt, ext, mt);
  else
    hipLaunchKernelGGL(sfx_run_reduce_kernel<false>, dim3(grid), th, 0, s, a, n, pw, part, lt, ext, mt);
  // carry[b] = s at the end of block b = sum_{b' > b} part[b'] (m^4096)^(b'-b-1)
  hipError_t e = suffix_scan(part, out ? carry : nullptr, nb, pw + kLgSeg, total, lt + nb * kScanThreads, s);
  if (e != hipSuccess || !out) return e;
  fr* none = nullptr;
  if (mt)
    hipLaunchKernelGGL((sfx_down_kernel<kLgPer, true, true>), dim3(sgrid(n)), th, 0, s, a, out, n, pw,
                       (const fr*)carry, none, (const fr*)lt, mt);
  else
    hipLaunchKernelGGL((sfx_down_kernel<kLgPer, true, false>), dim3(sgrid(n)), th, 0, s, a, out, n, pw,
                       (const fr*)carry, none, (const fr*)lt, mt);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// evaluation and division, latency form (kLatMin <= n <= kLatMax)
// ---------------------------------------------------------------------------
// A Fr product costs a wave about the same issue time whether or not other
// waves share its SIMD, so at these sizes the scan above is bound by the
// products its busiest SIMD issues in sequence: the powers chain, then the
// reduce (which waits for the powers), then the top level.  Here the powers
// are raised beside the data instead of before it:
//
//   launch 1  data blocks 1..G: thread t of block b owns the run of K
//             consecutive coefficients at (256 b + t) K and stores its
//             Horner value L = sum_k a_k m^k, which needs m alone;
//             table block 0 (on a CU of its own: G + 1 <= 256 blocks) raises
//             m: mu = m^K, its squares mu^(2^s), A_j = mu^j (j < 256) and
//             B_b = mu^(256 b) (b < G), multiplied up as the squares appear;
//   evaluation (m = x)
//   launch 2  block b: P_b = B_b sum_t L_(256 b + t) A_t;
//   launch 3  y = sum_b P_b;
//   division by X + c (m = -c; s_i = a_i + m s_(i+1), q_i = s_(i+1));
//             launch 1 also keeps each run's upper-half Horner value H
//   launch 2  block b scans its 256 run values with mu: the run suffixes S_t
//             and the block value P_b = S_0;
//   launch 3  two threads per run: each block forms its carry
//             C_b = sum_j P_(b+1+j) B_j; the carry at the end of run t is
//             S_(t+1) + mu^(255 - t) C_b, the lower half starts from
//             H_t + m^(K/2) times it, and both halves rescan in place.
//
// The launch boundaries carry the tables and values between blocks; a
// release/acquire hand-off inside one launch costs more than a launch here
// (it writes back and invalidates the L2 of every XCD involved).
// from here up three launches beat the powers chain and its single block
// (opening of 2001 42.3 against 47.9 us; of 1001 the single block's 40.4)
constexpr uint64_t kLatMin = (1ull << 10) + 1;
constexpr uint64_t kLatMax = 255ull * 256 * 28;  // runs of at most 28 coefficients (in registers)
constexpr uint32_t kLatMaxG = 255;
// workspace (Fr elements): A, B, P (256 each), mu^(2^s) (16), m^(K/2) (1), m
// (1), L (256 G; the division replaces it by the run suffixes S), and for the
// division the upper-half Horner values H (256 G).  The caller's point is read
// in launch 1 alone: the value, the remainder and the quotient, all written
// after it, may lie over the point.
constexpr uint64_t kWsA = 0, kWsB = 256, kWsP = 512, kWsPw = 768, kWsHalf = 784, kWsM = 785, kWsL = 800;

// the multiplier of a scan in stored form: x, or -c for a division by X + c
__device__ __forceinline__ fr load_m(const fr* x, int neg) {
  const fr m = fr_load(x);
  return neg ? fr_neg(m) : m;
}
// m R' as balanced digits within (-0.51 r, 0.51 r)
__device__ __forceinline__ v9 m_rp(const fr& m) {
  v9 a, b;
  split29_x32(m.l, a.l);
  reduce_centered(a.l, b.l);
  return b;
}

// Horner over a run held in registers, each element's digit split ordered
// after the previous step (an empty asm that reads the running value), so
// the loads issued before it are waited for one by one as the chain reaches
// them instead of all at once
// *upper (if not null): the value after the upper half, sum_(k >= K/2) a_k m^(k - K/2)
template <int K>
__device__ __forceinline__ fr horner29_inorder(fr (&v)[K], const rows_all& w, fr* upper) {
  v9 h;
  split29(v[K - 1].l, h.l);
  static_for<0, K - 1>([&](auto k_) {
    constexpr int k = K - 2 - decltype(k_)::value;
    fr e = v[k];
    asm volatile("" : "+v"(e.l[0]), "+v"(e.l[1]), "+v"(e.l[2]), "+v"(e.l[3]), "+v"(e.l[4]), "+v"(e.l[5]),
                 "+v"(e.l[6]), "+v"(e.l[7]) : "v"(h.l[0]));
    v9 xv;
    split29(e.l, xv.l);
    h = v9_add(v9_mul_all<false>(h, w), xv);
    if constexpr (k == K / 2) {
      if (upper) *upper = v9_canonical(h);
    }
  });
  return v9_canonical(h);
}

// a thread's run of K coefficients in registers, loaded top first; zeros
// past n (only the last data block checks, a uniform branch)
template <int K>
__device__ __forceinline__ void load_run(const fr* a, uint64_t n, uint64_t base, bool full, fr (&v)[K]) {
  if (full) {
    static_for<0, K>([&](auto j_) {
      constexpr int k = K - 1 - decltype(j_)::value;
      v[k] = fr_load(a + base + k);
    });
  } else {
    static_for<0, K>([&](auto j_) {
      constexpr int k = K - 1 - decltype(j_)::value;
      v[k] = base + k < n ? fr_load(a + base + k) : fr_zero();
    });
  }
}

// launch 1; steps: squares of mu the table block raises (8 for A, then B's);
// halves (division): also the upper-half Horner value of every run and m^(K/2)
template <int K>
__global__ void __launch_bounds__(kScanThreads) lat_runs_kernel(const fr* a, uint64_t n, const fr* x, int neg,
                                                                fr* ws, uint32_t G, int steps, int halves) {
  static_assert(K % 2 == 0, "runs split in two halves");
  const int t = threadIdx.x;
  if (blockIdx.x == 0) {
    // ---- table block: wave 0 raises mu, mu^2, mu^4, ... and publishes each;
    // a lane of the other waves multiplies up its own entries from the bits of
    // their index as the squares appear (wave 1: A_l, A_(l+64), ...; waves 2
    // and 3: B).  No step waits for another's table, so the chain is the
    // squarings and one product, about 21 at K = 20.
    __shared__ uint32_t pw_s[16][9];
    __shared__ int ready;
    const int w = t >> 6, l = t & 63;
    if (t == 0) ready = 0;
    __syncthreads();
    if (w == 0) {
      const fr m = load_m(x, neg);
      if (t == 0) fr_store(ws + kWsM, m);
      const v9 xp = m_rp(m);
      v9 mu = xp;  // m^K R', left to right; K is even, so m^(K/2) precedes the last squaring
      for (int bit = 30 - __builtin_clz(K); bit >= 0; bit--) {
        if (bit == 0 && t == 0) {
          fr o;
          pbd_pack(mu.l, o.l);
          fr_store(ws + kWsHalf, o);
        }
        mu = mul_r(mu, mu);
        if ((K >> bit) & 1) mu = mul_r(mu, xp);
      }
      for (int s = 0; s < steps; s++) {
        if (t == 0) {
#pragma unroll
          for (int i = 0; i < 9; i++) pw_s[s][i] = mu.l[i];
          __hip_atomic_store(&ready, s + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
          fr o;
          pbd_pack(mu.l, o.l);
          fr_store(ws + kWsPw + s, o);
        }
        if (s + 1 < steps) mu = mul_r(mu, mu);
      }
      return;
    }
    const int from = w == 1 ? 0 : 8, nb = w == 1 ? 8 : steps - 8;  // index bits of this table
    const uint64_t tab = w == 1 ? kWsA : kWsB;
    const int cnt = w == 1 ? kScanThreads : (int)G;
    auto square = [&](int s) {  // mu^(2^(from + s)) once wave 0 has it
      while (__hip_atomic_load(&ready, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) <= from + s)
        __builtin_amdgcn_s_sleep(1);
      v9 p;
#pragma unroll
      for (int i = 0; i < 9; i++) p.l[i] = pw_s[from + s][i];
      return p;
    };
    auto put = [&](int j, const v9& v) {
      if (j >= cnt) return;
      fr o;
      pbd_pack(v.l, o.l);
      fr_store(ws + tab + j, o);
    };
    v9 e0;
    unpack_ext(rp_one_fr().l, e0.l);
    for (int s = 0; s < 6 && s < nb; s++) {
      const v9 p = square(s), q = mul_r(e0, p);
      if ((l >> s) & 1) e0 = q;
    }
    if (w != 3) put(l, e0);
    if (nb > 6) {
      v9 e1;
      if (w != 3) {
        e1 = mul_r(e0, square(6));
        put(l + 64, e1);
      }
      if (nb > 7) {
        const v9 p = square(7);
        if (w != 2) put(l + 128, mul_r(e0, p));
        if (w != 3) put(l + 192, mul_r(e1, p));
      }
    }
    return;
  }
  // ---- data block b: the Horner value of each thread's run ----
  const uint32_t b = blockIdx.x - 1;
  v9 row = rows29_make<false>(load_m(x, neg));
  const uint64_t base = ((uint64_t)b * kScanThreads + t) * K;
  const bool full = (uint64_t)(b + 1) * kScanThreads * K <= n;
  fr v[K];
  load_run<K>(a, n, base, full, v);
  // the Horner chain starts after every load is issued (its rows pass through)
  asm volatile("" : "+v"(row.l[0]), "+v"(row.l[1]), "+v"(row.l[2]), "+v"(row.l[3]), "+v"(row.l[4]), "+v"(row.l[5]),
               "+v"(row.l[6]), "+v"(row.l[7]), "+v"(row.l[8])::"memory");
  fr upper;
  const fr L = horner29_inorder<K>(v, rows29_spread(row), halves ? &upper : nullptr);
  const uint64_t r = (uint64_t)b * kScanThreads + t;
  fr_store(ws + kWsL + r, L);
  if (halves) fr_store(ws + kWsL + (uint64_t)kScanThreads * G + r, upper);
}

// a word (stored form) times a pbd word in R'-form, canonical
__device__ __forceinline__ fr mul_word_pbd(const fr& a, const fr& w) {
  v9 x;
  uint32_t f[9];
  split29(a.l, x.l);
  pbd_unpack(w.l, f);
  return v9_canonical(v9_mul<false, false, false>(x, f));
}

// evaluation, launch 2: P_b = B_b sum_t L_(256 b + t) A_t
__global__ void __launch_bounds__(kScanThreads) lat_combine_kernel(fr* ws) {
  __shared__ uint4 l[2][kScanThreads];
  const int t = threadIdx.x;
  const uint32_t b = blockIdx.x;
  fr c = mul_word_pbd(fr_load(ws + kWsL + (uint64_t)b * kScanThreads + t), fr_load(ws + kWsA + t));
  lds_put(l, t, c);
  __syncthreads();
  for (int s = kScanThreads / 2; s > 0; s >>= 1) {
    if (t < s) {
      c = fr_add(c, lds_get(l, t + s));
      lds_put(l, t, c);
    }
    __syncthreads();
  }
  if (t == 0) fr_store(ws + kWsP + b, mul_word_pbd(c, fr_load(ws + kWsB + b)));
}

// evaluation, launch 3: y = sum of the G block values
__global__ void __launch_bounds__(kScanThreads) eval_lat_sum_kernel(const fr* ws, uint32_t G, fr* y) {
  __shared__ uint4 l[2][kScanThreads];
  const int t = threadIdx.x;
  fr v = t < (int)G ? fr_load(ws + kWsP + t) : fr_zero();
  lds_put(l, t, v);
  __syncthreads();
  for (int s = kScanThreads / 2; s > 0; s >>= 1) {
    if (t < s) {
      v = fr_add(v, lds_get(l, t + s));
      lds_put(l, t, v);
    }
    __syncthreads();
  }
  if (t == 0) fr_store(y, v);
}

// division, launch 2: the run suffixes of block b, S_t = sum_(t' >= t) L_t' mu^(t' - t)
// (S_t replaces L_t), and the block value P_b = S_0
__global__ void __launch_bounds__(kScanThreads) div_lat_suffix_kernel(fr* ws) {
  __shared__ uint32_t wt[4][9];
  const int t = threadIdx.x, lane = t & 63;
  const uint64_t r = (uint64_t)blockIdx.x * kScanThreads + t;
  fr pw[7];  // mu^(2^s), loaded once before the steps
#pragma unroll
  for (int s = 0; s < 7; s++) pw[s] = fr_load(ws + kWsPw + s);
  uint32_t f[9];
  pbd_unpack(fr_load(ws + kWsA + 64 - lane).l, f);  // mu^(64 - lane)
  v9 v;
  unpack_ext(fr_load(ws + kWsL + r).l, v.l);
  const fr S = run_suffix(v, f, wt, [&](int s, uint32_t* p) { pbd_unpack(pw[s].l, p); });
  fr_store(ws + kWsL + r, S);
  if (t == 0) fr_store(ws + kWsP + blockIdx.x, S);
}

// division, launch 3: two threads per run, each rescanning half of it in
// place.  Launch block d covers runs [(d mod 2) 128, +128) of launch-1 block
// b = d / 2.  C_b = s at the end of block b = sum_(j >= 0) P_(b+1+j) B_j (one
// product per thread and a sum); the carry at the end of run t is
// S_(t+1) + mu^(255 - t) C_b; the lower half starts from
// s at the middle = H_t + m^(K/2) (that carry).  q_i = s_(i+1),
// s_i = a_i + m s_(i+1).  Block 0 also writes the remainder s_0 = P_0 + M C_0.
// Every thread reads its half-run before writing it, so q may be a.
template <int K>
__global__ void __launch_bounds__(kScanThreads) div_lat_down_kernel(const fr* a, fr* q, uint64_t n, fr* ws,
                                                                    uint32_t G, fr* rem) {
  constexpr int H = K / 2;
  __shared__ uint4 l[2][kScanThreads];
  const int tid = threadIdx.x;
  const uint32_t b = blockIdx.x >> 1;
  const int t = (int)((blockIdx.x & 1) * 128 + (tid >> 1));
  const int upper = tid & 1;
  const uint64_t r = (uint64_t)b * kScanThreads + t;
  const uint64_t base = r * K + (upper ? H : 0);
  fr v[H];
  load_run<H>(a, n, base, (uint64_t)(b + 1) * kScanThreads * K <= n, v);
  v9 row = rows29_make<false>(fr_load(ws + kWsM));
  fr cb = b + 1 + tid < G ? mul_word_pbd(fr_load(ws + kWsP + b + 1 + tid), fr_load(ws + kWsB + tid)) : fr_zero();
  lds_put(l, tid, cb);
  __syncthreads();
  for (int s = kScanThreads / 2; s > 0; s >>= 1) {
    if (tid < s) {
      cb = fr_add(cb, lds_get(l, tid + s));
      lds_put(l, tid, cb);
    }
    __syncthreads();
  }
  cb = lds_get(l, 0);
  if (blockIdx.x == 0 && tid == 0 && rem) {
    const fr p0 = fr_load(ws + kWsP);
    fr_store(rem, G > 1 ? fr_add(p0, mul_word_pbd(cb, fr_load(ws + kWsB + 1))) : p0);
  }
  fr cin = mul_word_pbd(cb, fr_load(ws + kWsA + (kScanThreads - 1 - t)));
  if (t + 1 < kScanThreads) cin = fr_add(cin, fr_load(ws + kWsL + r + 1));
  if (!upper)
    cin = fr_add(fr_load(ws + kWsL + (uint64_t)kScanThreads * G + r), mul_word_pbd(cin, fr_load(ws + kWsHalf)));
  const rows_all m = rows29_spread(row);
  v9 sn;
  split29(cin.l, sn.l);
  static_for<0, H>([&](auto j_) {
    constexpr int k = H - 1 - decltype(j_)::value;
    if (base + k < n) fr_store(q + base + k, k == H - 1 ? cin : v9_canonical(sn));
    if constexpr (k > 0) {
      v9 xv;
      split29(v[k].l, xv.l);
      sn = v9_add(v9_mul_all<false>(sn, m), xv);
    }
  });
}

// run length K: the smallest multiple of 4 that keeps G <= 255 data blocks
static uint32_t lat_run(uint64_t n) {
  const uint64_t per4 = (uint64_t)kLatMaxG * kScanThreads * 4;
  return (uint32_t)(4 * ((n + per4 - 1) / per4));
}
static uint32_t lat_blocks(uint64_t n, uint32_t K) {
  return (uint32_t)((n + (uint64_t)kScanThreads * K - 1) / ((uint64_t)kScanThreads * K));
}
static uint64_t lat_ws_elems(uint64_t n) { return kWsL + 2ull * kScanThreads * lat_blocks(n, lat_run(n)); }

template <template <int> class F, typename... Args>
static void lat_dispatch(uint32_t K, Args... args) {
  switch (K) {
    case 4: F<4>::run(args...); break;
    case 8: F<8>::run(args...); break;
    case 12: F<12>::run(args...); break;
    case 16: F<16>::run(args...); break;
    case 20: F<20>::run(args...); break;
    case 24: F<24>::run(args...); break;
    default: F<28>::run(args...); break;
  }
}
template <int K>
struct LatRuns {
  static void run(dim3 g, hipStream_t s, const fr* a, uint64_t n, const fr* x, int neg, fr* ws, uint32_t G,
                  int steps, int halves) {
    hipLaunchKernelGGL(lat_runs_kernel<K>, g, dim3(kScanThreads), 0, s, a, n, x, neg, ws, G, steps, halves);
  }
};
template <int K>
struct LatDown {
  static void run(dim3 g, hipStream_t s, const fr* a, fr* q, uint64_t n, fr* ws, uint32_t G, fr* rem) {
    hipLaunchKernelGGL(div_lat_down_kernel<K>, g, dim3(kScanThreads), 0, s, a, q, n, ws, G, rem);
  }
};

// B and A need 8 + ceil(log2 G) squares
static int lat_steps(uint32_t G) { return 8 + (G > 1 ? 32 - __builtin_clz(G - 1) : 0); }

static hipError_t evaluate_lat(const fr* a, uint64_t n, const fr* x, fr* y, fr* ws, hipStream_t s) {
  const uint32_t K = lat_run(n), G = lat_blocks(n, K);
  lat_dispatch<LatRuns>(K, dim3(G + 1), s, a, n, x, 0, ws, G, lat_steps(G), 0);
  hipLaunchKernelGGL(lat_combine_kernel, dim3(G), dim3(kScanThreads), 0, s, ws);
  hipLaunchKernelGGL(eval_lat_sum_kernel, dim3(1), dim3(kScanThreads), 0, s, (const fr*)ws, G, y);
  return hipGetLastError();
}

// q <- s_(i+1), rem <- s_0 (if not null) with m = -c (neg) or c; q may be a
static hipError_t div_lat(const fr* a, fr* q, uint64_t n, const fr* c, int neg, fr* rem, fr* ws, hipStream_t s) {
  const uint32_t K = lat_run(n), G = lat_blocks(n, K);
  lat_dispatch<LatRuns>(K, dim3(G + 1), s, a, n, c, neg, ws, G, lat_steps(G), 1);
  hipLaunchKernelGGL(div_lat_suffix_kernel, dim3(G), dim3(kScanThreads), 0, s, ws);
  lat_dispatch<LatDown>(K, dim3(2 * G), s, a, q, n, ws, G, rem);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// entry points used by the C-ABI
// ---------------------------------------------------------------------------

uint64_t scan_scratch_elems(uint64_t n) {
  // the evaluation's m^t table sits between the powers and the scan
  uint64_t a = pfx_scratch_elems(n), b = sfx_scratch_elems(n) + kScanThreads;
  if (n >= kLatMin && n <= kLatMax && b < lat_ws_elems(n)) b = lat_ws_elems(n);
  return a > b ? a : b;
}

uint64_t grand_product_scratch_elems(uint64_t n) { return pfx_scratch_elems(n); }

hipError_t grand_product(fr* inout, fr* incl_out, uint64_t n, fr* scratch, hipStream_t s) {
  // in one buffer the exclusive products stay: the sweep stores an element's
  // inclusive product after its exclusive one
  if (incl_out == inout) incl_out = nullptr;
  return prefix_product<false>(inout, inout, incl_out, n, scratch, s);
}

// the scan of a division by X + c (neg) or an evaluation and division at x:
// q[i] = s_{i+1}, *total = s_0
static hipError_t divide(const fr* a, fr* q, uint64_t n, const fr* x, int neg, fr* total, fr* scratch,
                         hipStream_t s) {
  if (n >= kLatMin && n <= kLatMax) return div_lat(a, q, n, x, neg, total, scratch, s);
  fr* pw = scratch;
  const int np = sfx_pw_count(n);
  fr* mutab = scratch + np;  // mu^t for the run suffixes, when there is a level above
  const bool tab = n > (uint64_t)kSeg;
  hipLaunchKernelGGL(sfx_powers_kernel, dim3(1), dim3(tab ? 128 : 64), 0, s, x, neg, pw, sfx_pw_first(n),
                     tab ? mutab : nullptr, kLgPer);
  return suffix_scan(a, q, n, pw, total, mutab + kScanThreads, s, pw_ext(pw, np), tab ? mutab : nullptr);
}

hipError_t div_linear(fr* inout, uint64_t n, const fr* c, fr* rem, fr* scratch, hipStream_t s) {
  return divide(inout, inout, n, c, 1, rem, scratch, s);
}

hipError_t evaluate(const fr* coeffs, uint64_t n, const fr* x, fr* y, fr* scratch, hipStream_t s) {
  if (n >= kLatMin && n <= kLatMax) return evaluate_lat(coeffs, n, x, y, scratch, s);
  fr* pw = scratch;
  const int np = sfx_pw_count(n);
  // the reduce's factors m^t (t < 256) as a table beside the powers
  fr* mt = scratch + np;
  hipLaunchKernelGGL(sfx_powers_kernel, dim3(1), dim3(128), 0, s, x, 0, pw, sfx_pw_first(n), mt, 0);
  return suffix_scan(coeffs, nullptr, n, pw, y, mt + kScanThreads, s, pw_ext(pw, np), mt);
}

// one scan for an evaluation + division pair: q(X) = (p(X) - p(z)) / (X - z)
// (q[n-1] = 0) and y = p(z); the suffix s_i = a_i + z s_{i+1} gives both
hipError_t eval_div(const fr* in, fr* q, uint64_t n, const fr* z, fr* y, fr* scratch, hipStream_t s) {
  return divide(in, q, n, z, 0, y, scratch, s);
}

}  // namespace pl
