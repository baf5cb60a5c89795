// Element-wise Fr operators, batch inversion and the PLONK permutation ratio.
//
//  element-wise   add/sub/mul/div, scalar forms, neg, inv, to/from Montgomery
//                 [function.cuh:14-48; mont_arithmetic.cuh:17-69]
//  batch inverse  out[i] = num[i] / in[i] with x/0 = 0 (the reference's
//                 reciprocal: mont_t.cuh:1117-1126).  Montgomery's trick per
//                 2048-element block, then once more over the block totals,
//                 so one call performs a single field inversion.
//  perm ratio     p_i = prod_j (w_j + beta k_j w^i + gamma) / prod_j (w_j + beta s_j + gamma)
//                 (term shape of zksnark_compute_permutation_constraint.cu:13-14;
//                 the reference builds it from element-wise calls)
//
// The single inversion uses Pornin's optimized binary GCD (fr_inv.hpp) on the
// canonical residue and a Montgomery product with R^3 mod r to return to
// Montgomery form.
#include "pl_internal.hpp"
#include "fr29.hpp"
#include "fr_inv.hpp"

namespace pl {

constexpr int kOpThreads = 256;
// batch inversion: 256 threads x 8 elements per block (the down-sweep keeps
// each thread's eight local prefixes in registers)
constexpr int kOpLgPer = 3;
constexpr int kOpPer = 1 << kOpLgPer;
constexpr int kOpSeg = kOpThreads * kOpPer;

// R^2 and R^3 mod r (R = 2^256)
__host__ __device__ constexpr uint32_t rr_limb(int i) {
  return i == 0 ? 0xf3f29c6du : i == 1 ? 0xc999e990u : i == 2 ? 0x87925c23u : i == 3 ? 0x2b6cedcbu
       : i == 4 ? 0x7254398fu : i == 5 ? 0x05d31496u : i == 6 ? 0x9f59ff11u : 0x0748d9d9u;
}
__host__ __device__ constexpr uint32_t rrr_limb(int i) {
  return i == 0 ? 0x439b73afu : i == 1 ? 0xc62c1807u : i == 2 ? 0x8cf06990u : i == 3 ? 0x1b3e0d18u
       : i == 4 ? 0xc7b5f418u : i == 5 ? 0x73d13c71u : i == 6 ? 0xc8db33e9u : 0x6e2a5bb9u;
}

__device__ __forceinline__ fr const_fr(uint32_t (*f)(int)) {
  fr r;
#pragma unroll
  for (int i = 0; i < 8; i++) r.l[i] = f(i);
  return r;
}

// ---- single inversion ----------------------------------------------------
// Montgomery-form inverse of a (a = x R -> x^-1 R); zero maps to zero.  The
// integer inverse of the canonical value x R comes from the optimized binary
// GCD in fr_inv.hpp (at most 17 rounds of 31 steps),
// run by a whole wave: the four full-width updates of each round go to four
// lanes at once, one code path for the four, stopping once converged
// (about 12 of the 17 rounds for a random input; 70 -> ~34 us against one
// lane).  Call from all lanes of a wave, converged, with a the same on
// every lane (lane 0's is used); every lane returns the inverse.
__device__ fr fr_inv_wave(const fr& a_in) {
  const fr a = fr_reduce_once(a_in);
  fr r;
  inv::inverse_wave(a.l, r.l);  // zero maps to zero
  // r = (xR)^-1 = x^-1 R^-1 ; times R^3 under Montgomery: x^-1 R
  return fr_mul(r, const_fr(rrr_limb));
}

// ---- element-wise ----------------------------------------------------------
enum { OP_ADD = 0, OP_SUB, OP_MUL, OP_DIV, OP_ADD_S, OP_SUB_S, OP_MUL_S, OP_DIV_S, OP_NEG, OP_INV, OP_TO_MONT,
       OP_FROM_MONT };

__global__ void __launch_bounds__(256) vec_op_kernel(int op, const fr* a, const fr* b, fr* out, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  fr x = fr_load(a + i);
  fr r;
  switch (op) {
    case OP_ADD: r = fr_add(x, fr_load(b + i)); break;
    case OP_SUB: r = fr_sub(x, fr_load(b + i)); break;
    case OP_MUL: r = fr_mul(x, fr_load(b + i)); break;
    case OP_ADD_S: r = fr_add(x, fr_load(b)); break;
    case OP_SUB_S: r = fr_sub(x, fr_load(b)); break;
    case OP_MUL_S: r = fr_mul(x, fr_load(b)); break;
    case OP_NEG: r = fr_neg(x); break;
    case OP_TO_MONT: r = fr_mul(x, const_fr(rr_limb)); break;
    default: {  // OP_FROM_MONT: x * 1 (raw)
      fr one_raw = fr_zero();
      one_raw.l[0] = 1;
      r = fr_mul(x, one_raw);
    }
  }
  fr_store(out + i, r);
}

// ---- batch inversion ---------------------------------------------------------
__device__ __forceinline__ void lds_put2(uint4 (*l)[kOpThreads], int t, const fr& v) {
  l[0][t] = make_uint4(v.l[0], v.l[1], v.l[2], v.l[3]);
  l[1][t] = make_uint4(v.l[4], v.l[5], v.l[6], v.l[7]);
}
__device__ __forceinline__ fr lds_get2(uint4 (*l)[kOpThreads], int t) {
  uint4 a = l[0][t], b = l[1][t];
  fr v;
  v.l[0] = a.x; v.l[1] = a.y; v.l[2] = a.z; v.l[3] = a.w;
  v.l[4] = b.x; v.l[5] = b.y; v.l[6] = b.z; v.l[7] = b.w;
  return v;
}

// The batch inversion multiplies in signed radix-2^29 limbs (fr29.hpp) and
// reads every word W as the value W / R' (R' = 2^261, "R'-view"): the product
// P(W1, W2) = W1 W2 / R' is then closed (P of the words of a and b is the word
// of a b), and the R'-view one is the word R' mod r.  Only the single inversion
// and the final words relate to the stored form: a stored word S(x) = x R is
// the R'-view word of x / 32, so a level-0 output P(S(num), inverse of S(x)) =
// 32 S(num / x), and without num the inverse alone is 1024 S(1 / x).  Every
// output is linear in the one field inversion at the top, which absorbs that
// factor (inv_down_kernel's TOP).

// R' mod r: the R'-view one
__device__ __forceinline__ fr rp_one() {
  fr r;
  r.l[0] = 0xffffffbau; r.l[1] = 0x00000045u; r.l[2] = 0x0072d846u; r.l[3] = 0x1a25272eu;
  r.l[4] = 0x5dbeee8bu; r.l[5] = 0xfe2eedcdu; r.l[6] = 0x9eefbe41u; r.l[7] = 0x4d043f42u;
  return r;
}

// A word enters a product as plain 29-bit digits (split29, 17 VALU instructions
// against unpack_ext's 33 for balanced ones): with the other operand's digits
// below 2^30 a column stays below 9 * 2^59 + 8 * 2^58 + 2^35 < 2^62.8.  Only a
// word that is packed or summed as it is takes balanced digits.

// P(a, b) of two words, canonical
__device__ __forceinline__ fr mul_rp(const fr& a, const fr& b) {
  v9 x, y;
  split29(a.l, x.l);
  split29(b.l, y.l);
  return v9_canonical(v9_mul<false, false, false>(x, y.l));
}

__device__ __forceinline__ v9 shfl_xor9(const v9& v, int m) {
  v9 o;
#pragma unroll
  for (int i = 0; i < 9; i++) o.l[i] = (uint32_t)__shfl_xor((int)v.l[i], m);
  return o;
}

// E = the product over the block's other threads of their P (balanced digits,
// |value| < 1.08 r or a 256-bit word), and rest = that over the other waves.
// A lane carries the product of its group of 2^k lanes and of the group less
// itself, and takes its sibling group's: two products per step across the
// wave, no barriers; the four wave products meet in LDS once.  14 products
// per thread, a chain of 9, where an exclusive prefix and an exclusive suffix
// by up- and down-sweep took a chain of 34 through 64 barriers (the
// down-sweep of 2^21 quotients 157 -> 107 us, with the coalesced order below).
__device__ __forceinline__ void block_others(v9& P, v9& E, v9& rest) {
  __shared__ uint32_t wt[4][9];
  const int t = threadIdx.x, w = t >> 6;
  E = shfl_xor9(P, 1);
  P = v9_mul<false, false, true>(P, E.l);
#pragma unroll
  for (int m = 2; m < 64; m <<= 1) {
    const v9 sib = shfl_xor9(P, m);
    E = v9_mul<false, false, true>(E, sib.l);
    P = v9_mul<false, false, true>(P, sib.l);
  }
  if ((t & 63) == 0) {
#pragma unroll
    for (int i = 0; i < 9; i++) wt[w][i] = P.l[i];
  }
  __syncthreads();
  auto wave = [&](int k, v9& v) {
#pragma unroll
    for (int i = 0; i < 9; i++) v.l[i] = wt[(w + k) & 3][i];
  };
  v9 o;
  wave(1, rest);
  wave(2, o);
  rest = v9_mul<false, false, true>(rest, o.l);
  wave(3, o);
  rest = v9_mul<false, false, true>(rest, o.l);
  E = v9_mul<false, false, true>(E, rest.l);
}

// The exclusive prefix product of a and the exclusive suffix product of b
// over the 256 thread values (balanced digits, |value| < 1.1 r): six shuffle
// steps inside the wave, two independent products each, then the wave products
// of the waves before and after.  waves: how many waves hold values other than
// one (a single-block level of at most 64 threads' values skips the meeting).
__device__ __forceinline__ void block_scan2(v9& a, v9& b, const v9& one, int waves) {
  __shared__ uint32_t wa[4][9], wb[4][9];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    v9 oa, ob;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      oa.l[i] = (uint32_t)__shfl_up((int)a.l[i], s);
      ob.l[i] = (uint32_t)__shfl_down((int)b.l[i], s);
    }
    oa = v9_mul<false, false, true>(a, oa.l);
    ob = v9_mul<false, false, true>(b, ob.l);
    if (lane >= s) a = oa;
    if (lane + s < 64) b = ob;
  }
  if (waves > 1) {
    if (lane == 63) {
#pragma unroll
      for (int i = 0; i < 9; i++) wa[w][i] = a.l[i];
    }
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 9; i++) wb[w][i] = b.l[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 9; i++) {
    const uint32_t ua = (uint32_t)__shfl_up((int)a.l[i], 1), ub = (uint32_t)__shfl_down((int)b.l[i], 1);
    a.l[i] = lane > 0 ? ua : one.l[i];
    b.l[i] = lane < 63 ? ub : one.l[i];
  }
  if (waves > 1) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (k < w) a = v9_mul<false, false, true>(a, wa[k]);
      if (k > w) b = v9_mul<false, false, true>(b, wb[k]);
    }
  }
}

// Phase 1: total[b] = product over block b of in[i] (zeros taken as one).
__global__ void __launch_bounds__(kOpThreads) inv_reduce_kernel(const fr* in, uint64_t n, fr* total) {
  constexpr int kOpLgSeg = 8 + kOpLgPer;
  __shared__ uint4 l[2][kOpThreads];
  // order-free product: thread t takes elements b*kOpSeg + 256 k + t (coalesced)
  const uint64_t b0 = (uint64_t)blockIdx.x << kOpLgSeg;
  fr v[kOpPer];
  static_for<0, kOpPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const uint64_t i = b0 + (uint64_t)k * kOpThreads + threadIdx.x;
    fr x = i < n ? fr_load(in + i) : rp_one();
    v[k] = fr_is_zero(x) ? rp_one() : x;
  });
  // pairwise tree in registers: eight products of unpacked words, then the
  // products of products (all limbs normalized digits, so any pair is a valid
  // operand pair)
  v9 p[kOpPer / 2];
  static_for<0, kOpPer / 2>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    v9 x, y;
    split29(v[k].l, x.l);
    split29(v[k + kOpPer / 2].l, y.l);
    p[k] = v9_mul<false, false, false>(x, y.l);
  });
  static_for<0, kOpLgPer - 1>([&](auto s_) {
    constexpr int h = kOpPer / 2 >> (decltype(s_)::value + 1);
    static_for<0, h>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      p[k] = v9_mul<false, false, false>(p[k], p[k + h].l);
    });
  });
  fr acc = v9_canonical(p[0]);
  lds_put2(l, threadIdx.x, acc);
  __syncthreads();
  for (int s = kOpThreads / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      acc = mul_rp(acc, lds_get2(l, threadIdx.x + s));
      lds_put2(l, threadIdx.x, acc);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) fr_store(total + blockIdx.x, acc);
}

// Phase 3: with binv[b] the inverse of block b's product, out[i] = num[i] /
// in[i] (num == nullptr: one); zero inputs give zero.  out may equal in or num.
// The products are order-free, so thread t takes elements b*kOpSeg + 256 k + t
// (coalesced; a run of its own per thread fetched each line four times).
// Local prefixes L_k are kept as pbd words (products with balanced digits; a
// product of two values below 1.3 r lies in (-r, 0.03 r), inside a pbd word).
// TOP: the only block, which also inverts its product: times 2^-5 (level-0
// outputs with num) or 2^-10 (without), i.e. fr_inv_wave(W) times 32 or 1 (see
// the batch-inversion notes above).
template <int LG, bool TOP>
__global__ void __launch_bounds__(kOpThreads) __attribute__((amdgpu_waves_per_eu(TOP ? 1 : 3)))
inv_down_kernel(const fr* in, const fr* num, fr* out, uint64_t n, const fr* binv, int with_num) {
  constexpr int kOpPer = 1 << LG, kOpLgSeg = 8 + LG;
  const int t = threadIdx.x;
  // wave-uniform bases and 32-bit lane offsets: eight 64-bit indices per lane
  // would spill
  const uint64_t b0 = (uint64_t)blockIdx.x << kOpLgSeg;
  const uint32_t rem = (uint32_t)(n - b0 < kOpThreads * kOpPer ? n - b0 : kOpThreads * kOpPer);
  auto live = [&](int k) { return (uint32_t)(k * kOpThreads + t) < rem; };
  auto load_in = [&](int k) { return live(k) ? fr_load(in + b0 + k * kOpThreads + t) : rp_one(); };
  fr e[kOpPer];
  uint32_t zmask = 0;
  // local prefix L_k = x_0 ... x_k (pbd words in e[]); the thread product is
  // L_(kOpPer-1)
  v9 L;
  static_for<0, kOpPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    e[k] = load_in(k);
  });
  static_for<0, kOpPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    if (fr_is_zero(e[k])) {
      zmask |= 1u << k;
      e[k] = rp_one();
    }
    v9 x;
    split29(e[k].l, x.l);
    if constexpr (k == 0) {
      L = x;  // L_0 = x_0 as loaded (below 2^256, beyond a pbd word's range)
    } else {
      // |L_k| < 1.07 r: the product of a value below 1.07 r (or x_0 < 2^256) and
      // x_k < 2^256 lies in (-1.07 r, 0.07 r)
      L = v9_mul<false, false, true>(L, x.l);
      pbd_pack(L.l, e[k].l);
    }
  });
  // inv(L_last) = binv * (the block product over everything outside this
  // thread's elements)
  v9 cur, E, rest;
  block_others(L, E, rest);
  fr b;
  if constexpr (TOP) {
    __shared__ fr cinv;
    if (t < 64) {
      fr z = fr_inv_wave(v9_canonical(v9_mul<false, false, false>(rest, L.l)));
      if (with_num) {
#pragma unroll
        for (int d = 0; d < 5; d++) z = fr_add(z, z);
      }
      if (t == 0) cinv = z;
    }
    __syncthreads();
    b = cinv;
  } else {
    b = fr_load(binv + blockIdx.x);
  }
  split29(b.l, cur.l);
  cur = v9_mul<false, false, false>(cur, E.l);
  // walk back: inv(x_k) = inv(L_k) L_{k-1} (inv(x_0) = inv(L_0));
  // inv(L_{k-1}) = inv(L_k) x_k; each element and numerator is asked for one
  // step ahead, before the result in between is stored
  auto load_num = [&](int k) { return num && live(k) ? fr_load(num + b0 + k * kOpThreads + t) : rp_one(); };
  fr xn = load_in(kOpPer - 1);
  static_for<0, kOpPer>([&](auto k_) {
    constexpr int k = kOpPer - 1 - decltype(k_)::value;
    fr xk = xn;
    const fr nk = load_num(k);
    if constexpr (k > 0) xn = load_in(k - 1);
    __builtin_amdgcn_sched_barrier(0x0002 | 0x0004 | 0x0080);
    v9 inv_k = cur;
    if constexpr (k > 0) {
      uint32_t Lp[9];
      if constexpr (k - 1 == 0) split29(e[0].l, Lp);
      else pbd_unpack(e[k > 1 ? k - 1 : 1].l, Lp);
      inv_k = v9_mul<false, false, false>(cur, Lp);
      pin9(inv_k);  // one product at a time: fewer live temporaries
      pin9(cur);
      // x_k from the original input (one again for zeros)
      if ((zmask >> k) & 1) xk = rp_one();
      uint32_t X[9];
      split29(xk.l, X);
      cur = v9_mul<false, false, false>(cur, X);
      pin9(cur);
      pin9(inv_k);
    }
    if (live(k)) {
      fr r;
      if ((zmask >> k) & 1) {
        r = fr_zero();
      } else {
        if (num) {
          uint32_t N[9];
          split29(nk.l, N);
          inv_k = v9_mul<false, false, false>(inv_k, N);
        }
        r = v9_canonical(inv_k);
      }
      fr_store(out + b0 + k * kOpThreads + t, r);
    }
  });
}

static uint64_t inv_scratch_elems(uint64_t n) {
  uint64_t tot = 1;
  while (n > 1) {
    n = (n + kOpSeg - 1) / kOpSeg;
    tot += 2 * n;
  }
  return tot;
}

// out[i] = num[i] / in[i] (num == nullptr: 1/in[i]); x/0 = 0.  with_num: whether
// the level-0 call has num (sets the factor the single inversion absorbs).
static hipError_t batch_inverse_level(const fr* in, const fr* num, fr* out, uint64_t n, fr* scratch, int with_num,
                                      hipStream_t s) {
  const uint64_t nb = (n + kOpSeg - 1) / kOpSeg;
  fr* tot = scratch;
  fr* tinv = scratch + nb;
  if (nb == 1) {
    // one block: 256 x 2^LG with the smallest LG that covers n (1024 values, in
    // one launch instead of reduce, inversion and down-sweep: 72 -> 58 us, of
    // which the inversion takes 31)
    const dim3 g(1), b(kOpThreads);
    const fr* none = nullptr;
    if (n <= 256) hipLaunchKernelGGL((inv_down_kernel<0, true>), g, b, 0, s, in, num, out, n, none, with_num);
    else if (n <= 512) hipLaunchKernelGGL((inv_down_kernel<1, true>), g, b, 0, s, in, num, out, n, none, with_num);
    else if (n <= 1024) hipLaunchKernelGGL((inv_down_kernel<2, true>), g, b, 0, s, in, num, out, n, none, with_num);
    else hipLaunchKernelGGL((inv_down_kernel<kOpLgPer, true>), g, b, 0, s, in, num, out, n, none, with_num);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(inv_reduce_kernel, dim3((unsigned)nb), dim3(kOpThreads), 0, s, in, n, tot);
  // block totals are never zero (zeros were skipped): invert them as a batch
  hipError_t e = batch_inverse_level(tot, nullptr, tinv, nb, scratch + 2 * nb, with_num, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((inv_down_kernel<kOpLgPer, false>), dim3((unsigned)nb), dim3(kOpThreads), 0, s, in, num, out, n,
                     (const fr*)tinv, with_num);
  return hipGetLastError();
}

static hipError_t batch_inverse(const fr* in, const fr* num, fr* out, uint64_t n, fr* scratch, hipStream_t s) {
  return batch_inverse_level(in, num, out, n, scratch, num ? 1 : 0, s);
}

// ---- permutation ratio ------------------------------------------------------
struct RatioArgs {
  const fr* w[3];
  const fr* s[3];
  const fr* beta;
  const fr* gamma;
  const fr* w0;  // w^i = w0[i & 16383] * w1[i >> 14]
  const fr* w1;
  fr* tab;       // [3][tstride] pbd words of (beta k_j w0[lo]) R' (perm_table_kernel)
  uint32_t* brows;  // rows29 table of beta (perm_table_kernel)
  uint32_t tstride;  // min(n, 16384): the low-window entries in use
  fr k[3];
  fr k29[3];  // pbd words of (32 k_j) R' = 1024 k_j R mod r
  fr* num;
  fr* den;
  uint64_t n;
};

// Terms in signed radix-2^29 limbs (fr29.hpp).  With S(a) = a R (stored form)
// and the product P(x, y) = x y / 2^261:
//   P(S(w0), beta R') = S(beta w0)                (beta R' = 32 S(beta))
//   P(., (32 k) R')   = (beta k w0) R'            (host constant, pbd word)
//     -- once per call for the 16384 low-window entries (perm_table_kernel) --
//   P((beta k w0) R', S(w1)) = S(beta k w^i)      (w^i = w0[lo] w1[hi])
//   rows29(S(s_j), beta) = S(beta s_j)              (beta: the same for all lanes)
// so n_j = S(w_j + gamma + beta k_j w^i) and d_j = S(w_j + gamma + beta s_j)
// exactly, and the two products of three terms each carry 2^-10:
// num = S(n_0 n_1 n_2 / 1024), den = S(d_0 d_1 d_2 / 1024), whose ratio is the
// permutation ratio.  Limbs: the inputs are balanced digits (<= 2^28); the
// three-term sums <= 3 2^28 (products with balanced outputs), so a product of
// two of them stays below 81 2^56 + 2^61 < 2^62.8 per column.
constexpr int kWin = 16384;  // entries of the low window table
constexpr uint64_t kBRows = (81 * sizeof(uint32_t) + sizeof(fr) - 1) / sizeof(fr);  // beta's rows29 table
static uint64_t perm_table_elems(uint64_t n) { return 3 * std::min<uint64_t>(n, kWin) + kBRows; }

// tab[j][lo] = P(P(S(w0[lo]), beta R'), (32 k_j) R') = (beta k_j w0[lo]) R', so
// that P(tab[j][lo], S(w1[hi])) = S(beta k_j w^i)
__global__ void __launch_bounds__(256) perm_table_kernel(RatioArgs a, uint32_t count) {
  const uint32_t lo = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    const v9 r = rows29_make<false>(fr_load(a.beta));
    if (threadIdx.x < 9) {
#pragma unroll
      for (int j = 0; j < 9; j++) a.brows[9 * j + threadIdx.x] = r.l[j];
    }
  }
  if (lo >= count) return;
  fr b32 = fr_load(a.beta);  // beta R' = 32 S(beta)
#pragma unroll
  for (int d = 0; d < 5; d++) b32 = fr_add(b32, b32);
  uint32_t b[9];
  split29(b32.l, b);
  v9 w;
  split29(fr_load(a.w0 + lo).l, w.l);
  const v9 bw = v9_mul<false, false, false>(w, b);
#pragma unroll
  for (int j = 0; j < 3; j++) {
    uint32_t K[9];
    pbd_unpack(a.k29[j].l, K);
    const v9 t = v9_mul<false, false, true>(bw, K);  // within (-1.02 r, 0.02 r): a pbd word
    fr o;
    pbd_pack(t.l, o.l);
    fr_store(a.tab + j * a.tstride + lo, o);
  }
}

// v (nine signed limbs, |v_i| < 2^31) carried to balanced digits, the same
// integer: digits 0..7 in [-2^28, 2^28), the carries into the top limb
__device__ __forceinline__ void v9_carry_balanced(v9& v) {
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const uint32_t d = sext29(v.l[i]);
    v.l[i + 1] += (uint32_t)(((int32_t)v.l[i] - (int32_t)d) >> 29);  // exact
    v.l[i] = d;
  }
}

// num and den of element i (before reduction).  SK: k = (1, 7, 13), the
// reference's coset constants: t = S(beta w^i) is one product and the other
// two terms are 7 t and 13 t by limb shifts.  t has balanced digits
// (|t_i| <= 2^28), so 7 t_i fits a signed limb; carried back to balanced
// digits, 7 t plus 6 t fits again (13 t = 7 t + 6 t); each carried value is
// the same integer, so n_j = w_j + gamma + k_j t keeps the three-term bound.
// beta s_j takes beta as a wave-uniform factor (rows29): 117 VALU instructions
// of about 205, and beta's digits leave the vector registers (131 -> 95,
// five waves per SIMD instead of three; 2^20 rows 104 -> 95 us).
template <bool SK>
__device__ __forceinline__ void perm_terms_at(const RatioArgs& a, uint64_t i, v9& num, v9& den) {
  const uwords B = (uwords)a.brows;
  rows_cols g0 = rows29_open(B);
  v9 gam;
  unpack_ext(fr_load(a.gamma).l, gam.l);
  v9 w1;
  split29(fr_load(a.w1 + (i >> 14)).l, w1.l);
  v9 t1, t7;  // SK: beta w^i, then 7 beta w^i (balanced digits)
#pragma unroll
  for (int j = 0; j < 3; j++) {
    v9 wj, sj;
    unpack_ext(fr_load(a.w[j] + i).l, wj.l);
    const v9 wg = v9_add(wj, gam);
    v9 kt;
    if (!SK || j == 0) {
      uint32_t K[9];
      pbd_unpack(fr_load(a.tab + j * a.tstride + (i & (kWin - 1))).l, K);
      kt = v9_mul<false, false, true>(w1, K);
      if (SK) t1 = kt;
    } else if (j == 1) {
#pragma unroll
      for (int l = 0; l < 9; l++) t7.l[l] = (t1.l[l] << 3) - t1.l[l];
      v9_carry_balanced(t7);
      kt = t7;
    } else {
#pragma unroll
      for (int l = 0; l < 9; l++) kt.l[l] = t7.l[l] + (t1.l[l] << 2) + (t1.l[l] << 1);
      v9_carry_balanced(kt);
    }
    const v9 nj = v9_add(wg, kt);
    split29(fr_load(a.s[j] + i).l, sj.l);
    const v9 dj = v9_add(wg, v9_mul_rows<2, true>(sj, B, g0, B));
    num = j == 0 ? nj : v9_mul<false, false, false>(num, nj.l);  // the first factor needs no product
    den = j == 0 ? dj : v9_mul<false, false, false>(den, dj.l);
  }
}

// ZERO_DEN (grand product): a zero den is stored as num = 0, den = R' mod r,
// and the products of num and den over each run of 8 consecutive elements go
// to rn/rd, in three steps of a tree over the block: the first pairs
// neighbouring lanes (num on the even one, den on the odd one), the next two
// take their pairs through LDS into the block's first two waves and then the
// first, so that every lane of a wave that still runs holds a product of its
// own: 7 products of a wave per block.  As butterflies across the run's lanes
// all four waves take all three steps, 12, with a quarter of the lanes useful
// in the last (perm of 2^20 rows, whole call 203 us; so 196: the kernel is
// bound by its products).  Lanes past n carry R' mod r.
template <bool ZERO_DEN, bool SK>
__global__ void __launch_bounds__(256) perm_terms_kernel(RatioArgs a, fr* rn, fr* rd) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if constexpr (!ZERO_DEN) {
    if (i >= a.n) return;
    v9 num, den;
    perm_terms_at<SK>(a, i, num, den);
    fr_store(a.num + i, v9_canonical(num));
    fr_store(a.den + i, v9_canonical(den));
  } else {
    fr nw = rp_one(), dw = rp_one();
    if (i < a.n) {
      v9 num, den;
      perm_terms_at<SK>(a, i, num, den);
      nw = v9_canonical(num);
      dw = v9_canonical(den);
      if (fr_is_zero(dw)) {
        nw = fr_zero();
        dw = rp_one();
      }
      fr_store(a.num + i, nw);
      fr_store(a.den + i, dw);
    }
    const int lane = threadIdx.x & 1;
    v9 p;
    {
      const fr send = (lane & 1) ? nw : dw;
      v9 mine;
      split29(((lane & 1) ? dw : nw).l, mine.l);
      fr o;
#pragma unroll
      for (int j = 0; j < 8; j++) o.l[j] = (uint32_t)__shfl_xor((int)send.l[j], 1);
      uint32_t other[9];
      split29(o.l, other);
      p = v9_mul<false, false, false>(mine, other);
    }
    __shared__ uint32_t wp[2][9][256];
    static_for<0, 2>([&](auto s_) {
      constexpr int s = decltype(s_)::value;
      const int u = threadIdx.x;
      if (u < (256 >> s)) {
#pragma unroll
        for (int j = 0; j < 9; j++) wp[s][j][u] = p.l[j];
      }
      __syncthreads();
      if (u < (128 >> s)) {
        const int from = 4 * (u >> 1) + (u & 1);
        uint32_t q[9];
#pragma unroll
        for (int j = 0; j < 9; j++) {
          p.l[j] = wp[s][j][from];
          q[j] = wp[s][j][from + 2];
        }
        p = v9_mul<false, false, false>(p, q);
      }
    });
    const uint64_t run = (uint64_t)blockIdx.x * 32 + (threadIdx.x >> 1);
    if (threadIdx.x < 64 && run * 8 < a.n) fr_store((threadIdx.x & 1 ? rd : rn) + run, v9_canonical(p));
  }
}

// ---- permutation grand product without a ratio vector -----------------------
// z_i = prod_{j<i} num_j / den_j (exclusive, z_0 = 1) as
//   z_i = [prod_{j<i} num_j] [prod_{j>=i} den_j] / prod_j den_j,
// so the one field inversion multiplies carries only and no element needs an
// inverse of its own.  Up: per block of 2048 elements (256 threads x 8
// consecutive) the thread products of num and den (kept for the down-sweep)
// and the block products, recursively over the block products until one
// block holds them.  Top (one block): the thread scans, the inversion of the
// total den product, and the carries c_b = [prod_{b'<b} num] [prod_{b'>b} den]
// / total for the level below.  Down: each level rescans its blocks from their
// carries; level 0 takes its den suffix inclusive, upper levels exclusive.
// A zero den_j (ratio 0 under x/0 = 0) is stored as num_j = 0, den_j = 1,
// which gives the same z.
// Words are read in the R'-view (the batch-inversion notes above): num_j and
// den_j are stored words S(x), i.e. R'-view words of x / 32; the 32s cancel
// between the two products and the total but for one, which the inverse
// absorbs (32 fr_inv_wave(W) is the R'-view word of 1 / (32 W/R')), so level
// 0 yields the stored words S(z_i).

// the product over the wave's lanes (R'-view, balanced digits), on every lane
__device__ __forceinline__ void wave_product(v9& p) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) p = v9_mul<false, false, true>(p, shfl_xor9(p, m).l);
}

// Up-sweep over one level: thread products of num and den over each
// thread's 8 consecutive elements (tn, td: one per thread of every block, for
// the down-sweep) and the block products (bn, bd).  Half the block's 512
// threads take num and half den: at 2^20 the level is 64 blocks, one wave per
// SIMD and both chains in turn with 256 threads (27.6 us), two waves and half
// the chain with 512 (18.8 us).
constexpr int kUpThreads = 2 * kOpThreads;
__global__ void __launch_bounds__(kUpThreads) gp_up_kernel(const fr* nv, const fr* dv, uint64_t n, fr* tn, fr* td,
                                                           fr* bn, fr* bd) {
  __shared__ uint32_t wt[kUpThreads / 64][9];
  const int t = threadIdx.x & (kOpThreads - 1), w = threadIdx.x >> 6;
  const bool den = w >= 4;
  const uint64_t tid = (uint64_t)blockIdx.x * kOpThreads + t;
  const uint64_t base = tid * kOpPer;
  const fr* src = den ? dv : nv;
  v9 p;
  static_for<0, kOpPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const fr v = base + k < n ? fr_load(src + base + k) : rp_one();
    v9 x;
    split29(v.l, x.l);
    p = k == 0 ? x : v9_mul<false, false, true>(p, x.l);
  });
  fr_store((den ? td : tn) + tid, v9_canonical(p));
  wave_product(p);
  if ((t & 63) == 0) {
#pragma unroll
    for (int i = 0; i < 9; i++) wt[w][i] = p.l[i];
  }
  __syncthreads();
  if (t >= 64) return;  // wave 0 folds num, wave 4 den
#pragma unroll
  for (int k = 1; k < 4; k++) p = v9_mul<false, false, true>(p, wt[w + k]);
  if (t == 0) fr_store((den ? bd : bn) + blockIdx.x, v9_canonical(p));
}

// 32 fr_inv_wave(total): the R'-view word of 1 / (32 total / R'); by a whole
// wave, as fr_inv_wave
__device__ __forceinline__ fr gp_inverse(const fr& total) {
  fr z = fr_inv_wave(total);
#pragma unroll
  for (int d = 0; d < 5; d++) z = fr_add(z, z);
  return z;
}

// Down-sweep over one level (in place: out may be nv).  Thread t of block b
// owns elements base = (256 b + t) 2^LG + k, k < 2^LG, and writes
//   out = c_b pre_t suf_t prod_{k'<k} num [prod_{k'>=k} den (INCL) or k' > k]
// with pre_t / suf_t the products over the block's threads before / after t.
// TOP: a single block; the thread products are formed here and c =
// gp_inverse(total den), or c = one with the total stored to *tot when a
// later launch inverts it.  Otherwise the thread products come from the
// up-sweep (tn, td) and c_b = carry[b], or with nab > 0 block products
// (carry: nab of num, then nab of den) the block multiplies its own,
// [prod_{b'<b} num] [prod_{b'>b} den].
template <int LG, bool INCL, bool TOP>
__device__ __forceinline__ void gp_down_body(const fr* nv, const fr* dv, const fr* tn, const fr* td, uint64_t n,
                                             const fr* carry, uint32_t nab, fr* out, fr* tot, uint32_t blk) {
  constexpr int kPer = 1 << LG;
  __shared__ uint32_t cinv[8];
  const int t = threadIdx.x;
  const uint64_t tid = (uint64_t)blk * kOpThreads + t;
  const uint64_t base = tid * kPer;
  __shared__ uint32_t wc[4][9];
  if constexpr (!TOP) {
    if (nab) {  // first, while few registers are held: each wave's share of c_b
      const uint32_t j = t;
      v9 c;
      split29((j < nab && j != blk ? fr_load(carry + (j < blk ? j : nab + j)) : rp_one()).l, c.l);
      wave_product(c);
      if ((t & 63) == 0) {
#pragma unroll
        for (int i = 0; i < 9; i++) wc[t >> 6][i] = c.l[i];
      }
    }
  }
  v9 one;
  unpack_ext(rp_one().l, one.l);
  // local den suffixes S[k] (pbd words; a product of a value below 1.07 r and
  // one below r lies in (-1.07 r, 0.07 r))
  fr S[kPer];
  v9 acc;
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = kPer - 1 - decltype(k_)::value;
    const fr dw = base + k < n ? fr_load(dv + base + k) : rp_one();
    v9 y;
    if constexpr (k == kPer - 1) unpack_ext(dw.l, y.l);  // packed as it is: balanced digits
    else split29(dw.l, y.l);
    if constexpr (INCL) {
      acc = k == kPer - 1 ? y : v9_mul<false, false, true>(acc, y.l);
      pbd_pack(acc.l, S[k].l);
    } else {
      if constexpr (k == kPer - 1) {
        pbd_pack(one.l, S[k].l);
        acc = y;
      } else {
        pbd_pack(acc.l, S[k].l);
        acc = v9_mul<false, false, true>(acc, y.l);
      }
    }
  });
  // acc: the thread's den product; num's likewise
  v9 pre, suf;
  if constexpr (TOP) {
    static_for<0, kPer>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      const fr nw = base + k < n ? fr_load(nv + base + k) : rp_one();
      v9 x;
      unpack_ext(nw.l, x.l);
      pre = k == 0 ? x : v9_mul<false, false, true>(pre, x.l);
    });
    suf = acc;
  } else {
    unpack_ext(fr_load(tn + tid).l, pre.l);
    unpack_ext(fr_load(td + tid).l, suf.l);
  }
  const v9 mine = suf;
  block_scan2(pre, suf, one, TOP ? (int)((n + 64 * kPer - 1) / (64 * kPer)) : 4);
  v9 c;
  if constexpr (TOP) {
    if (t < 64) {
      // total den product = suf_0 x (thread 0's product): lane 0's value
      // (wave 0 runs it whole for the wave-wide inversion)
      const fr total = v9_canonical(v9_mul<false, false, false>(suf, mine.l));
      fr z;
      if (tot) {
        if (t == 0) fr_store(tot, total);  // inverted by gp_inverse beside the next sweep
        z = rp_one();
      } else {
        z = gp_inverse(total);
      }
      if (t == 0) {
#pragma unroll
        for (int i = 0; i < 8; i++) cinv[i] = z.l[i];
      }
    }
    __syncthreads();
    split29(cinv, c.l);
  } else if (nab) {
#pragma unroll
    for (int i = 0; i < 9; i++) c.l[i] = wc[0][i];  // past block_scan2's barrier
#pragma unroll
    for (int k = 1; k < 4; k++) c = v9_mul<false, false, true>(c, wc[k]);
  } else {
    split29(fr_load(carry + blk).l, c.l);
  }
  v9 cur = v9_mul<false, false, false>(v9_mul<false, false, false>(c, pre.l), suf.l);
  static_for<0, kPer>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const bool live = base + k < n;
    const fr nw = live ? fr_load(nv + base + k) : rp_one();  // read before out[] is written
    if (live) {
      uint32_t sk[9];
      pbd_unpack(S[k].l, sk);
      fr_store(out + base + k, v9_canonical(v9_mul<false, false, false>(cur, sk)));
    }
    if constexpr (k < kPer - 1) {
      uint32_t x[9];
      split29(nw.l, x);
      cur = v9_mul<false, false, false>(cur, x);
    }
  });
}

// bulk levels: three waves per SIMD (the local den suffixes stay in registers)
// inv != nullptr: one more block than the level needs; block 0 (dispatched
// first) has its wave 0 write gp_inverse(total den product) to inv while the
// other blocks sweep (the inverse then multiplies the run carries,
// gp_run_down_kernel).  The total is *tot, or with nab > 0 the product of the
// nab block products of den.
// With nab > 0 (the level above is nab <= kOwnCarry block products) every block
// multiplies its own carry, nine products of a wave, and the launch of the
// level above goes: 2^20 rows 18 + 33 -> 38 us, the whole call 190 -> 178 (173
// to 184 from one card to another); 2^15 79.4, 2^22 544.  With up to 512 block products, two per thread, 2^23
// gained nothing (27 + 65 -> 87 us).
constexpr uint32_t kOwnCarry = kOpThreads;
template <bool INCL>
__global__ void __launch_bounds__(kOpThreads) __attribute__((amdgpu_waves_per_eu(3)))
gp_down_kernel(const fr* nv, const fr* dv, const fr* tn, const fr* td, uint64_t n, const fr* carry, uint32_t nab,
               fr* out, const fr* tot, fr* inv) {
  uint32_t blk = blockIdx.x;
  if (inv) {
    if (blk == 0) {
      if (threadIdx.x < 64) {
        fr total;
        if (nab) {
          v9 p;
          split29((threadIdx.x < nab ? fr_load(carry + nab + threadIdx.x) : rp_one()).l, p.l);
          for (uint32_t j = threadIdx.x + 64; j < nab; j += 64) {
            uint32_t w[9];
            split29(fr_load(carry + nab + j).l, w);
            p = v9_mul<false, false, true>(p, w);
          }
          wave_product(p);
          total = v9_canonical(p);
        } else {
          total = fr_load(tot);
        }
        const fr z = gp_inverse(total);
        if (threadIdx.x == 0) fr_store(inv, z);
      }
      return;
    }
    blk--;
  }
  gp_down_body<kOpLgPer, INCL, false>(nv, dv, tn, td, n, carry, nab, out, nullptr, blk);
}

// the single-block top level
// tot == nullptr: the inversion runs here (no level below the top but the
// runs); otherwise the total is stored for gp_down_kernel's extra block
template <int LG, bool INCL>
__global__ void __launch_bounds__(kOpThreads) gp_top_kernel(const fr* nv, const fr* dv, uint64_t n, fr* out,
                                                             fr* tot) {
  gp_down_body<LG, INCL, true>(nv, dv, nullptr, nullptr, n, nullptr, 0, out, tot, 0);
}

// Level 0: thread = run of 8 consecutive elements with carry c (the num
// products of the runs before it, the den products of those after it, the
// inverse): z_k = c prod_{k'<k} num prod_{k'>=k} den.  No scans.
__global__ void __launch_bounds__(256) gp_run_down_kernel(const fr* nv, const fr* dv, uint64_t n, const fr* carry,
                                                          const fr* inv, fr* out) {
  const uint64_t run = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t base = run * kOpPer;
  if (base >= n) return;
  // local den suffixes (pbd words; products of a value below 1.07 r and one
  // below r lie in (-1.07 r, 0.07 r))
  fr S[kOpPer];
  v9 acc;
  static_for<0, kOpPer>([&](auto k_) {
    constexpr int k = kOpPer - 1 - decltype(k_)::value;
    const fr dw = base + k < n ? fr_load(dv + base + k) : rp_one();
    v9 y;
    if constexpr (k == kOpPer - 1) unpack_ext(dw.l, y.l);  // packed as it is: balanced digits
    else split29(dw.l, y.l);
    acc = k == kOpPer - 1 ? y : v9_mul<false, false, true>(acc, y.l);
    pbd_pack(acc.l, S[k].l);
  });
  v9 cur;
  split29(fr_load(carry + run).l, cur.l);
  if (inv) {
    uint32_t w[9];
    split29(fr_load(inv).l, w);
    cur = v9_mul<false, false, false>(cur, w);
  }
  // four quarters: each quarter's num values are loaded before its outputs
  // are written (out may equal nv), so a thread waits for four loads, not
  // eight, with few values live
  constexpr int Q = kOpPer / 4;
  static_for<0, 4>([&](auto g_) {
    constexpr int k0 = decltype(g_)::value * Q;
    fr nw[Q];
    static_for<0, Q>([&](auto j_) {
      constexpr int j = decltype(j_)::value;
      nw[j] = base + k0 + j < n ? fr_load(nv + base + k0 + j) : rp_one();
    });
    static_for<0, Q>([&](auto j_) {
      constexpr int j = decltype(j_)::value, k = k0 + j;
      if (base + k < n) {
        uint32_t sk[9];
        pbd_unpack(S[k].l, sk);
        fr_store(out + base + k, v9_canonical(v9_mul<false, false, false>(cur, sk)));
      }
      if constexpr (k < kOpPer - 1) {
        uint32_t x[9];
        split29(nw[j].l, x);
        cur = v9_mul<false, false, false>(cur, x);
      }
    });
  });
}

// is there a level above level L of the grand product, which has n values?  More
// than a block's do need one; the runs also from 1025 on, where an up-sweep, and
// the inversion beside the sweep, beat one block that does both in turn with
// eight values per thread (2^14 rows 88.6 -> 78.7 us; not at 2^12).
static bool gp_level_above(int L, uint64_t n) { return n > (uint64_t)(L == 0 ? 4 * kOpThreads : kOpSeg); }

// level sizes of the grand product: the runs of 8 elements (n_1 = ceil(n / 8)),
// then n_{L+1} = ceil(n_L / 2048) while gp_level_above; scratch holds den (n), the
// run products (2 n_1), then per up-swept level the thread products (2 x 256
// per block) and the next level's num and den, then the total and its inverse
static uint64_t gp_scratch_elems(uint64_t n) {
  uint64_t m = (n + kOpPer - 1) / kOpPer;
  uint64_t tot = n + 2 * m + 2;  // + the total den product and its inverse
  for (int L = 0; gp_level_above(L, m); L++) {
    const uint64_t nb = (m + kOpSeg - 1) / kOpSeg;
    tot += 2 * nb * kOpThreads + 2 * nb;
    m = nb;
  }
  return tot;
}

template <bool INCL>
static void gp_top(const fr* nv, const fr* dv, uint64_t n, fr* out, fr* tot, hipStream_t s) {
  const dim3 g(1), b(kOpThreads);
  if (n <= 256) hipLaunchKernelGGL((gp_top_kernel<0, INCL>), g, b, 0, s, nv, dv, n, out, tot);
  else if (n <= 512) hipLaunchKernelGGL((gp_top_kernel<1, INCL>), g, b, 0, s, nv, dv, n, out, tot);
  else if (n <= 1024) hipLaunchKernelGGL((gp_top_kernel<2, INCL>), g, b, 0, s, nv, dv, n, out, tot);
  else hipLaunchKernelGGL((gp_top_kernel<kOpLgPer, INCL>), g, b, 0, s, nv, dv, n, out, tot);
}

uint64_t ops_scratch_elems(uint64_t n) {
  return perm_table_elems(n) + std::max(n + inv_scratch_elems(n), gp_scratch_elems(n));
}

hipError_t vec_op(int op, const fr* a, const fr* b, fr* out, uint64_t n, fr* scratch, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (op == OP_INV) return batch_inverse(a, nullptr, out, n, scratch, s);
  if (op == OP_DIV) return batch_inverse(b, a, out, n, scratch, s);
  if (op == OP_DIV_S) {
    // out = a * (1/b): invert the scalar into scratch, then multiply
    fr* binv = scratch;
    hipError_t e = batch_inverse(b, nullptr, binv, 1, scratch + 1, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(vec_op_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (int)OP_MUL_S, a,
                       (const fr*)binv, out, n);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(vec_op_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, op, a, b, out, n);
  return hipGetLastError();
}

// ---- powers and broadcasts ------------------------------------------------------
// exp_mod: out[i] = a[i]^e, left-to-right square and multiply with the
// exponent uniform over the launch; e = 0 gives one and e = 1 a copy
// (mont_arithmetic.cu:258-273, cpu/mont_arithmetic.cpp:66-81).
__global__ void __launch_bounds__(256) exp_kernel(const fr* a, fr* out, uint64_t n, uint32_t e) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  fr_store(out + i, e == 0 ? fr_one() : fr_pow_u64(fr_load(a + i), e));
}

// gen_sequence: out[i] = x^i (poly_eval_kernel, mont_arithmetic.cu:104-114,
// raises x to each i alone).  Here the head out[0..min(n, 2^14)) is raised
// directly (at most 14 squarings), and every later tile of 2^14 elements is
// the head times one factor: out[(q << 14) + j] = out[j] * x^(q << 14), with
// x^(q << 14) = out[q]^(2^14) (q < 2^14 for n <= 2^28), one product per element.
constexpr uint32_t kSeqLgTile = 14;
__global__ void __launch_bounds__(256) seq_head_kernel(const fr* x, fr* out, uint64_t n0) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n0) return;
  fr_store(out + i, fr_pow_u64(fr_load(x), i));
}
// block b: tile q = b + 1; reads out[q] and out[0..2^14), writes tile q only
__global__ void __launch_bounds__(256) seq_tail_kernel(fr* out, uint64_t n) {
  __shared__ uint4 hq[2];
  const uint64_t q = (uint64_t)blockIdx.x + 1;
  if (threadIdx.x == 0) {
    fr h = fr_load(out + q);
    for (uint32_t k = 0; k < kSeqLgTile; k++) h = fr_sqr(h);
    hq[0] = make_uint4(h.l[0], h.l[1], h.l[2], h.l[3]);
    hq[1] = make_uint4(h.l[4], h.l[5], h.l[6], h.l[7]);
  }
  __syncthreads();
  fr h;
  h.l[0] = hq[0].x; h.l[1] = hq[0].y; h.l[2] = hq[0].z; h.l[3] = hq[0].w;
  h.l[4] = hq[1].x; h.l[5] = hq[1].y; h.l[6] = hq[1].z; h.l[7] = hq[1].w;
  const uint64_t base = q << kSeqLgTile;
  for (uint32_t j = threadIdx.x; j < (1u << kSeqLgTile) && base + j < n; j += blockDim.x)
    fr_store(out + base + j, fr_mul(fr_load(out + j), h));
}

// repeat_to_poly: out[i] = *x (repeat_kernel, mont_arithmetic.cu:214-220)
__global__ void __launch_bounds__(256) repeat_kernel(const fr* x, fr* out, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  fr_store(out + i, fr_load(x));
}

hipError_t exp_mod(const fr* a, fr* out, uint64_t n, uint32_t e, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(exp_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, out, n, e);
  return hipGetLastError();
}

hipError_t gen_sequence(const fr* x, fr* out, uint64_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const uint64_t n0 = std::min<uint64_t>(n, 1ull << kSeqLgTile);
  hipLaunchKernelGGL(seq_head_kernel, dim3((unsigned)((n0 + 255) / 256)), dim3(256), 0, s, x, out, n0);
  if (n > n0) {
    const uint64_t tiles = (n + (1ull << kSeqLgTile) - 1) >> kSeqLgTile;
    hipLaunchKernelGGL(seq_tail_kernel, dim3((unsigned)(tiles - 1)), dim3(256), 0, s, out, n);
  }
  return hipGetLastError();
}

hipError_t repeat_to_poly(const fr* x, fr* out, uint64_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(repeat_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, out, n);
  return hipGetLastError();
}

static RatioArgs ratio_args(const fr* const w[3], const fr* const sg[3], const fr* beta, const fr* gamma,
                            const fr* w0, const fr* w1, const host::fr64 k[3], uint64_t n) {
  RatioArgs a;
  for (int j = 0; j < 3; j++) {
    a.w[j] = w[j];
    a.s[j] = sg[j];
    memcpy(a.k[j].l, k[j].l, 32);
    // (32 k_j) R' = 1024 k_j R: the Montgomery product of k_j R and 1024 R
    const host::fr64 k1024 = host::mul(k[j], host::from_u64(1024));
    fr kk;
    memcpy(kk.l, k1024.l, 32);
    to_pbd(kk.l, a.k29[j].l);
  }
  a.beta = beta;
  a.gamma = gamma;
  a.w0 = w0;
  a.w1 = w1;
  a.tab = nullptr;
  a.brows = nullptr;
  a.tstride = 0;
  a.num = nullptr;
  a.den = nullptr;
  a.n = n;
  return a;
}

// k = (1, 7, 13) in Montgomery form, the coset constants of the miss_ops
// permutation workload (terms of the shape of
// zksnark_compute_permutation_constraint.cu:13-14): the terms kernel then
// forms k_1 t and k_2 t by limb shifts
static bool reference_ks(const host::fr64 k[3]) {
  const uint64_t v[3] = {1, 7, 13};
  for (int j = 0; j < 3; j++) {
    const host::fr64 m = host::from_u64(v[j]);
    if (memcmp(m.l, k[j].l, sizeof(m.l)) != 0) return false;
  }
  return true;
}

// the window tables at the front of scratch (perm_table_elems(n) elements)
static void perm_tables(RatioArgs& a, fr*& scratch, hipStream_t s) {
  const uint32_t count = (uint32_t)std::min<uint64_t>(a.n, kWin);
  a.tab = scratch;
  a.tstride = count;
  scratch += perm_table_elems(a.n);
  a.brows = (uint32_t*)(scratch - kBRows);
  hipLaunchKernelGGL(perm_table_kernel, dim3((count + 255) / 256), dim3(256), 0, s, a, count);
}

hipError_t perm_ratio(const fr* const w[3], const fr* const sg[3], const fr* beta, const fr* gamma,
                      const fr* w0, const fr* w1, const host::fr64 k[3], fr* ratio, uint64_t n, fr* scratch,
                      hipStream_t s) {
  RatioArgs a = ratio_args(w, sg, beta, gamma, w0, w1, k, n);
  perm_tables(a, scratch, s);
  a.num = ratio;
  a.den = scratch;
  if (reference_ks(k))
    hipLaunchKernelGGL((perm_terms_kernel<false, true>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a,
                       nullptr, nullptr);
  else
    hipLaunchKernelGGL((perm_terms_kernel<false, false>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a,
                       nullptr, nullptr);
  // ratio = num / den in place over num
  return batch_inverse(scratch, ratio, ratio, n, scratch + n, s);
}

hipError_t perm_grand_product(const fr* const w[3], const fr* const sg[3], const fr* beta, const fr* gamma,
                              const fr* w0, const fr* w1, const host::fr64 k[3], fr* z, uint64_t n, fr* scratch,
                              hipStream_t s) {
  RatioArgs a = ratio_args(w, sg, beta, gamma, w0, w1, k, n);
  perm_tables(a, scratch, s);
  a.num = z;
  a.den = scratch;
  const uint64_t nr = (n + kOpPer - 1) / kOpPer;
  fr* rn = scratch + n;
  fr* rd = rn + nr;
  if (reference_ks(k))
    hipLaunchKernelGGL((perm_terms_kernel<true, true>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, rn,
                       rd);
  else
    hipLaunchKernelGGL((perm_terms_kernel<true, false>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, rn,
                       rd);
  // levels above the elements: the runs, then block products
  struct Level {
    fr *nv, *dv, *tn, *td;
    uint64_t n;
  } lv[8];
  int top = 0;
  lv[0] = {rn, rd, nullptr, nullptr, nr};
  fr* p = rd + nr;
  while (gp_level_above(top, lv[top].n)) {
    Level& c = lv[top];
    const uint64_t nb = (c.n + kOpSeg - 1) / kOpSeg;
    c.tn = p;
    c.td = p + nb * kOpThreads;
    p += 2 * nb * kOpThreads;
    fr* bn = p;
    fr* bd = p + nb;
    p += 2 * nb;
    hipLaunchKernelGGL(gp_up_kernel, dim3((unsigned)nb), dim3(kUpThreads), 0, s, (const fr*)c.nv, (const fr*)c.dv,
                       c.n, c.tn, c.td, bn, bd);
    lv[++top] = {bn, bd, nullptr, nullptr, nb};
  }
  // carries in place over each level's num (the runs' carries over rn).  With
  // a level between the top and the runs, the first sweep below the top inverts
  // the total den product in an extra block; a top of at most kOwnCarry block
  // products has no launch of its own.
  fr* tot = top > 0 ? p : nullptr;
  fr* inv = top > 0 ? p + 1 : nullptr;
  const bool own = top > 0 && lv[top].n <= kOwnCarry;
  if (!own) gp_top<false>(lv[top].nv, lv[top].dv, lv[top].n, lv[top].nv, tot, s);
  for (int L = top - 1; L >= 0; L--) {
    const Level& c = lv[L];
    const bool first = L == top - 1;
    const unsigned nb = (unsigned)((c.n + kOpSeg - 1) / kOpSeg) + (first ? 1 : 0);
    hipLaunchKernelGGL(gp_down_kernel<false>, dim3(nb), dim3(kOpThreads), 0, s, c.nv, c.dv, c.tn, c.td, c.n,
                       (const fr*)lv[L + 1].nv, first && own ? (uint32_t)lv[top].n : 0u, c.nv, (const fr*)tot,
                       first ? inv : nullptr);
  }
  hipLaunchKernelGGL(gp_run_down_kernel, dim3((unsigned)((nr + 255) / 256)), dim3(256), 0, s, (const fr*)z,
                     (const fr*)scratch, n, (const fr*)rn, (const fr*)inv, z);
  return hipGetLastError();
}

}  // namespace pl
