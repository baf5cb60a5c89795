// Small transforms: one element per lane.
//
// The pass kernels (ntt_pass.hpp) hold eight elements per lane, so a lane
// works through some 23 products one after the other and a transform of 2^16
// elements occupies 128 waves of the 1024 that the chip's SIMDs could each take;
// below about 2^18 elements their time is that chain of products, not the
// chip's rate.  Here a lane holds one element and a column of M' = 2^m points
// (4 <= m <= 9) is one workgroup or part of one: m / 2 radix-4 steps (a
// radix-2 step first when m is odd), each one exchange through LDS and one
// product per lane.  A quad of lanes holds the four inputs x_q of a radix-4
// step; lane k forms its output with the twiddle that follows,
//
//   z_k = t_k (x_0 + (-1)^k x_2) + t_k i^k (x_1 + (-1)^k x_3),
//
// the sums by quad permutes of the limbs (DPP) and the two products with one
// reduction (dual29_dev, 234 multiply-adds): one chain of about 280 VALU
// instructions per two stages, against 107-196 per product and 23 products per
// six stages.  All factors come from one table of w_N^e, e < N, pbd words of
// w R' mod r (inverse: index N - e); the last step of the last pass takes its
// own four pairs, which carry 2^-lg for the inverse.
//
// lg <= kLaneOne: one launch.  Above: two, M'0 = 2^ceil(lg/2) columns at stride
// N / M'0 into the caller's scratch as 256-bit words (not reduced; the step's
// product centres its last Montgomery digit and adds r, mont29_word) with the
// twiddle w_N^(J kappa),
// then contiguous rows in natural order.  Against the pass kernels, one forward
// transform in a stream of calls: 2^5 13.2 -> 5.2 us, 2^9 25.1 -> 9.3, 2^12 30.8
// -> 10.4, 2^14 42.1 -> 11.1, 2^16 46.0 -> 14.9, 2^18 58.0 -> 44.6 (before, with
// the passes of then; pl_internal.hpp has both forms as they are now).
//
// Bounds: inputs are plain digits in [0, 2^29), so the sums have |l| < 2^30;
// values: a caller's 2^256 < 2.21 r makes the first sums 4.42 r each and the
// step's result within (-1.126 r, 0.126 r), later steps within (-1.07 r,
// 0.07 r) (x w / 2^261 < 0.01415 |x| for w < r), a stored word in (0.43 r,
// 1.57 r).
#include <type_traits>

#include "ntt_pass.hpp"

namespace pl {

// the limb of lane CTRL's choice within the quad
template <int P0, int P1, int P2, int P3>
__device__ __forceinline__ uint32_t quad(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, P0 | P1 << 2 | P2 << 4 | P3 << 6, 0xf, 0xf, true);
}

// log2 radix of step s and log2 size of its sub-problems, for 2^m points
constexpr int lane_lr(int m, int s) { return (m & 1) && s == 0 ? 1 : 2; }
constexpr int lane_mu(int m, int s) { return (m & 1) ? (s == 0 ? m : m - 1 - 2 * (s - 1)) : m - 2 * s; }

// position in the column of the element that lane tau holds in a step of
// radix 2^lr on sub-problems of 2^mu points: the radix's inputs are adjacent lanes
__device__ __forceinline__ uint32_t lane_pos(uint32_t tau, int mu, int lr) {
  const uint32_t q = tau & ((1u << lr) - 1), rest = tau >> lr;
  const uint32_t j = rest & ((1u << (mu - lr)) - 1), sub = rest >> (mu - lr);
  return (sub << mu) + (q << (mu - lr)) + j;
}

constexpr int kLaneMaxM = 9;  // the largest column that lane_args asks for
static_assert(kLaneOne == kLaneMaxM && (kLaneMaxLg + 1) / 2 <= kLaneMaxM, "lane_dispatch has every column size");
constexpr int lane_threads(int m) { return 1 << (m > 8 ? m : 8); }

template <int m, bool LAST>
__device__ __forceinline__ void ntt_lane_body(const LaneArgs& a, const uint32_t blk) {
  constexpr int T = lane_threads(m);
  constexpr int C = T >> m;  // columns per workgroup
  constexpr int LGC = C == 1 ? 0 : 8 - m;
  constexpr int NS = (m + 1) / 2;
  __shared__ uint3 ex[2][3][T];  // two exchange buffers: one barrier per step

  const uint32_t tid = threadIdx.x;
  const uint32_t c = (tid >> 2) & (C - 1);
  const uint32_t tau = (tid & 3) | ((tid >> (2 + LGC)) << 2);
  const uint32_t lg = a.lgN;
  const uint32_t nmask = (1u << lg) - 1;
  const uint32_t lgL = lg - m;  // log2 lines per polynomial
  const uint64_t line_of = (uint64_t)blk * C + c;
  // lanes beyond the launch's lines work on its last line and store nothing
  const uint64_t line = line_of < a.nlines ? line_of : a.nlines - 1;
  uint64_t poly;
  uint32_t lp;
  if (LAST && a.lgI) {
    poly = line & ((1ull << a.lgI) - 1);
    lp = (uint32_t)(line >> a.lgI);
  } else {
    poly = line >> lgL;
    lp = (uint32_t)(line & ((1ull << lgL) - 1));
  }
  auto lin = [&](uint32_t e) {  // w_N^(+-e)
    return fr_load(a.lin + ((a.inverse ? 0u - e : e) & nmask));
  };
  // twiddles of step s for this lane, not those after the pass
  auto twiddle = [&](auto s_, fr& w1, fr& w2) {
    constexpr int s = decltype(s_)::value, mu = lane_mu(m, s), lr = lane_lr(m, s);
    const uint32_t k = tau & ((1u << lr) - 1), j = (tau >> lr) & ((1u << (mu - lr)) - 1);
    w1 = lin((j * k) << (lg - mu));
    if constexpr (lr == 2) w2 = lin((k * (j + (1u << (mu - 2)))) << (lg - mu));
  };

  fr w1, w2;
  twiddle(std::integral_constant<int, 0>(), w1, w2);
  v9 x;
  {
    const uint32_t pos = lane_pos(tau, lane_mu(m, 0), lane_lr(m, 0));
    const uint32_t at = LAST ? (lp << m) + pos : lp + (pos << lgL);
    const fr raw = fr_load(a.in + poly * a.in_pstride + at);
    split29(raw.l, x.l);
    if (!LAST && a.premul) {
      uint32_t w[9];
      pbd_unpack(fr_load(a.premul + (((poly & a.pm_mask) << lg) + at)).l, w);
      x = v9_mul<false, false, false>(x, w);
    }
  }
  // kappa, the output index of this lane's last element: its position's
  // digits reversed
  uint32_t kappa = 0;
  {
    const uint32_t pos = tau;  // lane_pos of the last step
    int hi = m, sh = 0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const int lr = lane_lr(m, s);
      hi -= lr;
      kappa |= ((pos >> hi) & ((1u << lr) - 1)) << sh;
      sh += lr;
    }
  }
  static_for<0, NS>([&](auto s_) {
    constexpr int s = decltype(s_)::value, lr = lane_lr(m, s);
    constexpr bool word = !LAST && s + 1 == NS;  // this step's result is stored between launches
    uint32_t f1[9], f2[9];
    pbd_unpack(w1.l, f1);
    if constexpr (lr == 2) pbd_unpack(w2.l, f2);
    // the next step's factors, in flight during this step's product
    if constexpr (s + 2 < NS) {
      twiddle(std::integral_constant<int, s + 1>(), w1, w2);
    } else if constexpr (s + 1 < NS) {
      if constexpr (LAST) {
        const fr* f = a.post ? a.post + 2 * (lp + (kappa << lgL)) : a.fin + 2 * (tau & 3);
        w1 = fr_load(f);
        w2 = fr_load(f + 1);
      } else {
        // w_N^(J kappa), and times i^k
        w1 = lin(lp * kappa);
        w2 = lin(lp * kappa + ((tau & 3) << (lg - 2)));
      }
    }
    v9 u, v;
    if constexpr (lr == 1) {
      const uint32_t neg = 0u - (tau & 1);
#pragma unroll
      for (int i = 0; i < 9; i++) u.l[i] = quad<0, 0, 2, 2>(x.l[i]) + ((quad<1, 1, 3, 3>(x.l[i]) ^ neg) - neg);
      if constexpr (word) mont29_word_dev(u.l, f1, x.l);
      else x = v9_mul<false, false, false>(u, f1);
    } else {
      // lanes 0, 1: x_q + x_(q+2); lanes 2, 3: x_(q-2) - x_q
      const uint32_t neg = 0u - ((tau >> 1) & 1);
      uint32_t p[9];
#pragma unroll
      for (int i = 0; i < 9; i++) p[i] = quad<2, 3, 0, 1>(x.l[i]) + ((x.l[i] ^ neg) - neg);
#pragma unroll
      for (int i = 0; i < 9; i++) {
        u.l[i] = quad<0, 2, 0, 2>(p[i]);
        v.l[i] = quad<1, 3, 1, 3>(p[i]);
      }
      dual29_dev<word>(u.l, f1, v.l, f2, x.l);
    }
    if constexpr (s + 1 < NS) {
      const uint32_t wr = (c << m) + lane_pos(tau, lane_mu(m, s), lr);
      const uint32_t rd = (c << m) + lane_pos(tau, lane_mu(m, s + 1), lane_lr(m, s + 1));
      uint3(*const b)[T] = ex[s & 1];
#pragma unroll
      for (int h = 0; h < 3; h++) b[h][wr] = make_uint3(x.l[3 * h], x.l[3 * h + 1], x.l[3 * h + 2]);
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 3; h++) {
        const uint3 g = b[h][rd];
        x.l[3 * h] = g.x;
        x.l[3 * h + 1] = g.y;
        x.l[3 * h + 2] = g.z;
      }
    }
  });
  if (line_of >= a.nlines) return;
  if constexpr (LAST) {
    const uint32_t lgI = a.lgI;
    fr* const dst = a.out + ((poly >> lgI) << (lg + lgI)) + (poly & ((1ull << lgI) - 1));
    fr_store(dst + ((uint64_t)(lp + (kappa << lgL)) << lgI), v9_canonical(x));
  } else {
    fr o;
    join29(x.l, o.l);
    fr_store(a.out + (poly << lg) + lp + (kappa << lgL), o);
  }
}

template <int m, bool LAST>
__global__ void __launch_bounds__(lane_threads(m), 4) ntt_lane_kernel(LaneArgs a) {
  ntt_lane_body<m, LAST>(a, blockIdx.x);
}

// Ragged form, as ntt_pass_ragged_kernel: one launch for the columns of many
// transforms, of one column size; directions mix, the factors' index has it.
template <int m, bool LAST>
__global__ void __launch_bounds__(lane_threads(m), 4)
    ntt_lane_ragged_kernel(const LaneArgs* __restrict__ segs, const uint32_t* __restrict__ seg_block0, uint32_t nsegs) {
  const uint32_t b = blockIdx.x;
  uint32_t lo = 0, hi = nsegs - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (seg_block0[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  ntt_lane_body<m, LAST>(segs[lo], b - seg_block0[lo]);
}

uint32_t lane_blocks(int m, uint64_t nlines) {
  const int lgC = m >= 8 ? 0 : 8 - m;
  return (uint32_t)((nlines + (1u << lgC) - 1) >> lgC);
}

// f(m, last) as compile-time values
template <class F>
static void lane_dispatch(int m, bool last, F f) {
  auto both = [&](auto m_) {
    if (last) f(m_, std::true_type());
    else f(m_, std::false_type());
  };
  switch (m) {
    case 4: f(std::integral_constant<int, 4>(), std::true_type()); break;
    case 5: both(std::integral_constant<int, 5>()); break;
    case 6: both(std::integral_constant<int, 6>()); break;
    case 7: both(std::integral_constant<int, 7>()); break;
    case 8: both(std::integral_constant<int, 8>()); break;
    default: both(std::integral_constant<int, kLaneMaxM>()); break;
  }
}

static void launch_lane_m(int m, bool last, const LaneArgs& a, hipStream_t s) {
  lane_dispatch(m, last, [&](auto m_, auto last_) {
    constexpr int M = decltype(m_)::value;
    hipLaunchKernelGGL((ntt_lane_kernel<M, decltype(last_)::value>), dim3(lane_blocks(M, a.nlines)),
                       dim3(lane_threads(M)), 0, s, a);
  });
}

void launch_lane_ragged(int m, bool last, const LaneArgs* segs, const uint32_t* seg_block0, uint32_t nsegs,
                        uint32_t nblocks, hipStream_t s) {
  lane_dispatch(m, last, [&](auto m_, auto last_) {
    constexpr int M = decltype(m_)::value;
    hipLaunchKernelGGL((ntt_lane_ragged_kernel<M, decltype(last_)::value>), dim3(nblocks), dim3(lane_threads(M)), 0, s,
                       segs, seg_block0, nsegs);
  });
}

// fin[dir][k] = (s, s i^(+-k)) in the factors' form; ii[dir] = i^(+-1) = w_256^(+-64)
__global__ void lane_fin_kernel(fr* fin, const fr* w256, const fr* w256i, fr c32, fr n_inv32) {
  const int k = threadIdx.x & 3, dir = threadIdx.x >> 2;
  if (threadIdx.x >= 8) return;
  const fr s = dir ? n_inv32 : c32;
  fr o;
  to_pbd(s.l, o.l);
  fr_store(fin + 8 * dir + 2 * k, o);
  const fr v = fr_mul(s, fr_load((dir ? w256i : w256) + 64 * k));
  to_pbd(v.l, o.l);
  fr_store(fin + 8 * dir + 2 * k + 1, o);
}

hipError_t lane_tables(Domain& d, fr* fin, hipStream_t s) {
  auto dev = [](const host::fr64& h) {
    fr f;
    memcpy(f.l, h.l, 32);
    return f;
  };
  const host::fr64 c32 = host::from_u64(32);
  d.lane_fin = fin;
  hipLaunchKernelGGL(lane_fin_kernel, dim3(1), dim3(64), 0, s, fin, (const fr*)d.inner_fwd, (const fr*)d.inner_inv,
                     dev(c32), dev(host::mul(d.n_inv, c32)));
  return hipGetLastError();
}

// one thread per output index i; its last digit k is i's top two bits
__global__ void __launch_bounds__(256) lane_post_kernel(const fr* f, fr* post, const fr* w256i, fr n_inv32, uint32_t lg) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >> lg) return;
  const fr s = fr_mul(fr_load(f + i), n_inv32);
  const fr v = fr_mul(s, fr_load(w256i + 64 * (i >> (lg - 2))));
  fr o;
  to_pbd(s.l, o.l);
  fr_store(post + 2 * i, o);
  to_pbd(v.l, o.l);
  fr_store(post + 2 * i + 1, o);
}

hipError_t lane_post_table(const Domain& d, const fr* f, fr* post, hipStream_t s) {
  fr n_inv32;
  const host::fr64 h = host::mul(d.n_inv, host::from_u64(32));
  memcpy(n_inv32.l, h.l, 32);
  hipLaunchKernelGGL(lane_post_kernel, dim3(((1u << d.lg) + 255) / 256), dim3(256), 0, s, f, post,
                     (const fr*)d.inner_inv, n_inv32, (uint32_t)d.lg);
  return hipGetLastError();
}

bool lane_form(const Domain& d, const NttCall& c) {
  const uint64_t n = (uint64_t)c.npoly << d.lg;
  // One launch stores outputs while other workgroups still read.  In place each
  // reads its polynomials before it stores them; an output that lies over its
  // input in another way goes to the passes, which from 2^7 points on read all
  // of the input first.
  if (d.lg <= kLaneOne && !c.premul && !(c.in == c.out && c.in_pstride == 1ull << d.lg && !c.lgI) &&
      ranges_meet(c.in, c.in_pstride * (c.npoly - 1) + (1ull << d.lg), c.out, n))
    return false;
  return d.lane_lin && (n <= 1ull << 18 || (d.lg > 12 && n < 1ull << 19));
}

int lane_args(const Domain& d, const NttCall& c, LaneArgs (&a)[2], int (&m)[2]) {
  const int lg = d.lg;
  const bool one = lg <= kLaneOne;
  memset(a, 0, sizeof(a));
  a[0].lin = d.lane_lin;
  a[0].fin = d.lane_fin + (c.inverse ? 8 : 0);
  a[0].lgN = lg;
  a[0].lgI = c.lgI;
  a[0].inverse = c.inverse;
  a[0].in = c.in;
  a[0].in_pstride = c.in_pstride;
  a[0].pm_mask = c.pm_mask;
  a[0].out = c.out;
  a[0].post = c.post;
  m[0] = one ? lg : (lg + 1) / 2;
  a[0].nlines = (uint64_t)c.npoly << (lg - m[0]);
  if (one) return 1;
  a[1] = a[0];
  a[0].premul = c.premul;
  a[0].out = c.tmp;
  a[0].post = nullptr;
  m[1] = lg - m[0];
  a[1].in = c.tmp;
  a[1].in_pstride = 1ull << lg;
  a[1].nlines = (uint64_t)c.npoly << m[0];
  return 2;
}

hipError_t lane_launch(const Domain& d, const NttCall& c, hipStream_t s) {
  if (d.lg <= kLaneOne ? c.premul != nullptr : !c.tmp) return hipErrorInvalidValue;  // one launch: the caller multiplies first
  LaneArgs a[2];
  int m[2];
  const int np = lane_args(d, c, a, m);
  for (int p = 0; p < np; p++) launch_lane_m(m[p], p == np - 1, a[p], s);
  return hipGetLastError();
}

}  // namespace pl
