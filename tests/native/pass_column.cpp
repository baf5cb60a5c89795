// Host model of one column of an NTT pass (csrc/ntt_pass.hpp, ntt_pass_body) and
// of one element of the permutation terms (csrc/ops.hip, perm_terms_at) in the
// kernels' sequence of operations, on the fr29.hpp functions that state their
// products, with every bound they rely on checked:
//   * each limb of a sum or difference fits a signed 32-bit integer, but for the
//     one sum of eight that zero_bias brings back;
//   * a rows29 product with one Montgomery digit has limbs within 2^30;
//   * each product column fits a signed 64-bit accumulator at every term;
//   * words between passes join from plain digits and lie in (0.06 r, 1.94 r);
//     the last pass's values before the final subtraction in [0, 1.01 r).
#include <stdint.h>
#include <string.h>

#include "fr29.hpp"

using namespace pl;

namespace {

int g_bad = 0;
const __int128 kLim = ((__int128)1) << 63;

struct V {
  int64_t l[9];
};

V from_u(const uint32_t* b) {
  V v;
  for (int i = 0; i < 9; i++) v.l[i] = (int32_t)b[i];
  return v;
}
void check32(const V& v) {
  for (int i = 0; i < 9; i++)
    if (v.l[i] < INT32_MIN || v.l[i] > INT32_MAX) g_bad++;
}
void to_u(const V& v, uint32_t* u) {
  check32(v);
  for (int i = 0; i < 9; i++) u[i] = (uint32_t)v.l[i];
}
V add(const V& a, const V& b) {
  V s;
  for (int i = 0; i < 9; i++) s.l[i] = a.l[i] + b.l[i];
  return s;
}
V sub(const V& a, const V& b) {
  V s;
  for (int i = 0; i < 9; i++) s.l[i] = a.l[i] - b.l[i];
  check32(s);
  return s;
}
void bfly(V& a, V& b, bool wide = false) {
  const V s = add(a, b);
  b = sub(a, b);
  a = s;
  if (!wide) check32(a);
}

// a column term by term: acc += x y
void term(__int128& acc, int64_t x, int64_t y) {
  acc += (__int128)x * y;
  if (acc >= kLim || acc < -kLim) g_bad++;
}

// the columns of mont29 / mont29_word (word) beside the 64-bit product; w: signed limbs
void check_mont(const uint32_t* a, const uint32_t* w, bool word) {
  int64_t m[9];
  __int128 acc = 0;
  for (int k = 0; k < 17; k++) {
    const int lo = k > 8 ? k - 8 : 0, hi = k < 8 ? k : 8;
    for (int i = lo; i <= hi; i++) term(acc, (int32_t)a[i], (int32_t)w[k - i]);
    for (int i = lo; i <= hi; i++)
      if (i < k) term(acc, -m[i], r29(k - i));
    int64_t dig = (int64_t)((uint64_t)acc & kMask29);
    if (word && k == 8) dig = (int64_t)(int32_t)sext29((uint32_t)(uint64_t)acc) - (1 << 29);
    if (k <= 8) m[k] = dig;
    acc = (acc - dig) >> 29;
  }
}
template <bool BT>
V mul(const V& x, const uint32_t* w) {
  uint32_t u[9], t[9];
  to_u(x, u);
  check_mont(u, w, false);
  mont29<false, BT>(u, w, t);
  return from_u(t);
}
template <int D, bool BT>
V mul_rows(const V& x, const uint32_t* rows) {
  uint32_t u[9], t[9];
  to_u(x, u);
  if (D == 1)
    for (int i = 0; i < 9; i++)
      if (x.l[i] > (1 << 30) || x.l[i] < -(1 << 30)) g_bad++;
  int64_t m[D];
  __int128 acc = 0;
  for (int k = 0; k < 8 + D; k++) {
    if (k <= 8)
      for (int i = 0; i < 9; i++) term(acc, x.l[i], (int32_t)rows[9 * k + i]);
    for (int j = 0; j < D; j++)
      if (k - j >= 1 && k - j <= 8) term(acc, -m[j], r29(k - j));
    const int64_t dig =
        k >= D && BT ? (int64_t)(int32_t)sext29((uint32_t)(uint64_t)acc) : (int64_t)((uint64_t)acc & kMask29);
    if (k < D) m[k] = dig;
    acc = (acc - dig) >> 29;
  }
  rows29<D, BT>(u, rows, t);
  return from_u(t);
}

const uint32_t kR[8] = {0x00000001u, 0xffffffffu, 0xfffe5bfeu, 0x53bda402u,
                        0x09a1d805u, 0x3339d808u, 0x299d7d48u, 0x73eda753u};

// the kernels' fr_reduce_once
void reduce_once(uint32_t* o) {
  uint32_t d[8];
  int64_t b = 0;
  for (int i = 0; i < 8; i++) {
    const int64_t v = (int64_t)o[i] - kR[i] - b;
    d[i] = (uint32_t)v;
    b = v < 0;
  }
  if (!b) memcpy(o, d, sizeof d);
}

V reduce(const V& v) {
  uint32_t u[9], t[9];
  to_u(v, u);
  reduce_below_2r(u, t);
  if (t[8] >= (1u << 24)) g_bad++;
  return from_u(t);
}
void canonical(const V& v, uint32_t* o) {
  uint32_t t[9];
  to_u(reduce(v), t);
  join29(t, o);
  reduce_once(o);
}

int brev(int v, int bits) {
  int r = 0;
  for (int i = 0; i < bits; i++) r |= ((v >> i) & 1) << (bits - 1 - i);
  return r;
}

// dft_dif: f holds the rows of i, (w_8 + w_8^3) / 2 and (w_8 - w_8^3) / 2
void dft(V* x, int logb, const uint32_t* f) {
  const uint32_t *fi = f, *fa = f + 81, *fb = f + 162;
  if (logb == 1) {
    bfly(x[0], x[1]);
  } else if (logb == 2) {
    bfly(x[0], x[2]);
    bfly(x[1], x[3]);
    x[3] = mul_rows<1, false>(x[3], fi);
    bfly(x[0], x[1]);
    bfly(x[2], x[3]);
  } else if (logb == 3) {
    for (int i = 0; i < 4; i++) bfly(x[i], x[i + 4]);
    bfly(x[0], x[2]);
    bfly(x[1], x[3]);
    bfly(x[0], x[1], true);
    // zero_bias: 32-bit wrap-around of each limb's addition
    for (int i = 0; i < 9; i++)
      if (x[0].l[i] < INT32_MIN || x[0].l[i] >= ((int64_t)1 << 32)) g_bad++;
    x[0].l[0] = (int32_t)((uint32_t)x[0].l[0] ^ (1u << 31));
    for (int i = 1; i < 8; i++) x[0].l[i] = (int32_t)((uint32_t)x[0].l[i] + (4u - (1u << 31)));
    x[0].l[8] = (int32_t)((uint32_t)x[0].l[8] + 4);
    x[3] = mul_rows<1, false>(x[3], fi);
    bfly(x[2], x[3]);
    x[6] = mul_rows<1, false>(x[6], fi);
    bfly(x[4], x[6]);
    bfly(x[5], x[7]);
    x[5] = mul_rows<1, false>(x[5], fa);
    x[7] = mul_rows<1, false>(x[7], fb);
    bfly(x[5], x[7]);
    bfly(x[4], x[5]);
    bfly(x[6], x[7]);
  }
}

}  // namespace

extern "C" {

void t_row(const uint32_t* w, int i, uint32_t* rows) { rows29_row(w, i, rows); }
void t_to_pbd(const uint32_t* w, uint32_t* x) { to_pbd(w, x); }

// One column of M' = 8 2^la points in the kernel's order: point rho1 + A rho2 at
// in[rho1 + A rho2], output k = k2 + 8 k1 at out[k].  f: three D = 1 rows
// tables; inner: 64 D = 2 tables of w_64^e; premul: pbd words per input, or
// null; tw: pbd words per output (intermediate pass) or null (last pass);
// scale: a pbd word (last pass) or null.  Returns the number of broken bounds.
int t_column(int la, const uint32_t* in, const uint32_t* f, const uint32_t* inner, const uint32_t* premul,
             const uint32_t* tw, const uint32_t* scale, uint32_t* out) {
  g_bad = 0;
  const int A = 1 << la, m = 3 + la;
  V Y[8][8];  // [rho1][k2]
  for (int rho1 = 0; rho1 < A; rho1++) {
    V x[8];
    for (int r2 = 0; r2 < 8; r2++) {
      uint32_t a[9];
      split29(in + 8 * (rho1 + A * r2), a);
      x[r2] = from_u(a);
      if (premul) {
        uint32_t w[9];
        pbd_unpack(premul + 8 * (rho1 + A * r2), w);
        x[r2] = mul<false>(x[r2], w);
      }
    }
    dft(x, 3, f);
    if (la > 0) {
      x[0] = reduce(x[0]);
      for (int k2 = 1; k2 < 8; k2++) {
        V& v = x[brev(k2, 3)];
        if (rho1 == 0) v = reduce(v);
        else v = mul_rows<2, false>(v, inner + 81 * ((rho1 * k2) << (6 - m)));
      }
    }
    for (int k2 = 0; k2 < 8; k2++) Y[rho1][k2] = x[brev(k2, 3)];
  }
  for (int k2 = 0; k2 < 8; k2++) {
    V y[8];
    for (int r1 = 0; r1 < A; r1++) y[r1] = Y[r1][k2];
    dft(y, la, f);
    for (int k1 = 0; k1 < A; k1++) {
      const int k = k2 + 8 * k1;
      V v = y[brev(k1, la)];
      check32(v);
      if (tw) {
        uint32_t w[9], u[9], t[9];
        pbd_unpack(tw + 8 * k, w);
        to_u(v, u);
        check_mont(u, w, true);
        mont29_word(u, w, t);
        for (int i = 0; i < 8; i++)
          if (t[i] > kMask29) g_bad++;
        if (t[8] >= (1u << 24)) g_bad++;
        join29(t, out + 8 * k);
      } else {
        if (scale) {
          uint32_t w[9];
          pbd_unpack(scale, w);
          v = mul<false>(v, w);
        }
        canonical(v, out + 8 * k);
      }
    }
  }
  return g_bad;
}

// num and den of one element.  b32: 32 S(beta) mod r; beta, gamma, w0, w1, w[3],
// s[3]: words; shift: the factors of rows29_make<false> (nine of nine digits);
// k29: three pbd words; sk: k = (1, 7, 13) by limb shifts.
int t_perm_terms(const uint32_t* w0, const uint32_t* w1, const uint32_t* beta, const uint32_t* b32,
                 const uint32_t* gamma, const uint32_t* shift, const uint32_t* k29, int sk, const uint32_t* w,
                 const uint32_t* s, uint32_t* num_out, uint32_t* den_out) {
  g_bad = 0;
  uint32_t a[9], b[9], u[9];
  // beta's rows (perm_table_kernel): one product of its digits per row
  uint32_t rows[81];
  unpack_ext(beta, a);
  for (int i = 0; i < 9; i++) {
    const V r = mul<true>(from_u(a), shift + 9 * i);
    for (int j = 0; j < 9; j++) rows[9 * j + i] = (uint32_t)r.l[j];
  }
  // the table entries of w0
  split29(b32, b);
  split29(w0, a);
  const V bw = mul<false>(from_u(a), b);
  uint32_t T[3][8];
  for (int j = 0; j < 3; j++) {
    uint32_t K[9];
    pbd_unpack(k29 + 8 * j, K);
    const V t = mul<true>(bw, K);
    for (int i = 0; i < 8; i++)
      if (t.l[i] < -(1 << 28) || t.l[i] >= (1 << 28)) g_bad++;
    if (t.l[8] < -(1 << 23) || t.l[8] >= (1 << 23)) g_bad++;
    to_u(t, u);
    pbd_pack(u, T[j]);
  }
  auto carry = [](V& v) {  // v9_carry_balanced
    check32(v);
    for (int i = 0; i < 8; i++) {
      const int64_t d = (int32_t)sext29((uint32_t)v.l[i]);
      v.l[i + 1] += (v.l[i] - d) >> 29;
      v.l[i] = d;
    }
    check32(v);
  };
  unpack_ext(gamma, a);
  const V g = from_u(a);
  split29(w1, a);
  const V x1 = from_u(a);
  V num, den, t1, t7;
  for (int j = 0; j < 3; j++) {
    unpack_ext(w + 8 * j, a);
    const V wg = add(from_u(a), g);
    V kt;
    if (!sk || j == 0) {
      uint32_t K[9];
      pbd_unpack(T[j], K);
      kt = mul<true>(x1, K);
      t1 = kt;
    } else if (j == 1) {
      for (int l = 0; l < 9; l++) t7.l[l] = 7 * t1.l[l];
      carry(t7);
      kt = t7;
    } else {
      for (int l = 0; l < 9; l++) kt.l[l] = t7.l[l] + 6 * t1.l[l];
      carry(kt);
    }
    const V nj = add(wg, kt);
    split29(s + 8 * j, a);
    const V dj = add(wg, mul_rows<2, true>(from_u(a), rows));
    check32(nj);
    check32(dj);
    if (j == 0) {
      num = nj;
      den = dj;
    } else {
      to_u(nj, u);
      num = mul<false>(num, u);
      to_u(dj, u);
      den = mul<false>(den, u);
    }
  }
  canonical(num, num_out);
  canonical(den, den_out);
  return g_bad;
}

}  // extern "C"
