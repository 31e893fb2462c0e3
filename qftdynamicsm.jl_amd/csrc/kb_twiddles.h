// kb_twiddles.h -- exp(-2 pi i k / n), k < n, of every n <= TWIDDLE_MAX, one
// after another, worked out at compile time in pairs of doubles (some 100
// bits, Dekker's products) and rounded once; the quarter turns are exact.
#pragma once

namespace qftkb {

constexpr int TWIDDLE_MAX = 64;

struct DD {
  double h, l;
};
constexpr DD dd_sum(double a, double b) {  // a + b exactly
  const double s = a + b, t = s - a;
  return {s, (a - (s - t)) + (b - t)};
}
constexpr DD dd_add(DD a, DD b) {
  const DD s = dd_sum(a.h, b.h);
  return dd_sum(s.h, s.l + (a.l + b.l));
}
constexpr DD dd_neg(DD a) { return {-a.h, -a.l}; }
constexpr DD dd_mul(DD a, DD b) {
  const double ca = 134217729.0 * a.h, cb = 134217729.0 * b.h, p = a.h * b.h;
  const double ah = ca - (ca - a.h), al = a.h - ah, bh = cb - (cb - b.h), bl = b.h - bh;
  const double e = ((ah * bh - p) + ah * bl + al * bh) + al * bl;
  return dd_sum(p, e + (a.h * b.l + a.l * b.h));
}
constexpr DD dd_div(DD a, double d) {
  const double q = a.h / d;
  const DD r = dd_add(a, dd_neg(dd_mul({q, 0.0}, {d, 0.0})));
  return dd_sum(q, r.h / d);
}
// (aligned for the 16-byte loads of its pairs)
struct alignas(16) TwiddleTable {
  double v[TWIDDLE_MAX * (TWIDDLE_MAX + 1)];  // (re, im) pairs
};
constexpr int twiddle_start(int n) { return n * (n - 1) / 2; }
constexpr TwiddleTable make_twiddles() {
  TwiddleTable t{};
  for (int n = 1; n <= TWIDDLE_MAX; ++n) {
    // one step's cosine and sine by their series, at 1/16 of the angle, which
    // is then doubled four times
    const DD x = dd_div({6.283185307179586477, 2.4492935982947064e-16}, 16.0 * n);
    const DD xx = dd_mul(x, x);
    DD c{1.0, 0.0}, s = x, tc{1.0, 0.0}, ts = x;
    for (int j = 1; j <= 10; ++j) {
      tc = dd_neg(dd_div(dd_mul(tc, xx), (2.0 * j - 1.0) * (2.0 * j)));
      ts = dd_neg(dd_div(dd_mul(ts, xx), (2.0 * j) * (2.0 * j + 1.0)));
      c = dd_add(c, tc);
      s = dd_add(s, ts);
    }
    for (int j = 0; j < 4; ++j) {
      const DD cs = dd_mul(c, s), ss = dd_mul(s, s);
      c = dd_add({1.0, 0.0}, dd_neg(dd_add(ss, ss)));
      s = dd_add(cs, cs);
    }
    DD wc{1.0, 0.0}, ws{0.0, 0.0};
    for (int k = 0; k < n; ++k) {
      const int o = 2 * (twiddle_start(n) + k);
      // (the quarter turns exactly)
      t.v[o] = 4 * k == n || 4 * k == 3 * n ? 0.0 : 2 * k == n ? -1.0 : wc.h;
      t.v[o + 1] = k == 0 || 2 * k == n ? 0.0 : 4 * k == n ? -1.0 : 4 * k == 3 * n ? 1.0 : -ws.h;
      const DD a = dd_add(dd_mul(wc, c), dd_neg(dd_mul(ws, s)));
      ws = dd_add(dd_mul(wc, s), dd_mul(ws, c));
      wc = a;
    }
  }
  return t;
}

}  // namespace qftkb
