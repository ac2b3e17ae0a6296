// pair_table.h -- the radial factor of the short-range pair force as a table over r^2.
//
// The P2P kernels need, per pair at separation d (r = |d|), the factor
//     F(r) = G(r / 2 rs) / max(r, eps)^3,   G(u) = erfc(u) + 2u/sqrt(pi) exp(-u^2)
// (src/fmm.c:834-852, src/remotes.c:14-57), whose product with m d is the force.  F is
// tabulated directly over the squared separation, so that a pair takes no square root, no
// reciprocal and no softening branch: with s = lam^2 r^2 + 2, the row is the exponent of s
// and the leading six mantissa bits (64 rows per octave, equal relative widths, which
// suits a power law), and F is a polynomial in the distance of s from the row's middle.
//
//   * the added 2 keeps s at or above the first row (a particle with itself has d = 0 and
//     a finite F) and puts the first octave at exponent bits 0 (mod 32);
//   * lam^2 = (2^(j+1) - 2) / eps^2, so that r = eps, where F has a kink, is the start of
//     a row; j >= 1 is the smallest for which the first row (s in [2, 2 + 1/32)) resolves
//     the u^3 of G near 0, which is not smooth in s (u at s - 2 = 2: at most kUMin);
//   * rows end with the octave of r = u_end 2 rs, in FP64 at u = 8.7 at most, where they are
//     off by 9e-9 (G = 2e-32); the last one is zero.  (Ending at u = 8 costs: each batch with a pair beyond
//     the table is gone through again; 1M uniform particles 11.6 -> 12.6 ms, 256^3 248 -> 250.)
//
//             rows/octave  row                                   u up to   relative error of F
//   FP32      64           4 floats, cubic in s - s_mid          9.5       2e-7 (u < 1), 4e-7 (u < 3)
//   FP64      64           4 doubles + 4 floats, degree 7        8         1e-15 (u < 1), 2e-15 (u < 2),
//                          in the mantissa's distance                      3e-14 (u < 3)
// (the error of G stays below 1e-7 and 1e-15 of G(0) = 1 everywhere.)  The terms of degree 4
// and more are at most 1e-8 of F where it is a power law, so in the FP64 table their float
// coefficients are worth 3e-16 of F there.  Where G falls as exp(-u^2) they are worth more:
// 6e-13 of F at u = 4 (G = 5e-7), 7e-12 at 6 (2e-15), 3e-10 at 8 (1e-27), where k_p2p_f64 is 3e-14,
// 2e-11 and, by erfc and exp, 3e-14 off.  In the forces they do not
// show: against direct sums in 80 bits over 4,096 particles, mesh as fine as the particles and
// twice as fine, the relative error of all forces is 2.4e-16 and 2.2e-16 (clustered), 4.7e-16 and
// 4.6e-16 (lattice), 4.0e-16 and 3.9e-16 (uniform); by k_p2p_f64 2.7e-16, 2.6e-16, 6.2e-16,
// 5.6e-16, 5.2e-16 and 4.9e-16.  Rows of 56 bytes with degree 4 in double take five times as
// long (they are not 16-byte aligned); a table that ends at u = 6 takes 299 ms instead of 254 at
// 256^3 and 27 instead of 12 for 1M uniform particles, whose batches then hold pairs beyond it.
//
// Plain C++, so that it can be tested on the host.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

namespace photons {

struct PairRow32 {
    float c[4];
};
struct PairRow64 {
    double c[4];
    float h[4];
};
static_assert(sizeof(PairRow32) == 16 && sizeof(PairRow64) == 48, "rows as the kernels read them");

constexpr int kPairBits32 = 6, kPairBits64 = 6;  // rows per octave: 2^bits
// octaves at most (the row index takes the five low exponent bits): the FP64 rows, 3 KB
// per octave, share a workgroup's LDS with the staged particles
constexpr int kPairOctaves = 31;
constexpr double kPairUEnd32 = 9.5, kPairUEnd64 = 8.0, kPairUMost64 = 8.7;
constexpr double kPairUMin32 = 0.06, kPairUMin64 = 3.5e-4;

#ifdef __HIPCC__
#define PAIR_HD __host__ __device__
#else
#define PAIR_HD
#endif

// which rows a softening and split radius take; rows = 0: not covered (no softening, or a
// range of too many octaves) -- the kernels then evaluate the pair force from r
struct PairShape {
    double lam2 = 0, lam = 0;  // s = lam2 r^2 + 2 (FP32: lam is a float's value)
    int octaves = 0, rows = 0; // rows: octaves * 2^bits, then the zero row
};

inline PairShape pair_shape(double eps, double rs, bool f32)
{
    PairShape t;
    if (!(eps > 0.0) || !(rs > 0.0)) return t;
    const double uend = f32 ? kPairUEnd32 : kPairUEnd64, umin = f32 ? kPairUMin32 : kPairUMin64;
    int j = 1;
    while (j < 40 && std::sqrt(2.0 / (std::ldexp(1.0, j + 1) - 2.0)) * eps / (2.0 * rs) > umin) j++;
    const double q = std::ldexp(1.0, j + 1) - 2.0;
    if (f32) {
        t.lam = (double)(float)(std::sqrt(q) / eps);
        t.lam2 = t.lam * t.lam;
    } else {
        t.lam2 = q / (eps * eps);
        t.lam = std::sqrt(t.lam2);
    }
    const double end = uend * 2.0 * rs * t.lam;
    if (!std::isfinite(end) || end > 1e9) return t;
    int e = 0;
    std::frexp(end * end + 2.0, &e);  // end^2 + 2 <= 2^e
    t.octaves = e - 1;
    if (t.octaves < j) t.octaves = j;  // eps beyond the end of the split factor
    if (t.octaves > kPairOctaves) return t;
    t.rows = (t.octaves << (f32 ? kPairBits32 : kPairBits64)) + 1;
    if (!f32) {  // the octave may go on to u = 11.3, where the rows are off by some 1e-7
        const double most = kPairUMost64 * 2.0 * rs * t.lam, s = most * most + 2.0;
        uint64_t b;
        std::memcpy(&b, &s, 8);
        const int row = (int)((uint32_t)(b >> 32) - (1024u << 20)) >> (20 - kPairBits64);
        t.rows = std::min(t.rows, std::max(row + 1, j << kPairBits64) + 1);
    }
    return t;
}

// Row i's polynomial in tau = (s - s_mid) / h, |tau| <= 1, of degree 3 (FP32) or 7 (FP64),
// lowest power first: the Taylor series of F about the middle, by recurrence (one erfc and
// one exp a row), economised to that degree with the Chebyshev polynomials.  With
// x = s - 2 = a + h tau, v = u^2 = kappa x and y = sqrt(x) exp(-kappa x):
//     (a + h tau) y' = h (1/2 - kappa (a + h tau)) y
//     G' = -(2/sqrt(pi)) kappa^(3/2) h y           (d G / d v = -(2/sqrt(pi)) sqrt(v) e^-v)
//     (a + h tau) q' = -3/2 h q,  q = x^(-3/2)     (F = G q beyond eps, G / (lam eps)^3 within)
template <int DEG>
PAIR_HD inline void pair_row(int i, int bits, double lam2, double eps, double rs, double (&c)[DEG + 1])
{
    constexpr int N = 15;  // Taylor terms
    const double scale = ldexp(1.0, 1 + (i >> bits)), w = ldexp(1.0, -bits);
    const double h = 0.5 * w * scale;
    const double a = scale * (1.0 + w * ((i & ((1 << bits) - 1)) + 0.5)) - 2.0;
    const double kappa = 1.0 / (lam2 * (2.0 * rs) * (2.0 * rs));
    const double v = kappa * a, u = sqrt(v), g1 = 1.1283791670955125739;  // 2/sqrt(pi)
    double G[N], f[N];
    G[0] = erfc(u) + g1 * u * exp(-v);
    double y0 = sqrt(a) * exp(-v), ym = 0.0;
    for (int k = 0; k + 1 < N; k++) {
        G[k + 1] = -g1 * kappa * sqrt(kappa) * h * y0 / (k + 1);
        const double y1 = h * ((0.5 - kappa * a - k) * y0 - kappa * h * ym) / (a * (k + 1));
        ym = y0;
        y0 = y1;
    }
    if (a < lam2 * eps * eps) {
        const double x = lam2 * eps * eps, q = 1.0 / (x * sqrt(x));
        for (int k = 0; k < N; k++) f[k] = G[k] * q;
    } else {
        for (int k = 0; k < N; k++) f[k] = 0.0;
        double q = 1.0 / (a * sqrt(a));
        for (int j = 0; j < N; j++) {
            for (int k = 0; j + k < N; k++) f[j + k] += q * G[k];
            q *= -h * (1.5 + j) / (a * (j + 1));
        }
    }
    for (int k = N - 1; k > DEG; k--) {  // tau^k = 2^(1-k) T_k(tau) - lower powers: T_k goes
        double r = f[k];
        for (int j = 1; k - 2 * j >= 0; j++) {
            r *= -(double)((k - 2 * j + 2) * (k - 2 * j + 1)) / (4.0 * j * (k - j));
            f[k - 2 * j] -= r;
        }
    }
    for (int k = 0; k <= DEG; k++) c[k] = f[k];
}

PAIR_HD inline PairRow32 pair_row32(int i, int rows, double lam2, double eps, double rs)
{
    PairRow32 R{};
    if (i >= rows - 1) return R;
    double c[4];
    pair_row<3>(i, kPairBits32, lam2, eps, rs, c);
    const double ih = ldexp(1.0, kPairBits32 - (i >> kPairBits32));  // 1 / h
    double p = 1.0;  // in s - s_mid
    for (int k = 0; k < 4; k++, p *= ih) R.c[k] = (float)(c[k] * p);
    return R;
}

PAIR_HD inline PairRow64 pair_row64(int i, int rows, double lam2, double eps, double rs)
{
    PairRow64 R{};
    if (i >= rows - 1) return R;
    double c[8];
    pair_row<7>(i, kPairBits64, lam2, eps, rs, c);
    double p = 1.0;  // in the mantissa's distance: tau / 2^-(bits + 1)
    for (int k = 0; k < 8; k++, p *= ldexp(1.0, kPairBits64 + 1)) {
        if (k < 4) R.c[k] = c[k] * p;
        else R.h[k - 4] = (float)(c[k] * p);
    }
    return R;
}

// the high word of s from which on the FP64 rows end
inline uint32_t pair_top64(int rows) { return (1024u << 20) + ((uint32_t)(rows - 1) << (20 - kPairBits64)); }

// the table on the host (for tests; the library's is built on the device, row by row)
struct PairTable : PairShape {
    bool valid = false;
    std::vector<PairRow32> r32;
    std::vector<PairRow64> r64;
};

inline PairTable make_pair_table(double eps, double rs, bool f32)
{
    PairTable t;
    static_cast<PairShape &>(t) = pair_shape(eps, rs, f32);
    t.valid = t.rows > 0;
    for (int i = 0; i < t.rows; i++) {
        if (f32) t.r32.push_back(pair_row32(i, t.rows, t.lam2, eps, rs));
        else t.r64.push_back(pair_row64(i, t.rows, t.lam2, eps, rs));
    }
    return t;
}

// the tables evaluated on the host as the kernels do (for tests): F at separation r, in
// units of lam^3
inline float pair_eval32(const PairTable &t, float x /* lam r */)
{
    const float s = std::fma(x, x, 2.0f);
    uint32_t b;
    std::memcpy(&b, &s, 4);
    const uint32_t top = (uint32_t)(128 + t.octaves) << 23;
    if (b > top) b = top;
    const uint32_t m = (b & 0xfffe0000u) | 0x10000u;
    float sc, sm;
    std::memcpy(&sc, &b, 4);
    std::memcpy(&sm, &m, 4);
    const PairRow32 &R = t.r32[(b >> 17) & 0x7ff];
    const float d = sc - sm;
    return std::fma(std::fma(std::fma(R.c[3], d, R.c[2]), d, R.c[1]), d, R.c[0]);
}

inline double pair_eval64(const PairTable &t, double r)
{
    const double s = std::fma(r * r, t.lam2, 2.0);
    uint64_t b;
    std::memcpy(&b, &s, 8);
    const uint32_t hi = (uint32_t)(b >> 32), top = pair_top64(t.rows);
    if (hi >= top) return 0.0;  // the kernels evaluate the factor itself from there on
    const uint64_t xm = ((uint64_t)((hi & 0xfffffu) | 0x3ff00000u) << 32) | (b & 0xffffffffu);
    const uint64_t xc = (uint64_t)((hi & 0xfc000u) | 0x3ff02000u) << 32;
    double x, c;
    std::memcpy(&x, &xm, 8);
    std::memcpy(&c, &xc, 8);
    const double d = x - c;
    const float df = (float)d;
    const PairRow64 &R = t.r64[(hi >> 14) & 0x7ff];
    const float h = std::fma(std::fma(std::fma(R.h[3], df, R.h[2]), df, R.h[1]), df, R.h[0]);
    return std::fma(std::fma(std::fma(std::fma((double)h, d, R.c[3]), d, R.c[2]), d, R.c[1]), d, R.c[0]);
}

}  // namespace photons
