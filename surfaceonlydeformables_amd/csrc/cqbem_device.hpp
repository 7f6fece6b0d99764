// Device-side math shared by the CQBEM kernels: FP64 complex arithmetic and the
// Laplace-domain elastodynamic kernels in factored form.
//
// The reference evaluates each kernel entry (i,j) separately
// (G_collocation.cu:44-60, H_collocation.cu:45-76, B_trans_collocation.cu:41-58,
// B_angular_collocation.cu:44-63).  Here every kernel is written as a few
// complex scalar coefficients times frequency-independent geometric tensors, so
// one point/frequency evaluation costs two complex exponentials plus ~30 complex
// operations for all four matrices:
//   u_hat  = alpha rh rh^T + beta I
//   p_hat  = (1/4pi) [ h1 rh n^T + h2 (n rh^T + (rh.n) I) + h4 (rh.n) rh rh^T ]
//   b_hat  = t1 (rh n^T + n rh^T) + t2 (rh.n) I
//   b_hat_ijk = u1 (rh_i rh_k n_j + rh_j rh_k n_i) + (u1+u2)(d_jk n_i + d_ik n_j) + u3 d_ij n_k
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "cqbem_math_tables.hpp"

namespace cqbem {

struct cd {
    double x, y;
};

__host__ __device__ inline cd mkc(double a, double b) { return cd{a, b}; }
__host__ __device__ inline cd operator+(cd a, cd b) { return cd{a.x + b.x, a.y + b.y}; }
__host__ __device__ inline cd operator-(cd a, cd b) { return cd{a.x - b.x, a.y - b.y}; }
__host__ __device__ inline cd operator-(cd a) { return cd{-a.x, -a.y}; }
__host__ __device__ inline cd operator*(cd a, cd b) { return cd{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__host__ __device__ inline cd operator*(cd a, double s) { return cd{a.x * s, a.y * s}; }
__host__ __device__ inline cd operator*(double s, cd a) { return cd{a.x * s, a.y * s}; }
__host__ __device__ inline cd &operator+=(cd &a, cd b) {
    a.x += b.x, a.y += b.y;
    return a;
}
__host__ __device__ inline cd &operator-=(cd &a, cd b) {
    a.x -= b.x, a.y -= b.y;
    return a;
}
// a += b * s (complex times real)
__host__ __device__ inline void fma_cr(cd &a, cd b, double s) {
    a.x = fma(b.x, s, a.x);
    a.y = fma(b.y, s, a.y);
}

// Two real values side by side, with component-wise products: one quantity at the two frequencies of the half spectrum
// where s is real (l = 0, and l = L/2 for an even L).
struct rp {
    double x, y;
};
__host__ __device__ inline rp operator+(rp a, rp b) { return rp{a.x + b.x, a.y + b.y}; }
__host__ __device__ inline rp operator-(rp a, rp b) { return rp{a.x - b.x, a.y - b.y}; }
__host__ __device__ inline rp operator*(rp a, rp b) { return rp{a.x * b.x, a.y * b.y}; }
__host__ __device__ inline rp operator*(rp a, double s) { return rp{a.x * s, a.y * s}; }
__host__ __device__ inline rp operator*(double s, rp a) { return rp{a.x * s, a.y * s}; }
__host__ __device__ inline rp &operator+=(rp &a, rp b) { return a = a + b; }
__host__ __device__ inline rp &operator-=(rp &a, rp b) { return a = a - b; }
__host__ __device__ inline void fma_cr(rp &a, rp b, double s) {
    a.x = fma(b.x, s, a.x);
    a.y = fma(b.y, s, a.y);
}
// v + 1 at one frequency, or at both
__host__ __device__ inline cd add_one(cd v, double one) { return cd{v.x + one, v.y}; }
__host__ __device__ inline rp add_one(rp v, double one) { return rp{v.x + one, v.y + one}; }

// ---------------------------------------------------------------------------
// FP64 elementary functions for the kernel arguments.  The CQ exponent
// z = s r / c has Re z >= 0 (the BDF symbols are A-stable, so Re s_l > 0) and
// a moderate imaginary part, which allows an exact Cody-Waite reduction
// (W. J. Cody, W. Waite, "Software Manual for the Elementary Functions", 1980)
// followed by truncated Taylor series (the first omitted terms are below
// 1e-17 relative) whose leading terms are summed with their rounding errors
// carried (Fast2Sum), so e^{-a} stays within 0.65 ulp and sin, cos within
// 0.4 ulp of 1, at about half the instruction count of the library calls.
// Contraction is off inside them: every FMA is written out, so the error
// analysis holds as written.
// ---------------------------------------------------------------------------
constexpr double kLog2e = 1.4426950408889634;         // 1/ln 2
constexpr double kLn2Hi = 0x1.62e42fefa3800p-1;       // ln 2 to 42 bits: k kLn2Hi exact for |k| < 2^11
constexpr double kLn2Lo = 5.497923018708371e-14;      // ln 2 - kLn2Hi
constexpr double kTwoOverPi = 0.6366197723675814;     // 2/pi
constexpr double kPio2A = 0x1.921fb54400000p+0;       // pi/2 to 33 bits: k kPio2A exact for |k| < 2^20
constexpr double kPio2B = 0x1.0b4611a600000p-34;      // next 33 bits of pi/2
constexpr double kPio2C = 2.0222662487959506e-21;     // pi/2 - kPio2A - kPio2B
// |Im z| bound of the exact reduction (|k| < 2^20).  The host rejects jobs whose largest argument
// max|s_l| diam / min(c1, c2) reaches it.
constexpr double kTrigArgMax = 1.0e6;

// e^{-a}, a >= -700.  k = rint(-a / ln 2); f + c = -a - k ln 2 with |f| <= ln2/2 (the k kLn2Hi part
// is exact by Sterbenz); e^(f+c) = (1 + f) + (f^2 p(f) + c (1 + f)) with p the Taylor series of
// (e^f - 1 - f) / f^2 through f^11 (next term < 5e-18); 1 + f is split exactly.  Scaled by 2^k;
// -a is clamped at -740, where the result has underflowed to 0.  With `lo`, what the rounding of the result left out goes
// there (good to 2^-57 of the result).
__host__ __device__ inline double exp_neg(double a, double *lo = nullptr) {
#pragma clang fp contract(off)
    const double t = fmin(fmax(-a, -740.0), 700.0);
    const double k = rint(t * kLog2e);
    const double fh = fma(-k, kLn2Hi, t);
    const double fl = -k * kLn2Lo;
    const double f = fh + fl;
    const double c = (fh - f) + fl;
    double p = 1.0 / 6227020800.0;     // 1/13!
    p = fma(p, f, 1.0 / 479001600.0);  // 1/12!
    p = fma(p, f, 1.0 / 39916800.0);   // 1/11!
    p = fma(p, f, 1.0 / 3628800.0);
    p = fma(p, f, 1.0 / 362880.0);
    p = fma(p, f, 1.0 / 40320.0);
    p = fma(p, f, 1.0 / 5040.0);
    p = fma(p, f, 1.0 / 720.0);
    p = fma(p, f, 1.0 / 120.0);
    p = fma(p, f, 1.0 / 24.0);
    p = fma(p, f, 1.0 / 6.0);
    p = fma(p, f, 0.5);
    const double tail = fma(f * f, p, fma(c, f, c));
    const double s1 = 1.0 + f, e1 = ((1.0 - s1) + f) + tail, m = s1 + e1;
    if (lo) *lo = ldexp((s1 - m) + e1, (int)k);
    return ldexp(m, (int)k);
}

// sin y, cos y for |y| < kTrigArgMax.  k = rint(2y/pi); r + rr = y - k pi/2 to ~1e-30 (three-part
// pi/2, the first two products exact, the subtraction split by TwoSum); sin r through r^17 and
// cos r through r^18 (next terms < 1e-19), first-order in rr; 1 - r^2/2 split exactly.  The
// quadrant k mod 4 then selects and signs them.  With `lo`, lo[0] and lo[1] are what the roundings of s and c left out
// (good to 2^-57).
__host__ __device__ inline void cq_sincos(double y, double *s, double *c, double *lo = nullptr) {
#pragma clang fp contract(off)
    const double k = rint(y * kTwoOverPi);
    const double r1 = fma(-k, kPio2A, y);
    const double t = k * kPio2B;
    const double r = r1 - t;
    const double bb = r - r1;
    double rr = (r1 - (r - bb)) - (t + bb);
    rr = fma(-k, kPio2C, rr);
    const double x = r * r;
    double ps = 1.0 / 355687428096000.0;      // 1/17!
    ps = fma(ps, x, -1.0 / 1307674368000.0);  // -1/15!
    ps = fma(ps, x, 1.0 / 6227020800.0);
    ps = fma(ps, x, -1.0 / 39916800.0);
    ps = fma(ps, x, 1.0 / 362880.0);
    ps = fma(ps, x, -1.0 / 5040.0);
    ps = fma(ps, x, 1.0 / 120.0);
    ps = fma(ps, x, -1.0 / 6.0);
    double pc = -1.0 / 6402373705728000.0;    // -1/18!
    pc = fma(pc, x, 1.0 / 20922789888000.0);  // 1/16!
    pc = fma(pc, x, -1.0 / 87178291200.0);
    pc = fma(pc, x, 1.0 / 479001600.0);
    pc = fma(pc, x, -1.0 / 3628800.0);
    pc = fma(pc, x, 1.0 / 40320.0);
    pc = fma(pc, x, -1.0 / 720.0);
    pc = fma(pc, x, 1.0 / 24.0);
    const double st = fma(r * x, ps, rr * fma(-0.5, x, 1.0)), sr = r + st;
    const double xl = fma(r, r, -x);
    const double hz = 0.5 * x;
    const double w = 1.0 - hz, ct = ((1.0 - w) - hz) + fma(x * x, pc, -fma(0.5, xl, rr * r)), cr = w + ct;
    const int q = (int)k;
    const double so = (q & 1) ? cr : sr, co = (q & 1) ? sr : cr;
    *s = (q & 2) ? -so : so;
    *c = ((q + 1) & 2) ? -co : co;
    if (lo) {
        const double sl = (r - sr) + st, cl = (w - cr) + ct, sv = (q & 1) ? cl : sl, cv = (q & 1) ? sl : cl;
        lo[0] = (q & 2) ? -sv : sv;
        lo[1] = ((q + 1) & 2) ? -cv : cv;
    }
}

// 1/sqrt(d), d > 0: hardware estimate refined by two Newton steps y += y (1 - d y^2) / 2.
__device__ inline double rsqrt_nr(double d) {
    double y = __builtin_amdgcn_rsq(d);
    double e = fma(-d * y, y, 1.0);
    y = fma(0.5 * y, e, y);
    e = fma(-d * y, y, 1.0);
    return fma(0.5 * y, e, y);
}

// 1/sqrt(d), d > 0, in one third-order step y += y e (1/2 + 3 e/8), e = 1 - d y^2, from the hardware estimate
// (relative error below 2^-22, so the step's own error is below 2^-64).
__device__ inline double rsqrt_h3(double d) {
    const double y = __builtin_amdgcn_rsq(d);
    const double e = fma(-d * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// ---------------------------------------------------------------------------
// Table-driven variants (P. T. P. Tang, "Table-driven implementation of the
// exponential function in IEEE floating-point arithmetic", ACM TOMS 15, 1989;
// the same scheme for sin/cos): the reduction goes to |r| <= ln2/128 and
// |r| <= pi/64 against 64-entry tables of 2^(j/64) and sin, cos(j pi/32) held as
// double-double (hi, lo) pairs, so short series suffice and the table value is
// added last: e^{-a}, sin and cos stay within about 0.52 ulp (of 1 for sin, cos).
// The kernels that use them copy the tables to LDS first (load_math_tables).
// ---------------------------------------------------------------------------
struct MathTables {
    double2 e[64];  // 2^(j/64): hi, lo
    double4 t[64];  // sin(j pi/32) hi, lo, cos(j pi/32) hi, lo
};

static __constant__ double kExpTable[64][2] = CQBEM_EXP_TABLE;
static __constant__ double kTrigTable[64][4] = CQBEM_TRIG_TABLE;

// Copies the tables (constant memory) into `s`; every thread of the block calls it, a barrier must follow.
__device__ inline void load_math_tables(MathTables *s) {
    const auto &kExp = kExpTable;
    const auto &kTrig = kTrigTable;
    for (int k = threadIdx.x; k < 64; k += blockDim.x) {
        s->e[k] = make_double2(kExp[k][0], kExp[k][1]);
        s->t[k] = make_double4(kTrig[k][0], kTrig[k][1], kTrig[k][2], kTrig[k][3]);
    }
}

// Both find k by adding 1.5 2^52, which leaves rint in the low bits of the sum's significand: the integer is read
// from there (no conversion) and the subtraction gives it back as a double.
constexpr double kRoundMagic = 6755399441055744.0;  // 1.5 2^52
__host__ __device__ inline int magic_int(double t) { return (int)(unsigned)__builtin_bit_cast(unsigned long long, t); }

// e^t, -740 <= t <= 700.  k = rint(t 64/ln2); r = t - k ln2/64 (the k hi product and the first subtraction exact);
// e^r - 1 = r + r^2 q(r), q the degree-4 Taylor polynomial with its last term replaced by its Chebyshev economization
// on |r| <= ln2/128 (error 5e-18 of the result); 2^(k/64) = 2^(k >> 6) T[k & 63], and T_hi + (T_hi p + T_lo) last.
__host__ __device__ inline double exp_tab_core(double t, const double2 *T) {
#pragma clang fp contract(off)
    constexpr double kR = 0.005415212348514945;  // ln2/128
    const double km = fma(t, CQBEM_64_OVER_LN2, kRoundMagic);
    const double k = km - kRoundMagic;
    const double r1 = fma(-k, CQBEM_LN2_OVER_64_HI, t);
    const double r = fma(-k, CQBEM_LN2_OVER_64_LO, r1);
    double q = fma(r, 1.0 / 120.0, 1.0 / 24.0 + kR * kR / 720.0);
    q = fma(q, r, 1.0 / 6.0);
    q = fma(q, r, 0.5 - kR * kR * kR * kR / 5760.0);
    const double p = fma(r * r, q, r);
    const int ki = magic_int(km);
    const double2 e = T[ki & 63];
    return ldexp(e.x + fma(e.x, p, e.y), ki >> 6);
}
// e^{-a}, clamped at a = 740 (underflowed to 0) and a = -700.
__host__ __device__ inline double exp_neg_tab(double a, const double2 *T) {
    return exp_tab_core(fmin(fmax(-a, -740.0), 700.0), T);
}

// sin y, cos y for |y| < kTrigArgMax, as cq_sincos.  k = rint(32 y/pi); r = y - k pi/32 in two FMAs (k A exact, so the
// first has no rounding error; the second part holds the next 53 bits of pi/32: r is off by 2^-58 at most, 0.02 ulp
// of 1); sin r - r = r^3 times the degree-3 Taylor polynomial in r^2 with its last term economized on |r| <= pi/64
// (error 2e-19), cos r - 1 through r^8 (next term < 1e-19); then sin(a + r) = S + (S (cos r - 1) + C sin r) and
// cos(a + r) = C + (C (cos r - 1) - S sin r) with a = (k mod 64) pi/32 and the table's lo parts added inside the
// brackets.
__host__ __device__ inline void sincos_tab(double y, const double4 *T, double *s, double *c) {
#pragma clang fp contract(off)
    constexpr double kX = 0.0024094971401247595;  // (pi/64)^2
    const double km = fma(y, CQBEM_32_OVER_PI, kRoundMagic);
    const double k = km - kRoundMagic;
    const double r1 = fma(-k, CQBEM_PI_OVER_32_A, y);
    const double r = fma(-k, CQBEM_PI_OVER_32_B + CQBEM_PI_OVER_32_C, r1);
    const double x = r * r;
    double ps = fma(x, -1.0 / 5040.0 + 1.5 * kX / 362880.0, 1.0 / 120.0 - 0.5625 * kX * kX / 362880.0);
    ps = fma(ps, x, -1.0 / 6.0 + kX * kX * kX / 32.0 / 362880.0);
    const double sr = fma(r * x, ps, r);  // sin r
    double pc = fma(x, 1.0 / 40320.0, -1.0 / 720.0);
    pc = fma(pc, x, 1.0 / 24.0);
    pc = fma(pc, x, -0.5);
    const double cm1 = x * pc;  // cos r - 1
    const double4 e = T[magic_int(km) & 63];
    *s = e.x + fma(e.z, sr, fma(e.x, cm1, e.y));
    *c = e.z + fma(-e.x, sr, fma(e.z, cm1, e.w));
}

// exp(-z), Re z >= 0, through the tables
__host__ __device__ inline cd cexp_neg_tab(cd z, const MathTables *M) {
    const double m = exp_tab_core(fmax(-z.x, -740.0), M->e);
    double sn, cs;
    sincos_tab(z.y, M->t, &sn, &cs);
    return cd{m * cs, -m * sn};
}

// exp(-z), Re z >= 0
__device__ inline cd cexp_neg(cd z) {
    const double m = exp_neg(z.x);
    double sn, cs;
    cq_sincos(z.y, &sn, &cs);
    return cd{m * cs, -m * sn};
}

// Tables that no kernel writes, read through the constant address space: uniform indices become scalar loads also where
// the pointer itself came from memory (scenes).
typedef const __attribute__((address_space(4))) double const_double;
typedef const __attribute__((address_space(4))) int const_int;
__device__ inline const_double *as_const(const double4 *p) { return (const_double *)p; }
__device__ inline const_int *as_const(const int4 *p) { return (const_int *)p; }

// Per-frequency constants, uniform across a wavefront (loaded with scalar loads).
// The table of the regular kernels' exponentials (exp_pair): four arrays of coarse nodes (a pair's values, then what their
// rounding left out, relative to them), whose last place is left to the block's counters, and two of fine nodes.  Arrays, not
// records: lanes at different nodes meet in an LDS bank only where the nodes are 16 apart.
constexpr int kExpCoarse = 64, kExpFine = 128;
constexpr int kExpWords = 4 * kExpCoarse + 2 * kExpFine;
constexpr int kExpCells = (kExpCoarse - 1) * kExpFine - kExpFine / 2;
constexpr int kExpCounters = 4 * kExpCoarse - 1;  // the word of the block's counters
constexpr int kExpDeg = 5;  // of the polynomial in the rest
struct Freq {
    cd s;    // s_l
    cd sc1;  // s / c1
    cd sc2;  // s / c2
    cd is;   // 1 / s
    cd is2;  // 1 / s^2
    // The regular kernels' exponentials (exp_pair): the cell h and 1 / h, the coefficients of d, .., d^5 in e^{-s d / c} for
    // c1 and c2, |d| <= h / 2; direct: s is beyond the table's reach.
    double h, ih;
    cd q[2][kExpDeg];
    int direct, pad;
};

// The cell over distances up to `reach` (n h is exact for every n + 1/2 up to kExpCells), and the largest |s / c| H that the
// table is used for, with H = h / 2 (+ 1/16: the cell index is rounded).  The polynomial of e^{-x d}, |d| <= H, is the
// Taylor series through d^6 with the last term economized (d^6 -> (48 H^2 d^4 - 18 H^4 d^2 + H^6) / 32, T. J. Rivlin,
// "Chebyshev Polynomials", 1990): its error 2 |x H|^6 / (32 6!), constant term left out included, is below 1e-17.  The line is
// at |s| reach / c = 99, where a fine node's value is e^{+-0.8} at most: up to there the table's values are no less exact than
// the direct functions' in any range of arguments (at 124 they have 1.1 times their error for |s r / c| in 0.3 .. 1).
inline double exp_table_cell(double reach) {
    if (!(reach > 0.0)) return 1.0;
    const double h = reach / (kExpCells - 1.5);
    const float f = (float)h;
    return f > 0.0f && f < INFINITY ? (double)__builtin_nextafterf(f, INFINITY) : h;
}
constexpr double kExpTableReach = 0.0066;
inline double exp_table_width(double h) { return 0.5 * h * (1.0 + 1.0 / 16); }
// Fills the fields of exp_pair from s / c1 and s / c2 and the cell.
inline void exp_table_plan(Freq &f, double h) {
    const double H = exp_table_width(h);
    f.h = h, f.ih = 1.0 / h, f.pad = 0;
    f.direct = !(H * std::max(std::hypot(f.sc1.x, f.sc1.y), std::hypot(f.sc2.x, f.sc2.y)) <= kExpTableReach);
    for (int c = 0; c < 2; c++) {
        const cd x = c ? f.sc2 : f.sc1, x2 = x * x, x4 = x2 * x2, x6 = x4 * x2;
        f.q[c][0] = x * -1.0;
        f.q[c][1] = x2 * 0.5 + x6 * (H * H * H * H / -1280.0);
        f.q[c][2] = x * x2 * (-1.0 / 6.0);
        f.q[c][3] = x4 * (1.0 / 24.0) + x6 * (H * H / 480.0);
        f.q[c][4] = x * x4 * (-1.0 / 120.0);
    }
}

// The constants that the regular-face kernels read, at one frequency (cd) or at the two real ones (rp), from the table
// through the constant address space.
template <class T> struct PointFreq {
    typedef T value;
    T s, sc1, sc2, is2;
};
// A frequency within the reach of the exponentials' table.
struct TableFreq : PointFreq<cd> {
    double h, ih;
    cd q[2][kExpDeg];
};
__device__ inline PointFreq<cd> point_freq(const Freq *f, int l, cd) {
    const_double *p = (const_double *)(f + l);
    return PointFreq<cd>{cd{p[0], p[1]}, cd{p[2], p[3]}, cd{p[4], p[5]}, cd{p[8], p[9]}};
}
__device__ inline PointFreq<rp> point_freq(const Freq *f, int hi, rp) {
    const_double *p = (const_double *)f, *q = (const_double *)(f + hi);
    return PointFreq<rp>{rp{p[0], q[0]}, rp{p[2], q[2]}, rp{p[4], q[4]}, rp{p[8], q[8]}};
}
__device__ inline TableFreq table_freq(const Freq *f, int l) {
    const_double *p = (const_double *)(f + l);
    TableFreq r{point_freq(f, l, cd{}), p[10], p[11]};
#pragma unroll
    for (int k = 0; k < 2 * kExpDeg; k++) r.q[k / kExpDeg][k % kExpDeg] = cd{p[12 + 2 * k], p[13 + 2 * k]};
    return r;
}
__device__ inline bool beyond_table(const Freq *f, int l) { return *(const_int *)&f[l].direct; }

// ---------------------------------------------------------------------------
// The regular kernels' exponentials e^{-s r / c1} and e^{-s r / c2}.  Both depend on the distance r alone once the
// frequency is fixed, so a block tabulates them: r = 128 k h + (j - 63.5) h + d with |d| <= h / 2 over the mesh's
// extent, e^{-s r / c} = C_k (1 + g_j) (1 + u(d)), g_j = e^{..} - 1 and u a polynomial of degree 5 in the real d with uniform
// coefficients, whose constant term is the relative rounding error of C_k, the lane's own.  It is summed as C + C v,
// v = g + (1 + g) u, so that a value carries the last sum's roundings and |v| (at most about 1, and small near r = 0, where C
// is 1) times the ones before: 0.3 to 0.7 units of 2^-53 rms over all arguments up to the table's reach (kExpTableReach), where
// the direct functions, whose argument s r / c is rounded, have 0.5 to 0.95 below |s r / c| = 3 and 22 at 100.  49
// instructions per point and pair, against 78 for two reductions with e^x, sin and cos, which remain beyond the reach.
// ---------------------------------------------------------------------------
constexpr double kNodeMagic = 422212465065984.0 + kExpFine / 2;  // 1.5 2^48 + 64: the low word of r / h + this holds 16 cell + 4 bits
// e^{-sc r} as the sum of two doubles, r exact.
__host__ __device__ inline cd node_exp(cd sc, double r, cd &lo) {
#pragma clang fp contract(off)
    const cd z{sc.x * r, sc.y * r};
    double m, ml, s, c, sl[2];
    m = exp_neg(z.x, &ml), cq_sincos(z.y, &s, &c, sl);
    const cd e{m * c, -m * s};
    // what the products, their factors' low parts and the argument's roundings add
    const cd t{fma(sc.x, r, -z.x), fma(sc.y, r, -z.y)};
    const cd l{fma(m, c, -e.x) + (m * sl[1] + ml * c) - (e.x * t.x - e.y * t.y),
               fma(-m, s, -e.y) - (m * sl[0] + ml * s) - (e.x * t.y + e.y * t.x)};
    const cd v{e.x + l.x, e.y + l.y};
    lo = cd{(e.x - v.x) + l.x, (e.y - v.y) + l.y};
    return v;
}
// a / b, to a few units of the last place
__host__ __device__ inline cd over(cd a, cd b) {
    const double i = 1.0 / (b.x * b.x + b.y * b.y);
    return cd{(a.x * b.x + a.y * b.y) * i, (a.y * b.x - a.x * b.y) * i};
}
// v - 1 from v's two parts
__host__ __device__ inline cd minus_one(cd v, cd lo) { return cd{(v.x - 1.0) + lo.x, v.y + lo.y}; }
// Node n of the table: coarse nodes, then fine ones, kExpCoarse - 1 + kExpFine in all.
__host__ __device__ inline void fill_exp_node(const TableFreq &f, int n, double2 *tab) {
    const bool fine = n >= kExpCoarse - 1;
    const int j = n - (kExpCoarse - 1);
    const double r = (fine ? j + (0.5 - kExpFine / 2) : (double)(n * kExpFine)) * f.h;
    cd l1, l2;
    const cd e1 = node_exp(f.sc1, r, l1), e2 = node_exp(f.sc2, r, l2);
    if (fine) {
        const cd g1 = minus_one(e1, l1), g2 = minus_one(e2, l2);
        double2 *p = tab + 4 * kExpCoarse + j;
        p[0] = make_double2(g1.x, g1.y), p[kExpFine] = make_double2(g2.x, g2.y);
    } else {
        const cd q1 = over(l1, e1), q2 = over(l2, e2);
        double2 *p = tab + n;
        p[0] = make_double2(e1.x, e1.y), p[kExpCoarse] = make_double2(e2.x, e2.y);
        p[2 * kExpCoarse] = make_double2(q1.x, q1.y), p[3 * kExpCoarse] = make_double2(q2.x, q2.y);
    }
}
static_assert(sizeof(MathTables) <= sizeof(double2) * kExpCounters, "the direct functions' tables fit in the same place");
// Fills `tab` (kExpWords words but the last coarse entry's, which are left alone): with the nodes, or with the direct
// functions' tables.
__device__ inline void fill_exp_table(const TableFreq &f, double2 *tab) {
    for (int n = threadIdx.x; n < kExpCoarse - 1 + kExpFine; n += blockDim.x) fill_exp_node(f, n, tab);
}
template <class T> __device__ inline void fill_exp_table(const PointFreq<T> &, double2 *tab) {
    load_math_tables(reinterpret_cast<MathTables *>(tab));
}
// q0 + d q[0] + .. + d^5 q[4], one component.
__host__ __device__ inline double exp_poly(double d, double q0, double q1, double q2, double q3, double q4, double q5) {
    return fma(fma(fma(fma(fma(d, q5, q4), d, q3), d, q2), d, q1), d, q0);
}
__host__ __device__ inline cd exp_poly(double d, double2 q0, const cd (&q)[kExpDeg]) {
    return cd{exp_poly(d, q0.x, q[0].x, q[1].x, q[2].x, q[3].x, q[4].x), exp_poly(d, q0.y, q[0].y, q[1].y, q[2].y, q[3].y, q[4].y)};
}
// C (1 + g) (1 + u)
__host__ __device__ inline cd node_value(cd C, cd g, cd u) {
    const double fx = g.x + 1.0;
    const cd v{fma(fx, u.x, fma(-g.y, u.y, g.x)), fma(fx, u.y, fma(g.y, u.x, g.y))};
    return cd{fma(C.x, v.x, fma(-C.y, v.y, C.x)), fma(C.x, v.y, fma(C.y, v.x, C.y))};
}
// The pair at distance r; z1 = s r / c1 and z2 = s r / c2, rounded.
__host__ __device__ __attribute__((always_inline)) inline void exp_pair(double r, const cd &, const cd &, const TableFreq &f,
                                                                        const double2 *tab, cd &e1, cd &e2) {
    const unsigned long long t = __builtin_bit_cast(unsigned long long, fma(r, f.ih, kNodeMagic));
    const unsigned lo = (unsigned)t & ~15u;
    const double n = __builtin_bit_cast(double, (t & 0xffffffff00000000ull) | lo) - (kNodeMagic - 0.5);
    const double d = fma(-f.h, n, r);
    // byte offsets of the two nodes, in bounds whatever r
    const unsigned j = lo & (16u * (kExpFine - 1)), k = (lo / kExpFine) & (16u * (kExpCoarse - 1));
    const double2 *fine = reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(tab + 4 * kExpCoarse) + j);
    const double2 *coarse = reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(tab) + k);
    const double2 a1 = coarse[0], a2 = coarse[kExpCoarse], l1 = coarse[2 * kExpCoarse], l2 = coarse[3 * kExpCoarse];
    const double2 b1 = fine[0], b2 = fine[kExpFine];
    e1 = node_value(cd{a1.x, a1.y}, cd{b1.x, b1.y}, exp_poly(d, l1, f.q[0]));
    e2 = node_value(cd{a2.x, a2.y}, cd{b2.x, b2.y}, exp_poly(d, l2, f.q[1]));
}
// The same directly, for a frequency beyond the table's reach, and for the two real ones, where there are no trigonometric
// functions to save and e^x is exact to half an ulp of the rounded argument's.
__host__ __device__ __attribute__((always_inline)) inline void exp_pair(double, const cd &z1, const cd &z2, const PointFreq<cd> &,
                                                                        const double2 *tab, cd &e1, cd &e2) {
    const MathTables *M = reinterpret_cast<const MathTables *>(tab);
    e1 = cexp_neg_tab(z1, M), e2 = cexp_neg_tab(z2, M);
}
__host__ __device__ __attribute__((always_inline)) inline void exp_pair(double, const rp &z1, const rp &z2, const PointFreq<rp> &,
                                                                        const double2 *tab, rp &e1, rp &e2) {
    const double2 *T = reinterpret_cast<const MathTables *>(tab)->e;
    auto e = [T](double z) { return exp_tab_core(fmax(-z, -740.0), T); };
    e1 = rp{e(z1.x), e(z1.y)}, e2 = rp{e(z2.x), e(z2.y)};
}

// Material constants.
struct Mat {
    double c1, c2, rho;
    double ic1, ic2;    // 1/c1, 1/c2
    double ic1s, ic2s;  // 1/c1^2, 1/c2^2
    double kap;         // c2^2 / c1^2
    double six_c2s;     // 6 c2^2
    double g_scale;     // 1 / (4 pi rho)
};

// Shared exponentials of one (point pair, frequency): everything the four
// kernels need that depends on the frequency.
struct Expo {
    cd e1, e2;  // exp(-r s/c1), exp(-r s/c2)
    cd dA;      // A1 - A2, A_k = (s r/c_k + 1) exp(-r s/c_k) / s^2
    cd A2;
};

__device__ inline Expo expo(double r, const Freq &f) {
    Expo E;
    const cd z1 = f.sc1 * r, z2 = f.sc2 * r;
    E.e1 = cexp_neg(z1);
    E.e2 = cexp_neg(z2);
    const cd A1 = (z1 + cd{1.0, 0.0}) * E.e1 * f.is2;
    E.A2 = (z2 + cd{1.0, 0.0}) * E.e2 * f.is2;
    E.dA = A1 - E.A2;
    return E;
}

// expo with the table-driven exponentials (tables in LDS)
__device__ inline Expo expo(double r, const Freq &f, const MathTables *M) {
    Expo E;
    const cd z1 = f.sc1 * r, z2 = f.sc2 * r;
    E.e1 = cexp_neg_tab(z1, M);
    E.e2 = cexp_neg_tab(z2, M);
    const cd A1 = (z1 + cd{1.0, 0.0}) * E.e1 * f.is2;
    E.A2 = (z2 + cd{1.0, 0.0}) * E.e2 * f.is2;
    E.dA = A1 - E.A2;
    return E;
}

// u_hat = alpha rh rh^T + beta I  (times r if `times_r`: r*u_hat for polar rules).
__device__ inline void g_coef(const Expo &E, double ir, double ir2, const Mat &m, cd &alpha, cd &beta) {
    const cd t = E.dA * ir2;
    alpha = 3.0 * t + E.e1 * m.ic1s - E.e2 * m.ic2s;
    beta = E.e2 * m.ic2s - t;
    alpha = alpha * m.g_scale, beta = beta * m.g_scale;
}

// p_hat coefficients without the 1/(4 pi) factor.
__device__ inline void h_coef(const Expo &E, double ir, double ir2, const Freq &f, const Mat &m, cd &h1, cd &h2, cd &h4) {
    const cd irs = f.is * ir;  // 1/(r s)
    const cd D = (((E.e1 * m.ic1) - (E.e2 * m.ic2)) * irs + (E.e1 - E.e2) * (irs * irs)) * (m.six_c2s * ir2);
    const cd T1 = E.e1 * ir2, T2 = E.e2 * ir2;
    const cd T3 = E.e1 * f.sc1 * ir, T4 = E.e2 * f.sc2 * ir;
    const double k = m.kap;
    h1 = D + T1 * (4.0 * k - 1.0) - T2 * 2.0 - T3 * (1.0 - 2.0 * k);
    h2 = D + T1 * (2.0 * k) - T2 * 3.0 - T4;
    h4 = D * (-5.0) - T1 * (12.0 * k) + T2 * 12.0 - T3 * (2.0 * k) + T4 * 2.0;
}

constexpr double kInv4Pi = 0.079577471545947667884;  // 1/(4 pi)
constexpr double kInv8Pi = 0.039788735772973833942;  // 1/(8 pi)

// symmetric 3x3 packed index: 00 11 22 01 02 12
__host__ __device__ inline int sidx(int a, int b) {
    if (a == b) return a;
    const int lo = a < b ? a : b, hi = a < b ? b : a;
    return lo == 0 ? (hi == 1 ? 3 : 4) : 5;
}

// ---------------------------------------------------------------------------
// Regular faces in the face's own frame.  With the axes t1, t2 in the face's plane and n its normal, a source point
// y of the face seen from x is y - x = (ar, br, cr) with cr the same at every point of the face, and the direction is
// h = (a, b, c).  The traction kernel then has 8 different entries (xy = yx) and no separate normal:
//   p_xx = h2 c + h4 c a^2, p_yy = h2 c + h4 c b^2, p_xy = h4 c a b, p_xz = a (h1 + h4 c^2), p_zx = a (h2 + h4 c^2),
//   p_yz, p_zy alike with b, p_zz = c (h1 + 2 h2 + h4 c^2)
// and one rotation per face and corner, after the quadrature, brings the sums to the global axes.
// ---------------------------------------------------------------------------
struct FaceFrame {
    double L1, u, v;       // corners in the plane: (0, 0), (L1, 0), (u, v)
    double xa, xb, cr;     // -x in the plane, and the constant third coordinate of y - x
};
// Columns t1, t2, n of the axes of the face with edges e1 = y1 - y0 and e2 = y2 - y0, and twice its area.
__device__ inline void face_axes(const double *e1, const double *e2, double Q[3][3], double *L1, double *area2) {
    const double l2 = e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2], il = rsqrt_h3(l2);
    double c[3], c2 = 0;
    for (int k = 0; k < 3; k++) c[k] = e1[(k + 1) % 3] * e2[(k + 2) % 3] - e1[(k + 2) % 3] * e2[(k + 1) % 3], c2 = fma(c[k], c[k], c2);
    const double ic = rsqrt_h3(c2);
    for (int k = 0; k < 3; k++) Q[0][k] = e1[k] * il, Q[2][k] = c[k] * ic;
    for (int k = 0; k < 3; k++) Q[1][k] = Q[2][(k + 1) % 3] * Q[0][(k + 2) % 3] - Q[2][(k + 2) % 3] * Q[0][(k + 1) % 3];
    *L1 = l2 * il, *area2 = c2 * ic;
}
// Frame of the face (y0, y1, y2) seen from x.
__device__ inline FaceFrame face_frame(const double y[3][3], double x0, double x1, double x2) {
    FaceFrame F;
    double e1[3], e2[3], Q[3][3], area2;
    for (int k = 0; k < 3; k++) e1[k] = y[1][k] - y[0][k], e2[k] = y[2][k] - y[0][k];
    const double xr[3] = {y[0][0] - x0, y[0][1] - x1, y[0][2] - x2};
    face_axes(e1, e2, Q, &F.L1, &area2);
    auto dot = [](const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; };
    F.u = dot(e2, Q[0]), F.v = dot(e2, Q[1]);
    F.xa = dot(xr, Q[0]), F.xb = dot(xr, Q[1]), F.cr = dot(xr, Q[2]);
    return F;
}

// Frequency- and material-dependent factors of one point: with w_k = z_k e_k and dd = (A1 - A2) / r^2 every
// coefficient is a short sum, the traction's in units of 1/r^2 (their static part 6 c2^2 dd is the first bracket of
// H_collocation.cu:45-76, which the displacement kernel shares).
template <class T> struct PointExpo {
    double ir, ir2, r;
    T e1, e2, w1, w2, s2, q2;  // s2 = (z2 + 1) e2, q2 = 1 / (s r)^2
    T dd;
};
template <class F> __device__ inline PointExpo<typename F::value> point_expo(double d2, const F &f, const double2 *tab) {
    typedef typename F::value T;
    PointExpo<T> E;
    E.ir = rsqrt_h3(d2), E.r = d2 * E.ir, E.ir2 = E.ir * E.ir;
    const T z1 = f.sc1 * E.r, z2 = f.sc2 * E.r;
    exp_pair(E.r, z1, z2, f, tab, E.e1, E.e2);
    E.w1 = z1 * E.e1, E.w2 = z2 * E.e2;
    E.s2 = E.w2 + E.e2, E.q2 = f.is2 * E.ir2;
    E.dd = ((E.w1 + E.e1) - E.s2) * E.q2;
    return E;
}

// Local entries of one point in direction (a, b, c), not weighted: G (xx yy zz xy xz yz) = (alpha h h^T + beta I) / r
// without 1/(4 pi rho), and H (xx yy zz xy xz yz zx zy) without 1/(4 pi).
template <class T>
__device__ inline void point_g(const PointExpo<T> &E, double a, double b, double c, const Mat &m, T *G) {
    const T t = E.e2 * m.ic2s;
    const T al = (3.0 * E.dd + (E.e1 * m.ic1s - t)) * E.ir, be = (t - E.dd) * E.ir;
    G[0] = G[1] = G[2] = be;
    fma_cr(G[0], al, a * a), fma_cr(G[1], al, b * b), fma_cr(G[2], al, c * c);
    G[3] = al * (a * b), G[4] = al * (a * c), G[5] = al * (b * c);
}
template <class T>
__device__ inline void point_h(const PointExpo<T> &E, double a, double b, double c, const Mat &m, T *H) {
    const double k = m.kap, a2 = a * E.ir2, b2 = b * E.ir2, c2 = c * E.ir2, cc = c * c;
    const T d6 = E.dd * m.six_c2s;
    T h1 = d6, h2 = d6, h4 = d6 * (-5.0);
    fma_cr(h1, E.e1, 4.0 * k - 1.0), fma_cr(h1, E.e2, -2.0), fma_cr(h1, E.w1, 2.0 * k - 1.0);
    fma_cr(h2, E.e1, 2.0 * k), fma_cr(h2, E.e2, -3.0), h2 -= E.w2;
    fma_cr(h4, E.e1, -12.0 * k), fma_cr(h4, E.e2, 12.0), fma_cr(h4, E.w1, -2.0 * k), fma_cr(h4, E.w2, 2.0);
    const T hc = h4 * c2;
    H[0] = H[1] = h2 * c2;
    fma_cr(H[0], hc, a * a), fma_cr(H[1], hc, b * b);
    H[3] = hc * (a * b);
    T p1 = h1, p2 = h2;
    fma_cr(p1, h4, cc), fma_cr(p2, h4, cc);
    H[4] = p1 * a2, H[5] = p1 * b2, H[6] = p2 * a2, H[7] = p2 * b2;
    fma_cr(p1, h2, 2.0);
    H[2] = p1 * c2;
}

// out (xx yy zz xy xz yz) = Q S Q^T for one real part of a symmetric local block S, columns t1, t2, n of Q; `A` holds
// Q times a factor (the face's area).
__device__ inline void rotate_sym(const double S[6], const double Q[3][3], const double A[3][3], double *out) {
    const int ix[3][3] = {{0, 3, 4}, {3, 1, 5}, {4, 5, 2}};
    double P[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int b = 0; b < 3; b++) P[i][b] = fma(S[ix[i][0]], Q[0][b], fma(S[ix[i][1]], Q[1][b], S[ix[i][2]] * Q[2][b]));
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = a; b < 3; b++) out[sidx(a, b)] = fma(A[0][a], P[0][b], fma(A[1][a], P[1][b], A[2][a] * P[2][b]));
}
// The same for a general block given as xx yy zz xy(= yx) xz yz zx zy; out is row-major.
__device__ inline void rotate_gen(const double S[8], const double Q[3][3], const double A[3][3], double *out) {
    const int ix[3][3] = {{0, 3, 4}, {3, 1, 5}, {6, 7, 2}};
    double P[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int b = 0; b < 3; b++) P[i][b] = fma(S[ix[i][0]], Q[0][b], fma(S[ix[i][1]], Q[1][b], S[ix[i][2]] * Q[2][b]));
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) out[a * 3 + b] = fma(A[0][a], P[0][b], fma(A[1][a], P[1][b], A[2][a] * P[2][b]));
}

// b_hat (translational) and b_hat_ijk (angular) coefficients.
__device__ inline void b_coef(const Expo &E, double ir, double ir2, const Freq &f, const Mat &m, cd &t1, cd &t2, cd &u1,
                              cd &u12, cd &u3) {
    t1 = E.dA * (ir2 * kInv8Pi);
    t2 = (E.A2 - f.is2) * (ir2 * kInv4Pi);
    u1 = E.dA * (ir * kInv8Pi);
    const cd u2 = ((E.e2 * m.ic2) - (E.e1 * m.ic1)) * f.is * kInv8Pi;
    u12 = u1 + u2;
    u3 = E.e2 * f.is * (m.ic2 * kInv4Pi);
}

}  // namespace cqbem
