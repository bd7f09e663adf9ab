// lmie_gpu.hip -- gfx950 kernels of the size-integrated Mie path and the thin C
// ABI of include/lmie_gpu.h.
//
// Forward call:
//   front            one launch for what is serial in an order: Gauss-Legendre
//                    angles (misc/rtutil_math.c:231-316), pi_n +- tau_n at the
//                    positive angles, split 16-bit or FP64
//                    (src/lmie_core.c:669-691), P^{00}, P^{02}, P^{22}, P^{2-2},
//                    P_l (misc/rtutil_math.c:867-1017), and per size D_n
//                    downward, psi_n, chi_n (src/lmie_core.c:298-405)
//   mie_terms        per (size, 2 or 8 orders): a_n, b_n, contraction operand, series partials
//                                                              (src/lmie_core.c:453-652)
//   mie_sums         series per size                          (src/lmie_core.c:537-596)
//   mie_tan_*        the same with the derivatives along x and m
//   angular_mix      S sums on the 16-bit matrix cores (split operands), Stokes in
//                    FP64, weighted sums per angle            (src/lmie_core.c:658-791)
//   angular_f64      the same on the FP64 matrix cores
//   reduce_channels  fixed-order sums of the per-tile partials and of the series
//                    (src/lmie_schedule.c:109-147)
//   expand_*         generalized-spherical / Legendre expansion (misc/rtutil_scat_int.c:20-480)
//   saved_sums       save_control 2: re-weighting of saved per-size arrays
//                                                              (src/lmie_schedule.c:1087-1124)
// Reverse call: expand_adjoint_*, adj_weights, adj_tables, adj_gbuild,
// adj_gsplit, adj_ugemm32 (the kernel matrix G and U = G A), rev_orders and
// rev_carry (per-size reverse sweep); angular_adj_f64 on the FP64 path.
//
// Batches (lmie_gpu_batch_*): the same kernels in batched form (name_b, and
// the batch flag of adj_ugemm32), one launch for all cases of a batch, with
// copy_jobs moving the staged uploads and results.
//
// HBM layouts: orders are rows and sizes (padded to N_p) columns, so the 64
// lanes of a wave (64 consecutive sizes) move 512 contiguous bytes per row;
// split 16-bit operands are blocked by 8 along the contraction index
// ([plane][K / 8][column][8]), one 16-byte fragment per lane.
#include <hip/hip_runtime.h>

#include <math.h>
#include <pthread.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/lmie_gpu.h"
#include "../../include/lmie_hip.h"

namespace {

constexpr double kPi = 3.14159265358979323846264338327950288;
constexpr int KC = 16;     // orders per LDS stage of the contraction
constexpr int TILE = 64;   // size-point tile of the padded layouts

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Mixed path scaling: the split operands hold (2n+1)(a_n +- b_n) * kSA and
// (pi_n +- tau_n) / (n(n+1)) * kSB, so that their product is
// fv4_n (a_n +- b_n)(pi_n +- tau_n) * kSA * kSB with both factors inside the
// normal range of fp16 (|A| <= 4 * 7622, |B| <= 2^14); powers of two, so the
// scaling is exact.
constexpr double kSA = 4.0, kSB = 16384.0;
constexpr int KM = 32;     // orders per LDS stage of the mixed contraction (4 groups of 8)
// planes of the split angle table: (pi+tau) high, middle, low, (pi-tau) high, middle, low
constexpr int B16_PLANES = 6;

// 16-bit element types of the split operands
struct F16 {
     typedef _Float16 T;
     typedef v8h V;
     static __device__ __forceinline__ unsigned short bits(double v, double *rounded) {
          _Float16 h = (_Float16) (float) v;
          *rounded = (double) (float) h;
          return __builtin_bit_cast(unsigned short, h);
     }
     static __device__ __forceinline__ double value(unsigned short b) {
          return (double) (float) __builtin_bit_cast(_Float16, b);
     }
     static __device__ __forceinline__ v4f mfma(v4u a, v4u b, v4f c) {
          return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
     }
     static __device__ __forceinline__ v16f mfma32(v4u a, v4u b, v16f c) {
          return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
     }
};
struct BF16 {
     typedef __bf16 T;
     typedef v8b V;
     static __device__ __forceinline__ unsigned short bits(double v, double *rounded) {
          __bf16 h = (__bf16) (float) v;
          *rounded = (double) (float) h;
          return __builtin_bit_cast(unsigned short, h);
     }
     static __device__ __forceinline__ double value(unsigned short b) {
          return (double) __builtin_bit_cast(float, (unsigned) b << 16);
     }
     static __device__ __forceinline__ v4f mfma(v4u a, v4u b, v4f c) {
          return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
     }
     static __device__ __forceinline__ v16f mfma32(v4u a, v4u b, v16f c) {
          return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
     }
};

// high and low 16-bit parts of v: hi = round(v), lo = round(v - hi)
template <class E>
__device__ __forceinline__ void split16(double v, unsigned short *hi, unsigned short *lo) {
     double r, r2;
     *hi = E::bits(v, &r);
     *lo = E::bits(v - r, &r2);
}
// three parts: hi = round(v), mid = round(v - hi), lo = round(v - hi - mid)
// (hi and mid are split16's two parts)
template <class E>
__device__ __forceinline__ void split16x3(double v, unsigned short *hi, unsigned short *mid, unsigned short *lo) {
     double r, r2, r3;
     *hi = E::bits(v, &r);
     *mid = E::bits(v - r, &r2);
     *lo = E::bits((v - r) - r2, &r3);
}

// Row of the 16x16 f32 result held in lane l, element v, for the 16-bit
// matrix instructions (checked by lmie_gpu_selftest_mfma16).
__device__ __forceinline__ int mfma16_row(int l, int v) { return 4 * (l >> 4) + v; }
// Row of the 32x32 f32 result held in lane l, value v, for the 32x32x16
// 16-bit instructions (column l % 32; checked by lmie_gpu_selftest_mfma32).
__device__ __forceinline__ int mfma32_row(int l, int v) { return 8 * (v >> 2) + 4 * (l >> 5) + (v & 3); }

thread_local char g_err[512];
thread_local double g_times[LMIE_N_TIMERS];
int g_timing = 0;

int set_err(const char *fmt, ...) {
     va_list ap;
     va_start(ap, fmt);
     vsnprintf(g_err, sizeof g_err, fmt, ap);
     va_end(ap);
     return -1;
}

#define HIPCHECK(expr)                                                                     \
     do {                                                                                  \
          hipError_t e_ = (expr);                                                          \
          if (e_ != hipSuccess)                                                            \
               return set_err("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_),        \
                              __FILE__, __LINE__);                                         \
     } while (0)

inline int rup(int a, int b) { return (a + b - 1) / b * b; }

// ---------------------------------------------------------------------------
// complex helpers (double2 = re, im)
struct cd {
     double r, i;
};
__device__ __forceinline__ cd cmk(double r, double i) { return cd{r, i}; }
__device__ __forceinline__ cd cadd(cd a, cd b) { return cd{a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ cd csub(cd a, cd b) { return cd{a.r - b.r, a.i - b.i}; }
__device__ __forceinline__ cd cmul(cd a, cd b) { return cd{a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; }
__device__ __forceinline__ cd cscale(cd a, double s) { return cd{a.r * s, a.i * s}; }
__device__ __forceinline__ cd cconj(cd a) { return cd{a.r, -a.i}; }
__device__ __forceinline__ double cabs2(cd a) { return a.r * a.r + a.i * a.i; }
__device__ __forceinline__ double cdot(cd a, cd b) { return a.r * b.r + a.i * b.i; }   // Re(conj(a) b)
__device__ __forceinline__ double cim(cd a, cd b) { return a.r * b.i - a.i * b.r; }    // Im(conj(a) b)
// Smith's division: scaled by the larger component of the divisor, so no
// intermediate overflows where |b|^2 would.
__device__ __forceinline__ cd cdiv(cd a, cd b) {
     if (fabs(b.r) >= fabs(b.i)) {
          double t = b.i / b.r, d = b.r + b.i * t;
          return cd{(a.r + a.i * t) / d, (a.i - a.r * t) / d};
     }
     double t = b.r / b.i, d = b.r * t + b.i;
     return cd{(a.r * t + a.i) / d, (a.i * t - a.r) / d};
}
__device__ __forceinline__ cd crecip(cd b) { return cdiv(cd{1., 0.}, b); }
// 1/q from the hardware reciprocal and two Newton steps (about 1 ulp; no
// special-value handling), for the dependence chains of the recurrences
__device__ __forceinline__ double rcp_nr(double q) {
     double r = __builtin_amdgcn_rcp(q);
     double e = __builtin_fma(-q, r, 1.);
     r = __builtin_fma(r, e, r);
     e = __builtin_fma(-q, r, 1.);
     return __builtin_fma(r, e, r);
}
__device__ __forceinline__ cd crecip_nr(cd b) {
     const double q = rcp_nr(b.r * b.r + b.i * b.i);
     return cd{b.r * q, -b.i * q};
}
// Smith's division with the reciprocals of rcp_nr (about 1 ulp).  Both of
// Smith's cases in one instruction stream: with (p, q) the divisor's larger
// and smaller component and (u, v) the dividend's matching pair, the quotient
// is ((u + v t) / d, s (v - u t) / d), t = q / p, d = p + q t, s = +1 when
// the real part is the larger (else -1); the same operations as the two
// branches, so the same bits, without divergent lanes.
__device__ __forceinline__ cd cdiv_nr(cd a, cd b) {
     const bool rr = fabs(b.r) >= fabs(b.i);
     const double p = rr ? b.r : b.i, q = rr ? b.i : b.r;
     const double u = rr ? a.r : a.i, v = rr ? a.i : a.r;
     const double t = q * rcp_nr(p), rd = rcp_nr(p + q * t);
     const double im = (v - u * t) * rd;
     return cd{(u + v * t) * rd, rr ? im : -im};
}

// ---------------------------------------------------------------------------
// The front of a call: everything that is serial in an order and independent of
// the rest, one wave per role in one launch (kernel front, below): the angle
// tables and the per-size chains take about the same time (both grow with the
// largest order), so they share the launch and no stream waits for another.
//
// Gauss-Legendre angles: one lane per root.  Newton steps with the
// second-order correction, stopped at a step <= DBL_EPSILON
// (misc/rtutil_math.c:73-129); nodes ascending, weights
// (1 - y^2) 2 / (n P_{n-1}(y'))^2 with y' the last-but-one iterate
// (misc/rtutil_math.c:279-310).  Near mu = +-1 that weight formula is
// sensitive (about 1e-8 relative per ulp of y') to the iteration path, so the
// initial guesses come from the host (the C library's cos and tan, as the
// reference) and every operation here is a separately rounded IEEE operation
// (no contraction): the rule is the reference's rule bit for bit.
// Bound: the Legendre recurrence's chain of four dependent operations per order
// and Newton step.  Its factors j / (j + 1) are the same in every lane: each lane
// divides for one order of the next 64, and the steps read them back from LDS as
// broadcasts, ahead of the chain (uniform_steps), so every table wave can run
// the Newton steps of its own 64 angles and none waits for another.
// Orders the LDS accesses of one wave: what its lanes wrote before is read after
// (LDS serves a wave's accesses in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
     __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
     __builtin_amdgcn_wave_barrier();
}

// Runs step(i, factor(i)) for i = 0 .. n-1 where factor is the same in every lane
// of the wave: 64 factors at a time, one formed per lane, through two LDS buffers
// (lds: UF_LDS doubles of the wave), the next 64 formed and the next eight read
// while the steps run.  (Reading them from the forming lane by v_readlane cost two
// more issue slots per step inside the dependence chain: the Gauss rule of 3810
// angles took 0.26 ms.)
constexpr int UF_ROW = 72, UF_LDS = 2 * UF_ROW;
template <class G, class F>
__device__ __forceinline__ void uniform_steps(int n, double *lds, G factor, F step) {
     const int lane = threadIdx.x & 63;
     wave_lds_fence();
     lds[lane] = factor(lane);
     wave_lds_fence();
     for (int i0 = 0, c = 0; i0 < n; i0 += 64, c ^= 1) {
          if (i0 + 64 < n) lds[(c ^ 1) * UF_ROW + lane] = factor(i0 + 64 + lane);
          wave_lds_fence();
          const double *t = lds + c * UF_ROW;
          if (n - i0 >= 64) {
               // (a loop of a constant count: with the remainder in the same loop a step
               // took a fifth longer)
               double a[8], b[8];
#pragma unroll
               for (int k = 0; k < 8; ++k) a[k] = t[k];
               for (int e = 0; e < 64; e += 16) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) b[k] = t[e + 8 + k];
#pragma unroll
                    for (int k = 0; k < 8; ++k) step(i0 + e + k, a[k]);
#pragma unroll
                    for (int k = 0; k < 8; ++k) a[k] = t[e + 16 + k];      // (past 64: spare entries, unused)
#pragma unroll
                    for (int k = 0; k < 8; ++k) step(i0 + e + 8 + k, b[k]);
               }
          } else {
               const int m = n - i0;
               double a[8], b[8];
#pragma unroll
               for (int k = 0; k < 8; ++k) a[k] = t[k];
               int e = 0;
               for (; e + 8 <= m; e += 8) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) b[k] = t[e + 8 + k];
#pragma unroll
                    for (int k = 0; k < 8; ++k) step(i0 + e + k, a[k]);
#pragma unroll
                    for (int k = 0; k < 8; ++k) a[k] = b[k];
               }
#pragma unroll
               for (int k = 0; k < 7; ++k)
                    if (e + k < m) step(i0 + e + k, a[k]);
          }
          wave_lds_fence();
     }
}

// y: initial guess in, last iterate out; pb: P_{n-1} at the last-but-one.  The
// whole wave takes part; a lane that has stopped keeps its values.
__device__ __forceinline__ void gauss_newton(int n, bool run, double &y, double &pb, double *lds) {
#pragma clang fp contract(off)
     const double dn = (double) n, nn1 = (double) (n * (n + 1));
     int it = 0;
     while (__ballot(run)) {
          double pa = 1., pm = 0., pc = 0.;
          uniform_steps(n, lds, [](int j) { return (double) j / (j + 1.); },
                        [&](int, double c) {
                             pm = pc;
                             pc = pa;
                             const double u = y * pc;
                             pa = c * (u - pm) + u;
                        });
          const double s = 1. - y * y;
          const double d1 = dn * (pc - y * pa) / s;
          const double d2 = (2. * y * d1 - nn1 * pa) / s;
          const double h = pa / d1;
          const double yn = y - h * (1. + h * d2 / (2. * d1));
          if (run) {
               run = fabs(yn - y) > 2.220446049250313e-16 && ++it < 100;
               y = yn;
               pb = pc;
          }
     }
}

// Roots of the rule of n angles from their guesses: mu[0 .. n), w[0 .. n).
__device__ __forceinline__ void gauss_role(int n, const double *guess, double *mu, double *w, int block, double *lds) {
#pragma clang fp contract(off)
     const int i = block * 64 + threadIdx.x, nr = (n + 1) / 2;
     double y = guess[i < nr ? i : nr - 1], pb = 0.;
     gauss_newton(n, i < nr, y, pb, lds);
     if (i >= nr) return;
     double c = (double) n * pb;
     c = 2. / (c * c);
     const double off = 1. * y;
     mu[i] = 0. - off;
     mu[n - 1 - i] = 0. + off;
     w[i] = w[n - 1 - i] = (1. - off * y) * c;
}

// Positive angle j < H of this lane (0 past H): its own Newton steps, or the
// given angles mu[H + j] without guesses.
__device__ __forceinline__ double angle_of(int Q, int H, const double *guess, const double *mu, int j, double *lds) {
#pragma clang fp contract(off)
     if (!guess) return j < H ? mu[H + j] : 0.;
     double y = guess[j < H ? H - 1 - j : 0], pb;
     gauss_newton(Q, j < H, y, pb, lds);
     return j < H ? 0. + 1. * y : 0.;
}

// pi_n +- tau_n at the positive angles mu_{H+j}: one lane per angle, upward
// recurrences pi_{n+1} = mu pi_n + (n+1)/n (mu pi_n - pi_{n-1}),
// tau_n = n (mu pi_n - pi_{n-1}) - pi_{n-1} (src/lmie_core.c:669-691), in
// separately rounded operations in the reference's order: the tables are
// the reference's pi_n, tau_n bit for bit.  f(n, pi + tau, pi - tau) takes
// orders 1 .. n1max.
template <class F>
__device__ __forceinline__ void pitau_steps(int n1max, double m, double *lds, F f) {
#pragma clang fp contract(off)
     double p0 = 0., p1 = 1.;
     uniform_steps(n1max, lds, [](int i) { return (i + 2.) / (i + 1.); },      // (n + 1) / n, n = i + 1
                   [&](int i, double q) {
                        const int n = i + 1;
                        const double a1 = m * p1, a2 = a1 - p0;
                        const double tau = n * a2 - p0;
                        f(n, p1 + tau, p1 - tau);
                        p0 = p1;
                        p1 = a1 + q * a2;
                   });
}

// FP64 tables [Kp][Hp], zero rows past n1max and columns past H.
__device__ __forceinline__ void pitau_role(int H, int Hp, int n1max, int Kp, double m, double *Bp, double *Bm, int j, double *lds) {
     const bool live = j < H;
     pitau_steps(n1max, m, lds, [&](int n, double bp, double bm) {
          Bp[(size_t) (n - 1) * Hp + j] = live ? bp : 0.;
          Bm[(size_t) (n - 1) * Hp + j] = live ? bm : 0.;
     });
     for (int n = n1max + 1; n <= Kp; ++n) Bp[(size_t) (n - 1) * Hp + j] = Bm[(size_t) (n - 1) * Hp + j] = 0.;
}

// Split 16-bit tables for the mixed path, blocked by 8 orders:
// [6 planes: (pi+tau) hi, mid, lo, (pi-tau) hi, mid, lo][Kb][Hb][8], value
// (pi_n +- tau_n) / (n (n+1)) * kSB.  A lane (angle) writes 16 bytes per plane
// per group of 8 orders; consecutive lanes are consecutive 16-byte chunks.
// The splits take eight times the recurrence's own operations, so PITAU_SHARE
// waves run the recurrence of the same 64 angles and each splits and writes
// every PITAU_SHARE-th group.
constexpr int PITAU_SHARE = 8;

template <class E>
__device__ __forceinline__ void pitau16_role(int H, int Hb, int n1max, int Kb, double m, unsigned short *B16, int j, int share,
                                             double *lds) {
     const size_t plane = (size_t) Kb * Hb * 8;
     const int lane = threadIdx.x & 63;
     const bool live = j < H;
     double p0 = 0., p1 = 1.;
     for (int g = 0; g < Kb; ++g) {
          if ((g & 7) == 0) {          // factors of the next 64 orders, one per lane
               const double n = 8 * g + 1 + lane;
               wave_lds_fence();
               lds[lane] = (n + 1.) / n;
               lds[UF_ROW + lane] = kSB / (n * (n + 1.));
               wave_lds_fence();
          }
          const double *qs = lds + 8 * (g & 7), *ss = qs + UF_ROW;
          double q[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) q[e] = qs[e];
          if ((g & (PITAU_SHARE - 1)) != share) {
#pragma unroll
               for (int e = 0; e < 8; ++e) {
                    const double a1 = m * p1, a2 = a1 - p0;
                    p0 = p1;
                    p1 = a1 + q[e] * a2;
               }
               continue;
          }
          unsigned short v[B16_PLANES][8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
               const int n = 8 * g + e + 1;
               const double a1 = m * p1, a2 = a1 - p0;
               const double tau = n * a2 - p0, sc = ss[e];
               const bool on = live && n <= n1max;
               split16x3<E>(on ? (p1 + tau) * sc : 0., &v[0][e], &v[1][e], &v[2][e]);
               split16x3<E>(on ? (p1 - tau) * sc : 0., &v[3][e], &v[4][e], &v[5][e]);
               p0 = p1;
               p1 = a1 + q[e] * a2;
          }
#pragma unroll
          for (int b = 0; b < B16_PLANES; ++b) {
               v4u w;
#pragma unroll
               for (int k = 0; k < 4; ++k) w[k] = (unsigned) v[b][2 * k] | ((unsigned) v[b][2 * k + 1] << 16);
               *(v4u *) (B16 + b * plane + ((size_t) g * Hb + j) * 8) = w;
          }
     }
}

// Generalized spherical functions at the positive angles, l = 0 .. C-1, by
// their three-term recurrences in l (misc/rtutil_math.c:956-1016).  Layout
// [4][C][Hp] (+ plane 4: P_l for the Legendre expansion,
// misc/rtutil_math.c:506-513): lanes (angles) store contiguously for every l.
// The five recurrences are independent, one wave each (FN 0: P00, 1: P02,
// 2: P22, 3: P2-2, 4: P_l).  Columns H .. Hp-1 are written as zeros.
// Each step divides the reference's numerator by its divisor d_l (L1, sqrt(L1^2
// - 4) or L (L1^2 - 4)) in the reference's order of operations; the quotient
// is q = RN(x y) corrected once, q + y RN(x - q d), with y = RN(1 / d_l):
// Markstein's correction, which gives the correctly rounded x / d (the IEEE
// division's bits) when y is the correctly rounded reciprocal and q is
// within an ulp.  All that a step needs besides the angle (divisor,
// reciprocal, square roots, polynomials in l) is formed for 64 l at a time, one
// l per lane, and read back from LDS as broadcasts, ahead of the chain of five
// dependent operations that bounds the step.
constexpr int GSF_CST = 6, GSF_USED = 5;   // doubles per l: divisor, reciprocal, three factors
// The wave's functions go to f(l, l odd, value), l = 0 .. C-1 in order, and each 64
// l are announced by at(l0); a lane that is not live gets zeros.
template <int FN, class A, class F>
__device__ __forceinline__ void gsf_steps(int C, double m, bool live, double *cst, A at, F f) {
     // separately rounded operations in the reference's order (bitwise the
     // reference's functions)
#pragma clang fp contract(off)
     const int lane = threadIdx.x & 63;
     const double m2 = m * m;
     double a0 = 0., b0 = 0.;
     for (int l0 = 0; l0 < C; l0 += 64) {
          {
               const int lc = l0 + lane;
               const double L = lc - 1, L1 = lc, t = 2. * L + 1.;
               double d = 1., a = 0., b = 0., c = 0.;
               if constexpr (FN == 4) {
                    a = lc >= 2 ? (lc - 1) / (double) lc : 0.;
               } else if (lc >= 3) {
                    if constexpr (FN == 0) { d = L1; a = t; b = L; }
                    else if constexpr (FN == 1) { d = sqrt(L1 * L1 - 4.); a = t; b = sqrt(L * L - 4.); }
                    else { d = L * (L1 * L1 - 4); a = t * (L * L1); b = L1 * (L * L - 4); c = t * 4; }
               }
               // (the wave's own buffer: no other wave to wait for)
               double *o = cst + GSF_CST * lane;
               wave_lds_fence();
               o[0] = d; o[1] = 1. / d; o[2] = a; o[3] = b; o[4] = c;
               wave_lds_fence();
          }
          const int ne = min(64, C - l0);
          at(l0);
          auto put = [&](int e, bool odd, double v) {
               f(l0 + e, odd, v);
               a0 = b0;
               b0 = v;
          };
          // l = 0, 1, 2 by their closed forms, then the recurrence steps (no
          // per-step test of l)
          int e0 = 0;
          if (l0 == 0) {
               for (int l = 0; l < 3 && l < C; ++l) {
                    double v;
                    if constexpr (FN == 4) v = l == 0 ? 1. : l == 1 ? m : cst[GSF_CST * l + 2] * (m * b0 - a0) + m * b0;
                    else if (l == 0) v = FN == 0 ? 1. : 0.;
                    else if (l == 1) v = FN == 0 ? m : 0.;
                    else if constexpr (FN == 0) v = (3. * m2 - 1.) / 2.;
                    else if constexpr (FN == 1) v = .25 * sqrt(6.) * (m2 - 1.);
                    else if constexpr (FN == 2) v = .25 * (1. + m) * (1. + m);
                    else v = .25 * (1. - m) * (1. - m);
                    put(l, l & 1, live ? v : 0.);       // dead lanes stay zero from here
               }
               e0 = 3;
          }
          struct Cst { double v[GSF_USED]; };
          auto load = [&](int e) {
               Cst s;
#pragma unroll
               for (int k = 0; k < GSF_USED; ++k) s.v[k] = cst[GSF_CST * e + k];
               return s;
          };
          // the factor of the last value, formed one step ahead of its use: a m -+ c
          auto lead = [&](const Cst &s) {
               const double da = s.v[2] * m;
               return FN < 2 || FN == 4 ? da : FN == 2 ? da - s.v[4] : da + s.v[4];
          };
          auto step = [&](int e, bool odd, const Cst &s, double da) {
               if constexpr (FN == 4) {
                    // P_l = a (m P_{l-1} - P_{l-2}) + m P_{l-1}, a = (l-1)/l
                    const double bb = m * b0;
                    put(e, odd, s.v[2] * (bb - a0) + bb);
               } else {
                    const double x = da * b0 - s.v[3] * a0, q = x * s.v[1];
                    put(e, odd, __builtin_fma(__builtin_fma(-q, s.v[0], x), s.v[1], q));
               }
          };
          auto one = [&](int e) {
               const Cst s = load(e);
               step(e, e & 1, s, lead(s));
          };
          int e = e0;
          for (; e < ne && (e & 3); ++e) one(e);
          // groups of four, the next group's factors read one group ahead
          // (past the last one: the buffer's four spare entries)
          Cst c0[4], c1[4];
          auto read = [&](Cst *c, int o) {
#pragma unroll
               for (int k = 0; k < 4; ++k) c[k] = load(o + k);
          };
          double da;
          auto four = [&](const Cst *c, const Cst *n, int o) {
#pragma unroll
               for (int k = 0; k < 4; ++k) {
                    const double d = lead(k < 3 ? c[k + 1] : n[0]);
                    step(o + k, k & 1, c[k], da);
                    da = d;
               }
          };
          read(c0, e);
          da = lead(c0[0]);
          for (; e + 8 <= ne; e += 8) {
               read(c1, e + 4);
               four(c0, c1, e);
               read(c0, e + 8);
               four(c1, c0, e + 4);
          }
          for (; e < ne; ++e) one(e);
     }
}
// One plane of the expansion tables, zero columns past H: rows of two l, [(C + 1) /
// 2][Hp][2], so a step stores half as often (16 bytes a lane every second l): a
// wave issues its stores inside the chain (42 ns a step with one per l, 32 with one
// per two, 3810 l).
template <int FN>
__device__ __forceinline__ void gsf_role(int H, int Hp, int C, double m, double *P, int j, double *cst) {
     // rows from a uniform pointer, the lane's byte offset a 32-bit register
     const unsigned oj = (unsigned) j * 16u;
     typedef double d2 __attribute__((ext_vector_type(2)));
     double held = 0.;
     auto row = [&](int l) { return (d2 *) ((char *) (P + (size_t) (l >> 1) * 2 * Hp) + oj); };
     gsf_steps<FN>(C, m, j < H, cst, [](int) {},
                   [&](int l, bool odd, double v) {
                        if (odd) *row(l) = d2{held, v};
                        else held = v;
                   });
     if (C & 1) *row(C - 1) = d2{held, 0.};
}
// doubles of one plane of the expansion tables
__host__ __device__ inline size_t gsf_plane(int C, int Hp) { return (size_t) ((C + 1) / 2) * 2 * Hp; }

// ---------------------------------------------------------------------------
// Per-size Mie coefficients.
//
// Element i of row `row` of a [rows][Np] array: the row pointer is uniform
// over the wave (row and the base are), the lane's byte offset a 32-bit
// register, so each load is one scalar-based address and no 64-bit lane
// arithmetic.
// (double2: one 16-byte load, read as a built-in vector type.)
template <class T>
struct LdRowType {
     typedef T type;
};
template <>
struct LdRowType<double2> {
     typedef double type __attribute__((ext_vector_type(2)));
};
template <class T>
__device__ __forceinline__ T ld_row(const T *base, int row, size_t Np, unsigned ioff) {
     // the row pointer through readfirstlane: scalar registers, and the loop
     // optimiser cannot fold the lane offset into a 64-bit pointer per lane
     typedef typename LdRowType<T>::type L;
     const unsigned long long a = (unsigned long long) (base + (size_t) row * Np);
     const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned) a);
     const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned) (a >> 32));
     typedef const char __attribute__((address_space(1))) *gchar;
     typedef const L __attribute__((address_space(1))) *gL;
     const gchar rp = (gchar) (((unsigned long long) hi << 32) | lo);
     const L v = *(gL) (rp + ioff);
     if constexpr (std::is_same<T, double2>::value) return double2{v.x, v.y};
     else return v;
}

// Stores v at element i of row `row` (as ld_row: ioff = i * sizeof(T)).
template <class T>
__device__ __forceinline__ void st_row(T *base, int row, size_t Np, unsigned ioff, T v) {
     typedef typename LdRowType<T>::type L;
     const unsigned long long a = (unsigned long long) (base + (size_t) row * Np);
     const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned) a);
     const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned) (a >> 32));
     typedef char __attribute__((address_space(1))) *gchar;
     typedef L __attribute__((address_space(1))) *gL;
     const gchar rp = (gchar) (((unsigned long long) hi << 32) | lo);
     if constexpr (std::is_same<T, double2>::value) *(gL) (rp + ioff) = L{v.x, v.y};
     else *(gL) (rp + ioff) = v;
}

// Largest and smallest n of the wave's active lanes.
__device__ __forceinline__ int wave_max(int n) {
     int r = __builtin_amdgcn_readfirstlane(n);
     while (const unsigned long long b = __ballot(n > r)) r = __builtin_amdgcn_readlane(n, __builtin_ctzll(b));
     return r;
}
__device__ __forceinline__ int wave_min(int n) { return -wave_max(-n); }

// 1/q from the hardware reciprocal r (about 2^-24 relative) and the series
// r (1 + e + e^2), e = 1 - q r: three dependent operations after the
// reciprocal instead of the four of two Newton steps, error e^3 (< 2^-72)
// plus one rounding.  For the D chain, whose steps are latency bound.
__device__ __forceinline__ double rcp_s3(double q) {
     const double r = __builtin_amdgcn_rcp(q);
     const double e = __builtin_fma(-q, r, 1.);
     return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// ---------------------------------------------------------------------------
// The front runs the three recurrences that are serial in n, two threads per
// size in different waves (the D chain; the psi and chi chains); mie_terms forms a_n, b_n, the
// contraction operand and the partial series sums in parallel, one thread
// per (size, group of 8 or 2 orders); mie_sums adds the partial sums per size.  The
// serial part is a few operations per order, the parallel part fills the GPU.
// D_j is kept as a complex pair, one 16-byte element per (order, size), so
// each step of the D chain stores one element.
struct ChainArgs {
     int N, Np, n1max, n2rows;
     const double *x, *sx, *cx;
     const int *n1, *n2;
     double mr, mi;
     int d_all;                 // store D_j up to n2 - 1 (reverse pass) instead of n1
     double *D;                 // [n2rows][Np][2]: D_j (re, im) at row j
     double *PC;                // [2][n1max + 1][Np]: U_j (psi_j = s U_j), chi_j at row j
     double *PS;                // [Np]: s
     double *Dz, *PQ;           // TAN: dD_j/dz as D; [2][Np] p and q of psi' (see mie_tan_terms)
};

// TAN: forward tangents follow (mie_tan_terms): the D chain carries dD_j/dz too,
// dD_j/dz = c' + (dD_{j+1}/dz + c') / w_j^2 with c' = -(j+1)/z^2, beside the
// chain of w, which stays the longer dependence.
template <bool TAN>
__device__ __forceinline__ void mie_chain_d(const ChainArgs &p, int i) {
#pragma clang fp contract(off)
     if (i >= p.N) return;
     const size_t Np = p.Np;
     const double x = p.x[i];
     const int n1 = p.n1[i], n2 = p.n2[i], dtop = p.d_all ? n2 - 1 : n1;
     // (taken once: the arguments of a batch lie in memory that the stores may alias)
     double2 *const Dv = (double2 *) p.D, *const Dzv = (double2 *) p.Dz;
     // downward D_j(z) = (j+1)/z - 1 / w_j, w_j = D_{j+1} + (j+1)/z,
     // D_{n2} = 0.  The chain carries w: w_{j-1} = (2j+1)/z - 1 / w_j,
     // w_{n2-1} = n2 / z, with 1 / w = conj(w) / |w|^2 (|w| stays between
     // about 1/|z| and n2/|z|) and each update one fused multiply-add per
     // component; D_j = (j+1)/z - 1 / w_j is formed beside the chain.  The
     // recurrence damps its last-bit differences.
     const cd z = cscale(cmk(p.mr, -p.mi), x), iz = crecip(z);
     const cd w0 = cscale(iz, (double) n2), iz2 = cmul(iz, iz);
     cd w = w0, dz = cmk(0., 0.);
     // The loop is the wave's (from its largest n2 to 1; a branch on the lane's
     // own n2 or store range in every step took as long as the chain): down to
     // the smallest n2 a lane that has not started keeps its first w, and a row is
     // stored by every lane as soon as one keeps it (rows past a lane's own
     // range are never read).
     const int jt = wave_max(n2) - 1, js = wave_max(dtop), jm = min(wave_min(n2), jt + 1);
     const unsigned oi = (unsigned) i * 16u;
     auto run = [&](int j0, int j1, auto sel, auto st) {
          for (int j = j0; j >= j1; --j) {
               const double fj = j;
               const cd c1 = cscale(iz, fj + 1.), e = cscale(iz, 2. * fj + 1.);
               const double q = rcp_s3(__builtin_fma(w.r, w.r, w.i * w.i));
               const bool on = !sel.value || j < n2;
               if constexpr (TAN) {
                    const cd dc = cscale(iz2, -(fj + 1.)), r = cmk(w.r * q, -w.i * q), r2 = cmul(r, r), t = cadd(dz, dc);
                    const cd d = cmk(__builtin_fma(t.r, r2.r, __builtin_fma(-t.i, r2.i, dc.r)),
                                     __builtin_fma(t.r, r2.i, __builtin_fma(t.i, r2.r, dc.i)));
                    dz = on ? d : cmk(0., 0.);
                    if (st.value) st_row(Dzv, j, Np, oi, double2{dz.r, dz.i});
               }
               if (st.value) st_row(Dv, j, Np, oi, double2{__builtin_fma(-w.r, q, c1.r), __builtin_fma(w.i, q, c1.i)});
               const cd wn = cmk(__builtin_fma(-w.r, q, e.r), __builtin_fma(w.i, q, e.i));
               w = on ? wn : w0;
          }
     };
     const std::true_type yes;
     const std::false_type no;
     // (js < jt: the kept rows lie below the largest n2)
     const int ja = max(jm, js + 1);
     run(jt, ja, yes, no);
     if (jm > js) run(jm - 1, js + 1, no, no);
     else run(min(js, jt), jm, yes, yes);
     run(min(jm - 1, js), 1, no, yes);
}

// Quotients f / x by 1/x in two parts (two operations).  1/x rounded once is the same
// relative shift of x in every step of a chain: at x = 300 pi + 0.8 it cost psi 4e-14
// of its largest value and psi' 2e-13, at 300 pi + 0.01 4e-12 and 1e-9; now 4e-15, 9e-15 and
// 2e-13, 4e-11 (the reference's ratio chain: 4e-15, 3e-13 and 2e-13, 4e-11: near x = k pi psi
// keeps its loss eps / sin x from psi_0 = sin x, and psi' eps / sin^2 x).
struct OverX {
     double hi, lo;
     __device__ __forceinline__ explicit OverX(double x) {
#pragma clang fp contract(off)
          hi = 1. / x;
          lo = __builtin_fma(-x, hi, 1.) * hi;
     }
     __device__ __forceinline__ double operator()(double f) const {
#pragma clang fp contract(off)
          return __builtin_fma(f, hi, f * lo);
     }
};

// The other chains, in another wave, one loop: psi by
// Miller's downward recurrence, U_{n1} = 0, U_{n1-1} = 1,
// U_{j-1} = (2j+1)/x U_j - U_{j+1}, psi_j = s U_j with s = sin x / U_0 (the
// ratios r_j = U_j / U_{j-1} of the reference's ratio chain, whose
// product from psi_0 = sin x is the same psi_j), beside the upward
// chi_{j+1} = (2j+1)/x chi_j - chi_{j-1}; two independent dependence
// chains of two operations per order and no round trip through memory.
// U grows downward by at most the decay of psi_j between n1 - 1 and 0.
template <bool TAN>
__device__ __forceinline__ void mie_chain_psi(const ChainArgs &p, int i) {
#pragma clang fp contract(off)
     if (i >= p.N) return;
     const size_t Np = p.Np;
     const double x = p.x[i];
     const int n1 = p.n1[i];
     const size_t ppl = (size_t) (p.n1max + 1) * Np;
     double *U = p.PC, *Chi = p.PC + ppl;
     const OverX over(x);
     const double sx = p.sx[i], cx = p.cx[i];
     double ua = 0., ub = 1.;               // U_{j+1}, U_j, starting at j = n1 - 1
     double chi0 = cx, chi1 = over.hi * cx + sx, chn = 0.;
     // as the D chain, one loop for the wave: U waits at its start down to the
     // lane's n1 - 1 (its rows from n1 up are zero), chi runs on past it
     const int nt = wave_max(n1), nm = nt - wave_min(n1);
     const unsigned oi = (unsigned) i * 8u;
     st_row(U, nt, Np, oi, 0.);
     st_row(Chi, 0, Np, oi, chi0);
     auto run = [&](int t0, int t1, auto sel) {
          for (int t = t0; t <= t1; ++t) {
               const double ft = t;
               st_row(Chi, t, Np, oi, chi1);
               if (TAN) chn = t == n1 ? chi1 : chn;
               const double chi2 = over(2. * ft + 1.) * chi1 - chi0;
               chi0 = chi1;
               chi1 = chi2;
               // U_j of j = nt - t, then U_{j-1}
               const int j = nt - t;
               if (sel.value) {
                    const bool on = j < n1;
                    st_row(U, j, Np, oi, on ? ub : 0.);
                    const double un = over(2. * j + 1.) * ub - ua;
                    ua = on ? ub : 0.;
                    ub = on ? un : 1.;
               } else {
                    st_row(U, j, Np, oi, ub);
                    const double un = over(2. * j + 1.) * ub - ua;
                    ua = ub;
                    ub = un;
               }
          }
     };
     run(1, nm, std::true_type{});
     run(nm + 1, nt - 1, std::false_type{});
     // t = nt: U_0 is there
     st_row(Chi, nt, Np, oi, chi1);
     if (TAN) chn = nt == n1 ? chi1 : chn;
     st_row(U, 0, Np, oi, ub);
     const double s = sx / ub;
     p.PS[i] = s;
     if constexpr (TAN) {               // chn = chi_{n1}, ua = U_1
          const double q = -s / chn;
          p.PQ[i] = (cx - sx * over.hi + s * ua - q * cx) / sx;
          p.PQ[Np + i] = q;
     }
}
// a_j, b_j (src/lmie_core.c:557-583), jx = j / x
__device__ __forceinline__ void mie_ab(double jx, cd m, cd im, cd Dj, double psi, double psi0, double chi1,
                                          double chi0, cd *a, cd *b) {
#pragma clang fp contract(off)
     const cd zj = cmk(psi, chi1), zjm = cmk(psi0, chi0);
     const cd u = cadd(cmul(Dj, im), cmk(jx, 0.));   // D/m with im = 1/m
     const cd v = cadd(cmul(m, Dj), cmk(jx, 0.));
     const cd na = csub(cscale(u, psi), cmk(psi0, 0.)), da = csub(cmul(u, zj), zjm);
     const cd nb = csub(cscale(v, psi), cmk(psi0, 0.)), db = csub(cmul(v, zj), zjm);
     *a = cdiv_nr(na, da);
     *b = cdiv_nr(nb, db);
}

// Size-independent factors of order j (the reference's expressions, so the
// same bits), one row each over j = 0 .. n: fv4 = (2j+1) / (j (j+1)),
// fv3m = (j+1) / (j / (j-1)) and fv4m = (2j-1) / ((j-1) j) for j > 1 (else 0),
// fv3 = (j+2) / ((j+1) / j).  The per-order kernels read them as uniform loads
// instead of dividing in every lane.
constexpr int FT_FV4 = 0, FT_FV3M = 1, FT_FV4M = 2, FT_FV3 = 3, FT_ROWS = 4;

__device__ __forceinline__ void order_factors(int n, double *ft, int j) {
#pragma clang fp contract(off)
     if (j > n) return;
     const size_t ld = (size_t) n + 1;
     const double fv1 = 2. * j + 1.;
     ft[FT_FV4 * ld + j] = j > 0 ? fv1 / (j * (j + 1.)) : 0.;
     ft[FT_FV3M * ld + j] = j > 1 ? (j + 1.) / ((double) j / (j - 1.)) : 0.;
     ft[FT_FV4M * ld + j] = j > 1 ? (2. * j - 1.) / ((j - 1.) * j) : 0.;
     ft[FT_FV3 * ld + j] = j > 0 ? (j + 2.) / ((j + 1.) / j) : 0.;
}
// One launch for the roles of the front: blocks of one wave, the longest
// dependence chains first.  Measured at 3810 angles and 32768 sizes (each
// role launched alone): the Gauss rule 0.14 ms (three Newton steps in its
// slowest wave), with the expansion tables behind it 0.27, with the pi/tau tables
// 0.22 (split: 0.21), the chains 0.24 (0.31 with D kept to n2; 0.27 and 0.36 with
// a branch per lane and step); all of them 0.29 (0.36).  The factors common to a
// wave taken from its lanes instead of LDS: 0.26, 0.39, 0.36, and 0.39 for all.
// Block ranges (ends): the expansion tables (planes
// x angle blocks), the pi/tau tables (x PITAU_SHARE split), the Gauss rule, the
// D chains, the psi and chi chains (heaviest sizes first), the order factors.
// PK: pi/tau tables, 0 none, 1 FP64, 2 split fp16, 3 split bf16.
struct FrontArgs {
     int Q, H, Hp, C, n1max;
     const double *guess;       // [(Q + 1) / 2] guesses of the roots, or NULL: angles given in mu
     double *mu, *w;
     double *T;                 // expansion tables, planes of [(C + 1) / 2][Hp][2]
     int Kp, Kb, Hb;
     double *Bp, *Bm;           // [Kp][Hp]
     unsigned short *B16;
     double *ft;                // order factors over 0 .. n1max + 1
     ChainArgs ch;
     unsigned e_gsf, e_pi, e_gauss, e_d, e_psi, e_ft;
     void plan(int planes, int pk, bool gauss, int tiles, bool factors) {
          e_gsf = (unsigned) (Hp / 64 * planes);
          e_pi = e_gsf + (unsigned) (pk == 0 ? 0 : pk == 1 ? Hp / 64 : Hb / 64 * PITAU_SHARE);
          e_gauss = e_pi + (unsigned) (gauss ? ((Q + 1) / 2 + 63) / 64 : 0);
          e_d = e_gauss + (unsigned) tiles;
          e_psi = e_d + (unsigned) tiles;
          e_ft = e_psi + (unsigned) (factors ? (n1max + 2 + 63) / 64 : 0);
     }
};

template <int PK, bool TAN>
__device__ __forceinline__ void front_body(const FrontArgs &p, unsigned b) {
     __shared__ __align__(16) double cst[68 * GSF_CST];      // (also the Newton steps' and pi/tau factors)
     static_assert(68 * GSF_CST >= UF_LDS, "factor buffers");
     const int lane = threadIdx.x;
     if (b < p.e_gsf) {
          const int na = p.Hp / 64, fn = b / na, j = (b % na) * 64 + lane;
          const double m = angle_of(p.Q, p.H, p.guess, p.mu, j, cst);
          double *P = p.T + (size_t) fn * gsf_plane(p.C, p.Hp);
          switch (fn) {
          case 0: gsf_role<0>(p.H, p.Hp, p.C, m, P, j, cst); break;
          case 1: gsf_role<1>(p.H, p.Hp, p.C, m, P, j, cst); break;
          case 2: gsf_role<2>(p.H, p.Hp, p.C, m, P, j, cst); break;
          case 3: gsf_role<3>(p.H, p.Hp, p.C, m, P, j, cst); break;
          default: gsf_role<4>(p.H, p.Hp, p.C, m, P, j, cst); break;
          }
     } else if (b < p.e_pi) {
          if constexpr (PK == 1) {
               const int j = (b - p.e_gsf) * 64 + lane;
               pitau_role(p.H, p.Hp, p.n1max, p.Kp, angle_of(p.Q, p.H, p.guess, p.mu, j, cst), p.Bp, p.Bm, j, cst);
          } else if constexpr (PK > 1) {
               const int e = b - p.e_gsf, j = e / PITAU_SHARE * 64 + lane;
               typedef typename std::conditional<PK == 2, F16, BF16>::type E;
               pitau16_role<E>(p.H, p.Hb, p.n1max, p.Kb, angle_of(p.Q, p.H, p.guess, p.mu, j, cst), p.B16, j, e % PITAU_SHARE, cst);
          }
     } else if (b < p.e_gauss) gauss_role(p.Q, p.guess, p.mu, p.w, b - p.e_pi, cst);
     else if (b < p.e_d) mie_chain_d<TAN>(p.ch, (int) (p.e_d - 1 - b) * 64 + lane);
     else if (b < p.e_psi) mie_chain_psi<TAN>(p.ch, (int) (p.e_psi - 1 - b) * 64 + lane);
     else if (b < p.e_ft) order_factors(p.n1max + 1, p.ft, (int) (b - p.e_psi) * 64 + lane);
}
template <int PK, bool TAN>
__global__ __launch_bounds__(64) void front(FrontArgs p) { front_body<PK, TAN>(p, blockIdx.x); }
// Batched form of each kernel used by fused batches (name_b): one launch for
// all cases, blockIdx.z picks the case, whose own grid (gx, gy blocks) may be
// smaller than the launch grid; its surplus blocks exit.
template <int PK>
__global__ __launch_bounds__(64) void front_b(const FrontArgs *cases) { front_body<PK, false>(cases[blockIdx.z], blockIdx.x); }

int launch_front(const FrontArgs &p, int pk, bool tan, hipStream_t s) {
     const dim3 g(p.e_ft);
     if (p.e_ft == 0) return 0;
     if (pk == 0) hipLaunchKernelGGL((front<0, false>), g, dim3(64), 0, s, p);
     else if (pk == 2) hipLaunchKernelGGL((front<2, false>), g, dim3(64), 0, s, p);
     else if (pk == 3) hipLaunchKernelGGL((front<3, false>), g, dim3(64), 0, s, p);
     else if (tan) hipLaunchKernelGGL((front<1, true>), g, dim3(64), 0, s, p);
     else hipLaunchKernelGGL((front<1, false>), g, dim3(64), 0, s, p);
     HIPCHECK(hipGetLastError());
     return 0;
}

struct TermArgs {
     int N, Np, n1max, n2rows, Kp, Kb, ng;
     const double *ft;          // order_factors rows over 0 .. n1max + 1
     const double *x;
     const int *n1;
     const int *kfill;          // [Np / TILE]
     double mr, mi;
     const double *D, *PC, *PS; // from the chains: [n2rows][Np][2] D_j, [2][n1max + 1][Np] U_j and
                                // chi_j, [Np] s (psi_j = s U_j)
     double *A;                 // FP64 planes [4][Kp][Np] (E = void)
     unsigned short *A16;       // split planes [8][Kb][Np][8] (E = F16 / BF16)
     double *part;              // [5][ng][Np]: se, ss, cb re, cb im, sg of each group
};

template <class E, int OPT>
__device__ __forceinline__ void mie_terms_body(TermArgs p) {
#pragma clang fp contract(off)
     constexpr bool MIX = !std::is_void<E>::value;
     const int i = blockIdx.x * blockDim.x + threadIdx.x, g = blockIdx.y;
     if (i >= p.Np || g >= p.ng) return;
     const size_t Np = p.Np;
     const size_t plane = (size_t) p.Kp * Np, p16 = (size_t) p.Kb * Np * 8, gp = (size_t) p.ng * Np;
     const size_t ld = (size_t) p.n1max + 2;
     const int kf = p.kfill[i / TILE];
     const int n1 = i < p.N ? p.n1[i] : 0;
     const int j0 = OPT * g + 1, j1 = min(OPT * g + OPT, n1);
     double se = 0., ss = 0., sg = 0.;
     cd cb = cmk(0., 0.);
     // split operand of the orders, [plane][order pair]; orders past n1 stay 0
     static_assert(OPT == 8 || !MIX, "whole groups of the split operand");
     unsigned buf[8][4];
#pragma unroll
     for (int q = 0; q < 8; ++q)
#pragma unroll
          for (int k = 0; k < 4; ++k) buf[q][k] = 0u;
     if (j0 <= j1) {
          // (quotients by x, j/x of the terms among them, from OverX: two operations
          // where an IEEE division takes ten; with divisions for j/x the two-mode
          // workload's 32768 sizes took 412 us, now 384)
          const OverX over(p.x[i]);
          const cd m = cmk(p.mr, -p.mi), im = crecip(m);
          // the group's rows are the same in every lane: the D rows are all
          // loaded at once (rows clamped to the array; those past a lane's
          // n1 are read, not used), so the loads overlap
          const double2 *Dv = (const double2 *) p.D;
          const double *U = p.PC, *Chi = p.PC + (size_t) (p.n1max + 1) * Np;
          const unsigned o8 = (unsigned) i * 8u, o16 = (unsigned) i * 16u;
          const int pmax = p.n1max, dmax = p.n2rows - 1;
          const double sc = p.PS[i];
          double ps[OPT + 2], ch[OPT + 2], dr[OPT + 1], di[OPT + 1];   // rows j0 - 2 .. j0 + OPT - 1 (psi, chi), j0 - 1 .. (D)
          // U and chi of the group's rows from two seed rows each, by the
          // chains' own steps (the same bits as the stored rows): U downward
          // from rows j0 + OPT, j0 + OPT - 1 (U_{n1} = 0, U_{n1-1} = 1 where those rows
          // fall inside, as the chain starts), chi upward from rows j0 - 2,
          // j0 - 1 (rows 0 and 1 for the first group).  Rows past a lane's n1
          // are computed from unused values and never used.
          {
               double u[OPT + 3];             // rows j0 - 2 .. j0 + OPT
               u[OPT + 2] = ld_row(U, min(j0 + OPT, pmax), Np, o8);
               u[OPT + 1] = ld_row(U, min(j0 + OPT - 1, pmax), Np, o8);
#pragma unroll
               for (int e = OPT; e >= 0; --e) {
                    const int r = j0 - 2 + e, jj = r + 1;
                    const double un = over(2. * jj + 1.) * u[e + 1] - u[e + 2];
                    u[e] = r == n1 ? 0. : r == n1 - 1 ? 1. : un;
               }
#pragma unroll
               for (int e = 0; e < OPT + 2; ++e) ps[e] = sc * u[e];
               const bool first = j0 == 1;
               ch[0] = first ? 0. : ld_row(Chi, max(j0 - 2, 0), Np, o8);
               ch[1] = ld_row(Chi, j0 - 1, Np, o8);
               ch[2] = first ? ld_row(Chi, 1, Np, o8) : 0.;
#pragma unroll
               for (int e = 2; e < OPT + 2; ++e) {
                    const int t = j0 - 2 + e - 1;
                    const double fv1 = 2. * t + 1.;
                    const double c2 = over(fv1) * ch[e - 1] - ch[e - 2];
                    if (e > 2 || !first) ch[e] = c2;
               }
          }
#pragma unroll
          for (int e = 0; e < OPT + 1; ++e) {
               const double2 v = ld_row(Dv, min(j0 - 1 + e, dmax), Np, o16);
               dr[e] = v.x;
               di[e] = v.y;
          }
          cd ap = cmk(0., 0.), bp = cmk(0., 0.);
          double psi0 = ps[1], chi0 = ch[1];
          if (j0 > 1) mie_ab(over(j0 - 1.), m, im, cmk(dr[0], di[0]), psi0, ps[0], chi0, ch[0], &ap, &bp);
          double sgn = (j0 & 1) ? -1. : 1.;
          // the orders unrolled: the split halves land in registers
#pragma unroll
          for (int e = 0; e < OPT; ++e) {
               const int j = j0 + e;
               if (j <= j1) {
                    const double psi = ps[e + 2], chi = ch[e + 2];
                    cd a, b;
                    mie_ab(over((double) j), m, im, cmk(dr[e + 1], di[e + 1]), psi, psi0, chi, chi0, &a, &b);
                    const double fv1 = 2. * j + 1.;
                    se += fv1 * (a.r + b.r);
                    ss += fv1 * (cabs2(a) + cabs2(b));
                    cb = cadd(cb, cscale(csub(a, b), fv1 * sgn));
                    if (j > 1)
                         sg += p.ft[FT_FV3M * ld + j] * ((ap.r * a.r + ap.i * a.i) + (bp.r * b.r + bp.i * b.i)) +
                               p.ft[FT_FV4M * ld + j] * (ap.r * bp.r + ap.i * bp.i);
                    if constexpr (MIX) {
                         const double sc = fv1 * kSA;
                         unsigned short h[8];
                         split16<E>(sc * (a.r + b.r), &h[0], &h[1]);
                         split16<E>(sc * (a.i + b.i), &h[2], &h[3]);
                         split16<E>(sc * (a.r - b.r), &h[4], &h[5]);
                         split16<E>(sc * (a.i - b.i), &h[6], &h[7]);
#pragma unroll
                         for (int q = 0; q < 8; ++q) buf[q][e / 2] |= (unsigned) h[q] << (16 * (e & 1));
                    } else {
                         const size_t o = (size_t) (j - 1) * Np + i;
                         const double fv4 = p.ft[FT_FV4 * ld + j];
                         p.A[o] = fv4 * (a.r + b.r);
                         p.A[plane + o] = fv4 * (a.i + b.i);
                         p.A[2 * plane + o] = fv4 * (a.r - b.r);
                         p.A[3 * plane + o] = fv4 * (a.i - b.i);
                    }
                    ap = a;
                    bp = b;
                    psi0 = psi;
                    chi0 = chi;
                    sgn = -sgn;
               }
          }
     }
     // operand rows of orders beyond n1 (up to the tile's depth) are zero
     if constexpr (MIX) {
          if (8 * g < kf) {
#pragma unroll
               for (int q = 0; q < 8; ++q) {
                    const v4u w = {buf[q][0], buf[q][1], buf[q][2], buf[q][3]};
                    *(v4u *) (p.A16 + q * p16 + ((size_t) g * Np + i) * 8) = w;
               }
          }
     } else {
          for (int r = max(OPT * g, n1); r < min(OPT * g + OPT, kf); ++r)
               for (int c = 0; c < 4; ++c) p.A[c * plane + (size_t) r * Np + i] = 0.;
     }
     // mie_sums reads the groups below (n1 + OPT - 1) / OPT only
     if (j0 > n1) return;
     double *pt = p.part + (size_t) g * Np + i;
     pt[0] = se;
     pt[gp] = ss;
     pt[2 * gp] = cb.r;
     pt[3 * gp] = cb.i;
     pt[4 * gp] = sg;
}
template <class E, int OPT>
__global__ __launch_bounds__(64) void mie_terms(TermArgs p) { mie_terms_body<E, OPT>(p); }
struct mie_terms_B {
     TermArgs p;
     unsigned gx, gy;
};
template <class E>
__global__ __launch_bounds__(64) void mie_terms_b(const mie_terms_B *cases) {
     const mie_terms_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     mie_terms_body<E, 8>(a.p);
}


// Series per size from the group partials (src/lmie_core.c:586-596): a block
// of 32 sizes x 8 lanes, lane l adds the groups g = l mod 8, then the eight
// lane sums are added in a fixed order (deterministic).
__device__ __forceinline__ void mie_sums_body(const double *part, int N, int Np, int ng, int opt, const int *n1, double *S, double *CB) {
     __shared__ double red[5][8][32];
     const int il = threadIdx.x & 31, l = threadIdx.x >> 5, i = blockIdx.x * 32 + il;
     const size_t gp = (size_t) ng * Np;
     double v[5] = {0., 0., 0., 0., 0.};
     if (i < Np) {
          const int gn = i < N ? (n1[i] + opt - 1) / opt : 0;
          for (int g = l; g < gn; g += 8) {
               const double *pt = part + (size_t) g * Np + i;
#pragma unroll
               for (int q = 0; q < 5; ++q) v[q] += pt[q * gp];
          }
     }
#pragma unroll
     for (int q = 0; q < 5; ++q) red[q][l][il] = v[q];
     __syncthreads();
     if (l || i >= Np) return;
     double se = 0., ss = 0., sg = 0.;
     cd cb = cmk(0., 0.);
     for (int k = 0; k < 8; ++k) {
          se += red[0][k][il];
          ss += red[1][k][il];
          cb = cadd(cb, cmk(red[2][k][il], red[3][k][il]));
          sg += red[4][k][il];
     }
     S[i] = se;
     S[Np + i] = ss;
     S[2 * Np + i] = cabs2(cb);
     S[3 * Np + i] = sg;
     if (CB) {
          CB[i] = cb.r;
          CB[Np + i] = cb.i;
     }
}
__global__ __launch_bounds__(256) void mie_sums(const double *part, int N, int Np, int ng, int opt, const int *n1, double *S, double *CB) { mie_sums_body(part, N, Np, ng, opt, n1, S, CB); }
struct mie_sums_B {
     const double *part;
     int N;
     int Np;
     int ng;
     const int *n1;
     double *S;
     double *CB;
     unsigned gx, gy;
};
__global__ __launch_bounds__(256) void mie_sums_b(const mie_sums_B *cases) {
     const mie_sums_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     mie_sums_body(a.part, a.N, a.Np, a.ng, 8, a.n1, a.S, a.CB);
}


// ---------------------------------------------------------------------------
// Forward tangents of the per-size coefficients.  a_n and b_n depend on the
// inputs through the size parameter x and, analytically, through the complex
// m, so the derivatives along x (HX) and along m (HM) give those of every
// direction.  The D chain carries dD_j/dz; everything
// else is closed per order from the kept D, U and chi:
//   chi'_j = chi_{j-1} - (j/x) chi_j,
//   psi'_j = psi_{j-1} - (j/x) psi_j + p psi_j + q chi_j,
// where psi_j = s U_j is the chain's psi, cut at psi_{n1} = 0: its derivative
// in x solves the same recurrence up to a solution p psi + q chi, fixed by the
// cut (psi'_{n1} = 0: q = -psi_{n1-1} / chi_{n1}) and by psi'_0 = cos x.
// One thread per (size, 8 or 4 orders), as mie_terms; the previous order is formed
// again for the g series.  Bound: FP64 VALU (about 400 operations per (size,
// order) with both derivatives) and the operand planes it writes, 32 bytes per
// (size, order) and operand set.
struct TanArgs {
     int N, Np, n1max, n2rows, Kp, ng;
     const double *ft;          // order_factors rows over 0 .. n1max + 1
     const double *x;
     const int *n1, *kfill;
     double mr, mi;
     const double *D, *Dz, *PC, *PS, *PQ;   // from the chains: D_j and dD_j/dz [n2rows][Np][2], U and chi, s, [2][Np] p and q
     double *A[3];              // operand planes [4][Kp][Np] of the value, then of d/dx, d/dm as present
     double *part;              // [rows][ng][Np]: the value's se, ss, cb (re, im), sg, then mie_tan_sums's rows
};

template <bool HX, bool HM, int OPT>
__global__ __launch_bounds__(64) void mie_tan_terms(TanArgs p) {
     constexpr int NB = 1 + HX + HM, BM = HX ? 2 : 1;
     const int i = blockIdx.x * 64 + threadIdx.x, g = blockIdx.y;
     const size_t Np = p.Np, plane = (size_t) p.Kp * Np, gp = (size_t) p.ng * Np, ld = (size_t) p.n1max + 2;
     const int kf = p.kfill[i / TILE];
     const int n1 = i < p.N ? p.n1[i] : 0;
     const int j0 = OPT * g + 1, j1 = min(OPT * g + OPT, n1);
     if (j0 <= j1) {
          const double x = p.x[i], ax = 1. / x, sc = p.PS[i], pc = p.PQ[i], qc = p.PQ[Np + i];
          const cd m = cmk(p.mr, -p.mi), im = crecip(m), m2 = cmul(m, m);
          const double2 *Dv = (const double2 *) p.D, *Dz = (const double2 *) p.Dz;
          const double *U = p.PC, *Chi = p.PC + (size_t) (p.n1max + 1) * Np;
          const unsigned o8 = (unsigned) i * 8u, o16 = (unsigned) i * 16u;
          // psi, chi and their derivatives of the order before the first one formed
          const int js = g ? j0 - 1 : 1;
          double ps = sc * ld_row(U, js - 1, Np, o8), ch = ld_row(Chi, js - 1, Np, o8), dps, dch;
          if (g) {
               const double jx = (js - 1) * ax;
               dps = sc * ld_row(U, js - 2, Np, o8) - jx * ps + (pc * ps + qc * ch);
               dch = ld_row(Chi, js - 2, Np, o8) - jx * ch;
          } else {
               dps = ch;                 // psi_0 = sin x, chi_0 = cos x
               dch = -ps;
          }
          double se = 0., ss = 0., sg = 0., xe = 0., xs = 0., xg = 0., mg = 0., mgi = 0.;
          cd cb = cmk(0., 0.), xb = cb, me = cb, ms = cb, mb = cb;
          cd ap = cb, bp = cb, axp = cb, bxp = cb, amp = cb, bmp = cb;
          const int jl = min(OPT * g + OPT, p.n1max);       // uniform: the group's last row
          double un = ld_row(U, js, Np, o8), cn = ld_row(Chi, js, Np, o8);
          double2 dn = ld_row(Dv, js, Np, o16), zn = ld_row(Dz, js, Np, o16);
          for (int j = js; j <= jl; ++j) {
               const double ps0 = ps, ch0 = ch, dps0 = dps, dch0 = dch;
               ps = sc * un;
               ch = cn;
               const cd D = cmk(dn.x, dn.y), Dd = cmk(zn.x, zn.y);
               // the next row, ahead of its use (clamped to the arrays)
               const int jn = min(j + 1, jl), kn = min(jn, p.n2rows - 1);
               un = ld_row(U, jn, Np, o8);
               cn = ld_row(Chi, jn, Np, o8);
               dn = ld_row(Dv, kn, Np, o16);
               zn = ld_row(Dz, kn, Np, o16);
               if (j > j1) continue;
               const double jx = j * ax, jxx = -jx * ax;
               dps = ps0 - jx * ps + (pc * ps + qc * ch);
               dch = ch0 - jx * ch;
               const cd zj = cmk(ps, ch), zp = cmk(ps0, ch0);
               const cd Di = cmul(D, im);               // D / m
               const cd u = cadd(Di, cmk(jx, 0.)), v = cadd(cmul(m, D), cmk(jx, 0.));
               const cd da = csub(cmul(u, zj), zp), db = csub(cmul(v, zj), zp);
               const cd a = cdiv_nr(csub(cscale(u, ps), cmk(ps0, 0.)), da), b = cdiv_nr(csub(cscale(v, ps), cmk(ps0, 0.)), db);
               const cd ra = cdiv_nr(cmk(1., 0.), da), rb = cdiv_nr(cmk(1., 0.), db);
               cd atx = cmk(0., 0.), btx = atx, atm = atx, btm = atx;
               if constexpr (HX) {
                    // (u_x psi + u psi' - psi'_{j-1} - a (u_x zeta + u zeta' - zeta'_{j-1})) / da
                    const cd dz = cmk(dps, dch), dzp = cmk(dps0, dch0);
                    const cd ux = cadd(Dd, cmk(jxx, 0.)), vx = cadd(cmul(m2, Dd), cmk(jxx, 0.));
                    const cd na = csub(cadd(cscale(ux, ps), cscale(u, dps)), cmk(dps0, 0.));
                    const cd nb = csub(cadd(cscale(vx, ps), cscale(v, dps)), cmk(dps0, 0.));
                    const cd ea = csub(cadd(cmul(ux, zj), cmul(u, dz)), dzp), eb = csub(cadd(cmul(vx, zj), cmul(v, dz)), dzp);
                    atx = cmul(csub(na, cmul(a, ea)), ra);
                    btx = cmul(csub(nb, cmul(b, eb)), rb);
               }
               if constexpr (HM) {
                    // u_m (psi - a zeta) / da, u_m = (x D' - D/m) / m, v_m = D + m x D'
                    const cd xd = cscale(Dd, x);
                    const cd um = cmul(csub(xd, Di), im), vm = cadd(D, cmul(m, xd));
                    atm = cmul(cmul(um, csub(cmk(ps, 0.), cmul(a, zj))), ra);
                    btm = cmul(cmul(vm, csub(cmk(ps, 0.), cmul(b, zj))), rb);
               }
               if (j >= j0) {
                    const double f1 = 2. * j + 1., fs = (j & 1) ? -f1 : f1;
                    const double f3 = p.ft[FT_FV3M * ld + j], f4 = p.ft[FT_FV4M * ld + j], fa = p.ft[FT_FV4 * ld + j];
                    const size_t o = (size_t) (j - 1) * Np + i;
                    auto put = [&](double *A, cd s, cd t) {
                         A[o] = fa * (s.r + t.r);
                         A[plane + o] = fa * (s.i + t.i);
                         A[2 * plane + o] = fa * (s.r - t.r);
                         A[3 * plane + o] = fa * (s.i - t.i);
                    };
                    se += f1 * (a.r + b.r);
                    ss += f1 * (cabs2(a) + cabs2(b));
                    cb = cadd(cb, cscale(csub(a, b), fs));
                    sg += f3 * (cdot(ap, a) + cdot(bp, b)) + f4 * cdot(ap, bp);
                    put(p.A[0], a, b);
                    if constexpr (HX) {
                         xe += f1 * (atx.r + btx.r);
                         xs += f1 * 2. * (cdot(a, atx) + cdot(b, btx));
                         xb = cadd(xb, cscale(csub(atx, btx), fs));
                         xg += f3 * (cdot(axp, a) + cdot(ap, atx) + cdot(bxp, b) + cdot(bp, btx)) +
                               f4 * (cdot(axp, bp) + cdot(ap, bxp));
                         put(p.A[1], atx, btx);
                    }
                    if constexpr (HM) {
                         // complex sums: the derivative along t is Re(t (.))
                         me = cadd(me, cscale(cadd(atm, btm), f1));
                         ms = cadd(ms, cscale(cadd(cmul(cconj(a), atm), cmul(cconj(b), btm)), 2. * f1));
                         mb = cadd(mb, cscale(csub(atm, btm), fs));
                         mg += f3 * (cdot(amp, a) + cdot(ap, atm) + cdot(bmp, b) + cdot(bp, btm)) +
                               f4 * (cdot(amp, bp) + cdot(ap, bmp));
                         mgi += f3 * (cim(amp, a) - cim(ap, atm) + cim(bmp, b) - cim(bp, btm)) +
                                f4 * (cim(amp, bp) - cim(ap, bmp));
                         put(p.A[BM], atm, btm);
                    }
               }
               ap = a;
               bp = b;
               if constexpr (HX) { axp = atx; bxp = btx; }
               if constexpr (HM) { amp = atm; bmp = btm; }
          }
          double *pt = p.part + (size_t) g * Np + i;
          pt[0] = se; pt[gp] = ss; pt[2 * gp] = cb.r; pt[3 * gp] = cb.i; pt[4 * gp] = sg;
          if constexpr (HX) {
               pt += 5 * gp;
               pt[0] = xe; pt[gp] = xs; pt[2 * gp] = xb.r; pt[3 * gp] = xb.i; pt[4 * gp] = xg;
          }
          if constexpr (HM) {
               pt += 5 * gp;
               pt[0] = me.r; pt[gp] = me.i; pt[2 * gp] = ms.r; pt[3 * gp] = ms.i;
               pt[4 * gp] = mb.r; pt[5 * gp] = mb.i; pt[6 * gp] = mg; pt[7 * gp] = mgi;
          }
     }
     // operand rows of orders beyond n1 (up to the tile's depth) are zero
     for (int r = max(OPT * g, n1); r < min(OPT * g + OPT, kf); ++r)
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
               for (int c = 0; c < 4; ++c) p.A[b][c * plane + (size_t) r * Np + i] = 0.;
}

// Series per size from the group partials (as mie_sums): S [4][Np] of the
// value (ext, sca, |c_bak|^2, asym), then 4 rows of d/dx (HX), then 4 rows
// each of the derivatives along Re m and Im m (HM).
// A block of 32 sizes x 32 lanes: every partial of up to 256 orders is in flight
// at once (with 8 lanes the sum waited for one group after the other: 18.6 us of
// 4000 sizes of up to 250 orders, 13 rows; now 12.9 of twice the groups, and 90 -> 41
// us at 16384 sizes to x = 914).  Lane l adds the groups g = l mod 32,
// the two lanes of a wave add up, then the 16 waves in a fixed order.
template <bool HX, bool HM>
__global__ __launch_bounds__(1024) void mie_tan_sums(const double *part, int N, int Np, int ng, int opt, const int *n1, double *S) {
     constexpr int R = 5 + 5 * HX + 8 * HM;
     __shared__ double red[R][16][32];
     const int il = threadIdx.x & 31, l = threadIdx.x >> 5, i = blockIdx.x * 32 + il;
     const size_t gp = (size_t) ng * Np;
     double v[R];
#pragma unroll
     for (int q = 0; q < R; ++q) v[q] = 0.;
     if (i < Np) {
          const int gn = i < N ? (n1[i] + opt - 1) / opt : 0;
          for (int g = l; g < gn; g += 32) {
               const double *pt = part + (size_t) g * Np + i;
#pragma unroll
               for (int q = 0; q < R; ++q) v[q] += pt[q * gp];
          }
     }
#pragma unroll
     for (int q = 0; q < R; ++q) {
          const double t = v[q] + __shfl_xor(v[q], 32);
          if (!(l & 1)) red[q][l >> 1][il] = t;
     }
     __syncthreads();
     if (l < R) {
          double t = red[l][0][il];
#pragma unroll
          for (int k = 1; k < 16; ++k) t += red[l][k][il];
          red[l][0][il] = t;             // (read by this thread only so far)
     }
     __syncthreads();
     if (l || i >= Np) return;
#pragma unroll
     for (int q = 0; q < R; ++q) v[q] = red[q][0][il];
     const size_t n = Np;
     const cd cb = cmk(v[2], v[3]);
     double *s = S + i;
     s[0] = v[0]; s[n] = v[1]; s[2 * n] = cabs2(cb); s[3 * n] = v[4];
     if constexpr (HX) {
          s += 4 * n;
          s[0] = v[5]; s[n] = v[6]; s[2 * n] = 2. * cdot(cb, cmk(v[7], v[8])); s[3 * n] = v[9];
     }
     if constexpr (HM) {
          constexpr int q = 5 + 5 * HX;
          const cd mb = cmk(v[q + 4], v[q + 5]);
          s += 4 * n;
          s[0] = v[q]; s[n] = v[q + 2]; s[2 * n] = 2. * cdot(cb, mb); s[3 * n] = v[q + 6];
          s += 4 * n;
          s[0] = -v[q + 1]; s[n] = -v[q + 3]; s[2 * n] = 2. * cim(mb, cb); s[3 * n] = v[q + 7];
     }
}

// ---------------------------------------------------------------------------
// Weighted sums over sizes: out[k] = sum_i u_k[i] v_k[i],
// one workgroup per output, fixed-order tree reduction (deterministic).
struct DotJob {
     const double *u, *v;
};

__device__ __forceinline__ void weighted_dots_body(const DotJob *jobs, int n, double *out, int k) {
     __shared__ double red[256];
     const DotJob jb = jobs[k];
     double s = 0.;
     int i = threadIdx.x;
     // eight elements in flight, added in the order of the plain loop
     for (; i + 7 * 256 < n; i += 8 * 256) {
          double a[8], b[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
               a[e] = jb.u[i + 256 * e];
               b[e] = jb.v[i + 256 * e];
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) s += a[e] * b[e];
     }
     for (; i < n; i += 256) s += jb.u[i] * jb.v[i];
     red[threadIdx.x] = s;
     __syncthreads();
     for (int w = 128; w > 0; w >>= 1) {
          if ((int) threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
          __syncthreads();
     }
     if (threadIdx.x == 0) out[k] = red[0];
}


// ---------------------------------------------------------------------------
// Stokes elements of one (size, angle) from the sums sp = S1 + S2, sm = S1 - S2
// (src/lmie_core.c:726-749), and their tangents.
__device__ __forceinline__ void stokes(double spr, double spi, double smr, double smi, double P[4]) {
     const double s1r = .5 * (spr + smr), s1i = .5 * (spi + smi);
     const double s2r = .5 * (spr - smr), s2i = .5 * (spi - smi);
     const double q1 = s1r * s1r + s1i * s1i, q2 = s2r * s2r + s2i * s2i;
     P[0] = (q1 + q2) * .5;
     P[1] = s1r * s2r + s1i * s2i;            // Re S1 S2*
     P[2] = -(q1 - q2) * .5;
     P[3] = s1i * s2r - s1r * s2i;            // Im S1 S2*
}

__device__ __forceinline__ void stokes_tan(double spr, double spi, double smr, double smi, double tpr,
                                           double tpi, double tmr, double tmi, double dP[4]) {
     const double s1r = .5 * (spr + smr), s1i = .5 * (spi + smi);
     const double s2r = .5 * (spr - smr), s2i = .5 * (spi - smi);
     const double t1r = .5 * (tpr + tmr), t1i = .5 * (tpi + tmi);
     const double t2r = .5 * (tpr - tmr), t2i = .5 * (tpi - tmi);
     const double dq1 = 2. * (t1r * s1r + t1i * s1i), dq2 = 2. * (t2r * s2r + t2i * s2i);
     // d(S1 S2*) = dS1 S2* + S1 dS2*
     const double dxr = t1r * s2r + t1i * s2i + s1r * t2r + s1i * t2i;
     const double dxi = t1i * s2r - t1r * s2i + s1i * t2r - s1r * t2i;
     dP[0] = (dq1 + dq2) * .5;
     dP[1] = dxr;
     dP[2] = -(dq1 - dq2) * .5;
     dP[3] = dxi;
}

// Staging of one LDS stage of a blocked split operand: plane-major rows of
// `cols` 16-byte columns, [plane][group of 8][column], `rows` = planes x G rows
// per stage.  Thread tid of NT copies elements tid + NT t; with R = NT / cols
// rows per step, element t of thread tid sits at the thread's base address
// plus a compile-time offset in (plane, group), and each stage adds one
// uniform stride, so no address arithmetic runs inside the stage loop.
template <int NT, int COLS, int G>
struct Stager {
     static constexpr int R = NT / COLS;
     static_assert(NT % COLS == 0 && (R % G == 0 || G % R == 0), "staging shape");
     const unsigned short *base;    // thread's element 0 at stage 0
     size_t plane, row;             // strides in unsigned shorts: plane, group of 8
     __device__ Stager(const unsigned short *src, size_t plane_, size_t row_, int col0, int tid)
         : plane(plane_), row(row_) {
          const int r = tid / COLS, col = tid % COLS;
          base = src + (size_t) (r / G) * plane + (size_t) (r % G) * row + (size_t) (col0 + col) * 8;
     }
     __device__ __forceinline__ const v4u *at(int t, int stage) const {
          return (const v4u *) (base + (size_t) ((R * t) / G) * plane + (size_t) ((R * t) % G) * row +
                                (size_t) stage * G * row);
     }
};

// The split 16-bit contraction on the 16x16x32 instruction: the four complex
// sums of the FP64 contraction with the size operand in two 16-bit parts
// (A = Ah + Al, 22 bits) and the angle operand in three (B = Bh + Bm + Bl,
// 33 bits), on the matrix cores with fp32 accumulation:
//   NP = 5:  A B ~ Ah Bh + [Ah Bm + Al Bh + Ah Bl + Al Bm]   (dropped: Al Bl ~ 2^-34)
//   NP = 3:  A B ~ Ah Bh + [Ah Bm + Al Bh]                   (dropped: ~ 2^-24 of A B)
// The leading product and the bracketed corrections accumulate separately and
// meet in FP64 in the epilogue: an fp32 accumulator rounds at every product
// it takes, relative to its own running value, so the corrections (2^-11 of
// the sums) would otherwise add four roundings of the sums' size per stage.
// The angle operand is the same for every size point, so its rounding errors
// add up coherently over the size integral (two parts of B leave expansion
// coefficients with relative errors of a few 1e-5); the size operand's
// rounding is independent from size to size.
// One workgroup of four waves (one per SIMD) per (size tile of 64, angle tile
// of 64) task, two LDS stages of 32 orders filled straight from memory
// (global_load_lds_dwordx4: a wave moves one 1 KiB row, 64 lanes x 16 bytes,
// into LDS without registers) while the matrix cores work on the other stage,
// one barrier per stage.  Waves in a 2 x 2 grid, each 32 sizes x 32 angles
// (2 x 2 blocks of 16 x 16), 8 sums per element: at +mu and at -mu, whose
// products flip the sign of the odd orders of the size operand
// (s_n = (-1)^(n-1)).  The (size tile, angle tile) of each workgroup comes
// from a host-built list dealt over the XCDs (xcd_tasks).  Partials per size
// tile: part[tile][NW][4][Q].
struct Mix2Args {
     int Np, Kb, Hb, H, Q;
     const unsigned short *A16;     // [8][Kb][Np][8]: S re h/l, S im h/l, T re h/l, T im h/l
     const unsigned short *B16;     // [6][Kb][Hb][8]: (pi+tau) h/m/l, (pi-tau) h/m/l
     const int *ktile;              // orders per size tile of 64 (multiple of KM)
     const int2 *task;              // (size tile, angle tile) per workgroup, (-1, -1) = none
     const double *W[4];            // weight channels [Np]
     double *part;                  // [nT][NW][4][Q]
};

// Shapes of the forward contraction (environment LMIE_MIX_SHAPE, read at every
// call).  A workgroup owns TM sizes x TN angles; its NT / 64 waves form a
// WM x WN grid, each wave 16 MA sizes x 16 NB angles; SEP: the corrections
// have accumulators of their own (else every product goes to one
// accumulator per sum); ST LDS stages, loads ST - 1 stages ahead; OCC
// workgroups per CU.
//   0: 64 x 128, eight waves (two per SIMD), one accumulator, 2 x 80 KiB
//   1: 64 x 64, four waves (one per SIMD), separate corrections, 2 x 56 KiB
//   2: 32 x 64, four waves, separate corrections, 2 x 40 KiB, two workgroups per CU
//   3: 64 x 64, eight waves (two per SIMD), separate corrections, 2 x 56 KiB
constexpr int MIX_G = KM / 8;
constexpr int MIX_SHAPE_DEFAULT = 3;
struct MixS0 { static constexpr int NT = 512, TM = 64, TN = 128, WM = 2, WN = 4, MA = 2, NB = 2, ST = 2, OCC = 1; static constexpr bool SEP = false; };
struct MixS1 { static constexpr int NT = 256, TM = 64, TN = 64, WM = 2, WN = 2, MA = 2, NB = 2, ST = 2, OCC = 1; static constexpr bool SEP = true; };
struct MixS2 { static constexpr int NT = 256, TM = 32, TN = 64, WM = 2, WN = 2, MA = 1, NB = 2, ST = 2, OCC = 2; static constexpr bool SEP = true; };
struct MixS3 { static constexpr int NT = 512, TM = 64, TN = 64, WM = 4, WN = 2, MA = 1, NB = 2, ST = 2, OCC = 1; static constexpr bool SEP = true; };
template <class S> constexpr int mix_sa() { return 8 * MIX_G * S::TM; }              // v4u of A per stage
template <class S> constexpr int mix_sb() { return B16_PLANES * MIX_G * S::TN; }     // v4u of B per stage
// direct loads one wave issues per stage (its vmcnt events)
template <class S> constexpr int mix_loads() {
     return (8 * MIX_G * ((S::TM + 63) / 64) + B16_PLANES * MIX_G * ((S::TN + 63) / 64)) / (S::NT / 64);
}

typedef __attribute__((address_space(3))) void *lds_ptr;

// One wave's share of a stage: the A rows (plane, group) of the size tile and
// the B rows of the angle tile, cut into segments of at most 64 columns of 16
// bytes; wave w takes segments w, w + NT / 64, ...  Each segment is one direct
// load (lane l: column l of the segment).
template <class S>
__device__ __forceinline__ void mix_stage_load(const Mix2Args &p, v4u *sA, v4u *sB, int c, int it0, int jt0,
                                               int wave, int lane) {
     constexpr int NWAVE = S::NT / 64, SEGA = (S::TM + 63) / 64, SEGB = (S::TN + 63) / 64;
     constexpr int LA = S::TM < 64 ? S::TM : 64, LB = S::TN < 64 ? S::TN : 64;
     const size_t Np = p.Np, Hb = p.Hb;
     const size_t pA = (size_t) p.Kb * Np * 8, pB = (size_t) p.Kb * Hb * 8;
     if (lane < LA) {
#pragma unroll
          for (int t = 0; t < 8 * MIX_G * SEGA / NWAVE; ++t) {
               const int r = wave + NWAVE * t, row = r / SEGA, seg = r % SEGA, q = row / MIX_G, g = row % MIX_G;
               const unsigned short *src = p.A16 + q * pA + ((size_t) (c * MIX_G + g) * Np + it0 + 64 * seg + lane) * 8;
               __builtin_amdgcn_global_load_lds((const void *) src, (lds_ptr) (sA + row * S::TM + 64 * seg), 16, 0, 0);
          }
     }
     if (lane < LB) {
#pragma unroll
          for (int t = 0; t < B16_PLANES * MIX_G * SEGB / NWAVE; ++t) {
               const int r = wave + NWAVE * t, row = r / SEGB, seg = r % SEGB, q = row / MIX_G, g = row % MIX_G;
               const unsigned short *src = p.B16 + q * pB + ((size_t) (c * MIX_G + g) * Hb + jt0 + 64 * seg + lane) * 8;
               __builtin_amdgcn_global_load_lds((const void *) src, (lds_ptr) (sB + row * S::TN + 64 * seg), 16, 0, 0);
          }
     }
}

// The products of four sums (x_k times b_k, k = 0..3; x = (h, l) parts,
// b = (h, m, l) parts), interleaved so that consecutive instructions are
// independent: the leading product into m, the corrections into c.
template <class E, int NP>
__device__ __forceinline__ void mix_products(const v4u *x0, const v4u *b0, const v4u *x1, const v4u *b1,
                                             const v4u *x2, const v4u *b2, const v4u *x3, const v4u *b3,
                                             v4f *m, v4f *c) {
     m[0] = E::mfma(x0[0], b0[0], m[0]); m[1] = E::mfma(x1[0], b1[0], m[1]);
     m[2] = E::mfma(x2[0], b2[0], m[2]); m[3] = E::mfma(x3[0], b3[0], m[3]);
     c[0] = E::mfma(x0[0], b0[1], c[0]); c[1] = E::mfma(x1[0], b1[1], c[1]);
     c[2] = E::mfma(x2[0], b2[1], c[2]); c[3] = E::mfma(x3[0], b3[1], c[3]);
     c[0] = E::mfma(x0[1], b0[0], c[0]); c[1] = E::mfma(x1[1], b1[0], c[1]);
     c[2] = E::mfma(x2[1], b2[0], c[2]); c[3] = E::mfma(x3[1], b3[0], c[3]);
     if constexpr (NP >= 4) {
          c[0] = E::mfma(x0[0], b0[2], c[0]); c[1] = E::mfma(x1[0], b1[2], c[1]);
          c[2] = E::mfma(x2[0], b2[2], c[2]); c[3] = E::mfma(x3[0], b3[2], c[3]);
     }
     if constexpr (NP == 5) {
          c[0] = E::mfma(x0[1], b0[1], c[0]); c[1] = E::mfma(x1[1], b1[1], c[1]);
          c[2] = E::mfma(x2[1], b2[1], c[2]); c[3] = E::mfma(x3[1], b3[1], c[3]);
     }
}

template <class E, int NP, int NW, class S>
__device__ __forceinline__ void angular_mix_body(const Mix2Args &p, int2 tk) {
     constexpr int NT = S::NT, TM = S::TM, TN = S::TN, G = MIX_G, MA = S::MA, NB = S::NB, ST = S::ST;
     constexpr int SA = mix_sa<S>(), SB = mix_sb<S>();
     __shared__ v4u lds[ST * (SA + SB)];
     static_assert(sizeof(lds) >= sizeof(double) * S::WM * 4 * 8 * TN, "epilogue buffer");
     static_assert(S::WM * 16 * MA == TM && S::WN * 16 * NB == TN && S::WM * S::WN == NT / 64, "wave grid");

     if (tk.x < 0) return;
     const int st = tk.x, jt = tk.y;
     const int it0 = st * TM, jt0 = jt * TN, nch = p.ktile[st] / KM;
     const int lane = threadIdx.x & 63;
     const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
     const int wm = wave % S::WM, wn = wave / S::WM;
     const int l16 = lane & 15, lg = lane >> 4;
     // the first weight channel of this lane's sizes, loaded now so the
     // epilogue does not wait for it
     double w0[MA][4];
#pragma unroll
     for (int a = 0; a < MA; ++a)
#pragma unroll
          for (int v = 0; v < 4; ++v) w0[a][v] = p.W[0][it0 + wm * 16 * MA + 16 * a + mfma16_row(lane, v)];
     const v4u flip = {0x80000000u, 0x80000000u, 0x80000000u, 0x80000000u};
     // stage buffer b: A rows at lds + b (SA + SB), B rows after them
     auto sA = [&](int b_) { return lds + b_ * (SA + SB); };
     auto sB = [&](int b_) { return lds + b_ * (SA + SB) + SA; };

     // leading product and corrections (the same accumulators without SEP)
     v4f am[MA][NB][8], ac_[S::SEP ? MA : 1][S::SEP ? NB : 1][8];
#pragma unroll
     for (int a = 0; a < MA; ++a)
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
               for (int k = 0; k < 8; ++k) am[a][b][k] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
     for (int a = 0; a < (S::SEP ? MA : 1); ++a)
#pragma unroll
          for (int b = 0; b < (S::SEP ? NB : 1); ++b)
#pragma unroll
               for (int k = 0; k < 8; ++k) ac_[a][b][k] = v4f{0.f, 0.f, 0.f, 0.f};
     auto acc_c = [&](int a, int b) -> v4f * { if constexpr (S::SEP) return ac_[a][b]; else return am[a][b]; };

     // stages 0 .. ST-2 in flight before the loop; stage c + ST - 1 is issued
     // at stage c into the buffer of stage c - 1
#pragma unroll
     for (int c = 0; c < ST - 1; ++c)
          if (c < nch) mix_stage_load<S>(p, sA(c), sB(c), c, it0, jt0, wave, lane);
     for (int c = 0; c < nch; ++c) {
          const int buf = c % ST;
          // this wave's rows of stage c have landed; after the barrier every
          // wave's have, and every wave is done with stage c - 1
          __builtin_amdgcn_s_waitcnt(0);
          // the plain barrier: each wave has waited for its own rows above, and
          // a workgroup fence here would also wait for the younger stages
          __builtin_amdgcn_s_barrier();
          __asm__ volatile("" ::: "memory");
          if (c + ST - 1 < nch) {
               const int nb = (c + ST - 1) % ST;
               mix_stage_load<S>(p, sA(nb), sB(nb), c + ST - 1, it0, jt0, wave, lane);
          }
          // B fragments of the angle blocks: (pi+tau) h/m/l, (pi-tau) h/m/l
          v4u bp[NB][3], bm[NB][3];
#pragma unroll
          for (int b = 0; b < NB; ++b) {
               const int jc = wn * 16 * NB + 16 * b + l16;
#pragma unroll
               for (int q = 0; q < 3; ++q) {
                    bp[b][q] = sB(buf)[(q * G + lg) * TN + jc];
                    bm[b][q] = sB(buf)[((3 + q) * G + lg) * TN + jc];
               }
          }
#pragma unroll
          for (int a = 0; a < MA; ++a) {
               const int ic = wm * 16 * MA + 16 * a + l16;
               v4u x[8];
#pragma unroll
               for (int k = 0; k < 8; ++k) x[k] = sA(buf)[(k * G + lg) * TM + ic];
               // +mu: sp = S (pi+tau), sm = T (pi-tau)
#pragma unroll
               for (int b = 0; b < NB; ++b)
                    mix_products<E, NP>(x + 0, bp[b], x + 2, bp[b], x + 4, bm[b], x + 6, bm[b], am[a][b], acc_c(a, b));
               // -mu: the odd orders change sign, sp = s S (pi-tau), sm = s T (pi+tau)
#pragma unroll
               for (int k = 0; k < 8; ++k) x[k] ^= flip;
#pragma unroll
               for (int b = 0; b < NB; ++b)
                    mix_products<E, NP>(x + 0, bm[b], x + 2, bm[b], x + 4, bp[b], x + 6, bp[b], am[a][b] + 4,
                                        acc_c(a, b) + 4);
          }
     }

     // epilogue: the sums in double (leading product plus corrections), the
     // Stokes elements, weighted sums over this lane's sizes per angle; the
     // partial sums of every (wave row block, lane group) go to LDS and one
     // thread per output adds them (no cross-lane shuffles), one weight
     // channel at a time (the Stokes elements are recomputed per channel), so
     // few doubles are live beside the accumulators
     const double unscale = 1. / (kSA * kSB);
     double *sR = (double *) lds;            // [WM][4 lane groups][8][TN]
     __syncthreads();                        // every wave is done with the stages
     double *out = p.part + (size_t) st * NW * 4 * p.Q;
#pragma unroll
     for (int c = 0; c < NW; ++c) {
          if (c > 0) __syncthreads();        // the previous channel's sums are read
#pragma unroll
          for (int b = 0; b < NB; ++b) {
               const int jl = wn * 16 * NB + 16 * b + l16;
               double ew[8];
#pragma unroll
               for (int k = 0; k < 8; ++k) ew[k] = 0.;
#pragma unroll
               for (int a = 0; a < MA; ++a)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                         const v4f *qm = am[a][b], *qc = acc_c(a, b);
                         double q[8];
#pragma unroll
                         for (int k = 0; k < 8; ++k)
                              q[k] = (S::SEP ? (double) qm[k][v] + (double) qc[k][v] : (double) qm[k][v]) * unscale;
                         const int i = it0 + wm * 16 * MA + 16 * a + mfma16_row(lane, v);
                         double Pp[4], Pm[4];
                         stokes(q[0], q[1], q[2], q[3], Pp);
                         stokes(q[4], q[5], q[6], q[7], Pm);
                         const double wv = c == 0 ? w0[a][v] : p.W[c][i];
#pragma unroll
                         for (int k = 0; k < 4; ++k) {
                              ew[k] += wv * Pp[k];
                              ew[4 + k] += wv * Pm[k];
                         }
                    }
#pragma unroll
               for (int k = 0; k < 8; ++k) sR[((wm * 4 + lg) * 8 + k) * TN + jl] = ew[k];
          }
          __syncthreads();
          for (int e = threadIdx.x; e < 8 * TN; e += NT) {
               const int jl = e % TN, k = e / TN, j = jt0 + jl;
               if (j >= p.H) continue;
               double v = 0.;
#pragma unroll
               for (int m = 0; m < S::WM * 4; ++m) v += sR[(m * 8 + k) * TN + jl];
               // k < 4: direct angle H + j; k >= 4: mirrored angle H - 1 - j
               out[((size_t) c * 4 + (k & 3)) * p.Q + (k < 4 ? p.H + j : p.H - 1 - j)] = v;
          }
     }
}
template <class E, int NP, int NW, class S>
__global__ __launch_bounds__(S::NT) __attribute__((amdgpu_waves_per_eu(S::NT / 256 * S::OCC)))
void angular_mix(Mix2Args p) {
     angular_mix_body<E, NP, NW, S>(p, p.task[blockIdx.x]);
}
// angular_mix over the cases of a batch: one task list for all cases, task
// (size tile, angle tile | case << 16), padding tasks (-1, case << 16).
template <class E, int NP, int NW, class S>
__global__ __launch_bounds__(S::NT) __attribute__((amdgpu_waves_per_eu(S::NT / 256 * S::OCC)))
void angular_mix_b(const Mix2Args *cases, const int2 *task) {
     const int2 t = task[blockIdx.x];
     const Mix2Args p = cases[t.y >> 16];
     angular_mix_body<E, NP, NW, S>(p, make_int2(t.x, t.y & 0xffff));
}


// ---------------------------------------------------------------------------
// Reverse pass.
//
// Transpose of the expansion (misc/rtutil_scat_int.c:63-230 read backwards):
// from the cotangents of the raw coefficients to the cotangents of the raw
// matrix elements F11, F33, F12, F34 at the Gauss angles.  Two kernels: the
// sums over l in chunks of EXA_L (one thread per positive node j and chunk,
// partials [chunk][24][Hp]), then the fixed-order sum over chunks.
constexpr int EXA_L = 32;

template <bool G, bool L>
__device__ __forceinline__ void expand_adjoint_part_of(const double *T, const double *gbar, const double *lbar, int H, int Hp, int C, double *part) {
     const int j = blockIdx.x * blockDim.x + threadIdx.x, ck = blockIdx.y;
     if (j >= Hp) return;
     typedef double d2 __attribute__((ext_vector_type(2)));
     const size_t plane = gsf_plane(C, Hp) / 2;
     const d2 *T2 = (const d2 *) T;
     double Em[6] = {0, 0, 0, 0, 0, 0}, Ep[6] = {0, 0, 0, 0, 0, 0};   // GSF rows
     double Lm[6] = {0, 0, 0, 0, 0, 0}, Lp[6] = {0, 0, 0, 0, 0, 0};   // Legendre rows
     const int l1 = min(C, (ck + 1) * EXA_L);
     static_assert(EXA_L % 2 == 0, "whole rows of two l");
     d2 q00 = {0., 0.}, q02 = q00, q22 = q00, q2m = q00, qpl = q00;
     auto step = [&](int l, int u) {
          const double sl = u ? -1. : 1., fl = (2 * l + 1) / 2.;
          if constexpr (G) {
               double cb[6];
               for (int k = 0; k < 6; ++k) cb[k] = gbar[(size_t) k * C + l] * fl;
               const double e1 = (cb[1] + cb[2]) / 2., e2 = (cb[1] - cb[2]) / 2.;
               const double p00 = q00[u], p02 = q02[u], p22 = q22[u], p2m = q2m[u];
               Em[0] += sl * cb[0] * p00;  Ep[0] += cb[0] * p00;
               Em[1] += sl * e1 * p2m;     Ep[1] += e1 * p22;
               Em[2] += sl * e2 * p22;     Ep[2] += e2 * p2m;
               Em[3] += sl * cb[3] * p00;  Ep[3] += cb[3] * p00;
               Em[4] += sl * cb[4] * p02;  Ep[4] += cb[4] * p02;
               Em[5] += sl * cb[5] * p02;  Ep[5] += cb[5] * p02;
          }
          if constexpr (L) {
               const double pl = qpl[u];
               for (int k = 0; k < 6; ++k) {
                    const double c = lbar[(size_t) k * C + l] * fl * (k == 5 ? -1. : 1.);
                    Lm[k] += sl * c * pl;
                    Lp[k] += c * pl;
               }
          }
     };
     auto load = [&](int l) {
          const size_t o = (size_t) (l / 2) * Hp + j;
          if constexpr (G) { q00 = T2[o]; q02 = T2[plane + o]; q22 = T2[2 * plane + o]; q2m = T2[3 * plane + o]; }
          if constexpr (L) qpl = T2[4 * plane + o];
     };
     if (j < H) {
          int l = ck * EXA_L;
          // four pairs' loads in flight (a pair at a time waited for memory 16 times a
          // chunk: 17.5 us of 255 nodes and 510 l, now 11.3; 32 cases 37 and 29)
#pragma unroll 4
          for (; l + 2 <= l1; l += 2) {
               load(l);
               step(l, 0);
               step(l + 1, 1);
          }
          if (l < l1) {
               load(l);
               step(l, 0);
          }
     }
     double *out = part + (size_t) ck * 24 * Hp + j;
     for (int k = 0; k < 6; ++k) {
          out[(size_t) k * Hp] = Em[k];
          out[(size_t) (6 + k) * Hp] = Ep[k];
          out[(size_t) (12 + k) * Hp] = Lm[k];
          out[(size_t) (18 + k) * Hp] = Lp[k];
     }
}
// (the kinds of cotangents as template arguments: no branch in the loop, so the
// loads of several l are in flight)
__device__ __forceinline__ void expand_adjoint_part_body(const double *T, const double *gbar, const double *lbar, int H, int Hp, int C, double *part) {
     if (gbar && lbar) expand_adjoint_part_of<true, true>(T, gbar, lbar, H, Hp, C, part);
     else if (gbar) expand_adjoint_part_of<true, false>(T, gbar, lbar, H, Hp, C, part);
     else expand_adjoint_part_of<false, true>(T, gbar, lbar, H, Hp, C, part);
}
__global__ __launch_bounds__(64) void expand_adjoint_part(const double *T, const double *gbar, const double *lbar, int H, int Hp, int C, double *part) { expand_adjoint_part_body(T, gbar, lbar, H, Hp, C, part); }
struct expand_adjoint_part_B {
     const double *T;
     const double *gbar;
     const double *lbar;
     int H;
     int Hp;
     int C;
     double *part;
     unsigned gx, gy;
};
__global__ __launch_bounds__(64) void expand_adjoint_part_b(const expand_adjoint_part_B *cases) {
     const expand_adjoint_part_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     expand_adjoint_part_body(a.T, a.gbar, a.lbar, a.H, a.Hp, a.C, a.part);
}


// Sums of the chunk partials: a workgroup of 32 nodes x 24 rows, one thread
// per (node, row) adding the chunks in order, then the row combinations per
// node through LDS.
constexpr int EXF_J = 32;
// adjw: the halved combinations that the FP64 reverse contraction takes
// (AdjArgs::wts), zero up to a whole stage of angles past H, or NULL.
__device__ __forceinline__ void expand_adjoint_fin_body(const double *part, int nck, const double *w, int H, int Hp, int Q, double *pfbar,
                                                        double *adjw) {
     __shared__ double sv[24][EXF_J];
     const int jj = threadIdx.x % EXF_J, k = threadIdx.x / EXF_J, j = blockIdx.x * EXF_J + jj;
     double v = 0.;
     if (j < H) {
          const double *pk = part + (size_t) k * Hp + j;
          const size_t step = (size_t) 24 * Hp;
          int ck = 0;
          for (; ck + 8 <= nck; ck += 8) {   // eight loads in flight, added in order
               double t[8];
#pragma unroll
               for (int e = 0; e < 8; ++e) t[e] = pk[(size_t) (ck + e) * step];
#pragma unroll
               for (int e = 0; e < 8; ++e) v += t[e];
          }
          for (; ck < nck; ++ck) v += pk[(size_t) ck * step];
     }
     sv[k][jj] = v;
     __syncthreads();
     if (k) return;
     if (j >= H) {
          if (adjw && j < Hp)
               for (int r = 0; r < 8; ++r) adjw[(size_t) j * 8 + r] = 0.;
          return;
     }
     double vv[24];
     for (int r = 0; r < 24; ++r) vv[r] = sv[r][jj];
     const int ip = H + j, im = H - 1 - j;
     const double wq = w[ip];
     for (int s = 0; s < 2; ++s) {
          const double *E = vv + (s ? 6 : 0), *L = vv + (s ? 18 : 12);
          const int a = s ? ip : im;
          const double p0 = wq * (E[0] + E[1] + E[2] + L[0] + L[1]), p1 = wq * (E[1] - E[2] + E[3] + L[2] + L[3]);
          const double p2 = wq * (E[4] + L[4]), p3 = wq * (E[5] + L[5]);
          pfbar[a] = p0;
          pfbar[Q + a] = p1;
          pfbar[2 * Q + a] = p2;
          pfbar[3 * Q + a] = p3;
          if (adjw) {
               double *o = adjw + (size_t) j * 8 + (s ? 0 : 4);
               o[0] = .5 * (p0 + p1);
               o[1] = .5 * (p0 - p1);
               o[2] = .5 * p2;
               o[3] = .5 * p3;
          }
     }
}
__global__ __launch_bounds__(24 * EXF_J) void expand_adjoint_fin(const double *part, int nck, const double *w, int H, int Hp, int Q, double *pfbar, double *adjw) { expand_adjoint_fin_body(part, nck, w, H, Hp, Q, pfbar, adjw); }
struct expand_adjoint_fin_B {
     const double *part;
     int nck;
     const double *w;
     int H;
     int Hp;
     int Q;
     double *pfbar;
     unsigned gx, gy;
};
__global__ __launch_bounds__(24 * EXF_J) void expand_adjoint_fin_b(const expand_adjoint_fin_B *cases) {
     const expand_adjoint_fin_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     expand_adjoint_fin_body(a.part, a.nck, a.w, a.H, a.Hp, a.Q, a.pfbar, nullptr);
}


// Cotangents of the two complex sums at one (size, angle) from those of the
// four matrix elements (gradient convention d/dRe + i d/dIm):
//   sp^ = (p0 + p1) sp/2 - (p2 + i p3) sm/2,  sm^ = (p0 - p1) sm/2 - (p2 - i p3) sp/2,
// the adjoint of P11 = (|sp|^2 + |sm|^2)/4, P33 = (|sp|^2 - |sm|^2)/4,
// P12 = -Re(sp sm*)/2, P34 = -Im(sp sm*)/2 (src/lmie_core.c:726-744);
// w = (p0 + p1)/2, (p0 - p1)/2, p2/2, p3/2.
__device__ __forceinline__ void stokes_adj(double spr, double spi, double smr, double smi, const double w[4],
                                           double out[4]) {
     const double a = w[0], c = w[1], p2 = w[2], p3 = w[3];
     out[0] = a * spr - (p2 * smr - p3 * smi);
     out[1] = a * spi - (p2 * smi + p3 * smr);
     out[2] = c * smr - (p2 * spr + p3 * spi);
     out[3] = c * smi - (p2 * spi - p3 * spr);
}

// Angular part of the size-weight cotangent: fbar_i = sum_{j, +-, k} pfbar_k P_k(i, j),
// one wave per size point.
__global__ __launch_bounds__(256) void fbar_angular(const double *sst, const double *pfbar, int N, int Np, int H, int Hp,
                                                    int Q, double *fang) {
     const int lane = threadIdx.x & 63;
     const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
     if (i >= N) return;
     const size_t plane = (size_t) Np * Hp;
     double acc = 0.;
     for (int j = lane; j < H; j += 64) {
          const double *o = sst + (size_t) i * Hp + j;
          double q[8], Pp[4], Pm[4];
#pragma unroll
          for (int c = 0; c < 8; ++c) q[c] = o[c * plane];
          stokes(q[0], q[1], q[2], q[3], Pp);
          stokes(q[4], q[5], q[6], q[7], Pm);
          for (int k = 0; k < 4; ++k)
               acc += pfbar[k * Q + H + j] * Pp[k] + pfbar[k * Q + H - 1 - j] * Pm[k];
     }
     for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
     if (lane == 0) fang[i] = acc;
}

// waits until at most n of this wave's vector memory operations are in
// flight (vmcnt in bits 3:0 and 15:14) and its LDS reads have returned (lgkmcnt 0, so
// a barrier behind it frees the buffer they read); expcnt left open
template <int n>
__device__ __forceinline__ void wait_vm() {
     static_assert(n < 64, "vmcnt field");
     __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | ((n >> 4) << 14));
}

// Transposed angular contraction on FP64 matrix cores: for every size i and
// order n,
//   Sbar_n = f_i sum_j [sp^+ (pi+tau)_n + s_n sp^- (pi-tau)_n],
//   Tbar_n = f_i sum_j [sm^+ (pi-tau)_n + s_n sm^- (pi+tau)_n],
// K = the positive angles.  Both operands lie along K in memory (the checkpointed
// sums [8][Np][Hp], the tables [Kp][Hp]), so a stage of ADJ_KS = 8 angles is 64
// bytes a row, filled by direct loads (16 bytes a lane, 16 rows a load).  LDS rows
// have no padding; the four 16-byte pieces of row r sit at piece ^ (r / 4 & 3)
// (each lane fetches the piece its place belongs to), so the 16 rows x 2 angles that
// half a wave reads fall in different banks.  A wave owns 16 sizes x 16 BO orders,
// 4 sums each; it forms the cotangents of its 16 sizes from the sums and the
// angle's weights in registers (28 operations for BO x 8 matrix instructions), so
// no pass over the checkpoint writes them.  Four waves (2 x 2) share a tile of 32
// sizes and its two stages, one barrier each, one stage ahead; three workgroups
// per CU.
// What bounds it: the FP64 matrix cores (64 cycles per instruction and SIMD), at about
// 85% of the rate of angular_f64 (two modes of 32768 sizes, 3810 angles: 17.8 ms with
// the passes around it, 14.3 for the same products there): the cotangents' vector
// operations, and half lines per row and stage.
constexpr int ADJ_KS = 8;

// Orders per task of the contraction over size tiles of 32 with kt orders each:
// 64 (three of every four products then share their cotangents with another)
// unless the tasks of 32 are all resident at once (three workgroups on each of
// 256 CUs) and leave the fullest CU less to do: it gets ceil(tasks / 256) tasks of
// one unit, or half as many of two.  Measured, 32 and 64: 1024 sizes of up to 135
// orders (91 and 53 tasks) 48 and 58 us for the angular part, 3965 of 251 (577, 319)
// 121 and 134, 2048 of 372 (424, 227) 126 and 122, 4096 of 372 (842, 452) 200 and
// 184, 16384 of 954 (8063, 4159) 3150 and 2660.  128 orders on eight waves gave
// the same as 64; stages of 16 angles, which leave one workgroup to a CU, 3040-3650.
// The kernel before (32 x 32, the checkpoint by size and angle, staged through
// registers) took 65, 215, 260, 394 and 6490.
int adj_f64_orders(const std::vector<int> &kt) {
     int t32 = 0, t64 = 0;
     for (int k : kt) {
          t32 += (k + 31) / 32;
          t64 += (k + 63) / 64;
     }
     return t32 <= 3 * 256 && (t32 + 255) / 256 < 2 * ((t64 + 255) / 256) ? 32 : 64;
}

struct AdjArgs {
     int Np, Kp, Hp, H;
     const double *sst;         // [8][Np][Hp]
     const double *wts;         // [Hp + 8][8]: stokes_adj's w at +mu_j, then at -mu_j
     const double *Bp, *Bm;     // [Kp][Hp]
     const double *f;           // [Np]
     const int2 *task;          // (size tile, order tile), (-1, -1) none
     double *bar;               // [4][Kp][Np]: Sbar re, im, Tbar re, im
};

template <int BO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void angular_adj_f64(AdjArgs p) {
     constexpr int WO = 2, WI = 2, NW = WO * WI, KS = ADJ_KS, TO = 16 * WO * BO, TI = 16 * WI;
     constexpr int XSTG = 8 * TI * KS, BSTG = 2 * TO * KS, STG = XSTG + BSTG + 128;
     constexpr int NL = (XSTG + BSTG) / (128 * NW);   // direct loads per wave and stage, and the weights'
     static_assert((XSTG + BSTG) % (128 * NW) == 0 && XSTG % 128 == 0, "whole 1 KiB loads");
     __shared__ double sh[2 * STG];

     const int2 tk = p.task[blockIdx.x];
     if (tk.x < 0) return;
     const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
     const int wo = wave % WO, wi = wave / WO;
     const int l16 = lane & 15, lg = lane >> 4;
     const int it0 = tk.x * TI, n0 = tk.y * TO;
     const size_t Np = p.Np, Hp = p.Hp, plane = (size_t) p.Kp * Np, splane = Np * Hp;

     // this lane's source of each of the wave's loads (row, swizzled piece) at
     // angle 0; rows past the tables are clamped (their orders are not stored)
     const double *src[NL];
#pragma unroll
     for (int u = 0; u < NL; ++u) {
          const int e = (wave + NW * u) * 128 + 2 * lane;
          const int row = (e < XSTG ? e : e - XSTG) / KS, piece = (lane & 3) ^ (row >> 2 & 3);
          if (e < XSTG) src[u] = p.sst + (row / TI) * splane + (size_t) (it0 + row % TI) * Hp + 2 * piece;
          else src[u] = (row / TO ? p.Bm : p.Bp) + (size_t) min(n0 + row % TO, p.Kp - 1) * Hp + 2 * piece;
     }
     const double *wsrc = p.wts + 2 * lane;
     auto stage_load = [&](int buf) {
#pragma unroll
          for (int u = 0; u < NL; ++u) {
               __builtin_amdgcn_global_load_lds((const void *) src[u], (lds_ptr) (sh + buf * STG + (wave + NW * u) * 128), 16, 0, 0);
               src[u] += KS;
          }
          // 1 KiB of weights: this stage's 8 angles and the next 8 (unused)
          if (wave == 0) __builtin_amdgcn_global_load_lds((const void *) wsrc, (lds_ptr) (sh + buf * STG + XSTG + BSTG), 16, 0, 0);
          wsrc += KS * 8;
     };

     v4d acc[BO][4];
#pragma unroll
     for (int b = 0; b < BO; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[b][q] = v4d{0., 0., 0., 0.};
     // s_n of this lane's table rows n0 + ... + l16 (row n holds order n + 1)
     const unsigned long long sgn = (unsigned long long) (l16 & 1) << 63;
     auto flip = [&](double v) { return __longlong_as_double((long long) ((unsigned long long) __double_as_longlong(v) ^ sgn)); };
     // this lane's angle 4 ks + lg of row l16 in a tile of rows
     const int o0 = l16 * KS + (((lg >> 1) ^ (l16 >> 2 & 3)) << 1) + (lg & 1);
     const int nst = (p.H + KS - 1) / KS;
     if (nst > 0) stage_load(0);
     for (int k = 0; k < nst; ++k) {
          const int buf = k & 1;
          wait_vm<0>();                           // this wave's loads of the stage
          __builtin_amdgcn_s_barrier();           // everyone's; the other buffer is free
          __asm__ volatile("" ::: "memory");
          if (k + 1 < nst) stage_load(buf ^ 1);
          const double *x0 = sh + buf * STG + 16 * wi * KS, *b0 = sh + buf * STG + XSTG + 16 * BO * wo * KS;
          const double *w0 = sh + buf * STG + XSTG + BSTG + lg * 8;
#pragma unroll
          for (int ks = 0; ks < KS / 4; ++ks) {
               const int o = o0 ^ (4 * ks);       // pieces 0, 1 <-> 2, 3
               double x[8], wq[8], xp[4], xm[4];
#pragma unroll
               for (int c = 0; c < 8; ++c) x[c] = x0[c * TI * KS + o];
#pragma unroll
               for (int c = 0; c < 8; ++c) wq[c] = w0[ks * 32 + c];
               stokes_adj(x[0], x[1], x[2], x[3], wq, xp);          // sp^+, sm^+
               stokes_adj(x[4], x[5], x[6], x[7], wq + 4, xm);      // sp^-, sm^-
#pragma unroll
               for (int b = 0; b < BO; ++b) {
                    const double bp = b0[16 * b * KS + o], bm = b0[(TO + 16 * b) * KS + o];
                    const double sbp = flip(bp), sbm = flip(bm);
                    v4d *q = acc[b];
                    q[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(bp, xp[0], q[0], 0, 0, 0);
                    q[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(bp, xp[1], q[1], 0, 0, 0);
                    q[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(bm, xp[2], q[2], 0, 0, 0);
                    q[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(bm, xp[3], q[3], 0, 0, 0);
                    q[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(sbm, xm[0], q[0], 0, 0, 0);
                    q[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(sbm, xm[1], q[1], 0, 0, 0);
                    q[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(sbp, xm[2], q[2], 0, 0, 0);
                    q[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(sbp, xm[3], q[3], 0, 0, 0);
               }
          }
     }
     // result rows (orders) l / 16 + 4 v, column (size) l % 16
     const int i = it0 + 16 * wi + l16;
     const double fi = p.f[i];
#pragma unroll
     for (int b = 0; b < BO; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
               const int n = n0 + 16 * (BO * wo + b) + lg + 4 * v;
               if (n >= p.Kp) continue;
#pragma unroll
               for (int c = 0; c < 4; ++c) p.bar[c * plane + (size_t) n * Np + i] = fi * acc[b][c][v];
          }
}

// ---------------------------------------------------------------------------
// Reverse pass of the mixed path through the order-by-order kernel matrix.
//
// The cotangents of the four complex sums at an angle are linear in the sums
// (stokes_adj): at +mu_j sp^ = a_j sp - beta_j sm, sm^ = c_j sm - conj(beta_j) sp
// with a = (p0 + p1)/2, c = (p0 - p1)/2, beta = (p2 + i p3)/2 of that angle's
// matrix-element cotangents, and likewise (a', c', beta') at -mu_j.  Putting
// the forward sums sp = sum_m S_m (pi+tau)_m, ... into the transposed
// contraction gives, for every size,
//   Sbar_n = f (sum_m Gss(n,m) S_m - Gst(n,m) T_m)
//   Tbar_n = f (sum_m Gtt(n,m) T_m - conj(Gst(m,n)) S_m)
// with the size-independent matrices (P+- = pi +- tau at the positive nodes,
// s_n s_m = (-1)^(n+m) from the mirrored nodes)
//   Gss = sum_j a_j P+_n P+_m + s_n s_m a'_j P-_n P-_m,   Gtt = sum_j c_j P-_n P-_m + s_n s_m c'_j P+_n P+_m,
//   Gst = sum_j beta_j P+_n P-_m + s_n s_m beta'_j P-_n P+_m,
// and the angular part of the size-weight cotangent is the quadratic form
// sum_j pfbar . P(i, j) = 1/2 sum_n Re(conj S_n U_S,n + conj T_n U_T,n), U = Sbar / f.
// So the reverse contraction needs no per-(size, angle) checkpoint: five
// kernels build the weights, the split tables, G (split 16-bit, fp32
// accumulation), its split operand, and U = G A on the matrix cores.
struct AdjScal {
     double wmax;               // largest |weight| (weights are stored divided by it)
     unsigned gmax;             // bits of the largest |G| (non-negative float)
};

// Weights of the eight right-hand tables per positive node j (row q of wts):
// a, a', c, c', beta_r, beta_i, beta'_r, beta'_i, divided by their largest
// magnitude.  One workgroup.
__device__ __forceinline__ void adj_weights_body(const double *pfbar, int H, int Hq, int Q, double *wts, AdjScal *sc) {
     __shared__ double red[1024];
     double mx = 0.;
     for (int j = threadIdx.x; j < H; j += blockDim.x)
          for (int k = 0; k < 4; ++k)
               mx = fmax(mx, fmax(fabs(pfbar[k * Q + H + j]), fabs(pfbar[k * Q + H - 1 - j])));
     red[threadIdx.x] = mx;
     __syncthreads();
     for (int o = blockDim.x / 2; o > 0; o >>= 1) {
          if ((int) threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
          __syncthreads();
     }
     // |a|, |c| <= max(|p0|, |p1|) and |beta parts| <= |p| / 2: the bound of the pfbar
     // magnitudes bounds every weight
     const double wmax = red[0] > 0. ? red[0] : 1., iw = 1. / wmax;
     for (int j = threadIdx.x; j < Hq; j += blockDim.x) {
          double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
          if (j < H) {
               const double *pp = pfbar + H + j, *pm = pfbar + H - 1 - j;
               v[0] = .5 * (pp[0] + pp[Q]);
               v[1] = .5 * (pm[0] + pm[Q]);
               v[2] = .5 * (pp[0] - pp[Q]);
               v[3] = .5 * (pm[0] - pm[Q]);
               v[4] = .5 * pp[2 * Q];
               v[5] = .5 * pp[3 * Q];
               v[6] = .5 * pm[2 * Q];
               v[7] = .5 * pm[3 * Q];
          }
          for (int q = 0; q < 8; ++q) wts[(size_t) q * Hq + j] = v[q] * iw;
     }
     if (threadIdx.x == 0) {
          sc->wmax = wmax;
          sc->gmax = 0u;
     }
}
__global__ __launch_bounds__(1024) void adj_weights(const double *pfbar, int H, int Hq, int Q, double *wts, AdjScal *sc) { adj_weights_body(pfbar, H, Hq, Q, wts, sc); }
struct adj_weights_B {
     const double *pfbar;
     int H;
     int Hq;
     int Q;
     double *wts;
     AdjScal *sc;
     unsigned gx, gy;
};
__global__ __launch_bounds__(1024) void adj_weights_b(const adj_weights_B *cases) {
     const adj_weights_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     adj_weights_body(a.pfbar, a.H, a.Hq, a.Q, a.wts, a.sc);
}


// Split tables with angles along the contraction: [plane][Hq / 8][Kq][8],
// 8 consecutive positive nodes per 16 bytes, from the forward's split tables
// B16 ([6][Kb][Hb][8], orders along the contraction): left (4 planes) P+ and
// P- of order r + 1 over r (r + 1) (r + 2) times kSB, high and middle parts
// (two of the B16 parts, transposed); right (16 planes) weight q times P+
// (q = 0, 3, 6, 7) or P- (q = 1, 2, 4, 5), from P = high + middle + low,
// high and low parts.  One thread per (order, group of 8 nodes).
template <class E>
__device__ __forceinline__ void adj_tables_body(const unsigned short *B16, int Kb, int Hb, const double *wts, int H, int Hq, int Kq, int n1max, unsigned short *L16, unsigned short *R16) {
     const int r = blockIdx.x * 64 + threadIdx.x, jg = blockIdx.y;
     if (r >= Kq) return;
     const size_t plane = (size_t) (Hq / 8) * Kq * 8, o = ((size_t) jg * Kq + r) * 8, bpl = (size_t) Kb * Hb * 8;
     unsigned short lv[4][8], rv[16][8];
     for (int e = 0; e < 8; ++e) {
          const int j = 8 * jg + e;
          double pp = 0., pm = 0.;
          if (j < H && r < n1max) {
               const size_t bo = ((size_t) (r / 8) * Hb + j) * 8 + (r % 8);
               lv[0][e] = B16[0 * bpl + bo];
               lv[1][e] = B16[1 * bpl + bo];
               lv[2][e] = B16[3 * bpl + bo];
               lv[3][e] = B16[4 * bpl + bo];
               pp = E::value(lv[0][e]) + E::value(lv[1][e]) + E::value(B16[2 * bpl + bo]);
               pm = E::value(lv[2][e]) + E::value(lv[3][e]) + E::value(B16[5 * bpl + bo]);
          } else {
#pragma unroll
               for (int q = 0; q < 4; ++q) lv[q][e] = 0;
          }
          for (int q = 0; q < 8; ++q) {
               const bool plus = q == 0 || q == 3 || q == 6 || q == 7;
               // the planes of the sigma-sigma products (q = 1, 3, 6, 7) carry
               // sigma_m = (-1)^r of their order (an exact sign change)
               const bool odd = (q == 1 || q == 3 || q == 6 || q == 7) && (r & 1);
               const double v = wts[(size_t) q * Hq + j] * (plus ? pp : pm);
               split16<E>(odd ? -v : v, &rv[2 * q][e], &rv[2 * q + 1][e]);
          }
     }
     for (int q = 0; q < 4; ++q) {
          v4u w;
          for (int k = 0; k < 4; ++k) w[k] = (unsigned) lv[q][2 * k] | ((unsigned) lv[q][2 * k + 1] << 16);
          *(v4u *) (L16 + q * plane + o) = w;
     }
     for (int q = 0; q < 16; ++q) {
          v4u w;
          for (int k = 0; k < 4; ++k) w[k] = (unsigned) rv[q][2 * k] | ((unsigned) rv[q][2 * k + 1] << 16);
          *(v4u *) (R16 + q * plane + o) = w;
     }
}
template <class E>
__global__ __launch_bounds__(64) void adj_tables(const unsigned short *B16, int Kb, int Hb, const double *wts, int H, int Hq, int Kq, int n1max, unsigned short *L16, unsigned short *R16) { adj_tables_body<E>(B16, Kb, Hb, wts, H, Hq, Kq, n1max, L16, R16); }
struct adj_tables_B {
     const unsigned short *B16;
     int Kb;
     int Hb;
     const double *wts;
     int H;
     int Hq;
     int Kq;
     int n1max;
     unsigned short *L16;
     unsigned short *R16;
     unsigned gx, gy;
};
template <class E>
__global__ __launch_bounds__(64) void adj_tables_b(const adj_tables_B *cases) {
     const adj_tables_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     adj_tables_body<E>(a.B16, a.Kb, a.Hb, a.wts, a.H, a.Hq, a.Kq, a.n1max, a.L16, a.R16);
}


// G on the 32x32x16 matrix instruction: one workgroup per 64 x 64 tile of
// (n, m), four waves of 32 x 32, contraction over the positive nodes in
// stages of 16 (two LDS stages, 80 KiB: two workgroups per CU).  Each G
// element is a sum of two products, the second with the factor
// sigma_n sigma_m = (-1)^(n+m): the right planes of those products carry
// sigma_m (adj_tables) and the left fragment is negated on the lanes of odd
// rows, so both products accumulate into one accumulator:
// 0 P+ a P+ + P- a' P-, 1 P- c P- + P+ c' P+, 2 P+ br P- + P- b'r P+,
// 3 P+ bi P- + P- b'i P+.  Output in fp32, Gf[4][Kq][Kq] = Gss, Gtt, Re Gst,
// Im Gst (row n, column m, scaled by kSB^2 / (wmax n (n+1) m (m+1))), and the
// largest magnitude.
template <class E>
__device__ __forceinline__ void adj_gbuild_body(const unsigned short *L16, const unsigned short *R16, int Hq, int Kq, float *Gf, AdjScal *sc,
                                                int tn, int tm) {
     constexpr int T = 64, G = 2, KS = 8 * G;
     constexpr int NL = 4 * G * T / 256, NR = 16 * G * T / 256;
     __shared__ v4u sL[2][4 * G][T];
     __shared__ v4u sR[2][16 * G][T];
     const int n0 = tn * T, m0 = tm * T, nch = Hq / KS;
     const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
     const int wa = wave & 1, wb = wave >> 1, l32 = lane & 31, lh = lane >> 5;
     const size_t plane = (size_t) (Hq / 8) * Kq * 8;
     // odd rows n (lane parity) negate the left fragment of the sigma-sigma products
     const unsigned sg = (lane & 1) ? 0x80008000u : 0u;
     const v4u neg = {sg, sg, sg, sg};
     v4u rl[NL], rr[NR];
     const Stager<256, T, G> stL(L16, plane, (size_t) Kq * 8, n0, threadIdx.x);
     const Stager<256, T, G> stR(R16, plane, (size_t) Kq * 8, m0, threadIdx.x);
     auto load = [&](int c) {
#pragma unroll
          for (int t = 0; t < NL; ++t) rl[t] = *stL.at(t, c);
#pragma unroll
          for (int t = 0; t < NR; ++t) rr[t] = *stR.at(t, c);
     };
     auto store = [&](int s) {
#pragma unroll
          for (int t = 0; t < NL; ++t) {
               const int e = threadIdx.x + 256 * t;
               sL[s][e / T][e % T] = rl[t];
          }
#pragma unroll
          for (int t = 0; t < NR; ++t) {
               const int e = threadIdx.x + 256 * t;
               sR[s][e / T][e % T] = rr[t];
          }
     };
     v16f acc[4];
#pragma unroll
     for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[k][v] = 0.f;
     load(0);
     store(0);
     if (nch > 1) load(1);
     for (int c = 0; c < nch; ++c) {
          const int s = c & 1;
          __syncthreads();
          // lane l: row (n or m) l % 32, nodes 8 (l / 32) + e of the stage
          v4u y[16], x[8];
#pragma unroll
          for (int q = 0; q < 16; ++q) y[q] = sR[s][q * G + lh][wb * 32 + l32];
          // left planes: 0 P+ hi, 1 P+ lo, 2 P- hi, 3 P- lo; 4..7 the same
          // negated on odd rows
#pragma unroll
          for (int q = 0; q < 4; ++q) x[q] = sL[s][q * G + lh][wa * 32 + l32];
#pragma unroll
          for (int q = 0; q < 4; ++q) x[4 + q] = x[q] ^ neg;
          if (c + 1 < nch) store(s ^ 1);
          if (c + 2 < nch) load(c + 2);
#define GB(k, L, R) acc[k] = E::mfma32(x[L], y[2 * (R)], acc[k]); acc[k] = E::mfma32(x[L], y[2 * (R) + 1], acc[k]); \
          acc[k] = E::mfma32(x[(L) + 1], y[2 * (R)], acc[k]);
          GB(0, 0, 0) GB(1, 2, 2) GB(2, 0, 4) GB(3, 0, 5)
          GB(0, 6, 1) GB(1, 4, 3) GB(2, 6, 6) GB(3, 6, 7)
#undef GB
     }
     float mx = 0.f;
#pragma unroll
     for (int v = 0; v < 16; ++v) {
          const int r = n0 + wa * 32 + mfma32_row(lane, v);
          const int cm = m0 + wb * 32 + l32;
          const float g0 = acc[0][v], g1 = acc[1][v], g2 = acc[2][v], g3 = acc[3][v];
          const size_t o = (size_t) r * Kq + cm, pl = (size_t) Kq * Kq;
          Gf[o] = g0;
          Gf[pl + o] = g1;
          Gf[2 * pl + o] = g2;
          Gf[3 * pl + o] = g3;
          mx = fmaxf(mx, fmaxf(fmaxf(fabsf(g0), fabsf(g1)), fmaxf(fabsf(g2), fabsf(g3))));
     }
     for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
     if (lane == 0) atomicMax(&sc->gmax, __float_as_uint(mx));
}
// Tile (row tile, column tile) of workgroup id L of a g x g tile grid.  The
// hardware deals workgroup ids round robin over the 8 XCDs, so XCD x runs ids
// x, x + 8, ...; those take the consecutive tiles start_x, start_x + 1, ... of
// the column-major order, so the workgroups in flight on one XCD share one or
// two right-hand column tiles (4 MB each at Kq 1920) and stream the left-hand
// rows together, from that XCD's L2.
__device__ __forceinline__ int2 xcd_tile(int L, int g) {
     const int nt = g * g, x = L & 7, k = L >> 3, q = nt >> 3, r = nt & 7;
     const int t = x * q + min(x, r) + k;
     return make_int2(t % g, t / g);
}
template <class E>
__global__ __launch_bounds__(256) void adj_gbuild(const unsigned short *L16, const unsigned short *R16, int Hq, int Kq, float *Gf, AdjScal *sc) {
     const int2 t = xcd_tile(blockIdx.x, Kq / 64);
     adj_gbuild_body<E>(L16, R16, Hq, Kq, Gf, sc, t.x, t.y);
}
struct adj_gbuild_B {
     const unsigned short *L16;
     const unsigned short *R16;
     int Hq;
     int Kq;
     float *Gf;
     AdjScal *sc;
     unsigned gx, gy;
};
template <class E>
__global__ __launch_bounds__(256) void adj_gbuild_b(const adj_gbuild_B *cases) {
     const adj_gbuild_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     adj_gbuild_body<E>(a.L16, a.R16, a.Hq, a.Kq, a.Gf, a.sc, blockIdx.x, blockIdx.y);
}


// Exponent k with |G| * 2^(14 - k) < 2^14 for every entry (0 for G = 0).
__device__ __forceinline__ int adj_gexp(const AdjScal *sc) {
     const float g = __uint_as_float(sc->gmax);
     if (!(g > 0.f)) return 0;
     int k;
     (void) frexpf(g, &k);
     return k;
}

// Split operand of U = G A: [12][Kq / 8][Kq][8], contraction index m in
// groups of 8, column n: Gss, -Re Gst, Im Gst, Gtt, -Re Gts, Im Gts (high,
// low) with Gts(n, m) = conj Gst(m, n), all times 2^(14 - k).  One thread per
// (group of 8 m, n).
template <class E>
__device__ __forceinline__ void adj_gsplit_body(const float *Gf, const AdjScal *sc, int Kq, unsigned short *G16) {
     const int n = blockIdx.x * 64 + threadIdx.x, mg = blockIdx.y;
     if (n >= Kq) return;
     const double s = ldexp(1., 14 - adj_gexp(sc));
     const size_t pl = (size_t) Kq * Kq, plane = (size_t) (Kq / 8) * Kq * 8, o = ((size_t) mg * Kq + n) * 8;
     unsigned short v[12][8];
     for (int e = 0; e < 8; ++e) {
          const int m = 8 * mg + e;
          const size_t nm = (size_t) n * Kq + m, mn = (size_t) m * Kq + n;
          const double val[6] = {Gf[nm], -(double) Gf[2 * pl + nm], Gf[3 * pl + nm], Gf[pl + nm],
                                 -(double) Gf[2 * pl + mn], -(double) Gf[3 * pl + mn]};
          for (int q = 0; q < 6; ++q) split16<E>(val[q] * s, &v[2 * q][e], &v[2 * q + 1][e]);
     }
     for (int q = 0; q < 12; ++q) {
          v4u w;
          for (int k = 0; k < 4; ++k) w[k] = (unsigned) v[q][2 * k] | ((unsigned) v[q][2 * k + 1] << 16);
          *(v4u *) (G16 + q * plane + o) = w;
     }
}
template <class E>
__global__ __launch_bounds__(64) void adj_gsplit(const float *Gf, const AdjScal *sc, int Kq, unsigned short *G16) { adj_gsplit_body<E>(Gf, sc, Kq, G16); }
struct adj_gsplit_B {
     const float *Gf;
     const AdjScal *sc;
     int Kq;
     unsigned short *G16;
     unsigned gx, gy;
};
template <class E>
__global__ __launch_bounds__(64) void adj_gsplit_b(const adj_gsplit_B *cases) {
     const adj_gsplit_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     adj_gsplit_body<E>(a.Gf, a.sc, a.Kq, a.G16);
}


// Operands of U = G A (adj_ugemm32).  Accumulators: U_S re, im, U_T re, im;
// output Uf[4][Kq][Np] in fp32, unscaled to U = Sbar / f.
struct UArgs {
     int Np, Kb, Kq;
     const unsigned short *A16;     // [8][Kb][Np][8]
     const unsigned short *G16;     // [12][Kq / 8][Kq][8]
     const int *ktile;              // per size tile of 64
     const int2 *task;              // (size tile, order tile), heaviest first
     const AdjScal *sc;
     float *Uf;                     // [4][Kq][Np]
};

// U = G A with the 32x32x16 matrix instruction: one workgroup per (size tile
// of TS, order tile of 64) task, stages of 16 orders in two LDS buffers
// (112 KiB for TS = 128, 80 KiB for TS = 64).  Waves in a grid of TS / 32 / WA
// size blocks x 2 order blocks, each wave 32 orders (matrix rows) x 32 WA
// sizes, 4 accumulators per element (U_S, U_T re, im).  TS = 128, WA = 1:
// eight waves, two per SIMD, which hide each other's LDS and barrier waits;
// WA = 2: four waves, each operand fragment read for twice the products;
// TS = 64: four waves, two workgroups per CU.
template <class E, int WA, int TS, bool B>
__global__ __launch_bounds__(TS * 4 / WA) __attribute__((amdgpu_waves_per_eu(TS == 64 ? 2 : 1)))
void adj_ugemm32(UArgs p0, const UArgs *cases, const int2 *btask) {
     constexpr int TO = 64, G = 2;                           // orders, groups of 8 per stage
     constexpr int NT = TS * 4 / WA, WS = TS / 32 / WA;      // threads, size-block waves
     constexpr int NA = 8 * G * TS / NT, NG = 12 * G * TO / NT;
     static_assert(NA * NT == 8 * G * TS && NG * NT == 12 * G * TO, "staging split");
     __shared__ v4u sA[2][8 * G][TS];
     __shared__ v4u sG[2][12 * G][TO];
     // B: one task list for the cases of a batch, task (size tile, order tile | case << 16)
     int2 tk;
     UArgs p;
     if constexpr (B) {
          const int2 t = btask[blockIdx.x];
          p = cases[t.y >> 16];
          tk = make_int2(t.x, t.y & 0xffff);
     } else {
          p = p0;
          tk = p.task[blockIdx.x];
     }
     if (tk.x < 0) return;
     const int it0 = tk.x * TS, n0 = tk.y * TO, nch = p.ktile[tk.x] / (8 * G);
     const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
     const int wm = wave % WS, wn = wave / WS, l32 = lane & 31, lh = lane >> 5;
     const size_t Np = p.Np, Kq = p.Kq;
     const size_t pA = (size_t) p.Kb * Np * 8, pG = (Kq / 8) * Kq * 8;
     const v4u neg = {0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
     v4u ra[NA], rg[NG];
     const Stager<NT, TS, G> stA(p.A16, pA, Np * 8, it0, threadIdx.x);
     const Stager<NT, TO, G> stG(p.G16, pG, Kq * 8, n0, threadIdx.x);
     auto load = [&](int c) {
#pragma unroll
          for (int t = 0; t < NA; ++t) ra[t] = *stA.at(t, c);
#pragma unroll
          for (int t = 0; t < NG; ++t) rg[t] = *stG.at(t, c);
     };
     auto store = [&](int s) {
#pragma unroll
          for (int t = 0; t < NA; ++t) {
               const int e = threadIdx.x + NT * t;
               sA[s][e / TS][e % TS] = ra[t];
          }
#pragma unroll
          for (int t = 0; t < NG; ++t) {
               const int e = threadIdx.x + NT * t;
               sG[s][e / TO][e % TO] = rg[t];
          }
     };
     v16f acc[WA][4];
#pragma unroll
     for (int a = 0; a < WA; ++a)
#pragma unroll
          for (int k = 0; k < 4; ++k)
#pragma unroll
               for (int v = 0; v < 16; ++v) acc[a][k][v] = 0.f;
     if (nch > 0) {
          load(0);
          store(0);
          load(min(1, nch - 1));
     }
     // terms per accumulator: (G plane pair, A plane hi, A plane lo); A planes
     // 0..7 as A16, 8 = -A+r hi, 9 = -A+r lo, 10 = -A-r hi, 11 = -A-r lo
     constexpr int term[4][3][3] = {{{0, 0, 1}, {1, 4, 5}, {2, 6, 7}},     // U_S re
                                    {{0, 2, 3}, {1, 6, 7}, {2, 10, 11}},   // U_S im
                                    {{3, 4, 5}, {4, 0, 1}, {5, 2, 3}},     // U_T re
                                    {{3, 6, 7}, {4, 2, 3}, {5, 8, 9}}};    // U_T im
     for (int c = 0; c < nch; ++c) {
          const int s = c & 1;
          __syncthreads();
          v4u g[12];
#pragma unroll
          for (int q = 0; q < 12; ++q) g[q] = sG[s][q * G + lh][wn * 32 + l32];
          v4u x[WA][12];
#pragma unroll
          for (int a = 0; a < WA; ++a) {
#pragma unroll
               for (int q = 0; q < 8; ++q) x[a][q] = sA[s][q * G + lh][(wm * WA + a) * 32 + l32];
               x[a][8] = x[a][0] ^ neg;
               x[a][9] = x[a][1] ^ neg;
               x[a][10] = x[a][4] ^ neg;
               x[a][11] = x[a][5] ^ neg;
          }
          // hi x hi, lo(G) x hi(A), hi(G) x lo(A) for every (term, size block,
          // accumulator): 4 WA independent accumulators between dependent products
#pragma unroll
          for (int t = 0; t < 3; ++t) {
#pragma unroll
               for (int pr = 0; pr < 3; ++pr) {
#pragma unroll
                    for (int a = 0; a < WA; ++a)
#pragma unroll
                         for (int k = 0; k < 4; ++k) {
                              const int gp = term[k][t][0], xh = term[k][t][1], xl = term[k][t][2];
                              const v4u gv = g[2 * gp + (pr == 1 ? 1 : 0)];
                              const v4u xv = x[a][pr == 2 ? xl : xh];
                              acc[a][k] = E::mfma32(gv, xv, acc[a][k]);
                         }
               }
               // the stage body is one basic block: the last stages store and
               // load a repeat of the last stage (the other LDS buffer is not
               // read again, the repeated rows are in bounds)
               if (t == 0) {
                    store(s ^ 1);
                    load(min(c + 2, nch - 1));
               }
          }
     }
     // U = acc n (n+1) wmax / (2^(14 - k) kSB^2 kSA); rows are orders
     const double base = p.sc->wmax * ldexp(1., adj_gexp(p.sc) - 14) / (kSB * kSB * kSA);
#pragma unroll
     for (int a = 0; a < WA; ++a)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
               const int r = n0 + wn * 32 + mfma32_row(lane, v);
               const int i = it0 + (wm * WA + a) * 32 + l32;
               const double f = base * (r + 1.) * (r + 2.);
#pragma unroll
               for (int k = 0; k < 4; ++k) p.Uf[((size_t) k * Kq + r) * Np + i] = (float) (acc[a][k][v] * f);
          }
}


// Shape of the reverse contraction (environment LMIE_UGEMM_WAVES, read at
// every call): 8 (default) eight waves on 128 sizes, 4 four waves on 128
// sizes, 2 four waves on 64 sizes with two workgroups per CU.
int ugemm_waves() {
     const char *e = getenv("LMIE_UGEMM_WAVES");
     const int r = e ? atoi(e) : 8;
     return (r == 4 || r == 2) ? r : 8;
}

// Per-size reverse sweep (adjoint of src/lmie_core.c:298-611) over the
// forward's kept recurrences (D_j up to n2 - 1, psi_j, chi_j, the reciprocals
// 1 / (D_{j+1} + (j+1)/z)), in two kernels:
//   rev_orders one thread per (size, chunk of rch orders j in [1, n2)):
//              for j <= n1 the cotangents of a_j, b_j from the angular part
//              (Sbar, Tbar) and the series, through a = (u psi - psi0) /
//              (u zeta - zeta0), u = D/m + j/x and b (v = m D + j/x), to the
//              local cotangent of D_j and the direct part of the cotangent of
//              m; and the adjoint of the downward recurrence
//              D_j = (j+1)/z - 1/(D_{j+1} + (j+1)/z), a first-order linear
//              recurrence upward in j carrying the D cotangent to z = m x,
//              which the chunk returns as an affine function of the carry
//              entering it;
//   rev_carry  one thread per size: chains the chunks, then the per-size totals.
// Outputs per size: the cotangent of m (re, im as d/dRe + i d/dIm), of f_i and
// (when asked for) of x_i.

// Orders per chunk of rev_orders: 64, or 32 where the waves of 64 would not fill
// the chip's 1024 SIMDs once (every chunk forms two orders again, and its twelve
// results go through memory to rev_carry).  Measured, rev_orders + rev_carry: 3965
// sizes of up to 270 orders (315 waves of 64) 68 + 5 us with 64, 38 + 7 with 32, 28 +
// 12 with 16; 16384 sizes to x = 914 155 + 12, 145 + 23, 144 + 44; 32768 to 1848
// 539 + 32, 537 + 61, 565 + 131.  By the case also in a batch, so a case's results are
// the same bits alone and in one (32 cases of 4000 sizes: 436 + 17, 412 + 27, 413 + 48).
int rev_chunk(int Np, int n2rows) { return (size_t) (Np / 64) * ((n2rows + 62) / 64) <= 1024 ? 32 : 64; }

struct RevArgs {
     int N, Np, Kp, n1max, n2rows, rch, nch;
     const double *ft;          // order_factors rows over 0 .. n1max + 1
     const double *x, *f;
     const int *n1, *n2;
     double mr, mi;
     double im1r, im1i, im2r, im2i;   // 1/m, 1/m^2 (uniform, formed on the host)
     const double *D, *PC, *PS; // forward recurrences (the chains, D up to n2 - 1)
     const double *CB;          // [2][Np]
     const double *S;           // series [4][Np]
     const double *bar;         // [4][Kp][Np] f-weighted cotangents (FP64 path), or
     const float *Uf;           // [4][Kq][Np] U = Sbar / f (mixed path; fang from U)
     int Kq;
     const double *fang;        // [Np] (FP64 path), or NULL
     double sb0, sb1, sb2, sb3; // cotangents of the raw sums
     double *scan;              // [nch][REV_ROWS][Np]: P, C0, Q, Z0 (re, im), m cotangent (re, im),
                                // f quadratic form, local x cotangent
     double *mbar;              // [Np / 64][2] m cotangent (re, im) of 64 sizes
     double *fbar;              // [N]
     double *xbar;              // [N] cotangent of x_i, or null (not formed)
};
constexpr int REV_ROWS = 12;

// 1/m and 1/m^2 of m = mr - i mi for the reverse sweep, by Smith's division
static void host_crecip(double br, double bi, double *rr, double *ri) {
     if (fabs(br) >= fabs(bi)) {
          const double t = bi / br, d = br + bi * t;
          *rr = 1. / d;
          *ri = -t / d;
     } else {
          const double t = br / bi, d = br * t + bi;
          *rr = t / d;
          *ri = -1. / d;
     }
}
static void rev_recips(RevArgs &r) {
     const double mr = r.mr, mi = -r.mi;
     host_crecip(mr, mi, &r.im1r, &r.im1i);
     host_crecip(mr * mr - mi * mi, 2. * mr * mi, &r.im2r, &r.im2i);
}

// a_j, b_j for the reverse sweep, with the reciprocals the adjoint reuses:
// ra = 1/(u zeta_j - zeta_{j-1}), rb = 1/(v zeta_j - zeta_{j-1}) of the
// denominators of a and b, u = D/m + j/x, v = m D + j/x; a = (u psi_j -
// psi_{j-1}) ra.  Not the forward's bits (conj(d) / |d|^2 and a product with
// the reciprocal instead of Smith's division; a few ulp): the reverse pass
// needs the values, and d a / d u = (psi_j - a zeta_j) ra reuses ra.  |d|^2
// stays far inside the double range: |d| >= |a numerator| and zeta_j of the
// orders j <= n1(x) grows at most like (2j-1)!! / x^j.
struct AbRev {
     cd a, b, ra, rb;
};
__device__ __forceinline__ AbRev mie_ab_rev(double jx, cd m, cd im, cd Dj, double psi, double psi0, double chi1,
                                            double chi0) {
     AbRev o;
     const cd zj = cmk(psi, chi1), zjm = cmk(psi0, chi0);
     const cd u = cadd(cmul(Dj, im), cmk(jx, 0.)), v = cadd(cmul(m, Dj), cmk(jx, 0.));
     o.ra = crecip_nr(csub(cmul(u, zj), zjm));
     o.rb = crecip_nr(csub(cmul(v, zj), zjm));
     o.a = cmul(csub(cscale(u, psi), cmk(psi0, 0.)), o.ra);
     o.b = cmul(csub(cscale(v, psi), cmk(psi0, 0.)), o.rb);
     return o;
}

// Per chunk, with the carry entering it as c, every carry and D cotangent
// inside is affine in c: carry out = P c + C0, z cotangent = Q c + Z0.
// The order j of the loop is the same in every lane (the chunk is the
// workgroup's), so the rows read are uniform: each window load takes a row
// clamped to the array's extent (in bounds for every lane), unconditionally,
// so no wait follows it before the value's use an order later.  Rows of psi,
// chi and U past a lane's n1 are read but never used (every use is under
// j <= n1); D past n2 - 1 is replaced by 0 (D_{n2} = 0 starts the
// recurrence).  UP: the angular cotangents come from U (mixed path), else
// from the FP64 cotangent planes.
template <bool UP>
__device__ __forceinline__ void rev_orders_body(RevArgs p) {
     const int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
     if (i >= p.Np) return;
     const size_t Np = p.Np, plane = (size_t) p.Kp * Np, ld = (size_t) p.n1max + 2;
     const unsigned o4 = (unsigned) i * 4u, o8 = (unsigned) i * 8u, o16 = (unsigned) i * 16u;
     cd P = cmk(1., 0.), C0 = cmk(0., 0.), Q = cmk(0., 0.), Z0 = cmk(0., 0.), mb = cmk(0., 0.);
     double fq = 0., xq = 0.;
     const int n1 = i < p.N ? p.n1[i] : 0, n2 = i < p.N ? p.n2[i] : 0;
     const int lo = 1 + k * p.rch, hi = min(n2, lo + p.rch);
     if (lo < hi) {
          const double x = p.x[i], f = p.f[i];
          // m, 1/m, 1/m^2 from the arguments: scalar operands, no registers per lane
          const cd m = cmk(p.mr, -p.mi), im1 = cmk(p.im1r, p.im1i), im2 = cmk(p.im2r, p.im2i);
          const cd iz = cscale(im1, 1. / x);   // 1/z, z = m x
          const double2 *Dv = (const double2 *) p.D;
          const double *U = p.PC, *Chi = p.PC + (size_t) (p.n1max + 1) * Np;
          const double sc = p.PS[i];
          const int pmax = p.n1max, dmax = p.n2rows - 1;
          // a_n, b_n recomputed from the kept recurrences, one order ahead for
          // the asymmetry series.  The recurrences are read through a window
          // (psi, chi at j-1, j, j+1; D at j, j+1; the U row of j) whose next
          // entries are loaded one order ahead of their use.
          auto rpc = [&](int n) {   // (psi_n, chi_n)
               const int r = min(n, pmax);
               return double2{sc * ld_row(U, r, Np, o8), ld_row(Chi, r, Np, o8)};
          };
          auto rD = [&](int n) {
               const double2 v = ld_row(Dv, min(n, dmax), Np, o16);
               return n < n2 ? cmk(v.x, v.y) : cmk(0., 0.);
          };
          const size_t uq = (size_t) p.Kq * Np;
          auto rdu = [&](int q, int n) { return UP ? ld_row(p.Uf + q * uq, min(n, p.Kq) - 1, Np, o4) : 0.f; };
          const double2 pcm = rpc(lo - 1), pc0 = rpc(lo), pc1 = rpc(lo + 1);
          double psm = pcm.x, ps0 = pc0.x, ps1 = pc1.x;
          double chm = pcm.y, ch0 = pc0.y, ch1 = pc1.y;
          cd D0 = rD(lo), D1 = rD(lo + 1);
          float u0 = rdu(0, lo), u1 = rdu(1, lo), u2 = rdu(2, lo), u3 = rdu(3, lo);
          cd am = cmk(0., 0.), bm = cmk(0., 0.);
          AbRev cur, nxt;
          cur.a = cur.b = cur.ra = cur.rb = cmk(0., 0.);
          nxt = cur;
          if (lo <= n1) {
               if (lo > 1) {
                    const double2 pc2 = rpc(lo - 2);
                    const AbRev pr = mie_ab_rev((lo - 1) / x, m, im1, rD(lo - 1), psm, pc2.x, chm, pc2.y);
                    am = pr.a;
                    bm = pr.b;
               }
               cur = mie_ab_rev(lo / x, m, im1, D0, ps0, psm, ch0, chm);
          }
          const cd cbv = cmk(p.CB[i], p.CB[Np + i]);
          // U path: every cotangent below is linear in f (U = Sbar / f and the
          // series parts carry f), so the sweep runs with f = 1 and the chunk's
          // f-linear results are scaled once at the end
          const double fw = UP ? 1. : f;
          const double sb0 = p.sb0 * fw, sb1 = p.sb1 * fw, sb2 = p.sb2 * fw, sb3 = p.sb3 * fw;
          double sgn = (lo & 1) ? -1. : 1.;
          const double ix = 1. / x;
          for (int j = lo; j < hi; ++j) {
               // the window's next entries
               const double2 pc2 = rpc(j + 2);
               const double ps2 = pc2.x, ch2 = pc2.y;
               const cd D2 = rD(j + 2);
               const float v0 = rdu(0, j + 1), v1 = rdu(1, j + 1), v2 = rdu(2, j + 1), v3 = rdu(3, j + 1);
               cd lc = cmk(0., 0.);
               if (j <= n1) {
                    if (j < n1) nxt = mie_ab_rev((j + 1) * ix, m, im1, D1, ps1, ps0, ch1, ch0);
                    const cd a = cur.a, b = cur.b, an = nxt.a, bn = nxt.b;
                    const double psi = ps0;
                    const cd zj = cmk(ps0, ch0);
                    const cd Dj = D0;
                    const double fv1 = 2. * j + 1., fv4 = p.ft[FT_FV4 * ld + j];
                    cd Sb, Tb;
                    if constexpr (UP) {
                         const cd us = cmk(u0, u1), ut = cmk(u2, u3);
                         // 1/2 Re(conj S U_S + conj T U_T), S = fv4 (a + b), T = fv4 (a - b)
                         fq += .5 * fv4 * ((a.r + b.r) * us.r + (a.i + b.i) * us.i + (a.r - b.r) * ut.r + (a.i - b.i) * ut.i);
                         Sb = us;
                         Tb = ut;
                    } else {
                         Sb = cmk(ld_row(p.bar, j - 1, Np, o8), ld_row(p.bar + plane, j - 1, Np, o8));
                         Tb = cmk(ld_row(p.bar + 2 * plane, j - 1, Np, o8), ld_row(p.bar + 3 * plane, j - 1, Np, o8));
                    }
                    // angular part
                    cd ab = cscale(cadd(Sb, Tb), fv4), bb = cscale(csub(Sb, Tb), fv4);
                    // series parts: ext, sca, bak, asym
                    ab.r += sb0 * fv1;
                    bb.r += sb0 * fv1;
                    ab = cadd(ab, cscale(a, 2. * sb1 * fv1));
                    bb = cadd(bb, cscale(b, 2. * sb1 * fv1));
                    ab = cadd(ab, cscale(cbv, 2. * sb2 * fv1 * sgn));
                    bb = csub(bb, cscale(cbv, 2. * sb2 * fv1 * sgn));
                    if (j < n1) {
                         const double fv3 = p.ft[FT_FV3 * ld + j];
                         ab = cadd(ab, cadd(cscale(an, sb3 * fv3), cscale(b, sb3 * fv4)));
                         bb = cadd(bb, cadd(cscale(bn, sb3 * fv3), cscale(a, sb3 * fv4)));
                    }
                    if (j > 1) {
                         const double fv3m = p.ft[FT_FV3M * ld + j];
                         ab = cadd(ab, cscale(am, sb3 * fv3m));
                         bb = cadd(bb, cscale(bm, sb3 * fv3m));
                    }
                    // a = (u psi - psi0) / (u zeta - zeta0), da/du = (psi - a zeta) / den
                    const cd dua = cmul(csub(cmk(psi, 0.), cmul(a, zj)), cur.ra);
                    const cd dvb = cmul(csub(cmk(psi, 0.), cmul(b, zj)), cur.rb);
                    const cd ub = cmul(cconj(dua), ab), vb = cmul(cconj(dvb), bb);
                    if (p.xbar) {
                         // d a / d x at fixed D_j (psi_j, psi_{j-1}, chi_j, chi_{j-1}
                         // and j / x move): with P = psi_j - a zeta_j the definition
                         // of a gives psi_{j-1} - a zeta_{j-1} = u P, and with
                         // psi_j' = psi_{j-1} - j psi_j / x, psi_{j-1}' = j psi_{j-1} / x - psi_j
                         // (the same for chi) it reduces to
                         // (d a / d u) (1 + (D / m)^2 - j (j + 1) / x^2); b likewise
                         // with m D.  The D_j part goes through the z cotangent.
                         const double c0 = 1. - j * (j + 1.) * (ix * ix);
                         const cd dm = cmul(Dj, im1), md = cmul(m, Dj);
                         const cd wu = cmul(dm, dm), wv = cmul(md, md);
                         xq += (c0 + wu.r) * ub.r + wu.i * ub.i + (c0 + wv.r) * vb.r + wv.i * vb.i;
                    }
                    // u = D/m + j/x, v = m D + j/x
                    lc = cadd(cmul(cconj(im1), ub), cmul(cconj(m), vb));
                    mb = cadd(mb, cadd(cmul(cconj(cscale(cmul(Dj, im2), -1.)), ub), cmul(cconj(Dj), vb)));
                    sgn = -sgn;
                    am = a;
                    bm = b;
                    cur = nxt;
               }
               // D_j = c1 - 1/c2, c2 = D_{j+1} + c1, c1 = (j+1)/z, D_{n2} = 0; 1/c2
               // by the forward's own operations (the same bits).  D cotangent
               // = P c + (C0 + lc); carry = g D cotangent
               const cd c1 = cscale(iz, j + 1.);
               const cd rc = crecip_nr(cadd(D1, c1));
               const cd ic22 = cmul(rc, rc);
               const cd g = cconj(ic22);
               const cd h = cconj(cmul(cadd(cmk(1., 0.), ic22), cscale(cmul(c1, iz), -1.)));
               const cd t = cadd(C0, lc);
               Q = cadd(Q, cmul(h, P));
               Z0 = cadd(Z0, cmul(h, t));
               P = cmul(g, P);
               C0 = cmul(g, t);
               psm = ps0; ps0 = ps1; ps1 = ps2;
               chm = ch0; ch0 = ch1; ch1 = ch2;
               D0 = D1; D1 = D2;
               u0 = v0; u1 = v1; u2 = v2; u3 = v3;
          }
     }
     // rev_carry reads the chunks below (n2 - 1 + rch - 1) / rch only
     if (lo >= n2) return;
     if constexpr (UP) {
          const double f = p.f[i];
          C0 = cscale(C0, f);
          Z0 = cscale(Z0, f);
          mb = cscale(mb, f);
          xq *= f;
     }
     double *o = p.scan + (size_t) k * REV_ROWS * Np + i;
     o[0] = P.r; o[Np] = P.i; o[2 * Np] = C0.r; o[3 * Np] = C0.i;
     o[4 * Np] = Q.r; o[5 * Np] = Q.i; o[6 * Np] = Z0.r; o[7 * Np] = Z0.i;
     o[8 * Np] = mb.r; o[9 * Np] = mb.i; o[10 * Np] = fq; o[11 * Np] = xq;
}
template <bool UP>
__global__ __launch_bounds__(64) void rev_orders(RevArgs p) { rev_orders_body<UP>(p); }
struct rev_orders_B {
     RevArgs p;
     unsigned gx, gy;
};
__global__ __launch_bounds__(64) void rev_orders_b(const rev_orders_B *cases) {
     const rev_orders_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     rev_orders_body<true>(a.p);
}


__device__ __forceinline__ void rev_carry_body(RevArgs p) {
     const int i = blockIdx.x * blockDim.x + threadIdx.x;
     if (i >= p.Np) return;
     const size_t Np = p.Np;
     const bool live = i < p.N;
     const double x = p.x[i];
     const int nk = live ? (p.n2[i] - 1 + p.rch - 1) / p.rch : 0;
     // chain the chunks upward from j = 1 with carry 0
     cd carry = cmk(0., 0.), zb = cmk(0., 0.), mb = cmk(0., 0.);
     double fq = 0., xq = 0.;
     for (int k = 0; k < nk; ++k) {
          const double *q = p.scan + (size_t) k * REV_ROWS * Np + i;
          const cd P = cmk(q[0], q[Np]), C0 = cmk(q[2 * Np], q[3 * Np]);
          const cd Q = cmk(q[4 * Np], q[5 * Np]), Z0 = cmk(q[6 * Np], q[7 * Np]);
          zb = cadd(zb, cadd(cmul(Q, carry), Z0));
          carry = cadd(cmul(P, carry), C0);
          mb = cadd(mb, cmk(q[8 * Np], q[9 * Np]));
          fq += q[10 * Np];
          xq += q[11 * Np];
     }
     mb = cadd(mb, cscale(zb, x));
     // z = m x with m = mr - i mi: the x cotangent of z is Re(conj(m) zbar)
     if (live && p.xbar) p.xbar[i] = xq + p.mr * zb.r - p.mi * zb.i;
     // the wave's 64 sizes added in a fixed order; the host adds the waves
#pragma unroll
     for (int o = 32; o > 0; o >>= 1) {
          mb.r += __shfl_xor(mb.r, o);
          mb.i += __shfl_xor(mb.i, o);
     }
     if (threadIdx.x == 0) {
          p.mbar[2 * blockIdx.x] = mb.r;
          p.mbar[2 * blockIdx.x + 1] = mb.i;
     }
     if (!live) return;
     // size-weight cotangent: angular part plus the series part
     const double fser = p.sb0 * p.S[i] + p.sb1 * p.S[Np + i] + p.sb2 * p.S[2 * Np + i] + p.sb3 * p.S[3 * Np + i];
     p.fbar[i] = (p.Uf ? fq : p.fang ? p.fang[i] : 0.) + fser;
}
__global__ __launch_bounds__(64) void rev_carry(RevArgs p) { rev_carry_body(p); }
struct rev_carry_B {
     RevArgs p;
     unsigned gx, gy;
};
__global__ __launch_bounds__(64) void rev_carry_b(const rev_carry_B *cases) {
     const rev_carry_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     rev_carry_body(a.p);
}


// Directions from the raw channels of the sums over sizes: direction o is
// sum_t c_t raw[r_t] (r_t < 0: none).
struct ChComb {
     int r[4];
     double c[4];
};

// Sum of the per-tile partials per (raw channel, element, angle) and the
// directions formed from them; the last ndot blocks are the series sums of the
// raw channels (weighted_dots), which wait for nothing here.  Eight lanes per
// output element, each summing every eighth tile, then the eight partials in a
// fixed order: deterministic, and eight times the threads of a plain
// per-element loop.
struct ReduceArgs {
     const double *part;        // [nblk][nraw][4 Q]
     int nblk, nraw, Q, nch;
     const ChComb *comb;        // [nch], or NULL: channels as they are
     double *out;               // [nch][4 Q]
     const DotJob *jobs;
     int n, ndot;
     double *dots;
     unsigned gx;
};
__device__ __forceinline__ void reduce_channels_body(const ReduceArgs &p, unsigned block) {
     const int per = 4 * p.Q, all = p.nraw * per;
     const unsigned nred = (unsigned) ((p.nch * per + 31) / 32);
     if (block >= nred) {
          if (block < p.gx) weighted_dots_body(p.jobs, p.n, p.dots, (int) (block - nred));
          return;
     }
     const int e = block * 32 + (threadIdx.x >> 3), l = threadIdx.x & 7;
     const bool live = e < p.nch * per;
     const int o = live ? e / per : 0, rem = e - o * per;
     double out = 0.;
     const int nt = p.comb ? 4 : 1;
     for (int t = 0; t < nt; ++t) {
          const int r = !live ? -1 : p.comb ? p.comb[o].r[t] : o;
          double s = 0.;
          if (r >= 0) {
               const double *q = p.part + (size_t) r * per + rem;
               int b = l;
               for (; b + 56 < p.nblk; b += 64) {   // eight partials in flight, added in order
                    double v[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = q[(size_t) (b + 8 * k) * all];
#pragma unroll
                    for (int k = 0; k < 8; ++k) s += v[k];
               }
               for (; b < p.nblk; b += 8) s += q[(size_t) b * all];
          }
          s += __shfl_xor(s, 1);
          s += __shfl_xor(s, 2);
          s += __shfl_xor(s, 4);
          if (r >= 0) out += p.comb ? p.comb[o].c[t] * s : s;
     }
     if (live && l == 0) p.out[e] = out;
}
__global__ __launch_bounds__(256) void reduce_channels(ReduceArgs p) { reduce_channels_body(p, blockIdx.x); }
__global__ __launch_bounds__(256) void reduce_channels_b(const ReduceArgs *cases) { reduce_channels_body(cases[blockIdx.z], blockIdx.x); }


// ---------------------------------------------------------------------------
// Expansion.  For channel c the quadrature-weighted element rows at the
// mirrored (-) and direct (+) angles of every positive node j:
//   GSF      F11, F11+F33, F11-F33, F33, F12, F34   (misc/rtutil_scat_int.c:173-183)
//   Legendre F11, F11, F33, F33, F12, F34.
// One wave per (two l, channel): twelve dot products per l over the positive
// nodes, folded with (-1)^l for the mirrored half, then the alpha/zeta
// recombination and the (2l+1)/2 factor (misc/rtutil_scat_int.c:185-213,
// :436-469).  The rows are formed from the elements as they are read (a launch of
// their own otherwise), once for both l.
__device__ __forceinline__ void expand_coefs_body(const double *T, const double *pf, const double *w, int Q, int Hp, int C, int gsf,
                                                  double *coefs) {
     const int lane = threadIdx.x & 63, H = Q / 2;
     const int l0 = 2 * (blockIdx.x * 4 + (threadIdx.x >> 6));
     const int c = blockIdx.y;
     if (l0 >= C) return;
     typedef double d2 __attribute__((ext_vector_type(2)));
     const size_t plane = gsf_plane(C, Hp), row = (size_t) l0 * Hp;
     const d2 *P00 = (const d2 *) (T + (gsf ? 0 : 4 * plane) + row), *P02 = (const d2 *) (T + plane + row);
     const d2 *P22 = (const d2 *) (T + 2 * plane + row), *P2m = (const d2 *) (T + 3 * plane + row);
     const double *P = pf + (size_t) c * 4 * Q;
     double d[2][12];
#pragma unroll
     for (int r = 0; r < 12; ++r) d[0][r] = d[1][r] = 0.;
     for (int j = lane; j < H; j += 64) {
          const d2 q00 = P00[j];
          const double wq = w[H + j];
          double e[2][4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
               e[0][k] = P[(size_t) k * Q + H - 1 - j] * wq;
               e[1][k] = P[(size_t) k * Q + H + j] * wq;
          }
          d2 q02 = {0., 0.}, q22 = q02, q2m = q02;
          if (gsf) { q02 = P02[j]; q22 = P22[j]; q2m = P2m[j]; }
#pragma unroll
          for (int u = 0; u < 2; ++u) {
               const double p00 = q00[u];
               if (gsf) {
                    const double p02 = q02[u], p22 = q22[u], p2m = q2m[u];
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                         const double f11 = e[s][0], f33 = e[s][1], sum = f11 + f33, dif = f11 - f33;
                         d[u][6 * s + 0] += p00 * f11;
                         d[u][6 * s + 1] += (s ? p22 : p2m) * sum;
                         d[u][6 * s + 2] += (s ? p2m : p22) * dif;
                         d[u][6 * s + 3] += p00 * f33;
                         d[u][6 * s + 4] += p02 * e[s][2];
                         d[u][6 * s + 5] += p02 * e[s][3];
                    }
               } else {
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                         d[u][6 * s + 0] += p00 * e[s][0];
                         d[u][6 * s + 1] += p00 * e[s][0];
                         d[u][6 * s + 2] += p00 * e[s][1];
                         d[u][6 * s + 3] += p00 * e[s][1];
                         d[u][6 * s + 4] += p00 * e[s][2];
                         d[u][6 * s + 5] += p00 * e[s][3];
                    }
               }
          }
     }
#pragma unroll
     for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < 12; ++r) {
               double s = d[u][r];
#pragma unroll
               for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
               d[u][r] = s;
          }
     if (lane == 0) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
               const int l = l0 + u;
               if (l >= C) break;
               const double sl = (l & 1) ? -1. : 1., fl = (2 * l + 1) / 2.;
               double e[6];
#pragma unroll
               for (int k = 0; k < 6; ++k) e[k] = d[u][k] * sl + d[u][6 + k];
               double *out = coefs + (size_t) c * 6 * C;
               if (gsf) {
                    const double t = e[1];
                    e[1] = (t + e[2]) / 2.;
                    e[2] = (t - e[2]) / 2.;
               } else {
                    e[5] = -e[5];
               }
#pragma unroll
               for (int k = 0; k < 6; ++k) out[(size_t) k * C + l] = e[k] * fl;
          }
     }
}
__global__ __launch_bounds__(256) void expand_coefs(const double *T, const double *pf, const double *w, int Q, int Hp, int C, int gsf, double *coefs) { expand_coefs_body(T, pf, w, Q, Hp, C, gsf, coefs); }
struct expand_coefs_B {
     const double *T, *pf, *w;
     int Q, Hp, C, gsf;
     double *coefs;
     unsigned gx, gy;
};
__global__ __launch_bounds__(256) void expand_coefs_b(const expand_coefs_B *cases) {
     const expand_coefs_B a = cases[blockIdx.z];
     if (blockIdx.x >= a.gx || blockIdx.y >= a.gy) return;
     expand_coefs_body(a.T, a.pf, a.w, a.Q, a.Hp, a.C, a.gsf, a.coefs);
}


// Scattering matrix at user angles from coefficients (misc/rtutil_scat_int.c:510-797).
// Generalized spherical functions: a block takes 64 angles and PH_SETS coefficient
// sets, a wave per function (P00, P02, P22, P2-2) with its sums in registers;
// Legendre: a wave per set.  The coefficients of 64 l at a time are staged in the
// wave's LDS and read as broadcasts beside the recurrence's factors (gsf_steps).
// Bound: the recurrence's chain of five operations per l.  A call with 181 angles,
// 4 tangents and truncated at 1e-7 (the example program's) takes 0.64 ms against
// 0.93 with one thread per (set, angle) running all four functions with IEEE
// divisions, two launches and device allocations per call.
constexpr int PH_SETS = 4;
constexpr int PH_LDS = 68 * GSF_CST + 64 * 2 * PH_SETS;   // doubles per wave

// acc[k] += x_k[l] v for the rows of one wave: GSF FN 0 sums rows 0 and 3 of
// each set, 1 rows 4 and 5, 2 and 3 the sum and difference of rows 1 and 2;
// FN 4 (Legendre) all six rows of one set.
template <int FN>
__device__ __forceinline__ void phase_sums(int ncoef, int ld, const double *X, int s0, int ns, double m, bool live,
                                           double *lds, double *acc) {
#pragma clang fp contract(off)
     constexpr int NR = FN == 4 ? 6 : FN < 2 ? 2 * PH_SETS : PH_SETS;
     const int lane = threadIdx.x & 63;
     double *cst = lds, *xs = lds + 68 * GSF_CST;
     int base = 0;
     gsf_steps<FN>(ncoef, m, live, cst,
          [&](int l0) {
               base = l0;
               const int l = min(l0 + lane, ncoef - 1);
               wave_lds_fence();
#pragma unroll
               for (int r = 0; r < NR; ++r) {
                    const int set = FN == 4 ? s0 : s0 + min(FN < 2 ? r / 2 : r, ns - 1);
                    const double *x = X + (size_t) set * 6 * ld + l;
                    double v;
                    if constexpr (FN == 4) v = x[(size_t) r * ld];
                    else if constexpr (FN == 0) v = x[(size_t) (r & 1 ? 3 : 0) * ld];
                    else if constexpr (FN == 1) v = x[(size_t) (4 + (r & 1)) * ld];
                    else v = FN == 2 ? x[ld] + x[2 * (size_t) ld] : x[ld] - x[2 * (size_t) ld];
                    xs[lane * NR + r] = v;
               }
               wave_lds_fence();
          },
          [&](int l, bool, double v) {
               if (FN > 0 && FN < 4 && l < 2) return;     // the functions start at l = 2
               const double *x = xs + (l - base) * NR;
#pragma unroll
               for (int r = 0; r < NR; ++r) acc[r] += x[r] * v;
          });
}

template <bool GSF>
__global__ __launch_bounds__(256) void phase_at_angles(int nset, int ncoef, int ld, const double *X, int nth, const double *theta,
                                                       double *pf) {
#pragma clang fp contract(off)
     __shared__ __align__(16) double lds[4 * PH_LDS];
     const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
     const int i = blockIdx.x * 64 + lane;
     const bool live = i < nth;
     const double m = cos(theta[live ? i : 0] * (kPi / 180.));
     double *my = lds + wave * PH_LDS;
     if constexpr (!GSF) {
          const int set = blockIdx.y * 4 + wave;
          if (set >= nset) return;
          double acc[6] = {0., 0., 0., 0., 0., 0.};
          phase_sums<4>(ncoef, ld, X, set, 1, m, live, my, acc);
          if (!live) return;
          double *o = pf + (size_t) set * 6 * nth + i;
#pragma unroll
          for (int k = 0; k < 6; ++k) o[(size_t) k * nth] = k == 5 ? -acc[k] : acc[k];
     } else {
          const int s0 = blockIdx.y * PH_SETS, ns = min(PH_SETS, nset - s0);
          double acc[2 * PH_SETS];
#pragma unroll
          for (int k = 0; k < 2 * PH_SETS; ++k) acc[k] = 0.;
          if (wave == 0) phase_sums<0>(ncoef, ld, X, s0, ns, m, live, my, acc);
          else if (wave == 1) phase_sums<1>(ncoef, ld, X, s0, ns, m, live, my, acc);
          else if (wave == 2) phase_sums<2>(ncoef, ld, X, s0, ns, m, live, my, acc);
          else phase_sums<3>(ncoef, ld, X, s0, ns, m, live, my, acc);
          // F22 and F33 from the sums over P22 (wave 2) and P2-2 (wave 3)
          __syncthreads();
          if (wave == 3)
#pragma unroll
               for (int k = 0; k < PH_SETS; ++k) lds[k * 64 + lane] = acc[k];
          __syncthreads();
          if (!live || wave == 3) return;
#pragma unroll
          for (int k = 0; k < PH_SETS; ++k) {
               if (k >= ns) break;
               double *o = pf + (size_t) (s0 + k) * 6 * nth + i;
               if (wave == 0) { o[0] = acc[2 * k]; o[(size_t) 3 * nth] = acc[2 * k + 1]; }
               else if (wave == 1) { o[(size_t) 4 * nth] = acc[2 * k]; o[(size_t) 5 * nth] = acc[2 * k + 1]; }
               else {
                    const double b = lds[k * 64 + lane];
                    o[nth] = (acc[k] + b) / 2.;
                    o[(size_t) 2 * nth] = (acc[k] - b) / 2.;
               }
          }
     }
}

int launch_phase(int n_set, int n_coef, int ld, const double *X, int n_theta, const double *theta, double *pf, int gsf, hipStream_t s) {
     const unsigned gx = (unsigned) ((n_theta + 63) / 64);
     // the grid's y extent is bounded: the sets go in launches of at most 65535 rows
     const int per = 65535 * 4;
     for (int s0 = 0; s0 < n_set; s0 += per) {
          const int n = std::min(per, n_set - s0);
          const dim3 g(gx, (unsigned) ((n + 3) / 4));
          const double *x = X + (size_t) s0 * 6 * ld;
          double *o = pf + (size_t) s0 * 6 * n_theta;
          if (gsf) hipLaunchKernelGGL(phase_at_angles<true>, g, dim3(256), 0, s, n, n_coef, ld, x, n_theta, theta, o);
          else hipLaunchKernelGGL(phase_at_angles<false>, g, dim3(256), 0, s, n, n_coef, ld, x, n_theta, theta, o);
     }
     HIPCHECK(hipGetLastError());
     return 0;
}
static_assert(PH_SETS == 4, "launch_phase");

// ---------------------------------------------------------------------------
// Workspace: device buffers and a stream, reused across calls, one per
// concurrent caller (a mutex-guarded pool), so the API stays reentrant.
struct Buf {
     void *p = nullptr;
     size_t n = 0;
     int get(size_t bytes) {
          if (bytes <= n) return 0;
          if (p) (void) hipFree(p);
          p = nullptr;
          n = 0;
          bytes = bytes < 256 ? 256 : bytes;
          if (hipMalloc(&p, bytes) != hipSuccess) return set_err("hipMalloc(%zu bytes) failed", bytes);
          n = bytes;
          return 0;
     }
     template <class T> T *as() const { return (T *) p; }
};

struct PinBuf {      // pinned host memory, grown on demand
     void *p = nullptr;
     size_t n = 0;
     int get(size_t bytes) {
          if (bytes <= n) return 0;
          if (p) (void) hipHostFree(p);
          p = nullptr;
          n = 0;
          if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) return set_err("hipHostMalloc(%zu bytes) failed", bytes);
          n = bytes;
          return 0;
     }
};

// Many small copies as one: each job moves n doubles.  A fused batch sends its
// results with it from the device straight into each case's pinned landing area.
struct CopyJob {
     const double *src;
     double *dst;
     size_t n;
};
__global__ __launch_bounds__(256) void copy_jobs(const CopyJob *jobs) {
     const CopyJob j = jobs[blockIdx.y];
     for (size_t e = (size_t) blockIdx.x * 256 + threadIdx.x; e < j.n; e += (size_t) gridDim.x * 256)
          j.dst[e] = j.src[e];
}

// Place of an input inside a call's uploaded block (Stage).
struct Ref {
     void *p = nullptr;
     template <class T> T *as() const { return (T *) p; }
};

struct Workspace {
     int device = -1;
     hipStream_t stream = nullptr;
     hipEvent_t uploaded = nullptr;  // a batch case's inputs are on the device (its own stream)
     hipEvent_t ev[2 * LMIE_N_TIMERS + 2];
     // inputs of the last forward call, in finDev (f: the weight rows, row 0 the density)
     Ref x, sx, cx, f, n1, n2, kfill, ktile32, ktile64, ktile128, comb, guess, dotjobs, order, tasks;
     std::vector<int2> rtask;       // host copy of tasks: (size tile, order tile) of the reverse contraction
     Buf mu, w, Bp, Bm, B16, A16, T, A, S, part, pf, res, save2;
     // reverse-pass checkpoint and buffers
     Buf CB, sst, pfbar, bar, fang, gbar, expart;
     Buf rres;                      // results: f cotangents [N], x cotangents [N], m cotangents per 64 sizes [Np / 64][2]
     Buf wts, scal, L16, R16, Gf, G16, Uf;   // mixed reverse pass
     Buf chD, chPC, chPS, chPart, revScan;   // per-size recurrences
     Buf chDz, chPQ;                // and what their tangents need
     Buf ftab;                      // order_factors of the value channel
     Buf sw, s1, s2, sguess, dots;  // save_control 2: channel weights, saved per-size arrays, guesses, sums
     Buf bargs;                     // per-case arguments of a batch launched from here
     PinBuf pargs;
     PinBuf pres;                   // pinned landing area of a call's results
     PinBuf pin;                    // pinned staging of the cotangents
     Buf finDev;                    // a call's inputs, one copy
     Buf phIn, phOut;               // phase function: coefficients and angles, elements
     PinBuf finPin;
     int home = -1, busy = 0;       // batch slot of this workspace (-1: general pool)
     int n2rows = 0;
     int rch = 64;                  // reverse pass: orders per chunk (rev_chunk)
     int ushape = 8;                // reverse contraction: shape (FP64: orders per task)
     int valid = 0;
     int N = 0, Np = 0, Kp = 0, Hp = 0, H = 0, Q = 0, C = 0, n1max = 0, n2max = 0, calc_gc = 0, calc_lc = 0;
     int mixed = 0, bf16 = 0, Kb = 0, Hb = 0;
     double mr = 0., mi = 0.;
};

pthread_mutex_t g_pool_mu = PTHREAD_MUTEX_INITIALIZER;
std::vector<Workspace *> g_pool;
std::vector<Workspace *> g_home;     // workspaces of batch slots (Workspace::home)

// Makes device d current on this thread (hipSetDevice only when it is not).
int use_device(int d) {
     int cur = -1;
     if (hipGetDevice(&cur) != hipSuccess || cur != d) HIPCHECK(hipSetDevice(d));
     return 0;
}

int ws_create(int device, Workspace **out) {
     Workspace *w = new Workspace();
     w->device = device;
     HIPCHECK(hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking));
     HIPCHECK(hipEventCreateWithFlags(&w->uploaded, hipEventDisableTiming));
     for (auto &e : w->ev) HIPCHECK(hipEventCreate(&e));
     *out = w;
     return 0;
}


int ws_acquire(int device, Workspace **out) {
     pthread_mutex_lock(&g_pool_mu);
     Workspace *w = nullptr;
     for (size_t k = 0; k < g_pool.size(); ++k)
          if (g_pool[k]->device == device) {
               w = g_pool[k];
               g_pool.erase(g_pool.begin() + k);
               break;
          }
     pthread_mutex_unlock(&g_pool_mu);
     if (use_device(device)) return -1;
     if (!w && ws_create(device, &w)) return -1;
     *out = w;
     return 0;
}

// The workspace of slot `slot` of a batch on `device` (the current device):
// the same one at every batch call while it is free, so a retrieval loop that
// passes its cases in the same order finds buffers of the right sizes.
int ws_acquire_home(int device, int slot, Workspace **out) {
     pthread_mutex_lock(&g_pool_mu);
     Workspace *w = nullptr;
     for (Workspace *h : g_home)
          if (h->device == device && h->home == slot && !h->busy) {
               w = h;
               break;
          }
     if (w) w->busy = 1;
     pthread_mutex_unlock(&g_pool_mu);
     if (!w) {
          if (ws_create(device, &w)) return -1;
          w->home = slot;
          w->busy = 1;
          pthread_mutex_lock(&g_pool_mu);
          g_home.push_back(w);
          pthread_mutex_unlock(&g_pool_mu);
     }
     *out = w;
     return 0;
}

void ws_release(Workspace *w) {
     pthread_mutex_lock(&g_pool_mu);
     if (w->home >= 0) w->busy = 0;
     else g_pool.push_back(w);
     pthread_mutex_unlock(&g_pool_mu);
}

struct Timer {
     Workspace *w;
     int on;
     void mark(int id, int end, hipStream_t st = nullptr) {
          if (on) (void) hipEventRecord(w->ev[2 * id + end], st ? st : w->stream);
     }
     void collect(const int *ids, int n) {
          for (int k = 0; k < LMIE_T_HOST_GRID; ++k) g_times[k] = 0.;
          if (!on) return;
          for (int k = 0; k < n; ++k) {
               float ms = 0.f;
               if (hipEventElapsedTime(&ms, w->ev[2 * ids[k]], w->ev[2 * ids[k] + 1]) == hipSuccess)
                    g_times[ids[k]] = ms;
          }
     }
};

// ---------------------------------------------------------------------------
// Angular contraction, FP64 matrix cores.
//
// For a tile of sizes i and positive angles j the four complex sums
//   sp+ = sum_n S_n (pi+tau)_n   sm+ = sum_n T_n (pi-tau)_n
//   sp- = sum_n s_n S_n (pi-tau)_n   sm- = sum_n s_n T_n (pi+tau)_n,
// S_n = fv4 (a+b), T_n = fv4 (a-b), s_n = (-1)^(n-1) (the -mu mirror,
// src/lmie_core.c:617-652,682-686), are 8 real GEMM accumulators of
// v_mfma_f64_16x16x4 (operand lane layout: A[i][k] in lane i + 16 k, B[k][j] in
// lane j + 16 k; result D[l/16 + 4 v][l % 16] in lane l, element v -- checked by
// lmie_gpu_selftest_mfma_f64).
//
// Forward tangents: every direction's derivative of the sums is
//   dS = dx_i S_x + dm S_m,
// with S_x the derivative along the size parameter and S_m the (complex,
// analytic) derivative along m, so two further operand sets (HX, HM) serve
// any number of directions.  The epilogue forms the elements P and their
// derivatives along x, Re m and Im m, and sums them over the sizes with one
// weight row per raw channel: rows 0 .. nP-1 of W weigh P (the density, its
// tangents), rows nP .. nP+nX-1 weigh dP/dx (f dx_i of each direction that
// moves x), and the two last channels are dP/dRe m and dP/dIm m with the
// weight of row 0.  reduce_channels forms the directions from the sums.
//
// What bounds it: the FP64 matrix cores (64 cycles per instruction and SIMD).
// A wave owns one 16 x 16 block with all its sums in registers (8
// accumulators per operand set); WM x WN waves share an LDS tile of 16 WM
// sizes x 16 WN angles, filled by direct loads (global_load_lds_dwordx4, 64
// lanes x 16 bytes straight into LDS) one stage of KS orders ahead, one
// barrier per stage; a wave waits only for its own loads of the stage.  The
// products' LDS reads are 16 consecutive doubles per lane group, so rows need
// no padding.  (size tile, angle tile) tasks come from a host-built list dealt
// over the XCDs.  Partials per size tile: part[tile][channel][4][Q].
struct F64Args {
     int Np, Kp, Hp, H, Q, N;
     const double *A[3];        // operand planes [4][Kp][Np] of the value, then of d/dx, d/dm as present
     const double *Bp, *Bm;     // [Kp][Hp]
     const int *ktile;          // rows to contract per size tile
     const int2 *task;          // (size tile, angle tile), (-1, -1) none
     const double *W;           // [nP + nX][Np] weight rows, row 0 the density
     int nP, nX;
     double *part;              // [size tiles][channels][4][Q]
     double *save2;             // [4][N][Q] per-size matrix (save_control 1) or NULL
     double *sst;               // reverse-pass checkpoint [8][Np][Hp]: sp+, sm+, sp-, sm- (re, im) or NULL
};

template <int WM, int WN, bool HX, bool HM, int KS, int OCC>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(OCC))) void angular_f64(F64Args p) {
     constexpr int NB = 1 + HX + HM, NW = WM * WN, TM = 16 * WM, TN = 16 * WN;
     constexpr int ASTG = NB * 4 * KS * TM, STG = ASTG + 2 * KS * TN;
     constexpr int NL = STG / (128 * NW);             // direct loads per wave and stage
     static_assert(STG % (128 * NW) == 0 && ASTG % 128 == 0 && KS % 4 == 0, "whole 1 KiB loads");
     constexpr int CHB = 8 * WM * TN;                 // epilogue buffer per channel
     constexpr int CAP = 2 * STG / CHB;               // channels per flush
     __shared__ double sh[2 * STG];

     const int2 tk = p.task[blockIdx.x];
     if (tk.x < 0) return;
     const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
     const int wm = wave % WM, wn = wave / WM;
     const int l16 = lane & 15, lg = lane >> 4;
     const int tile = tk.x, it0 = tile * TM, jt0 = tk.y * TN;
     const size_t Np = p.Np, Hp = p.Hp, plane = (size_t) p.Kp * Np;
     const int nch = p.ktile[tile] / KS;

     // this lane's source of each of the wave's loads at stage 0, and the step
     // to the next stage
     const double *src[NL];
     size_t step[NL];
#pragma unroll
     for (int u = 0; u < NL; ++u) {
          const int c = wave + NW * u;
          if (c < ASTG / 128) {
               const int e = c * 128 + 2 * lane, row = e / TM, pl = row / KS;
               const double *base = p.A[0];
               if (NB > 1 && pl >= 4) base = p.A[1];
               if (NB > 2 && pl >= 8) base = p.A[2];
               src[u] = base + (size_t) (pl & 3) * plane + (size_t) (row % KS) * Np + it0 + e % TM;
               step[u] = (size_t) KS * Np;
          } else {
               const int e = c * 128 - ASTG + 2 * lane, row = e / TN;
               src[u] = (row / KS ? p.Bm : p.Bp) + (size_t) (row % KS) * Hp + jt0 + e % TN;
               step[u] = (size_t) KS * Hp;
          }
     }
     auto stage_load = [&](int buf) {
#pragma unroll
          for (int u = 0; u < NL; ++u) {
               __builtin_amdgcn_global_load_lds((const void *) src[u], (lds_ptr) (sh + buf * STG + (wave + NW * u) * 128), 16, 0, 0);
               src[u] += step[u];
          }
     };

     v4d acc[NB][8];
#pragma unroll
     for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int q = 0; q < 8; ++q) acc[b][q] = v4d{0., 0., 0., 0.};

     // s_n of this lane's orders (k0 + 4 ks + lg + 1: alternate lane groups)
     const unsigned long long sgn = (unsigned long long) (lg & 1) << 63;
     auto flip = [&](double v) { return __longlong_as_double((long long) ((unsigned long long) __double_as_longlong(v) ^ sgn)); };
     if (nch > 0) stage_load(0);
     int buf = 0;
     for (int kc = 0; kc < nch; ++kc) {
          // this wave's loads of the stage have landed, then everyone's; every
          // wave is also done with the buffer of stage kc - 1, which takes
          // stage kc + 1
          wait_vm<0>();
          __builtin_amdgcn_s_barrier();
          __asm__ volatile("" ::: "memory");
          if (kc + 1 < nch) stage_load(buf ^ 1);
          const double *a0 = sh + buf * STG + lg * TM + 16 * wm + l16;
          const double *b0 = sh + buf * STG + ASTG + lg * TN + 16 * wn + l16;
#pragma unroll
          for (int ks = 0; ks < KS / 4; ++ks) {
               // the -mu products take s_n on the angle operand
               const double bp = b0[4 * ks * TN], bm = b0[(KS + 4 * ks) * TN];
               const double sbp = flip(bp), sbm = flip(bm);
#pragma unroll
               for (int b = 0; b < NB; ++b) {
                    const double Sr = a0[((4 * b + 0) * KS + 4 * ks) * TM], Si = a0[((4 * b + 1) * KS + 4 * ks) * TM];
                    const double Tr = a0[((4 * b + 2) * KS + 4 * ks) * TM], Ti = a0[((4 * b + 3) * KS + 4 * ks) * TM];
                    v4d *q = acc[b];
                    q[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(Sr, bp, q[0], 0, 0, 0);
                    q[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(Si, bp, q[1], 0, 0, 0);
                    q[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(Tr, bm, q[2], 0, 0, 0);
                    q[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ti, bm, q[3], 0, 0, 0);
                    q[4] = __builtin_amdgcn_mfma_f64_16x16x4f64(Sr, sbm, q[4], 0, 0, 0);
                    q[5] = __builtin_amdgcn_mfma_f64_16x16x4f64(Si, sbm, q[5], 0, 0, 0);
                    q[6] = __builtin_amdgcn_mfma_f64_16x16x4f64(Tr, sbp, q[6], 0, 0, 0);
                    q[7] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ti, sbp, q[7], 0, 0, 0);
               }
          }
          buf ^= 1;
     }

     // epilogue: Stokes elements, weighted sums over this wave's 16 sizes (four
     // per lane, then the four lane groups), over the WM waves of a column in
     // a fixed order through LDS
     const int i0 = it0 + 16 * wm + lg, j = jt0 + 16 * wn + l16;
     if (p.sst || p.save2) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
               const int i = i0 + 4 * v;
               if (p.sst) {
                    double *o = p.sst + (size_t) i * Hp + j;
#pragma unroll
                    for (int c = 0; c < 8; ++c) o[c * Np * Hp] = acc[0][c][v];
               }
               if (p.save2 && i < p.N && j < p.H) {
                    double Pp[4], Pm[4];
                    stokes(acc[0][0][v], acc[0][1][v], acc[0][2][v], acc[0][3][v], Pp);
                    stokes(acc[0][4][v], acc[0][5][v], acc[0][6][v], acc[0][7][v], Pm);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                         p.save2[((size_t) k * p.N + i) * p.Q + p.H + j] = Pp[k];
                         p.save2[((size_t) k * p.N + i) * p.Q + p.H - 1 - j] = Pm[k];
                    }
               }
          }
     }
     const int nraw = p.nP + p.nX + (HM ? 2 : 0);
     double *out = p.part + (size_t) tile * nraw * 4 * p.Q;
     for (int c0 = 0; c0 < nraw; c0 += CAP) {
          const int c1 = c0 + CAP < nraw ? c0 + CAP : nraw;
          __syncthreads();               // every wave is done with the stages (or the last flush)
#pragma unroll
          for (int sg = 0; sg < 2; ++sg) {
               // elements of kind kd (0: P, 1: dP/dx, 2, 3: dP/dRe m, dP/dIm m)
               // under the weight rows of channels k0 .. k1 - 1
               auto kind = [&](auto kdc, int k0, int k1) {
                    constexpr int kd = decltype(kdc)::value;
                    k0 = k0 < c0 ? c0 : k0;
                    k1 = k1 > c1 ? c1 : k1;
                    if (k0 >= k1) return;
                    double e[4][4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                         const v4d *q = acc[0] + 4 * sg, *d = acc[kd == 0 ? 0 : kd == 1 ? 1 : NB - 1] + 4 * sg;
                         if constexpr (kd == 0) stokes(q[0][v], q[1][v], q[2][v], q[3][v], e[v]);
                         else if constexpr (kd < 3)
                              stokes_tan(q[0][v], q[1][v], q[2][v], q[3][v], d[0][v], d[1][v], d[2][v], d[3][v], e[v]);
                         else
                              stokes_tan(q[0][v], q[1][v], q[2][v], q[3][v], -d[1][v], d[0][v], -d[3][v], d[2][v], e[v]);
                    }
                    for (int c = k0; c < k1; ++c) {
                         const double *w = p.W + (kd < 2 ? (size_t) c * Np : 0) + i0;
                         double r[4] = {0., 0., 0., 0.};
#pragma unroll
                         for (int v = 0; v < 4; ++v) {
                              const double wv = w[4 * v];
#pragma unroll
                              for (int k = 0; k < 4; ++k) r[k] += wv * e[v][k];
                         }
#pragma unroll
                         for (int k = 0; k < 4; ++k) {
                              r[k] += __shfl_xor(r[k], 16);
                              r[k] += __shfl_xor(r[k], 32);
                         }
                         // lane group k stores element k
                         const double t = lg == 0 ? r[0] : lg == 1 ? r[1] : lg == 2 ? r[2] : r[3];
                         sh[(c - c0) * CHB + ((4 * sg + lg) * WM + wm) * TN + 16 * wn + l16] = t;
                    }
               };
               kind(std::integral_constant<int, 0>{}, 0, p.nP);
               if constexpr (HX) kind(std::integral_constant<int, 1>{}, p.nP, p.nP + p.nX);
               if constexpr (HM) {
                    kind(std::integral_constant<int, 2>{}, p.nP + p.nX, p.nP + p.nX + 1);
                    kind(std::integral_constant<int, 3>{}, p.nP + p.nX + 1, p.nP + p.nX + 2);
               }
          }
          __syncthreads();
          for (int e = threadIdx.x; e < (c1 - c0) * 8 * TN; e += 64 * NW) {
               const int jc = e % TN, ck = e / TN, k = ck & 7, c = ck >> 3;
               const double *t = sh + (size_t) c * CHB + k * WM * TN + jc;
               double s = t[0];
#pragma unroll
               for (int m = 1; m < WM; ++m) s += t[m * TN];
               if (jt0 + jc < p.H)
                    out[((size_t) (c0 + c) * 4 + (k & 3)) * p.Q + (k < 4 ? p.H + jt0 + jc : p.H - 1 - jt0 - jc)] = s;
          }
     }
}

// Tiles of the FP64 contraction and the size tiles per group of its task list.
// 32 x 32 tiles on four waves, two stages: three workgroups per CU with one
// operand set, two with more (the accumulators then take 128 or 192
// registers).  Measured on the two-mode workload (32768 sizes, 3810 angles, one
// set) and the gamma mode with tangents of m (16384 sizes, 1922 angles, two
// sets): 14.7 and 4.3 ms; the same tiles with three stages and two workgroups
// per CU 15.2 and 4.6; 32 x 64 on eight waves 15.7 and 4.6; 64 x 64 on
// sixteen waves 15.3.  The instance with both derivative sets (192 accumulator
// registers, the loads' 64-bit sources beside them) spills 112 registers, the
// other three none; one workgroup per CU without the spill took 0.171-0.175 ms
// where it takes 0.135 (2257 sizes, 512 angles).  Groups of 1 or 2 size tiles took 0.3-0.4 ms less than 4
// or 8, of 16 1 ms more.
constexpr int F64_TILE = 32, F64_GROUP = 2;

int launch_angular_f64(const F64Args &a, bool hx, bool hm, unsigned ntask, hipStream_t s) {
     if (!hx && !hm) hipLaunchKernelGGL((angular_f64<2, 2, false, false, 16, 3>), dim3(ntask), dim3(256), 0, s, a);
     else if (!hm) hipLaunchKernelGGL((angular_f64<2, 2, true, false, 8, 2>), dim3(ntask), dim3(256), 0, s, a);
     else if (!hx) hipLaunchKernelGGL((angular_f64<2, 2, false, true, 8, 2>), dim3(ntask), dim3(256), 0, s, a);
     else hipLaunchKernelGGL((angular_f64<2, 2, true, true, 8, 2>), dim3(ntask), dim3(256), 0, s, a);
     HIPCHECK(hipGetLastError());
     return 0;
}

// Task list of a tiled contraction over (size tile, column tile) pairs for
// the XCD layout of the chip: the hardware deals workgroup ids round robin
// over the 8 XCDs, so id 8k + x is the k-th workgroup of XCD x.  Size tiles go
// heaviest first (ktile descending) to the XCDs in turn; inside an XCD they
// are taken in groups of `group`, and a group runs column tile by column tile.
// The workgroups in flight on one XCD then share a column tile's operand
// (angle or order tables) across the group and a size tile's operand across
// the column tiles, both from that XCD's L2.  ncol(s) = column tiles of size
// tile s.  Padding entries are (-1, -1).
template <class F>
void xcd_tasks(const std::vector<int> &kt, F ncol, int group, std::vector<int2> &out) {
     const int nT = (int) kt.size();
     std::vector<int> ord(nT);
     for (int t = 0; t < nT; ++t) ord[t] = t;
     std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return kt[a] > kt[b]; });
     std::vector<std::vector<int2>> per(8);
     for (int x = 0; x < 8; ++x) {
          std::vector<int> mine;
          for (int k = x; k < nT; k += 8) mine.push_back(ord[k]);
          for (size_t g0 = 0; g0 < mine.size(); g0 += group) {
               const size_t g1 = std::min(mine.size(), g0 + group);
               int cmax = 0;
               for (size_t k = g0; k < g1; ++k) cmax = std::max(cmax, ncol(mine[k]));
               for (int c = 0; c < cmax; ++c)
                    for (size_t k = g0; k < g1; ++k)
                         if (c < ncol(mine[k])) per[x].push_back(make_int2(mine[k], c));
          }
     }
     size_t len = 0;
     for (auto &v : per) len = std::max(len, v.size());
     out.assign(8 * len, make_int2(-1, -1));
     for (int x = 0; x < 8; ++x)
          for (size_t k = 0; k < per[x].size(); ++k) out[8 * k + x] = per[x][k];
}

// Split products of the forward mixed contraction (environment
// LMIE_MIX_PRODUCTS, read at every call): 5 (default), 4 (without A_lo B_mid;
// shape 3 only, else 5) or 3.
int mix_products() {
     const char *e = getenv("LMIE_MIX_PRODUCTS");
     const int r = e ? atoi(e) : 5;
     return (r == 3 || r == 4) ? r : 5;
}

// Shape of the forward mixed contraction (environment LMIE_MIX_SHAPE, read at
// every call; the shapes are listed at MixS0): size tile, angle tile.
struct MixShapeInfo { int id, tm, tn, nt; };
MixShapeInfo mix_shape() {
     const char *e = getenv("LMIE_MIX_SHAPE");
     const int id = e ? atoi(e) : MIX_SHAPE_DEFAULT;
     if (id == 0) return {0, MixS0::TM, MixS0::TN, MixS0::NT};
     if (id == 2) return {2, MixS2::TM, MixS2::TN, MixS2::NT};
     if (id == 3) return {3, MixS3::TM, MixS3::TN, MixS3::NT};
     return {1, MixS1::TM, MixS1::TN, MixS1::NT};
}

// Size tiles per group of xcd_tasks in the forward mixed contraction
// (environment LMIE_MIX_GROUP, read at every call, default 4): the 32
// workgroups in flight on one XCD are then 4 size tiles x 8 angle tiles, so
// each angle tile's operand is read into that XCD's L2 for 4 size tiles and
// each size tile's (the larger operand per tile) for 8 angle tiles.
int mix_group() {
     const char *e = getenv("LMIE_MIX_GROUP");
     const int g = e ? atoi(e) : 4;
     return (g < 1 || g > 64) ? 4 : g;
}

// Size tiles per group of xcd_tasks (environment LMIE_TILE_GROUP, read at
// every call, default 1: the workgroups of one XCD take the column tiles of
// one size tile together).
int tile_group() {
     const char *e = getenv("LMIE_TILE_GROUP");
     const int g = e ? atoi(e) : 1;
     return (g < 1 || g > 64) ? 1 : g;
}

// Initial guesses of the Gauss-Legendre roots, cos(t + (n-1)/(8 n^3) / tan t)
// with t = (4 i + 3) pi / (4 n + 2) (misc/rtutil_math.c:93-97), on the host.
void gauss_guesses(int n, double *g) {
     const int ia = 4 * n + 2;
     const double da = (n - 1) / (8. * pow((double) n, 3));
     for (int i = 0; i < (n + 1) / 2; ++i) {
          const double db = (4. * i + 3.) / ia * kPi;
          g[i] = cos(db + da / tan(db));
     }
}


// What the host works out of a forward job before its launches: padded extents,
// contraction depths, the raw channels of the sums over sizes and the task
// list of the contraction.
struct FwdPlan {
     int N, Np, n1max, Q, C, H, Hp, Kp, Kb, Hb, nt, nw, nch;
     int mixed, bf16, planes, keep, n2max, n2rows, ng, opt, tm, ntile;
     // raw channels: weight rows of the value (row 0 the density, then the
     // weight-only directions and the density tangents of the directions that
     // move x or m), weight rows f dx_i of the value's x derivative, then its
     // Re m and Im m derivatives under the density (angular_f64); comb[o] forms
     // direction o from them
     int nP, nX, nraw, nb;
     bool hx, hm;
     struct Row { const double *src; bool byf; };
     std::vector<Row> rows;
     std::vector<ChComb> comb;
     std::vector<int> kt32, kt64, kt128;
     std::vector<int2> task;
};

int plan_forward(const lmie_gpu_job *J, FwdPlan &p) {
     const int N = J->n_size, n1max = J->n1_max, Q = J->n_qang;
     if (N <= 0) return set_err("no size points");
     if (Q % 2) return set_err("odd n_qang");
     p.n2max = 0;
     for (int i = 0; i < N; ++i) {
          if (J->n1[i] > n1max || J->n1[i] < 1 || J->n2[i] < J->n1[i])
               return set_err("size point %d: order n1 = %d outside [1, %d] (n2 = %d)", i, J->n1[i], n1max, J->n2[i]);
          p.n2max = std::max(p.n2max, J->n2[i]);
     }
     p.N = N; p.Np = rup(N, 2 * TILE);                 // whole tiles of 128 sizes
     p.n1max = n1max; p.Q = Q; p.C = J->n_coef; p.H = Q / 2;
     p.Hp = rup(p.H > 0 ? p.H : 1, TILE); p.Kp = rup(n1max, 32); p.Kb = rup(n1max, KM) / 8;
     // angle padding of the split tables: tiles of 128 angles (whole angle
     // tiles of every contraction shape)
     p.Hb = rup(p.H > 0 ? p.H : 1, 128);
     p.nt = J->n_tan; p.nw = J->n_wgt; p.nch = 1 + p.nt + p.nw;
     // mixed path: value and weight-only channels on the split 16-bit kernel;
     // forward tangents and per-size matrix output stay on the FP64 kernel
     p.mixed = (J->precision == LMIE_PRECISION_MIXED || J->precision == LMIE_PRECISION_MIXED_BF16) && p.nt == 0 &&
               p.nw <= 3 && J->save_control != 1 && Q > 0;
     p.bf16 = J->precision == LMIE_PRECISION_MIXED_BF16;
     p.planes = Q <= 0 ? 0 : J->calc_lc ? 5 : J->calc_gc ? 4 : 0;
     p.keep = J->keep;
     if (p.keep && (p.nt || J->save_control == 1))
          return set_err("the reverse-pass checkpoint covers the value channel only");
     // per-tile contraction depths; operand rows are zero up to the depth of
     // the 128-size tile (the reverse contraction runs whole 128-size tiles)
     const int gran = p.mixed ? KM : KC, nt32 = p.Np / 32, nt64 = p.Np / 64;
     p.kt32.assign(nt32, 0);
     for (int i = 0; i < N; ++i) p.kt32[i / 32] = std::max(p.kt32[i / 32], J->n1[i]);
     for (int &k : p.kt32) k = rup(k, gran);
     p.kt64.resize(nt64);
     p.kt128.resize(nt64 / 2);
     for (int t = 0; t < nt64; ++t) p.kt64[t] = std::max(p.kt32[2 * t], p.kt32[2 * t + 1]);
     int kfmax = 0;
     for (int t = 0; t < nt64 / 2; ++t) kfmax = std::max(kfmax, p.kt128[t] = std::max(p.kt64[2 * t], p.kt64[2 * t + 1]));
     p.n2rows = p.n2max + 1;
     // channels
     auto moves = [&](const double *v) {
          for (int i = 0; i < N; ++i)
               if (v[i] != 0.) return true;
          return false;
     };
     p.rows.assign(1, FwdPlan::Row{J->f, false});
     p.comb.assign(p.nch, ChComb{{-1, -1, -1, -1}, {1., 1., 1., 1.}});
     p.comb[0].r[0] = 0;
     auto row = [&](const double *src, bool byf) { p.rows.push_back(FwdPlan::Row{src, byf}); return (int) p.rows.size() - 1; };
     for (int t = 0; t < p.nw; ++t) p.comb[1 + p.nt + t].r[0] = row(J->df_wgt + (size_t) t * N, false);
     for (int t = 0; t < p.nt; ++t)
          if (moves(J->df_tan + (size_t) t * N)) p.comb[1 + t].r[0] = row(J->df_tan + (size_t) t * N, false);
     p.nP = (int) p.rows.size();
     for (int t = 0; t < p.nt; ++t)
          if (moves(J->dx + (size_t) t * N)) p.comb[1 + t].r[1] = row(J->dx + (size_t) t * N, true);
     p.nX = (int) p.rows.size() - p.nP;
     p.hx = p.nX > 0;
     p.hm = false;
     for (int t = 0; t < p.nt; ++t)
          if (J->dm[2 * t] != 0. || J->dm[2 * t + 1] != 0.) {
               ChComb &c = p.comb[1 + t];
               c.r[2] = p.nP + p.nX; c.r[3] = p.nP + p.nX + 1;
               c.c[2] = J->dm[2 * t]; c.c[3] = J->dm[2 * t + 1];
               p.hm = true;
          }
     p.nraw = p.nP + p.nX + (p.hm ? 2 : 0);
     p.nb = 1 + p.hx + p.hm;
     // orders per thread of the terms: 8, or fewer where the waves of 8 leave the
     // chip's 1024 SIMDs mostly idle and a thread's orders in a row are what the
     // launch takes (every thread forms the order before its first again, so
     // more threads are more work).  Measured, terms of 8 and of fewer: one size
     // 9.1 and 5.7 us (2 orders; 12 waves of 8), 1000 sizes of up to 40 orders 8.6
     // and 5.6 (96), 4096 sizes with tangents 17.3 and 15.0 (4 orders), 4000 of up
     // to 250 orders 22.3 and 20.8 (2016).
     const int waves = p.Np / 64 * (kfmax / 8);
     p.opt = p.mixed ? 8 : p.hx || p.hm ? (waves <= 4096 ? 4 : 8) : waves <= 512 ? 2 : 8;
     p.ng = kfmax / p.opt;
     // the contraction's task list
     p.task.clear();
     p.tm = F64_TILE;
     if (p.mixed) {
          const MixShapeInfo ms = mix_shape();
          p.tm = ms.tm;
          xcd_tasks(ms.tm == 64 ? p.kt64 : p.kt32, [&](int) { return (p.H + ms.tn - 1) / ms.tn; }, mix_group(), p.task);
     } else if (Q > 0)
          xcd_tasks(p.kt32, [&](int) { return (p.H + F64_TILE - 1) / F64_TILE; }, F64_GROUP, p.task);
     p.ntile = p.Np / p.tm;
     return 0;
}

// The inputs of a call, laid out in one pinned buffer and sent as one copy; the
// kernels read them where they land (the pointers of the workspace).  They
// stay valid until the workspace's next forward call.
struct Stage {
     size_t n = 0;
     std::vector<std::pair<Ref *, size_t>> at;
     template <class T> void add(Ref &r, size_t count) {
          at.push_back({&r, n});
          n = (n + sizeof(T) * count + 255) & ~(size_t) 255;
     }
     // device addresses into the Refs; host(r) is r's place in the pinned copy
     unsigned char *hp = nullptr;
     int open(Buf &dev, PinBuf &pin) {
          if (dev.get(n) || pin.get(n)) return -1;
          hp = (unsigned char *) pin.p;
          for (auto &a : at) a.first->p = dev.as<unsigned char>() + a.second;
          return 0;
     }
     template <class T> T *host(const Ref &r, const Buf &dev) const { return (T *) (hp + ((unsigned char *) r.p - (unsigned char *) dev.p)); }
};

int stage_forward(Workspace *w, const lmie_gpu_job *J, const FwdPlan &p, bool batch, hipStream_t s) {
     const int N = p.N, Np = p.Np;
     const size_t nrow = p.rows.size();
     // what the reverse pass needs besides the cotangents goes up with the
     // forward's inputs: the task list and depths of the reverse contraction
     std::vector<int2> rtask;
     if (p.keep && p.mixed) {
          w->ushape = batch ? 8 : ugemm_waves();       // fused passes run the 128-size shape
          const std::vector<int> &kts = w->ushape == 2 ? p.kt64 : p.kt128;
          xcd_tasks(kts, [&](int t) { return (kts[t] + 63) / 64; }, tile_group(), rtask);
     } else if (p.keep && p.Q > 0) {
          w->ushape = adj_f64_orders(p.kt32);
          xcd_tasks(p.kt32, [&](int t) { return (p.kt32[t] + w->ushape - 1) / w->ushape; }, F64_GROUP, rtask);
     }
     w->rtask = rtask;
     w->rch = rev_chunk(Np, p.n2rows);
     Stage st;
     st.add<double>(w->x, Np); st.add<double>(w->sx, Np); st.add<double>(w->cx, Np);
     st.add<double>(w->f, nrow * Np);
     st.add<int>(w->n1, Np); st.add<int>(w->n2, Np);
     st.add<int>(w->kfill, Np / 64); st.add<int>(w->ktile32, Np / 32); st.add<int>(w->ktile64, Np / 64);
     st.add<int>(w->ktile128, Np / 64);
     st.add<ChComb>(w->comb, p.nch); st.add<double>(w->guess, p.H > 0 ? p.H : 1);
     st.add<DotJob>(w->dotjobs, 4 * (size_t) p.nraw);
     st.add<int2>(w->order, p.task.size()); st.add<int2>(w->tasks, rtask.size());
     if (st.open(w->finDev, w->finPin)) return -1;
     auto h = [&](const Ref &r) { return st.host<double>(r, w->finDev); };
     // x, f zero-padded to Np; sin x, cos x of every size from the host C
     // library, as the reference (padding 0, 1)
     auto pad = [&](double *d, const double *v, double fill) {
          memcpy(d, v, sizeof(double) * N);
          for (int i = N; i < Np; ++i) d[i] = fill;
     };
     pad(h(w->x), J->x, 0.);
     double *hs = h(w->sx), *hc = h(w->cx);
     if (J->sx) pad(hs, J->sx, 0.);
     else for (int i = 0; i < Np; ++i) hs[i] = i < N ? sin(J->x[i]) : 0.;
     if (J->cx) pad(hc, J->cx, 1.);
     else for (int i = 0; i < Np; ++i) hc[i] = i < N ? cos(J->x[i]) : 1.;
     for (size_t r = 0; r < nrow; ++r) {
          double *d = h(w->f) + r * Np;
          pad(d, p.rows[r].src, 0.);
          if (p.rows[r].byf)
               for (int i = 0; i < N; ++i) d[i] *= J->f[i];
     }
     auto ints = [&](const Ref &r, const int *v, size_t n, size_t cap) {
          int *d = st.host<int>(r, w->finDev);
          memcpy(d, v, sizeof(int) * n);
          for (size_t k = n; k < cap; ++k) d[k] = 0;
     };
     ints(w->n1, J->n1, N, Np);
     ints(w->n2, J->n2, N, Np);
     ints(w->ktile32, p.kt32.data(), p.kt32.size(), Np / 32);
     ints(w->ktile64, p.kt64.data(), p.kt64.size(), Np / 64);
     int *kf = st.host<int>(w->kfill, w->finDev);
     for (int t = 0; t < Np / 64; ++t) kf[t] = p.kt128[t / 2];
     const std::vector<int> &kts = p.keep && p.mixed && w->ushape == 2 ? p.kt64 : p.kt128;
     ints(w->ktile128, kts.data(), kts.size(), Np / 64);
     memcpy(st.host<ChComb>(w->comb, w->finDev), p.comb.data(), sizeof(ChComb) * p.nch);
     // initial guesses of the Gauss roots (host C library)
     if (p.Q > 0) gauss_guesses(p.Q, h(w->guess));
     // series dot products of every raw channel
     DotJob *dj = st.host<DotJob>(w->dotjobs, w->finDev);
     const double *S0 = w->S.as<double>(), *W0 = w->f.as<double>();
     const double *SX = S0 + 4 * (size_t) Np, *SM = S0 + 4 * (size_t) Np * (p.hx ? 2 : 1);
     for (int c = 0; c < p.nraw; ++c)
          for (int q = 0; q < 4; ++q)
               *dj++ = DotJob{W0 + (c < p.nP + p.nX ? (size_t) c * Np : 0),
                              (c < p.nP ? S0 : c < p.nP + p.nX ? SX : SM + 4 * (size_t) Np * (c - p.nP - p.nX)) + (size_t) q * Np};
     memcpy(st.host<int2>(w->order, w->finDev), p.task.data(), sizeof(int2) * p.task.size());
     memcpy(st.host<int2>(w->tasks, w->finDev), rtask.data(), sizeof(int2) * rtask.size());
     HIPCHECK(hipMemcpyAsync(w->finDev.p, w->finPin.p, st.n, hipMemcpyHostToDevice, s));
     return 0;
}

// Device buffers of a forward call.
int alloc_forward(Workspace *w, const lmie_gpu_job *J, const FwdPlan &p) {
     const size_t Np = p.Np, plane = (size_t) p.Kp * Np, C = p.C, Q = p.Q > 0 ? p.Q : 1, Hp = p.Hp;
     const bool tan = p.hx || p.hm;
     if (w->S.get(sizeof(double) * 4 * Np * (1 + p.hx + 2 * p.hm)) ||
         w->chD.get(sizeof(double) * 2 * (size_t) p.n2rows * Np) || w->chPC.get(sizeof(double) * 2 * (size_t) (p.n1max + 1) * Np) ||
         w->chPS.get(sizeof(double) * Np) || w->chPart.get(sizeof(double) * (5 + 5 * p.hx + 8 * p.hm) * (size_t) (p.ng > 0 ? p.ng : 1) * Np) ||
         (tan && (w->chDz.get(sizeof(double) * 2 * (size_t) p.n2rows * Np) || w->chPQ.get(sizeof(double) * 2 * Np))) ||
         w->ftab.get(sizeof(double) * FT_ROWS * (size_t) (p.n1max + 2)) ||
         (p.mixed ? w->A16.get(sizeof(unsigned short) * 8 * (size_t) p.Kb * Np * 8) : w->A.get(sizeof(double) * 4 * plane * p.nb)) ||
         w->res.get(sizeof(double) * ((size_t) p.nch * 12 * C + 4 * p.nraw)) ||
         w->pres.get(sizeof(double) * ((size_t) p.nch * 12 * C + 4 * p.nraw)) ||
         (p.keep && w->CB.get(sizeof(double) * 2 * Np)))
          return -1;
     if (p.Q <= 0) return 0;
     if (w->mu.get(sizeof(double) * Q) || w->w.get(sizeof(double) * Q) ||
         (p.planes && w->T.get(sizeof(double) * p.planes * gsf_plane(p.C, p.Hp))) ||
         (p.mixed ? w->B16.get(sizeof(unsigned short) * B16_PLANES * (size_t) p.Kb * p.Hb * 8)
                  : (w->Bp.get(sizeof(double) * (size_t) p.Kp * Hp) || w->Bm.get(sizeof(double) * (size_t) p.Kp * Hp))) ||
         w->pf.get(sizeof(double) * (size_t) p.nch * 4 * Q) ||
         w->part.get(sizeof(double) * (size_t) p.ntile * p.nraw * 4 * Q) ||
         (p.keep && !p.mixed && w->sst.get(sizeof(double) * 8 * Np * Hp)) ||
         (J->save_control == 1 && w->save2.get(sizeof(double) * (size_t) 4 * p.N * Q)))
          return -1;
     return 0;
}

// Kernel arguments of the front, the terms and the mixed contraction (shared by
// the single call and the fused batch).
void front_args(const Workspace *w, const lmie_gpu_job *J, const FwdPlan &p, FrontArgs &fa) {
     memset(&fa, 0, sizeof fa);
     ChainArgs &ca = fa.ch;
     ca.N = p.N; ca.Np = p.Np; ca.n1max = p.n1max; ca.n2rows = p.n2rows;
     ca.x = w->x.as<double>(); ca.sx = w->sx.as<double>(); ca.cx = w->cx.as<double>();
     ca.n1 = w->n1.as<int>(); ca.n2 = w->n2.as<int>(); ca.mr = J->mr; ca.mi = J->mi;
     ca.d_all = p.keep; ca.D = w->chD.as<double>(); ca.PC = w->chPC.as<double>(); ca.PS = w->chPS.as<double>();
     ca.Dz = w->chDz.as<double>(); ca.PQ = w->chPQ.as<double>();
     fa.Q = p.Q; fa.H = p.H; fa.Hp = p.Hp; fa.C = p.C; fa.n1max = p.n1max; fa.Kp = p.Kp; fa.Kb = p.Kb; fa.Hb = p.Hb;
     fa.guess = w->guess.as<double>(); fa.mu = w->mu.as<double>(); fa.w = w->w.as<double>();
     fa.T = w->T.as<double>(); fa.Bp = w->Bp.as<double>(); fa.Bm = w->Bm.as<double>();
     fa.B16 = w->B16.as<unsigned short>(); fa.ft = w->ftab.as<double>();
     fa.plan(p.planes, p.Q <= 0 ? 0 : p.mixed ? 2 : 1, p.Q > 0, p.Np / 64, true);
}

void term_args(const Workspace *w, const lmie_gpu_job *J, const FwdPlan &p, TermArgs &ta) {
     ta.N = p.N; ta.Np = p.Np; ta.n1max = p.n1max; ta.n2rows = p.n2rows; ta.Kp = p.Kp; ta.Kb = p.Kb; ta.ng = p.ng;
     ta.ft = w->ftab.as<double>();
     ta.x = w->x.as<double>(); ta.n1 = w->n1.as<int>(); ta.kfill = w->kfill.as<int>();
     ta.mr = J->mr; ta.mi = J->mi; ta.D = w->chD.as<double>(); ta.PC = w->chPC.as<double>(); ta.PS = w->chPS.as<double>();
     ta.A = p.mixed ? nullptr : w->A.as<double>();
     ta.A16 = p.mixed ? w->A16.as<unsigned short>() : nullptr;
     ta.part = w->chPart.as<double>();
}

void mix_args(const Workspace *w, const FwdPlan &p, Mix2Args &m) {
     memset(&m, 0, sizeof m);
     m.Np = p.Np; m.Kb = p.Kb; m.Hb = p.Hb; m.H = p.H; m.Q = p.Q;
     m.A16 = w->A16.as<unsigned short>();
     m.B16 = w->B16.as<unsigned short>();
     m.ktile = p.tm == 64 ? w->ktile64.as<int>() : w->ktile32.as<int>();
     m.task = w->order.as<int2>();
     for (int q = 0; q <= p.nw; ++q) m.W[q] = w->f.as<double>() + (size_t) q * p.Np;
     m.part = w->part.as<double>();
}

// Results of a call: the series sums of the raw channels [4 nraw], then the
// expansions, generalized spherical [nch][6][C] and Legendre [nch][6][C], in
// one buffer.
void reduce_args(const Workspace *w, const FwdPlan &p, double *res, ReduceArgs &r) {
     r.part = w->part.as<double>(); r.nblk = p.ntile; r.nraw = p.nraw; r.Q = p.Q > 0 ? p.Q : 0; r.nch = p.nch;
     r.comb = p.nt ? w->comb.as<ChComb>() : nullptr;
     r.out = w->pf.as<double>();
     r.jobs = w->dotjobs.as<DotJob>(); r.n = p.Np; r.ndot = 4 * p.nraw; r.dots = res;
     r.gx = (unsigned) ((r.nch * 4 * r.Q + 31) / 32 + r.ndot);
}

void keep_forward(Workspace *w, const lmie_gpu_job *J, const FwdPlan &p) {
     w->N = p.N; w->Np = p.Np; w->Kp = p.Kp; w->Hp = p.Hp; w->H = p.H; w->Q = p.Q; w->C = p.C; w->n1max = p.n1max;
     w->n2max = p.n2max; w->n2rows = p.n2rows;
     w->calc_gc = J->calc_gc; w->calc_lc = J->calc_lc; w->mr = J->mr; w->mi = J->mi;
     w->mixed = p.mixed; w->bf16 = p.bf16; w->Kb = p.Kb; w->Hb = p.Hb;
}

// Raw sums of every direction from those of the raw channels.
void unpack_sums(const FwdPlan &p, const double *dots, lmie_gpu_result *R) {
     for (int q = 0; q < 4; ++q) R->sums[q] = dots[q];
     for (int c = 1; c < p.nch; ++c)
          for (int q = 0; q < 4; ++q) {
               double v = 0.;
               for (int t = 0; t < 4; ++t)
                    if (p.comb[c].r[t] >= 0) v += p.comb[c].c[t] * dots[4 * p.comb[c].r[t] + q];
               R->sums_ch[4 * (c - 1) + q] = v;
          }
}

int forward_impl(const lmie_gpu_job *J, lmie_gpu_result *R, Workspace *w) {
     const auto t_entry = std::chrono::steady_clock::now();
     hipStream_t s = w->stream;
     Timer tm{w, g_timing};
     w->valid = 0;
     FwdPlan p;
     if (plan_forward(J, p) || alloc_forward(w, J, p) || stage_forward(w, J, p, false, s)) return -1;
     const int N = p.N, Np = p.Np, Q = p.Q, C = p.C, nch = p.nch, keep = p.keep;
     const bool tan = p.hx || p.hm;
     const double prep_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_entry).count();
     tm.mark(LMIE_T_TOTAL, 0);

     // angle tables, chains and order factors; terms; per-size sums
     tm.mark(LMIE_T_COEFS, 0);
     FrontArgs fa;
     front_args(w, J, p, fa);
     tm.mark(LMIE_T_TABLES, 0);
     if (launch_front(fa, !p.mixed ? 1 : p.bf16 ? 3 : 2, tan, s)) return -1;
     tm.mark(LMIE_T_TABLES, 1);
     const dim3 gt(Np / 64, p.ng), gs((Np + 31) / 32);
     if (tan) {
          TanArgs ta;
          ta.N = N; ta.Np = Np; ta.n1max = p.n1max; ta.n2rows = p.n2rows; ta.Kp = p.Kp; ta.ng = p.ng;
          ta.ft = w->ftab.as<double>();
          ta.x = w->x.as<double>(); ta.n1 = w->n1.as<int>(); ta.kfill = w->kfill.as<int>();
          ta.mr = J->mr; ta.mi = J->mi; ta.D = w->chD.as<double>(); ta.Dz = w->chDz.as<double>();
          ta.PC = w->chPC.as<double>(); ta.PS = w->chPS.as<double>(); ta.PQ = w->chPQ.as<double>();
          for (int b = 0; b < p.nb; ++b) ta.A[b] = w->A.as<double>() + 4 * (size_t) p.Kp * Np * b;
          ta.part = w->chPart.as<double>();
#define LMIE_TAN(X, M)                                                                                           \
          do {                                                                                                   \
               if (p.ng > 0 && p.opt == 4) hipLaunchKernelGGL((mie_tan_terms<X, M, 4>), gt, dim3(64), 0, s, ta);  \
               else if (p.ng > 0) hipLaunchKernelGGL((mie_tan_terms<X, M, 8>), gt, dim3(64), 0, s, ta);          \
               hipLaunchKernelGGL((mie_tan_sums<X, M>), gs, dim3(1024), 0, s, (const double *) w->chPart.as<double>(), N, Np, \
                                  p.ng, p.opt, (const int *) w->n1.as<int>(), w->S.as<double>());                       \
          } while (0)
          if (p.hx && p.hm) LMIE_TAN(true, true);
          else if (p.hx) LMIE_TAN(true, false);
          else LMIE_TAN(false, true);
#undef LMIE_TAN
     } else {
          TermArgs ta;
          term_args(w, J, p, ta);
          if (p.ng > 0) {
               if (!p.mixed && p.opt == 2) hipLaunchKernelGGL((mie_terms<void, 2>), gt, dim3(64), 0, s, ta);
               else if (!p.mixed) hipLaunchKernelGGL((mie_terms<void, 8>), gt, dim3(64), 0, s, ta);
               else if (p.bf16) hipLaunchKernelGGL((mie_terms<BF16, 8>), gt, dim3(64), 0, s, ta);
               else hipLaunchKernelGGL((mie_terms<F16, 8>), gt, dim3(64), 0, s, ta);
          }
          hipLaunchKernelGGL(mie_sums, gs, dim3(256), 0, s, (const double *) w->chPart.as<double>(), N, Np,
                             p.ng, p.opt, (const int *) w->n1.as<int>(), w->S.as<double>(), keep ? w->CB.as<double>() : nullptr);
     }
     HIPCHECK(hipGetLastError());
     tm.mark(LMIE_T_COEFS, 1);

     // angular contraction
     if (Q > 0) {
          tm.mark(LMIE_T_ANGULAR, 0);
          if (p.mixed) {
               Mix2Args m;
               mix_args(w, p, m);
               const dim3 grid((unsigned) p.task.size());
               const int nw = p.nw, id = mix_shape().id;
               // five split products (three with LMIE_MIX_PRODUCTS=3), in the
               // shape of LMIE_MIX_SHAPE
#define LMIE_MIX(E, NP, NWC, S) hipLaunchKernelGGL((angular_mix<E, NP, NWC, S>), grid, dim3(S::NT), 0, s, m)
#define LMIE_MIX_NW(E, NP, S)                                                                            \
               do {                                                                                      \
                    if (nw == 0) LMIE_MIX(E, NP, 1, S); else if (nw == 1) LMIE_MIX(E, NP, 2, S);        \
                    else if (nw == 2) LMIE_MIX(E, NP, 3, S); else LMIE_MIX(E, NP, 4, S);                \
               } while (0)
#define LMIE_MIX_NP(E, S)                                                                                \
               do {                                                                                      \
                    if (mix_products() == 3) LMIE_MIX_NW(E, 3, S);                                       \
                    else if (mix_products() == 4 && std::is_same<S, MixS3>::value) LMIE_MIX_NW(E, 4, MixS3); \
                    else LMIE_MIX_NW(E, 5, S);                                                          \
               } while (0)
#define LMIE_MIX_S(S) do { if (p.bf16) LMIE_MIX_NP(BF16, S); else LMIE_MIX_NP(F16, S); } while (0)
               if (id == 0) LMIE_MIX_S(MixS0);
               else if (id == 2) LMIE_MIX_S(MixS2);
               else if (id == 3) LMIE_MIX_S(MixS3);
               else LMIE_MIX_S(MixS1);
#undef LMIE_MIX_S
#undef LMIE_MIX_NP
#undef LMIE_MIX_NW
#undef LMIE_MIX
               HIPCHECK(hipGetLastError());
          } else {
               F64Args a;
               memset(&a, 0, sizeof a);
               a.Np = Np; a.Kp = p.Kp; a.Hp = p.Hp; a.H = p.H; a.Q = Q; a.N = N;
               for (int b = 0; b < p.nb; ++b) a.A[b] = w->A.as<double>() + 4 * (size_t) p.Kp * Np * b;
               a.Bp = w->Bp.as<double>(); a.Bm = w->Bm.as<double>();
               a.ktile = w->ktile32.as<int>();
               a.task = w->order.as<int2>();
               a.W = w->f.as<double>(); a.nP = p.nP; a.nX = p.nX;
               a.part = w->part.as<double>();
               a.save2 = J->save_control == 1 ? w->save2.as<double>() : nullptr;
               a.sst = keep ? w->sst.as<double>() : nullptr;
               if (launch_angular_f64(a, p.hx, p.hm, (unsigned) p.task.size(), s)) return -1;
          }
          tm.mark(LMIE_T_ANGULAR, 1);
     }
     // sums over the size tiles and the series sums, then the expansions
     double *res = w->res.as<double>(), *land = (double *) w->pres.p;
     const size_t ndot = 4 * (size_t) p.nraw, nx = (size_t) nch * 6 * C;
     tm.mark(LMIE_T_REDUCE, 0);
     ReduceArgs ra;
     reduce_args(w, p, res, ra);
     hipLaunchKernelGGL(reduce_channels, dim3(ra.gx), dim3(256), 0, s, ra);
     HIPCHECK(hipGetLastError());
     tm.mark(LMIE_T_REDUCE, 1);
     const bool gc = Q > 0 && J->calc_gc && R->gc_raw, lc = Q > 0 && J->calc_lc && R->lc_raw;
     if (Q > 0) {
          tm.mark(LMIE_T_EXPAND, 0);
          for (int gsf = 1; gsf >= 0; --gsf)
               if (gsf ? gc : lc)
                    hipLaunchKernelGGL(expand_coefs, dim3((C + 7) / 8, nch), dim3(256), 0, s, (const double *) w->T.as<double>(),
                                       (const double *) w->pf.as<double>(), (const double *) w->w.as<double>(), Q, p.Hp, C, gsf,
                                       res + ndot + (gsf ? 0 : nx));
          HIPCHECK(hipGetLastError());
          tm.mark(LMIE_T_EXPAND, 1);
          if (J->save_control == 1 && R->save2)
               HIPCHECK(hipMemcpyAsync(R->save2, w->save2.p, sizeof(double) * (size_t) 4 * N * Q, hipMemcpyDeviceToHost, s));
     }
     tm.mark(LMIE_T_TOTAL, 1);
     // results: one copy into the pinned landing area
     HIPCHECK(hipMemcpyAsync(land, res, sizeof(double) * (ndot + (lc ? 2 * nx : gc ? nx : 0)), hipMemcpyDeviceToHost, s));
     if (J->save_control == 1 && R->save1)
          for (int q = 0; q < 4; ++q)
               HIPCHECK(hipMemcpyAsync(R->save1 + (size_t) q * N, w->S.as<double>() + (size_t) q * Np,
                                       sizeof(double) * N, hipMemcpyDeviceToHost, s));
     HIPCHECK(hipStreamSynchronize(s));
     if (gc) memcpy(R->gc_raw, land + ndot, sizeof(double) * nx);
     if (lc) memcpy(R->lc_raw, land + ndot + nx, sizeof(double) * nx);
     unpack_sums(p, land, R);
     const int ids[] = {LMIE_T_TABLES, LMIE_T_COEFS, LMIE_T_REDUCE, LMIE_T_TOTAL, LMIE_T_ANGULAR, LMIE_T_EXPAND};
     tm.collect(ids, Q > 0 ? 6 : 4);
     lmie_gpu_host_time(LMIE_T_HOST_PREP, prep_ms);
     w->valid = 1;
     keep_forward(w, J, p);
     R->precision = p.mixed ? J->precision : LMIE_PRECISION_FP64;
     return 0;
}

// Re-weighting of the per-size series and matrix elements of an earlier call
// (save_control = 2, src/lmie_schedule.c:1087-1124): per channel c with
// weights W[c][i], pf[c][q][j] = sum_i W[c][i] s2[q][i][j] and
// dots[c][q] = sum_i W[c][i] s1[q][i].  Eight lanes per output, each adding
// every eighth size, then the eight partials in a fixed order.
__global__ __launch_bounds__(256) void saved_sums(const double *W, const double *s1, const double *s2, int N, int Q,
                                                  double *pf, double *dots) {
     const int per = 4 * (Q + 1), c = blockIdx.y;
     const int e = blockIdx.x * 32 + (threadIdx.x >> 3), l = threadIdx.x & 7;
     const double *w = W + (size_t) c * N;
     double s = 0.;
     if (e < 4 * Q) {
          const int q = e / Q, j = e % Q;
          for (int i = l; i < N; i += 8) s += w[i] * s2[((size_t) q * N + i) * Q + j];
     } else if (e < per) {
          const int q = e - 4 * Q;
          for (int i = l; i < N; i += 8) s += w[i] * s1[(size_t) q * N + i];
     }
     s += __shfl_xor(s, 1);
     s += __shfl_xor(s, 2);
     s += __shfl_xor(s, 4);
     if (l || e >= per) return;
     if (e < 4 * Q) pf[(size_t) c * 4 * Q + e] = s;
     else dots[4 * c + e - 4 * Q] = s;
}

// save_control = 2: the raw sums and expansions from the saved per-size
// arrays and new weights (FP64), on the main stream.  Channels as the
// forward: value, Mie tangents (zero: the saved arrays carry none), weights.
int saved_impl(const lmie_gpu_job *J, lmie_gpu_result *R, Workspace *w) {
     const int N = J->n_size, Q = J->n_qang, C = J->n_coef;
     const int nt = J->n_tan, nw = J->n_wgt, nch = 1 + nt + nw;
     const int H = Q / 2, Hp = rup(H > 0 ? H : 1, TILE);
     if (!J->saved1 || (Q > 0 && !J->saved2)) return set_err("save_control = 2 needs the saved per-size arrays");
     if (N < 1) return set_err("no size points");
     hipStream_t s = w->stream;
     Timer tm{w, g_timing};
     if (w->sw.get(sizeof(double) * (size_t) nch * N) || w->s1.get(sizeof(double) * 4 * (size_t) N) ||
         (Q > 0 && w->s2.get(sizeof(double) * 4 * (size_t) N * Q)) ||
         w->pf.get(sizeof(double) * (size_t) nch * 4 * (Q > 0 ? Q : 1)) || w->dots.get(sizeof(double) * 4 * nch) ||
         w->res.get(sizeof(double) * (size_t) nch * 6 * C))
          return -1;
     double *W = w->sw.as<double>();
     HIPCHECK(hipMemcpyAsync(W, J->f, sizeof(double) * N, hipMemcpyHostToDevice, s));
     if (nt) HIPCHECK(hipMemsetAsync(W + (size_t) N, 0, sizeof(double) * (size_t) nt * N, s));
     if (nw)
          HIPCHECK(hipMemcpyAsync(W + (size_t) (1 + nt) * N, J->df_wgt, sizeof(double) * (size_t) nw * N,
                                  hipMemcpyHostToDevice, s));
     HIPCHECK(hipMemcpyAsync(w->s1.p, J->saved1, sizeof(double) * 4 * (size_t) N, hipMemcpyHostToDevice, s));
     if (Q > 0)
          HIPCHECK(hipMemcpyAsync(w->s2.p, J->saved2, sizeof(double) * 4 * (size_t) N * Q, hipMemcpyHostToDevice, s));
     tm.mark(LMIE_T_TOTAL, 0);
     if (Q > 0) {
          // Gauss rule and expansion tables (as the forward)
          if (w->mu.get(sizeof(double) * Q) || w->w.get(sizeof(double) * Q) || w->sguess.get(sizeof(double) * H) ||
              w->pin.get(sizeof(double) * H))
               return -1;
          gauss_guesses(Q, (double *) w->pin.p);
          HIPCHECK(hipMemcpyAsync(w->sguess.p, w->pin.p, sizeof(double) * H, hipMemcpyHostToDevice, s));
          FrontArgs fa;
          memset(&fa, 0, sizeof fa);
          const int planes = J->calc_lc ? 5 : J->calc_gc ? 4 : 0;
          if (planes && w->T.get(sizeof(double) * planes * gsf_plane(C, Hp))) return -1;
          fa.Q = Q; fa.H = H; fa.Hp = Hp; fa.C = C;
          fa.guess = w->sguess.as<double>(); fa.mu = w->mu.as<double>(); fa.w = w->w.as<double>(); fa.T = w->T.as<double>();
          fa.plan(planes, 0, true, 0, false);
          if (launch_front(fa, 0, false, s)) return -1;
     }
     const int per = 4 * (Q + 1);
     hipLaunchKernelGGL(saved_sums, dim3((per + 31) / 32, nch), dim3(256), 0, s, (const double *) W,
                        (const double *) w->s1.as<double>(), (const double *) w->s2.as<double>(), N, Q,
                        w->pf.as<double>(), w->dots.as<double>());
     HIPCHECK(hipGetLastError());
     if (Q > 0) {
          for (int gsf = 1; gsf >= 0; --gsf) {
               double *dst = gsf ? R->gc_raw : R->lc_raw;
               if (!(gsf ? J->calc_gc : J->calc_lc) || !dst) continue;
               hipLaunchKernelGGL(expand_coefs, dim3((C + 7) / 8, nch), dim3(256), 0, s, (const double *) w->T.as<double>(),
                                  (const double *) w->pf.as<double>(), (const double *) w->w.as<double>(), Q, Hp, C, gsf,
                                  w->res.as<double>());
               HIPCHECK(hipGetLastError());
               HIPCHECK(hipMemcpyAsync(dst, w->res.p, sizeof(double) * (size_t) nch * 6 * C, hipMemcpyDeviceToHost, s));
          }
     }
     tm.mark(LMIE_T_TOTAL, 1);
     std::vector<double> dots((size_t) 4 * nch);
     HIPCHECK(hipMemcpyAsync(dots.data(), w->dots.p, sizeof(double) * 4 * nch, hipMemcpyDeviceToHost, s));
     HIPCHECK(hipStreamSynchronize(s));
     for (int q = 0; q < 4; ++q) R->sums[q] = dots[q];
     for (int c = 1; c < nch; ++c)
          for (int q = 0; q < 4; ++q) R->sums_ch[4 * (c - 1) + q] = dots[4 * c + q];
     const int ids[] = {LMIE_T_TOTAL};
     tm.collect(ids, 1);
     w->valid = 0;
     return 0;
}

int rev_chunks(const Workspace *w) { return (w->n2rows - 1 + w->rch - 1) / w->rch; }

// Buffers of a reverse pass (use_u: through G on the 16-bit matrix cores).
int alloc_reverse(Workspace *w, bool use_u) {
     const size_t Np = w->Np, Q = w->Q > 0 ? w->Q : 1, C = w->C > 0 ? w->C : 1;
     const size_t Kq = rup(w->n1max, 64), Hq = rup(w->H > 0 ? w->H : 1, KM);
     const size_t nck = (w->C + EXA_L - 1) / EXA_L, nch = rev_chunks(w);
     if (use_u && rup(w->n1max, KM) > w->Kb * 8) return set_err("internal: split operand depth");
     const size_t nres = 2 * (size_t) w->N + Np / 32;
     if (w->pfbar.get(sizeof(double) * 4 * Q) || w->gbar.get(sizeof(double) * 12 * C) || w->pin.get(sizeof(double) * 12 * C) ||
         w->rres.get(sizeof(double) * nres) || w->pres.get(sizeof(double) * nres) ||
         w->revScan.get(sizeof(double) * REV_ROWS * (nch > 0 ? nch : 1) * Np) ||
         (w->Q > 0 && w->expart.get(sizeof(double) * 24 * nck * w->Hp)))
          return -1;
     if (!use_u)
          return w->fang.get(sizeof(double) * Np) || w->bar.get(sizeof(double) * 4 * (size_t) w->Kp * Np) ||
                         w->wts.get(sizeof(double) * 8 * ((size_t) w->Hp + ADJ_KS)) ? -1 : 0;
     return w->wts.get(sizeof(double) * 8 * Hq) || w->scal.get(sizeof(AdjScal)) ||
                    w->L16.get(sizeof(unsigned short) * 4 * Hq * Kq) || w->R16.get(sizeof(unsigned short) * 16 * Hq * Kq) ||
                    w->Gf.get(sizeof(float) * 4 * Kq * Kq) || w->G16.get(sizeof(unsigned short) * 12 * Kq * Kq) ||
                    w->Uf.get(sizeof(float) * 4 * Kq * Np) ? -1 : 0;
}

// The expansion cotangents through the pinned staging area: gc [6][C] at 0,
// lc at 6 C of gbar.
int stage_reverse(Workspace *w, const lmie_gpu_adj_in *in, bool use_gc, bool use_lc, hipStream_t s) {
     const size_t n = 6 * (size_t) w->C, o = use_gc ? 0 : n, e = use_lc ? 2 * n : n;
     double *h = (double *) w->pin.p;
     if (!use_gc && !use_lc) return 0;
     if (use_gc) memcpy(h, in->gc_bar, sizeof(double) * n);
     if (use_lc) memcpy(h + n, in->lc_bar, sizeof(double) * n);
     HIPCHECK(hipMemcpyAsync(w->gbar.as<double>() + o, h + o, sizeof(double) * (e - o), hipMemcpyHostToDevice, s));
     return 0;
}

// Arguments of the per-size reverse sweep.
void rev_args(const Workspace *w, const lmie_gpu_adj_in *in, bool xbar, bool use_u, RevArgs &r) {
     const int nch = rev_chunks(w);
     r.rch = w->rch;
     r.N = w->N; r.Np = w->Np; r.Kp = w->Kp; r.n1max = w->n1max; r.n2rows = w->n2rows; r.nch = nch;
     r.ft = w->ftab.as<double>();
     r.x = w->x.as<double>(); r.f = w->f.as<double>();
     r.n1 = w->n1.as<int>(); r.n2 = w->n2.as<int>(); r.mr = w->mr; r.mi = w->mi; rev_recips(r);
     r.D = w->chD.as<double>(); r.PC = w->chPC.as<double>(); r.PS = w->chPS.as<double>();
     r.CB = w->CB.as<double>(); r.S = w->S.as<double>(); r.bar = use_u ? nullptr : w->bar.as<double>();
     r.Uf = use_u ? w->Uf.as<float>() : nullptr; r.Kq = rup(w->n1max, 64);
     r.fang = nullptr;
     r.sb0 = in->sums_bar[0]; r.sb1 = in->sums_bar[1]; r.sb2 = in->sums_bar[2]; r.sb3 = in->sums_bar[3];
     r.scan = w->revScan.as<double>();
     r.fbar = w->rres.as<double>();
     r.xbar = xbar ? r.fbar + w->N : nullptr;
     r.mbar = r.fbar + 2 * (size_t) w->N;
}

// A reverse pass's results out of its landing area.
void unpack_reverse(const Workspace *w, const double *land, lmie_gpu_adj_out *out) {
     const size_t N = w->N;
     memcpy(out->f_bar, land, sizeof(double) * N);
     if (out->x_bar) memcpy(out->x_bar, land + N, sizeof(double) * N);
     double mr = 0., mi = 0.;
     for (int b = 0; b < w->Np / 64; ++b) {
          mr += land[2 * N + 2 * b];
          mi += land[2 * N + 2 * b + 1];
     }
     // m = mr - i mi: dL/dmr = Re(mbar), dL/dmi = -Im(mbar)
     out->m_bar[0] = mr;
     out->m_bar[1] = -mi;
}

// Mixed reverse contraction: weights, split tables, G, its split operand and
// U = G A (Uf, [4][Kq][Np]).
int adjoint_mixed_angular(Workspace *w, hipStream_t s, Timer &tm) {
     const int Np = w->Np, H = w->H, Q = w->Q, n1max = w->n1max;
     const int Kq = rup(n1max, 64), Hq = rup(H, KM);
     const int shape = w->ushape;
     const unsigned ntask = (unsigned) w->rtask.size();
     if (ntask == 0) {
          HIPCHECK(hipMemsetAsync(w->Uf.p, 0, sizeof(float) * 4 * (size_t) Kq * Np, s));
          return 0;
     }
     AdjScal *sc = w->scal.as<AdjScal>();
     hipLaunchKernelGGL(adj_weights, dim3(1), dim3(1024), 0, s, (const double *) w->pfbar.as<double>(), H, Hq, Q,
                        w->wts.as<double>(), sc);
     UArgs u;
     u.Np = Np; u.Kb = w->Kb; u.Kq = Kq;
     u.A16 = w->A16.as<unsigned short>(); u.G16 = w->G16.as<unsigned short>();
     u.ktile = w->ktile128.as<int>(); u.task = w->tasks.as<int2>(); u.sc = sc; u.Uf = w->Uf.as<float>();
#define LMIE_ADJ(E)                                                                                            \
     do {                                                                                                     \
          hipLaunchKernelGGL(adj_tables<E>, dim3(Kq / 64, Hq / 8), dim3(64), 0, s,                              \
                             (const unsigned short *) w->B16.as<unsigned short>(), w->Kb, w->Hb,                      \
                             (const double *) w->wts.as<double>(), H, Hq, Kq, n1max, w->L16.as<unsigned short>(),    \
                             w->R16.as<unsigned short>());                                                            \
          hipLaunchKernelGGL(adj_gbuild<E>, dim3((Kq / 64) * (Kq / 64)), dim3(256), 0, s,                       \
                             (const unsigned short *) w->L16.as<unsigned short>(),                             \
                             (const unsigned short *) w->R16.as<unsigned short>(), Hq, Kq, w->Gf.as<float>(), sc); \
          hipLaunchKernelGGL(adj_gsplit<E>, dim3(Kq / 64, Kq / 8), dim3(64), 0, s, (const float *) w->Gf.as<float>(), \
                             (const AdjScal *) sc, Kq, w->G16.as<unsigned short>());                           \
          tm.mark(LMIE_T_ADJ_GEMM, 0);                                                                          \
          if (shape == 4)                                                                                       \
               hipLaunchKernelGGL((adj_ugemm32<E, 2, 128, false>), dim3(ntask), dim3(256), 0, s, u, nullptr, nullptr);  \
          else if (shape == 2)                                                                                  \
               hipLaunchKernelGGL((adj_ugemm32<E, 1, 64, false>), dim3(ntask), dim3(256), 0, s, u, nullptr, nullptr);   \
          else                                                                                                  \
               hipLaunchKernelGGL((adj_ugemm32<E, 1, 128, false>), dim3(ntask), dim3(512), 0, s, u, nullptr, nullptr);  \
          tm.mark(LMIE_T_ADJ_GEMM, 1);                                                                          \
     } while (0)
     if (w->bf16) LMIE_ADJ(BF16);
     else LMIE_ADJ(F16);
#undef LMIE_ADJ
     HIPCHECK(hipGetLastError());
     return 0;
}

int adjoint_impl(Workspace *w, const lmie_gpu_adj_in *in, lmie_gpu_adj_out *out) {
     if (!w->valid) return set_err("no forward state");
     const int N = w->N, Np = w->Np, Kp = w->Kp, Hp = w->Hp, H = w->H, Q = w->Q, C = w->C;
     hipStream_t s = w->stream;
     Timer tm{w, g_timing};
     const int use_gc = in->gc_bar && w->calc_gc && Q > 0, use_lc = in->lc_bar && w->calc_lc && Q > 0;
     const int use_u = w->mixed && (use_gc || use_lc);
     // the cotangents go to the device before the timed pipeline
     if (alloc_reverse(w, use_u) || stage_reverse(w, in, use_gc, use_lc, s)) return -1;
     double *g = w->gbar.as<double>();
     RevArgs r;
     rev_args(w, in, out->x_bar != nullptr, use_u, r);
     tm.mark(LMIE_T_TOTAL, 0);
     if (Q > 0 && (use_gc || use_lc)) {
          tm.mark(LMIE_T_ADJ_ANGULAR, 0);
          const int nck = (C + EXA_L - 1) / EXA_L;
          hipLaunchKernelGGL(expand_adjoint_part, dim3(Hp / 64, nck), dim3(64), 0, s, (const double *) w->T.as<double>(),
                             use_gc ? (const double *) g : nullptr, use_lc ? (const double *) (g + 6 * C) : nullptr,
                             H, Hp, C, w->expart.as<double>());
          hipLaunchKernelGGL(expand_adjoint_fin, dim3((H + EXF_J - 1) / EXF_J), dim3(24 * EXF_J), 0, s, (const double *) w->expart.as<double>(),
                             nck, (const double *) w->w.as<double>(), H, Hp, Q, w->pfbar.as<double>(),
                             w->mixed ? nullptr : w->wts.as<double>());
     }
     if (w->mixed && Q > 0 && (use_gc || use_lc)) {
          if (adjoint_mixed_angular(w, s, tm)) return -1;
          tm.mark(LMIE_T_ADJ_ANGULAR, 1);
     } else if (Q > 0 && (use_gc || use_lc)) {
          hipLaunchKernelGGL(fbar_angular, dim3((N + 3) / 4), dim3(256), 0, s, (const double *) w->sst.as<double>(),
                             (const double *) w->pfbar.as<double>(), N, Np, H, Hp, Q, w->fang.as<double>());
          r.fang = w->fang.as<double>();
          AdjArgs aa;
          aa.Np = Np; aa.Kp = Kp; aa.Hp = Hp; aa.H = H;
          aa.sst = w->sst.as<double>(); aa.wts = w->wts.as<double>();
          aa.Bp = w->Bp.as<double>(); aa.Bm = w->Bm.as<double>();
          aa.f = w->f.as<double>(); aa.task = w->tasks.as<int2>(); aa.bar = w->bar.as<double>();
          if (!w->rtask.empty()) {
               const dim3 g((unsigned) w->rtask.size());
               if (w->ushape == 64) hipLaunchKernelGGL(angular_adj_f64<2>, g, dim3(256), 0, s, aa);
               else hipLaunchKernelGGL(angular_adj_f64<1>, g, dim3(256), 0, s, aa);
          }
          HIPCHECK(hipGetLastError());
          tm.mark(LMIE_T_ADJ_ANGULAR, 1);
     } else {
          tm.mark(LMIE_T_ADJ_ANGULAR, 0);
          HIPCHECK(hipMemsetAsync(w->bar.p, 0, sizeof(double) * 4 * (size_t) Kp * Np, s));
          tm.mark(LMIE_T_ADJ_ANGULAR, 1);
     }
     tm.mark(LMIE_T_ADJ_COEFS, 0);
     if (r.nch > 0) {
          if (use_u) hipLaunchKernelGGL(rev_orders<true>, dim3(Np / 64, r.nch), dim3(64), 0, s, r);
          else hipLaunchKernelGGL(rev_orders<false>, dim3(Np / 64, r.nch), dim3(64), 0, s, r);
     }
     hipLaunchKernelGGL(rev_carry, dim3(Np / 64), dim3(64), 0, s, r);
     HIPCHECK(hipGetLastError());
     tm.mark(LMIE_T_ADJ_COEFS, 1);
     // results through the pinned landing area
     tm.mark(LMIE_T_TOTAL, 1);
     HIPCHECK(hipMemcpyAsync(w->pres.p, w->rres.p, sizeof(double) * (2 * (size_t) N + Np / 32), hipMemcpyDeviceToHost, s));
     HIPCHECK(hipStreamSynchronize(s));
     unpack_reverse(w, (const double *) w->pres.p, out);
     const int ids[] = {LMIE_T_ADJ_ANGULAR, LMIE_T_ADJ_COEFS, LMIE_T_TOTAL, LMIE_T_ADJ_GEMM};
     tm.collect(ids, use_u ? 4 : 3);
     return 0;
}

// ---------------------------------------------------------------------------
// Batches of independent cases in one launch per kernel.  The host thread
// that runs case k of a batch (lmie_gpu_batch_enter) hands its forward and
// later its reverse pass to the batch instead of running them; when every
// case has arrived (or left), one thread runs the pass for all cases: each
// case keeps its own workspace (buffers, reverse-pass state), and every kernel
// is launched once, with blockIdx.z (or the task list) picking the case.
// Fused: mixed precision, value channel only, angles, save_control 0, kept
// state (the forward of a reverse pass); other cases run one by one.


struct BatchBlob {   // host staging of per-case argument arrays, one upload
     std::vector<unsigned char> h;
     template <class T> size_t add(const std::vector<T> &v) {
          const size_t off = (h.size() + 255) & ~(size_t) 255;
          h.resize(off + sizeof(T) * (v.empty() ? 1 : v.size()));
          if (!v.empty()) memcpy(h.data() + off, v.data(), sizeof(T) * v.size());
          return off;
     }
};

template <class T> unsigned max_g(const std::vector<T> &v, unsigned T::*g) {
     unsigned m = 0;
     for (const T &x : v) m = std::max(m, x.*g);
     return m;
}

struct FwdCase {
     int slot;
     const lmie_gpu_job *J;
     lmie_gpu_result *R;
     Workspace *w;
     FwdPlan p;
};

int fused_forward_ok(const lmie_gpu_job *J) {
     return (J->precision == LMIE_PRECISION_MIXED || J->precision == LMIE_PRECISION_MIXED_BF16) && J->n_tan == 0 &&
            J->n_wgt == 0 && J->save_control == 0 && J->keep && J->n_qang > 0 && J->n_qang % 2 == 0 &&
            (J->calc_gc || J->calc_lc);
}

// Sends a batch's per-case arguments (from pinned memory) and gives their
// device address.
int send_args(Workspace *L, const std::vector<unsigned char> &h, hipStream_t s, unsigned char **d) {
     if (L->bargs.get(h.size()) || L->pargs.get(h.size())) return -1;
     memcpy(L->pargs.p, h.data(), h.size());
     HIPCHECK(hipMemcpyAsync(L->bargs.p, L->pargs.p, h.size(), hipMemcpyHostToDevice, s));
     *d = L->bargs.as<unsigned char>();
     return 0;
}

// Buffers and inputs of one case, sent on its own stream; no kernels.
int fused_prepare(FwdCase &c) {
     return plan_forward(c.J, c.p) || alloc_forward(c.w, c.J, c.p) || stage_forward(c.w, c.J, c.p, true, c.w->stream) ? -1 : 0;
}

// A case's results out of its landing area: the series sums, then the
// expansions.
void fused_unpack(const FwdCase &c) {
     const double *land = (const double *) c.w->pres.p;
     const size_t n = 6 * (size_t) c.p.C;
     unpack_sums(c.p, land, c.R);
     if (c.J->calc_gc && c.R->gc_raw) memcpy(c.R->gc_raw, land + 4, sizeof(double) * n);
     if (c.J->calc_lc && c.R->lc_raw) memcpy(c.R->lc_raw, land + 4 + n, sizeof(double) * n);
}

// One launch per kernel over the prepared cases, on the stream of workspace L.
template <class E>
int fused_launch(std::vector<FwdCase *> &cs, Workspace *L) {
     hipStream_t s = L->stream;
     const unsigned n = (unsigned) cs.size();
     std::vector<FrontArgs> fronts(n);
     std::vector<mie_terms_B> terms(n);
     std::vector<mie_sums_B> sums(n);
     std::vector<Mix2Args> mix(n);
     std::vector<ReduceArgs> red(n);
     std::vector<expand_coefs_B> coefs[2];
     std::vector<int2> task;
     std::vector<CopyJob> out(n);
     for (unsigned k = 0; k < n; ++k) {
          const FwdCase &c = *cs[k];
          const FwdPlan &p = c.p;
          Workspace *w = c.w;
          front_args(w, c.J, p, fronts[k]);
          term_args(w, c.J, p, terms[k].p);
          terms[k].gx = (unsigned) p.Np / 64;
          terms[k].gy = (unsigned) p.ng;
          sums[k] = mie_sums_B{w->chPart.as<double>(), p.N, p.Np, p.ng, w->n1.as<int>(), w->S.as<double>(),
                               w->CB.as<double>(), (unsigned) (p.Np + 31) / 32, 1};
          mix_args(w, p, mix[k]);
          mix[k].task = nullptr;
          for (const int2 &t : p.task)
               task.push_back(make_int2(t.x, ((t.x < 0 ? 0 : t.y) & 0xffff) | (int) (k << 16)));
          double *res = w->res.as<double>();
          const size_t nx = 6 * (size_t) p.C;
          reduce_args(w, p, res, red[k]);
          for (int gs = 0; gs < 2; ++gs) {
               const unsigned on = (gs ? c.J->calc_gc : c.J->calc_lc) ? 1u : 0u;
               coefs[gs].push_back(expand_coefs_B{w->T.as<double>(), w->pf.as<double>(), w->w.as<double>(), p.Q, p.Hp, p.C, gs,
                                                  res + 4 + (gs ? 0 : nx), (unsigned) (p.C + 7) / 8, on});
          }
          out[k] = CopyJob{res, (double *) w->pres.p, 4 + (c.J->calc_lc ? 2 * nx : nx)};
     }
     BatchBlob b;
     const size_t o_front = b.add(fronts), o_terms = b.add(terms), o_sums = b.add(sums),
                  o_mix = b.add(mix), o_task = b.add(task), o_red = b.add(red),
                  o_coefs0 = b.add(coefs[0]), o_coefs1 = b.add(coefs[1]), o_out = b.add(out);
     unsigned char *d;
     if (send_args(L, b.h, s, &d)) return -1;
#define LMIE_B(T, off) ((const T *) (d + (off)))
     hipLaunchKernelGGL((front_b<std::is_same<E, F16>::value ? 2 : 3>), dim3(max_g(fronts, &FrontArgs::e_ft), 1, n), dim3(64),
                        0, s, LMIE_B(FrontArgs, o_front));
     const unsigned tgy = max_g(terms, &mie_terms_B::gy);
     if (tgy > 0)
          hipLaunchKernelGGL(mie_terms_b<E>, dim3(max_g(terms, &mie_terms_B::gx), tgy, n), dim3(64), 0, s,
                             LMIE_B(mie_terms_B, o_terms));
     hipLaunchKernelGGL(mie_sums_b, dim3(max_g(sums, &mie_sums_B::gx), 1, n), dim3(256), 0, s,
                        LMIE_B(mie_sums_B, o_sums));
     // contraction, one task list for all cases
     if (!task.empty())
     {
          const dim3 g((unsigned) task.size());
          const int np = mix_products(), id = mix_shape().id;
#define LMIE_MIXB(NP, S) hipLaunchKernelGGL((angular_mix_b<E, NP, 1, S>), g, dim3(S::NT), 0, s, LMIE_B(Mix2Args, o_mix), LMIE_B(int2, o_task))
          if (id == 0) { if (np == 3) LMIE_MIXB(3, MixS0); else LMIE_MIXB(5, MixS0); }
          else if (id == 2) { if (np == 3) LMIE_MIXB(3, MixS2); else LMIE_MIXB(5, MixS2); }
          else if (id == 3) { if (np == 3) LMIE_MIXB(3, MixS3); else if (np == 4) LMIE_MIXB(4, MixS3); else LMIE_MIXB(5, MixS3); }
          else { if (np == 3) LMIE_MIXB(3, MixS1); else LMIE_MIXB(5, MixS1); }
#undef LMIE_MIXB
     }
     hipLaunchKernelGGL(reduce_channels_b, dim3(max_g(red, &ReduceArgs::gx), 1, n), dim3(256), 0, s,
                        LMIE_B(ReduceArgs, o_red));
     // expansion: generalized spherical, then Legendre
     for (int gs = 1; gs >= 0; --gs) {
          if (max_g(coefs[gs], &expand_coefs_B::gy) == 0) continue;
          hipLaunchKernelGGL(expand_coefs_b, dim3(max_g(coefs[gs], &expand_coefs_B::gx), 1, n), dim3(256), 0, s,
                             LMIE_B(expand_coefs_B, gs ? o_coefs1 : o_coefs0));
     }
     hipLaunchKernelGGL(copy_jobs, dim3(8, n), dim3(256), 0, s, LMIE_B(CopyJob, o_out));
#undef LMIE_B
     HIPCHECK(hipGetLastError());
     HIPCHECK(hipStreamSynchronize(s));
     for (FwdCase *c : cs) {
          keep_forward(c->w, c->J, c->p);
          c->w->valid = 1;
     }
     return 0;
}

struct RevCase {
     int slot;
     Workspace *w;
     const lmie_gpu_adj_in *in;
     lmie_gpu_adj_out *out;
     int use_gc, use_lc;
};

// (fused passes run the 128-size shape; a state whose forward ran alone with
// LMIE_UGEMM_WAVES=2 holds the tasks and depths of 64-size tiles)
int fused_reverse_ok(Workspace *w, const lmie_gpu_adj_in *in) {
     return w->valid && w->mixed && w->ushape != 2 && w->Q > 0 &&
            ((in->gc_bar && w->calc_gc) || (in->lc_bar && w->calc_lc));
}

// Buffers of one reverse pass (the mixed branch of adjoint_impl) and its
// cotangents in its pinned staging area.
int fused_rev_prepare(RevCase &c) {
     Workspace *w = c.w;
     c.use_gc = c.in->gc_bar && w->calc_gc;
     c.use_lc = c.in->lc_bar && w->calc_lc;
     if (alloc_reverse(w, true)) return -1;
     double *h = (double *) w->pin.p;
     const size_t n = 6 * (size_t) w->C;
     if (c.use_gc) memcpy(h, c.in->gc_bar, sizeof(double) * n);
     if (c.use_lc) memcpy(h + n, c.in->lc_bar, sizeof(double) * n);
     return 0;
}

template <class E>
int fused_rev_launch(std::vector<RevCase *> &cs, Workspace *L) {
     hipStream_t s = L->stream;
     const unsigned n = (unsigned) cs.size();
     std::vector<expand_adjoint_part_B> epart(n);
     std::vector<expand_adjoint_fin_B> efin(n);
     std::vector<adj_weights_B> wts(n);
     std::vector<adj_tables_B> tabs(n);
     std::vector<adj_gbuild_B> gb(n);
     std::vector<adj_gsplit_B> gsp(n);
     std::vector<UArgs> ua(n);
     std::vector<int2> task;
     std::vector<rev_orders_B> ro(n);
     std::vector<rev_carry_B> rc(n);
     std::vector<CopyJob> in(n), out(n);
     for (unsigned k = 0; k < n; ++k) {
          const RevCase &c = *cs[k];
          Workspace *w = c.w;
          const int H = w->H, Hp = w->Hp, Q = w->Q, C = w->C, Np = w->Np;
          const int Kq = rup(w->n1max, 64), Hq = rup(H, KM), nck = (C + EXA_L - 1) / EXA_L;
          const double *g = w->gbar.as<double>();
          AdjScal *sc = w->scal.as<AdjScal>();
          // cotangents from the case's pinned staging area, results into its
          // landing area
          const size_t o = c.use_gc ? 0 : 6 * (size_t) C;
          in[k] = CopyJob{(const double *) w->pin.p + o, w->gbar.as<double>() + o, (c.use_lc ? 12 * (size_t) C : 6 * (size_t) C) - o};
          out[k] = CopyJob{w->rres.as<double>(), (double *) w->pres.p, 2 * (size_t) w->N + Np / 32};
          epart[k] = expand_adjoint_part_B{w->T.as<double>(), c.use_gc ? g : nullptr, c.use_lc ? g + 6 * C : nullptr,
                                           H, Hp, C, w->expart.as<double>(), (unsigned) Hp / 64, (unsigned) nck};
          efin[k] = expand_adjoint_fin_B{w->expart.as<double>(), nck, w->w.as<double>(), H, Hp, Q,
                                         w->pfbar.as<double>(), (unsigned) (H + EXF_J - 1) / EXF_J, 1};
          wts[k] = adj_weights_B{w->pfbar.as<double>(), H, Hq, Q, w->wts.as<double>(), sc, 1, 1};
          tabs[k] = adj_tables_B{w->B16.as<unsigned short>(), w->Kb, w->Hb, w->wts.as<double>(), H, Hq, Kq,
                                 w->n1max, w->L16.as<unsigned short>(), w->R16.as<unsigned short>(),
                                 (unsigned) Kq / 64, (unsigned) Hq / 8};
          gb[k] = adj_gbuild_B{w->L16.as<unsigned short>(), w->R16.as<unsigned short>(), Hq, Kq,
                               w->Gf.as<float>(), sc, (unsigned) Kq / 64, (unsigned) Kq / 64};
          gsp[k] = adj_gsplit_B{w->Gf.as<float>(), sc, Kq, w->G16.as<unsigned short>(), (unsigned) Kq / 64,
                                (unsigned) Kq / 8};
          UArgs &u = ua[k];
          u.Np = Np; u.Kb = w->Kb; u.Kq = Kq;
          u.A16 = w->A16.as<unsigned short>(); u.G16 = w->G16.as<unsigned short>();
          u.ktile = w->ktile128.as<int>(); u.task = nullptr; u.sc = sc; u.Uf = w->Uf.as<float>();
          for (const int2 &t : w->rtask)
               task.push_back(make_int2(t.x, ((t.x < 0 ? 0 : t.y) & 0xffff) | (int) (k << 16)));
          RevArgs r;
          rev_args(w, c.in, c.out->x_bar != nullptr, true, r);
          ro[k] = rev_orders_B{r, (unsigned) Np / 64, (unsigned) r.nch};
          rc[k] = rev_carry_B{r, (unsigned) Np / 64, 1};
     }
     BatchBlob b;
     const size_t o_ep = b.add(epart), o_ef = b.add(efin), o_w = b.add(wts), o_t = b.add(tabs), o_gb = b.add(gb),
                  o_gs = b.add(gsp), o_u = b.add(ua), o_task = b.add(task), o_ro = b.add(ro), o_rc = b.add(rc),
                  o_in = b.add(in), o_out = b.add(out);
     unsigned char *d;
     if (send_args(L, b.h, s, &d)) return -1;
#define LMIE_B(T, off) ((const T *) (d + (off)))
     hipLaunchKernelGGL(copy_jobs, dim3(8, n), dim3(256), 0, s, LMIE_B(CopyJob, o_in));
     hipLaunchKernelGGL(expand_adjoint_part_b, dim3(max_g(epart, &expand_adjoint_part_B::gx),
                                                    max_g(epart, &expand_adjoint_part_B::gy), n),
                        dim3(64), 0, s, LMIE_B(expand_adjoint_part_B, o_ep));
     hipLaunchKernelGGL(expand_adjoint_fin_b, dim3(max_g(efin, &expand_adjoint_fin_B::gx), 1, n), dim3(24 * EXF_J), 0, s,
                        LMIE_B(expand_adjoint_fin_B, o_ef));
     hipLaunchKernelGGL(adj_weights_b, dim3(1, 1, n), dim3(1024), 0, s, LMIE_B(adj_weights_B, o_w));
     hipLaunchKernelGGL(adj_tables_b<E>, dim3(max_g(tabs, &adj_tables_B::gx), max_g(tabs, &adj_tables_B::gy), n),
                        dim3(64), 0, s, LMIE_B(adj_tables_B, o_t));
     hipLaunchKernelGGL(adj_gbuild_b<E>, dim3(max_g(gb, &adj_gbuild_B::gx), max_g(gb, &adj_gbuild_B::gy), n),
                        dim3(256), 0, s, LMIE_B(adj_gbuild_B, o_gb));
     hipLaunchKernelGGL(adj_gsplit_b<E>, dim3(max_g(gsp, &adj_gsplit_B::gx), max_g(gsp, &adj_gsplit_B::gy), n),
                        dim3(64), 0, s, LMIE_B(adj_gsplit_B, o_gs));
     if (!task.empty())
          hipLaunchKernelGGL((adj_ugemm32<E, 1, 128, true>), dim3((unsigned) task.size()), dim3(512), 0, s,
                             UArgs{}, LMIE_B(UArgs, o_u), LMIE_B(int2, o_task));
     const unsigned rgy = max_g(ro, &rev_orders_B::gy);
     if (rgy > 0)
          hipLaunchKernelGGL(rev_orders_b, dim3(max_g(ro, &rev_orders_B::gx), rgy, n), dim3(64), 0, s,
                             LMIE_B(rev_orders_B, o_ro));
     hipLaunchKernelGGL(rev_carry_b, dim3(max_g(rc, &rev_carry_B::gx), 1, n), dim3(64), 0, s,
                        LMIE_B(rev_carry_B, o_rc));
     hipLaunchKernelGGL(copy_jobs, dim3(8, n), dim3(256), 0, s, LMIE_B(CopyJob, o_out));
#undef LMIE_B
     HIPCHECK(hipGetLastError());
     HIPCHECK(hipStreamSynchronize(s));
     return 0;
}

// The collective: cases register their pass; the last to arrive (or to
// leave without arriving) runs it for all.
struct Batch {
     int n = 0, device = 0;
     pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
     pthread_cond_t cv = PTHREAD_COND_INITIALIZER;
     int arrived[2] = {0, 0}, left[2] = {0, 0}, state[2] = {0, 0};   // state: 0 open, 1 running, 2 done
     std::vector<char> in[2];
     std::vector<const lmie_gpu_job *> job;
     std::vector<lmie_gpu_result *> res;
     std::vector<Workspace *> ws;
     std::vector<const lmie_gpu_adj_in *> ain;
     std::vector<lmie_gpu_adj_out *> aout;
     std::vector<int> rc[2];
     std::vector<std::string> err[2];
     int fused_cases[2] = {0, 0};
     // forward cases prepared by their own threads before they arrive
     // (buffers, host tables and inputs), so the thread that runs the pass
     // only launches; a case takes its results out of its landing area itself
     std::vector<char> prepped, done[2];
     std::vector<FwdCase> pre;
     std::vector<int> prerc;
     std::vector<std::string> preerr;
     // the same for the reverse pass
     std::vector<char> rprepped;
     std::vector<RevCase> rpre;
     std::vector<int> rprerc;
     std::vector<std::string> rpreerr;
};

thread_local Batch *t_batch = nullptr;
thread_local int t_slot = -1, t_phase = 0;

int forward_one(const lmie_gpu_job *job, lmie_gpu_result *res);
int adjoint_one(Workspace *w, const lmie_gpu_adj_in *in, lmie_gpu_adj_out *out);

// A forward case of a fused batch prepared on its own thread, before it
// arrives: its workspace, host tables and staged uploads (fused_prepare).
void batch_prepare(Batch *b, int k, const lmie_gpu_job *J, lmie_gpu_result *res) {
     g_err[0] = 0;
     FwdCase &c = b->pre[k];
     c.slot = k; c.J = J; c.R = res; c.w = nullptr;
     int rc = use_device(J->device);
     if (rc == 0) rc = ws_acquire_home(J->device, k, &c.w);
     if (rc == 0) {
          // the case's inputs go up from here, on its own stream, one pinned
          // copy; the launch waits for the event
          rc = fused_prepare(c);
          if (rc == 0 && hipEventRecord(c.w->uploaded, c.w->stream) != hipSuccess)
               rc = set_err("hipEventRecord failed");
          if (rc) {
               (void) hipStreamSynchronize(c.w->stream);
               ws_release(c.w);
               c.w = nullptr;
          }
     }
     b->prerc[k] = rc;
     b->preerr[k] = rc ? g_err : "";
     b->prepped[k] = 1;
}

// A reverse case of a fused batch prepared on its own thread, before it
// arrives (fused_rev_prepare); the pass reads the cotangents from its pinned
// staging area.
void batch_rev_prepare(Batch *b, int k, Workspace *w, const lmie_gpu_adj_in *in, lmie_gpu_adj_out *out) {
     g_err[0] = 0;
     RevCase &c = b->rpre[k];
     c.slot = k; c.w = w; c.in = in; c.out = out;
     int rc = use_device(w->device);
     if (rc == 0) rc = fused_rev_prepare(c);
     b->rprerc[k] = rc;
     b->rpreerr[k] = rc ? g_err : "";
     b->rprepped[k] = 1;
}

void batch_run_forward(Batch *b) {
     std::vector<FwdCase *> f16, b16;
     Workspace *L = nullptr;           // the workspace whose stream launches the batch
     for (int k = 0; k < b->n; ++k) {
          if (!b->in[0][k]) continue;
          const lmie_gpu_job *J = b->job[k];
          g_err[0] = 0;
          int rc;
          if (b->prepped[k] && b->prerc[k]) {
               b->rc[0][k] = b->prerc[k];
               b->err[0][k] = b->preerr[k];
               continue;
          } else if (b->prepped[k] && J->device == b->device) {
               // its inputs are on the way on its own stream (batch_prepare)
               FwdCase &c = b->pre[k];
               if (!L) L = c.w;
               if (hipStreamWaitEvent(L->stream, c.w->uploaded, 0) != hipSuccess) {
                    (void) hipStreamSynchronize(c.w->stream);
                    if (c.w != L) ws_release(c.w);
                    b->rc[0][k] = set_err("hipStreamWaitEvent failed");
                    b->err[0][k] = g_err;
                    continue;
               }
               const bool bf = J->precision == LMIE_PRECISION_MIXED_BF16;
               (bf ? b16 : f16).push_back(&c);
               continue;
          }
          // another device's case, or one that the fused kernels do not cover
          if (b->prepped[k]) {
               (void) hipStreamSynchronize(b->pre[k].w->stream);
               ws_release(b->pre[k].w);
          }
          rc = forward_one(J, b->res[k]);
          b->rc[0][k] = rc;
          b->err[0][k] = rc ? g_err : "";
     }
     if (!L) return;
     bool L_kept = false;
     for (int t = 0; t < 2; ++t) {     // one arithmetic type per launch
          std::vector<FwdCase *> &v = t ? b16 : f16;
          if (v.empty()) continue;
          g_err[0] = 0;
          const int rc = t ? fused_launch<BF16>(v, L) : fused_launch<F16>(v, L);
          if (rc) (void) hipStreamSynchronize(L->stream);
          for (FwdCase *c : v) {
               b->rc[0][c->slot] = rc;
               b->err[0][c->slot] = rc ? g_err : "";
               b->done[0][c->slot] = rc == 0;
               c->R->state = rc ? nullptr : c->w;
               c->R->precision = c->J->precision;
               if (rc == 0 && c->w == L) L_kept = true;
               if (rc && c->w != L) ws_release(c->w);
               b->fused_cases[0]++;
          }
     }
     if (!L_kept) ws_release(L);
}

void batch_run_reverse(Batch *b) {
     std::vector<RevCase *> f16, b16;
     Workspace *L = nullptr;
     for (int k = 0; k < b->n; ++k) {
          if (!b->in[1][k]) continue;
          Workspace *w = b->ws[k];
          g_err[0] = 0;
          if (b->rprepped[k] && b->rprerc[k]) {
               b->rc[1][k] = b->rprerc[k];
               b->err[1][k] = b->rpreerr[k];
               continue;
          } else if (b->rprepped[k] && w->device == b->device) {
               if (!L) L = w;
               (w->bf16 ? b16 : f16).push_back(&b->rpre[k]);
               continue;
          }
          const int rc = adjoint_one(w, b->ain[k], b->aout[k]);
          b->rc[1][k] = rc;
          b->err[1][k] = rc ? g_err : "";
     }
     for (int t = 0; t < 2; ++t) {
          std::vector<RevCase *> &v = t ? b16 : f16;
          if (v.empty()) continue;
          g_err[0] = 0;
          const int rc = t ? fused_rev_launch<BF16>(v, L) : fused_rev_launch<F16>(v, L);
          if (rc) (void) hipStreamSynchronize(L->stream);
          for (RevCase *c : v) {
               b->rc[1][c->slot] = rc;
               b->err[1][c->slot] = rc ? g_err : "";
               b->done[1][c->slot] = rc == 0;
               b->fused_cases[1]++;
          }
     }
}

void batch_fire(Batch *b, int p) {   // with b->mu held; runs phase p if complete
     if (b->state[p] != 0 || b->arrived[p] + b->left[p] != b->n) return;
     if (b->arrived[p] == 0) {
          b->state[p] = 2;
          return;
     }
     b->state[p] = 1;
     pthread_mutex_unlock(&b->mu);
     (void) use_device(b->device);
     if (p == 0) batch_run_forward(b);
     else batch_run_reverse(b);
     pthread_mutex_lock(&b->mu);
     b->state[p] = 2;
     pthread_cond_broadcast(&b->cv);
}

int batch_arrive(int p, const lmie_gpu_job *job, lmie_gpu_result *res, Workspace *w, const lmie_gpu_adj_in *ain,
                 lmie_gpu_adj_out *aout) {
     Batch *b = t_batch;
     const int k = t_slot;
     // a fused case does its own preparation first, beside the others
     if (p == 0 && fused_forward_ok(job)) batch_prepare(b, k, job, res);
     if (p == 1 && fused_reverse_ok(w, ain)) batch_rev_prepare(b, k, w, ain, aout);
     pthread_mutex_lock(&b->mu);
     if (p == 0) {
          b->job[k] = job;
          b->res[k] = res;
          if (b->arrived[0] == 0) b->device = job->device;
     } else {
          b->ws[k] = w;
          b->ain[k] = ain;
          b->aout[k] = aout;
          if (b->arrived[1] == 0) b->device = w->device;
     }
     b->in[p][k] = 1;
     b->arrived[p]++;
     t_phase = p + 1;
     batch_fire(b, p);
     while (b->state[p] != 2) pthread_cond_wait(&b->cv, &b->mu);
     const int rc = b->rc[p][k], done = b->done[p][k];
     const std::string e = b->err[p][k];
     pthread_mutex_unlock(&b->mu);
     if (done && p == 0) fused_unpack(b->pre[k]);
     if (done && p == 1) unpack_reverse(w, (const double *) w->pres.p, aout);
     if (rc) return set_err("%s", e.c_str());
     return 0;
}

// Plain 16-byte-per-lane copy: the calibration point for HBM traffic counters
// (n16 elements of 16 bytes read and written once).
__global__ __launch_bounds__(256) void copy16(const v4u *src, v4u *dst, size_t n16) {
     for (size_t e = (size_t) blockIdx.x * blockDim.x + threadIdx.x; e < n16; e += (size_t) gridDim.x * blockDim.x)
          dst[e] = src[e];
}

// Lane-layout check of the FP64 matrix instruction used by the contraction:
// D = A (16x4) B (4x16), all row-major, one wave.
__global__ void mfma_f64_probe(const double *A, const double *B, double *D) {
     const int l = threadIdx.x;
     const double a = A[(l & 15) * 4 + (l >> 4)];
     const double b = B[(l >> 4) * 16 + (l & 15)];
     v4d c = {0., 0., 0., 0.};
     c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
     for (int v = 0; v < 4; ++v) D[((l >> 4) + 4 * v) * 16 + (l & 15)] = c[v];
}

// Lane-layout check of the 32x32x16 fp16 matrix instruction: D = A (32x16)
// B (16x32), row-major float inputs, one wave.  Operand lane l: row (column)
// l % 32, elements 8 (l / 32) .. +7 of the contraction; result lane l, value v:
// column l % 32, row given by mfma32_row (checked by lmie_gpu_selftest_mfma32).


__global__ void mfma32_probe(const float *A, const float *B, float *D) {
     const int l = threadIdx.x;
     unsigned short av[8], bv[8];
     double r;
     for (int e = 0; e < 8; ++e) {
          av[e] = F16::bits(A[(l & 31) * 16 + 8 * (l >> 5) + e], &r);
          bv[e] = F16::bits(B[(8 * (l >> 5) + e) * 32 + (l & 31)], &r);
     }
     v4u a, b;
     for (int k = 0; k < 4; ++k) {
          a[k] = (unsigned) av[2 * k] | ((unsigned) av[2 * k + 1] << 16);
          b[k] = (unsigned) bv[2 * k] | ((unsigned) bv[2 * k + 1] << 16);
     }
     v16f c;
     for (int v = 0; v < 16; ++v) c[v] = 0.f;
     c = F16::mfma32(a, b, c);
     for (int v = 0; v < 16; ++v) D[mfma32_row(l, v) * 32 + (l & 31)] = c[v];
}

// Lane-layout check of the 16-bit matrix instructions used by the mixed
// contraction: D = A (16x32) B (32x16), row-major float inputs (exactly
// representable in the 16-bit type), one wave.
template <class E>
__global__ void mfma16_probe(const float *A, const float *B, float *D) {
     const int l = threadIdx.x;
     unsigned short av[8], bv[8];
     double r;
     for (int e = 0; e < 8; ++e) {
          av[e] = E::bits(A[(l & 15) * 32 + 8 * (l >> 4) + e], &r);
          bv[e] = E::bits(B[(8 * (l >> 4) + e) * 16 + (l & 15)], &r);
     }
     v4u a, b;
     for (int k = 0; k < 4; ++k) {
          a[k] = (unsigned) av[2 * k] | ((unsigned) av[2 * k + 1] << 16);
          b[k] = (unsigned) bv[2 * k] | ((unsigned) bv[2 * k + 1] << 16);
     }
     v4f c = {0.f, 0.f, 0.f, 0.f};
     c = E::mfma(a, b, c);
     for (int v = 0; v < 4; ++v) D[mfma16_row(l, v) * 16 + (l & 15)] = c[v];
}

}  // namespace

extern "C" {

const char *lmie_gpu_last_error(void) { return g_err; }

int lmie_set_timing(int on) {
     g_timing = on ? 1 : 0;
     return 0;
}

void lmie_gpu_host_time(int k, double ms) {
     if (g_timing && k >= LMIE_T_HOST_GRID && k < LMIE_N_TIMERS) g_times[k] = ms;
}

void lmie_gpu_host_times_clear(void) {
     for (int k = LMIE_T_HOST_GRID; k < LMIE_N_TIMERS; ++k) g_times[k] = 0.;
}

int lmie_get_timing(double *ms, int n) {
     for (int k = 0; k < n && k < LMIE_N_TIMERS; ++k) ms[k] = g_times[k];
     return 0;
}

int lmie_gpu_forward(const lmie_gpu_job *job, lmie_gpu_result *res) {
     g_err[0] = 0;
     if (!job || !res) return set_err("null argument");
     if (t_batch && t_phase == 0) {
          res->state = nullptr;
          return batch_arrive(0, job, res, nullptr, nullptr, nullptr);
     }
     return forward_one(job, res);
}

int lmie_gpu_adjoint(void *state, const lmie_gpu_adj_in *in, lmie_gpu_adj_out *out) {
     g_err[0] = 0;
     if (!state || !in || !out || !in->sums_bar || !out->f_bar) return set_err("null argument");
     if (t_batch && t_phase == 1) return batch_arrive(1, nullptr, nullptr, (Workspace *) state, in, out);
     return adjoint_one((Workspace *) state, in, out);
}

void *lmie_gpu_batch_open(int n_case) {
     g_err[0] = 0;
     if (n_case < 1 || n_case > 32767) {
          set_err("batch of %d cases (1 .. 32767)", n_case);
          return nullptr;
     }
     Batch *b = new Batch();
     b->n = n_case;
     for (int p = 0; p < 2; ++p) {
          b->in[p].assign(n_case, 0);
          b->rc[p].assign(n_case, 0);
          b->err[p].assign(n_case, std::string());
     }
     b->job.assign(n_case, nullptr);
     b->res.assign(n_case, nullptr);
     b->ws.assign(n_case, nullptr);
     b->ain.assign(n_case, nullptr);
     b->aout.assign(n_case, nullptr);
     b->prepped.assign(n_case, 0);
     b->pre.resize(n_case);
     b->done[0].assign(n_case, 0);
     b->done[1].assign(n_case, 0);
     b->prerc.assign(n_case, 0);
     b->preerr.assign(n_case, std::string());
     b->rprepped.assign(n_case, 0);
     b->rpre.resize(n_case);
     b->rprerc.assign(n_case, 0);
     b->rpreerr.assign(n_case, std::string());
     return b;
}

int lmie_gpu_batch_enter(void *batch, int slot) {
     g_err[0] = 0;
     Batch *b = (Batch *) batch;
     if (!b || slot < 0 || slot >= b->n) return set_err("batch slot %d", slot);
     if (t_batch) return set_err("this thread is already in a batch");
     t_batch = b;
     t_slot = slot;
     t_phase = 0;
     return 0;
}

void lmie_gpu_batch_leave(void) {
     Batch *b = t_batch;
     if (!b) return;
     pthread_mutex_lock(&b->mu);
     for (int p = t_phase; p < 2; ++p) b->left[p]++;
     for (int p = 0; p < 2; ++p) batch_fire(b, p);
     pthread_mutex_unlock(&b->mu);
     t_batch = nullptr;
     t_slot = -1;
     t_phase = 0;
}

int lmie_gpu_batch_fused(void *batch, int pass) {
     Batch *b = (Batch *) batch;
     return b && pass >= 0 && pass < 2 ? b->fused_cases[pass] : 0;
}

void lmie_gpu_batch_close(void *batch) { delete (Batch *) batch; }
}

namespace {
int forward_one(const lmie_gpu_job *job, lmie_gpu_result *res) {
     if (job->precision != LMIE_PRECISION_FP64 && job->precision != LMIE_PRECISION_MIXED &&
         job->precision != LMIE_PRECISION_MIXED_BF16)
          return set_err("unknown precision %d", job->precision);
     if (job->save_control == 2 && job->keep) return set_err("save_control = 2 keeps no reverse-pass state");
     Workspace *w = nullptr;
     if (ws_acquire(job->device, &w)) return -1;
     res->state = nullptr;
     res->precision = LMIE_PRECISION_FP64;   /* the re-weighting of save_control 2 is FP64 */
     int rc = job->save_control == 2 ? saved_impl(job, res, w) : forward_impl(job, res, w);
     if (rc) {
          (void) hipStreamSynchronize(w->stream);
     }
     if (rc == 0 && job->keep) {
          res->state = w;          // owned by the caller until lmie_gpu_release
          return 0;
     }
     ws_release(w);
     return rc;
}

int adjoint_one(Workspace *w, const lmie_gpu_adj_in *in, lmie_gpu_adj_out *out) {
     if (use_device(w->device)) return -1;
     int rc = adjoint_impl(w, in, out);
     if (rc) (void) hipStreamSynchronize(w->stream);
     return rc;
}
}  // namespace

extern "C" {

void lmie_gpu_release(void *state) {
     if (state) ws_release((Workspace *) state);
}

// Coefficients (the n_coef columns in use) and angles go up as one pinned copy,
// the phase function comes back as one, on a pooled workspace.
static int phase_func_ws(Workspace *w, int n_set, int n_coef, int ld, const double *coefs, int n_theta, const double *theta,
                         double *pf, int gsf) {
     hipStream_t s = w->stream;
     const size_t rows = (size_t) n_set * 6, nx = rows * n_coef, np = rows * n_theta, in = nx + (size_t) n_theta;
     if (w->phIn.get(sizeof(double) * in) || w->pin.get(sizeof(double) * in) || w->phOut.get(sizeof(double) * np) ||
         w->pres.get(sizeof(double) * np))
          return -1;
     double *h = (double *) w->pin.p, *d = w->phIn.as<double>();
     for (size_t r = 0; r < rows; ++r) memcpy(h + r * n_coef, coefs + r * ld, sizeof(double) * n_coef);
     memcpy(h + nx, theta, sizeof(double) * n_theta);
     HIPCHECK(hipMemcpyAsync(d, h, sizeof(double) * in, hipMemcpyHostToDevice, s));
     if (launch_phase(n_set, n_coef, n_coef, d, n_theta, d + nx, w->phOut.as<double>(), gsf, s)) return -1;
     HIPCHECK(hipMemcpyAsync(w->pres.p, w->phOut.p, sizeof(double) * np, hipMemcpyDeviceToHost, s));
     HIPCHECK(hipStreamSynchronize(s));
     memcpy(pf, w->pres.p, sizeof(double) * np);
     return 0;
}

int lmie_gpu_phase_func(int n_set, int n_coef, int ld, const double *coefs, int n_theta, const double *theta,
                        double *pf, int gsf, int device) {
     g_err[0] = 0;
     if (n_set <= 0 || n_theta <= 0) return 0;
     if (n_coef > ld || n_coef < 0) return set_err("n_coef %d outside [0, %d]", n_coef, ld);
     Workspace *w = nullptr;
     if (ws_acquire(device, &w)) return -1;
     const int rc = phase_func_ws(w, n_set, n_coef, ld, coefs, n_theta, theta, pf, gsf);
     if (rc) (void) hipStreamSynchronize(w->stream);
     ws_release(w);
     return rc;
}

// Staging of lmie_gpu_phase_func_static: the coefficients, the angles and the
// phase function of one call, in one file-scope device array in place of the
// workspace buffers that lmie_gpu_phase_func grows as its calls do.  Every GPU the
// library runs on holds its own copy of the array (16 MiB) until the process
// ends.  In host code the name `scratch` is not a device address: the address
// of each device's copy is taken once (hipGetSymbolAddress, with that device
// current) and kept in pf_scratch[device]; only that address is passed on.
constexpr size_t PF_SCRATCH_DOUBLES = (size_t) 1 << 21;
constexpr int PF_MAX_DEVICES = 64;
static __device__ __align__(256) double scratch[PF_SCRATCH_DOUBLES];
static double *pf_scratch[PF_MAX_DEVICES];     // guarded by pf_lock[device]
static std::mutex pf_lock[PF_MAX_DEVICES];

static int phase_func_static_locked(int n_set, int n_coef, int ld, const double *coefs, int n_theta,
                                    const double *theta, double *pf, int gsf, int device, size_t ot, size_t op) {
     HIPCHECK(hipSetDevice(device));
     if (!pf_scratch[device]) {
          void *p = nullptr;
          HIPCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
          if (!p) return set_err("hipGetSymbolAddress gave no address for the phase-function scratch");
          pf_scratch[device] = (double *) p;
     }
     double *dX = pf_scratch[device], *dT = dX + ot, *dP = dX + op;
     const size_t nx = (size_t) n_set * 6 * ld, np = (size_t) n_set * 6 * n_theta;
     if (nx) HIPCHECK(hipMemcpy(dX, coefs, sizeof(double) * nx, hipMemcpyHostToDevice));
     HIPCHECK(hipMemcpy(dT, theta, sizeof(double) * n_theta, hipMemcpyHostToDevice));
     if (launch_phase(n_set, n_coef, ld, dX, n_theta, dT, dP, gsf, nullptr)) return -1;
     HIPCHECK(hipMemcpy(pf, dP, sizeof(double) * np, hipMemcpyDeviceToHost));
     return 0;
}

int lmie_gpu_phase_func_static(int n_set, int n_coef, int ld, const double *coefs, int n_theta,
                               const double *theta, double *pf, int gsf, int device) {
     g_err[0] = 0;
     if (n_set <= 0 || n_theta <= 0) return 0;
     if (n_coef > ld || n_coef < 0) return set_err("n_coef %d outside [0, %d]", n_coef, ld);
     if (device < 0 || device >= PF_MAX_DEVICES)
          return set_err("device %d outside [0, %d)", device, PF_MAX_DEVICES);
     // layout in the array (doubles): coefficients at 0, angles at ot, phase
     // function at op, each start a multiple of 32 (256 bytes); every factor
     // is bounded first so that the products cannot wrap
     const size_t cap = PF_SCRATCH_DOUBLES;
     if ((size_t) n_set > cap || (size_t) ld > cap || (size_t) n_theta > cap)
          return set_err("lmie_gpu_phase_func_static: n_set %d, ld %d, n_theta %d exceed its static scratch of %zu doubles",
                         n_set, ld, n_theta, cap);
     const size_t nx = (size_t) n_set * 6 * ld, np = (size_t) n_set * 6 * n_theta;
     const size_t ot = (nx + 31) / 32 * 32, op = (ot + (size_t) n_theta + 31) / 32 * 32;
     if (op + np > cap)
          return set_err("lmie_gpu_phase_func_static: %zu doubles of staging (coefficients %zu, angles %d, "
                         "phase function %zu) exceed its static scratch of %zu doubles",
                         op + np, nx, n_theta, np, cap);
     std::lock_guard<std::mutex> hold(pf_lock[device]);
     return phase_func_static_locked(n_set, n_coef, ld, coefs, n_theta, theta, pf, gsf, device, ot, op);
}

int lmie_gpu_gauss_rule(int n, double *x, double *wt, int device) {
     if (n < 1) return set_err("n < 1");
     HIPCHECK(hipSetDevice(device));
     std::vector<double> g((n + 1) / 2);
     gauss_guesses(n, g.data());
     double *d = nullptr;
     HIPCHECK(hipMalloc(&d, sizeof(double) * (g.size() + 2 * (size_t) n)));
     HIPCHECK(hipMemcpy(d, g.data(), sizeof(double) * g.size(), hipMemcpyHostToDevice));
     FrontArgs fa;
     memset(&fa, 0, sizeof fa);
     fa.Q = n; fa.guess = d; fa.mu = d + g.size(); fa.w = d + g.size() + n;
     fa.plan(0, 0, true, 0, false);
     if (launch_front(fa, 0, false, nullptr)) return -1;
     HIPCHECK(hipMemcpy(x, d + g.size(), sizeof(double) * n, hipMemcpyDeviceToHost));
     HIPCHECK(hipMemcpy(wt, d + g.size() + n, sizeof(double) * n, hipMemcpyDeviceToHost));
     HIPCHECK(hipFree(d));
     return 0;
}

int lmie_gpu_gsf_table(int n_mu, const double *mu, int n_l, double *out, int device) {
     if (n_mu < 1 || n_l < 1) return set_err("n_mu < 1 or n_l < 1");
     if (!mu || !out) return set_err("missing argument");
     HIPCHECK(hipSetDevice(device));
     // the expansion tables' role reads the angles at mu[H + j], j < H, and writes 5 planes of rows of two l
     const int H = n_mu, Hp = rup(H, 64);
     const size_t pl = gsf_plane(n_l, Hp), tab = 5 * pl;
     double *d = nullptr;
     HIPCHECK(hipMalloc(&d, sizeof(double) * (2 * (size_t) H + tab)));
     HIPCHECK(hipMemcpy(d + H, mu, sizeof(double) * H, hipMemcpyHostToDevice));
     FrontArgs fa;
     memset(&fa, 0, sizeof fa);
     fa.H = H; fa.Hp = Hp; fa.C = n_l; fa.mu = d; fa.T = d + 2 * H;
     fa.plan(5, 0, false, 0, false);
     if (launch_front(fa, 0, false, nullptr)) return -1;
     std::vector<double> t(tab);
     HIPCHECK(hipMemcpy(t.data(), d + 2 * H, sizeof(double) * tab, hipMemcpyDeviceToHost));
     HIPCHECK(hipFree(d));
     for (int q = 0; q < 5; ++q)
          for (int l = 0; l < n_l; ++l)
               for (int j = 0; j < H; ++j)
                    out[((size_t) q * n_l + l) * H + j] = t[q * pl + ((size_t) (l / 2) * Hp + j) * 2 + (l & 1)];
     return 0;
}

int lmie_gpu_pitau_table(int n_mu, const double *mu, int n, double *bp, double *bm, int device) {
     if (n_mu < 1 || n < 1) return set_err("n_mu < 1 or n < 1");
     if (!mu || !bp || !bm) return set_err("missing argument");
     HIPCHECK(hipSetDevice(device));
     // the pi/tau tables' role reads the angles at mu[H + j], j < H, and writes [n][Hp] twice
     const int H = n_mu, Hp = rup(H, 64);
     const size_t tab = (size_t) n * Hp;
     double *d = nullptr;
     HIPCHECK(hipMalloc(&d, sizeof(double) * (2 * (size_t) H + 2 * tab)));
     HIPCHECK(hipMemcpy(d + H, mu, sizeof(double) * H, hipMemcpyHostToDevice));
     FrontArgs fa;
     memset(&fa, 0, sizeof fa);
     fa.H = H; fa.Hp = Hp; fa.n1max = fa.Kp = n; fa.mu = d; fa.Bp = d + 2 * H; fa.Bm = d + 2 * H + tab;
     fa.plan(0, 1, false, 0, false);
     if (launch_front(fa, 1, false, nullptr)) return -1;
     std::vector<double> t(2 * tab);
     HIPCHECK(hipMemcpy(t.data(), d + 2 * H, sizeof(double) * 2 * tab, hipMemcpyDeviceToHost));
     HIPCHECK(hipFree(d));
     for (size_t r = 0; r < (size_t) n; ++r) {
          memcpy(bp + r * H, t.data() + r * Hp, sizeof(double) * H);
          memcpy(bm + r * H, t.data() + tab + r * Hp, sizeof(double) * H);
     }
     return 0;
}

int lmie_gpu_selftest_mfma16(int bf16, const float *A, const float *B, float *D, int device) {
     HIPCHECK(hipSetDevice(device));
     float *d = nullptr;
     HIPCHECK(hipMalloc(&d, sizeof(float) * (512 + 512 + 256)));
     HIPCHECK(hipMemcpy(d, A, sizeof(float) * 512, hipMemcpyHostToDevice));
     HIPCHECK(hipMemcpy(d + 512, B, sizeof(float) * 512, hipMemcpyHostToDevice));
     if (bf16)
          hipLaunchKernelGGL(mfma16_probe<BF16>, dim3(1), dim3(64), 0, 0, (const float *) d, (const float *) (d + 512), d + 1024);
     else
          hipLaunchKernelGGL(mfma16_probe<F16>, dim3(1), dim3(64), 0, 0, (const float *) d, (const float *) (d + 512), d + 1024);
     HIPCHECK(hipGetLastError());
     HIPCHECK(hipMemcpy(D, d + 1024, sizeof(float) * 256, hipMemcpyDeviceToHost));
     HIPCHECK(hipFree(d));
     return 0;
}

// Copies n_bytes (a multiple of 16) device to device `reps` times with copy16
// and returns the average kernel time in ms through *ms.
int lmie_gpu_selftest_copy(size_t n_bytes, int reps, int device, double *ms) {
     if (n_bytes == 0 || n_bytes % 16 || reps < 1) return set_err("copy size must be a positive multiple of 16");
     HIPCHECK(hipSetDevice(device));
     void *a = nullptr, *b = nullptr;
     hipEvent_t e0, e1;
     HIPCHECK(hipMalloc(&a, n_bytes));
     HIPCHECK(hipMalloc(&b, n_bytes));
     HIPCHECK(hipMemset(a, 1, n_bytes));
     HIPCHECK(hipEventCreate(&e0));
     HIPCHECK(hipEventCreate(&e1));
     const size_t n16 = n_bytes / 16;
     HIPCHECK(hipEventRecord(e0, 0));
     for (int r = 0; r < reps; ++r)
          hipLaunchKernelGGL(copy16, dim3(2048), dim3(256), 0, 0, (const v4u *) a, (v4u *) b, n16);
     HIPCHECK(hipGetLastError());
     HIPCHECK(hipEventRecord(e1, 0));
     HIPCHECK(hipEventSynchronize(e1));
     float t = 0.f;
     HIPCHECK(hipEventElapsedTime(&t, e0, e1));
     if (ms) *ms = t / reps;
     (void) hipEventDestroy(e0);
     (void) hipEventDestroy(e1);
     HIPCHECK(hipFree(a));
     HIPCHECK(hipFree(b));
     return 0;
}

int lmie_gpu_selftest_mfma32(const float *A, const float *B, float *D, int device) {
     HIPCHECK(hipSetDevice(device));
     float *d = nullptr;
     HIPCHECK(hipMalloc(&d, sizeof(float) * (512 + 512 + 1024)));
     HIPCHECK(hipMemcpy(d, A, sizeof(float) * 512, hipMemcpyHostToDevice));
     HIPCHECK(hipMemcpy(d + 512, B, sizeof(float) * 512, hipMemcpyHostToDevice));
     hipLaunchKernelGGL(mfma32_probe, dim3(1), dim3(64), 0, 0, (const float *) d, (const float *) (d + 512), d + 1024);
     HIPCHECK(hipGetLastError());
     HIPCHECK(hipMemcpy(D, d + 1024, sizeof(float) * 1024, hipMemcpyDeviceToHost));
     HIPCHECK(hipFree(d));
     return 0;
}

int lmie_gpu_selftest_mfma_f64(const double *A, const double *B, double *D, int device) {
     HIPCHECK(hipSetDevice(device));
     double *d = nullptr;
     HIPCHECK(hipMalloc(&d, sizeof(double) * (64 + 64 + 256)));
     HIPCHECK(hipMemcpy(d, A, sizeof(double) * 64, hipMemcpyHostToDevice));
     HIPCHECK(hipMemcpy(d + 64, B, sizeof(double) * 64, hipMemcpyHostToDevice));
     hipLaunchKernelGGL(mfma_f64_probe, dim3(1), dim3(64), 0, 0, (const double *) d, (const double *) (d + 64), d + 128);
     HIPCHECK(hipGetLastError());
     HIPCHECK(hipMemcpy(D, d + 128, sizeof(double) * 256, hipMemcpyDeviceToHost));
     HIPCHECK(hipFree(d));
     return 0;
}

}  // extern "C"
