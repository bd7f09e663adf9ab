/*
 * tangent_quad.c -- the per-size Mie coefficients and their derivatives in
 * 113-bit arithmetic, from the recurrences themselves: D_j downward from
 * D_{n2} = 0, psi_j = sin x U_j / U_0 with U_{n1} = 0, U_{n1-1} = 1 downward,
 * chi_j upward (src/lmie_core.c:298-405), each differentiated step by step
 * along x and m with n1 and n2 held.
 *
 *   tangent_quad check   the arithmetic of the kernels' size chains
 *                        (lmie_amd/csrc/lmie_gpu.hip, mie_chain_psi, and the psi'
 *                        of mie_tan_terms) in double against it: psi_j and psi'_j.
 *   tangent_quad         per line "x mr mi n1 n2" of stdin, the series sums ext,
 *                        sca, |bak|^2, asym (src/lmie_core.c:537-596), their
 *                        derivatives along x, mr and mi (16 values), for each the
 *                        sum of the magnitudes of its terms (16), and the same 16
 *                        values by the reference's recurrences in double: the
 *                        ratios r_j and their derivatives downward, psi_j = r_j
 *                        psi_{j-1} from sin x.
 */
#include <complex.h>
#include <math.h>
#include <quadmath.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef __float128 q;
typedef __complex128 cq;
#define QI 1.0iQ

static q mag(cq a) { return cabsq(a); }
static q re(cq a) { return crealq(a); }

typedef struct { q *ps, *dps, *ch, *dch; } chains;

static void free_chains(chains c) { free(c.ps); free(c.dps); free(c.ch); free(c.dch); }

static chains quad_chains(double xd, int n1) {
     const q x = xd, sx = sinq(x), cx = cosq(x);
     chains c;
     q *U = calloc(n1 + 2, sizeof *U), *V = calloc(n1 + 2, sizeof *V);     /* U and U' */
     c.ps = calloc(n1 + 2, sizeof(q)); c.dps = calloc(n1 + 2, sizeof(q));
     c.ch = calloc(n1 + 2, sizeof(q)); c.dch = calloc(n1 + 2, sizeof(q));
     U[n1 - 1] = 1;
     for (int j = n1 - 1; j >= 1; --j) {
          const q f = (2 * j + 1) / x;
          U[j - 1] = f * U[j] - U[j + 1];
          V[j - 1] = f * V[j] - f / x * U[j] - V[j + 1];
     }
     const q s = sx / U[0], ds = (cx - s * V[0]) / U[0];
     c.ch[0] = cx; c.dch[0] = -sx;
     c.ch[1] = cx / x + sx; c.dch[1] = -cx / (x * x) - sx / x + cx;
     for (int j = 1; j <= n1; ++j) {
          const q f = (2 * j + 1) / x;
          c.ch[j + 1] = f * c.ch[j] - c.ch[j - 1];
          c.dch[j + 1] = f * c.dch[j] - f / x * c.ch[j] - c.dch[j - 1];
     }
     for (int j = 0; j <= n1; ++j) {
          c.ps[j] = s * U[j];
          c.dps[j] = ds * U[j] + s * V[j];
     }
     free(U); free(V);
     return c;
}

/* ------------------------------------------------------------------------- */
static void ratio_sums(double x, double mr, double mi, int n1, int n2);

static int sums(double xd, double mr, double mi, int n1, int n2) {
     if (n1 < 1 || n2 < n1 || !(xd > 0.)) return 1;
     const q x = xd;
     const cq m = (q) mr - (q) mi * QI, z = m * x;
     cq *D = calloc(n2 + 1, sizeof *D), *Dx = calloc(n2 + 1, sizeof *Dx), *Dm = calloc(n2 + 1, sizeof *Dm);
     for (int j = n2 - 1; j >= 1; --j) {
          const cq c = (j + 1) / z, w = D[j + 1] + c, cx = -c / z * m, cm = -c / z * x;
          D[j] = c - 1 / w;
          Dx[j] = cx + (Dx[j + 1] + cx) / (w * w);
          Dm[j] = cm + (Dm[j + 1] + cm) / (w * w);
     }
     const chains c = quad_chains(xd, n1);
     /* index 0 the value, 1 along x, 2 along mr, 3 along mi */
     q E[4] = {0}, S[4] = {0}, G[4] = {0}, eE[4] = {0}, eS[4] = {0}, eG[4] = {0}, eB[4] = {0};
     cq B[4] = {0}, ap[4] = {0}, bp[4] = {0};
     for (int j = 1; j <= n1; ++j) {
          const cq zj = c.ps[j] + c.ch[j] * QI, zm = c.ps[j - 1] + c.ch[j - 1] * QI;
          const cq dz = c.dps[j] + c.dch[j] * QI, dzm = c.dps[j - 1] + c.dch[j - 1] * QI;
          const cq u = D[j] / m + j / x, v = m * D[j] + j / x;
          const cq ux = Dx[j] / m - j / (x * x), vx = m * Dx[j] - j / (x * x);
          const cq um = Dm[j] / m - D[j] / (m * m), vm = D[j] + m * Dm[j];
          const cq da = u * zj - zm, db = v * zj - zm;
          cq a[4], b[4];
          a[0] = (u * c.ps[j] - c.ps[j - 1]) / da;
          b[0] = (v * c.ps[j] - c.ps[j - 1]) / db;
          a[1] = (ux * c.ps[j] + u * c.dps[j] - c.dps[j - 1] - a[0] * (ux * zj + u * dz - dzm)) / da;
          b[1] = (vx * c.ps[j] + v * c.dps[j] - c.dps[j - 1] - b[0] * (vx * zj + v * dz - dzm)) / db;
          a[2] = um * (c.ps[j] - a[0] * zj) / da;
          b[2] = vm * (c.ps[j] - b[0] * zj) / db;
          a[3] = -QI * a[2];            /* m = mr - i mi */
          b[3] = -QI * b[2];
          const q f1 = 2 * j + 1, f3 = j > 1 ? (q) (j - 1) * (j + 1) / j : 0, f4 = j > 1 ? (2 * j - 1) / ((q) (j - 1) * j) : 0;
          for (int d = 0; d < 4; ++d) {
               E[d] += f1 * re(a[d] + b[d]);
               eE[d] += f1 * (mag(a[d]) + mag(b[d]));
               B[d] += (j & 1 ? -f1 : f1) * (a[d] - b[d]);
               eB[d] += f1 * (mag(a[d]) + mag(b[d]));
               const q t = d ? 2 : 1;
               S[d] += t * f1 * re(conjq(a[0]) * a[d] + conjq(b[0]) * b[d]);
               eS[d] += t * f1 * (mag(a[0]) * mag(a[d]) + mag(b[0]) * mag(b[d]));
               const cq ga = conjq(ap[d]) * a[0] + (d ? conjq(ap[0]) * a[d] : 0), gb = conjq(bp[d]) * b[0] + (d ? conjq(bp[0]) * b[d] : 0);
               const cq gc = conjq(ap[d]) * bp[0] + (d ? conjq(ap[0]) * bp[d] : 0);
               G[d] += f3 * re(ga + gb) + f4 * re(gc);
               eG[d] += f3 * (mag(ap[d]) * mag(a[0]) + mag(ap[0]) * mag(a[d]) + mag(bp[d]) * mag(b[0]) + mag(bp[0]) * mag(b[d])) +
                        f4 * (mag(ap[d]) * mag(bp[0]) + mag(ap[0]) * mag(bp[d]));
          }
          memcpy(ap, a, sizeof a);
          memcpy(bp, b, sizeof b);
     }
     for (int d = 0; d < 4; ++d)
          printf("%.17g %.17g %.17g %.17g ", (double) E[d], (double) S[d],
                 (double) (d ? 2 * re(conjq(B[0]) * B[d]) : re(conjq(B[0]) * B[0])), (double) G[d]);
     for (int d = 0; d < 4; ++d)
          printf("%.6g %.6g %.6g %.6g ", (double) eE[d], (double) eS[d],
                 (double) (d ? 2 * (mag(B[0]) * eB[d] + eB[0] * mag(B[d])) : 2 * mag(B[0]) * eB[0]), (double) eG[d]);
     ratio_sums(xd, mr, mi, n1, n2);
     printf("\n");
     free(D); free(Dx); free(Dm);
     free_chains(c);
     return 0;
}

/* ------------------------------------------------------------------------- */
typedef double _Complex cd;

static void ratio_sums(double x, double mr, double mi, int n1, int n2) {
     const cd m = mr - I * mi, z = m * x;
     cd *D = calloc(n2 + 1, sizeof *D), *Dx = calloc(n2 + 1, sizeof *Dx), *Dm = calloc(n2 + 1, sizeof *Dm);
     double *r = calloc(n1 + 2, sizeof *r), *dr = calloc(n1 + 2, sizeof *dr);
     for (int j = n2 - 1; j >= 1; --j) {
          const cd c = (j + 1.) / z, w = D[j + 1] + c, c5 = -c / z * m, c6 = -c / z * x;
          D[j] = c - 1. / w;
          Dx[j] = c5 + (Dx[j + 1] + c5) / (w * w);
          Dm[j] = c6 + (Dm[j + 1] + c6) / (w * w);
     }
     for (int j = n1 - 1; j >= 1; --j) {
          const double c = (2. * j + 1.) / x, v = 1. / (c - r[j + 1]);
          dr[j] = -(-c / x - dr[j + 1]) * (v * v);
          r[j] = v;
     }
     const double sx = sin(x), cx = cos(x), ax = 1. / x;
     double ps0 = sx, ch0 = cx, ch1 = ax * cx + sx, dps0 = cx, dch0 = -sx, dch1 = -ax / x * cx + ax * dch0 + cx;
     double E[4] = {0}, S[4] = {0}, G[4] = {0};
     cd B[4] = {0}, ap[4] = {0}, bp[4] = {0};
     for (int j = 1; j <= n1; ++j) {
          const double ps = r[j] * ps0, dps = dr[j] * ps0 + r[j] * dps0, jx = j / x, djx = -jx / x;
          const cd zj = ps + I * ch1, zm = ps0 + I * ch0, dz = dps + I * dch1, dzm = dps0 + I * dch0;
          const cd u = D[j] / m + jx, v = m * D[j] + jx;
          const cd na = u * ps - ps0, da = u * zj - zm, nb = v * ps - ps0, db = v * zj - zm;
          const cd du = Dx[j] / m + djx, dv = m * Dx[j] + djx;
          const cd um = Dm[j] / m - D[j] / (m * m), vm = D[j] + m * Dm[j];
          cd a[4], b[4];
          a[0] = na / da;
          b[0] = nb / db;
          a[1] = (du * ps + u * dps - dps0) / da - na * (du * zj + u * dz - dzm) / (da * da);
          b[1] = (dv * ps + v * dps - dps0) / db - nb * (dv * zj + v * dz - dzm) / (db * db);
          a[2] = um * ps / da - na * (um * zj) / (da * da);
          b[2] = vm * ps / db - nb * (vm * zj) / (db * db);
          a[3] = -I * a[2];
          b[3] = -I * b[2];
          const double f1 = 2. * j + 1., f3 = j > 1 ? (j - 1.) * (j + 1.) / j : 0., f4 = j > 1 ? (2. * j - 1.) / ((j - 1.) * j) : 0.;
          for (int d = 0; d < 4; ++d) {
               E[d] += f1 * creal(a[d] + b[d]);
               S[d] += (d ? 2. : 1.) * f1 * creal(conj(a[0]) * a[d] + conj(b[0]) * b[d]);
               B[d] += (j & 1 ? -f1 : f1) * (a[d] - b[d]);
               G[d] += f3 * creal(conj(ap[d]) * a[0] + conj(bp[d]) * b[0]) + f4 * creal(conj(ap[d]) * bp[0]);
               if (d) G[d] += f3 * creal(conj(ap[0]) * a[d] + conj(bp[0]) * b[d]) + f4 * creal(conj(ap[0]) * bp[d]);
          }
          memcpy(ap, a, sizeof a);
          memcpy(bp, b, sizeof b);
          const double c = (2. * j + 1.) / x, dch2 = -c / x * ch1 + c * dch1 - dch0, ch2 = c * ch1 - ch0;
          dch0 = dch1; dch1 = dch2; ch0 = ch1; ch1 = ch2; dps0 = dps; ps0 = ps;
     }
     for (int d = 0; d < 4; ++d)
          printf("%.17g %.17g %.17g %.17g ", E[d], S[d], (d ? 2. : 1.) * creal(conj(B[0]) * B[d]), G[d]);
     free(D); free(Dx); free(Dm); free(r); free(dr);
}

/* ------------------------------------------------------------------------- */
static double f_over_x(double f, double hi, double lo) { return fma(f, hi, f * lo); }

/* The kernels' arithmetic against the quad chains: the largest errors of psi_j
   and psi'_j, j = 1 .. n1, over the largest |psi|, |psi'|. */
static void kernel_chains(double x, int n1, double *e0, double *e1) {
     const chains c = quad_chains(x, n1);
     double *U = calloc(n1 + 2, sizeof *U), *X = calloc(n1 + 2, sizeof *X);
     const double hi = 1. / x, lo = fma(-x, hi, 1.) * hi, sx = sin(x), cx = cos(x);
     U[n1 - 1] = 1.;
     for (int j = n1 - 1; j >= 1; --j) U[j - 1] = f_over_x(2. * j + 1., hi, lo) * U[j] - U[j + 1];
     X[0] = cx;
     X[1] = hi * cx + sx;
     for (int j = 1; j < n1; ++j) X[j + 1] = f_over_x(2. * j + 1., hi, lo) * X[j] - X[j - 1];
     const double s = sx / U[0], qf = -s / X[n1], pf = (cx - sx * hi + s * U[1] - qf * cx) / sx;
     double m0 = 0., m1 = 0.;
     *e0 = *e1 = 0.;
     for (int j = 1; j <= n1; ++j) {
          const double ps = s * U[j], dps = s * U[j - 1] - j * hi * ps + (pf * ps + qf * X[j]);
          m0 = fmax(m0, fabs((double) c.ps[j]));
          m1 = fmax(m1, fabs((double) c.dps[j]));
          *e0 = fmax(*e0, (double) fabsq(ps - c.ps[j]));
          *e1 = fmax(*e1, (double) fabsq(dps - c.dps[j]));
     }
     *e0 /= m0;
     *e1 /= m1;
     free(U); free(X);
     free_chains(c);
}

/* Each of the n1 steps rounds its quotient, product and difference, at most two
   ulp together, of random sign: 2 sqrt(n1) ulp one standard deviation, eps four of
   them.  psi_0 = sin x sets the scale of psi and psi'_0 = cos x that of psi', so past
   x = 1 the relative errors of U_0 and U_1 come in divided by |sin x| and sin^2 x.
   (1/x rounded once breaks the bound away from and near x = k pi.) */
static int check(void) {
     const double k[] = {0, 1, 2, 5, 30, 100, 300, 588}, d[] = {.8, -.3, 1e-2, -1e-4, 1e-6};
     const double small[] = {1e-3, 0.02, 0.3, .7, .9};
     int fails = 0;
     for (int a = 0; a < 8; ++a)
          for (int b = 0; b < 5; ++b)
               for (int t = 0; t < 5; ++t) {
                    const double x = k[a] ? (k[a] + t) * M_PI + d[b] * (1. + .01 * t) : small[t] * (1. + .02 * b);
                    const int n1 = (int) (x + 4.05 * pow(x, 1. / 3.) + 8);
                    double e0, e1;
                    kernel_chains(x, n1, &e0, &e1);
                    const double eps = 8. * sqrt(n1) * 2.3e-16, is = x > 1. ? 1. / fabs(sin(x)) : 1.;
                    if (!(e0 <= eps * is && e1 <= eps * is * is)) {
                         printf("x %.17g n1 %d: psi %.2e of %.2e, psi' %.2e of %.2e\n", x, n1, e0, eps * is, e1, eps * is * is);
                         fails = 1;
                    }
               }
     if (!fails) printf("tangent arithmetic: ok\n");
     return fails;
}

int main(int argc, char **argv) {
     if (argc > 1 && strcmp(argv[1], "check") == 0) return check();
     double x, mr, mi;
     int n1, n2;
     while (scanf("%lf %lf %lf %d %d", &x, &mr, &mi, &n1, &n2) == 5)
          if (sums(x, mr, mi, n1, n2)) return 1;
     return 0;
}
