/*
 * alloc_checks.c -- the host C layer (lmie_amd/csrc/lmie_host.c compiled with
 * -Dmalloc=test_malloc -Dcalloc=test_calloc and linked with the device test double
 * tests/c/gpu_double.c) when a large block cannot be had: for k = 1, 2, ... the k-th allocation of 64 KiB
 * or more of a call fails, in a process of its own.  The call returns -1 with an
 * error text and leaves nothing behind, or its results are those of a call
 * without the failure; a call after it succeeds.
 * Prints "allocation checks: ok" and returns 0 when every check passes.
 */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include <sys/wait.h>
#include <unistd.h>

#include "lmie_hip.h"
#include "lmie_interface.h"

#define LARGE ((size_t) 65536)
static int fail_at, n_large;       /* atomic: the host layer allocates on its helper thread too */

static int refused(size_t n) {
     return n >= LARGE && __atomic_add_fetch(&n_large, 1, __ATOMIC_RELAXED) == __atomic_load_n(&fail_at, __ATOMIC_RELAXED);
}
void *test_malloc(size_t n) { return refused(n) ? NULL : malloc(n); }
void *test_calloc(size_t n, size_t m) { return refused(n * m) ? NULL : calloc(n, m); }

/* 16384 sizes, 1484 coefficients: every per-size and per-coefficient block is large */
static void make_in(lmie_in_data *in, int dist) {
     memset(in, 0, sizeof *in);
     in->calc_gc = 1; in->calc_lc = 1;
     in->dist_type = dist;
     in->n_int1 = 1; in->n_int2 = 64; in->n_quad = 256;
     in->lambda = 0.63; in->mr = 1.5; in->mi = 0.01;
     in->a1 = 0.3; in->a2 = 0.2; in->r1 = 0.02; in->r2 = 70.; in->accuracy = -1.;
}

static int cot(const lmie_out_data *out, lmie_adj_in *adj, void *user) {
     (void) user;
     adj->cext = 1.;
     adj->gc = out->gc[0];
     return 0;
}

#define N_RES 32
/* kind 0: forward with four tangents; 1, 2: gradient of one mode, of two */
static int call(int kind, double *res) {
     lmie_in_data in[2];
     lmie_in_data *pin[2] = {&in[0], &in[1]};
     lmie_out_data out;
     memset(&out, 0, sizeof out);
     memset(res, 0, N_RES * sizeof *res);
     make_in(&in[0], SIZE_DIST_LOG_NORMAL);
     make_in(&in[1], SIZE_DIST_GAMMA);
     int rc;
     if (kind == 0) {
          if (lmie_in_alloc(&in[0], 4)) return 2;
          lmie_in_zero_derivs(&in[0], 4);
          in[0].n_derivs = 4;
          in[0].mr_l[0] = in[0].a1_l[1] = in[0].r2_l[2] = in[0].lambda_l[3] = 1.;
          rc = lmie_solution(&in[0], &out, 1, 0, 1, 0);
          if (rc == 0) {
               res[0] = out.cext; res[1] = out.reff; res[2] = out.gc[0][1]; res[3] = out.lc[5][700];
               for (int d = 0; d < 4; ++d) {
                    res[4 + 4 * d] = out.cext_l[d]; res[5 + 4 * d] = out.reff_l[d];
                    res[6 + 4 * d] = out.norm_l[d]; res[7 + 4 * d] = out.gc_l[d][1][3];
               }
          }
          lmie_out_free(&out, 1);
          lmie_in_free(&in[0], 1);
     } else {
          lmie_grad g;
          memset(&g, 0, sizeof g);
          rc = lmie_solution_adjoint(pin, NULL, kind, &out, 1, NULL, cot, NULL, &g, res + 10);
          if (rc == 0) {
               const double v[10] = {g.lambda, g.mr, g.mi, g.a1, g.a2, g.a3, g.a4, g.a5, g.r1, g.r2};
               memcpy(res, v, sizeof v);
          }
          lmie_out_free(&out, 0);     /* (a failed reverse pass leaves the outputs to the caller) */
     }
     return rc;
}

/* the k-th large allocation refused: 0 ok, 3 ok and the call made fewer, else a fault */
static int child(int kind, int k, const double *ref) {
     double res[N_RES];
     fail_at = k;
     const int rc = call(kind, res);
     const int made = n_large;
     fail_at = 0;
     if (rc == 0 && memcmp(res, ref, sizeof res)) {
          printf("kind %d, allocation %d refused: success with other results\n", kind, k);
          return 1;
     }
     if (rc != 0 && (rc != -1 || !lmie_last_error()[0])) {
          printf("kind %d, allocation %d refused: returned %d without an error text\n", kind, k, rc);
          return 1;
     }
     if (call(kind, res) != 0 || memcmp(res, ref, sizeof res)) {
          printf("kind %d, allocation %d refused: the next call fails or differs\n", kind, k);
          return 1;
     }
     return made < k ? 3 : 0;
}

int main(void) {
     double (*ref)[N_RES] = mmap(NULL, 4096, PROT_READ | PROT_WRITE, MAP_SHARED | MAP_ANONYMOUS, -1, 0);
     if (ref == MAP_FAILED) return 1;
     int bad = 0;
     for (int kind = 0; kind < 3; ++kind) {
          for (int k = 0; k < 500; ++k) {
               fflush(stdout);
               const pid_t pid = fork();
               if (pid < 0) return 1;
               if (pid == 0) exit(k == 0 ? call(kind, ref[kind]) : child(kind, k, ref[kind]));
               int st = 0;
               waitpid(pid, &st, 0);
               if (!WIFEXITED(st)) {
                    printf("kind %d, allocation %d refused: signal %d\n", kind, k, WTERMSIG(st));
                    ++bad;
               } else if (WEXITSTATUS(st) == 3) break;
               else if (WEXITSTATUS(st)) {
                    if (WEXITSTATUS(st) != 1) printf("kind %d, allocation %d refused: exit status %d\n", kind, k, WEXITSTATUS(st));
                    ++bad;
               }
          }
          double s = 0.;
          for (int q = 0; q < N_RES; ++q) s += fabs(ref[kind][q]);
          if (!(s > 0.)) return 1;
     }
     if (!bad) printf("allocation checks: ok\n");
     return bad != 0;
}
