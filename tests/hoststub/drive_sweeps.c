/*
 * drive_sweeps.c -- TEST INFRASTRUCTURE: relax-6 calls on one-level
 * hierarchies through a solver's own layouts (dev_sweeps.c carries the launches
 * out) against the recurrence on the matrix.  Exit status 0 = all agree.
 *   drive_sweeps n rowlen symmetric zero_every
 */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "jxamd.h"
#include "jxamd_dev.h"

extern void (*jxamd_stub_relax)(int done, int xt, int n, int ncalls, const void *f, int fs, const void *uo, void *un);

static jxamd_csr A;
static double *ref;   /* the reference result of the launch under way */
static double worst;  /* largest error against it, relative to its largest entry */
static int exact, chunked; /* launches */
static unsigned long long state = 88172645463325252ull;

static double uniform(void)
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return (double)(state >> 11) / 9007199254740992.0;
}
static double at(const void *p, int xt, size_t i)
{
    return xt == JXAMD_T_F64 ? ((const double *)p)[i] : (double)((const float *)p)[i];
}

/* relax-6 calls (ncalls > 0: exact; else one call on -ncalls chunks) on ref */
static void relax(int ncalls, const void *f, int fs, int xt)
{
    const int n = A.n, T = ncalls > 0 ? 1 : -ncalls, size = n / T, rest = n - size * T;
    double *old = (double *)malloc(sizeof(double) * (size_t)n);
    for (int call = 0; call < (ncalls > 0 ? ncalls : 1); call++) {
        memcpy(old, ref, sizeof(double) * (size_t)n);
        for (int c = 0; c < T; c++) {
            const int ns = c < rest ? c * (size + 1) : c * size + rest, len = c < rest ? size + 1 : size;
            for (int k = 0; k < 2 * len; k++) {
                const int i = ns + (k < len ? k : 2 * len - 1 - k);
                double s = at(f, xt, (size_t)i * fs);
                if (A.a[A.ia[i]] == 0.0) continue;
                for (int q = A.ia[i] + 1; q < A.ia[i + 1]; q++) {
                    const int j = A.ja[q];
                    s -= A.a[q] * (j >= ns && j < ns + len ? ref[j] : old[j]);
                }
                ref[i] = s / A.a[A.ia[i]];
            }
        }
    }
    free(old);
}

static void hook(int done, int xt, int n, int ncalls, const void *f, int fs, const void *uo, void *un)
{
    if (!done) {
        for (int i = 0; i < n; i++) {
            const double v = uniform() - 0.5;
            if (xt == JXAMD_T_F64) ((double *)f)[(size_t)i * fs] = v;
            else ((float *)f)[(size_t)i * fs] = (float)v;
            ref[i] = uo ? uniform() - 0.5 : 0.0;
            if (uo && xt == JXAMD_T_F64) ((double *)uo)[i] = ref[i];
            else if (uo) ((float *)uo)[i] = (float)ref[i];
        }
        relax(ncalls, f, fs, xt);
        return;
    }
    double err = 0.0, top = 0.0;
    for (int i = 0; i < n; i++) {
        err = fmax(err, fabs(at(un, xt, i) - ref[i]));
        top = fmax(top, fabs(ref[i]));
    }
    if (ncalls > 0) exact++;
    else chunked++;
    worst = fmax(worst, err / top / (xt == JXAMD_T_F64 ? 1e-16 : 6e-8));
}

static int less(const void *a, const void *b) { return *(const int *)a - *(const int *)b; }

int main(int argc, char **argv)
{
    if (argc < 5) return 2;
    const int n = atoi(argv[1]), half = atoi(argv[2]) / 2, sym = atoi(argv[3]), zero = atoi(argv[4]);
    /* each row's distinct columns, a random pattern near the diagonal */
    int *cnt = (int *)calloc((size_t)n, sizeof(int)), **cols = (int **)calloc((size_t)n, sizeof(int *));
    for (int i = 0; i < n; i++) cols[i] = (int *)malloc(sizeof(int) * (size_t)(8 * half + 64));
    for (int i = 0; i < n; i++)
        for (int k = 0; k < half; k++) {
            const int j = i + (int)((uniform() - 0.5) * (6 * half + 8));
            if (j < 0 || j >= n || j == i) continue;
            if (cnt[i] < 8 * half + 64) cols[i][cnt[i]++] = j;
            if (sym && cnt[j] < 8 * half + 64) cols[j][cnt[j]++] = i;
            else if (sym) cnt[i]--;
        }
    long nnz = n;
    int longest = 0;
    for (int i = 0; i < n; i++) {
        int m = 0;
        qsort(cols[i], (size_t)cnt[i], sizeof(int), less);
        for (int k = 0; k < cnt[i]; k++)
            if (!m || cols[i][k] != cols[i][m - 1]) cols[i][m++] = cols[i][k];
        nnz += cnt[i] = m;
        if (m > longest) longest = m;
    }
    int *ia = (int *)malloc(sizeof(int) * ((size_t)n + 1)), *ja = (int *)malloc(sizeof(int) * (size_t)nnz);
    double *a = (double *)malloc(sizeof(double) * (size_t)nnz);
    ia[0] = 0;
    for (int i = 0; i < n; i++) {
        double sum = 0.5;
        int q = ia[i];
        ja[q++] = i;
        for (int k = cnt[i] - 1; k >= 0; k--) { /* behind the diagonal in any order */
            ja[q] = cols[i][k];
            a[q] = -0.1 - uniform();
            sum -= 1.1 * a[q++];
        }
        a[ia[i]] = zero && i % zero == 1 ? 0.0 : sum;
        ia[i + 1] = q;
        free(cols[i]);
    }
    free(cols);
    free(cnt);
    A = (jxamd_csr){n, n, ia[n], ia, ja, a};
    ref = (double *)malloc(sizeof(double) * (size_t)n);
    /* identity 2x2 blocks around it */
    int *bi = (int *)malloc(sizeof(int) * ((size_t)n + 1)), *bj = (int *)malloc(sizeof(int) * (size_t)n);
    double *ba = (double *)calloc(4 * (size_t)n, sizeof(double)), *r = (double *)calloc(2 * (size_t)n, sizeof(double));
    double *x = (double *)calloc(2 * (size_t)n, sizeof(double));
    for (int i = 0; i <= n; i++) bi[i] = i;
    for (int i = 0; i < n; i++) {
        bj[i] = i;
        ba[4 * i] = ba[4 * i + 3] = 1.0;
    }
    jxamd_bsr B = {n, n, n, 2, bi, bj, ba};
    jxamd_hierarchy H;
    memset(&H, 0, sizeof(H));
    H.num_levels = 1;
    H.A[0] = A;
    jxamd_stub_relax = hook;
    const int chunks[] = {0, 1, 2, 3, 4, 7, 8};
    int rc = 0;
    for (int c = 0; c < 7 && !rc; c++)
        for (int prec = 0; prec < 2 && !rc; prec++) {
            jxamd_params p;
            jxamd_params_default(&p);
            p.relax_chunk = chunks[c];
            p.precond_precision = prec;
            p.stage2_maxit = 0;
            jxamd_solver *s = NULL;
            rc = jxamd_solver_create(&s, &B, &H, &p);
            if (!rc) rc = jxamd_cpr_precond_device(s, r, x); /* from a zero guess, f strided in FP64 */
            if (!rc) rc = jxamd_solver_profile(s, 1);
            const int e0 = exact;
            if (!rc) rc = jxamd_op_hsgs(s, 0, r, x);         /* from u */
            if (!rc && exact > e0) {
                /* the bytes it is priced at: forward, backward, and the sums
                 * over the upper couplings before */
                const double xsz = prec ? 4.0 : 8.0;
                double ms, bytes = 0.0, want = 9.0 * xsz * n;
                long count = 0;
                for (int i = 0; i < n; i++)
                    for (int k = ia[i] + 1; k < ia[i + 1]; k++) want += (ja[k] < i ? 1.0 : 2.0) * (xsz + 4.0);
                rc = jxamd_solver_profile_read(s, JXAMD_PROF_GS_SWEEP, &count, &ms, &bytes);
                if (!rc && (count != 1 || bytes != want)) {
                    fprintf(stderr, "exact sweep priced at %.0f bytes in %ld launches, not %.0f\n", bytes, count, want);
                    rc = 10;
                }
            }
            if (s) jxamd_solver_destroy(s);
        }
    free(ia); free(ja); free(a); free(ref); free(bi); free(bj); free(ba); free(r); free(x);
    /* a row's new value is off by at most a rounding per entry and one per
     * entry's storage, and by 1 / 1.1 of its neighbours' errors */
    const double most = 11.0 * (2.0 * longest + 8.0);
    printf("rc %d exact %d chunked %d worst error %.1f of %.0f roundings\n", rc, exact, chunked, worst, most);
    return rc || worst > most ? 1 : 0;
}
