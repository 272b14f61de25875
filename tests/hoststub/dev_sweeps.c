/*
 * dev_sweeps.c -- TEST INFRASTRUCTURE: the relax-6 launches whose layouts only
 * the host knows how to build, carried out on the host: the schedules and
 * records of the one-workgroup sweeps, and the blocks of the chunked sweeps
 * from a zero guess, are walked entry by entry as the kernels walk them, the
 * reads ahead and past the last row included, so AddressSanitizer sees each.
 * What no layout may hold (a row left out or taken twice, a value read in the
 * step that writes it, a padding entry that is not zero) ends the program.
 */
#include <stdio.h>
#include <stdlib.h>

#include "jxamd_dev.h"

/* set by a driver: called with the launch's operands before it and after it */
void (*jxamd_stub_relax)(int done, int xt, int n, int ncalls, const void *f, int fs, const void *uo, void *un);

static void need(int ok, const char *what)
{
    if (ok) return;
    fprintf(stderr, "relax-6 layout: %s\n", what);
    exit(9);
}
static double get(const void *p, int xt, size_t i)
{
    return xt == JXAMD_T_F64 ? ((const double *)p)[i] : (double)((const float *)p)[i];
}
static void put(void *p, int xt, size_t i, double v)
{
    if (xt == JXAMD_T_F64) ((double *)p)[i] = v;
    else ((float *)p)[i] = (float)v;
}
static double rnd(int xt, double v) { return xt == JXAMD_T_F64 ? v : (double)(float)v; }

int jxamd_gs_lds_rows(int xt) { return 160 * 1024 / (xt == JXAMD_T_F64 ? 8 : 4) - 1; }

typedef struct { size_t i; double x; } store;

/* one pass over a direction's steps, x in the rows' order: the sweep from
 * g = f less the sum over the other couplings, or (g NULL) only the sums over
 * the direction's own; h: f less these */
static void pass(int G, int U, int W, int xt, int n, const jxamd_lds_sweep *sw, const void *diag, const void *fo,
                 const void *g, void *h, double *x, int keep)
{
    const int R = 64 / G, xsz = xt == JXAMD_T_F64 ? 8 : 4, E = 16 / xsz;
    double *acc = (double *)calloc((size_t)W * 64, sizeof(double));
    store *st = (store *)malloc(sizeof(store) * (size_t)W * 64);
    int *wrote = (int *)malloc(sizeof(int) * (size_t)n), rows = 0;
    volatile double sink = 0.0;
    for (int i = 0; i < n; i++) wrote[i] = -1;
    need(sw->steps % JXAMD_LDS_DEPTH == 0, "steps in whole rounds");
    /* the steps of padding behind the last are read ahead */
    for (int t = 0; t < sw->steps + 2 * JXAMD_LDS_DEPTH; t++) {
        int ns = 0;
        for (int w = 0; w < W; w++) {
            const int *q = sw->sched + 2 * ((size_t)t * W + w);
            const int e = q[0], b = e & JXAMD_LDS_ROW, cnt = JXAMD_LDS_COUNT(e);
            const size_t rec = (size_t)q[1];
            need(t < sw->steps || (e == 0 && rec == 0), "steps past the last are padding");
            need(cnt <= R && b + cnt <= n, "a slice's rows");
            for (int r = 0; r < R; r++) /* a wavefront's rows of the vectors, those past the slice too */
                sink += get(fo, xt, (size_t)b + r) + get(diag, xt, 2 * ((size_t)b + r) + 1) +
                        (g ? get(g, xt, (size_t)b + r) : 0.0);
            for (int lane = 0; lane < 64; lane++) {
                double *a = acc + (size_t)w * 64 + lane;
                if (!(e & JXAMD_LDS_CONT)) *a = 0.0;
                for (int u = 0; u < U; u++) {
                    const unsigned c = sw->col[((rec * (U / 4) + u / 4) * 64 + lane) * 4 + u % 4];
                    const double v = get(sw->val, xt, ((rec * (U / E) + u / E) * 64 + lane) * E + u % E);
                    const size_t j = c / xsz;
                    need(c % xsz == 0 && j <= (size_t)n, "a column");
                    if (j == (size_t)n) need(v == 0.0, "a padding entry");
                    else if (g) need(wrote[j] != t, "a value read in the step that writes it");
                    *a = rnd(xt, *a + v * x[j]);
                }
            }
            for (int r = 0; r < cnt && (e & JXAMD_LDS_LAST); r++) {
                const size_t i = (size_t)b + r;
                double s = 0.0;
                for (int k = 0; k < G; k++) s = rnd(xt, s + acc[(size_t)w * 64 + r * G + k]);
                need(wrote[i] < 0, "a row taken twice");
                wrote[i] = t;
                rows++;
                const double d = get(diag, xt, 2 * i);
                if (g && d != 0.0) {
                    st[ns].i = i;
                    st[ns++].x = rnd(xt, rnd(xt, get(g, xt, i) - s) / d);
                }
                if (!g || keep) put(h, xt, i, get(fo, xt, i) - s);
            }
        }
        for (int k = 0; k < ns; k++) x[st[k].i] = st[k].x;
    }
    need(rows == n, "a row left out");
    (void)sink;
    free(acc);
    free(st);
    free(wrote);
}

int jxamd_k_gs_lds(int G, int U, int waves, int xt, int n, const jxamd_lds_sweep *fw, const jxamd_lds_sweep *bw,
                   const int *order, const void *diag, int ncalls, const void *f, int fs, const void *uo, void *un,
                   void *work, void *stream)
{
    (void)stream;
    need((U == 4 || U == 8) && G >= 1 && G <= 16 && waves >= 1 && waves <= JXAMD_LDS_WAVES(U, xt), "G, U, waves");
    need(n >= 1 && n <= jxamd_gs_lds_rows(xt), "rows");
    if (jxamd_stub_relax) jxamd_stub_relax(0, xt, n, ncalls, f, fs, uo, un);
    void *fo = work, *h = (char *)work + (xt == JXAMD_T_F64 ? 8 : 4) * ((size_t)n + JXAMD_LDS_PAD);
    double *x = (double *)calloc((size_t)n + 1, sizeof(double));
    for (int q = 0; q < n; q++) {
        put(fo, xt, q, get(f, xt, (size_t)order[q] * fs));
        x[q] = uo ? get(uo, xt, order[q]) : 0.0;
    }
    /* the last of the padding that may be read */
    put(h, xt, (size_t)n + JXAMD_LDS_PAD - 1, 0.0);
    if (uo) pass(G, U, waves, xt, n, bw, diag, fo, NULL, h, x, 1);
    for (int q = 0; q < 2 * ncalls; q++)
        pass(G, U, waves, xt, n, q & 1 ? bw : fw, diag, fo, q > 0 || uo ? h : fo, h, x, q + 1 < 2 * ncalls);
    for (int q = 0; q < n; q++) put(un, xt, order[q], x[q]);
    free(x);
    if (jxamd_stub_relax) jxamd_stub_relax(1, xt, n, ncalls, f, fs, uo, un);
    return 0;
}

int jxamd_k_gs_chunk_zero(int L, int xt, int n, int nchunks, const void *blk, const void *diag, const void *f, int fs,
                          void *un, void *stream)
{
    (void)stream;
    need(L == 2 || L == 4 || L == 8, "rows of a block");
    need(nchunks >= 1 && jxamd_gs_chunk_lds_rows(n, nchunks) <= L, "chunks fit their blocks");
    if (jxamd_stub_relax) jxamd_stub_relax(0, xt, n, -nchunks, f, fs, NULL, un);
    const int size = n / nchunks, rest = n - size * nchunks, NE = L * (L - 1);
    for (int c = 0; c < nchunks; c++) {
        const int ns = c < rest ? c * (size + 1) : c * size + rest, len = c < rest ? size + 1 : size;
        double B[8 * 7], u[8] = {0};
        for (int e = 0; e < NE; e++) B[e] = get(blk, xt, ((size_t)(c / 64) * NE + e) * 64 + c % 64);
        for (int k = 0; k < 2 * len; k++) {
            const int t = k < len ? k : 2 * len - 1 - k;
            const double d = get(diag, xt, (size_t)ns + t);
            double x = get(f, xt, ((size_t)ns + t) * fs);
            if (d == 0.0) continue;
            for (int q = 0; q < len; q++)
                if (q != t) x = rnd(xt, x - B[t * (L - 1) + (q < t ? q : q - 1)] * u[q]);
            u[t] = rnd(xt, x / d);
        }
        for (int t = 0; t < len; t++) put(un, xt, (size_t)ns + t, u[t]);
    }
    if (jxamd_stub_relax) jxamd_stub_relax(1, xt, n, -nchunks, f, fs, NULL, un);
    return 0;
}
