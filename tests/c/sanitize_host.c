/* sanitize_host.c - the host C code under AddressSanitizer and UndefinedBehaviorSanitizer
 * (tests/test_sanitize.py builds it with tests/c/Makefile's sanitize_host target): the
 * product's parameter clamps and sample.h layer (qs_params.c, qs_sampler.c, over
 * stub_device.c: no device, so every pick takes the reference's out-of-memory answer) and
 * the CPU restatement (oracle/orc_*.c) through each of its branches.  Exits 0 when every
 * check holds; a sanitizer report aborts it. */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "quasar_sampler.h"
#include "../../oracle/orc_sampler.h"

extern int stub_allocs;
static int fails;
#define CHECK(c) do { if (!(c)) { fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); fails++; } } while (0)

static uint64_t st = 88172645463325252ull;
static float frand(void) {
    st ^= st << 13; st ^= st >> 7; st ^= st << 17;
    return (float)((double)(st >> 11) / 9007199254740992.0) * 8.0f - 4.0f;
}

static void fill(float *x, int n) {
    for (int i = 0; i < n; i++) x[i] = frand();
}

/* the product's host layer: clamps, history mirror, argmax answer, state read-back */
static void product(void) {
    enum { V = 3001 };
    float *x = malloc(sizeof(float) * V);
    int32_t hist[16];
    uint64_t rng = 0;
    int len = -1;
    quasar_sampler *s = quasar_sampler_new();
    CHECK(s != NULL);
    fill(x, V);
    (void)quasar_sampler_pick(s, x, V);
    CHECK(stub_allocs == 1);                 /* the row of logits and nothing else */
    for (int round = 0; round < 3; round++) {
        quasar_sampler_config(s, 0.8f, 0.9f, 40 * round, 0.05f, 1.3f, 4 + round, 77u + round);
        for (int t = 0; t < 9; t++) {
            fill(x, V);
            if (t == 3) x[0] = NAN;
            if (t == 5) x[V - 1] = INFINITY;
            int bi = 0;
            for (int i = 1; i < V; i++) if (x[i] > x[bi]) bi = i;
            CHECK(quasar_sampler_pick(s, x, V) == bi);
        }
        CHECK(qs_sampler_get_state(s, &rng, hist, 16, &len) == 0);
        CHECK(len == 4 + round && rng == 77u + (uint64_t)round);
        quasar_sampler_reset(s);
        CHECK(qs_sampler_get_state(s, &rng, hist, 16, &len) == 0 && len == 0);
        CHECK(quasar_sampler_pick(s, x, 0) == 0);
    }
    quasar_sampler_config(s, 0.0f, 1.0f, 0, 0.0f, 1.0f, 0, 5u);   /* keeps the ring */
    CHECK(quasar_sampler_pick(s, x, 17) >= 0);
    CHECK(qs_sampler_get_state(s, &rng, hist, 1, &len) == 0 && len == 1);
    CHECK(qs_sampler_get_state(NULL, &rng, hist, 1, &len) == QS_EINVAL);
    CHECK(qs_debug_fail_picks(-1) == QS_EINVAL);
    quasar_sampler_free(s);
    quasar_sampler_free(NULL);
    free(x);
}

/* the restatement: every branch of sample.c:111-179 on small rows */
static void restatement(void) {
    enum { V = 700 };
    float *x = malloc(sizeof(float) * V);
    orc_diag d;
    orc_sampler *s = orc_sampler_new();
    const float cfg[][6] = {{0.0f, 1, 0, 0, 1, 0}, {0.7f, 0.9f, 40, 0.05f, 1.1f, 8},
                            {1.0f, 1, 0, 0, 1, 3}, {2.0f, 0.5f, 0, 0.2f, 1.5f, 700},
                            {0.3f, 0.99f, 700, 0, 1, 1}};
    for (size_t c = 0; c < sizeof cfg / sizeof cfg[0]; c++) {
        orc_sampler_config(s, cfg[c][0], cfg[c][1], (int)cfg[c][2], cfg[c][3], cfg[c][4],
                           (int)cfg[c][5], 1000u + c);
        for (int t = 0; t < 12; t++) {
            fill(x, V);
            if (t == 2) for (int i = 0; i < V; i++) x[i] = 1.0f;       /* all equal */
            if (t == 4) x[7] = NAN;
            if (t == 6) x[3] = -INFINITY;
            if (t == 8) { x[11] = INFINITY; x[12] = INFINITY; }
            const int id = orc_sampler_pick_diag(s, x, V - (t % 3), &d);
            CHECK(id >= 0 && id < V);
        }
        orc_sampler_fail_scratch(s, 1);
        CHECK(orc_sampler_pick(s, x, V) >= 0);
        orc_sampler_fail_scratch(s, 0);
        orc_sampler_reset(s);
    }
    int32_t ids[4] = {1, 2, 699, 0}, back[8];
    orc_sampler_set_history(s, ids, 4);
    CHECK(orc_sampler_get_history(s, back, 8) == 1);          /* capacity 1 */
    orc_sampler_free(s);
    /* the threaded row driver */
    enum { R = 6 };
    float *rows = malloc(sizeof(float) * R * V);
    fill(rows, R * V);
    int32_t out[R], hist2[R * 3];
    uint64_t seeds[R];
    orc_diag dg[R];
    for (int r = 0; r < R; r++) { seeds[r] = 5u + r; for (int k = 0; k < 3; k++) hist2[r * 3 + k] = r + k; }
    orc_params p = {0.8f, 0.95f, 0.05f, 1.1f, 40, 3};
    CHECK(orc_pick_rows_diag(&p, rows, V, R, V, hist2, 3, seeds, out, dg, 3) >= 0.0);
    for (int r = 0; r < R; r++) CHECK(out[r] == dg[r].id);
    free(rows);
    free(x);
}

int main(void) {
    product();
    restatement();
    if (fails) { fprintf(stderr, "%d checks failed\n", fails); return 1; }
    printf("sanitize_host: all checks passed\n");
    return 0;
}
