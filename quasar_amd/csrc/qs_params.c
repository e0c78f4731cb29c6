/* qs_params.c - parameter clamps and the error channel (C host code). */
#define _POSIX_C_SOURCE 200809L
#include <stdarg.h>
#include <stdio.h>
#include <string.h>
#include <time.h>

#include "../../include/quasar_sampler.h"
#include "qs_internal.h"

#define QS_DEFAULT_RNG 0x9E3779B97F4A7C15ull

void qs_default_param(qs_row_param *out, uint64_t *rng_out) {
    memset(out, 0, sizeof *out);
    out->temperature = 0.0f;
    out->top_p = 1.0f;
    out->top_k = 0;
    out->min_p = 0.0f;
    out->repeat_penalty = 1.0f;
    out->ring_cap = 0;
    out->inv_t = 0.0f;
    *rng_out = QS_DEFAULT_RNG;
}

void qs_clamp_config(float temperature, float top_p, int top_k, float min_p,
                     float repeat_penalty, int repeat_last_n, uint64_t seed, int prev_cap,
                     qs_row_param *out, uint64_t *rng_out) {
    memset(out, 0, sizeof *out);
    out->temperature = temperature;
    out->top_p = (top_p > 0.0f && top_p < 1.0f) ? top_p : 1.0f;
    out->top_k = top_k > 0 ? top_k : 0;
    out->min_p = min_p > 0.0f ? min_p : 0.0f;
    out->repeat_penalty = repeat_penalty > 1.0f ? repeat_penalty : 1.0f;
    out->ring_cap = repeat_last_n > 0 ? repeat_last_n : prev_cap;
    /* Used whenever the row samples, i.e. unless temperature <= 0 (a NaN temperature
     * samples, as in sample.c:130); the same float division sample.c:137 does per pick.
     * volatile keeps it a run-time IEEE division. */
    volatile float t = temperature;
    out->inv_t = temperature <= 0.0f ? 0.0f : 1.0f / t;
    if (seed == 0) seed = (uint64_t)time(NULL) * 2654435761u + 0x1234567u;
    *rng_out = seed ? seed : QS_DEFAULT_RNG;
}

static int qs_fail_left;   /* injected pick failures (qs_debug_fail_picks) */

int qs_debug_fail_picks(int n) {
    if (n < 0) return QS_EINVAL;
    __atomic_store_n(&qs_fail_left, n, __ATOMIC_RELAXED);
    return 0;
}

static int qs_open_fail_left;   /* injected failures of k_open's launch */

int qs_debug_fail_open_launches(int n) {
    if (n < 0) { qs_set_error("qs_debug_fail_open_launches: n %d", n); return QS_EINVAL; }
    __atomic_store_n(&qs_open_fail_left, n, __ATOMIC_RELAXED);
    return 0;
}

int qs_debug_take_open_failure(void) {
    int left = __atomic_load_n(&qs_open_fail_left, __ATOMIC_RELAXED);
    while (left > 0)
        if (__atomic_compare_exchange_n(&qs_open_fail_left, &left, left - 1, 0,
                                        __ATOMIC_RELAXED, __ATOMIC_RELAXED))
            return 1;
    return 0;
}

int qs_debug_take_failure(void) {
    int v = __atomic_load_n(&qs_fail_left, __ATOMIC_RELAXED);
    while (v > 0) {
        if (__atomic_compare_exchange_n(&qs_fail_left, &v, v - 1, 0, __ATOMIC_RELAXED,
                                        __ATOMIC_RELAXED)) {
            qs_set_error("injected device failure");
            return 1;
        }
    }
    return 0;
}

static _Thread_local char qs_err[512];

void qs_set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(qs_err, sizeof qs_err, fmt, ap);
    va_end(ap);
}

const char *qs_last_error(void) { return qs_err; }
