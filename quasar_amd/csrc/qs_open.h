// qs_open.h - the whole-window decision of rows without a top-k, spread over workgroups
// (device code, included by qs_part.hip; sample.c:136-178 where the kept prefix may be the
// whole 30-nat window).
//
// A flat row keeps tens of thousands of ids, and sorting and adding them one after another
// in one workgroup (full_row) takes 12 to 19 ms at 151,936 logits: a chain of dependent
// binary64 additions and eight radix passes by four wavefronts.  Neither is needed.  The
// pick is one id: the first, in (p desc, id asc) order, whose running sum reaches r = u *
// rsum, and the top-p cut the first whose running sum reaches top_p.  Both are found by
// selection, in two passes over the row split into parts of OP logits:
//
//   sums (open_sum): each part's exact numerators e (the host-libm-equal expf), their
//     binary64 sum, and a histogram of their mass over ONB bins of the scaled logit.
//   select (k_open): inv from the parts' sums; from the histogram the few bins that hold
//     the top-p cut and the drawn position; each part then adds up p = fl(e * inv) above
//     those bins and lists the (p, id) inside them.  The row's last part to finish finds
//     the two positions in the lists.
//
// Both passes serve the rows that the decision kernel leaves undecided.  In picks of few rows
// the sums are taken by workgroups of that kernel past its row decisions, beside them and for
// every row without a top-k (the chip is otherwise idle).  In larger picks that would hold up
// rows that need none: there the decision kernel queues its undecided rows, and a launch of its
// own (k_open_sum), then k_open, take the queue's.  Rows that were decided cost these launches
// one load a workgroup.
//
// Why it is the reference's result.  inv is proved to be the reference's float (inv_settled).
// Every p is the reference's float.  Any order of adding n nonnegative binary64 numbers
// lies within (n - 1) 2^-53 (relative) of their exact sum, so the reference's running sums
// lie within eps = 8 n 2^-53 of these; a position counts only when its sums clear the target
// by eps on both sides.  The order inside a list is exact, and a position counts only when
// its p lies strictly between the least p above the list and the largest below it, so no
// tie reaches across the list's ends.  Where inv is not settled (about one row in 1,000 at
// 151,936 logits) the sum is taken again in id order; what is not proved (3 of 60,000 rows of
// N(0, 2) x 151,936, and rows of few values) takes full_row, as every such row did.
// The histogram only chooses the bins: its error can cost a retry, never a result.
//
// Measured (8 rows of N(0, 2) x 151,936 logits, a pick with its ids on the host): 50 to 60 us
// without cuts (by the logits: the ranked sub-bins hold up to 1,024 entries) and 54 us at top-p
// 0.9, against 18.7 and 12.1 ms in one workgroup a row; the ids left on the device, 37 and 41.
// Bounds: 8 rows x 151,936 logits are 4.9 MB, read from the last-level cache; the two
// passes are instruction-bound (an expf a logit each) at about 300 workgroups, and the end
// is a chain of block steps in one workgroup a row.
#pragma once

#include "qs_decide.h"

namespace qs {
namespace open {

using dec::DecLds;
using dec::ND;
using dec::PartArgs;

constexpr int OP = QS_OPEN_PART;     // logits a workgroup takes (16 a thread, one load each):
constexpr int OQ = OP / ND;          // 304 workgroups for 8 rows of 151,936
constexpr int ONB = QS_OPEN_BINS;    // histogram bins over the row's range (at most 30 nats)
constexpr int OLCAP = QS_OPEN_LIST;  // entries a row's list holds
constexpr int OSUB = 256;            // sub-bins of a list (one a thread)
constexpr int OSMALL = 1024;         // entries of the sub-bins ranked against each other
// Edges are moved off the multiples of the bin width: logits rounded to a coarse grid
// (bf16) would put whole groups of equal values exactly on them.
constexpr float OFF_EDGE = 0.37f;
constexpr double MASS = 0x1p43;      // histogram units of a numerator of 1
constexpr double BIN_SLACK = 0x1p-20;    // histogram and rounding slack around a target

static_assert(OP % ND == 0 && ONB == 4 * ND && OSUB == ND && OQ <= 32, "the thread mapping");

struct OpenArgs {
    OpenScratch s;
    int parts;                       // open parts per row
    int beside;                      // 1: the sums are taken beside the decisions
};

// The rows this path takes: sampling rows whose top-k cuts nothing.
__host__ __device__ __forceinline__ bool open_row(const qs_row_param &P, int vocab) {
    return !row_greedy(P) && (P.top_k <= 0 || P.top_k >= vocab);
}

struct Cross {
    double cum;                      // running sum up to and with the entry
    uint64_t key;
    int pos;                         // its position in the row's order
    int ok;
};

struct OpenSumLds {                  // what a part's sums need
    uint64_t tab[QS_EXPF_TAB_N];
    uint64_t hist[ONB];              // the part's histogram; later the ranked entries
    uint32_t bm[OP / 32];
    double rd[5][ND / 64];
    uint32_t ru[8][ND / 64];
};
struct OpenLds : OpenSumLds {
    uint64_t list[OLCAP];
    uint64_t sub[OSUB];
    uint64_t base;
    Cross cross;
    int ns, flag;
};
static_assert(sizeof(uint64_t) * ONB >= sizeof(uint64_t) * OSMALL, "ranked entries alias hist");

// x * 2^k rounded to an integer, for 0 <= x * 2^k < 2^51 (unit = 2^-k): one addition.
__device__ __forceinline__ uint64_t to_units(double x, double unit) {
    const double magic = 0x1.8p52 * unit;
    return (uint64_t)__double_as_longlong(x + magic) - (uint64_t)__double_as_longlong(magic);
}

// The bin of a scaled logit's distance x = s - msc <= 0: non-decreasing as x falls.
__device__ __forceinline__ int open_bin(float x, float scale) {
    const float b = __builtin_fmaf(-x, scale, OFF_EDGE);
    return (int)fminf(fmaxf(b, 0.0f), (float)(ONB - 1));
}

// The part's logits, one load each (what does not depend on them runs under their latency).
__device__ __forceinline__ void open_load(const PartArgs &a, int row, int part, float (&w)[OQ]) {
    const int lo = part * OP, hi = min(lo + OP, a.vocab);
    const float *x = a.logits + (int64_t)row * a.stride;
#pragma unroll
    for (int k = 0; k < OQ; ++k) {
        const int i = lo + k * ND + (int)threadIdx.x;
        w[k] = i < hi ? x[i] : -INFINITY;
    }
}

// Visit the part's loaded logits in the window: f(k, id, x) for this thread's k-th (all
// threads; the history bitmap in L.bm).
template <typename F>
__device__ __forceinline__ void open_visit(const PartArgs &a, int row, const qs_row_param &P,
                                           int part, float msc, OpenSumLds &L,
                                           float (&w)[OQ], F &&f) {
    const int tid = threadIdx.x, lo = part * OP, hi = min(lo + OP, a.vocab);
    const float rp = P.repeat_penalty, inv_t = P.inv_t, thr = msc - 30.0f;
    // (uniform from the parameters alone: a decision beside the first pass may change the
    // history's length, and build_bitmap's barriers need every thread)
    const bool pen = rp > 1.0f && P.ring_cap > 0;
    if (pen) build_bitmap<ND>(L.bm, OP / 32, lo, hi, a.st, row, P.ring_cap);
#pragma unroll
    for (int k = 0; k < OQ; ++k) {
        const int q = k * ND + tid;
        if (pen && ((L.bm[q >> 5] >> (q & 31)) & 1u)) w[k] = penalise(w[k], rp);
        const float s = w[k] * inv_t;
        if (s >= thr) f(k, lo + q, s - msc);
    }
}

// Block sums in a fixed order (all threads; the result in every thread).
__device__ __forceinline__ double block_sum_d(double v, double (&r)[ND / 64]) {
    v = wave_sum_d(v);
    if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    for (int j = 0; j < ND / 64; ++j) t += r[j];
    return t;
}

// One part of the first pass.  Beside the row decisions the decision of its own row may record
// an id meanwhile, and then nothing here is used (the bitmap reads stay in range whatever the
// ring holds, and a bin is always inside the histogram).
__device__ __forceinline__ void open_sum(const PartArgs &a, const OpenArgs &o, int row, int part,
                                         OpenSumLds &L, const uint64_t *ctab) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const qs_row_param P = row_param(a.st, row);
    if (!open_row(P, a.vocab)) return;
    float w[OQ];
    open_load(a, row, part, w);
    if (tid < QS_EXPF_TAB_N) L.tab[tid] = ctab[tid];
    for (int j = tid; j < ONB; j += ND) L.hist[j] = 0ull;
    // the row's largest and least penalised logits from the streaming kernel's records
    const int NL = a.parts * QS_PART_WAVES;
    const WaveRec *rec = a.sc.wrec + (int64_t)row * NL;
    uint32_t mk = 0u, mn = 0xFFFFFFFFu;
    for (int j = tid; j < NL; j += ND) {
        mk = max(mk, rec[j].maxk);
        mn = min(mn, rec[j].mink);
    }
    mk = wave_max_u(mk);
    mn = wave_min_u(mn);
    if (lane == 0) { L.ru[0][wv] = mk; L.ru[1][wv] = mn; }
    __syncthreads();
    for (int j = 0; j < ND / 64; ++j) {
        mk = max(mk, L.ru[0][j]);
        mn = min(mn, L.ru[1][j]);
    }
    const float maxl = key2f(mk > KEY_NEG_INF ? mk : KEY_NEG_INF);
    const float msc = maxl * P.inv_t;
    if (!isfinite(msc)) return;                       // decided by the row's workgroup
    // bins over the row's own range, so a row of nearly equal logits spreads over them too
    float range = msc - key2f(mn) * P.inv_t;
    if (!(range < 30.0f)) range = 30.0f;
    const float scale = (float)(ONB - 1) / fmaxf(range, 0x1p-10f);
    if (part == 0 && tid == 0) {
        o.s.ctl[row].maxl = maxl;
        o.s.ctl[row].scale = scale;
    }
    const float mp_in = P.min_p * (1.0f + 0x1p-20f), mp_out = P.min_p * (1.0f - 0x1p-20f);
    double acc = 0.0, m_in = 0.0, m_out = 0.0;
    int cnt = 0;
    open_visit(a, row, P, part, msc, L, w, [&](int, int, float x) {
        const float e = qs_expf_core(x, L.tab);
        acc += (double)e;
        ++cnt;
        m_in += e >= mp_in ? (double)e : 0.0;
        m_out += e >= mp_out ? (double)e : 0.0;
        atomicAdd((unsigned long long *)&L.hist[open_bin(x, scale)],
                  (unsigned long long)to_units((double)e, 1.0 / MASS));
    });
    acc = wave_sum_d(acc);
    m_in = wave_sum_d(m_in);
    m_out = wave_sum_d(m_out);
    cnt = wave_sum_i(cnt);
    if (lane == 0) {
        L.rd[0][wv] = acc;
        L.rd[1][wv] = m_in;
        L.rd[2][wv] = m_out;
        L.ru[2][wv] = (uint32_t)cnt;
    }
    __syncthreads();
    for (int b = tid; b < ONB; b += ND)
        if (L.hist[b] != 0ull) add_dev(&o.s.hist[(int64_t)row * ONB + b], L.hist[b]);
    if (tid == 0) {
        OpenSum s{0.0, 0.0, 0.0, 0, 0};
        for (int j = 0; j < ND / 64; ++j) {
            s.sum += L.rd[0][j];
            s.m_in += L.rd[1][j];
            s.m_out += L.rd[2][j];
            s.cnt += (int)L.ru[2][j];
        }
        o.s.sum[(int64_t)row * o.parts + part] = s;
    }
}

// The first position, in list order continued from `base` (the sum of the `above` positions
// before the list), whose running sum reaches `target`: proved as the header says, or
// L.cross.ok = 0.  list: cnt entries in LDS (any order).  All threads; ends synchronised.
__device__ __forceinline__ void list_cross(OpenLds &L, int cnt, double base, int above,
                                           uint32_t min_above, uint32_t max_below,
                                           double target, double eps) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t pmx = 0u, pmn = 0xFFFFFFFFu;
    for (int j = tid; j < cnt; j += ND) {
        const uint32_t b = (uint32_t)(L.list[j] >> 32);
        pmx = max(pmx, b);
        pmn = min(pmn, b);
    }
    pmx = wave_max_u(pmx);
    pmn = wave_min_u(pmn);
    if (lane == 0) { L.ru[0][wv] = pmx; L.ru[1][wv] = pmn; }
    L.sub[tid] = 0ull;
    if (tid == 0) {
        L.cross.ok = 0;
        L.ns = 0;
    }
    if (tid < 2) L.ru[2][tid] = OSUB;
    __syncthreads();
    for (int j = 0; j < ND / 64; ++j) {
        pmx = max(pmx, L.ru[0][j]);
        pmn = min(pmn, L.ru[1][j]);
    }
    if (cnt < 1) return;                              // (uniform; cross.ok is 0)
    // sub-bins of the p bits, with the mass in units of 2^-40 of the power of two above pmx
    const uint32_t span = pmx - pmn;
    const int bits = span ? 32 - __builtin_clz(span) : 0, sh = bits > 8 ? bits - 8 : 0;
    const double unit = ldexp(1.0, (int)(pmx >> 23) - 127 + 1 - 40);
    for (int j = tid; j < cnt; j += ND) {
        const uint32_t b = (uint32_t)(L.list[j] >> 32);
        atomicAdd((unsigned long long *)&L.sub[(pmx - b) >> sh],
                  (unsigned long long)to_units((double)__uint_as_float(b), unit));
    }
    __syncthreads();
    {
        double incl = wave_scan_d((double)L.sub[tid]);
        if (lane == 63) L.rd[0][wv] = incl;
        __syncthreads();
        for (int j = 0; j < wv; ++j) incl += L.rd[0][j];
        const double tgt = (target - base) / unit;
        const double tol = (double)cnt + 1.0 + fabs(target) * eps / unit;
        const uint64_t m0 = __ballot(incl >= tgt - tol), m1 = __ballot(incl >= tgt + tol);
        if (lane == 0) {
            if (m0) atomicMin(&L.ru[2][0], (uint32_t)(wv * 64 + __builtin_ctzll(m0)));
            if (m1) atomicMin(&L.ru[2][1], (uint32_t)(wv * 64 + __builtin_ctzll(m1)));
        }
    }
    __syncthreads();
    const uint32_t s_lo = L.ru[2][0], s_hi = min(L.ru[2][1], (uint32_t)OSUB - 1u);
    double before = 0.0;
    int nb = 0;
    for (int j = tid; j < cnt; j += ND) {
        const uint64_t k = L.list[j];
        const uint32_t s = (pmx - (uint32_t)(k >> 32)) >> sh;
        if (s < s_lo) {
            before += (double)key_p(k);
            ++nb;
        } else if (s <= s_hi) {
            const int at = atomicAdd(&L.ns, 1);
            if (at < OSMALL) L.hist[at] = k;
        }
    }
    nb = wave_sum_i(nb);
    if (lane == 0) L.ru[3][wv] = (uint32_t)nb;
    before = block_sum_d(before, L.rd[1]);            // (synchronises)
    nb = 0;
    for (int j = 0; j < ND / 64; ++j) nb += (int)L.ru[3][j];
    const int m = L.ns;
    if (m <= OSMALL) {
        const double b0 = base + before;
        for (int i = tid; i < m; i += ND) {
            const uint64_t k = L.hist[i];
            double sb = 0.0;
            int rank = 0;
            for (int j = 0; j < m; ++j) {
                const uint64_t kj = L.hist[j];
                if (kj > k) {
                    sb += (double)key_p(kj);
                    ++rank;
                }
            }
            const double prev = b0 + sb, cum = prev + (double)key_p(k);
            const int pos = above + nb + rank;
            const uint32_t pb = (uint32_t)(k >> 32);
            if (cum * (1.0 - eps) >= target && (pos == 0 || prev * (1.0 + eps) < target) &&
                pb < min_above && pb > max_below) {
                L.cross.cum = cum;
                L.cross.key = k;
                L.cross.pos = pos;
                L.cross.ok = 1;
            }
        }
    }
    __syncthreads();
}

// A row's list that other workgroups stored: its first OPRE entries a thread requested into
// registers (before the count is known), then all cnt of them into LDS (all threads).
constexpr int OPRE = 4;
__device__ __forceinline__ void ask_list(const uint64_t *src, uint64_t (&pre)[OPRE]) {
#pragma unroll
    for (int k = 0; k < OPRE; ++k) pre[k] = ld_dev(src + k * ND + threadIdx.x);
}
__device__ __forceinline__ void load_list(OpenLds &L, const uint64_t *src,
                                          const uint64_t (&pre)[OPRE], int cnt) {
#pragma unroll
    for (int k = 0; k < OPRE; ++k)
        if (k * ND + (int)threadIdx.x < cnt) L.list[k * ND + threadIdx.x] = pre[k];
    for (int j = OPRE * ND + threadIdx.x; j < cnt; j += ND) L.list[j] = ld_dev(src + j);
    __syncthreads();
}

// First bins whose running mass reaches t0 and t1 (ONB: none), the thread's four bins'
// inclusive sums in c.  All threads; out: two words of LDS set to ONB and synchronised.
__device__ __forceinline__ void first_bins(const double (&c)[4], double t0, double t1,
                                           uint32_t *out) {
    uint32_t b0 = ONB, b1 = ONB;
#pragma unroll
    for (int q = 3; q >= 0; --q) {
        if (c[q] >= t0) b0 = 4 * threadIdx.x + q;
        if (c[q] >= t1) b1 = 4 * threadIdx.x + q;
    }
    b0 = wave_min_u(b0);
    b1 = wave_min_u(b1);
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&out[0], b0);
        atomicMin(&out[1], b1);
    }
    __syncthreads();
}

// The row's end: its last part finds the cut and the drawn position (all threads).  Returns
// whether the row was decided and recorded.
__device__ __forceinline__ bool open_finish(const PartArgs &a, const OpenArgs &o, int row,
                                            const qs_row_param &P, double S, float inv, int nwin,
                                            float maxl, float msc, uint64_t rs, double u,
                                            int reason, OpenLds &L) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // one round of requests: the counts, the parts' sums and the head of both lists
    const uint64_t cnts = ld_dev(&o.s.ctl[row].cnt);
    const uint64_t *lists = o.s.list + (int64_t)row * 2 * OLCAP;
    uint64_t pre1[OPRE], pre2[OPRE];
    if (P.top_p < 1.0f) ask_list(lists, pre1);
    ask_list(lists + OLCAP, pre2);
    // the parts' sums, in a fixed order
    uint64_t v[8] = {};
    if (tid < o.parts) {
        const uint64_t *src = (const uint64_t *)(o.s.prec + (int64_t)row * o.parts + tid);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = ld_dev(src + j);
    } else {
        v[6] = v[7] = 0xFFFFFFFFull;                  // (min, max) pairs: none
    }
    const int cnt1 = (int)(uint32_t)cnts, cnt2 = (int)(uint32_t)(cnts >> 32);
    if (cnt1 > OLCAP || cnt2 > OLCAP) return false;
    double sums[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) sums[j] = wave_sum_d(__longlong_as_double((long long)v[j]));
    const int n1 = wave_sum_i((int)(uint32_t)v[4]), n2 = wave_sum_i((int)(uint32_t)(v[4] >> 32));
    const int nm = wave_sum_i((int)(uint32_t)v[5]);
    const uint32_t mn1 = wave_min_u((uint32_t)v[6]), mx1 = wave_max_u((uint32_t)(v[6] >> 32));
    const uint32_t mn2 = wave_min_u((uint32_t)v[7]), mx2 = wave_max_u((uint32_t)(v[7] >> 32));
    if (lane == 0) {
        for (int j = 0; j < 4; ++j) L.rd[j][wv] = sums[j];
        L.ru[0][wv] = (uint32_t)n1;
        L.ru[1][wv] = (uint32_t)n2;
        L.ru[2][wv] = (uint32_t)nm;
        L.ru[3][wv] = mn1;
        L.ru[4][wv] = mx1;
        L.ru[5][wv] = mn2;
        L.ru[6][wv] = mx2;
    }
    __syncthreads();
    double a1 = 0.0, a2 = 0.0, am = 0.0, all = 0.0;
    int above1 = 0, above2 = 0, kept_m = 0;
    uint32_t min1 = 0xFFFFFFFFu, max1 = 0u, min2 = 0xFFFFFFFFu, max2 = 0u;
    for (int j = 0; j < ND / 64; ++j) {
        a1 += L.rd[0][j];
        a2 += L.rd[1][j];
        am += L.rd[2][j];
        all += L.rd[3][j];
        above1 += (int)L.ru[0][j];
        above2 += (int)L.ru[1][j];
        kept_m += (int)L.ru[2][j];
        min1 = min(min1, L.ru[3][j]);
        max1 = max(max1, L.ru[4][j]);
        min2 = min(min2, L.ru[5][j]);
        max2 = max(max2, L.ru[6][j]);
    }
    __syncthreads();
    const double eps = 8.0 * (double)nwin * 0x1p-53;
    // sample.c:155-160: the shortest prefix whose running sum reaches top_p
    int n_topp = nwin;
    double rsum = all;
    if (P.top_p < 1.0f) {
        const double tp = (double)P.top_p;
        if (!(all * (1.0 + eps) < tp)) {
            load_list(L, lists, pre1, cnt1);
            list_cross(L, cnt1, a1, above1, min1, max1, tp, eps);
            if (!L.cross.ok) return false;
            n_topp = L.cross.pos + 1;
            rsum = L.cross.cum;
            __syncthreads();
        }
    }
    // sample.c:161-168: the ids below min_p p0 go, the first position stays
    int n = n_topp;
    if (P.min_p > 0.0f) {
        const int nk = max(kept_m, 1);
        if (nk < n) {
            n = nk;
            rsum = kept_m > 0 ? am : (double)inv;     // (p0 = fl(1 * inv))
        }
    }
    const double r = u * rsum;                        // sample.c:170-175
    load_list(L, lists + OLCAP, pre2, cnt2);
    list_cross(L, cnt2, a2, above2, min2, max2, r, eps);
    if (!L.cross.ok || L.cross.pos >= n) return false;
    if (tid == 0) {
        const int id = key_id(L.cross.key);
        a.st.rng[row] = rs;
        ring_record(a.st.ring + (int64_t)row * a.st.ring_stride, a.st.hlen + row,
                    a.st.hhead + row, P.ring_cap, id);
        a.out[row] = id;
        add_dev(o.s.selected, 1);
        if (a.diag) {
            qs_pick_diag d;
            memset(&d, 0, sizeof d);
            d.id = id;
            d.path = QS_PATH_FULL;
            d.n_window = nwin;
            d.n_cand = nwin;
            d.keep_topk = nwin;
            d.keep_topp = n_topp;
            d.keep = n;
            d.rank = L.cross.pos;
            d.maxl = maxl;
            d.msc = msc;
            d.inv = inv;
            d.inv_hi = inv;
            d.p0 = inv;
            d.fallback = reason;
            d.sum = S;
            d.sum_hi = S;
            d.rsum = rsum;
            d.u = u;
            a.diag[row] = d;
        }
    }
    return true;
}

// The row's softmax denominator exactly as sample.c:147-149 adds it, by one workgroup: a part's
// numerators at a time into LDS (0 outside the window, which adds nothing), then one binary64
// chain over them in id order.  All threads; the sum in every thread.
__device__ __forceinline__ double open_sum_in_order(const PartArgs &a, const OpenArgs &o, int row,
                                                    const qs_row_param &P, float msc,
                                                    OpenLds &L) {
    static_assert(OLCAP >= OP && OP % 16 == 0, "a part's numerators in the list's LDS");
    const int tid = threadIdx.x;
    double *e = (double *)L.list;
    double acc = 0.0;
    for (int q = 0; q < o.parts; ++q) {
        float w[OQ];
        open_load(a, row, q, w);
#pragma unroll
        for (int k = 0; k < OQ; ++k) e[k * ND + tid] = 0.0;
        open_visit(a, row, P, q, msc, L, w, [&](int k, int, float x) {
            e[k * ND + tid] = (double)qs_expf_core(x, L.tab);
        });
        __syncthreads();
        if (tid < 64) {                               // (every lane the same chain)
            const double2 *d = (const double2 *)e;
            for (int i = 0; i < OP / 2; i += 8) {
                double2 v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = d[i + j];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    acc += v[j].x;
                    acc += v[j].y;
                }
            }
        }
        __syncthreads();
    }
    if (tid == 0) L.rd[4][0] = acc;
    __syncthreads();
    return L.rd[4][0];
}

// The second pass: one part of a row of the queue.
template <bool UNAL>
__device__ __forceinline__ void open_select(const PartArgs &a, const OpenArgs &o, int row,
                                            int part, OpenLds &L, DecLds &dl,
                                            const uint64_t *ctab) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    OpenCtl *ctl = o.s.ctl + row;
    uint64_t *ghist = o.s.hist + (int64_t)row * ONB;
    const qs_row_param P = row_param(a.st, row);
    float w[OQ];
    open_load(a, row, part, w);
    const int reason = ctl->reason;
    if (tid < QS_EXPF_TAB_N) L.tab[tid] = ctab[tid];
    if (tid < 4) L.ru[7][tid] = ONB;
    const float maxl = ctl->maxl, scale = ctl->scale, msc = maxl * P.inv_t;
    OpenSum os{0.0, 0.0, 0.0, 0, 0};
    if (tid < o.parts) os = o.s.sum[(int64_t)row * o.parts + tid];
    double c[4];
    {
        const ulong2 *src = (const ulong2 *)(ghist + 4 * tid);
        const ulong2 q0 = src[0], q1 = src[1];
        c[0] = (double)q0.x;
        c[1] = c[0] + (double)q0.y;
        c[2] = c[1] + (double)q1.x;
        c[3] = c[2] + (double)q1.y;
    }
    os.sum = wave_sum_d(os.sum);
    os.m_in = wave_sum_d(os.m_in);
    os.m_out = wave_sum_d(os.m_out);
    os.cnt = wave_sum_i(os.cnt);
    const double incl = wave_scan_d(c[3]);
    if (lane == 0) {
        L.rd[0][wv] = os.sum;
        L.rd[1][wv] = os.m_in;
        L.rd[2][wv] = os.m_out;
        L.ru[0][wv] = (uint32_t)os.cnt;
    }
    if (lane == 63) L.rd[3][wv] = incl;
    __syncthreads();
    double S = 0.0, m_in = 0.0, m_out = 0.0, T = 0.0, cb = incl - c[3];
    int nwin = 0;
    for (int j = 0; j < ND / 64; ++j) {
        S += L.rd[0][j];
        m_in += L.rd[1][j];
        m_out += L.rd[2][j];
        T += L.rd[3][j];
        if (j < wv) cb += L.rd[3][j];
        nwin += (int)L.ru[0][j];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) c[q] += cb;
    const bool good = !a.sc.sum_in_order && inv_settled(S, nwin);   // (uniform)
    float inv = (float)(1.0 / S);
    uint64_t rs = a.st.rng[row];
    const double u = rng_unit(rs);
    // the bins of the top-p cut, and the sum the draw scales with (histogram units)
    const bool topp = P.top_p < 1.0f;
    int c_lo = ONB, c_hi = ONB, d_lo, d_hi;
    {
        double r_lo = T, r_hi = T;
        if (topp) {
            const double m = (double)P.top_p * T;
            first_bins(c, m * (1.0 - BIN_SLACK), m * (1.0 + BIN_SLACK), &L.ru[7][0]);
            c_lo = (int)L.ru[7][0];
            c_hi = min((int)L.ru[7][1], ONB - 1);
            // the prefix ends with an id of those bins: at most the largest numerator of
            // the first one past the target
            const float top = c_lo > 0 ? __expf(-((float)c_lo - OFF_EDGE) / scale) : 1.0f;
            r_lo = m * (1.0 - BIN_SLACK);
            r_hi = fmin(m * (1.0 + BIN_SLACK) + (double)top * 1.01 * MASS, T);
        }
        if (P.min_p > 0.0f) {
            r_lo = fmin(r_lo, fmax(m_in, 1.0) * MASS);
            r_hi = fmin(r_hi, fmax(m_out, 1.0) * MASS);
        }
        first_bins(c, u * r_lo * (1.0 - BIN_SLACK), u * r_hi * (1.0 + BIN_SLACK) + 1.0,
                   &L.ru[7][2]);
        d_lo = (int)L.ru[7][2];
        d_hi = min((int)L.ru[7][3], ONB - 1);
    }
    // Each part takes its own share.  Where the parts' sum leaves inv open (about one row in
    // 1,000 at 151,936 logits), the last part adds the row's numerators in id order (1 ms) and
    // takes every part's share itself (the whole-window sort took 12 to 19 ms).
    bool all_parts = false;
    for (int q = part;;) {
        if (good || all_parts) {
            // the part's share: sums above the bins, the entries inside them
            const float floor_p = P.min_p * inv;
            double a1 = 0.0, a2 = 0.0, am = 0.0, all = 0.0;
            int n1 = 0, n2 = 0, nm = 0;
            uint32_t min1 = 0xFFFFFFFFu, max1 = 0u, min2 = 0xFFFFFFFFu, max2 = 0u;
            uint32_t in1 = 0u, in2 = 0u;
            float p[OQ];
#pragma unroll
            for (int k = 0; k < OQ; ++k) p[k] = 0.0f;
            open_visit(a, row, P, q, msc, L, w, [&](int k, int, float x) {
                const float pk = qs_expf_core(x, L.tab) * inv;
                const uint32_t pb = __float_as_uint(pk);
                const double pd = (double)pk;
                const int b = open_bin(x, scale);
                p[k] = pk;
                all += pd;
                if (topp) {
                    if (b < c_lo) {
                        a1 += pd;
                        ++n1;
                        min1 = min(min1, pb);
                    } else if (b <= c_hi) {
                        in1 |= 1u << k;
                    } else {
                        max1 = max(max1, pb);
                    }
                }
                if (b < d_lo) {
                    a2 += pd;
                    ++n2;
                    min2 = min(min2, pb);
                } else if (b <= d_hi) {
                    in2 |= 1u << k;
                } else {
                    max2 = max(max2, pb);
                }
                if (pk >= floor_p) {
                    am += pd;
                    ++nm;
                }
            });
            // the entries' places: one addition to the row's two counts for the workgroup
            const uint32_t mine = (uint32_t)__popc(in1) | ((uint32_t)__popc(in2) << 16);
            const uint32_t pre = wave_scan(mine);         // (counts up to 4096: 16 bits each)
            a1 = wave_sum_d(a1);
            a2 = wave_sum_d(a2);
            am = wave_sum_d(am);
            all = wave_sum_d(all);
            n1 = wave_sum_i(n1);
            n2 = wave_sum_i(n2);
            nm = wave_sum_i(nm);
            min1 = wave_min_u(min1);
            max1 = wave_max_u(max1);
            min2 = wave_min_u(min2);
            max2 = wave_max_u(max2);
            __syncthreads();                              // (rd and ru were read above)
            if (lane == 63) L.ru[7][wv] = pre;
            if (lane == 0) {
                L.rd[0][wv] = a1;
                L.rd[1][wv] = a2;
                L.rd[2][wv] = am;
                L.rd[3][wv] = all;
                L.ru[0][wv] = (uint32_t)n1;
                L.ru[1][wv] = (uint32_t)n2;
                L.ru[2][wv] = (uint32_t)nm;
                L.ru[3][wv] = min1;
                L.ru[4][wv] = max1;
                L.ru[5][wv] = min2;
                L.ru[6][wv] = max2;
            }
            __syncthreads();
            uint32_t off = pre - mine, tot = 0u;
            for (int j = 0; j < ND / 64; ++j) {
                if (j < wv) off += L.ru[7][j];
                tot += L.ru[7][j];
            }
            if (tid == 0) {
                L.base = tot ? add_dev(&ctl->cnt, (uint64_t)(tot & 0xFFFFu) |
                                                      ((uint64_t)(tot >> 16) << 32))
                             : 0ull;
                a1 = a2 = am = all = 0.0;
                n1 = n2 = nm = 0;
                min1 = min2 = 0xFFFFFFFFu;
                max1 = max2 = 0u;
                for (int j = 0; j < ND / 64; ++j) {
                    a1 += L.rd[0][j];
                    a2 += L.rd[1][j];
                    am += L.rd[2][j];
                    all += L.rd[3][j];
                    n1 += (int)L.ru[0][j];
                    n2 += (int)L.ru[1][j];
                    nm += (int)L.ru[2][j];
                    min1 = min(min1, L.ru[3][j]);
                    max1 = max(max1, L.ru[4][j]);
                    min2 = min(min2, L.ru[5][j]);
                    max2 = max(max2, L.ru[6][j]);
                }
                uint64_t *dst = (uint64_t *)(o.s.prec + (int64_t)row * o.parts + q);
                st_dev(dst + 0, (uint64_t)__double_as_longlong(a1));
                st_dev(dst + 1, (uint64_t)__double_as_longlong(a2));
                st_dev(dst + 2, (uint64_t)__double_as_longlong(am));
                st_dev(dst + 3, (uint64_t)__double_as_longlong(all));
                st_dev(dst + 4, (uint64_t)(uint32_t)n1 | ((uint64_t)(uint32_t)n2 << 32));
                st_dev(dst + 5, (uint64_t)(uint32_t)nm);
                st_dev(dst + 6, (uint64_t)min1 | ((uint64_t)max1 << 32));
                st_dev(dst + 7, (uint64_t)min2 | ((uint64_t)max2 << 32));
            }
            __syncthreads();
            const uint64_t gb = L.base;
            uint32_t at1 = (uint32_t)gb + (off & 0xFFFFu), at2 = (uint32_t)(gb >> 32) + (off >> 16);
            uint64_t *lists = o.s.list + (int64_t)row * 2 * OLCAP;
#pragma unroll
            for (int k = 0; k < OQ; ++k) {
                const uint64_t key = pid_key(p[k], q * OP + k * ND + tid);
                if ((in1 >> k) & 1u) {
                    if (at1 < OLCAP) st_dev(lists + at1, key);
                    ++at1;
                }
                if ((in2 >> k) & 1u) {
                    if (at2 < OLCAP) st_dev(lists + OLCAP + at2, key);
                    ++at2;
                }
            }
        }
        stores_done();                                // every wavefront's, then counted
        __syncthreads();
        if (all_parts) {
            if (++q == o.parts) break;
        } else {
            if (tid == 0) L.flag = add_dev(&ctl->done, 1) == o.parts - 1;
            __syncthreads();
            if (!L.flag) return;
            if (good) break;
            S = open_sum_in_order(a, o, row, P, msc, L);
            inv = (float)(1.0 / S);
            all_parts = true;
            q = 0;
        }
        open_load(a, row, q, w);
    }
    const bool ok = open_finish(a, o, row, P, S, inv, nwin, maxl, msc, rs, u, reason, L);
    // every part has read the histogram and the counts: zero for the next pick
    for (int b = tid; b < ONB; b += ND) st_dev(ghist + b, (uint64_t)0);
    if (tid == 0) {
        st_dev(&ctl->cnt, (uint64_t)0);
        st_dev(&ctl->done, 0);
    }
    if (ok) return;
    // not proved: the whole window sorted by this workgroup
    __syncthreads();
    if (tid < QS_EXPF_TAB_N) dl.dl.tab[tid] = ctab[tid];
    __syncthreads();
    double sum = 0.0;
    int nw = 0;
    dec::exact_totals<UNAL>(a, row, P, msc, dl, sum, nw);
    full_row<ND>(a.logits + (int64_t)row * a.stride, a.vocab, row, P, maxl, sum, a.st, a.sc,
                 a.out, a.diag, dl.dl.tab, *(FullLds<ND> *)dl.keys, -1);
    __syncthreads();
    if (tid == 0 && a.diag) a.diag[row].fallback = reason;
}

}  // namespace open
}  // namespace qs
