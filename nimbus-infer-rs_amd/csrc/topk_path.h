// topk_path.h — top-k rows with a repetition-penalty history, or longer than
// the registers hold (256 <= V <= 262141, 1 <= k <= 960, T > 0, any
// top-p > 0; src/sampler.rs:83-116, 118-160, 201-216).  One row per
// 1024-lane workgroup; the row is streamed once and only its head is kept.
//
// What bounds it: one CU's HBM stream of the row, then a chain of short
// workgroup steps.  The stream keeps no element: each lane holds the
// maxima of 16 groups of its float4s (G float4s each), and a chunk of 64
// float4s costs five VALU instructions, far below the CU's share of HBM.
//
// Threshold.  With need = k + (distinct history ids), the need-th largest
// group maximum tau is at most the need-th largest logit, because the groups
// are disjoint; so at least `need` logits, and at least k that no penalty
// touches, are >= tau, whatever the distribution.  (need is cut at kTNeed so
// that the lists can hold the candidates; a row left with fewer than k of
// them is declined.)  The workgroup finds a tau
// that at least `need` maxima reach by counting their order-preserving keys
// in 256 buckets (again inside one bucket while the count is more than a
// quarter above `need`).  The groups reaching tau are read again (they are in
// L2 or the MALL) and their elements >= tau become the candidates; penalised
// elements are left out there and join as f64 values y, wherever y / T
// reaches tau / T.  Every value at or above the k-th largest is then a
// candidate.
//
// Finish.  w = v / T in f64 as the reference computes it.  More than a few
// candidates beyond k are cut by the same search.  Every candidate then
// counts the larger ones (kept by top-k while fewer than k are strictly
// larger, sampler.rs:110-114) and sums the masses before it in the stable
// descending order (sampler.rs:140-154); the kept ones sum the masses at or
// before their index, and the one whose sum crosses r = u Z is the token
// (sampler.rs:209-214).  Both sums are pairwise over LDS entries, the pairs
// split over all 16 waves.  Masses are f64 exp(w - max); their sums are
// integers in units of 2^-52 (of at most 1024 terms <= 1), so they do not
// depend on the order in which the candidates were listed.
//
// Measured against the general path, which these rows took before: 64 rows of
// V = 128256, k = 50, top-p 0.9: 343 -> 19.4 us a call; a decode step of 64
// rows of V = 50257, k = 50, top-p 0.9, penalty 1.1, 200-id histories: 346 ->
// 16.8 us (one row alone: 12.8 us, of it the stream 4.7, the threshold 0.9,
// the candidates 2.5, the cut to the final ones 1.2, the finish 3.5; the
// steps after the stream are bound by their instructions, 16 waves on 4
// SIMDs, so waves without work leave early or skip them).
//
// A row this path cannot prove (k past 960, a history past 4096 ids, NaN or
// +inf, more candidates than the lists hold) returns a reject code before
// anything is written; the kernel then runs the general path.
#pragma once
#include "penalty_bits.h"
#include "sparse_path.h"

namespace nis {

constexpr int kTB = 1024;                     // lanes per workgroup
constexpr int kTW = kTB / 64;                 // waves per workgroup
constexpr int kTN = 16;                       // float4 groups per lane
constexpr int kTMaxV = kTB * 4 * kTN * 4 - 3; // 262141: groups of up to 4 float4s
constexpr int kTMaxK = 960;   // (the final step holds ties and the search's excess beyond k, up to 1024)
constexpr int kTCap = 4096;                   // candidates (4 per lane)
constexpr int kTNeed = 2800;                  // group maxima to reach tau, at most
constexpr int kTGl = 4096;                    // float4 groups read again
constexpr int kTFin = 1024;                   // candidates of the final step (1 per lane)
constexpr int kTLev = 4;                      // levels of one search, 256 buckets each
constexpr int kTD = 8;                        // loads in flight ahead of the chunk in use
constexpr uint32_t kTFinite = 0x00800000u;    // key32 of the lowest finite float
constexpr double kTFix = 4503599627370496.0;  // 2^52: units of the mass sums

struct alignas(16) TEnt {
    double w;
    unsigned long long fx;  // exp(w - max) in 2^-52 units
};

struct TopkShared {
    uint32_t bitmap[(kTMaxV + 31) / 32];      // the penalised ids
    double cv[kTCap];                         // candidates: value (penalised),
    uint32_t ci[kTCap];                       //   row index
    union alignas(16) {
        uint32_t gl[kTGl];                    // groups to read again: first float4 slot
        struct {
            TEnt ent[kTFin];                  // the final candidates (after the listing)
        };
    };
    uint32_t ei[kTFin];
    unsigned long long kfx[kTFin];            // the kept ones: mass,
    uint32_t ki[kTFin];                       //   row index
    unsigned long long psum[kTB];             // partial pairwise sums [part][candidate]
    uint32_t pcnt[kTB];
    uint32_t hist[2][kTLev][256];             // the two searches' buckets
    unsigned long long zred[2][kTW];          // per-wave sums: top-k mass, kept mass
    unsigned long long wmax;                  // key64 of the largest w
    double u;
    uint32_t kmax;                            // key32 of the largest logit
    uint32_t kmin[4];                         //   of the smallest finite maximum: 4 lanes', a lane's, 4 groups', one group's
    uint32_t kpen;                            //   of the largest penalised candidate
    uint32_t nfin[4];                         // finite maxima: 4 lanes', a lane's, 4 groups', one group's
    uint32_t hd;                              // distinct history ids
    uint32_t bad;                             // NaN or an infinite penalised value
    uint32_t ng, n, m, m2;                    // groups listed, candidates, final ones, kept ones
};
static_assert(sizeof(TopkShared) <= 163840, "LDS of one workgroup");

__host__ __device__ __forceinline__ bool topk_eligible(const RowArgs& a) {
    return a.V >= 256 && a.V <= kTMaxV && a.temperature > 0.0f && !(a.top_p <= 0.0f) && a.top_k > 0 &&
           a.top_k < (uint64_t)a.V;
}

// A value t <= hi that at least `need` of the workgroup's values x reach and,
// where they allow, about `enough` at most (at least `need` reach the given
// lo; none passes hi).  Each level counts the values of [lo, hi] in 256 equal
// buckets and goes on inside the bucket that holds the need-th largest: one
// level in most rows.  t lies a rounding margin below that bucket's lower
// edge, so every value counted reaches it.  Every lane of the workgroup takes
// part with its N values and gets the same result.
template <int N>
__device__ __forceinline__ float topk_search(uint32_t (*hist)[256], const float (&x)[N], float lo, float hi,
                                             uint32_t need, uint32_t enough) {
    const int l = lane_id();
    uint32_t live = 0u;
#pragma unroll
    for (int i = 0; i < N; ++i) live |= x[i] >= lo ? 1u << i : 0u;
    for (int lev = 0; lev < kTLev; ++lev) {
        // (quarters: the span of finite floats may overflow)
        const float lo4 = 0.25f * lo, span = 0.25f * hi - lo4;
        if (!(span > 1.0e-35f)) break;  // (ties)
        const float sc = 255.99f / span;
        int bin[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            bin[i] = (live >> i) & 1u ? min(max((int)((0.25f * x[i] - lo4) * sc), 0), 255) : -1;
            if (bin[i] >= 0) atomicAdd(&hist[lev][bin[i]], 1u);
        }
        lds_barrier();
        // lane l: buckets 255 - 4 l .. 252 - 4 l, counted from the top
        const u4v h = *reinterpret_cast<const u4v*>(&hist[lev][252 - 4 * l]);
        const uint32_t c0 = h.w, c1 = c0 + h.z, c2 = c1 + h.y, c3 = c2 + h.x;
        const uint32_t incl = wscan_u32(c3), ex = incl - c3;
        const uint64_t m = __ballot(incl >= need);
        const int at = m ? __ffsll((long long)m) - 1 : 63;
        const int q = (ex + c0 >= need) ? 0 : (ex + c1 >= need) ? 1 : (ex + c2 >= need) ? 2 : 3;
        const uint32_t thru = ex + (q == 0 ? c0 : q == 1 ? c1 : q == 2 ? c2 : c3);
        const uint32_t own = (q == 0 ? h.w : q == 1 ? h.z : q == 2 ? h.y : h.x);
        const int b = (int)bcast_u32((uint32_t)(255 - 4 * l - q), at);
        const uint32_t cum = bcast_u32(thru, at), cnt = bcast_u32(own, at);
        const float wd = 1.0f / sc, mg = (fabsf(lo4) + span) * 2.0e-6f + 1.0e-37f;
        hi = fminf(hi, 4.0f * (lo4 + (float)(b + 1) * wd + mg));
        lo = fmaxf(lo, 4.0f * (lo4 + (float)b * wd - mg));
        if (cum <= enough) break;
        need -= cum - cnt;  // (the buckets above stay counted)
        enough -= min(enough, cum - cnt);
#pragma unroll
        for (int i = 0; i < N; ++i) live &= bin[i] == b ? 0xFFFFFFFFu : ~(1u << i);
    }
    return lo;
}

// Wave maximum of f64 values that are not NaN, uniform (DPP scan).
__device__ __forceinline__ double wmax_f64(double v) {
#define NIS_DPPM(C, M)                                                                       \
    {                                                                                        \
        const uint64_t b_ = (uint64_t)__double_as_longlong(v);                               \
        const uint32_t lo_ = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)b_, (int)(uint32_t)b_, C, M, 0xF, false); \
        const uint32_t hi_ = (uint32_t)__builtin_amdgcn_update_dpp((int)(b_ >> 32), (int)(b_ >> 32), C, M, 0xF, false);     \
        v = fmax(v, __longlong_as_double((long long)(((uint64_t)hi_ << 32) | lo_)));         \
    }
    NIS_DPPM(0x111, 0xF)
    NIS_DPPM(0x112, 0xF)
    NIS_DPPM(0x114, 0xF)
    NIS_DPPM(0x118, 0xF)
    NIS_DPPM(0x142, 0xA)
    NIS_DPPM(0x143, 0xC)
#undef NIS_DPPM
    return bcast_f64(v, 63);
}

// Pairs (j, t), j and t < m <= 1024: f(j, t) over every t for every j, split
// over the 16 waves: wave w takes candidates 64 (w % jb) .. + 63 (lane l: j =
// 64 (w % jb) + l) and the t of part w / jb.  acc returns its part's sum for
// slot part * 64 jb + j.
struct TPairs {
    int jb, tb, j, slot, t0, t1;
};
__device__ __forceinline__ TPairs topk_pairs(int m, int w, int l) {
    TPairs p;
    const int nb = (m + 63) >> 6;
    p.jb = nb <= 1 ? 1 : (nb <= 2 ? 2 : (nb <= 4 ? 4 : (nb <= 8 ? 8 : 16)));
    p.tb = kTW / p.jb;
    const int part = w / p.jb;
    const int per = (m + p.tb - 1) / p.tb;
    p.j = 64 * (w % p.jb) + l;
    p.slot = part * 64 * p.jb + p.j;
    p.t0 = min(part * per, m);
    p.t1 = min(p.t0 + per, m);
    return p;
}

// Returns NIS_REJECT_NONE when the row is done, else (uniformly across the
// workgroup) why it must be recomputed; nothing has been written then.
template <int G>
__device__ __forceinline__ uint32_t topk_row(const RowArgs a, const int row, TopkShared& sh) {
    const int tid = (int)threadIdx.x, l = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(wave_id());
    const int V = (int)a.V;
    if (a.top_k > (uint64_t)kTMaxK) return NIS_REJECT_WINDOW;
    const uint32_t topk = (uint32_t)a.top_k;
    const gfp rowp = (gfp)(a.logits + (int64_t)row * a.ld);
    const int mis = (int)(((uintptr_t)rowp >> 2) & 3);  // elements before the row in its 16 B block
    const gf4p base = (gf4p)(rowp - mis);
    const int f_lo = mis ? 1 : 0;          // first float4 slot lying fully inside the row
    const int f_hi = (V + mis - 4) >> 2;   // last one
    const int nsl = (V + mis + 3) >> 2;    // slots touching the row
    const int cpw = (((nsl + 63) >> 6) + kTW - 1) / kTW;  // chunks per wave (<= kTN * G)
    const int wbase = 64 * cpw * w;
    const int Kw = min(max((nsl - wbase + 63) >> 6, 0), cpw);
    const int slot0 = wbase + l;

    // ---- the row's first chunks, then the history's ids -------------------------
    const uint64_t bptr = (uint64_t)(uintptr_t)base;
    const i4v rsrc = {(int32_t)(uint32_t)bptr, (int32_t)(uint32_t)((bptr >> 32) & 0xFFFFu),
                      16 * (f_hi + 1), 0x00020000};
    const int voff = 16 * slot0;
    // chunk k's load (past the wave's range: an offset that reads nothing)
    auto load = [&](int k) -> f4v {
        const int off = (k == 0) ? 16 * max(slot0, f_lo) : voff + 1024 * k;
        return nis_buffer_load_f4(rsrc, (k < Kw) ? off : 0x7FFFFFF0, 0, 0);
    };
    f4v ring[kTD];
#pragma unroll
    for (int k = 0; k < kTD; ++k) {
        ring[k] = load(k);
        __builtin_amdgcn_sched_barrier(0);
    }
    // the (at most 3 + 3) elements of partial head / tail slots, in lanes 0..5
    const int nhead = mis ? 4 - mis : 0, ntail = (V + mis) & 3;
    const int eidx = l < 3 ? l : V - 6 + l;
    const bool eon = (l < 3) ? l < nhead : (l < 6 && 6 - l <= ntail);
    const float ev = eon ? rowp[eidx] : -INFINITY;
    // (an empty history costs the clearing of the bitmap: its length is not
    // waited for here)
    const bool pen = a.penalty != 1.0f && a.gen_ids != nullptr;
    uint32_t hid[kPHist / kPB];
    bool hlong = false;
    // ---- the shared state cleared, ordered by one barrier before any use -----
    if (pen)
        for (int i = tid; i < (V + 31) >> 5; i += kTB) sh.bitmap[i] = 0u;
#pragma unroll
    for (int i = tid; i < 2 * kTLev * 256; i += kTB) (&sh.hist[0][0][0])[i] = 0u;
    if (tid == 0) {
        sh.wmax = 0ull;
        sh.kmax = sh.kpen = 0u;
        sh.kmin[0] = sh.kmin[1] = sh.kmin[2] = sh.kmin[3] = 0xFFFFFFFFu;
        sh.nfin[0] = sh.nfin[1] = sh.nfin[2] = sh.nfin[3] = 0u;
        sh.hd = sh.bad = 0u;
        sh.ng = sh.n = sh.m = sh.m2 = 0u;
    }
    lds_barrier();
    if (pen) hlong = pen_load_ids(a, row, tid, hid);

    // ---- stream: the maxima of the lane's groups -------------------------------
    float mx[kTN];
#pragma unroll
    for (int i = 0; i < kTN; ++i) mx[i] = -INFINITY;
    bool nan = false;
#pragma unroll
    for (int k = 0; k < kTN * G; ++k) {
        if (k < Kw) {
            f4v x = ring[k % kTD];
            const int fb0 = wbase + 64 * k;
            if (fb0 < f_lo || fb0 + 63 > f_hi) {  // lanes outside the row's whole slots
                const int f = slot0 + 64 * k;
                if (f < f_lo || f > f_hi) x = f4v{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            }
            nan |= __builtin_isunordered(x.x, x.y) | __builtin_isunordered(x.z, x.w);
            mx[k / G] = s_max(mx[k / G], s_max4(x));
        }
        if (k + kTD < kTN * G) ring[k % kTD] = load(k + kTD);
    }
    float km[4];  // the maxima of every fourth group
#pragma unroll
    for (int i = 0; i < 4; ++i) km[i] = s_max(s_max(mx[i], mx[i + 4]), s_max(mx[i + 8], mx[i + 12]));
    // the penalised ids: each distinct one belongs to the lane that sets its
    // bit, which reads its logit now and adds its penalised value later (after
    // the stream: the ids' loads were queued behind the row's first chunks)
    float hx[kPHist / kPB];
    uint32_t own = 0u;
    if (pen) {
        uint32_t hd = 0u;
#pragma unroll
        for (int i = 0; i < kPHist / kPB; ++i) {
            bool mine = false;
            if (hid[i] < (uint32_t)V) {
                const uint32_t bit = 1u << (hid[i] & 31u);
                mine = (atomicOr(&sh.bitmap[hid[i] >> 5], bit) & bit) == 0u;
            }
            own |= mine ? 1u << i : 0u;
            hx[i] = mine ? rowp[hid[i]] : -INFINITY;
            hd += (uint32_t)__popcll(__ballot(mine));
        }
        if (l == 0 && hd) atomicAdd(&sh.hd, hd);
    }
    const float ml = s_max(s_max(km[0], km[1]), s_max(km[2], km[3]));  // the lane's
    {
        // the wave's largest logit, and the smallest finite maximum of 4 lanes:
        // at least as many elements reach it as there are such maxima
        float mq = s_max(ml, dpp_ninf<0xB1>(ml));
        mq = s_max(mq, dpp_ninf<0x4E>(mq));
        const float mw = wmax_f32(w == 0 ? s_max(mq, ev) : mq);
        const uint32_t klq = wmin_u32(mq > -INFINITY ? key32(mq) : 0xFFFFFFFFu);
        const uint32_t nq = (uint32_t)__popcll(__ballot(mq > -INFINITY)) >> 2;
        bool bad = nan;
        if (w == 0) bad |= eon & !(ev < INFINITY);
        const bool anyb = __ballot(bad) != 0ull;
        if (l == 0) {
            atomicAdd(&sh.nfin[0], nq);
            atomicMin(&sh.kmin[0], klq);
            atomicMax(&sh.kmax, key32(mw));
            if (anyb | hlong) atomicOr(&sh.bad, anyb ? 1u : 2u);
        }
    }
    typedef const __attribute__((address_space(1))) uint64_t* gu64p;
    uint64_t rsv = 0;
    if (w == 0) rsv = ((gu64p)(a.rng + 4 * (int64_t)row))[l & 3];
    uint64_t rst = 0;  // wave 0, lane j < 4: word j of the advanced state
    if (w == 0) {
        uint64_t st[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            st[j] = ((uint64_t)bcast_u32((uint32_t)(rsv >> 32), j) << 32) | bcast_u32((uint32_t)rsv, j);
        const double u0 = rng_next_f64(st);
        if (l == 0) sh.u = u0;
        rst = (l == 0) ? st[0] : (l == 1) ? st[1] : (l == 2) ? st[2] : st[3];
    }
    lds_barrier();

    // ---- tau: reached by at least `need` group maxima ---------------------------
    const uint32_t kmax = sh.kmax;
    if (sh.bad & 1u) return NIS_REJECT_NONFINITE;
    if (sh.bad) return NIS_REJECT_CAPACITY;
    if (kmax < kTFinite || kmax >= key32(INFINITY)) return NIS_REJECT_NONFINITE;
    const uint32_t need = min(topk + sh.hd, (uint32_t)kTNeed);
    const uint32_t enough = need + (need >> 2) + 16u;
    const float top = unkey32(kmax);
    float tau = -3.402823466e38f;
    bool whole = false;  // fewer groups than that: every finite element is a candidate
    if (need <= sh.nfin[0]) {
        tau = topk_search<4>(sh.hist[0], km, unkey32(sh.kmin[0]), top, need, enough);
    } else {
        // smaller groups: the maxima of a lane, of 4 groups, of one group (which
        // are searched when `need` is more than half of the maxima of 4)
        uint32_t n4 = 0u, n1 = 0u;
        float lo4 = INFINITY, lo1 = INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo4 = fminf(lo4, km[i] > -INFINITY ? km[i] : INFINITY);
            n4 += (uint32_t)__popcll(__ballot(km[i] > -INFINITY));
        }
#pragma unroll
        for (int i = 0; i < kTN; ++i) {
            lo1 = fminf(lo1, mx[i] > -INFINITY ? mx[i] : INFINITY);
            n1 += (uint32_t)__popcll(__ballot(mx[i] > -INFINITY));
        }
        const uint32_t kll = wmin_u32(ml > -INFINITY ? key32(ml) : 0xFFFFFFFFu);
        const uint32_t kl4 = wmin_u32(key32(lo4)), kl1 = wmin_u32(key32(lo1));
        const uint32_t nl = (uint32_t)__popcll(__ballot(ml > -INFINITY));
        if (l == 0) {
            atomicAdd(&sh.nfin[1], nl);
            atomicAdd(&sh.nfin[2], n4);
            atomicAdd(&sh.nfin[3], n1);
            atomicMin(&sh.kmin[1], kll);
            atomicMin(&sh.kmin[2], kl4);
            atomicMin(&sh.kmin[3], kl1);
        }
        lds_barrier();
        if (2u * need <= sh.nfin[2])
            tau = topk_search<4>(sh.hist[0], km, unkey32(need <= sh.nfin[1] ? sh.kmin[1] : sh.kmin[2]), top, need,
                                 enough);
        else if (need <= sh.nfin[3])
            tau = topk_search<kTN>(sh.hist[0], mx, unkey32(sh.kmin[3]), top, need, enough);
        else
            whole = true;
    }

    // ---- the groups reaching tau ---------------------------------------------------
    {
        uint32_t hits = 0u;  // bit kTN - 1 - i: the lane's group i
#pragma unroll
        for (int i = 0; i < kTN; ++i) hits = hits + hits + (mx[i] >= tau ? 1u : 0u);
        if (__ballot(hits != 0u)) {
            const uint32_t nh = (uint32_t)__popc(hits), incl = wscan_u32(nh);
            uint32_t at = 0u;
            if (l == 63) at = atomicAdd(&sh.ng, incl);
            at = bcast_u32(at, 63) + incl - nh;
            while (hits) {
                const int i = kTN - 32 + __clz((int)hits);
                hits &= ~(0x80000000u >> __clz((int)hits));
                if (at < (uint32_t)kTGl) sh.gl[at] = (uint32_t)(slot0 + 64 * G * i);
                ++at;
            }
        }
    }
    lds_barrier();
    const uint32_t ng = sh.ng;
    if (ng > (uint32_t)kTGl) return NIS_REJECT_CAPACITY;

    // ---- the candidates ---------------------------------------------------------------
    const double temp = fmax((double)a.temperature, 1e-6);  // sampler.rs:183
    // one append per wave of up to N entries per lane
    auto put = [&](auto& in, auto& v, auto& idx) {
        constexpr int N = (int)(sizeof(in) / sizeof(in[0]));
        uint64_t im[N];
        uint32_t tot = 0u;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            im[i] = __ballot(in[i]);
            tot += (uint32_t)__popcll(im[i]);
        }
        if (tot == 0u) return;
        uint32_t at = 0u;
        if (l == 0) at = atomicAdd(&sh.n, tot);
        at = bcast_u32(at, 0);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t pos = at + lane_rank(im[i]);
            if (in[i] && pos < (uint32_t)kTCap) {
                sh.cv[pos] = (double)v[i];
                sh.ci[pos] = (uint32_t)idx[i];
            }
            at += (uint32_t)__popcll(im[i]);
        }
    };
    auto free_id = [&](int idx) { return !pen || ((sh.bitmap[idx >> 5] >> (idx & 31)) & 1u) == 0u; };
    for (uint32_t b0 = 64u * (uint32_t)w; b0 < ng; b0 += (uint32_t)kTB) {
        const bool v = b0 + (uint32_t)l < ng;
        const int f0 = v ? (int)sh.gl[b0 + (uint32_t)l] : 0x1000000;
        // (a group ends with its wave's range)
        const int fe = (G == 1) ? f_hi : min(f_hi, 64 * cpw * (f0 / (64 * cpw) + 1) - 1);
        f4v xs[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int f = f0 + 64 * g;
            xs[g] = nis_buffer_load_f4(rsrc, (v && f >= f_lo && f <= fe) ? 16 * f : 0x7FFFFFF0, 0, 0);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int f = f0 + 64 * g;
            const bool in = v && f >= f_lo && f <= fe;
            bool hit[4];
            float hv[4];
            int hi[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                hv[q] = elem(xs[g], q);
                hi[q] = 4 * f + q - mis;
                hit[q] = in && hv[q] >= tau;
                if (hit[q]) hit[q] = free_id(hi[q]);
            }
            put(hit, hv, hi);
        }
    }
    if (w == 0) {
        bool hit[1] = {eon && ev >= tau};
        if (hit[0]) hit[0] = free_id(eidx);
        const float hv[1] = {ev};
        const int hi[1] = {eidx};
        put(hit, hv, hi);
    }
    if (pen && __ballot(own != 0u)) {
        const double wt = (double)tau / temp, penf = (double)a.penalty;
        bool hit[kPHist / kPB];
        double y[kPHist / kPB];
        bool inf = false;
        uint32_t kp = 0u;
#pragma unroll
        for (int i = 0; i < kPHist / kPB; ++i) {
            hit[i] = false;
            y[i] = 0.0;
            if (__ballot((own >> i) & 1u)) {
                const bool mine = (own >> i) & 1u;
                y[i] = pen_value(hx[i], penf);
                inf |= mine && !(y[i] < INFINITY);
                hit[i] = mine && y[i] > -INFINITY && y[i] / temp >= wt;
                if (hit[i]) kp = max(kp, key32((float)y[i]));
            }
        }
        kp = ~wmin_u32(~kp);
        if (l == 0 && kp) atomicMax(&sh.kpen, kp);
        if (__ballot(inf) && l == 0) atomicOr(&sh.bad, 1u);
        put(hit, y, hid);
    }
    lds_barrier();
    const uint32_t n = sh.n;
    if (sh.bad) return NIS_REJECT_NONFINITE;
    if (n == 0u) return NIS_REJECT_NONFINITE;
    // (fewer than k: the whole row listed, or a long history's bound cut at kTNeed)
    if (n > (uint32_t)kTCap || (n < topk && !whole)) return NIS_REJECT_CAPACITY;

    // ---- the final candidates: a few beyond the k-th at most -----------------------
    {
        double cv[kTCap / kTB];
        float cf[kTCap / kTB];  // the value in f32 (monotone)
#pragma unroll
        for (int i = 0; i < kTCap / kTB; ++i) {
            const uint32_t e = (uint32_t)(tid + kTB * i);
            cv[i] = -INFINITY;
            if (i == 0 || n > (uint32_t)(kTB * i)) cv[i] = e < n ? sh.cv[e] : -INFINITY;
            cf[i] = (float)cv[i];
        }
        // (the search's margin below its bucket also keeps the values that the
        // division by T could merge with the k-th)
        float t2 = -3.402823466e38f;
        const uint32_t enough2 = min(max(topk + (topk >> 3) + 8u, 64u), (uint32_t)kTFin);
        if (n > enough2)
            t2 = topk_search<kTCap / kTB>(sh.hist[1], cf, tau, unkey32(max(kmax, sh.kpen)), topk, enough2);
#pragma unroll
        for (int i = 0; i < kTCap / kTB; ++i) {
            if (i > 0 && n <= (uint32_t)(kTB * i)) break;
            const bool in = cf[i] >= t2;
            const uint64_t im = __ballot(in);
            if (im) {
                uint32_t at = 0u;
                if (l == 0) at = atomicAdd(&sh.m, (uint32_t)__popcll(im));
                at = bcast_u32(at, 0) + lane_rank(im);
                if (in && at < (uint32_t)kTFin) {
                    sh.ent[at].w = cv[i] / temp;  // sampler.rs:184-186
                    sh.ei[at] = sh.ci[tid + kTB * i];
                }
            }
        }
    }
    lds_barrier();
    const uint32_t m = sh.m;
    if (m > (uint32_t)kTFin) return NIS_REJECT_BUCKET;  // ties around the k-th
    if (w == 0 && l < 4) a.rng[4 * (int64_t)row + l] = rst;
    const bool topp_on = a.top_p > 0.0f && a.top_p < 1.0f;
    if (m <= 64u) {
        // a wave's worth: waves 0..3 (one per SIMD) each hold all candidates,
        // one per lane, and take a quarter of the pairs; wave 0 finishes
        constexpr int kPw = 4;
        if (w >= kPw) return NIS_REJECT_NONE;
        const bool in = l < (int)m;
        const double wq = in ? sh.ent[l].w : -INFINITY;
        const uint32_t iq = in ? sh.ei[l] : 0xFFFFFFFFu;
        const double wmax = wmax_f64(wq);
        const double eq = in ? exp(wq - wmax) : 0.0;  // sampler.rs:202
        const unsigned long long fq = (unsigned long long)(eq * kTFix + 0.5);
        uint32_t cnt = 0u;
        unsigned long long pre = 0ull;
#pragma unroll 4
        for (int t = w; t < (int)m; t += kPw) {
            const double wt = bcast_f64(wq, t);
            const uint32_t it = bcast_u32(iq, t);
            const unsigned long long ft = bcast_u64(fq, t);
            const bool gt = wt > wq;
            cnt += gt ? 1u : 0u;
            pre += (gt || (wt == wq && it < iq)) ? ft : 0ull;
        }
        sh.pcnt[tid] = cnt;
        sh.psum[tid] = pre;
        lds_barrier();
        if (w != 0) return NIS_REJECT_NONE;
#pragma unroll
        for (int q = 1; q < kPw; ++q) {
            cnt += sh.pcnt[64 * q + l];
            pre += sh.psum[64 * q + l];
        }
        const bool intop = in && cnt < topk;  // sampler.rs:112: w >= the k-th largest
        const unsigned long long zall = bcast_u64(wscan_u64(intop ? fq : 0ull), 63);
        // sampler.rs:150
        const bool kept = intop && (!topp_on || (double)((long long)pre - (long long)fq) <= (double)a.top_p * (double)zall);
        const unsigned long long fk = kept ? fq : 0ull;
        const unsigned long long zk = bcast_u64(wscan_u64(fk), 63);
        // the walk: the kept mass at or before each index
        unsigned long long cum = 0ull;
        uint64_t todo = __ballot(kept);
        const int m2 = __popcll(todo);
        while (todo) {
            const int t = __ffsll((long long)todo) - 1;
            todo &= todo - 1ull;
            cum += bcast_u32(iq, t) <= iq ? bcast_u64(fk, t) : 0ull;
        }
        const double u = sh.u;
        const double r = u * (double)zk;
        // the crossing (u = 0 stops the reference's walk at index 0)
        const bool hit = u == 0.0 ? l == 0 : (kept && (double)cum >= r && (double)(cum - fk) < r);
        if (hit) {
            const uint32_t tok = u == 0.0 ? 0u : iq;
            emit_token(a, row, tok);
            if (a.stats) {
                const double z = (double)zk / kTFix;
                write_row_stats(a, row, tok, NIS_PATH_DRAW, wmax, z, topp_on ? (double)zall / kTFix : 0.0, u,
                                u == 0.0 ? 0.0 : eq / z, (uint64_t)m2, 1);
            }
        }
        return NIS_REJECT_NONE;
    }
    const bool mine = tid < (int)m;
    const double wj = mine ? sh.ent[tid].w : -INFINITY;
    {
        const double wm = wmax_f64(wj);
        if (l == 0 && wm > -INFINITY) atomicMax(&sh.wmax, key64(wm));
    }
    lds_barrier();
    const double wmax = unkey64(sh.wmax);
    const double ej = mine ? exp(wj - wmax) : 0.0;  // sampler.rs:202
    const unsigned long long fj = (unsigned long long)(ej * kTFix + 0.5);
    if (mine) sh.ent[tid].fx = fj;
    const uint32_t ij = mine ? sh.ei[tid] : 0u;
    lds_barrier();

    // ---- every candidate: the strictly larger ones, the mass before it ------------
    const TPairs p1 = topk_pairs((int)m, w, l);
    {
        const bool in = p1.j < (int)m;
        const double wq = in ? sh.ent[p1.j].w : INFINITY;
        const uint32_t iq = in ? sh.ei[p1.j] : 0u;
        uint32_t cnt = 0u;
        unsigned long long pre = 0ull;
#pragma unroll 4
        for (int t = p1.t0; t < p1.t1; ++t) {
            const TEnt e = sh.ent[t];
            const uint32_t it = sh.ei[t];
            const bool gt = e.w > wq;
            cnt += gt ? 1u : 0u;
            pre += (gt || (e.w == wq && it < iq)) ? e.fx : 0ull;
        }
        sh.pcnt[p1.slot] = cnt;
        sh.psum[p1.slot] = pre;
    }
    lds_barrier();
    uint32_t cnt = 0u;
    unsigned long long pre = 0ull;
    if (mine)
        for (int q = 0; q < p1.tb; ++q) {
            cnt += sh.pcnt[q * 64 * p1.jb + tid];
            pre += sh.psum[q * 64 * p1.jb + tid];
        }
    const bool intop = mine && cnt < topk;  // sampler.rs:112: w >= the k-th largest
    {
        const unsigned long long z = bcast_u64(wscan_u64(intop ? fj : 0ull), 63);
        if (l == 0) sh.zred[0][w] = z;
    }
    lds_barrier();
    unsigned long long zall = 0ull, zk = 0ull;
#pragma unroll
    for (int i = 0; i < kTW; ++i) zall += sh.zred[0][i];
    // sampler.rs:150
    const bool kept = intop && (!topp_on || (double)((long long)pre - (long long)fj) <= (double)a.top_p * (double)zall);
    {
        const unsigned long long z = bcast_u64(wscan_u64(kept ? fj : 0ull), 63);
        const uint64_t im = __ballot(kept);
        uint32_t at = 0u;
        if (l == 0) {
            sh.zred[1][w] = z;
            if (im) at = atomicAdd(&sh.m2, (uint32_t)__popcll(im));
        }
        at = bcast_u32(at, 0) + lane_rank(im);
        if (kept) {
            sh.kfx[at] = fj;
            sh.ki[at] = ij;
        }
    }
    lds_barrier();

    // ---- the walk: each kept candidate's mass at or before its index -------------
    const int m2 = (int)sh.m2;
#pragma unroll
    for (int i = 0; i < kTW; ++i) zk += sh.zred[1][i];
    const TPairs p2 = topk_pairs(m2, w, l);
    {
        const uint32_t iq = p2.j < m2 ? sh.ki[p2.j] : 0u;
        unsigned long long s = 0ull;
#pragma unroll 4
        for (int t = p2.t0; t < p2.t1; ++t) s += sh.ki[t] <= iq ? sh.kfx[t] : 0ull;
        sh.psum[p2.slot] = s;
    }
    lds_barrier();
    if (tid < m2) {
        const unsigned long long fq = sh.kfx[tid];
        unsigned long long cum = 0ull;
        for (int q = 0; q < p2.tb; ++q) cum += sh.psum[q * 64 * p2.jb + tid];
        const double u = sh.u;
        const double r = u * (double)zk;
        const uint32_t iq = sh.ki[tid];
        // the crossing (u = 0 stops the reference's walk at index 0)
        const bool hit = u == 0.0 ? tid == 0 : ((double)cum >= r && (double)(cum - fq) < r);
        if (hit) {
            const uint32_t tok = u == 0.0 ? 0u : iq;
            emit_token(a, row, tok);
            if (a.stats) {
                const double z = (double)zk / kTFix;
                write_row_stats(a, row, tok, NIS_PATH_DRAW, wmax, z, topp_on ? (double)zall / kTFix : 0.0, u,
                                u == 0.0 ? 0.0 : ((double)fq / kTFix) / z, (uint64_t)m2, 1);
            }
        }
    }
    return NIS_REJECT_NONE;
}

}  // namespace nis
