// smallupd.h -- sort, heads, probe, plan and offsets of a small update batch
// in one workgroup (included by update.hip).
//
// The update pipeline's passes over tiles of a batch are launches of four to
// twelve microseconds each; below some thousands of triples the launches are the
// time (1,000 triples: 56 us of kernels and as much between them when there
// were nine; 5,000: 67 us).
// Here one workgroup of 1,024 threads
//   1. packs and sorts the triples in LDS: a key's bucket is its place between
//      the batch's smallest and largest key, buckets are counted by LDS
//      atomics and a key is ranked by (key, arrival) inside its own bucket, so
//      keys that spread over the range cost a few LDS accesses each; a batch
//      that crowds into few buckets (a few rows take it all) is sorted by a
//      stable 8-bit LSD radix sort of the same LDS arrays;
//   2. emits the coordinate and row records of the heads pass;
//   3. places every coordinate in its row by bisection (one lane each; a row is
//      not streamed, so its length costs a logarithm) and gives it its code;
//   4. takes the prefix sums, plans the rows and decides the batch.
// Up to SMALL_FUSED triples the steps are one launch (17 us for 1,000); above,
// steps 1 and 2 are (14 us for 3,000, 25 for 7,000), and the device-wide
// bisection, plan and offsets passes follow (5 + 4 + 5), because one CU's gathers
// (one line per clock) would take longer.  Above SMALL_MAX the tiled passes sort
// and emit in the time that this workgroup needs (a whole update: 72 us for 7,000
// here, 83 for 7,300 there, 105 for 10,000 in one workgroup).  Every array and
// DevState field is the pipeline's own, so the move, write and re-plan kernels
// that follow are the same.
#pragma once

constexpr int SU_TB = 1024;
constexpr int SU_NW = SU_TB / 64;
constexpr int64_t SMALL_FUSED = 2048;
constexpr int SU_IT_MAX = 7;                                // triples per thread
constexpr int64_t SMALL_MAX = (int64_t)SU_IT_MAX * SU_TB;
constexpr uint32_t SU_CROWD = 64;                           // keys per bucket before the radix sort takes over
constexpr int SU_RADIX_WORDS = SU_NW * 256;

struct SmallArgs {
    const int32_t *rows, *cols;
    const float *vals;
    uint32_t n;
    int64_t R, C;
    int cbits;
    unsigned long long pool_cap;
    DevState *ds;
    const uint32_t *row_start;
    const int32_t *row_len, *row_cap;
    const int32_t *pcol;
    const float *pval;
    int32_t *ucol;
    float *usum, *uval;
    uint32_t *ut, *upos, *ucode, *upre;
    uint32_t *trow, *tubeg, *trs, *tlen, *tcap, *tins, *tdel, *tnewl, *tmode, *tmoved, *tpre;
    uint32_t *mspan;
    uint64_t *rowt;
    uint32_t rtag;
};

template <int IT>
struct SmallLds {
    static constexpr int NB = SU_TB * (IT < 2 ? 2 : IT + (IT & 1));  // buckets: whole counter words per thread
    static constexpr int HW = NB / 2 + 2 > SU_RADIX_WORDS ? NB / 2 + 2 : SU_RADIX_WORDS;
    uint64_t key[IT * SU_TB];   // in bucket order (sorted after the radix sort)
    uint16_t arr[IT * SU_TB];   // arrival index of key[i]
    uint16_t perm[IT * SU_TB];  // sorted place -> i
    uint32_t hist[HW];          // 16-bit bucket counters / starts; radix counters
    uint64_t mm[NPLAN * SU_NW];
    uint32_t lw[SU_NW];
};

// Exclusive scan of one value per thread of the workgroup.
__device__ __forceinline__ uint32_t su_excl(uint32_t v, uint32_t *lw, uint32_t *total)
{
    const uint32_t inc = wave_incl_scan_u32(v);
    if (lane_id() == 63) lw[threadIdx.x >> 6] = inc;
    __syncthreads();
    uint32_t carry = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SU_NW; ++i) {
        const uint32_t t = lw[i];
        if (i < (int)(threadIdx.x >> 6)) carry += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return carry + inc - v;
}

// Exclusive prefix over the waves of a wave-uniform value; *total: their sum.
__device__ __forceinline__ uint32_t su_wave_excl(uint32_t v, uint32_t *lw, uint32_t *total)
{
    if (lane_id() == 0) lw[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t before = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SU_NW; ++i) {
        const uint32_t t = lw[i];
        if (i < (int)(threadIdx.x >> 6)) before += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return before;
}

// Workgroup totals of the plan counters: v[i] in thread i < NPLAN's lds[i].
__device__ __forceinline__ void su_sum_plan(const long long (&v)[NPLAN], uint64_t *lds)
{
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NPLAN; ++i) {
        const long long w = wave_sum_i64(v[i]);
        if (lane_id() == 0) lds[i * SU_NW + (threadIdx.x >> 6)] = (uint64_t)w;
    }
    __syncthreads();
    if (threadIdx.x < NPLAN) {
        uint64_t t = 0;
        for (int w = 0; w < SU_NW; ++w) t += lds[threadIdx.x * SU_NW + w];
        lds[threadIdx.x * SU_NW] = t;
    }
    __syncthreads();
}

// Stable LSD radix sort of key[0..n) (arrival order) with arr = 0..n-1 along,
// over the key bits below `bits`; in place: a pass holds its items in
// registers.  Wave w ranks the contiguous items from w * IT * 64.
template <int IT>
__device__ __forceinline__ void su_radix_sort(SmallLds<IT> &S, uint32_t n, int bits)
{
    const uint32_t lane = (uint32_t)lane_id(), w = threadIdx.x >> 6;
    const uint32_t wb = w * (IT * 64);
    const uint64_t lt = lanemask_lt();
    uint32_t(*cnt)[256] = reinterpret_cast<uint32_t(*)[256]>(S.hist);
    for (int shift = 0; shift < bits; shift += 8) {
        for (int i = threadIdx.x; i < SU_RADIX_WORDS; i += SU_TB) S.hist[i] = 0u;
        __syncthreads();
        uint64_t k[IT];
        uint32_t a[IT], rk[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const uint32_t i = wb + j * 64 + lane;
            k[j] = i < n ? S.key[i] : 0ull;
            a[j] = i < n ? S.arr[i] : 0u;
        }
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const bool ok = wb + j * 64 + lane < n;
            const uint32_t d = (uint32_t)(k[j] >> shift) & 255u;
            const uint64_t peers = wave_match_digit8(d, __ballot(ok));
            const int leader = __ffsll((long long)peers) - 1;
            // every lane of the digit reads its count before the leader adds
            // to it (a wave's LDS accesses complete in order)
            const uint32_t b = cnt[w][d];
            if (ok && (int)lane == leader) cnt[w][d] = b + (uint32_t)__popcll(peers);
            rk[j] = b + (uint32_t)__popcll(peers & lt);
        }
        __syncthreads();
        uint32_t c[SU_NW], sum = 0, tot;
        if (threadIdx.x < 256) {
#pragma unroll
            for (int i = 0; i < SU_NW; ++i) {
                c[i] = cnt[i][threadIdx.x];
                sum += c[i];
            }
        }
        uint32_t base = su_excl(sum, S.lw, &tot);
        if (threadIdx.x < 256) {
#pragma unroll
            for (int i = 0; i < SU_NW; ++i) {
                cnt[i][threadIdx.x] = base;
                base += c[i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            if (wb + j * 64 + lane >= n) continue;
            const uint32_t p = cnt[w][(uint32_t)(k[j] >> shift) & 255u] + rk[j];
            S.key[p] = k[j];
            S.arr[p] = (uint16_t)a[j];
        }
        __syncthreads();
    }
    for (uint32_t i = threadIdx.x; i < n; i += SU_TB) S.perm[i] = (uint16_t)i;
    __syncthreads();
}

// Steps 1 and 2.  Returns (every thread) whether the batch is valid; *nu and
// *nt receive its coordinates and touched rows.
template <int IT, bool FUSED>
__device__ __forceinline__ bool su_heads(const SmallArgs &A, SmallLds<IT> &S, uint32_t *nu, uint32_t *nt)
{
    constexpr uint32_t NB = SmallLds<IT>::NB;
    constexpr int BPT = NB / SU_TB;  // buckets per thread
    const uint32_t t = threadIdx.x, n = A.n;
    uint64_t k[IT];
    bool bad = false;
    {
        int32_t r[IT], c[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const uint32_t i = t + (uint32_t)j * SU_TB < n ? t + (uint32_t)j * SU_TB : n - 1;
            r[j] = A.rows[i];
            c[j] = A.cols[i];
        }
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            bad |= (r[j] < 0) | (r[j] >= A.R) | (c[j] < 0) | (c[j] >= A.C);
            k[j] = ((uint64_t)(uint32_t)r[j] << A.cbits) | (uint32_t)c[j];
        }
    }
    for (uint32_t i = t; i < NB / 2 + 2; i += SU_TB) S.hist[i] = 0u;
    *nu = *nt = 0;
    if (__syncthreads_or(bad)) return false;
    // the batch's key range
    uint64_t lo = ~0ull, hi = 0ull;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        lo = k[j] < lo ? k[j] : lo;
        hi = k[j] > hi ? k[j] : hi;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint64_t l2 = __shfl_xor((unsigned long long)lo, o), h2 = __shfl_xor((unsigned long long)hi, o);
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
    }
    if (lane_id() == 0) {
        S.mm[2 * (t >> 6)] = lo;
        S.mm[2 * (t >> 6) + 1] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SU_NW; ++i) {
        lo = S.mm[2 * i] < lo ? S.mm[2 * i] : lo;
        hi = S.mm[2 * i + 1] > hi ? S.mm[2 * i + 1] : hi;
    }
    // buckets: a float product is monotone in the key
    const float scale = (float)NB / ((float)(hi - lo) + 1.0f);
    uint32_t bo[IT];  // bucket, arrival in it << 16
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        bo[j] = 0;
        if (t + (uint32_t)j * SU_TB < n) {
            uint32_t b = (uint32_t)((float)(k[j] - lo) * scale);
            b = b < NB ? b : NB - 1;
            const uint32_t sh = (b & 1u) * 16u;
            bo[j] = b | (((atomicAdd(&S.hist[b >> 1], 1u << sh) >> sh) & 0xffffu) << 16);
        }
    }
    __syncthreads();
    uint32_t tot;
    {
        uint32_t w[BPT / 2], sum = 0;
#pragma unroll
        for (int i = 0; i < BPT / 2; ++i) {
            w[i] = S.hist[t * (BPT / 2) + i];
            sum += (w[i] & 0xffffu) + (w[i] >> 16);
        }
        uint32_t run = su_excl(sum, S.lw, &tot);
#pragma unroll
        for (int i = 0; i < BPT / 2; ++i) {
            const uint32_t a = run + (w[i] & 0xffffu);
            S.hist[t * (BPT / 2) + i] = run | (a << 16);
            run = a + (w[i] >> 16);
        }
        if (t == 0) S.hist[NB / 2] = n;
    }
    __syncthreads();
    const uint16_t *start = reinterpret_cast<const uint16_t *>(S.hist);
    uint32_t l[IT], cnt[IT], most = 0;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        l[j] = cnt[j] = 0;
        if (t + (uint32_t)j * SU_TB < n) {
            const uint32_t b = bo[j] & 0xffffu;
            l[j] = start[b];
            cnt[j] = start[b + 1] - l[j];
            most = cnt[j] > most ? cnt[j] : most;
        }
    }
    if (!__syncthreads_or(most > SU_CROWD)) {
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            if (t + (uint32_t)j * SU_TB < n) {
                S.key[l[j] + (bo[j] >> 16)] = k[j];
                S.arr[l[j] + (bo[j] >> 16)] = (uint16_t)(t + j * SU_TB);
            }
        }
        __syncthreads();
        uint32_t rk[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) rk[j] = l[j];
        for (uint32_t d = 0; __any(most > 1 && d < most); ++d) {
#pragma unroll
            for (int j = 0; j < IT; ++j) {
                if (d < cnt[j]) {
                    const uint64_t kk = S.key[l[j] + d];
                    rk[j] += (uint32_t)(kk < k[j] || (kk == k[j] && S.arr[l[j] + d] < t + (uint32_t)j * SU_TB));
                }
            }
        }
#pragma unroll
        for (int j = 0; j < IT; ++j)
            if (t + (uint32_t)j * SU_TB < n) S.perm[rk[j]] = (uint16_t)(l[j] + (bo[j] >> 16));
        __syncthreads();
    } else {
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const uint32_t i = t + (uint32_t)j * SU_TB;
            if (i < n) {
                S.key[i] = k[j];
                S.arr[i] = (uint16_t)i;
            }
        }
        __syncthreads();
        // keys differ only in the bits below the highest one of lo ^ hi
        su_radix_sort<IT>(S, n, lo == hi ? 0 : 64 - __clzll((long long)(lo ^ hi)));
    }
    // heads: wave w takes the sorted items from w * 64 * IT, 64 at a time, so
    // that ranks are ballot counts and the records leave in whole lines
    const uint32_t lane = (uint32_t)lane_id(), wb = (t >> 6) * (64 * IT);
    float vb[IT];
    uint64_t hm[IT], rm[IT];
    uint32_t hc = 0, rc = 0;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t p = wb + j * 64 + lane;
        const bool in = p < n;
        const uint32_t i = S.perm[in ? p : 0u];
        k[j] = S.key[i];
        const uint64_t prev = S.key[S.perm[in && p > 0 ? p - 1 : 0u]];
        vb[j] = A.vals[S.arr[i]];
        hm[j] = __ballot(in && (p == 0 || k[j] != prev));
        rm[j] = __ballot(in && (p == 0 || (k[j] >> A.cbits) != (prev >> A.cbits)));
        hc += (uint32_t)__popcll(hm[j]);
        rc += (uint32_t)__popcll(rm[j]);
    }
    uint32_t at = su_wave_excl(hc | (rc << 16), S.lw, &tot);
    uint32_t ub = at & 0xffffu, tb = at >> 16;
    const uint64_t lt = lanemask_lt(), le = lt | (1ull << lane);
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t r = (uint32_t)(k[j] >> A.cbits);
        const uint32_t u = ub + (uint32_t)__popcll(hm[j] & lt);
        const uint32_t tt = tb + (uint32_t)__popcll(rm[j] & le) - 1u;  // the last row head up to here
        if ((rm[j] >> lane) & 1u) {
            A.trow[tt] = r;
            A.tubeg[tt] = u;
            if constexpr (!FUSED) {
                A.tins[tt] = 0u;
                A.tdel[tt] = 0u;
            }
            if (A.rowt) A.rowt[r] = ((uint64_t)A.rtag << 32) | (uint64_t)tt;
        }
        if ((hm[j] >> lane) & 1u) {
            // duplicates left to right from 0, in arrival order
            float s = 0.0f + vb[j];
            for (uint32_t m = wb + j * 64 + lane + 1; m < n && S.key[S.perm[m]] == k[j]; ++m)
                s = s + A.vals[S.arr[S.perm[m]]];
            A.ucol[u] = (int32_t)(k[j] & ((1ull << A.cbits) - 1ull));
            A.usum[u] = s;
            A.ut[u] = tt;
        }
        ub += (uint32_t)__popcll(hm[j]);
        tb += (uint32_t)__popcll(rm[j]);
    }
    *nu = tot & 0xffffu;
    *nt = tot >> 16;
    if (t == 0) A.tubeg[tot >> 16] = tot & 0xffffu;
    return true;
}

// Step 3 for coordinates u0 + q * step < nu, PT of them.  FROM: where a row's
// pool start and length come from and what else is recorded.  P_FUSED: the row
// table; a row's first coordinate records its entry for step 4.  P_SPLIT: the
// same, and the rows' insert and delete counts for the plan pass.  P_TILES: the
// records of the heads pass, and the counts.
enum { P_FUSED, P_SPLIT, P_TILES };
template <int PT, int FROM>
__device__ __forceinline__ void su_probe(const SmallArgs &A, uint32_t u0, uint32_t step, uint32_t nu)
{
    uint32_t st[PT], len[PT], pos[PT], tq[PT], rq[PT], most = 0;
    int32_t want[PT];
    float sum[PT], old[PT];
    bool hit[PT];
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const uint32_t u = u0 + (uint32_t)q * step;
        st[q] = len[q] = pos[q] = 0;
        want[q] = 0;
        sum[q] = 0.0f;
        hit[q] = false;
        tq[q] = rq[q] = 0;
        if (u < nu) {
            tq[q] = A.ut[u];
            want[q] = A.ucol[u];
            sum[q] = A.usum[u];
        }
    }
    if constexpr (FROM == P_TILES) {
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            if (u0 + (uint32_t)q * step < nu) {
                st[q] = A.trs[tq[q]];
                len[q] = A.tlen[tq[q]];
            }
        }
    } else {
        uint32_t first[PT];
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            first[q] = ~0u;
            if (u0 + (uint32_t)q * step < nu) {
                rq[q] = A.trow[tq[q]];
                first[q] = A.tubeg[tq[q]];
            }
        }
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const uint32_t u = u0 + (uint32_t)q * step;
            if (u < nu) {
                st[q] = A.row_start[rq[q]];
                len[q] = (uint32_t)A.row_len[rq[q]];
                rq[q] = first[q] == u ? (uint32_t)A.row_cap[rq[q]] : 0u;
            }
        }
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            if (first[q] == u0 + (uint32_t)q * step) {
                A.trs[tq[q]] = st[q];
                A.tlen[tq[q]] = len[q];
                A.tcap[tq[q]] = rq[q];
            }
        }
    }
#pragma unroll
    for (int q = 0; q < PT; ++q) most = len[q] > most ? len[q] : most;
    // every round leaves at most half of the longest row
    for (; __any(most > 0); most >>= 1) {
        int32_t c[PT];
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            c[q] = 0;
            if (len[q]) c[q] = A.pcol[(uint64_t)st[q] + (pos[q] + (len[q] >> 1))];
        }
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const uint32_t half = len[q] >> 1;
            const bool below = len[q] && c[q] < want[q];
            hit[q] = hit[q] || (len[q] && c[q] == want[q]);
            pos[q] = below ? pos[q] + half + 1 : pos[q];
            len[q] = below ? len[q] - half - 1 : half;
        }
    }
#pragma unroll
    for (int q = 0; q < PT; ++q) old[q] = hit[q] ? A.pval[(uint64_t)st[q] + pos[q]] : 0.0f;
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const uint32_t u = u0 + (uint32_t)q * step;
        float v = sum[q];
        uint32_t code = C_NOP;
        if (u < nu) {
            if (hit[q]) {
                v = old[q] + v;
                code = v != 0.0f ? C_ADD : C_DEL;
            } else {
                code = v != 0.0f ? C_INS : C_NOP;
            }
            A.uval[u] = v;
            A.upos[u] = pos[q];
            A.ucode[u] = code;
        }
        if constexpr (FROM != P_FUSED) {
            // the wave's coordinates are in row order: the first one of a row adds
            // the row's counts.  One atomic per coordinate took 5,583 us where
            // 500,000 of them fall into four rows (93 so) and 117 for 10,000 (6)
            static_assert(PT == 1, "a wave's coordinates are consecutive");
            const int lane = lane_id();
            const uint32_t before = (uint32_t)__shfl_up((int)tq[q], 1);
            const uint64_t heads = __ballot(u < nu && (lane == 0 || before != tq[q]));
            const uint64_t im = __ballot(code == C_INS), dm = __ballot(code == C_DEL);
            if ((heads >> lane) & 1u) {
                const uint64_t next = heads & ~((2ull << lane) - 1ull);
                const uint64_t own = (next ? (next & (0ull - next)) - 1ull : ~0ull) & ~((1ull << lane) - 1ull);
                const uint32_t ni = (uint32_t)__popcll(im & own), nd = (uint32_t)__popcll(dm & own);
                if (ni) atomicAdd(&A.tins[tq[q]], ni);
                if (nd) atomicAdd(&A.tdel[tq[q]], nd);
            }
        }
    }
}

// Step 4 (the plan, offsets and decision kernels' work).
template <int IT>
__device__ __forceinline__ void su_plan(const SmallArgs &A, uint32_t nu, uint32_t nt, uint32_t *lw, uint64_t *lds64)
{
    const uint32_t t = threadIdx.x, lane = (uint32_t)lane_id(), wb = (t >> 6) * (64 * IT);
    const uint64_t lt = lanemask_lt();
    uint32_t c = 0, nadd = 0, tot;
    uint64_t im[IT], dm[IT];
    {
        uint32_t code[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const uint32_t e = wb + j * 64 + lane;
            code[j] = e < nu ? A.ucode[e] : (uint32_t)C_NOP;
        }
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            im[j] = __ballot(code[j] == C_INS);
            dm[j] = __ballot(code[j] == C_DEL);
            c += (uint32_t)__popcll(im[j]) + ((uint32_t)__popcll(dm[j]) << 16);
            nadd += (uint32_t)__popcll(__ballot(code[j] == C_ADD));
        }
    }
    const uint32_t at = su_wave_excl(c, lw, &tot);
    const uint32_t ins_total = tot & 0xffffu, del_total = tot >> 16;
    uint2 *upre = reinterpret_cast<uint2 *>(A.upre);
    uint32_t ib = at & 0xffffu, db = at >> 16;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t e = wb + j * 64 + lane;
        if (e < nu) upre[e] = make_uint2(ib + (uint32_t)__popcll(im[j] & lt), db + (uint32_t)__popcll(dm[j] & lt));
        ib += (uint32_t)__popcll(im[j]);
        db += (uint32_t)__popcll(dm[j]);
    }
    if (t == 0) upre[nu] = make_uint2(ins_total, del_total);
    (void)su_wave_excl(nadd, lw, &nadd);  // its barriers also publish upre to the workgroup
    uint32_t L[IT], cap[IT], claim[IT], csum = 0, msum = 0;
    uint2 a[IT], b[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t e = wb + j * 64 + lane;
        L[j] = cap[j] = 0;
        a[j] = b[j] = make_uint2(0u, 0u);
        if (e < nt) {
            L[j] = A.tlen[e];
            cap[j] = A.tcap[e];
            a[j] = upre[A.tubeg[e]];
            b[j] = upre[A.tubeg[e + 1]];
        }
    }
    long long v[NPLAN] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t e = wb + j * 64 + lane;
        const uint32_t ni = b[j].x - a[j].x, nd = b[j].y - a[j].y;
        const uint32_t nl = L[j] + ni - nd;
        const bool rewrite = e < nt && (ni | nd) != 0u;
        uint32_t moved = 0;
        claim[j] = 0;
        if (rewrite) {
            claim[j] = chunk_round(nl);
            moved = L[j];
            const int hub_now = nl > DCSR_HUB_LEN, hub_was = L[j] > DCSR_HUB_LEN;
            v[0] += (long long)nl - (long long)L[j];
            v[1] += (long long)cap[j];
            v[2] += hub_now - hub_was;
            v[3] += (hub_now ? ((long long)nl + DCSR_HUB_CHUNK - 1) / DCSR_HUB_CHUNK : 0) -
                    (hub_was ? ((long long)L[j] + DCSR_HUB_CHUNK - 1) / DCSR_HUB_CHUNK : 0);
            v[4] += hub_now | hub_was;
        }
        if (e < nt) {
            A.tins[e] = ni;
            A.tdel[e] = nd;
            A.tnewl[e] = nl;
            A.tmode[e] = rewrite ? M_REWRITE : M_VALUES;
            A.tmoved[e] = moved;
        }
        L[j] = moved;
        // the wave's prefixes; its base follows
        const uint32_t ci = wave_incl_scan_u32(claim[j]), mi = wave_incl_scan_u32(moved);
        claim[j] = csum + ci - claim[j];
        cap[j] = msum + mi - moved;
        csum += wave_read_lane_u32(ci, 63);
        msum += wave_read_lane_u32(mi, 63);
    }
    uint32_t claim_total, moved_total;
    const uint32_t cb = su_wave_excl(csum, lw, &claim_total);
    const uint32_t mb = su_wave_excl(msum, lw, &moved_total);
    uint2 *tpre = reinterpret_cast<uint2 *>(A.tpre);
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t e = wb + j * 64 + lane;
        if (e >= nt) continue;
        const uint32_t sm = mb + cap[j];
        tpre[e] = make_uint2(cb + claim[j], sm);
        if (A.mspan)
            for (uint32_t k = (sm + MV_SPAN - 1u) / MV_SPAN; k * MV_SPAN < sm + L[j]; ++k) A.mspan[k] = e;
    }
    su_sum_plan(v, lds64);
    if (t == 0) {
        tpre[nt] = make_uint2(claim_total, moved_total);
        DevState *ds = A.ds;
        ds->claim_total = claim_total;
        ds->nrewrite_old = moved_total;
        ds->n_ins = ins_total;
        ds->n_add = nadd;
        ds->n_del = del_total;
        ds->d_nnz = (long long)lds64[0];
        ds->d_garbage = (long long)lds64[SU_NW];
        ds->d_hubs = (long long)lds64[2 * SU_NW];
        ds->d_hub_chunks = (long long)lds64[3 * SU_NW];
        ds->hub_touch = (unsigned)lds64[4 * SU_NW];
        const unsigned long long base = ds->bump;  // claims start at the current bump
        ds->need = claim_total;
        ds->bump_saved = base;
        ds->ubad_last = 0;
        const bool go = base + claim_total <= A.pool_cap;
        ds->go = go ? 1u : 0u;
        if (go) ds->bump = base + claim_total;
    }
}

// FUSED: all steps.  Else steps 1 and 2; a batch with an index outside the
// matrix goes on without coordinates to the decision, which rejects it.
template <int IT, bool FUSED>
__global__ __launch_bounds__(SU_TB) void k_upd_small(SmallArgs A)
{
    __shared__ SmallLds<IT> S;
    uint32_t nu, nt;
    const bool ok = su_heads<IT, FUSED>(A, S, &nu, &nt);
    if (threadIdx.x == 0) {
        A.ds->nuniq = ok ? nu : 0u;
        A.ds->ntouched = ok ? nt : 0u;
        if constexpr (FUSED) {
            A.ds->ubad = 0;
            A.ds->ubad_last = ok ? 0 : 1;
            if (!ok) {  // rejected whole
                A.ds->nrewrite_old = 0;
                A.ds->go = 0;
            }
        } else {
            A.ds->ubad = ok ? 0 : 1;
        }
    }
    if constexpr (FUSED) {
        if (!ok) return;
        __syncthreads();
        su_probe<IT, P_FUSED>(A, threadIdx.x, SU_TB, nu);
        __syncthreads();
        su_plan<IT>(A, nu, nt, S.lw, S.mm);
    }
}

template <int FROM>
__global__ __launch_bounds__(TB) void k_upd_bisect(SmallArgs A)
{
    su_probe<1, FROM>(A, blockIdx.x * TB + threadIdx.x, 0u, A.ds->nuniq);
}
