// batch.hip -- many small DCSR matrices updated and multiplied in one
// persistent launch.
//
// No reference counterpart: the reference handles one matrix at a time with
// a process-global bin table (include/Matrix_Test.h:57, include/load.h:606).
// The matrices of a batch live block-diagonally in one DCSR handle (matrix m
// owns global rows [row_base[m], row_base[m+1]) and keeps local column
// indices), so they share one pool and one allocator.  One persistent kernel
// does a whole step: every workgroup takes matrix ids from a work counter and,
// for each, applies that matrix's insert-or-add batch with all of its records
// in LDS (triples bucketed by row and ranked inside their row, left-to-right
// duplicate sums, each touched row met by 16 lanes that hold its entries in
// registers, prefix-sum chunk claims, merge into the new chunk, commit), then
// computes that matrix's SpMV with TEAM lanes per row and a whole wave for
// rows longer than a threshold.  Semantics per matrix are those of
// dcsr_update followed by dcsr_spmv.  The last workgroup to finish resets the
// counter, so the launch can be captured in a hipGraph and replayed.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <map>
#include <vector>
#include "dcsr_internal.h"
#include "prims.h"
#include "wave.h"

namespace {

// 16 waves and 73 KB of LDS: two workgroups fill a CU's waves.  A matrix is a
// chain of short phases with a barrier between them, so what bounds a step is
// how many rows are in flight per CU: 4,096 matrices (4.0M rows, 68M entries,
// 2,000 triples each) take 0.91 ms per step; 4 waves per matrix with the records
// in memory and one lane per touched row took 2.44.  Everything is inlined: as a
// function the update spilled its registers through memory (1.31 ms).
constexpr int BT = 1024;
constexpr int NW = BT / 64;
constexpr uint32_t BMAX = 4096;  // triples per matrix per step
constexpr int KB = 12;           // bits of a local row / column / arrival index
constexpr uint32_t LMAX = 1u << KB;
constexpr int PT = BMAX / BT;    // records per thread
// Triples of one row before the batch is sorted by digits instead of ranked inside
// its rows, a round per triple of the fullest.  600 matrices, two steps: 4,096
// triples at one coordinate 6,554 -> 1,648 us, 1,000 in one row 1,885 -> 1,214; 100 in
// one row 409 -> 404.  Limits of 16 to 128 differ by less than the runs do.
constexpr uint32_t BT_CROWD = 64;
constexpr int RL = 16;           // lanes per touched row
constexpr int NTM = BT / RL;     // rows in flight per workgroup
constexpr int RC = 2 * RL;       // entries of a row met at once (two per lane)
static_assert(BMAX == LMAX && PT % 2 == 0, "row counters and records share their split over the threads");
enum { C_NOP = 0, C_ADD = 1, C_DEL = 2, C_INS = 3 };

enum { SM_CROWD = 0, SM_OK, SM_BASE, SM_INS, SM_ADD, SM_DEL, SM_LONG, SM_WORDS };
// A workgroup's records.  Reused in order: buckets -> coordinates; sorted keys
// -> positions and codes, new row lengths; sorted values -> chunk offsets; row
// counters -> row starts in the buckets -> first coordinate of each row.
struct BatchLds {
    uint32_t urc[BMAX];  // bucketed column << 12 | arrival; then coordinate u: row << 12 | column
    uint32_t sk[BMAX];   // sorted row << 12 | column; then upc and tnl
    float sv[BMAX];      // sorted values; then tdst
    float uval[BMAX];    // coordinate u: sum, then new value
    uint32_t cnt[BMAX / 2 + 2];  // 16-bit: triples of each row, bucket starts; then tub
    uint32_t done[LMAX / 32];    // rows whose product the update has written
    uint32_t lw[NW];
    uint32_t sm[SM_WORDS];
    uint32_t next;
    // coordinate u: position in its old row | code << 14
    __device__ uint16_t *upc() { return reinterpret_cast<uint16_t *>(sk); }
    // touched row t: new length | rewritten << 15
    __device__ uint16_t *tnl() { return reinterpret_cast<uint16_t *>(sk) + BMAX; }
    // touched row t: its chunk's offset in the matrix's claim
    __device__ uint32_t *tdst() { return reinterpret_cast<uint32_t *>(sv); }
    // touched row t: first coordinate (t == touched rows: their count)
    __device__ uint16_t *tub() { return reinterpret_cast<uint16_t *>(cnt); }
};

struct BatchState {
    unsigned int work;  // next matrix id
    unsigned int done;  // workgroups finished
};

#define BST_BAD_INDEX 0x1u
#define BST_TOO_BIG 0x2u
#define BST_EXHAUSTED 0x4u

// Block-wide exclusive scan of one value per thread; *total receives the sum.
__device__ __forceinline__ uint32_t block_excl(uint32_t v, uint32_t *lw, uint32_t *total)
{
    const uint32_t inc = wave_incl_scan_u32(v);
    if (lane_id() == 63) lw[threadIdx.x >> 6] = inc;
    __syncthreads();
    uint32_t carry = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const uint32_t t = lw[i];
        if (i < (int)(threadIdx.x >> 6)) carry += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return carry + inc - v;
}

// Stable sort of the nb keys in S.sk (below 2^24, in arrival order) with S.sv
// along: LSD passes of 8 bits in place, a pass's records in registers, wave w
// ranking those from w * 64 * PT.  The 16-bit counters of every wave and digit
// lie in S.cnt.  The caller has synchronized.
__device__ __forceinline__ void batch_radix_sort(BatchLds &S, uint32_t nb)
{
    static_assert(NW * 256 <= 2 * (BMAX / 2 + 2), "the counters fit the row counters");
    uint16_t *cnt = reinterpret_cast<uint16_t *>(S.cnt);
    // opaque to the compiler: what follows from it is computed here, not kept in
    // registers across the matrices (18 registers spilled, not 22)
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const uint32_t lane = t & 63u, w = t >> 6, wb = w * (64 * PT);
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll 1
    for (int shift = 0; shift < 2 * KB; shift += 8) {
        for (uint32_t i = t; i < NW * 128; i += BT) S.cnt[i] = 0u;
        __syncthreads();
#pragma unroll 1
        for (uint32_t i = wb + lane; i < wb + 64 * PT; i += 64) {
            const bool ok = i < nb;
            const uint32_t d = ok ? (S.sk[i] >> shift) & 255u : 0u;
            const uint64_t peers = wave_match_digit8(d, __ballot(ok));
            const int leader = __ffsll((long long)peers) - 1;
            const uint32_t b = cnt[w * 256 + d];
            if (ok && (int)lane == leader) cnt[w * 256 + d] = (uint16_t)(b + (uint32_t)__popcll(peers));
            S.urc[i] = b + (uint32_t)__popcll(peers & lt);
        }
        __syncthreads();
        uint32_t sum = 0, tot;
        if (t < 256)
#pragma unroll 1
            for (int i = 0; i < NW; ++i) sum += cnt[i * 256 + t];
        uint32_t base = block_excl(sum, S.lw, &tot);
        if (t < 256) {
#pragma unroll 1
            for (int i = 0; i < NW; ++i) {
                const uint32_t c = cnt[i * 256 + t];
                cnt[i * 256 + t] = (uint16_t)base;
                base += c;
            }
        }
        __syncthreads();
        uint32_t k[PT], p[PT];
        float v[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t i = wb + (uint32_t)j * 64 + lane;
            k[j] = S.sk[i];
            v[j] = S.sv[i];
            p[j] = cnt[w * 256 + ((k[j] >> shift) & 255u)] + S.urc[i];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            if (wb + (uint32_t)j * 64 + lane >= nb) continue;
            S.sk[p[j]] = k[j];
            S.sv[p[j]] = v[j];
        }
        __syncthreads();
    }
}

// Counters of the matrices one workgroup updated, kept by its thread 0 and
// added to the device state once when the workgroup is done (one atomic per
// counter and workgroup instead of per matrix).
struct BatchAcc {
    long long dnnz, dgarbage;
    unsigned long long ins, add, del;
    uint32_t touched;
};

// Update of matrix m inside one workgroup.  Returns nothing; status bits go
// to mstat[m].  reserved: the host has made room in the pool for every
// matrix's largest claim, so claims take a plain atomic add; otherwise a
// compare-and-swap that advances the bump pointer only when the claim fits.
__device__ __forceinline__ void batch_update(uint32_t m, const uint32_t *__restrict__ row_base, const uint32_t *__restrict__ col_base,
                             const int64_t *__restrict__ tri_off, int64_t ntri, const int32_t *__restrict__ trow,
                             const int32_t *__restrict__ tcol, const float *__restrict__ tval,
                             uint32_t *__restrict__ row_start, int32_t *__restrict__ row_len,
                             int32_t *__restrict__ row_cap, int32_t *__restrict__ pcol, float *__restrict__ pval,
                             unsigned long long pool_cap, DevState *ds, uint32_t *__restrict__ mstat,
                             const float *__restrict__ x, float *__restrict__ y, BatchLds &S, bool reserved,
                             BatchAcc &acc)
{
    const uint32_t t = threadIdx.x;
    const uint32_t gbase = row_base[m];
    const uint32_t Rm = row_base[m + 1] - gbase;
    const uint32_t Cm = col_base[m + 1] - col_base[m];
    const int64_t t0 = tri_off[m];
    const int64_t t1 = tri_off[m + 1];
    if (t0 < 0 || t1 < t0 || t1 > ntri) {  // offsets outside the triple arrays
        if (t == 0) mstat[m] |= BST_BAD_INDEX;
        return;
    }
    const int64_t nb64 = t1 - t0;
    if (nb64 == 0) return;
    if (nb64 > (int64_t)BMAX) {
        if (t == 0) mstat[m] |= BST_TOO_BIG;
        return;
    }
    const uint32_t nb = (uint32_t)nb64;
    // U1: sort the triples by (row, column, arrival).  Row counters in LDS
    // give every triple a place in its row's bucket, in any order; its rank
    // among the bucket's (column, arrival) pairs is its sorted place.  A
    // thread's triples are all loaded before the first LDS access; indices
    // clamp to the matrix's last triple.
    int32_t rr[PT], cc[PT];
    float vv[PT];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const uint32_t i = t + (uint32_t)j * BT;
        const int64_t gi = t0 + (i < nb ? i : nb - 1);
        rr[j] = trow[gi];
        cc[j] = tcol[gi];
        vv[j] = tval[gi];
    }
    for (uint32_t i = t; i < BMAX / 2 + 2; i += BT) S.cnt[i] = 0u;
    if (t < SM_WORDS) S.sm[t] = 0u;
    __syncthreads();
    uint32_t off[PT];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const int32_t r = rr[j], c = cc[j];
        off[j] = 0;
        if (t + (uint32_t)j * BT >= nb) continue;
        if (r < 0 || (uint32_t)r >= Rm || c < 0 || (uint32_t)c >= Cm) {
            bad = true;
        } else {
            const uint32_t sh = ((uint32_t)r & 1u) * 16u;
            off[j] = (atomicAdd(&S.cnt[(uint32_t)r >> 1], 1u << sh) >> sh) & 0xffffu;
            if (off[j] == BT_CROWD) S.sm[SM_CROWD] = 1u;
        }
    }
    if (__syncthreads_or(bad)) {
        if (t == 0) mstat[m] |= BST_BAD_INDEX;
        return;
    }
    uint32_t tot;
    if (S.sm[SM_CROWD]) {
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t i = t + (uint32_t)j * BT;
            if (i < nb) {
                S.sk[i] = ((uint32_t)rr[j] << KB) | (uint32_t)cc[j];
                S.sv[i] = vv[j];
            }
        }
        __syncthreads();
        batch_radix_sort(S, nb);
    } else {
        // bucket starts: PT rows (two to a counter word) per thread
        {
            uint32_t w[PT / 2], sum = 0;
#pragma unroll
            for (int i = 0; i < PT / 2; ++i) {
                w[i] = S.cnt[t * (PT / 2) + i];
                sum += (w[i] & 0xffffu) + (w[i] >> 16);
            }
            uint32_t b = block_excl(sum, S.lw, &tot);
#pragma unroll
            for (int i = 0; i < PT / 2; ++i) {
                const uint32_t a = b + (w[i] & 0xffffu);
                S.cnt[t * (PT / 2) + i] = b | (a << 16);
                b = a + (w[i] >> 16);
            }
            if (t == 0) S.cnt[BMAX / 2] = nb;
        }
        __syncthreads();
        const uint16_t *start = reinterpret_cast<const uint16_t *>(S.cnt);
        uint32_t lo[PT], n[PT], me[PT], most = 0;
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t i = t + (uint32_t)j * BT;
            lo[j] = n[j] = me[j] = 0;
            if (i < nb) {
                lo[j] = start[rr[j]];
                n[j] = start[rr[j] + 1] - lo[j];
                me[j] = ((uint32_t)cc[j] << KB) | i;
                S.urc[lo[j] + off[j]] = me[j];
                most = n[j] > most ? n[j] : most;
            }
        }
        __syncthreads();
        uint32_t rk[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) rk[j] = lo[j];
        for (uint32_t d = 0; __any(most > 1 && d < most); ++d) {
#pragma unroll
            for (int j = 0; j < PT; ++j)
                if (d < n[j]) rk[j] += (uint32_t)(S.urc[lo[j] + d] < me[j]);
        }
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            if (t + (uint32_t)j * BT < nb) {
                S.sk[rk[j]] = ((uint32_t)rr[j] << KB) | (uint32_t)cc[j];
                S.sv[rk[j]] = vv[j];
            }
        }
        __syncthreads();
    }
    // U2: distinct coordinates (heads) and touched rows (row heads), four
    // consecutive records per thread; duplicates are summed from 0 in arrival
    // order
    uint32_t nu, nt;
    {
        const uint32_t p0 = t * PT;
        uint32_t k[PT], h = 0, rh = 0;
        uint32_t prev = p0 > 0 && p0 - 1 < nb ? S.sk[p0 - 1] : ~0u;
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            k[j] = p0 + j < nb ? S.sk[p0 + j] : ~0u;
            if (p0 + j < nb && k[j] != prev) h |= 1u << j;
            if (p0 + j < nb && (prev == ~0u || (k[j] >> KB) != (prev >> KB))) rh |= 1u << j;
            prev = k[j];
        }
        uint32_t at = block_excl((uint32_t)__popc(h) | ((uint32_t)__popc(rh) << 16), S.lw, &tot);
        nu = tot & 0xffffu;
        nt = tot >> 16;
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            if ((h >> j) & 1u) {
                float s = 0.0f + S.sv[p0 + j];
                for (uint32_t q = p0 + j + 1; q < nb && S.sk[q] == k[j]; ++q) s = s + S.sv[q];
                const uint32_t u = at & 0xffffu;
                S.urc[u] = k[j];
                S.uval[u] = s;
                if ((rh >> j) & 1u) {
                    S.tub()[at >> 16] = (uint16_t)u;
                    at += 1u << 16;
                }
                ++at;
            }
        }
        if (t == 0) S.tub()[nt] = (uint16_t)nu;
    }
    __syncthreads();
    // U3: one lane per coordinate finds its place among its row's columns (a
    // bisection in memory: the first probe brings the row's line, the others
    // hit it) and the old value of a match; its code and new value follow
    uint16_t *upc = S.upc();
    const uint16_t *tub = S.tub();
    uint32_t nins = 0, nadd = 0, ndel = 0;
    {
        uint32_t k[PT], st[PT], pos[PT], len[PT], most_len = 0;
        bool hit[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t u = t + (uint32_t)j * BT;
            k[j] = u < nu ? S.urc[u] : 0u;
            st[j] = pos[j] = len[j] = 0;
            hit[j] = false;
            if (u < nu) {
                st[j] = row_start[gbase + (k[j] >> KB)];
                len[j] = (uint32_t)row_len[gbase + (k[j] >> KB)];
            }
        }
#pragma unroll
        for (int j = 0; j < PT; ++j) most_len = len[j] > most_len ? len[j] : most_len;
        // every round leaves at most half of the longest row
        for (; __any(most_len > 0); most_len >>= 1) {
            int32_t c[PT];
#pragma unroll
            for (int j = 0; j < PT; ++j) {
                c[j] = 0;
                if (len[j]) c[j] = pcol[(uint64_t)st[j] + (pos[j] + (len[j] >> 1))];
            }
#pragma unroll
            for (int j = 0; j < PT; ++j) {
                const int32_t want = (int32_t)(k[j] & (LMAX - 1));
                const uint32_t half = len[j] >> 1;
                const bool below = len[j] && c[j] < want;
                hit[j] = hit[j] || (len[j] && c[j] == want);
                pos[j] = below ? pos[j] + half + 1 : pos[j];
                len[j] = below ? len[j] - half - 1 : half;
            }
        }
        float old[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) old[j] = hit[j] ? pval[(uint64_t)st[j] + pos[j]] : 0.0f;
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t u = t + (uint32_t)j * BT;
            if (u >= nu) continue;
            float v = S.uval[u];
            uint32_t code;
            if (hit[j]) {
                v = old[j] + v;
                code = v != 0.0f ? C_ADD : C_DEL;
            } else {
                code = v != 0.0f ? C_INS : C_NOP;
            }
            S.uval[u] = v;
            upc[u] = (uint16_t)(pos[j] | (code << 14));
            nins += code == C_INS;
            nadd += code == C_ADD;
            ndel += code == C_DEL;
        }
    }
    const uint32_t tm = t / RL, tl = t % RL;
    auto row_of = [&](uint32_t tt) { return gbase + (S.urc[tub[tt]] >> KB); };
    nins = wave_sum_u32(nins);
    nadd = wave_sum_u32(nadd);
    ndel = wave_sum_u32(ndel);
    if (lane_id() == 0) {
        atomicAdd(&S.sm[SM_INS], nins);
        atomicAdd(&S.sm[SM_ADD], nadd);
        atomicAdd(&S.sm[SM_DEL], ndel);
    }
    __syncthreads();
    // U4: plan and claim, four consecutive rows per thread
    uint16_t *tnl = S.tnl();
    uint32_t *tdst = S.tdst();
    uint32_t dgar = 0, claim_tot;
    {
        uint32_t claim[PT], sum = 0;
        uint32_t L[PT], cap[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t tt = t * PT + j;
            L[j] = cap[j] = 0;
            if (tt < nt) {
                const uint32_t g = row_of(tt);
                L[j] = (uint32_t)row_len[g];
                cap[j] = (uint32_t)row_cap[g];
            }
        }
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t tt = t * PT + j;
            claim[j] = 0;
            if (tt < nt) {
                // a coordinate's place becomes its place in the new row: the
                // inserts less the deletes before it in the row shift it
                uint32_t ni = 0, nd = 0;
                for (uint32_t u = tub[tt], ue = tub[tt + 1]; u < ue; ++u) {
                    const uint32_t w = upc[u], code = w >> 14;
                    upc[u] = (uint16_t)(w + ni - nd);
                    ni += code == C_INS;
                    nd += code == C_DEL;
                }
                const uint32_t nl = L[j] + ni - nd;
                tnl[tt] = (uint16_t)(nl | ((ni | nd) ? 0x8000u : 0u));
                if (ni | nd) {
                    claim[j] = chunk_round(nl);
                    dgar += cap[j];
                }
            }
            sum += claim[j];
        }
        uint32_t at = block_excl(sum, S.lw, &claim_tot);
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            if (t * PT + j < nt) tdst[t * PT + j] = at;
            at += claim[j];
        }
    }
    uint32_t dg;
    (void)block_excl(dgar, S.lw, &dg);
    if (t == 0) {
        // claim by compare-and-swap: the bump pointer advances only when the
        // claim fits, so a matrix that does not fit leaves room for later
        // (smaller) matrices of the same step
        unsigned long long base = 0ull;
        bool ok = true;
        if (claim_tot && reserved) {
            base = atomicAdd(&ds->bump, (unsigned long long)claim_tot);
        } else if (claim_tot) {
            unsigned long long cur = __hip_atomic_load(&ds->bump, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (;;) {
                if (cur + claim_tot > pool_cap) {
                    ok = false;
                    break;
                }
                const unsigned long long seen = atomicCAS(&ds->bump, cur, cur + claim_tot);
                if (seen == cur) {
                    base = cur;
                    break;
                }
                cur = seen;  // another matrix claimed first: retry from its end
            }
        }
        S.sm[SM_OK] = ok ? 1u : 0u;
        S.sm[SM_BASE] = (uint32_t)base;
        if (!ok) mstat[m] |= BST_EXHAUSTED;
        if (ok) {
            acc.dnnz += (long long)S.sm[SM_INS] - (long long)S.sm[SM_DEL];
            acc.dgarbage += (long long)dg;
            acc.ins += S.sm[SM_INS];
            acc.add += S.sm[SM_ADD];
            acc.del += S.sm[SM_DEL];
            acc.touched += nt;
        }
    }
    __syncthreads();
    if (!S.sm[SM_OK]) return;
    const uint32_t base = S.sm[SM_BASE];
    // U5: RL lanes merge a rewritten row into its new chunk, holding RC of its
    // entries at a time: an entry moves by the inserts at or before its place
    // less the deletes before it.  The entries of the team's next row, and the
    // row table entry of the one after, are in flight meanwhile.  Rows of
    // unchanged structure get their added values written in place.  With x, the
    // row's product is taken from the entries at hand (each lane's in order, then
    // a fixed tree): reading the rewritten rows again for it would be a third of
    // the step's bytes.  It is summed in double, whatever the row's length: 16
    // chains in float were 7.4e-8 rms off over 4,096 entries, where batch_spmv's 64
    // lanes were 4.3e-8; now 3.4e-8 at most from 4 to 4,000
    {
        uint32_t st = 0, L = 0, st1 = 0, L1 = 0;
        int32_t c0 = 0, c1 = 0;
        float v0 = 0.0f, v1 = 0.0f;
        if (tm < nt) {
            const uint32_t g = row_of(tm);
            st = row_start[g];
            L = (uint32_t)row_len[g];
        }
        if (tm + NTM < nt) {
            const uint32_t g = row_of(tm + NTM);
            st1 = row_start[g];
            L1 = (uint32_t)row_len[g];
        }
        if (tl < L) {
            c0 = pcol[(uint64_t)st + tl];
            v0 = pval[(uint64_t)st + tl];
        }
        if (tl + RL < L) {
            c1 = pcol[(uint64_t)st + tl + RL];
            v1 = pval[(uint64_t)st + tl + RL];
        }
        for (uint32_t tt = tm; tt < nt; tt += NTM) {
            uint32_t st2 = 0, L2 = 0;
            int32_t d0 = 0, d1 = 0;
            float w0 = 0.0f, w1 = 0.0f;
            if (tl < L1) {
                d0 = pcol[(uint64_t)st1 + tl];
                w0 = pval[(uint64_t)st1 + tl];
            }
            if (tl + RL < L1) {
                d1 = pcol[(uint64_t)st1 + tl + RL];
                w1 = pval[(uint64_t)st1 + tl + RL];
            }
            if (tt + 2 * NTM < nt) {
                const uint32_t g = row_of(tt + 2 * NTM);
                st2 = row_start[g];
                L2 = (uint32_t)row_len[g];
            }
            uint32_t u = tub[tt];
            const uint32_t ue = tub[tt + 1];
            const uint32_t nl = tnl[tt];
            if (!(nl & 0x8000u)) {
                for (uint32_t q = u + tl; q < ue; q += RL)
                    if (upc[q] >> 14 == C_ADD) pval[(uint64_t)st + (upc[q] & 0x3fffu)] = S.uval[q];
            } else {
                const uint32_t g = gbase + (S.urc[u] >> KB);
                const uint32_t dst = base + tdst[tt];
                double prod = 0.0;
                for (uint32_t q = u + tl; q < ue; q += RL) {
                    if (upc[q] >> 14 != C_INS) continue;
                    const uint64_t d = (uint64_t)dst + (upc[q] & 0x3fffu);
                    const int32_t c = (int32_t)(S.urc[q] & (LMAX - 1));
                    pcol[d] = c;
                    pval[d] = S.uval[q];
                    if (x) prod = prod + (double)(S.uval[q] * x[c]);
                }
                uint32_t sh = 0;  // inserts less deletes so far
                for (uint32_t i0 = 0;;) {
                    const bool last = i0 + RC >= L;
                    const uint32_t p0 = i0 + tl, p1 = p0 + RL;
                    uint32_t s0 = sh, s1 = sh;
                    bool k0 = p0 < L, k1 = p1 < L;
                    float x0 = 0.0f, x1 = 0.0f;
                    if (x && k0) x0 = x[c0];
                    if (x && k1) x1 = x[c1];
                    for (; u < ue; ++u) {
                        const uint32_t w = upc[u];
                        const uint32_t pos = (w & 0x3fffu) - sh, code = w >> 14;  // place in the old row
                        if (!last && pos >= i0 + RC) break;  // among later entries
                        const float nv = S.uval[u];
                        const uint32_t ins = code == C_INS, del = code == C_DEL;
                        const bool add = code == C_ADD;
                        s0 += (p0 >= pos ? ins : 0u) - (p0 > pos ? del : 0u);
                        s1 += (p1 >= pos ? ins : 0u) - (p1 > pos ? del : 0u);
                        k0 = k0 && !(del && p0 == pos);
                        k1 = k1 && !(del && p1 == pos);
                        v0 = add && p0 == pos ? nv : v0;
                        v1 = add && p1 == pos ? nv : v1;
                        sh += ins - del;
                    }
                    if (k0) {
                        pcol[(uint64_t)dst + (p0 + s0)] = c0;
                        pval[(uint64_t)dst + (p0 + s0)] = v0;
                        prod = prod + (double)(v0 * x0);
                    }
                    if (k1) {
                        pcol[(uint64_t)dst + (p1 + s1)] = c1;
                        pval[(uint64_t)dst + (p1 + s1)] = v1;
                        prod = prod + (double)(v1 * x1);
                    }
                    if (last) break;
                    i0 += RC;
                    if (i0 + tl < L) {
                        c0 = pcol[(uint64_t)st + i0 + tl];
                        v0 = pval[(uint64_t)st + i0 + tl];
                    }
                    if (i0 + RL + tl < L) {
                        c1 = pcol[(uint64_t)st + i0 + RL + tl];
                        v1 = pval[(uint64_t)st + i0 + RL + tl];
                    }
                }
                prod = dpp_row_sum_f64(prod);
                if (tl == 0) {
                    if (x) {
                        y[g] = (float)prod;
                        atomicOr(&S.done[(g - gbase) >> 5], 1u << ((g - gbase) & 31u));
                    }
                    row_start[g] = dst;
                    row_len[g] = (int32_t)(nl & 0x7fffu);
                    row_cap[g] = (int32_t)chunk_round(nl & 0x7fffu);
                }
            }
            st = st1;
            L = L1;
            c0 = d0;
            c1 = d1;
            v0 = w0;
            v1 = w1;
            st1 = st2;
            L1 = L2;
        }
    }
    __syncthreads();
}

// SpMV of matrix m, but for the rows whose product its update has written: TEAM
// lanes per row for rows up to `thresh` entries, one
// wave per longer row; fixed-order reductions.  The first pass lists the longer
// rows in LDS (looking for them again, one row length per wave and round trip,
// took longer than the products).
template <int TEAM>
__device__ __forceinline__ void batch_spmv(uint32_t m, const uint32_t *__restrict__ row_base, const uint32_t *__restrict__ col_base,
                           const uint32_t *__restrict__ row_start, const int32_t *__restrict__ row_len,
                           const int32_t *__restrict__ pcol, const float *__restrict__ pval,
                           const float *__restrict__ x, float *__restrict__ y, uint32_t thresh, BatchLds &S)
{
    if (threadIdx.x == 0) S.sm[SM_LONG] = 0u;
    __syncthreads();
    const uint32_t gbase = row_base[m];
    const uint32_t Rm = row_base[m + 1] - gbase;
    const float *xm = x + col_base[m];
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));  // not kept from matrix to matrix: 13 registers spilled, not 18
    const uint32_t tl = t % TEAM;
    for (uint32_t r0 = 0; r0 < Rm; r0 += BT / TEAM) {
        const uint32_t r = r0 + t / TEAM;
        float acc = 0.0f;
        bool mine = false;
        if (r < Rm && !((S.done[r >> 5] >> (r & 31u)) & 1u)) {
            const uint32_t L = (uint32_t)row_len[gbase + r];
            mine = L <= thresh;
            if (!mine && tl == 0) S.urc[atomicAdd(&S.sm[SM_LONG], 1u)] = r;
            if (mine) {
                const uint64_t st = row_start[gbase + r];
                // four entries of the lane in flight, the last ones masked;
                // the lane still sums its entries in ascending order
                for (uint32_t k = tl; k < L; k += 4 * TEAM) {
                    int32_t c[4];
                    float v[4], xv[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        c[j] = 0;
                        v[j] = 0.0f;
                        if (k + j * TEAM < L) {
                            c[j] = pcol[st + k + j * TEAM];
                            v[j] = pval[st + k + j * TEAM];
                        }
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) xv[j] = k + j * TEAM < L ? xm[c[j]] : 0.0f;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (k + j * TEAM < L) acc = acc + v[j] * xv[j];
                }
            }
        }
#pragma unroll
        for (int o = TEAM / 2; o >= 1; o >>= 1) acc += __shfl_xor(acc, o);
        if (mine && tl == 0) y[gbase + r] = acc;
    }
    __syncthreads();
    // loads that the rows above left behind would be waited for in every round below,
    // and with them the row's store (100 matrices of 2,000 rows with 600 entries:
    // 613 -> 563 us)
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    const uint32_t nlong = S.sm[SM_LONG];
    for (uint32_t i = t >> 6; i < nlong; i += NW) {
        const uint32_t r = S.urc[i];
        const uint32_t L = (uint32_t)row_len[gbase + r];
        const uint64_t st = row_start[gbase + r];
        float acc = 0.0f;
        uint32_t k = lane_id();
        for (; k + 3 * 64 < L; k += 4 * 64) {
            const int32_t c0 = pcol[st + k], c1 = pcol[st + k + 64], c2 = pcol[st + k + 128], c3 = pcol[st + k + 192];
            const float v0 = pval[st + k], v1 = pval[st + k + 64], v2 = pval[st + k + 128], v3 = pval[st + k + 192];
            const float x0 = xm[c0], x1 = xm[c1], x2 = xm[c2], x3 = xm[c3];
            acc = acc + v0 * x0;
            acc = acc + v1 * x1;
            acc = acc + v2 * x2;
            acc = acc + v3 * x3;
        }
        for (; k < L; k += 64) acc = acc + pval[st + k] * xm[pcol[st + k]];
        acc = wave_sum_f32(acc);
        if (lane_id() == 0) y[gbase + r] = acc;
    }
}

template <int TEAM>
__global__ __launch_bounds__(BT, 2 * BT / 256) void k_batch_step(uint32_t M, const uint32_t *__restrict__ order,
                                                   const uint32_t *__restrict__ row_base,
                                                   const uint32_t *__restrict__ col_base,
                                                   const int64_t *__restrict__ tri_off, int64_t ntri,
                                                   const int32_t *__restrict__ trow, const int32_t *__restrict__ tcol,
                                                   const float *__restrict__ tval,
                                                   uint32_t *__restrict__ row_start, int32_t *__restrict__ row_len,
                                                   int32_t *__restrict__ row_cap, int32_t *__restrict__ pcol,
                                                   float *__restrict__ pval, unsigned long long pool_cap, DevState *ds,
                                                   uint32_t *__restrict__ mstat,
                                                   const float *__restrict__ x, float *__restrict__ y, uint32_t thresh,
                                                   BatchState *bs, int do_update, int do_spmv, int reserved)
{
    __shared__ BatchLds S;
    __shared__ BatchAcc acc;
    if (threadIdx.x == 0) acc = BatchAcc{0, 0, 0, 0, 0, 0};
    // the first matrix is the workgroup's own, the others come from the work
    // counter (which counts past the grid), asked for while the one before is
    // in work: 512 workgroups that wait for the same word take microseconds
    for (uint32_t i = blockIdx.x; i < M;) {
        if (threadIdx.x == 0) S.next = gridDim.x + atomicAdd(&bs->work, 1u);
        const uint32_t m = order[i];
        if (do_spmv && threadIdx.x < LMAX / 32) S.done[threadIdx.x] = 0u;  // a barrier follows before its first use
        if (do_update)
            batch_update(m, row_base, col_base, tri_off, ntri, trow, tcol, tval, row_start, row_len, row_cap, pcol, pval,
                         pool_cap, ds, mstat, do_spmv ? x + col_base[m] : nullptr, y, S, reserved != 0, acc);
        if (do_spmv) batch_spmv<TEAM>(m, row_base, col_base, row_start, row_len, pcol, pval, x, y, thresh, S);
        __syncthreads();
        i = S.next;
        __syncthreads();
    }
    // the workgroup's counters, then: the last workgroup out resets the work
    // counters (no memset: replay-safe).  No fence: both counters are
    // atomics, every workgroup's last work claim returned before its finish
    // count, and the kernel boundary publishes the reset (a release fence
    // would write back the XCD's whole L2 here)
    if (threadIdx.x == 0) {
        if (acc.touched) {
            atomicAdd((unsigned long long *)&ds->nnz, (unsigned long long)acc.dnnz);
            atomicAdd((unsigned long long *)&ds->garbage, (unsigned long long)acc.dgarbage);
            atomicAdd((unsigned long long *)&ds->n_ins, acc.ins);
            atomicAdd((unsigned long long *)&ds->n_add, acc.add);
            atomicAdd((unsigned long long *)&ds->n_del, acc.del);
            atomicAdd(&ds->ntouched, acc.touched);
        }
        if (atomicAdd(&bs->done, 1u) == gridDim.x - 1) {  // every workgroup has asked for its last matrix
            bs->work = 0;
            bs->done = 0;
        }
    }
}

__global__ void k_batch_globalize(const int64_t *__restrict__ tri_off, uint32_t M, int64_t n,
                                  const uint32_t *__restrict__ row_base, const uint32_t *__restrict__ col_base,
                                  const int32_t *__restrict__ rows, const int32_t *__restrict__ cols,
                                  int32_t *__restrict__ grows, int32_t *__restrict__ gcols, DevState *ds)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t lo = 0, hi = M;  // matrix of entry i: largest m with tri_off[m] <= i
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (tri_off[mid] <= i) lo = mid; else hi = mid;
    }
    const uint32_t Rm = row_base[lo + 1] - row_base[lo], Cm = col_base[lo + 1] - col_base[lo];
    const int32_t r = rows[i], c = cols[i];
    const bool bad = r < 0 || (uint32_t)r >= Rm || c < 0 || (uint32_t)c >= Cm;
    grows[i] = bad ? -1 : (int32_t)(row_base[lo] + r);
    gcols[i] = c;
    if (bad) atomicOr(&ds->status, ST_BAD_INDEX);
}

__global__ void k_batch_zero_stat(uint32_t *mstat, uint32_t M, DevState *ds)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) mstat[i] = 0;
    if (i == 0) {
        ds->n_ins = ds->n_add = ds->n_del = 0;
        ds->ntouched = 0;
    }
}

}  // namespace

dcsr_status load_coo_internal(dcsr_handle h, const int32_t *rows, const int32_t *cols, const float *vals, int64_t n,
                              hipStream_t s);

struct TuneKey {
    int mbucket, lbucket;
    bool operator<(const TuneKey &o) const { return mbucket != o.mbucket ? mbucket < o.mbucket : lbucket < o.lbucket; }
};
struct TuneVal {
    int team;
    int thresh;
};
static std::map<TuneKey, TuneVal> g_tune_cache;  // process-wide autotuner choices

struct dcsr_batch_s {
    uint32_t M;
    dcsr_handle h;  // block-diagonal storage
    uint32_t *row_base, *col_base;  // device, M+1
    // device, M: the matrices by rows, largest first, so that the last ones
    // taken are small (in given order a 4,096-row matrix taken last left the
    // other workgroups idle: 1.36 -> 1.31 ms per step)
    uint32_t *order;
    std::vector<uint32_t> row_base_h, col_base_h;
    uint32_t *mstat;                // device, per-matrix status bits
    BatchState *bs;
    int grid;
    int team, thresh;               // SpMV launch shape (autotuned)
    hipStream_t cs;                 // capture stream (graphs replay on the caller's stream)
    hipGraph_t graph;
    hipGraphExec_t gexec;
    const void *gkey[13];           // launch arguments the captured graph was built with
};

static int bucket_log2(double v)
{
    int b = 0;
    while (v >= 2.0 && b < 30) {
        v /= 2.0;
        ++b;
    }
    return b;
}

dcsr_status dcsr_batch_create(dcsr_batch *out, int32_t count, const int32_t *rows, const int32_t *cols,
                              const dcsr_config *cfg)
{
    if (!out || count <= 0 || !rows || !cols) return DCSR_ERR_INVALID;
    uint64_t R = 0, Cmax = 1;
    std::vector<uint32_t> rb(count + 1), cb(count + 1);
    uint64_t cacc = 0;
    for (int i = 0; i < count; ++i) {
        if (rows[i] < 0 || cols[i] < 0 || (uint32_t)rows[i] > LMAX || (uint32_t)cols[i] > LMAX)
            return DCSR_ERR_UNSUPPORTED;  // local indices are 12-bit
        rb[i] = (uint32_t)R;
        cb[i] = (uint32_t)cacc;
        R += (uint32_t)rows[i];
        cacc += (uint32_t)cols[i];
        if ((uint64_t)cols[i] > Cmax) Cmax = cols[i];
    }
    rb[count] = (uint32_t)R;
    cb[count] = (uint32_t)cacc;
    if (R >= (1ull << 31) || cacc >= (1ull << 31)) return DCSR_ERR_UNSUPPORTED;
    dcsr_batch b = new dcsr_batch_s();
    b->M = (uint32_t)count;
    b->row_base_h = rb;
    b->col_base_h = cb;
    b->team = 8;
    b->thresh = 128;
    dcsr_status st = dcsr_create(&b->h, (int64_t)R, (int64_t)Cmax, cfg);
    if (st != DCSR_OK) {
        delete b;
        return st;
    }
    int dev = 0, ncu = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    b->grid = (ncu > 0 ? ncu : 256) * 2;
    if ((uint32_t)b->grid > b->M) b->grid = (int)b->M;
    if (hipMalloc(&b->row_base, (count + 1) * 4) != hipSuccess || hipMalloc(&b->col_base, (count + 1) * 4) != hipSuccess ||
        hipMalloc(&b->mstat, count * 4) != hipSuccess || hipMalloc(&b->order, count * 4) != hipSuccess ||
        hipMalloc(&b->bs, sizeof(BatchState)) != hipSuccess ||
        hipStreamCreateWithFlags(&b->cs, hipStreamNonBlocking) != hipSuccess) {
        dcsr_batch_destroy(b);
        return DCSR_ERR_OOM;
    }
    std::vector<uint32_t> order(count);
    for (int i = 0; i < count; ++i) order[i] = (uint32_t)i;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t p, uint32_t q) { return rows[p] > rows[q]; });
    if (hipMemcpy(b->order, order.data(), count * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b->row_base, rb.data(), (count + 1) * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b->col_base, cb.data(), (count + 1) * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(b->mstat, 0, count * 4) != hipSuccess || hipMemset(b->bs, 0, sizeof(BatchState)) != hipSuccess) {
        dcsr_batch_destroy(b);
        return DCSR_ERR_HIP;
    }
    *out = b;
    return DCSR_OK;
}

dcsr_status dcsr_batch_destroy(dcsr_batch b)
{
    if (!b) return DCSR_ERR_INVALID;
    (void)hipDeviceSynchronize();
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    if (b->cs) (void)hipStreamDestroy(b->cs);
    (void)hipFree(b->row_base);
    (void)hipFree(b->col_base);
    (void)hipFree(b->mstat);
    (void)hipFree(b->order);
    (void)hipFree(b->bs);
    if (b->h) dcsr_destroy(b->h);
    delete b;
    return DCSR_OK;
}

dcsr_handle dcsr_batch_handle(dcsr_batch b) { return b ? b->h : nullptr; }

dcsr_status dcsr_batch_info(dcsr_batch b, int64_t *row_base, int64_t *col_base, int32_t *team, int32_t *thresh)
{
    if (!b) return DCSR_ERR_INVALID;
    for (uint32_t i = 0; i <= b->M; ++i) {
        if (row_base) row_base[i] = b->row_base_h[i];
        if (col_base) col_base[i] = b->col_base_h[i];
    }
    if (team) *team = b->team;
    if (thresh) *thresh = b->thresh;
    return DCSR_OK;
}

dcsr_status dcsr_batch_load_coo(dcsr_batch b, const int64_t *tri_off, const int32_t *rows, const int32_t *cols,
                                const float *vals, int64_t n, dcsr_stream_t stream)
{
    if (!b || !tri_off || n < 0 || (n > 0 && (!rows || !cols || !vals))) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    dcsr_handle h = b->h;
    int32_t *gr, *gc;
    DCSR_TRY(ws_get(h, WS_SG_KEY0, (size_t)(n + 1) * 4, (void **)&gr));
    DCSR_TRY(ws_get(h, WS_SG_KEY1, (size_t)(n + 1) * 4, (void **)&gc));
    if (n > 0)
        k_batch_globalize<<<grid_for(n, 256), 256, 0, s>>>(tri_off, b->M, n, b->row_base, b->col_base, rows, cols, gr,
                                                           gc, h->ds);
    DCSR_HIP(hipGetLastError());
    return load_coo_internal(h, gr, gc, vals, n, s);
}

template <int TEAM>
static void launch_step(dcsr_batch b, const int64_t *tri_off, int64_t n, const int32_t *rows, const int32_t *cols,
                        const float *vals, const float *x, float *y, int do_update, int do_spmv, int reserved,
                        hipStream_t s)
{
    dcsr_handle h = b->h;
    k_batch_step<TEAM><<<b->grid, BT, 0, s>>>(b->M, b->order, b->row_base, b->col_base, tri_off, n, rows, cols, vals, h->row_start,
                                              h->row_len, h->row_cap, h->pool_col, h->pool_val,
                                              (unsigned long long)h->pool_cap, h->ds, b->mstat, x, y,
                                              (uint32_t)b->thresh, b->bs, do_update, do_spmv, reserved);
}

static void launch_any(dcsr_batch b, const int64_t *tri_off, int64_t n, const int32_t *rows, const int32_t *cols,
                       const float *vals, const float *x, float *y, int do_update, int do_spmv, int reserved,
                       hipStream_t s)
{
    switch (b->team) {
    case 4: launch_step<4>(b, tri_off, n, rows, cols, vals, x, y, do_update, do_spmv, reserved, s); break;
    case 16: launch_step<16>(b, tri_off, n, rows, cols, vals, x, y, do_update, do_spmv, reserved, s); break;
    case 32: launch_step<32>(b, tri_off, n, rows, cols, vals, x, y, do_update, do_spmv, reserved, s); break;
    default: launch_step<8>(b, tri_off, n, rows, cols, vals, x, y, do_update, do_spmv, reserved, s); break;
    }
}

// Pool headroom for one step: every matrix may rewrite all its rows plus its
// batch.  Compacts/grows ahead of the launch so the kernel never runs out
// (*reserved = 1: the claims need no fit check).  With allow_grow = 0 the
// pool keeps its capacity (retired chunks are reclaimed first): if the room
// may still fall short (*reserved = 0), a matrix whose claim does not fit
// fails alone with its exhausted bit and leaves room for the others.
static dcsr_status batch_reserve(dcsr_batch b, int64_t n, hipStream_t s, int *reserved)
{
    dcsr_handle h = b->h;
    if (!h->state_known) DCSR_TRY(pull_state(h, s));
    const int64_t need = h->nnz_h + n + 4 * (int64_t)h->rows + 64;
    *reserved = 1;
    if (h->pool_cap - h->bump_h >= need) return DCSR_OK;
    if (!h->cfg.allow_grow) {
        if (h->bump_h > h->nnz_h) DCSR_TRY(compact_in_order(h, s));
        // after a compaction the bump pointer is the live count
        *reserved = h->pool_cap - h->nnz_h >= need ? 1 : 0;
        return DCSR_OK;
    }
    return pool_reserve(h, need, s, nullptr);
}

dcsr_status dcsr_batch_step(dcsr_batch b, const int64_t *tri_off, const int32_t *rows, const int32_t *cols,
                            const float *vals, int64_t n, const float *x, float *y, uint32_t flags,
                            dcsr_stream_t stream)
{
    if (!b) return DCSR_ERR_INVALID;
    const int do_update = tri_off != nullptr && n > 0;
    const int do_spmv = x != nullptr && y != nullptr;
    if (!do_update && !do_spmv) return DCSR_OK;
    if (do_update && (!rows || !cols || !vals)) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    dcsr_handle h = b->h;
    h->last_stream = s;
    if (!h->canonical) DCSR_TRY(canonicalize(h, s));
    int reserved = 0;
    if (do_update) {
        if (capturing(s)) h->replayed = true;
        else DCSR_TRY(refresh_replayed(h, s));
        DCSR_TRY(batch_reserve(b, n, s, &reserved));
    }
    k_batch_zero_stat<<<grid_for(b->M, 256), 256, 0, s>>>(b->mstat, b->M, h->ds);
    if (flags & DCSR_BATCH_GRAPH) {
        const void *key[13] = {tri_off, rows, cols, vals, x, y, h->pool_col, (const void *)(intptr_t)b->team,
                               (const void *)(intptr_t)b->thresh,
                               (const void *)(intptr_t)(reserved * 4 + do_update * 2 + do_spmv),
                               (const void *)(intptr_t)h->pool_cap, (const void *)(intptr_t)n, h->row_start};
        bool same = b->gexec != nullptr;
        for (int i = 0; i < 13 && same; ++i) same = key[i] == b->gkey[i];
        if (!same) {
            if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
            if (b->graph) (void)hipGraphDestroy(b->graph);
            b->gexec = nullptr;
            b->graph = nullptr;
            // capture on the batch's own stream (the caller's may be the null
            // stream, which cannot be captured); nothing runs during capture
            DCSR_HIP(hipStreamBeginCapture(b->cs, hipStreamCaptureModeThreadLocal));
            launch_any(b, tri_off, n, rows, cols, vals, x, y, do_update, do_spmv, reserved, b->cs);
            DCSR_HIP(hipStreamEndCapture(b->cs, &b->graph));
            DCSR_HIP(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
            for (int i = 0; i < 13; ++i) b->gkey[i] = key[i];
        }
        DCSR_HIP(hipGraphLaunch(b->gexec, s));
    } else {
        launch_any(b, tri_off, n, rows, cols, vals, x, y, do_update, do_spmv, reserved, s);
    }
    DCSR_HIP(hipGetLastError());
    if (do_update) {
        state_unknown(h, n, h->pool_cap);
        h->flat_dirty = true;
    }
    return DCSR_OK;
}

// Status of the last step: OR of the per-matrix bits (syncs); `per_matrix`
// (host, M entries) receives them when not NULL.  Also refreshes the handle's
// counters (nnz, inserted / added / deleted entries and touched rows of the
// step, summed over the matrices).
dcsr_status dcsr_batch_status(dcsr_batch b, uint32_t *per_matrix)
{
    if (!b) return DCSR_ERR_INVALID;
    std::vector<uint32_t> st(b->M);
    DCSR_HIP(hipMemcpyAsync(st.data(), b->mstat, b->M * 4, hipMemcpyDeviceToHost, b->h->last_stream));
    DCSR_HIP(hipStreamSynchronize(b->h->last_stream));
    // the step's counters (summed over matrices) become the handle's
    // "last update" figures reported by dcsr_query
    DCSR_TRY(pull_state(b->h, b->h->last_stream));
    b->h->last_ins = b->h->hs->n_ins;
    b->h->last_add = b->h->hs->n_add;
    b->h->last_del = b->h->hs->n_del;
    b->h->last_touched = b->h->hs->ntouched;
    uint32_t any = 0;
    for (uint32_t i = 0; i < b->M; ++i) {
        any |= st[i];
        if (per_matrix) per_matrix[i] = st[i];
    }
    if (any & BST_BAD_INDEX) return DCSR_ERR_BAD_INDEX;
    if (any & BST_TOO_BIG) return DCSR_ERR_UNSUPPORTED;
    if (any & BST_EXHAUSTED) return DCSR_ERR_POOL_EXHAUSTED;
    return DCSR_OK;
}

// Autotuner: times the SpMV part of the step (read-only) for every
// (lanes per row, long-row threshold) pair on the batch as loaded, keeps the
// fastest, and caches the choice per shape class (matrix count and mean row
// length, log2 buckets) for the process.
dcsr_status dcsr_batch_autotune(dcsr_batch b, const float *x, float *y, int32_t *team_out, int32_t *thresh_out,
                                dcsr_stream_t stream)
{
    if (!b || !x || !y) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    dcsr_handle h = b->h;
    if (!h->state_known) DCSR_TRY(pull_state(h, s));
    const double mean_len = h->rows ? (double)h->nnz_h / (double)h->rows : 0.0;
    TuneKey key{bucket_log2((double)b->M), bucket_log2(mean_len)};
    auto it = g_tune_cache.find(key);
    if (it != g_tune_cache.end()) {
        b->team = it->second.team;
        b->thresh = it->second.thresh;
    } else {
        const int teams[4] = {4, 8, 16, 32};
        const int threshs[3] = {64, 256, 1024};
        hipEvent_t e0, e1;
        DCSR_HIP(hipEventCreate(&e0));
        DCSR_HIP(hipEventCreate(&e1));
        float best = 1e30f;
        int bt = 8, bth = 128;
        for (int ti = 0; ti < 4; ++ti)
            for (int hi = 0; hi < 3; ++hi) {
                b->team = teams[ti];
                b->thresh = threshs[hi];
                launch_any(b, nullptr, 0, nullptr, nullptr, nullptr, x, y, 0, 1, 0, s);  // warm
                DCSR_HIP(hipEventRecord(e0, s));
                for (int rep = 0; rep < 3; ++rep) launch_any(b, nullptr, 0, nullptr, nullptr, nullptr, x, y, 0, 1, 0, s);
                DCSR_HIP(hipEventRecord(e1, s));
                DCSR_HIP(hipEventSynchronize(e1));
                float ms = 0.0f;
                DCSR_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (ms < best) {
                    best = ms;
                    bt = teams[ti];
                    bth = threshs[hi];
                }
            }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        b->team = bt;
        b->thresh = bth;
        g_tune_cache[key] = TuneVal{bt, bth};
    }
    if (team_out) *team_out = b->team;
    if (thresh_out) *thresh_out = b->thresh;
    return DCSR_OK;
}

dcsr_status dcsr_batch_set_shape(dcsr_batch b, int32_t team, int32_t thresh)
{
    if (!b || !(team == 4 || team == 8 || team == 16 || team == 32) || thresh < 0) return DCSR_ERR_INVALID;
    b->team = team;
    b->thresh = thresh;
    return DCSR_OK;
}
