// spgemm.hip -- C = A * B for DCSR operands.
//
// Replaces device::spmm(const dcsr& A, const dcsr& B, dcsr& C, streams)
// (include/spmm.h:30-391) and its binned ESC kernels (include/spmm.inl:361-668,
// 951-1061).  Result semantics are those of the host path
// (cusp/system/detail/sequential/multiply/csr_spgemm.h:75-150): the structure
// holds every (i, k) with a partial product whose FP32 sum, accumulated from
// 0 in A-row order then B-row order, is not exactly 0.
//
// Rows are bucketed by their partial-product count P_i:
//   P_i <=  128  a 16-lane team per row, four rows per wave, the same LDS
//                ESC as below with small per-row buffers (many rows in
//                flight per CU: a row is a chain of dependent loads);
//   P_i <= 1024  one wave per row, LDS ESC: the row's partials are expanded
//                with their generation index (A-entry order, then B-row
//                order), bucket-sorted in LDS by (column, generation), and
//                each run of equal columns is summed left-to-right;
//   P_i <= 4096  the same with one 256-thread workgroup per row;
//   P_i <= 16384 the same with one 1024-thread workgroup per row (8192 where
//                the sort key needs 64 bits);
//   larger       (power-law hub rows, which the reference skips) a global
//                ESC: expand, stable LSD radix sort by (row, column), reduce.
// Output rows come out column-sorted with exact zeros removed, and the
// accumulation order is fixed, so C is deterministic.
#include "dcsr_internal.h"
#include "prims.h"
#include "segments.h"

namespace {

constexpr int TB = 256;
constexpr uint32_t TEAM_MAX = 128;    // partials per row for the team kernel
constexpr int TEAM = 16;              // lanes per row in the team kernel
static_assert(TEAM_MAX <= 8 * TEAM, "team rows: the rank sort holds at most 8 keys per lane");
constexpr int TEAM_GB = 7;            // generation bits of the team kernel's 32-bit keys
// the team kernel's keys are 32-bit: B's columns must stay below this
constexpr int64_t TEAM_MAX_COLS = (1ll << (32 - TEAM_GB)) - 1;
constexpr int WAVE_GB = 10;           // generation bits of the wave kernel's keys
// the wave kernel's keys are 32-bit up to this many columns of B, else 64-bit
constexpr int64_t WAVE_MAX_COLS32 = (1ll << (32 - WAVE_GB)) - 1;
constexpr uint32_t WAVE_MAX = 1024;   // partials per row for the wave kernel
constexpr uint32_t BLOCK_MAX = 4096;  // partials per row for the workgroup kernel
constexpr int BLOCK_GB = 12;
constexpr int64_t BLOCK_MAX_COLS32 = (1ll << (32 - BLOCK_GB)) - 1;
// the large-row kernel: 1024 threads, most of a CU's LDS
constexpr int BIG_TB = 1024;
constexpr uint32_t BIG_MAX32 = 16384, BIG_MAX64 = 8192;  // partials per row by key width
constexpr int BIG_GB = 14;
constexpr int64_t BIG_MAX_COLS32 = (1ll << (32 - BIG_GB)) - 1;
constexpr int SG_EX = 8;              // partials per lane whose loads are in flight together
// row classes: hub, large, workgroup;
// team classes CL_TEAM + 2 i: rows of at most 2 (i + 1) * TEAM partials, sorted
// with 2 (i + 1) keys per lane;
// wave classes CL_WAVE + 2 i: rows of at most 256, 512, 1024 partials, sorted with
// 4, 8, 16 keys per lane (the registers of the widest would hold the shorter
// rows, which are most of them, to 3 waves per SIMD)
enum { CL_HUB = 0, CL_BIG = 1, CL_TEAM = 2, CL_BLOCK = 3, CL_WAVE = 5, NCLS = 10 };
constexpr int cl_team(int kpl) { return CL_TEAM + 2 * (kpl / 2 - 1); }
constexpr int cl_wave(int kpl) { return CL_WAVE + 2 * ((kpl > 4) + (kpl > 8)); }

// The rows of one class.  A row is in one class at most, so two classes share an
// array of R rows: the even one fills it from the front, the odd one from the back.
template <int CLS>
struct SgList {
    const uint32_t *p;
    SgList(const uint32_t *lists, uint32_t R) : p(lists + (uint64_t)(CLS / 2) * R + (CLS % 2 ? R - 1 : 0)) {}
    __device__ __forceinline__ uint32_t operator[](uint32_t i) const { return CLS % 2 ? *(p - i) : p[i]; }
};

struct SgState {
    unsigned long long total;  // sum of P_i (64-bit)
    unsigned int count[NCLS];  // rows per class
    unsigned int pad;
};

__device__ __forceinline__ uint32_t next_pow2(uint32_t v)
{
    v--;
    v |= v >> 1;
    v |= v >> 2;
    v |= v >> 4;
    v |= v >> 8;
    v |= v >> 16;
    return v + 1;
}

// What the kernels read: the operands' row tables and pools, and in a PAIRED
// product the B row of every A entry (A's flat order) and B's entries as (column,
// value) pairs in B's flat order.  A short row of B is one 128-byte line of pairs
// where the pool's two arrays cost one line each, and these lines bound the product
// of matrices past the L2 (2M-row Poisson(8): the 16-lane kernels 1083 -> 1006 us
// and the count 248 -> 181, the copy costs 77).  Small products read the operands
// as they are, for the copy is a launch: squares of 0.3M / 0.6M / 0.8M / 1.2M / 1.6M /
// 3.2M / 16M entries (Poisson rows of 3 and 8) take 99 / 113 / 163 / 160 / 224 / 382 /
// 1,879 us so and 104 / 124 / 164 / 161 / 207 / 302 / 1,260 with the copies, power-law
// squares of 0.1M / 0.4M / 0.8M / 1.6M / 2M 191 / 273 / 321 / 508 / 590 and 195 / 276 /
// 314 / 493 / 579: the line is at 1.6M entries of both operands.  So do products for
// which the copies do not fit the memory.
struct SgIn {
    const uint32_t *P, *Poff, *a_start;
    const int32_t *a_len, *a_col;
    const float *a_val;
    const uint32_t *b_start;
    const int32_t *b_len, *b_col;
    const float *b_val;
    const uint32_t *a_foff, *b_foff;
    const uint2 *ent, *b_ent;
};

// P_i = sum over the entries of A row i of len(B row col).  One wave per 64
// consecutive rows; entries folded per row with a DPP segmented scan.  PAIRED: the
// B row (flat start, length) of every A entry is kept in A's flat order (ent): the
// row kernels stream it instead of gathering it again.
template <bool PAIRED>
__global__ __launch_bounds__(TB) void k_sg_count(uint32_t R, SgIn in, uint2 *__restrict__ ent, uint32_t *__restrict__ P)
{
    __shared__ uint32_t s_ex[TB / 64][64];
    __shared__ uint32_t s_st[TB / 64][64];
    __shared__ uint32_t s_acc[TB / 64][64];
    const int w = threadIdx.x >> 6;
    const int lane = lane_id();
    const uint32_t r0 = (blockIdx.x * (TB / 64) + w) * 64u;
    const uint32_t r = r0 + lane;
    if (r0 >= R) return;
    uint32_t f0 = 0, tot, ex;
    if constexpr (PAIRED) {
        const uint32_t fo = in.a_foff[r < R ? r : R];
        f0 = wave_read_lane_u32(fo, 0);
        tot = in.a_foff[r0 + 64u < R ? r0 + 64u : R] - f0;
        ex = fo - f0;
    } else {
        const uint32_t L = r < R ? (uint32_t)in.a_len[r] : 0u, inc = wave_incl_scan_u32(L);
        tot = wave_read_lane_u32(inc, 63);
        ex = inc - L;
    }
    s_ex[w][lane] = ex;
    s_st[w][lane] = r < R ? in.a_start[r] : 0u;
    s_acc[w][lane] = 0;
    __builtin_amdgcn_wave_barrier();
    // four 64-entry chunks per round: their A-column loads, then their B-row
    // record loads, each issued together (two round trips per 256 entries)
    constexpr int CU = 4;
    for (uint32_t b = 0; b < tot; b += 64 * CU) {
        uint32_t j[CU];
        int32_t c[CU];
        uint2 q[CU];
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            const uint32_t e = b + (uint32_t)u * 64u + lane;
            j[u] = 64;
            c[u] = -1;
            if (e < tot) {
                j[u] = (uint32_t)find_seg64(s_ex[w], e);
                c[u] = in.a_col[(uint64_t)s_st[w][j[u]] + (e - s_ex[w][j[u]])];
            }
        }
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            if constexpr (PAIRED) {
                // neighbours in one array: one line, mostly
                q[u] = c[u] >= 0 ? make_uint2(in.b_foff[c[u]], in.b_foff[c[u] + 1]) : make_uint2(0u, 0u);
                q[u].y -= q[u].x;
            } else {
                q[u] = make_uint2(0u, c[u] >= 0 ? (uint32_t)in.b_len[c[u]] : 0u);
            }
        }
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            if (PAIRED && c[u] >= 0) ent[(uint64_t)f0 + b + (uint32_t)u * 64u + lane] = q[u];
            const uint32_t t = wave_seg_incl_scan_u32(q[u].y, j[u]);
            const uint32_t jn = __shfl_down(j[u], 1);
            if (j[u] < 64 && (lane == 63 || jn != j[u])) s_acc[w][j[u]] += t;
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (r < R) P[r] = s_acc[w][lane];
}

// Row classes (list appends aggregated per workgroup: one global atomic per
// class per workgroup of SG_CR * TB rows) and per-block 64-bit P sums.  Each
// thread classifies SG_CR rows; with 256 rows per workgroup the class
// counters took ~60K contended atomics per product (94 us on 2M rows).
constexpr int SG_CR = 8;
__global__ __launch_bounds__(TB) void k_sg_classify(uint32_t R, const uint32_t *__restrict__ P,
                                                    uint32_t *__restrict__ lists, SgState *st, uint32_t *__restrict__ cnt,
                                                    unsigned long long *__restrict__ bsum, uint32_t team_ok,
                                                    uint32_t big_max)
{
    __shared__ unsigned long long ws[TB / 64];
    __shared__ uint32_t s_cnt[NCLS], s_base[NCLS];
    if (threadIdx.x < NCLS) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t r0 = blockIdx.x * (TB * SG_CR) + threadIdx.x;
    uint32_t p[SG_CR], slot[SG_CR];
    int cls[SG_CR];
#pragma unroll
    for (int q = 0; q < SG_CR; ++q) {
        const uint32_t r = r0 + (uint32_t)q * TB;
        p[q] = r < R ? P[r] : 0u;
    }
    unsigned long long v = 0;
#pragma unroll
    for (int q = 0; q < SG_CR; ++q) {
        const uint32_t r = r0 + (uint32_t)q * TB;
        cls[q] = -1;
        slot[q] = 0;
        if (r < R) {
            // team rows in classes by rank-sort width (2, 4, 6 or 8 keys per
            // lane), so the four teams of a wave run the same sort over similar
            // row sizes
            cls[q] = p[q] == 0                         ? -1
                     : (p[q] <= TEAM_MAX && team_ok)   ? CL_TEAM + 2 * (int)((p[q] - 1) / (2 * TEAM))
                     : p[q] <= WAVE_MAX                ? CL_WAVE + 2 * ((p[q] > 256u) + (p[q] > 512u))
                     : p[q] <= BLOCK_MAX               ? CL_BLOCK
                     : p[q] <= big_max                 ? CL_BIG
                                                       : CL_HUB;
            if (p[q] == 0) cnt[r] = 0;
        }
        v += p[q];
        // slot of this row inside its workgroup's share of its class list
#pragma unroll
        for (int c = 0; c < NCLS; ++c) {
            const uint64_t m = __ballot(cls[q] == c);
            if (!m) continue;
            const int leader = __ffsll((long long)m) - 1;
            uint32_t base = 0;
            if (lane_id() == leader) base = atomicAdd(&s_cnt[c], (uint32_t)__popcll(m));
            base = __shfl(base, leader);
            if (cls[q] == c) slot[q] = base + (uint32_t)__popcll(m & lanemask_lt());
        }
    }
    __syncthreads();
    if (threadIdx.x < NCLS && s_cnt[threadIdx.x])
        s_base[threadIdx.x] = atomicAdd(&st->count[threadIdx.x], s_cnt[threadIdx.x]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SG_CR; ++q)
        if (cls[q] >= 0) {
            const uint32_t i = s_base[cls[q]] + slot[q];
            lists[(uint64_t)(cls[q] >> 1) * R + (cls[q] & 1 ? R - 1u - i : i)] = r0 + (uint32_t)q * TB;
        }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    if (lane_id() == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = (ws[0] + ws[1]) + (ws[2] + ws[3]);
}

__global__ void k_sg_state_zero(SgState *st)
{
    st->total = 0;
    for (int c = 0; c < NCLS; ++c) st->count[c] = 0;
}

__global__ __launch_bounds__(1024) void k_sg_total(SgState *st, const unsigned long long *__restrict__ bsum, int nb)
{
    __shared__ unsigned long long red[16];
    unsigned long long v = 0;
    for (int b = threadIdx.x; b < nb; b += 1024) v += bsum[b];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < 16; ++i) t += red[i];
        st->total = t;
    }
}

// ---------------------------------------------------------------------------
// Shared row routine: expand, sort, reduce.  NT threads cooperate (64 for the
// wave kernel, 256 and 1024 for the workgroup kernels); GB = generation-index
// bits.
// ---------------------------------------------------------------------------
// A team is NT threads: 16 (a quarter wave), 64 (a wave), 256 or 1024 (the
// workgroup).  Teams inside one wave never exchange data with each other.
template <int NT>
__device__ __forceinline__ void team_sync()
{
    if (NT <= 64) __builtin_amdgcn_wave_barrier();
    else __syncthreads();
}

// Exclusive scan of one uint32 per team thread.
template <int NT>
__device__ __forceinline__ uint32_t team_excl_scan(uint32_t v, uint32_t *lds_w, uint32_t *total)
{
    if (NT < 64) {
        static_assert(NT >= 64 || NT == 16, "a team is a DPP row");
        uint32_t inc = v, tot = v;
        inc += dpp_u32<DPP_ROW_SHR(1)>(0u, inc);
        inc += dpp_u32<DPP_ROW_SHR(2)>(0u, inc);
        inc += dpp_u32<DPP_ROW_SHR(4)>(0u, inc);
        inc += dpp_u32<DPP_ROW_SHR(8)>(0u, inc);
        tot += dpp_u32<DPP_ROW_ROR(8)>(0u, tot);
        tot += dpp_u32<DPP_ROW_ROR(4)>(0u, tot);
        tot += dpp_u32<DPP_ROW_ROR(2)>(0u, tot);
        tot += dpp_u32<DPP_ROW_ROR(1)>(0u, tot);
        *total = tot;
        return inc - v;
    }
    const uint32_t inc = wave_incl_scan_u32(v);
    if (NT == 64) {
        *total = wave_read_lane_u32(inc, 63);
        return inc - v;
    }
    const int w = (threadIdx.x % NT) >> 6;
    if (lane_id() == 63) lds_w[w] = inc;
    __syncthreads();
    uint32_t carry = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
        const uint32_t t = lds_w[i];
        if (i < w) carry += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return carry + inc - v;
}

// Largest j in [0, NT) with s[j] <= e.
template <int NT>
__device__ __forceinline__ uint32_t find_seg_team(const uint32_t *s, uint32_t e)
{
    uint32_t lo = 0, hi = NT;
#pragma unroll
    for (int it = 0; (1 << it) < NT; ++it) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s[mid] <= e) lo = mid; else hi = mid;
    }
    return lo;
}

// K: the sort key type, (column << GB) | generation.  32-bit keys halve the
// LDS per row (more rows in flight); they need columns below 2^(32-GB) - 1
// so that no key reaches the ~0 padding.
// What a row needs before its expansion: its partial count, output offset
// and A row.  Loaded one row ahead by the kernels' row loops (the loads of
// the next row are in flight while the current row is processed).
struct SgRowInfo {
    uint32_t row, P, ast, la, fo;
    uint32_t out_base;
};

// What they write: C's pool and the row's entry count.
struct SgOut {
    int32_t *tcol;
    float *tval;
    uint32_t *cnt;
};

// B's row (start in B's entries, length) of entry a of A's row.
template <bool PAIRED>
__device__ __forceinline__ uint2 sg_b_row(const SgIn &in, const SgRowInfo &ri, uint32_t a)
{
    if constexpr (PAIRED) return in.ent[(uint64_t)ri.fo + a];
    const int32_t c = in.a_col[(uint64_t)ri.ast + a];
    return make_uint2(in.b_start[c], (uint32_t)in.b_len[c]);
}

// Entry p of B: column and value bits.
template <bool PAIRED>
__device__ __forceinline__ uint2 sg_b_entry(const SgIn &in, uint32_t p)
{
    if constexpr (PAIRED) return in.b_ent[p];
    return make_uint2((uint32_t)in.b_col[p], __float_as_uint(in.b_val[p]));
}

template <bool PAIRED>
__device__ __forceinline__ SgRowInfo sg_row_info(uint32_t row, const SgIn &in)
{
    SgRowInfo r;
    r.row = row;
    r.P = in.P[row];
    r.out_base = in.Poff[row];
    r.ast = in.a_start[row];
    r.la = (uint32_t)in.a_len[row];
    r.fo = PAIRED ? in.a_foff[row] : 0u;
    return r;
}

// Rank sort of a team's P staged keys in LDS, for teams of at most a wave.
// The keys are distinct, so a key's sorted position is the number of smaller
// keys: lane t holds keys t, t + NT, ... in registers and compares them with
// every key of the row, read back one at a time (the team's lanes all read the
// same word: one broadcast per key), then every key is written to its
// position.  P * KPL compares per lane.
template <int NT, int KPL, typename K>
__device__ __forceinline__ void team_rank_sort(K *key, uint32_t P)
{
    const uint32_t t = threadIdx.x % NT;
    K mk[KPL];
    uint32_t rk[KPL];
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        const uint32_t i = t + (uint32_t)r * NT;
        mk[r] = i < P ? key[i] : (K)~0ull;
        rk[r] = 0;
    }
    uint32_t j = 0;
    for (; j + 4 <= P; j += 4) {
        K k0, k1, k2, k3;
        if constexpr (sizeof(K) == 4) {
            // four keys per read (the team's key row is 16-byte aligned)
            const uint4 q = *reinterpret_cast<const uint4 *>(key + j);
            k0 = q.x;
            k1 = q.y;
            k2 = q.z;
            k3 = q.w;
        } else {
            k0 = key[j];
            k1 = key[j + 1];
            k2 = key[j + 2];
            k3 = key[j + 3];
        }
#pragma unroll
        for (int r = 0; r < KPL; ++r)
            rk[r] += (uint32_t)(k0 < mk[r]) + (uint32_t)(k1 < mk[r]) + (uint32_t)(k2 < mk[r]) +
                     (uint32_t)(k3 < mk[r]);
    }
    for (; j < P; ++j) {
        const K kj = key[j];
#pragma unroll
        for (int r = 0; r < KPL; ++r) rk[r] += (uint32_t)(kj < mk[r]);
    }
    team_sync<NT>();  // every read of the row is done before the scatter
#pragma unroll
    for (int r = 0; r < KPL; ++r)
        if (t + (uint32_t)r * NT < P) key[rk[r]] = mk[r];
    team_sync<NT>();
}

// Bitonic network over LDS: the sort of the rows whose columns crowd into few
// buckets (keys past P are padding and sort last; key holds next_pow2(P)).
template <int NT, typename K>
__device__ void team_bitonic_sort(K *key, uint32_t P)
{
    const uint32_t t = threadIdx.x % NT;
    const uint32_t n2 = next_pow2(P < 2 * NT ? 2 * NT : P);
    for (uint32_t p = P + t; p < n2; p += NT) key[p] = (K)~0ull;
    team_sync<NT>();
    for (uint32_t k = 2; k <= n2; k <<= 1) {
        for (uint32_t js = k >> 1; js > 0; js >>= 1) {
            for (uint32_t c = t; c < n2 / 2; c += NT) {
                const uint32_t i1 = (c / js) * 2 * js + (c % js);
                const uint32_t i2 = i1 + js;
                const bool asc = (i1 & k) == 0;
                const K ka = key[i1], kb = key[i2];
                if ((ka > kb) == asc) {
                    key[i1] = kb;
                    key[i2] = ka;
                }
            }
            team_sync<NT>();
        }
    }
}

// Bucket sort of a team's P <= NT * KPL staged keys in LDS.  A key's bucket is
// its place between the row's smallest and largest key, in NT * BPL equal
// steps (a float product: monotone in the key, so buckets are in key order).
// The buckets are counted by LDS atomics, scanned, and filled in any order; a
// key's sorted position is then its bucket's start plus the smaller keys of
// its own bucket.  Columns that spread over the row's range leave about one
// key per bucket, so a key costs a few LDS accesses instead of a compare with
// every other key of the row (the rank sort) or log^2-many passes (the
// bitonic network).  Returns false, with all keys in LDS, when a bucket of
// the wave (of the workgroup for NT > 64) holds more than BK_CROWD keys: the
// caller then sorts them without buckets.
// hist: NT * BPL / 2 + 1 words, two 16-bit counters to a word.
constexpr uint32_t BK_CROWD = 24;
template <int KPL>
constexpr int bucket_bpl() { return KPL > 8 ? 8 : KPL; }
template <int NT, int KPL, int GB, typename K>
__device__ __forceinline__ bool team_bucket_sort(K *key, uint32_t *hist, uint32_t P, uint32_t *lds_w)
{
    constexpr int BPL = bucket_bpl<KPL>();
    constexpr uint32_t NB = (uint32_t)NT * BPL;
    static_assert(BPL % 2 == 0, "whole counter words per lane");
    const uint32_t t = threadIdx.x % NT;
    auto place = [](K k) { return sizeof(K) == 4 ? (uint32_t)k : (uint32_t)((uint64_t)k >> GB); };
    K mk[KPL];
    uint32_t lo = ~0u, hi = 0u;
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        const uint32_t i = t + (uint32_t)r * NT;
        mk[r] = key[i < P ? i : 0u];
        const uint32_t b = place(mk[r]);
        lo = b < lo ? b : lo;
        hi = b > hi ? b : hi;
    }
#pragma unroll
    for (int i = 0; i < BPL / 2; ++i) hist[(uint32_t)i * NT + t] = 0u;
    // over the 16 lanes of a DPP row by rotations, across rows by permutes
    auto both = [&](uint32_t l2, uint32_t h2) {
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
    };
    both(dpp_u32<DPP_ROW_ROR(8)>(lo, lo), dpp_u32<DPP_ROW_ROR(8)>(hi, hi));
    both(dpp_u32<DPP_ROW_ROR(4)>(lo, lo), dpp_u32<DPP_ROW_ROR(4)>(hi, hi));
    both(dpp_u32<DPP_ROW_ROR(2)>(lo, lo), dpp_u32<DPP_ROW_ROR(2)>(hi, hi));
    both(dpp_u32<DPP_ROW_ROR(1)>(lo, lo), dpp_u32<DPP_ROW_ROR(1)>(hi, hi));
    if constexpr (NT >= 64) {
#pragma unroll
        for (int d = 16; d < 64; d <<= 1) both((uint32_t)__shfl_xor((int)lo, d), (uint32_t)__shfl_xor((int)hi, d));
    }
    if constexpr (NT > 64) {
        constexpr int NW = NT / 64;
        if (lane_id() == 0) {
            lds_w[2 * (t >> 6)] = lo;
            lds_w[2 * (t >> 6) + 1] = hi;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            lo = lds_w[2 * i] < lo ? lds_w[2 * i] : lo;
            hi = lds_w[2 * i + 1] > hi ? lds_w[2 * i + 1] : hi;
        }
    }
    team_sync<NT>();
    const float scale = (float)NB / ((float)(hi - lo) + 1.0f);
    uint32_t bo[KPL];  // bucket, and the key's arrival in it << 16
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        bo[r] = 0;
        if (t + (uint32_t)r * NT < P) {
            uint32_t b = (uint32_t)((float)(place(mk[r]) - lo) * scale);
            b = b < NB ? b : NB - 1;
            const uint32_t sh = (b & 1u) * 16u;
            bo[r] = b | (((atomicAdd(&hist[b >> 1], 1u << sh) >> sh) & 0xffffu) << 16);
        }
    }
    team_sync<NT>();
    // exclusive starts, BPL consecutive buckets per lane
    uint32_t w[BPL / 2], sum = 0;
#pragma unroll
    for (int i = 0; i < BPL / 2; ++i) {
        w[i] = hist[t * (BPL / 2) + i];
        sum += (w[i] & 0xffffu) + (w[i] >> 16);
    }
    uint32_t tot;
    uint32_t run = team_excl_scan<NT>(sum, lds_w, &tot);
#pragma unroll
    for (int i = 0; i < BPL / 2; ++i) {
        const uint32_t a = run + (w[i] & 0xffffu);
        hist[t * (BPL / 2) + i] = run | (a << 16);
        run = a + (w[i] >> 16);
    }
    if (t == 0) hist[NB / 2] = P;
    team_sync<NT>();
    const uint16_t *start = reinterpret_cast<const uint16_t *>(hist);
    uint32_t l[KPL], n[KPL], most = 0;
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        l[r] = n[r] = 0;
        if (t + (uint32_t)r * NT < P) {
            const uint32_t b = bo[r] & 0xffffu;
            l[r] = start[b];
            n[r] = start[b + 1] - l[r];
            key[l[r] + (bo[r] >> 16)] = mk[r];
            most = n[r] > most ? n[r] : most;
        }
    }
    team_sync<NT>();
    bool crowded;
    if constexpr (NT > 64) crowded = __syncthreads_or(most > BK_CROWD);
    else crowded = __any(most > BK_CROWD);
    if (crowded) return false;
    // smaller keys of the own bucket: the wave's fullest bucket sets the
    // rounds, each with one independent read per key
    uint32_t rk[KPL];
#pragma unroll
    for (int r = 0; r < KPL; ++r) rk[r] = l[r];
    for (uint32_t d = 0; __any(most > 1 && d < most); ++d) {
#pragma unroll
        for (int r = 0; r < KPL; ++r)
            if (d < n[r]) rk[r] += (uint32_t)(key[l[r] + d] < mk[r]);
    }
    team_sync<NT>();
#pragma unroll
    for (int r = 0; r < KPL; ++r)
        if (n[r] > 1) key[rk[r]] = mk[r];
    team_sync<NT>();
    return true;
}

// Sort a team's row: buckets, with the smallest per-lane key count that holds
// it; where they are crowded, the rank sort (teams of at most a wave and at
// most 8 keys per lane) or the bitonic network.
template <int NT, int KPL, int GB, typename K>
__device__ __forceinline__ void team_sort(K *key, uint32_t *hist, uint32_t P, uint32_t *lds_w)
{
    if (team_bucket_sort<NT, KPL, GB, K>(key, hist, P, lds_w)) return;
    if constexpr (NT < 64) team_rank_sort<NT, KPL, K>(key, P);
    else if constexpr (NT == 64 && KPL <= 4) team_rank_sort<NT, KPL, K>(key, P);
    else team_bitonic_sort<NT, K>(key, P);
}

// The expansion of up to TEAM entries of a team's row (tot partials from
// generation gbase): the entries with partials leave a bit each at their first
// one in a map of the row's at most 32 * KPL / 2 partials (in hist, free until the sort)
// and, by their rank, their displacement and value in a table, so a partial's
// entry is a bit count; a search of the entries' offsets took four dependent LDS
// reads and 24 instructions per partial (the four classes on 2M Poisson rows with
// 8 entries: 994 -> 937 us).
template <bool PAIRED, int GB, int KPL>
__device__ __forceinline__ void sg_expand_team(const SgIn &in, uint32_t lb, uint32_t sb, float va, uint32_t ex,
                                               uint32_t tot, uint32_t gbase, uint32_t *key, float *val,
                                               uint32_t *map, uint32_t *s_sb, float *s_va)
{
    constexpr int W = KPL / 2;  // words of 32 partials
    static_assert(KPL % 2 == 0 && TEAM == 16, "two partials per lane and word");
    const uint32_t t = threadIdx.x % TEAM;
    if (t < W) map[t] = 0u;
    const uint32_t some = (uint32_t)(__ballot(lb > 0u) >> (lane_id() & ~(TEAM - 1))) & 0xffffu;
    team_sync<TEAM>();
    if (lb > 0u) {
        const uint32_t k = (uint32_t)__popc(some & ((1u << t) - 1u));
        s_sb[k] = sb - ex;  // B's entry of a partial less the partial
        s_va[k] = va;
        atomicOr(&map[ex >> 5], 1u << (ex & 31u));
    }
    team_sync<TEAM>();
    if (tot == 0u) return;
    uint32_t m[W], before[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        m[i] = map[i];
        before[i] = i ? before[i - 1] + (uint32_t)__popc(m[i - 1]) : ~0u;
    }
    // every load before the first use (a lane past tot reads entry 0 of B and
    // writes nothing)
    uint2 be[KPL];
    float av[KPL];
#pragma unroll
    for (int i = 0; i < KPL; ++i) {
        const uint32_t pe = (uint32_t)i * TEAM + t;
        const uint32_t q = before[i / 2] + (uint32_t)__popc(m[i / 2] & ((2u << ((i & 1) * TEAM + t)) - 1u));
        be[i] = sg_b_entry<PAIRED>(in, pe < tot ? s_sb[q] + pe : 0u);
        av[i] = s_va[q];
    }
#pragma unroll
    for (int i = 0; i < KPL; ++i) {
        const uint32_t pe = (uint32_t)i * TEAM + t;
        if (pe < tot) {
            const uint32_t g = gbase + pe;
            key[g] = (be[i].x << GB) | g;
            val[g] = av[i] * __uint_as_float(be[i].y);
        }
    }
}

// Sums of a workgroup's sorted row from key `from` > 0 on where columns are few: the
// starts of all runs of equal columns first, as 16-bit positions in list (the bucket
// counters), then a run per thread, so the row waits for its longest run once and not
// once per NT keys.  The product with 128 rows of 16,384 partials in 128 columns:
// 507 -> 236 us, with 2,000 rows of 4,096 in 64 columns: 434 -> 241; with runs of
// SG_RUN keys the list is worth its scan (500 rows of 16,384 in 4,096: 176 -> 161).
// Sums run left to right from 0, exact zeros are dropped; outc: the entries written
// before.  Returns those written now too.
constexpr uint32_t SG_RUN = 4;
template <int NT, int GB, int KPL, typename K>
__device__ uint32_t sg_sum_runs(const K *key, const float *val, uint32_t *list, uint32_t from, uint32_t P,
                                uint64_t out_base, uint32_t outc, const SgOut &out, uint32_t *lds_w)
{
    constexpr uint32_t GM = (1u << GB) - 1u, CAP = (uint32_t)NT * bucket_bpl<KPL>();
    static_assert((uint32_t)NT * KPL <= 2 * CAP, "half of the starts fit the list");
    uint16_t *start = reinterpret_cast<uint16_t *>(list);
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));  // positions of its own: those of the sort would spill
    while (from < P) {
        uint32_t own = 0;  // the starts among the thread's KPL positions, a bit each
#pragma unroll
        for (int r = 0; r < KPL; ++r) {
            const uint32_t p = from + t * KPL + (uint32_t)r;
            if (p < P && (uint32_t)(key[p - 1u] >> GB) != (uint32_t)(key[p] >> GB)) own |= 1u << r;
        }
        uint32_t runs, tot, at = team_excl_scan<NT>((uint32_t)__popc(own), lds_w, &runs);
        uint32_t to = P;
        if (runs > CAP) {  // those of the first half of the keys now
            if (t == NT / 2) lds_w[0] = at;
            if (t >= NT / 2) own = 0u;
            __syncthreads();
            runs = lds_w[0];
            to = from + (uint32_t)NT / 2 * KPL;
        }
        for (; own; own &= own - 1u) start[at++] = (uint16_t)(from + t * KPL + (uint32_t)__ffs((int)own) - 1u);
        __syncthreads();
        for (uint32_t i0 = 0; i0 < runs; i0 += NT) {
            const uint32_t i = i0 + t;
            float s = 0.0f;
            uint32_t c = 0;
            if (i < runs) {
                uint32_t q = start[i];
                const uint32_t end = i + 1u < runs ? start[i + 1u] : P;
                c = (uint32_t)(key[q] >> GB);
                for (; q + 4u <= end && (uint32_t)(key[q + 3u] >> GB) == c; q += 4u) {
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = val[(uint32_t)key[q + j] & GM];
#pragma unroll
                    for (int j = 0; j < 4; ++j) s = s + v[j];
                }
                for (; q < end && (uint32_t)(key[q] >> GB) == c; ++q) s = s + val[(uint32_t)key[q] & GM];
            }
            const bool emit = s != 0.0f;
            const uint32_t pos = team_excl_scan<NT>(emit ? 1u : 0u, lds_w, &tot);
            if (emit) {
                out.tcol[out_base + outc + pos] = (int32_t)c;
                out.tval[out_base + outc + pos] = s;
            }
            outc += tot;
        }
        __syncthreads();
        from = to;
    }
    return outc;
}

// KPL: keys per lane of the sort, fixed by the row's class (P <= KPL * NT).  The products stay where the expansion put them
// (generation order); only the keys are sorted, and a sorted key names its
// product by its generation bits.
template <bool PAIRED, int NT, int GB, typename K, int KPL>
__device__ void sg_row(const SgRowInfo &ri, const SgIn &in, const SgOut &out, K *key, float *val, uint32_t *hist,
                       uint32_t *s_ex, uint32_t *s_sb, float *s_va, uint32_t *lds_w)
{
    const uint32_t t = threadIdx.x % NT;
    const uint32_t row = ri.row, P = ri.P, ast = ri.ast, la = ri.la;
    const uint64_t out_base = ri.out_base;
    // 1. expand in generation order
    uint32_t gbase = 0;
    for (uint32_t a0 = 0; a0 < la; a0 += NT) {
        const uint32_t a = a0 + t;
        uint32_t lb = 0, sb = 0;
        float va = 0.0f;
        if (a < la) {
            const uint2 q = sg_b_row<PAIRED>(in, ri, a);
            va = in.a_val[(uint64_t)ast + a];
            sb = q.x;
            lb = q.y;
        }
        uint32_t tot;
        const uint32_t ex = team_excl_scan<NT>(lb, lds_w, &tot);
        if constexpr (NT == TEAM) {
            sg_expand_team<PAIRED, GB, KPL>(in, lb, sb, va, ex, tot, gbase, key, val, hist, s_sb, s_va);
            gbase += tot;
            team_sync<NT>();
            continue;
        }
        s_ex[t] = ex;
        s_sb[t] = sb;
        s_va[t] = va;
        team_sync<NT>();
        // up to SG_EX partials per lane per round, every load of a round
        // issued before the first wait (a lane past tot reads entry 0 of B
        // and writes nothing)
        constexpr int EX = KPL < SG_EX ? KPL : SG_EX;
        for (uint32_t e0 = 0; e0 < tot; e0 += EX * NT) {
            uint2 be[EX];
            float av[EX];
#pragma unroll
            for (int i = 0; i < EX; ++i) {
                const uint32_t pe = e0 + (uint32_t)i * NT + t;
                const uint32_t q = find_seg_team<NT>(s_ex, pe < tot ? pe : 0u);
                be[i] = sg_b_entry<PAIRED>(in, pe < tot ? s_sb[q] + (pe - s_ex[q]) : 0u);
                av[i] = s_va[q];
            }
#pragma unroll
            for (int i = 0; i < EX; ++i) {
                const uint32_t pe = e0 + (uint32_t)i * NT + t;
                if (pe < tot) {
                    const uint32_t g = gbase + pe;
                    key[g] = (K)(((uint64_t)be[i].x << GB) | g);
                    val[g] = av[i] * __uint_as_float(be[i].y);
                }
            }
        }
        gbase += tot;
        team_sync<NT>();
    }
    // 2. sort by (column, generation)
    if constexpr (KPL == 2) {
        // 32 partials: 64 compares per lane, no more than the buckets cost
        team_rank_sort<NT, KPL, K>(key, P);
    } else {
        team_sort<NT, KPL, GB, K>(key, hist, P, lds_w);
    }
    // 3. runs of equal columns, summed left to right from 0; drop exact zeros
    constexpr uint32_t GM = (1u << GB) - 1u;
    uint32_t outc = 0, from = P;
    for (uint32_t p0 = 0; p0 < P; p0 += NT) {
        const uint32_t p = p0 + t;
        bool emit = false;
        float s = 0.0f;
        uint32_t c = 0;
        // the key, its neighbours and its product without a branch: most runs
        // are one key
        const uint32_t pc = p < P ? p : 0u;
        const K k = key[pc], kp = key[pc > 0u ? pc - 1u : 0u], kn = key[pc + 1u < P ? pc + 1u : pc];
        c = (uint32_t)(k >> GB);
        if (p < P && (p == 0u || (uint32_t)(kp >> GB) != c)) {
            s = 0.0f + val[(uint32_t)k & GM];
            if (p + 1u < P && (uint32_t)(kn >> GB) == c) {
                for (uint32_t q = p + 1u; q < P; ++q) {
                    const K kq = key[q];
                    if ((uint32_t)(kq >> GB) != c) break;
                    s = s + val[(uint32_t)kq & GM];
                }
            }
            emit = s != 0.0f;
        }
        // place among the team's emitting threads
        uint32_t pos, tot;
        const uint64_t m = __ballot(emit);
        if constexpr (NT < 64) {
            const uint32_t mt = (uint32_t)(m >> (lane_id() & ~(NT - 1))) & ((1u << NT) - 1u);
            pos = (uint32_t)__popc(mt & ((1u << t) - 1u));
            tot = (uint32_t)__popc(mt);
        } else if constexpr (NT == 64) {
            pos = (uint32_t)__popcll(m & lanemask_lt());
            tot = (uint32_t)__popcll(m);
        } else {
            pos = team_excl_scan<NT>(emit ? 1u : 0u, lds_w, &tot);
        }
        if (emit) {
            out.tcol[out_base + outc + pos] = (int32_t)c;
            out.tval[out_base + outc + pos] = s;
        }
        outc += tot;
        if (NT > 64 && tot * SG_RUN <= NT) {
            from = p0 + NT;
            break;
        }
    }
    if constexpr (NT > 64) outc = sg_sum_runs<NT, GB, KPL, K>(key, val, hist, from, P, out_base, outc, out, lds_w);
    if (t == 0) out.cnt[row] = outc;
    team_sync<NT>();
}

// Team loop over a class list: team `first`, stride `step`.  The next row's
// id and info are loaded one and two iterations ahead.
template <bool PAIRED, int CLS, typename F>
__device__ __forceinline__ void sg_rows(SgList<CLS> list, uint32_t n, uint32_t first, uint32_t step, const SgIn &in, F &&body)
{
    if (first >= n) return;
    SgRowInfo cur = sg_row_info<PAIRED>(list[first], in);
    uint32_t next_id = first + step < n ? list[first + step] : 0u;
    for (uint32_t i = first; i < n; i += step) {
        SgRowInfo nxt{};
        if (i + step < n) nxt = sg_row_info<PAIRED>(next_id, in);
        const uint32_t nn_id = i + 2 * step < n ? list[i + 2 * step] : 0u;
        body(cur);
        cur = nxt;
        next_id = nn_id;
    }
}

// Wave rows: one wave per row, at most 64 * KPL partials.  K: 32-bit sort keys
// (half the LDS per row, more rows in flight) when B's columns allow.
template <bool PAIRED, int KPL, typename K>
__global__ __launch_bounds__(TB) void k_sg_wave(SgList<cl_wave(KPL)> list, const SgState *__restrict__ st,
                                                SgIn in, SgOut out)
{
    static_assert(64 * KPL <= WAVE_MAX, "generations fit their key bits");
    __shared__ __align__(16) K key[TB / 64][64 * KPL];
    __shared__ float val[TB / 64][64 * KPL];
    __shared__ uint32_t hist[TB / 64][64 * bucket_bpl<KPL>() / 2 + 1];
    __shared__ uint32_t s_ex[TB / 64][64], s_sb[TB / 64][64];
    __shared__ float s_va[TB / 64][64];
    const int w = threadIdx.x >> 6;
    const uint32_t n = st->count[cl_wave(KPL)];
    sg_rows<PAIRED>(list, n, blockIdx.x * (TB / 64) + w, gridDim.x * (TB / 64), in, [&](const SgRowInfo &ri) {
        sg_row<PAIRED, 64, WAVE_GB, K, KPL>(ri, in, out, key[w], val[w], hist[w], s_ex[w], s_sb[w], s_va[w], nullptr);
    });
}

// Rows of at most KPL * TEAM partials (class CL_TEAM + KPL / 2 - 1): 16-lane
// teams, four rows per wave.  A row is a chain of round trips, so waves in flight
// are what counts: a team is a DPP row, its scans and bounds stay in registers
// (44, 64, 72 and 96 of them for 2, 4, 6 and 8 keys per lane; with permutes 54, 72,
// 90 and 106), and six keys are held to the 72 that let seven waves share a SIMD.
// The four classes on 2M Poisson rows with 8 entries: 907 -> 866 us.  Loading the
// next row's A entries a row ahead cost more registers than it gave (866 -> 912).
template <bool PAIRED, int KPL>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(KPL == 6 ? 7 : 4))) void k_sg_team(
    SgList<cl_team(KPL)> list, const SgState *__restrict__ st, SgIn in, SgOut out)
{
    constexpr int NTEAM = TB / TEAM;
    // per-team rows padded so the four teams of a wave start on different
    // LDS banks; the pitch keeps every key row 16-byte aligned
    constexpr uint32_t PITCH = KPL * TEAM + 20;
    static_assert(PITCH % 4 == 0, "16-byte aligned key rows");
    __shared__ __align__(16) uint32_t key[NTEAM][PITCH];
    __shared__ float val[NTEAM][PITCH];
    __shared__ uint32_t hist[NTEAM][KPL * TEAM / 2 + 5];
    __shared__ uint32_t s_ex[NTEAM][TEAM], s_sb[NTEAM][TEAM];
    __shared__ float s_va[NTEAM][TEAM];
    const int tm = threadIdx.x / TEAM;
    static_assert(KPL * TEAM <= TEAM_MAX, "a team row fits its LDS row");
    const uint32_t n = st->count[cl_team(KPL)];
    sg_rows<PAIRED>(list, n, blockIdx.x * NTEAM + tm, gridDim.x * NTEAM, in, [&](const SgRowInfo &ri) {
        sg_row<PAIRED, TEAM, TEAM_GB, uint32_t, KPL>(ri, in, out, key[tm], val[tm], hist[tm], s_ex[tm], s_sb[tm], s_va[tm],
                                             nullptr);
    });
}

// One workgroup of NT threads per row of class CLS, at most MAXP partials.
template <bool PAIRED, int CLS, int NT, int GB, uint32_t MAXP, typename K>
__global__ __launch_bounds__(NT) void k_sg_block(SgList<CLS> list, const SgState *__restrict__ st, SgIn in, SgOut out)
{
    constexpr int KPL = MAXP / NT;
    __shared__ __align__(16) K key[MAXP];
    __shared__ float val[MAXP];
    __shared__ uint32_t hist[NT * bucket_bpl<KPL>() / 2 + 1];
    __shared__ uint32_t s_ex[NT], s_sb[NT];
    __shared__ float s_va[NT];
    __shared__ uint32_t lds_w[2 * NT / 64];
    const uint32_t n = st->count[CLS];
    sg_rows<PAIRED>(list, n, blockIdx.x, gridDim.x, in, [&](const SgRowInfo &ri) {
        sg_row<PAIRED, NT, GB, K, KPL>(ri, in, out, key, val, hist, s_ex, s_sb, s_va, lds_w);
    });
}

// ---------------------------------------------------------------------------
// global path for hub rows (more partials than the large-row kernel holds)
// ---------------------------------------------------------------------------
// pre[2h] = len(A row), pre[2h+1] = P for hub row h (index hn: zeros)
__global__ void k_sg_hprep(const uint32_t *__restrict__ hlist, uint32_t hn, const int32_t *__restrict__ a_len,
                           const uint32_t *__restrict__ P, uint32_t *__restrict__ pre)
{
    const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h > hn) return;
    pre[2 * h] = h < hn ? (uint32_t)a_len[hlist[h]] : 0u;
    pre[2 * h + 1] = h < hn ? P[hlist[h]] : 0u;
}

struct EA {
    uint32_t h;
    uint32_t bst;
    float va;
};

// One record per A entry of every hub row (flat over hpre[2h]).
__global__ __launch_bounds__(TB) void k_sg_hentries(const uint32_t *__restrict__ hlist, uint32_t hn,
                                                    const uint32_t *__restrict__ hpre, uint32_t total,
                                                    const uint32_t *__restrict__ a_start,
                                                    const int32_t *__restrict__ a_col, const float *__restrict__ a_val,
                                                    const uint32_t *__restrict__ b_start,
                                                    const int32_t *__restrict__ b_len, EA *__restrict__ ea,
                                                    uint32_t *__restrict__ blen)
{
    __shared__ uint32_t s_off[TB / 64][65];
    const int w = threadIdx.x >> 6;
    const uint64_t wave = (uint64_t)blockIdx.x * (TB / 64) + w;
    const uint32_t per = 256;
    const uint64_t e0 = wave * per;
    if (e0 >= total) return;
    const uint64_t e1 = e0 + per < total ? e0 + per : total;
    wave_visit<2>(hpre, hn, (uint32_t)e0, (uint32_t)e1, s_off[w], [&](bool valid, uint32_t h, uint32_t k, uint32_t e) {
        if (!valid) return;
        const uint64_t ap = (uint64_t)a_start[hlist[h]] + k;
        const int32_t j = a_col[ap];
        EA r;
        r.h = h;
        r.bst = b_start[j];
        r.va = a_val[ap];
        ea[e] = r;
        blen[e] = (uint32_t)b_len[j];
    });
}

// Partials of hub rows in generation order: key = (h, col), value a*b.
__global__ __launch_bounds__(TB) void k_sg_hexpand(const uint32_t *__restrict__ apos, uint32_t nent, uint32_t total,
                                                   const EA *__restrict__ ea, const int32_t *__restrict__ b_col,
                                                   const float *__restrict__ b_val, int cbits,
                                                   uint64_t *__restrict__ key, uint32_t *__restrict__ val)
{
    __shared__ uint32_t s_off[TB / 64][65];
    const int w = threadIdx.x >> 6;
    const uint64_t wave = (uint64_t)blockIdx.x * (TB / 64) + w;
    const uint32_t per = 256;
    const uint64_t e0 = wave * per;
    if (e0 >= total) return;
    const uint64_t e1 = e0 + per < total ? e0 + per : total;
    wave_visit(apos, nent, (uint32_t)e0, (uint32_t)e1, s_off[w], [&](bool valid, uint32_t q, uint32_t k, uint32_t e) {
        if (!valid) return;
        const EA r = ea[q];
        const uint64_t bp = (uint64_t)r.bst + k;
        key[e] = ((uint64_t)r.h << cbits) | (uint32_t)b_col[bp];
        val[e] = __float_as_uint(r.va * b_val[bp]);
    });
}

// Run heads of the sorted hub partials: left-to-right sums, emit flags.
__global__ void k_sg_hreduce(const uint64_t *__restrict__ key, const uint32_t *__restrict__ val, uint32_t n,
                             uint32_t *__restrict__ emit, float *__restrict__ sum)
{
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > n) return;
    uint32_t e = 0;
    if (p < n) {
        const uint64_t k = key[p];
        if (p == 0 || key[p - 1] != k) {
            float s = 0.0f + __uint_as_float(val[p]);
            for (uint32_t q = p + 1; q < n && key[q] == k; ++q) s = s + __uint_as_float(val[q]);
            e = s != 0.0f ? 1u : 0u;
            sum[p] = s;
        }
    }
    emit[p] = e;
}

__global__ void k_sg_hwrite(const uint64_t *__restrict__ key, uint32_t n, int cbits, const uint32_t *__restrict__ emit,
                            const uint32_t *__restrict__ epos, const float *__restrict__ sum,
                            const uint32_t *__restrict__ hlist, const uint32_t *__restrict__ hpre,
                            const uint32_t *__restrict__ Poff, int32_t *__restrict__ tcol, float *__restrict__ tval)
{
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || !emit[p]) return;
    const uint64_t k = key[p];
    const uint32_t h = (uint32_t)(k >> cbits);
    const uint32_t first = epos[hpre[2 * h + 1]];  // emits before this hub row
    const uint64_t o = (uint64_t)Poff[hlist[h]] + (epos[p] - first);
    tcol[o] = (int32_t)(k & ((1ull << cbits) - 1ull));
    tval[o] = sum[p];
}

__global__ void k_sg_hcount(const uint32_t *__restrict__ hlist, uint32_t hn, const uint32_t *__restrict__ hpre,
                            const uint32_t *__restrict__ epos, uint32_t *__restrict__ cnt)
{
    const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= hn) return;
    cnt[hlist[h]] = epos[hpre[2 * (h + 1) + 1]] - epos[hpre[2 * h + 1]];
}

// C row table from the output counts.
// Row r of C: chunk [Poff[r], Poff[r] + P[r]) holding cnt[r] entries.
__global__ void k_sg_set_rows(uint32_t R, const uint32_t *__restrict__ Poff, const uint32_t *__restrict__ P,
                              const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ nnz, uint32_t ptot,
                              uint32_t *__restrict__ start, int32_t *__restrict__ len, int32_t *__restrict__ cap,
                              DevState *ds)
{
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    // a row's chunk keeps its P_r slots at Poff[r]; the P_r - cnt_r it does
    // not fill are counted as garbage, so its capacity is its length (bump
    // = sum of capacities + garbage, as for every other producer)
    if (r < R) {
        start[r] = Poff[r];
        len[r] = (int32_t)cnt[r];
        cap[r] = (int32_t)cnt[r];
    }
    if (r == 0) {
        const uint32_t tot = nnz[0];
        ds->bump = ptot;
        ds->nnz = tot;
        ds->garbage = ptot - tot;
        ds->status &= ST_SCAN_FALLBACK;
    }
}

}  // namespace

// Launches `kernel` over the rows of class CLS, `per` rows to a workgroup of nt
// threads, on at most `most` workgroups (they stride over the rest).
struct RowLaunch {
    const SgState &hst;
    const uint32_t *lists;
    uint32_t R;
    const SgState *st;
    const SgIn &in;
    const SgOut &out;
    hipStream_t s;
    template <int CLS>
    void operator()(void (*kernel)(SgList<CLS>, const SgState *, SgIn, SgOut), uint32_t per, uint32_t most, int nt) const
    {
        const uint32_t want = (hst.count[CLS] + per - 1) / per;
        if (want) kernel<<<want < most ? want : most, nt, 0, s>>>(SgList<CLS>(lists, R), st, in, out);
    }
};

// The row kernels of every class; PAIRED as in SgIn.
template <bool PAIRED>
static void launch_rows(const RowLaunch &run, int64_t cols)
{
    run(k_sg_team<PAIRED, 2>, TB / TEAM, 8192, TB);
    run(k_sg_team<PAIRED, 4>, TB / TEAM, 8192, TB);
    run(k_sg_team<PAIRED, 6>, TB / TEAM, 8192, TB);
    run(k_sg_team<PAIRED, 8>, TB / TEAM, 8192, TB);
    if (cols <= WAVE_MAX_COLS32) {
        run(k_sg_wave<PAIRED, 4, uint32_t>, 4, 8192, TB);
        run(k_sg_wave<PAIRED, 8, uint32_t>, 4, 8192, TB);
        run(k_sg_wave<PAIRED, 16, uint32_t>, 4, 8192, TB);
    } else {
        run(k_sg_wave<PAIRED, 4, uint64_t>, 4, 8192, TB);
        run(k_sg_wave<PAIRED, 8, uint64_t>, 4, 8192, TB);
        run(k_sg_wave<PAIRED, 16, uint64_t>, 4, 8192, TB);
    }
    if (cols <= BLOCK_MAX_COLS32) run(k_sg_block<PAIRED, CL_BLOCK, TB, BLOCK_GB, BLOCK_MAX, uint32_t>, 1, 4096, TB);
    else run(k_sg_block<PAIRED, CL_BLOCK, TB, BLOCK_GB, BLOCK_MAX, uint64_t>, 1, 4096, TB);
    if (cols <= BIG_MAX_COLS32) run(k_sg_block<PAIRED, CL_BIG, BIG_TB, BIG_GB, BIG_MAX32, uint32_t>, 1, 1024, BIG_TB);
    else run(k_sg_block<PAIRED, CL_BIG, BIG_TB, BIG_GB, BIG_MAX64, uint64_t>, 1, 1024, BIG_TB);
}

// C = A * B (states known); paired: with the copies of SgIn, in C's workspace.
static dcsr_status spgemm_run(dcsr_handle A, dcsr_handle B, dcsr_handle C, bool paired, hipStream_t s)
{
    const uint32_t R = (uint32_t)A->rows;
    uint32_t *P, *Poff, *cnt, *coff, *lists, *part;
    SgState *st;
    unsigned long long *bsum;
    const unsigned nbR = grid_for(R, TB * SG_CR);  // classify workgroups
    DCSR_TRY(ws_get(C, WS_SG_P, (size_t)(R + 1) * 4, (void **)&P));
    DCSR_TRY(ws_get(C, WS_SG_POFF, (size_t)(R + 1) * 4, (void **)&Poff));
    DCSR_TRY(ws_get(C, WS_SG_CNT, (size_t)(R + 1) * 4, (void **)&cnt));
    DCSR_TRY(ws_get(C, WS_SG_COFF, (size_t)(R + 1) * 4, (void **)&coff));
    DCSR_TRY(ws_get(C, WS_SG_LIST, (size_t)R * 4 * (NCLS / 2), (void **)&lists));
    DCSR_TRY(ws_get(C, WS_SG_STATE, sizeof(SgState), (void **)&st));
    DCSR_TRY(ws_get(C, WS_SG_BSUM, (size_t)nbR * 8, (void **)&bsum));
    DCSR_TRY(ws_get_zeroed(C, WS_PART, scan_part_words(R + 1, 2) * 4, (void **)&part, s));

    SgIn in{P, Poff, A->row_start, A->row_len, A->pool_col, A->pool_val, B->row_start, B->row_len, B->pool_col,
            B->pool_val, nullptr, nullptr, nullptr, nullptr};
    uint2 *ent = nullptr;
    if (paired) {
        uint2 *b_ent;
        DCSR_TRY(ensure_flat(A, s));
        in.a_foff = (const uint32_t *)A->ws.ptr[WS_FOFF];
        DCSR_TRY(ws_get(C, WS_SG_BENT, (size_t)(B->nnz_h + 1) * 8, (void **)&b_ent));
        DCSR_TRY(copy_rows_paired(B, b_ent, B->nnz_h, &in.b_foff, s));
        DCSR_TRY(ws_get(C, WS_SG_ENT, (size_t)(A->nnz_h + 1) * 8, (void **)&ent));
        in.ent = ent;
        in.b_ent = b_ent;
    }

    // 1. partial counts, classes, offsets
    k_sg_state_zero<<<1, 1, 0, s>>>(st);
    if (R > 0) {
        if (paired) k_sg_count<true><<<grid_for(R, TB), TB, 0, s>>>(R, in, ent, P);
        else k_sg_count<false><<<grid_for(R, TB), TB, 0, s>>>(R, in, nullptr, P);
        k_sg_classify<<<nbR, TB, 0, s>>>(R, P, lists, st, cnt, bsum, B->cols <= TEAM_MAX_COLS ? 1u : 0u,
                                         B->cols <= BIG_MAX_COLS32 ? BIG_MAX32 : BIG_MAX64);
        k_sg_total<<<1, 1024, 0, s>>>(st, bsum, (int)nbR);
    }
    DCSR_HIP(scan_exclusive_u32(P, Poff, R, 1, part, Poff + R, s, fault_word(C)));
    SgState hst;
    DCSR_TRY(fetch_words(C, st, sizeof(SgState), &hst, s));
    if (hst.total >= 0xfffffff0ull) return DCSR_ERR_UNSUPPORTED;
    const uint32_t Ptot = (uint32_t)hst.total;

    // C's rows are written in place in its pool at their partial offsets:
    // row r owns the P_r slots from Poff[r] (its chunk; the slots its merged
    // columns do not fill are garbage), so no copy assembles C afterwards
    if ((int64_t)Ptot > C->pool_cap) {
        const int64_t want = (int64_t)(Ptot * C->cfg.pool_factor);
        DCSR_TRY(alloc_pool(C, want > (int64_t)Ptot ? want : (int64_t)Ptot));
    }
    int32_t *tcol = C->pool_col;
    float *tval = C->pool_val;

    // 2. numeric phases
    const SgOut out{tcol, tval, cnt};
    const RowLaunch run{hst, lists, R, st, in, out, s};
    paired ? launch_rows<true>(run, B->cols) : launch_rows<false>(run, B->cols);
    if (hst.count[CL_HUB]) {
        const uint32_t hn = hst.count[CL_HUB];
        static_assert(CL_HUB % 2 == 0, "its list runs forward");
        const uint32_t *hlist = SgList<CL_HUB>(lists, R).p;
        uint32_t *hpre_in, *hpre, *blen, *apos, *emit, *epos, *v0, *v1;
        uint64_t *k0, *k1;
        EA *ea;
        DCSR_TRY(ws_get(C, WS_SG_HPRE, (size_t)(hn + 1) * 16, (void **)&hpre_in));
        hpre = hpre_in + 2 * (hn + 1);
        k_sg_hprep<<<grid_for(hn + 1, TB), TB, 0, s>>>(hlist, hn, A->row_len, P, hpre_in);
        uint32_t htot[2];
        uint32_t *htot_d;
        DCSR_TRY(ws_get(C, WS_TMP2, 64, (void **)&htot_d));
        DCSR_HIP(scan_exclusive_u32(hpre_in, hpre, hn + 1, 2, part, htot_d, s, fault_word(C)));
        DCSR_TRY(fetch_words(C, htot_d, 8, htot, s));
        const uint32_t nent = htot[0], np = htot[1];
        DCSR_TRY(ws_get(C, WS_SG_EA, (size_t)(nent + 1) * sizeof(EA), (void **)&ea));
        DCSR_TRY(ws_get(C, WS_SG_APOS, (size_t)(nent + 2) * 8, (void **)&blen));
        apos = blen + (nent + 1);
        // hpre (the exclusive prefix), not hpre_in (the lengths): the segment
        // search needs monotone offsets
        k_sg_hentries<<<grid_for(nent, 4 * 256) + 1, TB, 0, s>>>(hlist, hn, hpre, nent, A->row_start, A->pool_col,
                                                               A->pool_val, B->row_start, B->row_len, ea, blen);
        size_t pw = scan_part_words(nent + 1, 1);
        if (scan_part_words((int64_t)np + 1, 1) > pw) pw = scan_part_words((int64_t)np + 1, 1);
        if (radix_part_words(np) > pw) pw = radix_part_words(np);
        DCSR_TRY(ws_get_zeroed(C, WS_SCAN, pw * 4, (void **)&part, s));
        DCSR_HIP(scan_exclusive_u32(blen, apos, nent, 1, part, apos + nent, s, fault_word(C)));
        DCSR_TRY(ws_get(C, WS_SG_KEY0, (size_t)(np + 1) * 8, (void **)&k0));
        DCSR_TRY(ws_get(C, WS_SG_KEY1, (size_t)(np + 1) * 8, (void **)&k1));
        DCSR_TRY(ws_get(C, WS_SG_VAL0, (size_t)(np + 1) * 4, (void **)&v0));
        DCSR_TRY(ws_get(C, WS_SG_VAL1, (size_t)(np + 1) * 4, (void **)&v1));
        k_sg_hexpand<<<grid_for(np, 4 * 256) + 1, TB, 0, s>>>(apos, nent, np, ea, B->pool_col, B->pool_val, C->cbits,
                                                              k0, v0);
        uint32_t *hist;
        DCSR_TRY(ws_get(C, WS_HIST, radix_hist_words(np) * 4, (void **)&hist));
        int which = 0;
        DCSR_HIP(radix_sort_pairs(k0, v0, k1, v1, np, bits_for(hn) + C->cbits, hist, part, &which, s));
        uint64_t *key = which ? k1 : k0;
        uint32_t *val = which ? v1 : v0;
        float *sum;
        DCSR_TRY(ws_get(C, WS_SG_FLAG, (size_t)(np + 2) * 8, (void **)&emit));
        sum = (float *)(emit + (np + 2));
        DCSR_TRY(ws_get(C, WS_SG_EPOS, (size_t)(np + 2) * 4, (void **)&epos));
        k_sg_hreduce<<<grid_for(np + 1, TB), TB, 0, s>>>(key, val, np, emit, sum);
        DCSR_HIP(scan_exclusive_u32(emit, epos, np + 1, 1, part, nullptr, s, fault_word(C)));
        k_sg_hwrite<<<grid_for(np, TB), TB, 0, s>>>(key, np, C->cbits, emit, epos, sum, hlist, hpre, Poff, tcol, tval);
        k_sg_hcount<<<grid_for(hn, TB), TB, 0, s>>>(hlist, hn, hpre, epos, cnt);
    }
    DCSR_HIP(hipGetLastError());

    // 3. C's row table: chunks at the partial offsets; nnz from a scan of
    // the row counts
    DCSR_TRY(ws_get_zeroed(C, WS_PART, scan_part_words(R + 1, 1) * 4, (void **)&part, s));
    DCSR_HIP(scan_exclusive_u32(cnt, coff, R, 1, part, coff + R, s, fault_word(C)));
    k_sg_set_rows<<<grid_for(R + 1, TB), TB, 0, s>>>(R, Poff, P, cnt, coff + R, Ptot, C->row_start, C->row_len,
                                                     C->row_cap, C->ds);
    DCSR_HIP(hipGetLastError());
    DCSR_TRY(pull_state(C, s));
    C->canonical = true;
    C->flat_dirty = true;
    C->hubs_dirty = true;
    return DCSR_OK;
}

dcsr_status dcsr_spgemm(dcsr_handle A, dcsr_handle B, dcsr_handle C, dcsr_stream_t stream)
{
    if (!A || !B || !C || C == A || C == B) return DCSR_ERR_INVALID;
    if (A->cols != B->rows || C->rows != A->rows || C->cols != B->cols) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    A->last_stream = B->last_stream = C->last_stream = s;
    DCSR_TRY(refresh_replayed(A, s));
    DCSR_TRY(refresh_replayed(B, s));
    if (!A->state_known) DCSR_TRY(pull_state(A, s));
    if (!B->state_known) DCSR_TRY(pull_state(B, s));
    if (A->nnz_h + B->nnz_h >= C->sg_pair_min) {
        const dcsr_status st = spgemm_run(A, B, C, true, s);
        if (st != DCSR_ERR_OOM) return st;
        // the copies leave no room for the rest (or find none): without them
        (void)hipGetLastError();
        DCSR_TRY(ws_release(C, WS_SG_BENT, s));
        DCSR_TRY(ws_release(C, WS_SG_ENT, s));
    }
    return spgemm_run(A, B, C, false, s);
}
