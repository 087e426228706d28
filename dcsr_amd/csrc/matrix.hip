// matrix.hip -- handle lifetime, COO/CSR -> DCSR load, DCSR -> CSR export,
// compaction (defrag), pool growth, hub-row list, status plumbing.
//
// Reference counterparts: dcsr_matrix::resize (include/dcsr_matrix.h:41-108),
// device::Initialize_Matrix (include/load.h:8-22), device::LoadMatrix
// (include/load.h:27-59, 207-253), device::SortMatrixRow (include/load.h:404-581),
// device::BinRows (include/load.h:583-610).
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <chrono>
#include "dcsr_internal.h"
#include "prims.h"
#include "rowscan.h"
#include "segments.h"

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
namespace {

constexpr int TB = 256;

__global__ void k_fill_i32(int32_t *p, int64_t n, int32_t v)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Empty rows with capacity L: start = r*L (InitializeMatrix_dcsr,
// include/sparse_update.inl:1155-1176).
__global__ void k_init_rows(int64_t R, uint32_t L, uint32_t *start, int32_t *len, int32_t *cap, DevState *ds)
{
    int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < R) {
        start[r] = (uint32_t)(r * L);
        len[r] = 0;
        cap[r] = (int32_t)L;
    }
    if (r == 0) {
        ds->bump = (unsigned long long)R * L;
        ds->nnz = 0;
        ds->garbage = 0;
        ds->status &= ST_SCAN_FALLBACK;
        ds->hub_count = 0;
        ds->hub_chunks = 0;
    }
}

// Raise a load flag from a workgroup in which any thread wants it (every
// thread calls this).  Looked at before it is set, and once per workgroup: on
// unordered input nearly every one raises it, and one access of the same word
// per wave took ten times as long as the rest of the pass (16 -> 143 us over
// 3.2M triples).
__device__ __forceinline__ void raise_load_flag(DevState *ds, uint32_t bit, bool any)
{
    if (__syncthreads_or(any) && threadIdx.x == 0 &&
        !(__hip_atomic_load(&ds->load_flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit))
        atomicOr(&ds->load_flags, bit);
}

// Pack (row, col) into a sort key, LD_PER triples per thread; invalid indices
// become ~0 and raise ST_BAD_INDEX.  Notes whether the triples are out of
// order (a sorted edge list needs no sort).
constexpr int LD_PER = 8;
__global__ __launch_bounds__(TB) void k_pack_keys(const int32_t *__restrict__ rows, const int32_t *__restrict__ cols,
                                                  const float *__restrict__ vals, int64_t n, int64_t R, int64_t C,
                                                  int cbits, uint64_t *__restrict__ key, uint32_t *__restrict__ val,
                                                  DevState *ds)
{
    const int64_t i0 = (int64_t)blockIdx.x * (TB * LD_PER) + threadIdx.x;
    int32_t r[LD_PER], c[LD_PER], rp[LD_PER], cp[LD_PER];
    uint32_t v[LD_PER];
    // all loads in flight first (clamped to the triples there are)
#pragma unroll
    for (int q = 0; q < LD_PER; ++q) {
        const int64_t i = i0 + (int64_t)q * TB < n ? i0 + (int64_t)q * TB : n - 1;
        const int64_t ip = i > 0 ? i - 1 : 0;
        r[q] = rows[i];
        c[q] = cols[i];
        rp[q] = rows[ip];
        cp[q] = cols[ip];
        v[q] = __float_as_uint(vals[i]);
    }
    bool bad = false, down = false;
#pragma unroll
    for (int q = 0; q < LD_PER; ++q) {
        const int64_t i = i0 + (int64_t)q * TB;
        if (i >= n) break;
        const bool b = (r[q] < 0) | (r[q] >= R) | (c[q] < 0) | (c[q] >= C);
        key[i] = b ? ~0ull : (((uint64_t)(uint32_t)r[q] << cbits) | (uint32_t)c[q]);
        val[i] = v[q];
        bad |= b;
        down |= rp[q] > r[q] || (rp[q] == r[q] && cp[q] > c[q]);
    }
    if (__ballot(bad) && lane_id() == 0) atomicOr(&ds->status, ST_BAD_INDEX);
    raise_load_flag(ds, LD_UNSORTED, down);
}

// The same keys for a CSR matrix: a wave owns KEY_SPAN consecutive entries and
// walks the rows they belong to 64 at a time (wave_visit), so an entry costs a
// search of 64 offsets in LDS instead of one of all R offsets in memory.  Entries
// that lie further apart than KEY_WALK rows (a matrix of mostly empty rows) are
// searched for instead, a lane's eight together: a load into 10M rows took 86 ms
// where one wave's entries were the first row's and the last's (now 0.2), 856 us for
// 100,000 entries a hundred rows apart (214).
constexpr uint32_t KEY_SPAN = 512, KEY_WALK = 1024;
__global__ __launch_bounds__(TB) void k_pack_keys_csr(const int32_t *__restrict__ off, uint32_t R,
                                                      const int32_t *__restrict__ cols,
                                                      const float *__restrict__ vals, uint32_t n, int64_t C, int cbits,
                                                      uint64_t *__restrict__ key, uint32_t *__restrict__ val,
                                                      DevState *ds)
{
    __shared__ uint32_t s_off[TB / 64][65];
    const uint32_t *uoff = (const uint32_t *)off;
    uint64_t e0 = ((uint64_t)blockIdx.x * (TB / 64) + (threadIdx.x >> 6)) * KEY_SPAN;
    if (e0 > n) e0 = n;
    const uint32_t e1 = n - (uint32_t)e0 < KEY_SPAN ? n : (uint32_t)e0 + KEY_SPAN;
    bool bad = false, down = false;
    auto pack = [&](bool valid, uint32_t r, uint32_t k, uint32_t e) {
        if (!valid) return;
        const int32_t c = cols[e];
        if (k > 0) down |= cols[e - 1] > c;
        const bool b = (c < 0) | (c >= C);
        key[e] = b ? ~0ull : (((uint64_t)r << cbits) | (uint32_t)c);
        val[e] = __float_as_uint(vals[e]);
        bad |= b;
    };
    if (e0 < e1) {
        const uint32_t j = wave_find_last_le(uoff, R, (uint32_t)e0);
        if (R - j <= KEY_WALK || uoff[j + KEY_WALK] >= e1) {
            wave_visit_from(uoff, R, j, (uint32_t)e0, e1, s_off[threadIdx.x >> 6], pack);
        } else {
            constexpr int PER = KEY_SPAN / 64;
            uint32_t lo[PER], hi[PER];  // off[lo] <= e < off[hi]
            const uint32_t j1 = wave_find_last_le(uoff, R, e1 - 1) + 1;
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                lo[q] = j;
                hi[q] = j1;
            }
            for (uint32_t span = j1 - j; span > 1; span = (span + 1) >> 1) {  // no interval is longer
#pragma unroll
                for (int q = 0; q < PER; ++q) {
                    const uint32_t e = (uint32_t)e0 + (uint32_t)q * 64 + lane_id();
                    const uint32_t mid = lo[q] + ((hi[q] - lo[q]) >> 1);
                    const bool left = uoff[mid] > e;  // mid == lo: it is not
                    hi[q] = left ? mid : hi[q];
                    lo[q] = left ? lo[q] : mid;
                }
            }
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const uint32_t e = (uint32_t)e0 + (uint32_t)q * 64 + lane_id();
                pack(e < e1, lo[q], e < e1 ? e - uoff[lo[q]] : 0u, e);
            }
        }
    }
    if (__ballot(bad) && lane_id() == 0) atomicOr(&ds->status, ST_BAD_INDEX);
    raise_load_flag(ds, LD_UNSORTED, down);
}

__global__ void k_check_offsets(const int32_t *__restrict__ off, int64_t R, DevState *ds)
{
    int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool bad = false;
    if (r < R) bad = off[r + 1] < off[r];
    if (r == 0) {
        bad |= R > 0 && off[0] != 0;
        ds->load_nnz = (unsigned int)off[R];
    }
    if (__ballot(bad) && lane_id() == 0) atomicOr(&ds->status, ST_BAD_INDEX);
}

// Sorted triples into the pool: natural row order without slack, so sorted
// entry i is pool slot i.  A row's length is its last entry's position plus 1
// less its first entry's: the entries at the two ends add them up in row_len
// (zero before; a row of one entry stores its 1).  Also notes duplicate
// coordinates and explicit zeros (non-canonical input).  Bound by the 16 bytes
// read and written per entry; finding a row's end by bisection of the keys
// instead took 275 us of a 3.2M-entry load, this pass takes 14.
__global__ __launch_bounds__(TB) void k_load_place(const uint64_t *__restrict__ key, const uint32_t *__restrict__ val,
                                                   int64_t n, int cbits, int32_t *__restrict__ row_len,
                                                   int32_t *__restrict__ pcol, float *__restrict__ pval, DevState *ds)
{
    const int64_t i0 = (int64_t)blockIdx.x * (TB * LD_PER) + threadIdx.x;
    uint64_t k[LD_PER], kp[LD_PER], kn[LD_PER];
    uint32_t v[LD_PER];
    // all loads in flight first (clamped to the entries there are)
#pragma unroll
    for (int q = 0; q < LD_PER; ++q) {
        const int64_t i = i0 + (int64_t)q * TB < n ? i0 + (int64_t)q * TB : n - 1;
        k[q] = key[i];
        kp[q] = key[i > 0 ? i - 1 : 0];
        kn[q] = key[i + 1 < n ? i + 1 : i];
        v[q] = val[i];
    }
    bool nc = false;
#pragma unroll
    for (int q = 0; q < LD_PER; ++q) {
        const int64_t i = i0 + (int64_t)q * TB;
        if (i >= n) break;
        const uint32_t r = (uint32_t)(k[q] >> cbits);
        const bool head = i == 0 || (uint32_t)(kp[q] >> cbits) != r;
        const bool tail = i == n - 1 || (uint32_t)(kn[q] >> cbits) != r;
        nc |= (i > 0 && kp[q] == k[q]) || __uint_as_float(v[q]) == 0.0f;
        pcol[i] = (int32_t)(k[q] & ((1ull << cbits) - 1ull));
        pval[i] = __uint_as_float(v[q]);
        if (head && tail) row_len[r] = 1;
        else if (head) atomicAdd(&row_len[r], (int32_t)(0u - (uint32_t)i));
        else if (tail) atomicAdd(&row_len[r], (int32_t)(uint32_t)(i + 1));
    }
    raise_load_flag(ds, LD_NONCANON, nc);
}

// Row table of a loaded matrix: the flat offsets are the row starts.
__global__ void k_set_loaded(int64_t R, const uint32_t *__restrict__ foff, uint32_t *__restrict__ start,
                             const int32_t *__restrict__ len, int32_t *__restrict__ cap, DevState *ds, uint64_t nnz)
{
    int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < R) {
        start[r] = foff[r];
        cap[r] = len[r];
    }
    if (r == 0) {
        ds->bump = nnz;
        ds->nnz = (long long)nnz;
        ds->garbage = 0;
        ds->hub_count = 0;
        ds->hub_chunks = 0;
    }
}

// Flat copy of every row into destination offsets (compaction / export).
// dst_off[r] is the row's new start; src rows are (start, len).  Each wave
// owns SPAN destination entries, in chunks of at most 64 rows: a start
// map of the chunk's rows (ranked to rows through `tab`: empty rows share a
// start) gives every entry its row without a search, and all of a lane's
// loads are in flight before its first store.  The wave's first row comes
// from the row map of the flat offsets (one load; a search only past a run of
// 64 or more empty rows).  With row_offsets (an export) the kernel also stores
// the offsets there; nothing is written when the rows hold more than `limit`
// entries, so a caller need not know the count before the launch.  PAIR: the
// entries go to dst_pair as (column, value bits) pairs.
//
// A wave's pass over its entries is one chain of loads, so up to CP_SHORT_MAX
// entries (fewer workgroups than CUs at CP_SPAN) the waves own CP_SHORT: 3,000
// entries 7.4 -> 3.8 us, 200,000 11.7 -> 5.1, 1M (as pairs) 10 -> 8.3; 4M takes
// 18 either way, and 16M (57 us) moves 4.5 TB/s.
constexpr uint32_t CP_SPAN = 1024, CP_SHORT = 256;
constexpr int64_t CP_SHORT_MAX = 1 << 20;
template <bool PAIR, uint32_t SPAN>
__global__ __launch_bounds__(TB) void k_copy_rows(const uint32_t *__restrict__ dst_off,
                                                  const uint32_t *__restrict__ rowmap, uint32_t R, uint64_t limit,
                                                  int32_t *__restrict__ row_offsets,
                                                  const uint32_t *__restrict__ src_start,
                                                  const int32_t *__restrict__ src_col, const float *__restrict__ src_val,
                                                  int32_t *__restrict__ dst_col, float *__restrict__ dst_val,
                                                  uint2 *__restrict__ dst_pair)
{
    constexpr uint32_t PER = SPAN / 64;
    struct Lds {
        uint32_t off[65];
        uint32_t src[64];
        uint32_t pmap[SPAN / 32];
        uint32_t tab[64];
    };
    __shared__ Lds sh[TB / 64];
    Lds &S = sh[threadIdx.x >> 6];
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t total = dst_off[R];  // the offsets decide, not the caller's count
    if (total > limit) return;
    if (row_offsets)
        for (uint64_t r = (uint64_t)blockIdx.x * TB + threadIdx.x; r <= R; r += (uint64_t)gridDim.x * TB)
            row_offsets[r] = (int32_t)dst_off[r];
    const uint64_t nwaves = (uint64_t)gridDim.x * (TB / 64);
    for (uint64_t wave = (uint64_t)blockIdx.x * (TB / 64) + (threadIdx.x >> 6); wave * SPAN < total;
         wave += nwaves) {
        const uint32_t e0 = (uint32_t)(wave * SPAN);
        const uint32_t e1 = total - e0 < SPAN ? total : e0 + SPAN;
        uint32_t j = rowmap[e0 / RS_GRAN];
        if (j + 64u <= R && dst_off[j + 64u] <= e0) j = wave_find_last_le(dst_off, R, e0);
        uint32_t e = e0;
        while (e < e1) {
            const uint32_t t = j + lane;
            const uint32_t off_t = t <= R ? dst_off[t] : 0xffffffffu;
            const uint32_t off_64 = j + 64u <= R ? dst_off[j + 64u] : 0xffffffffu;
            const uint32_t src = t < R ? src_start[t] : 0u;
            S.off[lane] = off_t;
            if (lane == 0) S.off[64] = off_64;
            S.src[lane] = src;
            if (lane < SPAN / 32) S.pmap[lane] = 0u;
            __builtin_amdgcn_wave_barrier();
            const uint32_t wend = S.off[64] < e1 ? S.off[64] : e1;
            const uint32_t cnt = wend - e;
            const int j0 = find_seg64(S.off, e);  // the row holding e
            // rows with entries starting in the chunk
            const bool starts_here = t < R && off_t >= e && off_t < wend && S.off[lane + 1] > off_t;
            if (starts_here) atomicOr(&S.pmap[(off_t - e) >> 5], 1u << ((off_t - e) & 31u));
            __builtin_amdgcn_wave_barrier();
            const StartMap pm = start_map_load(S.pmap, SPAN / 64);
            const uint32_t rank = start_map_rank(pm, starts_here ? off_t - e : 0u);  // every lane takes part
            if (starts_here) S.tab[rank] = lane;
            __builtin_amdgcn_wave_barrier();
            int32_t c[PER];
            float v[PER];
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q) {
                const uint32_t p = q * 64u + lane;
                const uint32_t nst = start_map_count(pm, (int)q);
                c[q] = 0;
                v[q] = 0.0f;
                if (p < cnt) {
                    const uint32_t jr = nst == 0u ? (uint32_t)j0 : S.tab[nst - 1u];
                    const uint64_t sp = (uint64_t)S.src[jr] + (e + p - S.off[jr]);
                    c[q] = src_col[sp];
                    v[q] = src_val[sp];
                }
            }
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q) {
                const uint32_t p = q * 64u + lane;
                if (p < cnt) {
                    if constexpr (PAIR) {
                        dst_pair[e + p] = make_uint2((uint32_t)c[q], __float_as_uint(v[q]));
                    } else {
                        dst_col[e + p] = c[q];
                        dst_val[e + p] = v[q];
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
            e = wend;
            j += 64;
        }
    }
}

// New row table after compaction: start = off[r], cap = len.
__global__ void k_set_compacted(int64_t R, const uint32_t *__restrict__ off, uint32_t *__restrict__ start,
                                const int32_t *__restrict__ len, int32_t *__restrict__ cap, DevState *ds,
                                const uint32_t *__restrict__ total)
{
    int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < R) {
        start[r] = off[r];
        cap[r] = len[r];
    }
    if (r == 0) {
        ds->bump = total ? total[0] : 0u;
        ds->nnz = total ? total[0] : 0;
        ds->garbage = 0;
    }
}

// Canonical form of a natural-order CSR: emit one entry per run of equal
// columns with value (0 + a1) + a2 + ... (stored order) when it is not 0.
//   k_canon_mark   one bit per entry that starts a row;
//   k_canon_count  sums every run into its first entry's value and notes
//                  which entries emit: one 64-bit word per 64 entries, and
//                  the count of each CN_TILE tile;
//   k_canon_write  the emitted entries at the tile's offset plus the bits
//                  before them, and per word the entries emitted before it;
//   k_canon_offsets  the new offset of a row is the count before its first
//                  entry: one word prefix and a popcount.
// The row of an entry is never searched for.  Measured on 3.2M entries in
// 325K rows against one search of the offsets per entry and a scan of one
// flag word per entry: 130 -> 36 us.
constexpr int CN_PER = 8;
constexpr int CN_TILE = TB * CN_PER;
__global__ void k_canon_mark(const uint32_t *__restrict__ off, int64_t R, unsigned long long *__restrict__ starts)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < R && off[r + 1] > off[r]) atomicOr(&starts[off[r] >> 6], 1ull << (off[r] & 63u));
}

__device__ __forceinline__ bool row_starts(const unsigned long long *__restrict__ starts, int64_t i)
{
    return (starts[i >> 6] >> (i & 63)) & 1ull;
}

// s plus the values from entry m on that continue a run of column c, in stored
// order.  Eight entries' loads in flight at a time: one by one, a run is a chain of
// round trips (an export of 1M entries at 100 coordinates: 2.6 ms, now 1.5).
__device__ __forceinline__ float canon_run(const unsigned long long *__restrict__ starts, const int32_t *__restrict__ col,
                                           const float *__restrict__ val, int64_t n, int64_t m, int32_t c, float s)
{
    constexpr int RUN = 8;
    for (;; m += RUN) {
        int32_t cc[RUN];
        float vv[RUN];
        unsigned long long w[RUN];
#pragma unroll
        for (int q = 0; q < RUN; ++q) {
            const int64_t i = m + q < n ? m + q : n - 1;
            cc[q] = col[i];
            vv[q] = val[i];
            w[q] = starts[i >> 6] >> (i & 63);
        }
#pragma unroll
        for (int q = 0; q < RUN; ++q) {
            if (m + q >= n || cc[q] != c || (w[q] & 1ull)) return s;
            s = s + vv[q];
        }
    }
}

__global__ __launch_bounds__(TB) void k_canon_count(const unsigned long long *__restrict__ starts,
                                                    const int32_t *__restrict__ col, float *__restrict__ val,
                                                    int64_t n, unsigned long long *__restrict__ emit,
                                                    uint32_t *__restrict__ tile_cnt)
{
    __shared__ uint32_t wcnt[TB / 64];
    const int w = threadIdx.x >> 6, lane = lane_id();
    const int64_t w0 = (int64_t)blockIdx.x * CN_TILE + w * (64 * CN_PER);  // this wave's entries
    int32_t c[CN_PER], cp[CN_PER], cn[CN_PER];
    float v[CN_PER];
    // all loads in flight first (clamped to the entries there are)
#pragma unroll
    for (int q = 0; q < CN_PER; ++q) {
        const int64_t i = w0 + q * 64 + lane < n ? w0 + q * 64 + lane : n - 1;
        c[q] = col[i];
        cp[q] = col[i > 0 ? i - 1 : 0];
        cn[q] = col[i + 1 < n ? i + 1 : i];
        v[q] = val[i];
    }
    uint32_t cnt = 0;
#pragma unroll
    for (int q = 0; q < CN_PER; ++q) {
        const int64_t i = w0 + q * 64 + lane;
        bool e = false;
        if (i < n && (cp[q] != c[q] || row_starts(starts, i))) {
            float s = 0.0f + v[q];
            // only a run of more than one entry reads on
            if (i + 1 < n && cn[q] == c[q]) {
                s = canon_run(starts, col, val, n, i + 1, c[q], s);
                val[i] = s;  // a run's first entry is read by no other thread's run
            }
            e = s != 0.0f;
        }
        const unsigned long long b = __ballot(e);
        if (lane == 0 && w0 + q * 64 < n) emit[(w0 >> 6) + q] = b;
        cnt += (uint32_t)__popcll(b);
    }
    if (lane == 0) wcnt[w] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) tile_cnt[blockIdx.x] = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
}

// total[0] > cap: the caller's buffers are too small, nothing is written.
__global__ __launch_bounds__(TB) void k_canon_write(const int32_t *__restrict__ col, const float *__restrict__ val,
                                                    int64_t n, const unsigned long long *__restrict__ emit,
                                                    const uint32_t *__restrict__ tile_off,
                                                    const uint32_t *__restrict__ total, uint64_t cap,
                                                    uint32_t *__restrict__ word_pre, int32_t *__restrict__ ocol,
                                                    float *__restrict__ oval)
{
    if (total[0] > cap) return;
    const int lane = lane_id();
    const int64_t t0 = (int64_t)blockIdx.x * CN_TILE;
    const int64_t w0 = t0 + (threadIdx.x >> 6) * (64 * CN_PER);
    // the tile's 32 words, one per lane, and the entries emitted before each
    const int64_t wi = (t0 >> 6) + lane;
    const unsigned long long word = lane < CN_TILE / 64 && wi * 64 < n ? emit[wi] : 0ull;
    const uint32_t pc = (uint32_t)__popcll(word);
    const uint32_t pre = tile_off[blockIdx.x] + wave_incl_scan_u32(pc) - pc;
    if (threadIdx.x < CN_TILE / 64 && wi * 64 < n) word_pre[wi] = pre;
#pragma unroll
    for (int q = 0; q < CN_PER; ++q) {
        const int64_t i = w0 + q * 64 + lane;
        const int src = (threadIdx.x >> 6) * CN_PER + q;
        const unsigned long long m = ((unsigned long long)(uint32_t)__shfl((int)(uint32_t)(word >> 32), src) << 32) |
                                     (uint32_t)__shfl((int)(uint32_t)word, src);
        const uint32_t p = (uint32_t)__shfl((int)pre, src) + (uint32_t)__popcll(m & lanemask_lt());
        if ((m >> lane) & 1ull) {
            ocol[p] = col[i];
            oval[p] = val[i];
        }
    }
}

__global__ void k_canon_offsets(const uint32_t *__restrict__ off_in, int64_t R,
                                const unsigned long long *__restrict__ emit, const uint32_t *__restrict__ word_pre,
                                const uint32_t *__restrict__ total, uint64_t cap, int32_t *__restrict__ off_out,
                                uint32_t n)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > R || total[0] > cap) return;
    const uint32_t o = off_in[r];
    off_out[r] = (int32_t)(o < n ? word_pre[o >> 6] + (uint32_t)__popcll(emit[o >> 6] & ((1ull << (o & 63u)) - 1ull))
                                 : total[0]);
}

// Number of rows longer than DCSR_HUB_LEN (reported by dcsr_query).
__global__ void k_count_hubs(int64_t R, const int32_t *__restrict__ len, DevState *ds)
{
    int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool hub = r < R && len[r] > DCSR_HUB_LEN;
    uint64_t m = __ballot(hub);
    if (m && lane_id() == 0) atomicAdd(&ds->hub_count, (uint32_t)__popcll(m));
}

__global__ void k_zero_hubs(DevState *ds) { ds->hub_count = 0; }

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
dcsr_status dcsr_hip_fail(hipError_t e, const char *what, const char *file, int line)
{
    if (getenv("DCSR_VERBOSE"))
        fprintf(stderr, "[dcsr] HIP error %d (%s) in %s at %s:%d\n", (int)e, hipGetErrorString(e), what, file, line);
    return e == hipErrorOutOfMemory ? DCSR_ERR_OOM : DCSR_ERR_HIP;
}

const char *dcsr_status_string(dcsr_status s)
{
    switch (s) {
    case DCSR_OK: return "ok";
    case DCSR_ERR_INVALID: return "invalid argument";
    case DCSR_ERR_BAD_INDEX: return "row or column index out of range";
    case DCSR_ERR_POOL_EXHAUSTED: return "entry pool exhausted";
    case DCSR_ERR_SEGMENT_OVERFLOW: return "row segment overflow";
    case DCSR_ERR_HIP: return "HIP runtime error";
    case DCSR_ERR_OOM: return "device out of memory";
    case DCSR_ERR_CAPACITY: return "output buffer too small";
    case DCSR_ERR_UNSUPPORTED: return "unsupported";
    case DCSR_ERR_TOO_LARGE: return "request exceeds the allocation-free entry point's fixed scratch";
    }
    return "unknown";
}

namespace {
__global__ void k_zero_words(uint32_t *p, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}
}  // namespace

static void release_retired(dcsr_handle h);

// Grow a slot.  The old buffer may still be read by work queued on any
// stream, so it is retired (freed at the next state read-back or at
// destroy), never freed here: hipFree would wait for the whole device.
static dcsr_status ws_grow(dcsr_handle h, WsSlot slot, size_t bytes)
{
    if (h->ws.ptr[slot]) {
        if (h->nretired == (int)(sizeof(h->retired) / sizeof(h->retired[0]))) {
            DCSR_HIP(hipDeviceSynchronize());
            release_retired(h);
        }
        h->retired[h->nretired++] = h->ws.ptr[slot];
    }
    h->ws.ptr[slot] = nullptr;
    h->ws.bytes[slot] = 0;
    const size_t nb = bytes + bytes / 4;  // headroom for growing batches
    DCSR_HIP(hipMalloc(&h->ws.ptr[slot], nb));
    h->ws.bytes[slot] = nb;
    return DCSR_OK;
}

dcsr_status ws_get(dcsr_handle h, WsSlot slot, size_t bytes, void **out)
{
    if (bytes == 0) bytes = 16;
    if (h->ws.bytes[slot] < bytes) DCSR_TRY(ws_grow(h, slot, bytes));
    *out = h->ws.ptr[slot];
    return DCSR_OK;
}

dcsr_status ws_release(dcsr_handle h, WsSlot slot, hipStream_t s)
{
    DCSR_HIP(hipStreamSynchronize(s));
    release_retired(h);
    if (h->ws.ptr[slot]) DCSR_HIP(hipFree(h->ws.ptr[slot]));
    h->ws.ptr[slot] = nullptr;
    h->ws.bytes[slot] = 0;
    return DCSR_OK;
}

dcsr_status ws_get_zeroed(dcsr_handle h, WsSlot slot, size_t bytes, void **out, hipStream_t s)
{
    if (bytes == 0) bytes = 16;
    if (h->ws.bytes[slot] < bytes) {
        DCSR_TRY(ws_grow(h, slot, bytes));
        // stream-ordered before the slot's first use on s
        const int64_t words = (int64_t)(h->ws.bytes[slot] / 4);
        int64_t blocks = (words + 255) / 256;
        if (blocks > 1024) blocks = 1024;
        k_zero_words<<<(unsigned)blocks, 256, 0, s>>>((uint32_t *)h->ws.ptr[slot], words);
        DCSR_HIP(hipGetLastError());
    }
    *out = h->ws.ptr[slot];
    return DCSR_OK;
}


namespace {
// One wave copies a few device words into coherent host memory, then stores the
// sequence number with a release at system scope.
__global__ void k_fetch(const uint32_t *__restrict__ src, int words, HostFetch *dst, uint64_t seq)
{
    for (int i = threadIdx.x; i < words; i += 64)
        __hip_atomic_store(&dst->words[i], src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    if (threadIdx.x == 0) __hip_atomic_store(&dst->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

// A kernel's store and a host poll instead of a copy and a stream wait: a read
// of the state after a small update took about 25 us of idle GPU, now about 10.
// The poll is bounded (FETCH_SPIN_US): a longer wait, and any error, is the
// stream wait's.
dcsr_status fetch_words(dcsr_handle h, const void *src, size_t bytes, void *dst, hipStream_t s)
{
    constexpr int FETCH_SPIN_US = 500;
    if (bytes > sizeof(h->hfetch->words) || bytes % 4 != 0) return DCSR_ERR_INVALID;
    const uint64_t seq = ++h->fetch_seq;
    k_fetch<<<1, 64, 0, s>>>((const uint32_t *)src, (int)(bytes / 4), h->dfetch, seq);
    DCSR_HIP(hipGetLastError());
    const auto t0 = std::chrono::steady_clock::now();
    auto landed = [&] { return __atomic_load_n(&h->hfetch->seq, __ATOMIC_ACQUIRE) == seq; };
    for (int polls = 0; !landed(); ++polls) {
        if ((polls & 63) == 63 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(FETCH_SPIN_US)) {
            DCSR_HIP(hipStreamSynchronize(s));
            if (!landed()) return DCSR_ERR_HIP;
            break;
        }
        __builtin_ia32_pause();
    }
    memcpy(dst, h->hfetch->words, bytes);
    return DCSR_OK;
}

dcsr_status pull_state(dcsr_handle h, hipStream_t s)
{
    DCSR_TRY(fetch_words(h, h->ds, sizeof(DevState), h->hs, s));
    if (h->nretired) release_retired(h);
    h->nnz_h = h->hs->nnz;
    h->bump_h = (int64_t)h->hs->bump;
    h->garbage_h = h->hs->garbage;
    state_exact(h);
    return DCSR_OK;
}

bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();  // the null stream beside another stream's capture
        return false;
    }
    return st != hipStreamCaptureStatusNone;
}

dcsr_status refresh_replayed(dcsr_handle h, hipStream_t s)
{
    if (!h->replayed) return DCSR_OK;
    h->flat_dirty = true;
    if (!capturing(s)) return pull_state(h, s);
    h->state_known = false;
    h->nnz_ub = h->bump_ub = h->pool_cap;
    h->snap_valid_from = h->snap_seq + 1;
    return DCSR_OK;
}

void state_exact(dcsr_handle h)
{
    h->state_known = true;
    h->snap_valid_from = h->snap_seq + 1;
}

void state_unknown(dcsr_handle h, int64_t added, int64_t claimed)
{
    const int64_t nnz = live_bound(h) + added, bump = bump_bound(h) + claimed;
    // neither can pass the pool: live entries sit in it and the device
    // rejects a batch whose claims would
    h->nnz_ub = nnz < h->pool_cap ? nnz : h->pool_cap;
    h->bump_ub = bump < h->pool_cap ? bump : h->pool_cap;
    h->cum_add += added;
    h->cum_claim += claimed;
    h->state_known = false;
    h->hubs_dirty = true;
}

// The next NOSYNC update's sequence number (its write kernel stores the
// snapshot under it).
uint64_t snapshot_next(dcsr_handle h) { return ++h->snap_seq; }

// After update seq's launches and its state_unknown: the running sums that
// its snapshot's values are to be read against.
void snapshot_note(dcsr_handle h, uint64_t seq)
{
    h->ring_add[seq % SNAP_RING] = h->cum_add;
    h->ring_claim[seq % SNAP_RING] = h->cum_claim;
}

// The newest landed snapshot k bounds the state: its values plus the sums
// added after update k.  The write kernel stores the values before k (a
// release at system scope), so values read after k was seen are those of k
// or of a later update j, whose sums after j are at least k's: the bound
// holds either way.  A snapshot older than the ring, or than the last change
// the sums do not count, is skipped.
void refresh_bounds(dcsr_handle h)
{
    const uint64_t k = __atomic_load_n(&h->hsnap->seq, __ATOMIC_ACQUIRE);
    if (k == h->snap_used || k < h->snap_valid_from || k > h->snap_seq || k + SNAP_RING <= h->snap_seq) return;
    h->snap_used = k;
    if (h->state_known) return;
    const int64_t nnz = (int64_t)__atomic_load_n(&h->hsnap->nnz, __ATOMIC_RELAXED) +
                        (h->cum_add - h->ring_add[k % SNAP_RING]);
    const int64_t bump = (int64_t)__atomic_load_n(&h->hsnap->bump, __ATOMIC_RELAXED) +
                         (h->cum_claim - h->ring_claim[k % SNAP_RING]);
    if (nnz < h->nnz_ub) h->nnz_ub = nnz;
    if (bump < h->bump_ub) h->bump_ub = bump;
}

static dcsr_status status_from_bits(unsigned bits)
{
    if (bits & ST_BAD_INDEX) return DCSR_ERR_BAD_INDEX;
    if (bits & ST_SEGMENT_OVERFLOW) return DCSR_ERR_SEGMENT_OVERFLOW;
    if (bits & ST_POOL_EXHAUSTED) return DCSR_ERR_POOL_EXHAUSTED;
    return DCSR_OK;
}

// Clears the error bits (the scan-fallback diagnostic stays for the handle's life).
__global__ void k_clear_status(DevState *ds)
{
    ds->status &= ST_SCAN_FALLBACK;
    ds->load_flags = 0;
}

dcsr_status dcsr_get_status(dcsr_handle h)
{
    if (!h) return DCSR_ERR_INVALID;
    DCSR_TRY(pull_state(h, h->last_stream));
    unsigned bits = h->hs->status;
    k_clear_status<<<1, 1, 0, h->last_stream>>>(h->ds);
    DCSR_HIP(hipGetLastError());
    return status_from_bits(bits);
}

static dcsr_status alloc_rows(dcsr_handle h)
{
    size_t R = (size_t)(h->rows > 0 ? h->rows : 1);
    DCSR_HIP(hipMalloc(&h->row_start, R * sizeof(uint32_t)));
    DCSR_HIP(hipMalloc(&h->row_len, R * sizeof(int32_t)));
    DCSR_HIP(hipMalloc(&h->row_cap, R * sizeof(int32_t)));
    return DCSR_OK;
}

dcsr_status alloc_pool(dcsr_handle h, int64_t cap)
{
    if (cap < h->cfg.min_pool) cap = h->cfg.min_pool;
    if (cap > (int64_t)0xfffffff0ll) cap = (int64_t)0xfffffff0ll;
    if (h->pool_col) DCSR_HIP(hipFree(h->pool_col));
    if (h->pool_val) DCSR_HIP(hipFree(h->pool_val));
    h->pool_col = nullptr;
    h->pool_val = nullptr;
    DCSR_HIP(hipMalloc(&h->pool_col, (size_t)cap * sizeof(int32_t)));
    DCSR_HIP(hipMalloc(&h->pool_val, (size_t)cap * sizeof(float)));
    h->pool_cap = cap;
    return DCSR_OK;
}

dcsr_status dcsr_create(dcsr_handle *out, int64_t rows, int64_t cols, const dcsr_config *cfg)
{
    if (!out || rows < 0 || cols < 0 || rows >= (1ll << 31) || cols >= (1ll << 31)) return DCSR_ERR_INVALID;
    dcsr_handle h = (dcsr_handle)calloc(1, sizeof(struct dcsr_matrix_s));
    if (!h) return DCSR_ERR_OOM;
    h->rows = rows;
    h->cols = cols;
    h->rbits = bits_for(rows);
    h->cbits = bits_for(cols);
    h->cfg.pool_factor = 2.0;
    h->cfg.min_pool = 1024;
    h->cfg.allow_grow = 1;
    if (cfg) {
        if (cfg->pool_factor >= 1.0) h->cfg.pool_factor = cfg->pool_factor;
        if (cfg->min_pool > 0) h->cfg.min_pool = cfg->min_pool;
        h->cfg.allow_grow = cfg->allow_grow;
    }
    h->canonical = true;
    h->hubs_dirty = false;
    h->flat_dirty = true;
    state_exact(h);
    // SpMV column panels: at most 1.25M columns (5 MB of x; a 10M x 10M
    // power-law matrix with 160M entries takes 1.56, 1.50, 1.46, 1.53, 1.73 ms
    // with 0.75M, 1M, 1.25M, 1.5M and 2M) for matrices of at least 8M entries;
    // both can be overridden for testing
    h->pnl_cols = 1280 << 10;
    h->pnl_prev_calls = DCSR_PNL_REUSE;  // no evidence yet: a fresh matrix is assumed to be reused
    h->pnl_min_nnz = 8ll << 20;
    if (const char *e = getenv("DCSR_SPMV_PANEL_COLS")) h->pnl_cols = atoll(e) > 0 ? atoll(e) : h->pnl_cols;
    if (const char *e = getenv("DCSR_SPMV_PANEL_MIN_NNZ")) h->pnl_min_nnz = atoll(e) >= 0 ? atoll(e) : h->pnl_min_nnz;
    // SpGEMM: entries of both operands from which it takes copies of them
    // (spgemm.hip); overridden for testing
    h->sg_pair_min = SG_PAIR_MIN;
    if (const char *e = getenv("DCSR_SPGEMM_PAIR_MIN")) h->sg_pair_min = atoll(e) >= 0 ? atoll(e) : h->sg_pair_min;
    // the update tag's starting value (a test of its wrap-around)
    if (const char *e = getenv("DCSR_UPDATE_TAG_START")) h->upd_tag = (uint32_t)strtoul(e, nullptr, 0);
    dcsr_status st = alloc_rows(h);
    if (st == DCSR_OK) st = alloc_pool(h, h->cfg.min_pool);
    if (st == DCSR_OK && hipMalloc(&h->ds, sizeof(DevState)) != hipSuccess) st = DCSR_ERR_OOM;
    if (st == DCSR_OK && hipHostMalloc(&h->hs, sizeof(DevState), hipHostMallocDefault) != hipSuccess) st = DCSR_ERR_OOM;
    // the NOSYNC snapshot: coherent, so the write kernel's stores reach the
    // host without a copy
    if (st == DCSR_OK &&
        hipHostMalloc(&h->hsnap, sizeof(HostSnap), hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
        st = DCSR_ERR_OOM;
    if (st == DCSR_OK &&
        hipHostMalloc(&h->hfetch, sizeof(HostFetch), hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
        st = DCSR_ERR_OOM;
    if (st == DCSR_OK) {
        memset(h->hfetch, 0, sizeof(HostFetch));
        if (hipHostGetDevicePointer((void **)&h->dfetch, h->hfetch, 0) != hipSuccess) st = DCSR_ERR_HIP;
    }
    if (st == DCSR_OK) {
        memset(h->hsnap, 0, sizeof(HostSnap));
        h->snap_valid_from = 1;
        if (hipHostGetDevicePointer((void **)&h->dsnap, h->hsnap, 0) != hipSuccess) st = DCSR_ERR_HIP;
    }
    if (st == DCSR_OK && hipMemset(h->ds, 0, sizeof(DevState)) != hipSuccess) st = DCSR_ERR_HIP;
    if (st == DCSR_OK) {
        // all rows empty
        k_init_rows<<<grid_for(rows, TB), TB>>>(rows, 0, h->row_start, h->row_len, h->row_cap, h->ds);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) st = DCSR_ERR_HIP;
    }
    if (st != DCSR_OK) {
        dcsr_destroy(h);
        return st;
    }
    *out = h;
    return DCSR_OK;
}

dcsr_status dcsr_destroy(dcsr_handle h)
{
    if (!h) return DCSR_ERR_INVALID;
    if (h->last_stream) (void)hipStreamSynchronize(h->last_stream);
    else (void)hipDeviceSynchronize();
    (void)hipFree(h->row_start);
    (void)hipFree(h->row_len);
    (void)hipFree(h->row_cap);
    (void)hipFree(h->pool_col);
    (void)hipFree(h->pool_val);
    (void)hipFree(h->spare_col);
    (void)hipFree(h->spare_val);
    release_retired(h);
    (void)hipFree(h->ds);
    if (h->hs) (void)hipHostFree(h->hs);
    if (h->hsnap) (void)hipHostFree(h->hsnap);
    if (h->hfetch) (void)hipHostFree(h->hfetch);
    for (int i = 0; i < WS_COUNT; ++i)
        if (h->ws.ptr[i]) (void)hipFree(h->ws.ptr[i]);
    free(h);
    return DCSR_OK;
}

dcsr_status dcsr_initialize(dcsr_handle h, int32_t bin_length, dcsr_stream_t stream)
{
    if (!h || bin_length < 0) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    int64_t need = h->rows * (int64_t)bin_length;
    if (need > (int64_t)0xfffffff0ll) return DCSR_ERR_INVALID;
    if (need > h->pool_cap) {
        DCSR_HIP(hipStreamSynchronize(s));
        DCSR_TRY(alloc_pool(h, (int64_t)(need * h->cfg.pool_factor)));
    }
    k_init_rows<<<grid_for(h->rows, TB), TB, 0, s>>>(h->rows, (uint32_t)bin_length, h->row_start, h->row_len,
                                                       h->row_cap, h->ds);
    DCSR_HIP(hipGetLastError());
    h->nnz_h = 0;
    h->bump_h = need;
    h->garbage_h = 0;
    h->hub_rows_h = 0;
    h->hub_chunks_h = 0;
    h->canonical = true;
    h->hubs_dirty = true;
    h->flat_dirty = true;
    state_exact(h);
    return DCSR_OK;
}

// Load sorted-by-key triples into a fresh natural-order pool.
static dcsr_status load_sorted(dcsr_handle h, const uint64_t *key, const uint32_t *val, int64_t n, hipStream_t s)
{
    const int64_t R = h->rows;
    int64_t want = (int64_t)(n * h->cfg.pool_factor);
    if (want < n) want = n;
    if (want > h->pool_cap || n > h->pool_cap) {
        DCSR_HIP(hipStreamSynchronize(s));
        DCSR_TRY(alloc_pool(h, want));
    }
    // the spare pool (compaction target) is sized with the main pool so that
    // compactions during updates allocate nothing
    if (h->spare_cap < h->pool_cap) {
        DCSR_HIP(hipStreamSynchronize(s));
        if (h->spare_col) (void)hipFree(h->spare_col);
        if (h->spare_val) (void)hipFree(h->spare_val);
        h->spare_col = nullptr;
        h->spare_val = nullptr;
        h->spare_cap = 0;
        DCSR_HIP(hipMalloc(&h->spare_col, (size_t)h->pool_cap * 4));
        DCSR_HIP(hipMalloc(&h->spare_val, (size_t)h->pool_cap * 4));
        h->spare_cap = h->pool_cap;
    }
    if (R > 0) k_fill_i32<<<grid_for(R, TB * 4), TB, 0, s>>>(h->row_len, R, 0);
    if (n > 0)
        k_load_place<<<grid_for(n, TB * LD_PER), TB, 0, s>>>(key, val, n, h->cbits, h->row_len, h->pool_col,
                                                             h->pool_val, h->ds);
    // natural order, no slack: the row starts are the SpMV's flat offsets,
    // which the next product finds ready
    h->flat_dirty = true;
    DCSR_TRY(ensure_flat(h, s, n));
    k_set_loaded<<<grid_for(R > 0 ? R : 1, TB), TB, 0, s>>>(R, (const uint32_t *)h->ws.ptr[WS_FOFF], h->row_start,
                                                            h->row_len, h->row_cap, h->ds, (uint64_t)n);
    DCSR_HIP(hipGetLastError());
    DCSR_TRY(pull_state(h, s));
    h->canonical = !(h->hs->load_flags & LD_NONCANON);
    h->hubs_dirty = true;
    h->hub_rows_h = -1;  // unknown until the hub list is rebuilt
    return DCSR_OK;
}

// Load triples whose keys are given by `pack` (a launch that fills key / val
// and raises ST_BAD_INDEX on an index outside the matrix).
template <class Pack>
static dcsr_status load_packed(dcsr_handle h, int64_t n, hipStream_t s, Pack &&pack)
{
    if (n >= (int64_t)0xfffffff0ll) return DCSR_ERR_INVALID;
    uint64_t *k0, *k1;
    uint32_t *v0, *v1, *hist, *part;
    DCSR_TRY(ws_get(h, WS_KEY_A, (size_t)n * 8, (void **)&k0));
    DCSR_TRY(ws_get(h, WS_VAL_A, (size_t)n * 4, (void **)&v0));
    k_clear_status<<<1, 1, 0, s>>>(h->ds);
    if (n > 0) pack(k0, v0);
    DCSR_HIP(hipGetLastError());
    // reject out-of-range indices before anything is modified
    DCSR_TRY(pull_state(h, s));
    if (h->hs->status & ST_BAD_INDEX) {
        k_clear_status<<<1, 1, 0, s>>>(h->ds);
        return DCSR_ERR_BAD_INDEX;
    }
    // a stable sort leaves keys that are in order as they are
    if (!(h->hs->load_flags & LD_UNSORTED)) return load_sorted(h, k0, v0, n, s);
    DCSR_TRY(ws_get(h, WS_KEY_B, (size_t)n * 8, (void **)&k1));
    DCSR_TRY(ws_get(h, WS_VAL_B, (size_t)n * 4, (void **)&v1));
    DCSR_TRY(ws_get(h, WS_HIST, radix_hist_words(n) * 4, (void **)&hist));
    DCSR_TRY(ws_get_zeroed(h, WS_SCAN, radix_part_words(n) * 4, (void **)&part, s));
    int which = 0;
    DCSR_HIP(radix_sort_pairs(k0, v0, k1, v1, n, h->rbits + h->cbits, hist, part, &which, s));
    return load_sorted(h, which ? k1 : k0, which ? v1 : v0, n, s);
}

static dcsr_status load_coo_impl(dcsr_handle h, const int32_t *rows, const int32_t *cols, const float *vals,
                                 int64_t n, hipStream_t s)
{
    return load_packed(h, n, s, [&](uint64_t *key, uint32_t *val) {
        k_pack_keys<<<grid_for(n, TB * LD_PER), TB, 0, s>>>(rows, cols, vals, n, h->rows, h->cols, h->cbits, key, val, h->ds);
    });
}

dcsr_status load_coo_internal(dcsr_handle h, const int32_t *rows, const int32_t *cols, const float *vals, int64_t n,
                              hipStream_t s)
{
    return load_coo_impl(h, rows, cols, vals, n, s);
}

dcsr_status dcsr_load_coo(dcsr_handle h, const int32_t *rows, const int32_t *cols, const float *vals, int64_t n,
                          dcsr_stream_t stream)
{
    if (!h || n < 0 || (n > 0 && (!rows || !cols || !vals))) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    return load_coo_impl(h, rows, cols, vals, n, s);
}

dcsr_status dcsr_load_csr(dcsr_handle h, const int32_t *row_offsets, const int32_t *cols, const float *vals,
                          dcsr_stream_t stream)
{
    if (!h || !row_offsets) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    int32_t nnz = 0;
    k_clear_status<<<1, 1, 0, s>>>(h->ds);
    k_check_offsets<<<grid_for(h->rows, TB), TB, 0, s>>>(row_offsets, h->rows, h->ds);
    DCSR_TRY(pull_state(h, s));
    nnz = (int32_t)h->hs->load_nnz;
    if (nnz < 0 || (h->hs->status & ST_BAD_INDEX)) return DCSR_ERR_INVALID;
    if (nnz > 0 && (!cols || !vals)) return DCSR_ERR_INVALID;
    if (nnz > 0 && h->rows == 0) return DCSR_ERR_BAD_INDEX;
    return load_packed(h, nnz, s, [&](uint64_t *key, uint32_t *val) {
        k_pack_keys_csr<<<grid_for(nnz, (TB / 64) * KEY_SPAN), TB, 0, s>>>(row_offsets, (uint32_t)h->rows, cols, vals,
                                                                           (uint32_t)nnz, h->cols, h->cbits, key, val,
                                                                           h->ds);
    });
}

// Flat exclusive offsets of the live rows (u32, R+1 entries) and their row
// map: the SpMV's own, scanned again only where they are not known to be
// current (a structural change outside the update pipeline; refresh_replayed).
static dcsr_status flat_rows(dcsr_handle h, hipStream_t s, const uint32_t **off, const uint32_t **rowmap)
{
    DCSR_TRY(ensure_flat(h, s));
    *off = (const uint32_t *)h->ws.ptr[WS_FOFF];
    *rowmap = (const uint32_t *)h->ws.ptr[WS_ROWMAP];
    return DCSR_OK;
}

// total: an upper bound of the entries (sizes the grid); see k_copy_rows.
static void launch_copy_rows(dcsr_handle h, const uint32_t *off, const uint32_t *rowmap, int64_t total, uint64_t limit,
                             int32_t *row_offsets, int32_t *dcol, float *dval, hipStream_t s, uint2 *dpair = nullptr)
{
    const int64_t R = h->rows;
    if (R <= 0 || (total <= 0 && !row_offsets)) return;
    const bool small = total <= CP_SHORT_MAX;
    const int64_t span = small ? CP_SHORT : CP_SPAN;
    const int64_t waves = (total + span - 1) / span;
    int64_t blocks = (waves + 3) / 4;
    if (row_offsets && blocks < (R + 1) / (TB * 8)) blocks = (R + 1) / (TB * 8);
    if (blocks > 2048) blocks = 2048;  // waves stride over the rest
    if (blocks < 1) blocks = 1;
    auto run = [&](auto *k) {
        k<<<(unsigned)blocks, TB, 0, s>>>(off, rowmap, (uint32_t)R, limit, row_offsets, h->row_start, h->pool_col,
                                          h->pool_val, dcol, dval, dpair);
    };
    if (dpair) small ? run(k_copy_rows<true, CP_SHORT>) : run(k_copy_rows<true, CP_SPAN>);
    else small ? run(k_copy_rows<false, CP_SHORT>) : run(k_copy_rows<false, CP_SPAN>);
}

// The live entries as (column, value) pairs in flat order; *off receives the
// flat offsets (state known; cap: the entries that dst holds).
dcsr_status copy_rows_paired(dcsr_handle h, uint2 *dst, int64_t cap, const uint32_t **off, hipStream_t s)
{
    const uint32_t *rowmap;
    DCSR_TRY(flat_rows(h, s, off, &rowmap));
    launch_copy_rows(h, *off, rowmap, h->nnz_h, (uint64_t)cap, nullptr, nullptr, nullptr, s, dst);
    DCSR_HIP(hipGetLastError());
    return DCSR_OK;
}

// Canonical export of a matrix with duplicates / zeros (state known).
static dcsr_status export_canonical(dcsr_handle h, int32_t *row_offsets, int32_t *cols, float *vals, int64_t cap,
                                    int64_t *nnz_out, hipStream_t s)
{
    const int64_t R = h->rows, nnz = h->nnz_h;
    const uint32_t *off, *rowmap;
    DCSR_TRY(flat_rows(h, s, &off, &rowmap));
    int32_t *tcol;
    float *tval;
    unsigned long long *starts, *emit;
    uint32_t *word_pre, *tile_cnt, *tile_off, *part, *tot;
    const int64_t words = (nnz + 63) / 64, tiles = (nnz + CN_TILE - 1) / CN_TILE;
    DCSR_TRY(ws_get(h, WS_UCOL, (size_t)nnz * 4 + 4, (void **)&tcol));
    DCSR_TRY(ws_get(h, WS_UVAL, (size_t)nnz * 4 + 4, (void **)&tval));
    DCSR_TRY(ws_get(h, WS_UPOS, (size_t)words * 8, (void **)&starts));
    DCSR_TRY(ws_get(h, WS_UCODE, (size_t)words * 8, (void **)&emit));
    DCSR_TRY(ws_get(h, WS_UPRE, (size_t)words * 4, (void **)&word_pre));
    DCSR_TRY(ws_get(h, WS_TINS, (size_t)(tiles + 1) * 4, (void **)&tile_cnt));
    DCSR_TRY(ws_get(h, WS_TDEL, (size_t)(tiles + 1) * 4, (void **)&tile_off));
    DCSR_TRY(ws_get_zeroed(h, WS_SCAN, scan_part_words(tiles + 1, 1) * 4, (void **)&part, s));
    DCSR_TRY(ws_get(h, WS_TMP2, 64, (void **)&tot));
    if (nnz > 0) {
        k_zero_words<<<grid_for(words * 2, TB * 4), TB, 0, s>>>((uint32_t *)starts, words * 2);
        k_canon_mark<<<grid_for(R, TB), TB, 0, s>>>(off, R, starts);
        launch_copy_rows(h, off, rowmap, nnz, ~0ull, nullptr, tcol, tval, s);
        k_canon_count<<<(unsigned)tiles, TB, 0, s>>>(starts, tcol, tval, nnz, emit, tile_cnt);
    }
    DCSR_HIP(scan_exclusive_u32(tile_cnt, tile_off, tiles, 1, part, tot, s, fault_word(h)));
    if (nnz > 0)
        k_canon_write<<<(unsigned)tiles, TB, 0, s>>>(tcol, tval, nnz, emit, tile_off, tot, (uint64_t)cap, word_pre,
                                                     cols, vals);
    if (R > 0)
        k_canon_offsets<<<grid_for(R + 1, TB), TB, 0, s>>>(off, R, emit, word_pre, tot, (uint64_t)cap, row_offsets,
                                                           (uint32_t)nnz);
    else
        k_fill_i32<<<1, 64, 0, s>>>(row_offsets, 1, 0);
    DCSR_HIP(hipGetLastError());
    uint32_t total = 0;
    DCSR_TRY(fetch_words(h, tot, 4, &total, s));
    if ((int64_t)total > cap) return DCSR_ERR_CAPACITY;
    *nnz_out = total;
    return DCSR_OK;
}

dcsr_status dcsr_export_csr(dcsr_handle h, int32_t *row_offsets, int32_t *cols, float *vals, int64_t cap,
                            int64_t *nnz_out, uint32_t flags, dcsr_stream_t stream)
{
    if (!h || !row_offsets || !nnz_out) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    const int64_t R = h->rows;
    DCSR_TRY(refresh_replayed(h, s));
    const bool canon = (flags & DCSR_EXPORT_CANONICAL) && !h->canonical;
    if (canon || !cols || !vals || cap < 0) {
        if (!h->state_known) DCSR_TRY(pull_state(h, s));
        if (!canon && cap < h->nnz_h) return DCSR_ERR_CAPACITY;
        if (h->nnz_h > 0 && (!cols || !vals)) return DCSR_ERR_INVALID;
        if (canon && cap < 0) return DCSR_ERR_CAPACITY;  // the kernels compare it unsigned
        if (canon) return export_canonical(h, row_offsets, cols, vals, cap, nnz_out, s);
    }
    if (h->state_known && cap < h->nnz_h) return DCSR_ERR_CAPACITY;
    if (R > 0) {
        const uint32_t *off, *rowmap;
        DCSR_TRY(flat_rows(h, s, &off, &rowmap));
        // a count the host does not know is read back after the copy, which
        // checks the capacity itself: one round trip instead of two
        launch_copy_rows(h, off, rowmap, live_bound(h), (uint64_t)cap, row_offsets, cols, vals, s);
    } else {
        k_fill_i32<<<1, 64, 0, s>>>(row_offsets, 1, 0);
    }
    DCSR_HIP(hipGetLastError());
    DCSR_TRY(pull_state(h, s));
    if (cap < h->nnz_h) return DCSR_ERR_CAPACITY;
    *nnz_out = h->nnz_h;
    return DCSR_OK;
}

// Rewrite every row contiguously into a pool of capacity new_cap (>= nnz).
// The destination is the handle's spare pool (allocated only when it is too
// small); the old pool becomes the spare, so steady-state compaction makes no
// allocation and no host synchronization beyond the state read-back.
// Copy the live rows, in natural order, into the spare pool (grown to
// new_cap when smaller) and swap pools.  Needs no read-back: the copy is
// sized from the host's bound of the live entries and stops at the device's
// count; the device's bump pointer becomes its live count.
// Free the retired spare buffers (the caller knows the stream is idle).
static void release_retired(dcsr_handle h)
{
    for (int i = 0; i < h->nretired; ++i) (void)hipFree(h->retired[i]);
    h->nretired = 0;
}

static dcsr_status compact_into(dcsr_handle h, int64_t new_cap, hipStream_t s)
{
    const int64_t R = h->rows;
    const int64_t nnz = live_bound(h);
    if (new_cap < nnz) new_cap = nnz;
    if (new_cap < h->cfg.min_pool) new_cap = h->cfg.min_pool;
    if (new_cap > (int64_t)0xfffffff0ll) return DCSR_ERR_POOL_EXHAUSTED;
    const uint32_t *off = nullptr, *rowmap = nullptr;
    if (R > 0) DCSR_TRY(flat_rows(h, s, &off, &rowmap));
    if (h->spare_cap < new_cap) {
        // kernels queued earlier may still read the old spare (the pool of
        // the compaction before): it is retired, not freed, so that growing
        // never waits for the stream
        if (h->nretired + 2 > (int)(sizeof(h->retired) / sizeof(h->retired[0]))) {
            DCSR_HIP(hipStreamSynchronize(s));
            release_retired(h);
        }
        if (h->spare_col) h->retired[h->nretired++] = h->spare_col;
        if (h->spare_val) h->retired[h->nretired++] = h->spare_val;
        h->spare_col = nullptr;
        h->spare_val = nullptr;
        h->spare_cap = 0;
        DCSR_HIP(hipMalloc(&h->spare_col, (size_t)new_cap * 4));
        DCSR_HIP(hipMalloc(&h->spare_val, (size_t)new_cap * 4));
        h->spare_cap = new_cap;
    }
    launch_copy_rows(h, off, rowmap, nnz, ~0ull, nullptr, h->spare_col, h->spare_val, s);
    ++h->ncompact;
    if (R > 0) k_set_compacted<<<grid_for(R, TB), TB, 0, s>>>(R, off, h->row_start, h->row_len, h->row_cap, h->ds, off + R);
    else k_set_compacted<<<1, 1, 0, s>>>(0, nullptr, h->row_start, h->row_len, h->row_cap, h->ds, nullptr);
    DCSR_HIP(hipGetLastError());
    int32_t *oc = h->pool_col;
    float *ov = h->pool_val;
    int64_t ocap = h->pool_cap;
    h->pool_col = h->spare_col;
    h->pool_val = h->spare_val;
    h->pool_cap = h->spare_cap;
    h->spare_col = oc;
    h->spare_val = ov;
    h->spare_cap = ocap;
    if (h->state_known) {
        h->bump_h = nnz;
        h->garbage_h = 0;
    } else {
        // the device's bump pointer is now its live count; a snapshot in
        // flight predates the swap
        h->bump_ub = h->nnz_ub;
        h->snap_valid_from = h->snap_seq + 1;
    }
    return DCSR_OK;
}

dcsr_status compact_in_order(dcsr_handle h, hipStream_t s) { return compact_into(h, h->pool_cap, s); }

dcsr_status grow_in_order(dcsr_handle h, int64_t new_cap, hipStream_t s)
{
    if (new_cap < h->pool_cap) new_cap = h->pool_cap;
    return compact_into(h, new_cap, s);
}

dcsr_status dcsr_compact(dcsr_handle h, dcsr_stream_t stream)
{
    if (!h) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    DCSR_TRY(refresh_replayed(h, s));
    if (!h->state_known) DCSR_TRY(pull_state(h, s));
    // keep the capacity, release retired chunks
    return compact_into(h, h->pool_cap, s);
}

// Make room for at least min_free entries past the bump pointer: compact
// (releasing retired chunks) and grow geometrically when live data plus the
// request would fill more than 2/3 of the pool.
dcsr_status pool_reserve(dcsr_handle h, int64_t min_free, hipStream_t s, const int32_t *)
{
    if (!h->state_known) DCSR_TRY(pull_state(h, s));
    if (h->pool_cap - h->bump_h >= min_free) return DCSR_OK;
    int64_t cap = h->pool_cap;
    int64_t want = h->nnz_h + min_free;
    if (want + want / 2 > cap) {
        int64_t grown = (int64_t)(want * h->cfg.pool_factor);
        if (grown < 2 * cap) grown = 2 * cap;
        cap = grown;
    }
    return compact_into(h, cap, s);
}

// Rewrite a non-canonical matrix (duplicates / explicit zeros from the load)
// into canonical rows, as the first host-path add does for every row
// (cusp/system/detail/sequential/elementwise.h:44-131 visits all rows of A).
dcsr_status canonicalize(dcsr_handle h, hipStream_t s)
{
    if (h->canonical) return DCSR_OK;
    const int64_t R = h->rows;
    int64_t nnz = h->nnz_h;
    int32_t *off, *ocol;
    float *oval;
    DCSR_HIP(hipMalloc(&off, (size_t)(R + 1) * 4));
    DCSR_HIP(hipMalloc(&ocol, (size_t)(nnz > 0 ? nnz : 1) * 4));
    DCSR_HIP(hipMalloc(&oval, (size_t)(nnz > 0 ? nnz : 1) * 4));
    int64_t cn = 0;
    dcsr_status st = dcsr_export_csr(h, off, ocol, oval, nnz, &cn, DCSR_EXPORT_CANONICAL, s);
    if (st == DCSR_OK) st = dcsr_load_csr(h, off, ocol, oval, s);
    (void)hipFree(off);
    (void)hipFree(ocol);
    (void)hipFree(oval);
    if (st == DCSR_OK) h->canonical = true;
    return st;
}

dcsr_status dcsr_rebin(dcsr_handle h, dcsr_stream_t stream)
{
    if (!h) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    h->flat_dirty = true;
    DCSR_TRY(ensure_flat(h, s));
    k_zero_hubs<<<1, 1, 0, s>>>(h->ds);
    if (h->rows > 0) k_count_hubs<<<grid_for(h->rows, TB), TB, 0, s>>>(h->rows, h->row_len, h->ds);
    DCSR_HIP(hipGetLastError());
    DCSR_TRY(pull_state(h, s));
    h->hub_rows_h = h->hs->hub_count;
    h->hubs_dirty = false;
    return DCSR_OK;
}

dcsr_status dcsr_query(dcsr_handle h, dcsr_info *info)
{
    if (!h || !info) return DCSR_ERR_INVALID;
    DCSR_TRY(pull_state(h, h->last_stream));
    memset(info, 0, sizeof(*info));
    info->rows = h->rows;
    info->cols = h->cols;
    info->nnz = h->nnz_h;
    info->pool_cap = h->pool_cap;
    info->pool_used = h->bump_h;
    info->garbage = h->garbage_h;
    info->hub_rows = h->hubs_dirty ? -1 : h->hub_rows_h;
    info->last_inserted = h->last_ins;
    info->last_added = h->last_add;
    info->last_deleted = h->last_del;
    info->last_touched_rows = h->last_touched;
    info->canonical = h->canonical ? 1 : 0;
    info->max_segments = 1;
    info->scan_fallback = (h->hs->status & ST_SCAN_FALLBACK) ? 1 : 0;
    info->spmv_paneled = h->pnl_valid ? 1 : 0;
    info->compactions = h->ncompact;
    return DCSR_OK;
}

dcsr_status dcsr_export_layout(dcsr_handle h, uint32_t *row_start, int32_t *row_len, int32_t *row_cap,
                               dcsr_stream_t stream)
{
    if (!h || (h->rows > 0 && (!row_start || !row_len || !row_cap))) return DCSR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    h->last_stream = s;
    const size_t R = (size_t)h->rows;
    if (R > 0) {
        DCSR_HIP(hipMemcpyAsync(row_start, h->row_start, R * 4, hipMemcpyDeviceToDevice, s));
        DCSR_HIP(hipMemcpyAsync(row_len, h->row_len, R * 4, hipMemcpyDeviceToDevice, s));
        DCSR_HIP(hipMemcpyAsync(row_cap, h->row_cap, R * 4, hipMemcpyDeviceToDevice, s));
    }
    return pull_state(h, s);
}
