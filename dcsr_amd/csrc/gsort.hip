// gsort.hip -- row-group sort of an update batch's (key, value) pairs.
//
// Keys are (row << cbits) | col; invalid ones are ~0.  The rows are split
// into G groups of 2^gshift consecutive rows, and a key's digit is its group
// (key >> lb with lb = gshift + cbits; ~0 goes to digit G, after every
// group).  The caller's pack pass counts the digits per 2048-pair tile into
// a blocked table; then
//
//   1. k_gs_scan: each digit's tile counts become exclusive offsets (one
//      workgroup per 64 digits, one lane per digit, every load in flight
//      before the first add);
//   2. k_gs_scatter: one stable scatter places each group's pairs
//      contiguously, in arrival order (digits ranked by wave ballots, staged
//      in LDS so runs are written together);
//   3. k_gs_sort: one workgroup per group sorts the group's pairs by their
//      low lb key bits (all of its keys share the bits above): groups of up to
//      GS_CAP pairs in LDS by buckets, larger ones out of global memory by
//      stable LSD passes.
//
// The result is exactly the stable sort of the batch by key, which the LSD
// radix sort (prims.hip) gives in one count/scan/scatter round per 8 key
// bits: here the pairs cross HBM in one scatter and one group pass.  Stable
// ranks keep equal keys in arrival order, which the insert-or-add sums rely
// on.
#include "prims.h"
#include "wave.h"

namespace {

constexpr int GT = 512;              // threads of the scatter
constexpr int GIPT = 4;              // pairs per lane in a scatter tile
constexpr int GTILE = GT * GIPT;     // 2048 == RADIX_TILE
static_assert(GTILE == RADIX_TILE, "pack counts tiles of the scatter's size");
constexpr int GS_SCAN_T = 1024;      // k_gs_scan: 16 waves per 64 digits
constexpr int GS_SCAN_Q = 32;        // tiles per wave per round

// Lanes holding the same digit of `bits` bits (every lane active).
__device__ __forceinline__ uint64_t wave_match_bits(uint32_t d, int bits)
{
    uint64_t peers = ~0ull;
    for (int b = 0; b < bits; ++b) {
        const uint64_t m = __ballot((d >> b) & 1u);
        peers &= ((d >> b) & 1u) ? m : ~m;
    }
    return peers;
}

__device__ __forceinline__ uint32_t group_digit(uint64_t k, int lb, int ndig)
{
    return k == ~0ull ? (uint32_t)(ndig - 1) : (uint32_t)(k >> lb);
}

// Exclusive offsets of each digit's tile counts, in place; dtot[d] receives
// the digit's total.  Block b covers digits [64b, 64b + 64): lane = digit.
// A round covers NW * GS_SCAN_Q consecutive tiles, GS_SCAN_Q per wave in
// wave order; the wave's counts stay in registers between the sum and the
// write of the prefixes.
__global__ __launch_bounds__(GS_SCAN_T) void k_gs_scan(uint32_t *__restrict__ hist, int64_t nb,
                                                       uint32_t *__restrict__ dtot)
{
    constexpr int NW = GS_SCAN_T / 64;
    __shared__ uint32_t wsum[NW][64];
    const int w = threadIdx.x >> 6, lane = lane_id();
    uint32_t *col = hist + (int64_t)blockIdx.x * nb * 64 + lane;
    uint32_t carry_in = 0;  // the digit's count in earlier rounds
    for (int64_t r0 = 0; r0 < nb; r0 += (int64_t)NW * GS_SCAN_Q) {
        const int64_t t0 = r0 + (int64_t)w * GS_SCAN_Q;
        const int64_t t1 = t0 + GS_SCAN_Q < nb ? t0 + GS_SCAN_Q : nb;
        uint32_t v[GS_SCAN_Q];
        uint32_t s = 0;
#pragma unroll
        for (int q = 0; q < GS_SCAN_Q; ++q) {
            const int64_t t = t0 + q;
            v[q] = t < t1 ? col[t * 64] : 0u;
        }
#pragma unroll
        for (int q = 0; q < GS_SCAN_Q; ++q) s += v[q];
        wsum[w][lane] = s;
        __syncthreads();
        uint32_t before = 0, tot = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const uint32_t x = wsum[i][lane];
            before += i < w ? x : 0u;
            tot += x;
        }
        __syncthreads();
        uint32_t p = carry_in + before;
#pragma unroll
        for (int q = 0; q < GS_SCAN_Q; ++q) {
            const int64_t t = t0 + q;
            if (t < t1) col[t * 64] = p;
            p += v[q];
        }
        carry_in += tot;
    }
    if (w == 0) dtot[(int64_t)blockIdx.x * 64 + lane] = carry_in;
}

// Stable scatter of one 2048-pair tile into the group order.  gbase_out
// (block 0) receives the exclusive offsets of the ndig digits plus the total.
// A tile's ranking is a serial chain per wave, so eight waves take four pairs per
// lane (four took eight: 22.7 us for 1M triples, 8.6 for 100K; now 19.7 and 6.4).
__global__ __launch_bounds__(GT) void k_gs_scatter(const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                   uint64_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                   int64_t n, int lb, int ndig, int dbits,
                                                   const uint32_t *__restrict__ hist, int64_t nb,
                                                   const uint32_t *__restrict__ dtot, uint32_t *__restrict__ gbase_out)
{
    __shared__ uint16_t wcnt[GT / 64][GS_MAX_DIGITS];  // at most a tile
    __shared__ uint32_t lofs[GS_MAX_DIGITS];
    __shared__ uint32_t gofs[GS_MAX_DIGITS];
    __shared__ uint64_t skey[GTILE];
    __shared__ uint32_t sval[GTILE];
    __shared__ uint32_t lds2[GT / 64][2];
    constexpr int DPT = GS_MAX_DIGITS / GT;  // digits per thread in the offset phase
    const int w = threadIdx.x >> 6, lane = lane_id();
    const int64_t tile = blockIdx.x;
    const int64_t base = tile * GTILE;
    const int64_t wbase = base + (int64_t)w * (GIPT * 64);
    // every load first: the tile's offsets and the digit totals of this
    // thread's digits (dpt contiguous digits per thread, spread over every
    // thread), then the pairs
    uint32_t ho[DPT], dt[DPT];
    const int dpt = (ndig + GT - 1) / GT;
    const int d0 = (int)threadIdx.x * dpt;
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
        const int d = d0 + q;
        const bool in = q < dpt && d < ndig;
        ho[q] = in ? hist[gs_hist_index(d, tile, nb)] : 0u;
        dt[q] = in ? dtot[d] : 0u;
    }
    uint64_t key[GIPT];
    uint32_t val[GIPT];
#pragma unroll
    for (int j = 0; j < GIPT; ++j) {
        const int64_t idx = wbase + j * 64 + lane;
        key[j] = kin[idx < n ? idx : base];
        val[j] = vin[idx < n ? idx : base];
    }
    for (int d = threadIdx.x; d < ndig; d += GT)
#pragma unroll
        for (int i = 0; i < GT / 64; ++i) wcnt[i][d] = 0;
    __syncthreads();
    // rank: items past n take the last digit and rank after every real one
    const uint64_t lt = lanemask_lt();
    uint32_t rnk[GIPT], dg[GIPT];
#pragma unroll
    for (int j = 0; j < GIPT; ++j) {
        const bool real = wbase + j * 64 + lane < n;
        const uint32_t d = real ? group_digit(key[j], lb, ndig) : (uint32_t)(ndig - 1);
        const uint64_t peers = wave_match_bits(d, dbits);
        const int leader = __ffsll((long long)peers) - 1;
        // every lane of the digit reads its count before the leader adds to
        // it (a wave's LDS accesses complete in order): no broadcast needed
        const uint32_t b = wcnt[w][d];
        if (lane == leader) wcnt[w][d] = (uint16_t)(b + (uint32_t)__popcll(peers));
        rnk[j] = b + (uint32_t)__popcll(peers & lt);
        dg[j] = d;
    }
    __syncthreads();
    {
        uint32_t cs[DPT], gs[DPT];
        uint32_t csum = 0, gsum = 0;
#pragma unroll
        for (int q = 0; q < DPT; ++q) {
            const int d = d0 + q;
            uint32_t c = 0;
            if (q < dpt && d < ndig) {
#pragma unroll
                for (int i = 0; i < GT / 64; ++i) {
                    const uint32_t x = wcnt[i][d];
                    wcnt[i][d] = (uint16_t)c;
                    c += x;
                }
            }
            cs[q] = csum;
            csum += c;
            gs[q] = gsum;
            gsum += dt[q];
        }
        uint32_t pre[2] = {csum, gsum}, tot[2];
        block_excl_scan_n<GT / 64>(pre, lds2, tot);
        const uint32_t lp = pre[0], gp = pre[1];
#pragma unroll
        for (int q = 0; q < DPT; ++q) {
            const int d = d0 + q;
            if (q < dpt && d < ndig) {
                lofs[d] = lp + cs[q];
                gofs[d] = gp + gs[q] + ho[q];
                if (tile == 0) gbase_out[d] = gp + gs[q];
            }
        }
        if (tile == 0 && threadIdx.x == 0) gbase_out[ndig] = tot[1];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < GIPT; ++j) {
        const uint32_t p = lofs[dg[j]] + wcnt[w][dg[j]] + rnk[j];
        skey[p] = key[j];
        sval[p] = val[j];
    }
    __syncthreads();
    const int64_t valid = (n - base) < GTILE ? (n - base) : GTILE;
#pragma unroll
    for (int j = 0; j < GIPT; ++j) {
        const int p = j * GT + (int)threadIdx.x;
        if (p < valid) {
            const uint64_t k = skey[p];
            const uint32_t d = group_digit(k, lb, ndig);
            const int64_t o = (int64_t)gofs[d] + (p - (int64_t)lofs[d]);
            kout[o] = k;
            vout[o] = sval[p];
        }
    }
}

// ---------------------------------------------------------------------------
// Per-group sort.  Ranking of one chunk of up to 4 * 64 * J items in their
// current order (wave w holds positions [w * 64J, (w + 1) * 64J), item j of
// a lane at w * 64J + 64 j + lane): rnk[j] = stable rank of item j among the
// chunk's items of its digit in earlier waves excluded; afterwards
// wcnt[w][d] = items of digit d in waves before w, loff[d] = items of the
// chunk with a smaller digit, cnt_out[d] (if not null) = items of digit d.
// ---------------------------------------------------------------------------
constexpr int ST = 512;          // threads of a group's workgroup
constexpr int SNW = ST / 64;
constexpr int SJ = GS_CAP / ST;  // items per lane in a full LDS group
constexpr int SD_BITS = 9;       // digits of the stable passes: one per thread
constexpr int SD = 1 << SD_BITS;
static_assert(SD == ST && GS_CAP % ST == 0, "a digit per thread");

template <int J>
__device__ __forceinline__ void rank_chunk(const uint32_t (&dg)[J], const bool (&real)[J], int jmax,
                                           uint32_t (&rnk)[J], uint16_t (*wcnt)[SD], uint32_t *loff,
                                           uint32_t (*lds)[1])
{
    const int w = threadIdx.x >> 6, lane = lane_id();
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int i = 0; i < SD / 64; ++i) wcnt[w][lane + 64 * i] = 0;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < J; ++j) {
        rnk[j] = 0;
        if (j >= jmax) continue;  // uniform over the workgroup
        const uint64_t act = __ballot(real[j]);
        if (!real[j]) continue;
        uint64_t peers = act;
#pragma unroll
        for (int b = 0; b < SD_BITS; ++b) {
            const uint64_t m = __ballot((dg[j] >> b) & 1u);
            peers &= ((dg[j] >> b) & 1u) ? m : ~m;
        }
        const int leader = __ffsll((long long)peers) - 1;
        // every lane of the digit reads its count before the leader adds to
        // it (a wave's LDS accesses complete in order): no broadcast needed
        const uint32_t c = wcnt[w][dg[j]];
        if (lane == leader) wcnt[w][dg[j]] = (uint16_t)(c + (uint32_t)__popcll(peers));
        rnk[j] = c + (uint32_t)__popcll(peers & lt);
    }
    __syncthreads();
    uint32_t s[1] = {0}, tot[1];
#pragma unroll
    for (int i = 0; i < SNW; ++i) {
        const uint32_t x = wcnt[i][threadIdx.x];
        wcnt[i][threadIdx.x] = (uint16_t)s[0];
        s[0] += x;
    }
    block_excl_scan_n<SNW>(s, lds, tot);
    loff[threadIdx.x] = s[0];
    __syncthreads();
}

// LDS sort of n <= GS_CAP pairs of a group.  A pair is one word, its local key
// above its position in the group (GS_POS bits: ties keep their arrival order).
//
// A key's bucket is its top GS_NBB local bits.  Buckets are counted by LDS
// atomics, their starts scanned, the words placed in bucket order, and a pair is
// ranked among its own bucket's words.  Keys and values stay in registers and go
// straight to their places.  The ranking's LDS reads are the cost (they conflict:
// a microsecond for every two words in the fullest bucket with the chip's groups
// in flight), so where a bucket holds more than GS_FEW pairs every bucket is
// split first; a group that still has more than GS_CROWD pairs in a part (a
// coordinate repeated, columns that crowd) takes stable digit passes.
// For 10,000, 100,000 and 1M triples spread over 1M rows the groups take 5.2, 6
// and 19 us; in digit passes alone (nine ballots per pair and pass, three to five
// passes) 12, 13 and 30.  1M power-law triples on 325K rows: 23 and 26.
constexpr int GS_POS = 12;  // position bits (GS_CAP <= 4096)
static_assert(GS_CAP <= (1 << GS_POS), "a position fits its field");
constexpr int GS_NBB = 11;
constexpr int GS_NB = 1 << GS_NBB;
constexpr uint32_t GS_FEW = 6;     // pairs in a bucket before the buckets are split
constexpr uint32_t GS_CROWD = 64;  // pairs in a part before the digit passes
constexpr uint32_t GS_PARTS = 2 * GS_CAP + GS_NB;
static_assert(GS_PARTS / 2 + 1 <= 2 * GS_CAP && GS_PARTS % (2 * ST) == 0, "16-bit part counters fit the words");

struct GsLds {
    uint64_t word[GS_CAP];
    union {
        uint32_t start[GS_NB + 1];
        struct {
            uint16_t wcnt[SNW][SD];
            uint32_t loff[SD];
        } r;
    };
    uint32_t lds[SNW][1];
};

// A crowded group of n pairs (lb + GS_POS <= 64): digit passes over its words.
__device__ void group_sort_crowded(GsLds &S, const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                   uint64_t *__restrict__ kout, uint32_t *__restrict__ vout, uint32_t n, int lb)
{
    const uint64_t lmask = (1ull << lb) - 1ull;
    const int cnt = (int)n;
    for (uint32_t i = threadIdx.x; i < n; i += ST) S.word[i] = ((kin[i] & lmask) << GS_POS) | (uint64_t)i;
    __syncthreads();
    const int w = threadIdx.x >> 6, lane = lane_id();
    const int jmax = (cnt + ST - 1) / ST, pw = jmax * 64;  // positions per wave
    for (int sh = GS_POS; sh < lb + GS_POS; sh += SD_BITS) {
        uint32_t dg[SJ], rnk[SJ];
        uint64_t wd[SJ];
        bool real[SJ];
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            const int p = w * pw + j * 64 + lane;
            real[j] = j < jmax && p < cnt;
            wd[j] = real[j] ? S.word[p] : 0ull;
            dg[j] = (uint32_t)(wd[j] >> sh) & (SD - 1u);
        }
        rank_chunk<SJ>(dg, real, jmax, rnk, S.r.wcnt, S.r.loff, S.lds);  // its barriers: every word is read
#pragma unroll
        for (int j = 0; j < SJ; ++j)
            if (real[j]) S.word[S.r.loff[dg[j]] + S.r.wcnt[w][dg[j]] + rnk[j]] = wd[j];
        __syncthreads();
    }
    for (uint32_t i = threadIdx.x; i < n; i += ST) {
        const uint32_t src = (uint32_t)S.word[i] & ((1u << GS_POS) - 1u);
        kout[i] = kin[src];
        vout[i] = vin[src];
    }
}

// Returns (every thread) false, with nothing written, for a crowded group.
__device__ bool group_sort_lds(GsLds &S, const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                               uint64_t *__restrict__ kout, uint32_t *__restrict__ vout, uint32_t n, int lb)
{
    const uint64_t lmask = (1ull << lb) - 1ull;
    const int bs = lb > GS_NBB ? lb - GS_NBB : 0;  // key bits below the bucket's
    const uint64_t rest = (1ull << bs) - 1ull;
    // every load in flight before the first use (indices clamped into the group)
    uint64_t k[SJ];
    uint32_t v[SJ];
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
        const uint32_t i = j * ST + threadIdx.x;
        if (j * ST >= n) break;
        k[j] = kin[i < n ? i : n - 1];
        v[j] = vin[i < n ? i : n - 1];
    }
    for (int i = threadIdx.x; i < GS_NB; i += ST) S.start[i] = 0u;
    __syncthreads();
    uint32_t at[SJ];  // arrival in the bucket
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
        const uint32_t i = j * ST + threadIdx.x;
        if (j * ST >= n) break;
        at[j] = i < n ? atomicAdd(&S.start[(uint32_t)((k[j] & lmask) >> bs)], 1u) : 0u;
    }
    __syncthreads();
    {
        constexpr int BPT = GS_NB / ST;
        uint32_t c[BPT], sum[1] = {0}, tot[1];
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            c[q] = S.start[threadIdx.x * BPT + q];
            sum[0] += c[q];
        }
        block_excl_scan_n<SNW>(sum, S.lds, tot);
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            S.start[threadIdx.x * BPT + q] = sum[0];
            sum[0] += c[q];
        }
        if (threadIdx.x == 0) S.start[GS_NB] = n;
    }
    __syncthreads();
    uint32_t lc[SJ], most = 0;  // bucket start, pairs in it << 16
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
        const uint32_t i = j * ST + threadIdx.x;
        if (j * ST >= n) break;
        const uint32_t b = (uint32_t)((k[j] & lmask) >> bs);
        const uint32_t l = S.start[b], c = i < n ? S.start[b + 1] - l : 0u;
        lc[j] = l | (c << 16);
        most = c > most ? c : most;
    }
    if (__syncthreads_or(most > GS_FEW)) {
        // a long row: every bucket is split into at least as many equal parts as it
        // has pairs, and the parts are counted (16 bits each, in the words'
        // place) and scanned like the buckets before
        uint32_t *parts = reinterpret_cast<uint32_t *>(S.word);
        constexpr int BPT = GS_NB / ST, PPT = GS_PARTS / 2 / ST;
        uint32_t lg[BPT], sum[1] = {0}, tot[1];
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            const uint32_t c = S.start[threadIdx.x * BPT + q + 1] - S.start[threadIdx.x * BPT + q];
            lg[q] = c > 1 ? 32u - (uint32_t)__clz(c - 1u) : 0u;
            lg[q] = lg[q] < (uint32_t)bs ? lg[q] : (uint32_t)bs;
            sum[0] += 1u << lg[q];
        }
        for (uint32_t i = threadIdx.x; i < GS_PARTS / 2; i += ST) parts[i] = 0u;
        block_excl_scan_n<SNW>(sum, S.lds, tot);
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            S.start[threadIdx.x * BPT + q] = sum[0] | (lg[q] << 16);
            sum[0] += 1u << lg[q];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            const uint32_t i = j * ST + threadIdx.x;
            if (j * ST >= n) break;
            const uint32_t e = S.start[(uint32_t)((k[j] & lmask) >> bs)];
            lc[j] = (e & 0xffffu) + (uint32_t)((k[j] & rest) >> (bs - (int)(e >> 16)));
            const uint32_t sh = (lc[j] & 1u) * 16u;
            at[j] = i < n ? (atomicAdd(&parts[lc[j] >> 1], 1u << sh) >> sh) & 0xffffu : 0u;
        }
        __syncthreads();
        uint32_t pc[PPT];
        sum[0] = 0;
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
            pc[q] = parts[threadIdx.x * PPT + q];
            sum[0] += (pc[q] & 0xffffu) + (pc[q] >> 16);
        }
        block_excl_scan_n<SNW>(sum, S.lds, tot);
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
            const uint32_t a = sum[0] + (pc[q] & 0xffffu);
            parts[threadIdx.x * PPT + q] = sum[0] | (a << 16);
            sum[0] = a + (pc[q] >> 16);
        }
        if (threadIdx.x == 0) parts[GS_PARTS / 2] = n;
        __syncthreads();
        const uint16_t *ps = reinterpret_cast<const uint16_t *>(S.word);
        most = 0;
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            const uint32_t i = j * ST + threadIdx.x;
            if (j * ST >= n) break;
            const uint32_t l = ps[lc[j]], c = i < n ? ps[lc[j] + 1] - l : 0u;
            lc[j] = l | (c << 16);
            most = c > most ? c : most;
        }
        if (__syncthreads_or(most > GS_CROWD)) return false;
    }
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
        const uint32_t i = j * ST + threadIdx.x;
        if (j * ST >= n) break;
        if (i < n) S.word[(lc[j] & 0xffffu) + at[j]] = ((k[j] & rest) << GS_POS) | (uint64_t)i;
        at[j] = lc[j] & 0xffffu;  // from here on the pair's place
    }
    __syncthreads();
    for (uint32_t d = 0; __any(d < most); ++d) {
        // all reads in flight before the first use
        uint64_t o[SJ];
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            if (j * ST >= n) break;
            o[j] = ~0ull;
            if (d < (lc[j] >> 16)) o[j] = S.word[(lc[j] & 0xffffu) + d];
        }
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            const uint64_t mine = ((k[j] & rest) << GS_POS) | (uint64_t)(j * ST + threadIdx.x);
            if (j * ST >= n) break;
            at[j] += o[j] < mine ? 1u : 0u;
        }
    }
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
        const uint32_t i = j * ST + threadIdx.x;
        if (j * ST >= n) break;
        if (i < n) {
            kout[at[j]] = k[j];
            vout[at[j]] = v[j];
        }
    }
    return true;
}

// A group larger than GS_CAP: stable LSD passes out of global memory by this
// workgroup alone, chunk after chunk (each chunk ranked as above, each
// digit's running offset carried in LDS).  Ping-pongs between the group's
// ranges of (a_k, a_v) (input) and (b_k, b_v) and ends in (b_k, b_v).
struct GsBig {
    uint16_t wcnt[SNW][SD];
    uint32_t loff[SD];
    uint32_t run[SD];
    uint32_t lds[SNW][1];
};

__device__ void group_sort_big(GsBig &S, uint64_t *__restrict__ a_k, uint32_t *__restrict__ a_v,
                               uint64_t *__restrict__ b_k, uint32_t *__restrict__ b_v, int64_t s0, int64_t cnt,
                               int lb)
{
    constexpr int BJ = 2;                 // items per lane per chunk
    constexpr int CH = ST * BJ;           // pairs per chunk
    const int w = threadIdx.x >> 6, lane = lane_id();
    uint64_t *sk = a_k, *dk = b_k;
    uint32_t *sv = a_v, *dv = b_v;
    bool in_b = false;
    for (int sh = 0; sh < lb; sh += SD_BITS) {
        // digit counts of the whole group
        S.run[threadIdx.x] = 0;
        __syncthreads();
        for (int64_t i = threadIdx.x; i < cnt; i += ST) atomicAdd(&S.run[(uint32_t)(sk[s0 + i] >> sh) & (SD - 1u)], 1u);
        __syncthreads();
        {
            uint32_t c[1] = {S.run[threadIdx.x]}, tot[1];
            block_excl_scan_n<SNW>(c, S.lds, tot);
            S.run[threadIdx.x] = c[0];
        }
        __syncthreads();
        for (int64_t c0 = 0; c0 < cnt; c0 += CH) {
            const int64_t left = cnt - c0;
            const int jmax = left >= CH ? BJ : (int)((left + ST - 1) / ST);
            const int pw = jmax * 64;
            // only digits and ranks stay in registers; the pairs are read
            // again for the scatter (L2 hits)
            uint32_t dg[BJ], rnk[BJ];
            bool real[BJ];
#pragma unroll
            for (int j = 0; j < BJ; ++j) {
                const int64_t p = (int64_t)w * pw + j * 64 + lane;
                real[j] = j < jmax && p < left;
                dg[j] = real[j] ? (uint32_t)(sk[s0 + c0 + p] >> sh) & (SD - 1u) : 0u;
            }
            rank_chunk<BJ>(dg, real, jmax, rnk, S.wcnt, S.loff, S.lds);
#pragma unroll
            for (int j = 0; j < BJ; ++j) {
                if (!real[j]) continue;
                const int64_t p = (int64_t)w * pw + j * 64 + lane;
                const int64_t o = (int64_t)S.run[dg[j]] + S.wcnt[w][dg[j]] + rnk[j];
                dk[s0 + o] = sk[s0 + c0 + p];
                dv[s0 + o] = sv[s0 + c0 + p];
            }
            __syncthreads();
            // the chunk's count of digit d: loff[d + 1] - loff[d]
            {
                const int d = threadIdx.x;
                const uint32_t c = (d == SD - 1 ? (uint32_t)(left < CH ? left : CH) : S.loff[d + 1]) - S.loff[d];
                S.run[d] += c;
            }
            __syncthreads();
        }
        uint64_t *tk = sk; sk = dk; dk = tk;
        uint32_t *tv = sv; sv = dv; dv = tv;
        in_b = !in_b;
    }
    if (!in_b) {
        for (int64_t i = threadIdx.x; i < cnt; i += ST) {
            b_k[s0 + i] = a_k[s0 + i];
            b_v[s0 + i] = a_v[s0 + i];
        }
    }
}

// One workgroup per digit (group); the last digit holds the invalid keys,
// copied as they are.  In: (kin, vin) in group order; out: (kout, vout)
// sorted.  gbase: ndig + 1 exclusive group offsets.
__global__ __launch_bounds__(ST) __attribute__((amdgpu_waves_per_eu(6))) void k_gs_sort(uint64_t *__restrict__ kin, uint32_t *__restrict__ vin,
                                                uint64_t *__restrict__ kout, uint32_t *__restrict__ vout, int lb,
                                                int ndig, const uint32_t *__restrict__ gbase)
{
    __shared__ union {
        GsLds lds;
        GsBig big;
    } S;
    const int g = blockIdx.x;
    const int64_t s0 = gbase[g];
    const int64_t cnt = (int64_t)gbase[g + 1] - s0;
    if (cnt <= 0) return;
    if (g == ndig - 1) {
        for (int64_t i = threadIdx.x; i < cnt; i += ST) {
            kout[s0 + i] = kin[s0 + i];
            vout[s0 + i] = vin[s0 + i];
        }
        return;
    }
    if (cnt <= GS_CAP) {
        if (group_sort_lds(S.lds, kin + s0, vin + s0, kout + s0, vout + s0, (uint32_t)cnt, lb)) return;
        __syncthreads();
        if (lb + GS_POS <= 64) {
            group_sort_crowded(S.lds, kin + s0, vin + s0, kout + s0, vout + s0, (uint32_t)cnt, lb);
            return;
        }
    }
    group_sort_big(S.big, kin, vin, kout, vout, s0, cnt, lb);
}

}  // namespace

size_t gs_hist_words(int64_t n, int ndig)
{
    const int64_t nb = (n + GTILE - 1) / GTILE;
    const int64_t blocks = (ndig + 63) / 64;
    return (size_t)((nb < 1 ? 1 : nb) * 64 * blocks) + 2 * (GS_MAX_DIGITS + 64);
}

hipError_t group_sort_pairs(uint64_t *k0, uint32_t *v0, uint64_t *k1, uint32_t *v1, int64_t n, int lb, int ndig,
                            uint32_t *hist, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (ndig < 1 || ndig > GS_MAX_DIGITS || lb < 1 || lb > 62) return hipErrorInvalidValue;
    const int64_t nb = (n + GTILE - 1) / GTILE;
    const int blocks = (ndig + 63) / 64;
    uint32_t *dtot = hist + nb * 64 * blocks;
    uint32_t *gbase = dtot + GS_MAX_DIGITS + 64;
    int dbits = 1;
    while ((1 << dbits) < ndig) ++dbits;
    k_gs_scan<<<blocks, GS_SCAN_T, 0, s>>>(hist, nb, dtot);
    k_gs_scatter<<<(unsigned)nb, GT, 0, s>>>(k0, v0, k1, v1, n, lb, ndig, dbits, hist, nb, dtot, gbase);
    k_gs_sort<<<ndig, ST, 0, s>>>(k1, v1, k0, v0, lb, ndig, gbase);
    return hipGetLastError();
}
