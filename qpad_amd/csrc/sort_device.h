// sort_device.h -- device side of the per-slice re-sort of a plasma species
// by radial cell (the order QPAD's update_bound leaves,
// part2d_class.f03:2307-2353, is not kept: particles are regrouped by cell so
// that one wave deposits one cell), shared by the sort (k_sort.hip) and the
// push that counts the cells of few particles (k_plasma.hip).
//
// Stable counting sort over the nr + 1 cell keys (key nr = left the box),
// chunk of T * PER particles per workgroup of T threads:
//   counting pass    histogram of the chunk's keys in LDS -> hist[chunk][bin];
//   k_sort_scan      per bin, exclusive prefix of the chunk counts (in place)
//                    and the bin totals (many chunks only);
//   scattering pass  bin starts from the totals; rank of each particle among
//                    the chunk's particles with the same key, in particle
//                    order; position = bin start + chunk offset + rank.  One
//                    workgroup more than there are chunks writes cell_start,
//                    numbers the overflow rows of crowded cells and lists
//                    their chunks for the deposits.
// Integer counting only, in a fixed order: the permutation is the same on
// every run.
//
// Both passes are chains of latencies, so they want many workgroups and few
// launches: small chunks up to kMidMax particles, and up to kDirectChunks of
// them without the scan launch (every scattering workgroup sums the histogram
// rows itself) and counted by the push.  A chunk's keys lie within a few
// cells of each other, so the ranks come from per-wave counters over a window
// of the keys (three barriers); a chunk whose keys spread wider takes its
// waves in turn.
#pragma once

#include <hip/hip_runtime.h>

#include "qpad_internal.h"

namespace qpad {

// the forms, by the number of particles (sort_form):
//   direct  chunks of kSmallChunk, no scan launch, counted by the push;
//   mid     chunks of kMidChunk;
//   large   chunks of kSortChunk (fewer histogram rows).
enum { SORT_LARGE = 0, SORT_MID = 1, SORT_DIRECT = 2, SORT_FORMS = 3 };
constexpr int kSortChunk = 2048;
constexpr int kMidChunk = 1024;
constexpr int kSmallChunk = 512;
// threads of every form's workgroups: with 1024 for the large one, two fit a
// CU and the closing workgroup waits for a second round (scatter, 2^20
// particles in 8192 cells 41.5 us, with 512 33.6; 524288 in 4096 20.6, 17.5)
constexpr int kSortThreads = 512;
static_assert(kSortThreads == kSmallChunk, "the direct form: a thread per particle");
constexpr int64_t kMidMax = 262144;          // most particles of the mid form
constexpr int64_t kMidWork = 1 << 20;        // most (chunks x cells) of its histogram
constexpr int kDirectChunks = 120;           // most chunks of the direct form
constexpr int64_t kDirectWork = 1 << 17;     // most (chunks x bins) it sums in every workgroup
constexpr int kDirectBins = 4097;            // bins the direct form keeps in LDS
static_assert(kDirectChunks * kSmallChunk < 65536, "the direct form counts in 16 bits");

// The cell of a stored position.  The fma is written out, so that every
// kernel that asks computes the same cell for the same particle.
__device__ __forceinline__ uint32_t cell_key(double x1, double x2, double idr, double edge, int nr)
{
    double r = sqrt(fma(x1, x1, x2 * x2));
    if (!(r < edge)) return (uint32_t)nr;   // leaves the box (update_bound)
    int c = (int)__dmul_rn(r, idr);
    return (uint32_t)(c < nr ? c : nr - 1);
}

struct SortArgs {
    int64_t n;
    int nb;                 // bins: keys 0 .. nb-1
    int nchunks;
    int form;               // SORT_*
    const uint32_t *key;
    uint32_t *key_w;        // counting pass of the push: keys out
    int *hist;              // [nchunks][nb]; direct: 16-bit rows of hist16_row(nb)
    int *tot;               // [nb]
    int32_t *cs;            // [nb + 1]
    const double *s[8];
    double *d[8];
    const int32_t *sid;
    int32_t *did;
    int32_t *os;            // [nb] overflow rows of cell c: os[c] .. os[c+1]-1; [nb] crowded chunks
    int4 *desc;             // [n_crowd_max] (cell, first particle, end, overflow row or -1)
    int n_ov_max, n_crowd_max, first;
};

// row length of the direct form's 16-bit histogram rows (16-byte loads)
__host__ __device__ inline int hist16_row(int nb) { return (nb + 7) & ~7; }

// particle of this thread in round j of the chunk (a wave owns 64 PER
// consecutive particles)
template <int T, int PER>
__device__ __forceinline__ int64_t sort_element(int j)
{
    return (int64_t)blockIdx.x * (T * PER) + (threadIdx.x >> 6) * (64 * PER) + j * 64 + (threadIdx.x & 63);
}

// histogram row of the chunk from its keys (cnt: nb ints of LDS)
template <int T, int PER>
__device__ __forceinline__ void chunk_hist(const SortArgs &a, const uint32_t (&kv)[PER], int *cnt)
{
    const bool direct = a.form == SORT_DIRECT;
    for (int b = threadIdx.x; b < a.nb; b += T) cnt[b] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; j++)
        if (sort_element<T, PER>(j) < a.n) atomicAdd(&cnt[min(kv[j], (uint32_t)(a.nb - 1))], 1);
    __syncthreads();
    if (direct) {
        const int row = hist16_row(a.nb);
        unsigned short *h = reinterpret_cast<unsigned short *>(a.hist) + (size_t)blockIdx.x * row;
        for (int b = threadIdx.x; b < row; b += T) h[b] = b < a.nb ? (unsigned short)cnt[b] : (unsigned short)0;
    } else {
        int *h = a.hist + (size_t)blockIdx.x * a.nb;
        for (int b = threadIdx.x; b < a.nb; b += T) h[b] = cnt[b];
    }
}

// direct form: total of every bin into base, the counts of the chunks before
// this workgroup's into off.  8 bins (16 bytes) a thread, the chunks shared by
// groups of threads, their rows loaded 8 at a time; the counts stay below
// 65536 and are added in pairs
template <int T>
__device__ __forceinline__ void sum_rows(const SortArgs &a, int *base, int *off)
{
    constexpr int R = 8;
    const int t = threadIdx.x, own = min((int)blockIdx.x, a.nchunks), row = hist16_row(a.nb), nv = row / 8;
    if (a.nchunks <= R) {
        // one round of loads without groups
        const uint32_t *h = reinterpret_cast<const uint32_t *>(a.hist);
        for (int v = t; 2 * v < a.nb; v += T) {
            uint32_t x[R], total = 0, mine = 0;
#pragma unroll
            for (int u = 0; u < R; u++) x[u] = h[max(min(u, a.nchunks - 1), 0) * (row / 2) + v];
#pragma unroll
            for (int u = 0; u < R; u++) {
                total += u < a.nchunks ? x[u] : 0u;
                mine += u < own ? x[u] : 0u;
            }
            *reinterpret_cast<int2 *>(base + 2 * v) = make_int2((int)(total & 0xffffu), (int)(total >> 16));
            *reinterpret_cast<int2 *>(off + 2 * v) = make_int2((int)(mine & 0xffffu), (int)(mine >> 16));
        }
        return;
    }
    const int groups = max(T / nv, 1);
    for (int q = t; q < a.nb; q += T) {
        base[q] = 0;
        off[q] = 0;
    }
    __syncthreads();
    const int grp = groups == 1 ? 0 : t / nv;
    if (grp >= groups) return;
    for (int v = t - grp * nv; v < nv; v += T) {
        const uint4 *h = reinterpret_cast<const uint4 *>(a.hist) + v;
        uint32_t total[4] = {0, 0, 0, 0}, mine[4] = {0, 0, 0, 0};
        for (int c0 = grp; c0 < a.nchunks; c0 += R * groups) {
            uint4 x[R];
#pragma unroll
            for (int u = 0; u < R; u++) x[u] = h[min(c0 + u * groups, a.nchunks - 1) * nv];
#pragma unroll
            for (int u = 0; u < R; u++) {
                const int c = c0 + u * groups;
                const uint32_t y[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    total[e] += c < a.nchunks ? y[e] : 0u;
                    mine[e] += c < own ? y[e] : 0u;
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int q = 8 * v + e;
            const int tv = (int)((total[e >> 1] >> (16 * (e & 1))) & 0xffffu);
            const int mv = (int)((mine[e >> 1] >> (16 * (e & 1))) & 0xffffu);
            if (tv && q < a.nb) {
                atomicAdd(&base[q], tv);
                if (mv) atomicAdd(&off[q], mv);
            }
        }
    }
}

// bin starts into base; with `direct` also this chunk's offset within each
// bin into off (else the scan left it in the histogram row)
template <int T>
__device__ inline void bin_starts(const SortArgs &a, int *base, int *off)
{
    __shared__ int wsum[T / 64];
    const int t = threadIdx.x;
    if (a.form == SORT_DIRECT) {
        sum_rows<T>(a, base, off);
    } else {
        for (int q0 = 0; q0 < a.nb; q0 += 8 * T) {
            int v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = a.tot[min(q0 + u * T + t, a.nb - 1)];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int q = q0 + u * T + t;
                if (q < a.nb) base[q] = v[u];
            }
        }
    }
    __syncthreads();
    const int bper = (a.nb + T - 1) / T;
    const int b0 = t * bper;
    int local = 0;
    for (int q = 0; q < bper; q++)
        if (b0 + q < a.nb) local += base[b0 + q];
    const int lane = t & 63, wave = t >> 6;
    int incl = local;
    for (int dd = 1; dd < 64; dd <<= 1) {
        const int y = __shfl_up(incl, dd, 64);
        if (lane >= dd) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int run = incl - local;
    for (int w = 0; w < wave; w++) run += wsum[w];
    for (int q = 0; q < bper; q++) {
        if (b0 + q < a.nb) {
            const int v = base[b0 + q];
            base[b0 + q] = run;
            run += v;
        }
    }
    __syncthreads();
}

// key window of the per-wave rank counters (bins); the counters of the waves
// are together at least one 16-bit counter per bin of 8192 cells
constexpr int kSortWindow = 1024;
template <int T>
constexpr int sort_counters() { return (T / 64) * (kSortWindow + 1); }
static_assert(sort_counters<kSortThreads>() >= 8192, "chunks whose keys spread wide: a counter per cell");

// lanes of the wave with this lane's value (of `bits` bits)
__device__ __forceinline__ uint64_t match_lanes(uint32_t v, int bits, bool valid)
{
    uint64_t match = __ballot(valid);
    for (int bit = 0; bit < bits; bit++) {
        const bool bv = (v >> bit) & 1u;
        const uint64_t bal = __ballot(bv);
        match &= bv ? bal : ~bal;
    }
    return match;
}

// rank of each of this thread's particles among the chunk's earlier particles
// with the same key
template <int T, int PER>
__device__ inline void chunk_ranks(const SortArgs &a, const uint32_t (&kv)[PER], unsigned short *cnt, int (&rank)[PER])
{
    constexpr int NW = T / 64, W = kSortWindow;
    __shared__ int kmin[NW], kmax[NW];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int nr = a.nb - 1;
    bool valid[PER];
    int lo = 0, width = nr;
#pragma unroll
    for (int j = 0; j < PER; j++) valid[j] = sort_element<T, PER>(j) < a.n && kv[j] < (uint32_t)nr;
    if (nr > W) {
        // the chunk's keys inside the box
        int mn = nr, mx = -1;
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (valid[j]) {
                mn = min(mn, (int)kv[j]);
                mx = max(mx, (int)kv[j]);
            }
        for (int d = 32; d > 0; d >>= 1) {
            mn = min(mn, __shfl_xor(mn, d, 64));
            mx = max(mx, __shfl_xor(mx, d, 64));
        }
        if (lane == 0) {
            kmin[wave] = mn;
            kmax[wave] = mx;
        }
        __syncthreads();
        mn = nr;
        mx = -1;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            mn = min(mn, kmin[w]);
            mx = max(mx, kmax[w]);
        }
        lo = __builtin_amdgcn_readfirstlane(mn);
        width = __builtin_amdgcn_readfirstlane(mx) - lo + 1;
    }
    if (width <= W) {
        const int wd = max(width, 1);
        for (int q = t; q < NW * wd; q += T) cnt[q] = 0;
        __syncthreads();
        int bits = 1;
        while ((1 << bits) < wd) bits++;
        unsigned short *mine = cnt + wave * wd;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const uint32_t w = valid[j] ? kv[j] - (uint32_t)lo : 0u;
            const uint64_t m = match_lanes(w, bits, valid[j]);
            // the group's lanes read the wave's running count, its highest
            // lane advances it
            const int c0 = mine[w];
            rank[j] = c0 + __popcll(m & lt);
            if (valid[j] && (m >> lane) == 1ull) mine[w] = (unsigned short)(c0 + __popcll(m));
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        __syncthreads();
        for (int q = t; q < wd; q += T) {
            int s = 0;
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const int v = cnt[w * wd + q];
                cnt[w * wd + q] = (unsigned short)s;
                s += v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < PER; j++) rank[j] += valid[j] ? mine[kv[j] - (uint32_t)lo] : 0;
        return;
    }
    // keys spread wide: one counter per bin, the waves in turn
    for (int q = t; q < nr; q += T) cnt[q] = 0;
    __syncthreads();
    int bits = 1;
    while ((1 << bits) < nr) bits++;
    uint64_t m[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) m[j] = match_lanes(valid[j] ? kv[j] : 0u, bits, valid[j]);
    for (int w = 0; w < NW; w++) {
        if (wave == w) {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const int c0 = valid[j] ? cnt[kv[j]] : 0;
                rank[j] = c0 + __popcll(m[j] & lt);
                if (valid[j] && (m[j] >> lane) == 1ull) cnt[kv[j]] = (unsigned short)(c0 + __popcll(m[j]));
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
        __syncthreads();
    }
}

// after bin_starts: cell c < nr (nr = nb - 1) with n_c
// particles is deposited in chunks of kDepChunk: chunk 0 into the cell's own
// partial row, chunks 1 .. into overflow rows, numbered cell by cell, chunk
// by chunk (os = exclusive prefix of their counts).  The chunks of cells of
// more than `first` particles are the crowded list of the deposits: desc =
// (cell, first particle, end, overflow row; -1: the cell's own row), their
// number at os[nr + 1].
template <int T>
__device__ inline void overflow_chunks(const SortArgs &a, const int *base)
{
    __shared__ uint64_t wsum[T / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int nr = a.nb - 1;
    const int per = (nr + T - 1) / T;
    const int c0 = t * per;
    // overflow rows (low half) and crowded chunks (high half) of n particles
    auto rows_of = [&](int n) -> uint64_t {
        const uint64_t k = n > 0 ? (uint64_t)((n - 1) / kDepChunk) : 0;
        return k | (n > a.first ? (k + 1) << 32 : 0);
    };
    uint64_t local = 0;
    for (int q = 0; q < per; q++)
        if (c0 + q < nr) local += rows_of(base[c0 + q + 1] - base[c0 + q]);
    uint64_t incl = local;
    for (int dd = 1; dd < 64; dd <<= 1) {
        const uint64_t y = __shfl_up(incl, dd, 64);
        if (lane >= dd) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    uint64_t run = incl - local;
    for (int w = 0; w < wave; w++) run += wsum[w];
    for (int q = 0; q < per; q++) {
        const int c = c0 + q;
        if (c >= nr) break;
        const int p0 = base[c], p1 = base[c + 1];
        const uint64_t k = rows_of(p1 - p0);
        const int row0 = (int)(uint32_t)run, at = (int)(run >> 32), chunks = (int)(k >> 32);
        a.os[c] = min(row0, a.n_ov_max);
        for (int u = 0; u < chunks; u++)
            if (at + u < a.n_crowd_max)
                a.desc[at + u] = make_int4(c, p0 + u * kDepChunk, min(p0 + (u + 1) * kDepChunk, p1),
                                           u == 0 ? -1 : min(row0 + u - 1, a.n_ov_max - 1));
        run += k;
    }
    // the last thread's running counts are the totals (its range may be
    // empty); overflow rows never exceed n_ov_max (the chunks of n particles
    // number < n / kDepChunk), crowded chunks never n_crowd_max
    if (t == T - 1) {
        a.os[nr] = min((int)(uint32_t)run, a.n_ov_max);
        a.os[nr + 1] = min((int)(run >> 32), a.n_crowd_max);
    }
}

// dynamic LDS of a scattering workgroup: bin starts, offsets (direct), rank
// counters
template <int T>
inline size_t scatter_lds(int nb, int form)
{
    return sizeof(int) * (size_t)hist16_row(nb) * (form == SORT_DIRECT ? 2 : 1) + sizeof(unsigned short) * (size_t)sort_counters<T>();
}

// the scattering pass up to the positions: destination of each of this
// thread's particles (-1: past the end, or left the box: nothing reads it
// again).  false for the extra workgroup, which closes the sort instead.
template <int T, int PER>
__device__ __forceinline__ bool scatter_positions(const SortArgs &a, const uint32_t (&kv)[PER], int *lds, int (&dp)[PER])
{
    int *base = lds, *off = lds + hist16_row(a.nb);
    unsigned short *cnt = reinterpret_cast<unsigned short *>(lds + (size_t)hist16_row(a.nb) * (a.form == SORT_DIRECT ? 2 : 1));
    bin_starts<T>(a, base, off);
    if ((int)blockIdx.x == a.nchunks) {
        for (int b = threadIdx.x; b < a.nb; b += T) a.cs[b] = base[b];
        if (threadIdx.x == 0) a.cs[a.nb] = (int32_t)a.n;
        overflow_chunks<T>(a, base);
        return false;
    }
    int rank[PER];
    chunk_ranks<T, PER>(a, kv, cnt, rank);
    const int *row = a.form == SORT_DIRECT ? off : a.hist + (size_t)blockIdx.x * a.nb;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const bool live = sort_element<T, PER>(j) < a.n && kv[j] < (uint32_t)(a.nb - 1);
        dp[j] = live ? base[kv[j]] + row[kv[j]] + rank[j] : -1;
    }
    return true;
}

// ---- host side (k_sort.hip) ----
// the form of species s by itself (SORT_LARGE takes every count)
int sort_form(qpad_ctx *c, int s);
// its arguments in that form or a more demanding species' (SORT_* below it)
SortArgs sort_args(qpad_ctx *c, int s, int form);
struct SortMulti {
    SortArgs s[kMaxSpecies];
};
// the sort of the species of m.s[0 .. ns-1], all in one form (workgroup rows
// by species); counted: the push has counted the keys already
int launch_sort_list(qpad_ctx *c, const SortMulti &m, int ns, bool counted);
// the sorted buffers become the current ones
void sort_swap(Species &sp);

}  // namespace qpad
