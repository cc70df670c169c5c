// k_sort.hip -- the re-sort of a plasma species by radial cell (of a slice,
// after injection, or when the caller sets particles): its launches and its
// host side; the passes are described in sort_device.h.
#include <algorithm>
#include <cstring>
#include <string>

#include "kernels.h"
#include "sort_device.h"

namespace qpad {

constexpr int kScanThreads = 512;
constexpr int kScanGroups = 16;       // chunk groups per bin in k_sort_scan
constexpr int kScanBins = kScanThreads / kScanGroups;

template <int T, int PER>
__device__ __forceinline__ void load_keys(const SortArgs &a, uint32_t (&kv)[PER])
{
#pragma unroll
    for (int j = 0; j < PER; j++)
        kv[j] = a.n ? min(a.key[min(sort_element<T, PER>(j), a.n - 1)], (uint32_t)(a.nb - 1)) : 0u;
}

template <int T, int PER>
__global__ __launch_bounds__(T) void k_sort_hist(const SortMulti m)
{
    const SortArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    if ((int)blockIdx.x >= a.nchunks) return;   // the species has fewer chunks than the grid
    extern __shared__ __attribute__((aligned(16))) int lds[];
    uint32_t kv[PER];
    load_keys<T, PER>(a, kv);
    chunk_hist<T, PER>(a, kv, lds);
}

// workgroup = kScanBins bins x kScanGroups chunk groups; each thread prefixes
// a contiguous run of at most RUN chunks of its bin (held in registers; RUN
// is the smallest of 8, 16, 32, 64 that covers nchunks / kScanGroups), the
// groups are then prefixed in LDS
constexpr int kScanRun = 64;
constexpr int kMaxSortChunks = kScanGroups * kScanRun;

template <int RUN>
__global__ __launch_bounds__(kScanThreads) void k_sort_scan(const SortMulti m)
{
    const SortArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    __shared__ int gsum[kScanGroups][kScanBins];
    const int t = threadIdx.x;
    const int lb = t % kScanBins, grp = t / kScanBins;
    const int b = blockIdx.x * kScanBins + lb;
    const int per = (a.nchunks + kScanGroups - 1) / kScanGroups;   // <= RUN
    const int c0 = grp * per;
    // clamped (always valid) addresses, masked values: no branches between
    // the loads, which all issue together
    const int bc = min(b, a.nb - 1);
    int h[RUN];
#pragma unroll
    for (int u = 0; u < RUN; u++) {
        const int c = min(c0 + u, max(a.nchunks - 1, 0));
        const int x = a.hist[(size_t)c * a.nb + bc];
        h[u] = (b < a.nb && u < per && c0 + u < a.nchunks) ? x : 0;
    }
    int run = 0;
#pragma unroll
    for (int u = 0; u < RUN; u++) {
        const int v = h[u];
        h[u] = run;
        run += v;
    }
    gsum[grp][lb] = run;
    __syncthreads();
    int goff = 0, total = 0;
    for (int q = 0; q < kScanGroups; q++) {
        const int v = gsum[q][lb];
        if (q < grp) goff += v;
        total += v;
    }
#pragma unroll
    for (int u = 0; u < RUN; u++) {
        const int c = c0 + u;
        if (b < a.nb && u < per && c < a.nchunks) a.hist[(size_t)c * a.nb + b] = h[u] + goff;
    }
    if (grp == 0 && b < a.nb) a.tot[b] = total;
}

template <int T, int PER>
__global__ __launch_bounds__(T) void k_sort_scatter(const SortMulti m)
{
    const SortArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    if ((int)blockIdx.x > a.nchunks) return;
    extern __shared__ __attribute__((aligned(16))) int lds[];
    uint32_t kv[PER];
    load_keys<T, PER>(a, kv);
    int dp[PER];
    if (!scatter_positions<T, PER>(a, kv, lds, dp)) return;
    // every load of the chunk first (all in flight), then the stores
    double v[8][PER];
    int32_t vi[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int64_t e = min(sort_element<T, PER>(j), a.n - 1);
#pragma unroll
        for (int f = 0; f < 8; f++) v[f][j] = a.s[f][e];
        vi[j] = a.sid[e];
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        if (dp[j] < 0) continue;
#pragma unroll
        for (int f = 0; f < 8; f++) a.d[f][dp[j]] = v[f][j];
        a.did[dp[j]] = vi[j];
    }
}

int sort_workspace(int64_t npmax, int nr, size_t *hist_ints)
{
    const int64_t nchunks = (npmax + kSortChunk - 1) / kSortChunk;
    if (nchunks > kMaxSortChunks) {
        set_error("too many particles per species for the cell sort (max " +
                  std::to_string((long long)kMaxSortChunks * kSortChunk) + ")");
        return QPAD_E_INVALID;
    }
    // up to kMidMax particles in smaller chunks; the direct form's rows hold
    // 16-bit counts, two small chunks in the space of a mid one
    const int64_t mid = (std::min(npmax, kMidMax) + kMidChunk - 1) / kMidChunk;
    static_assert(2 * kSmallChunk == kMidChunk, "16-bit rows of small chunks in the space of the mid ones");
    *hist_ints = (size_t)std::max(nchunks, mid) * (size_t)hist16_row(nr + 1);
    return 0;
}

int sort_form(qpad_ctx *c, int s)
{
    const int64_t n = c->sp[s].npp;
    const int nr = c->g.nr, nb = nr + 1;
    // direct: push and re-sort, us a slice, chunks of 2048 with the scan launch
    // -> direct: 4096 particles in 256 cells 24.1 -> 11.7, 21189 in 1009 23.4 ->
    // 15.5, 24576 in 768 27 -> 19.5 (the sum over the chunks grows with chunks x
    // bins: at 131072 its 2 us equal the scan launch)
    // mid: the sort's three launches, us, chunks of 2048 -> 1024: 65536 in 512
    // cells 18.5 -> 15.4, 262144 in 512 21.7 -> 17.9, in 2048 22.1 -> 19.7, in
    // 4096 23.8 -> 23.1; 131072 in 8192 24.6 -> 24.7.  Past the line the larger
    // histogram costs more than the shorter chunks give: 393216 in 512 23.6 ->
    // 23.6, in 2048 24.2 -> 25.2, in 4096 25.7 -> 28.3; 196608 in 8192 26.0 -> 28.4
    const int64_t small = (n + kSmallChunk - 1) / kSmallChunk, mid = (n + kMidChunk - 1) / kMidChunk;
    if (nb <= kDirectBins && small <= kDirectChunks && small * nb <= kDirectWork) return SORT_DIRECT;
    return n <= kMidMax && mid * nr <= kMidWork ? SORT_MID : SORT_LARGE;
}

SortArgs sort_args(qpad_ctx *c, int s, int form)
{
    Species &sp = c->sp[s];
    const int64_t n = sp.npp;
    SortArgs a;
    memset(&a, 0, sizeof(a));
    a.n = n;
    a.nb = c->g.nr + 1;
    a.form = form;
    const int chunk = a.form == SORT_LARGE ? kSortChunk : a.form == SORT_MID ? kMidChunk : kSmallChunk;
    a.nchunks = (int)((n + chunk - 1) / chunk);
    a.key = sp.key;
    a.key_w = sp.key;
    a.hist = sp.hist;
    a.tot = sp.tot;
    a.cs = sp.cell_start;
    const double *src[8] = {sp.x1, sp.x2, sp.p1, sp.p2, sp.p3, sp.q, sp.gamma, sp.psi};
    double *dst[8] = {sp.a_x1, sp.a_x2, sp.a_p1, sp.a_p2, sp.a_p3, sp.a_q, sp.a_gamma, sp.a_psi};
    for (int f = 0; f < 8; f++) {
        a.s[f] = src[f];
        a.d[f] = dst[f];
    }
    a.sid = sp.id;
    a.did = sp.a_id;
    a.os = sp.ov_start;
    a.desc = sp.ov_desc;
    a.n_ov_max = sp.n_ov_max;
    a.n_crowd_max = sp.n_crowd_max;
    a.first = sp.dep_first;
    return a;
}

void sort_swap(Species &sp)
{
    if (sp.npp <= 0) return;
    std::swap(sp.x1, sp.a_x1); std::swap(sp.x2, sp.a_x2);
    std::swap(sp.p1, sp.a_p1); std::swap(sp.p2, sp.a_p2); std::swap(sp.p3, sp.a_p3);
    std::swap(sp.q, sp.a_q); std::swap(sp.gamma, sp.a_gamma); std::swap(sp.psi, sp.a_psi);
    std::swap(sp.id, sp.a_id);
}

static int launch_sort_scan(qpad_ctx *c, const SortMulti &m, int ns, int maxc)
{
    const int nb = c->g.nr + 1;
    const dim3 sg((nb + kScanBins - 1) / kScanBins, ns), sb(kScanThreads);
    const int per = (maxc + kScanGroups - 1) / kScanGroups;
    if (per <= 8) hipLaunchKernelGGL(k_sort_scan<8>, sg, sb, 0, c->stream, m);
    else if (per <= 16) hipLaunchKernelGGL(k_sort_scan<16>, sg, sb, 0, c->stream, m);
    else if (per <= 32) hipLaunchKernelGGL(k_sort_scan<32>, sg, sb, 0, c->stream, m);
    else hipLaunchKernelGGL(k_sort_scan<kScanRun>, sg, sb, 0, c->stream, m);
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_sort_list(qpad_ctx *c, const SortMulti &m, int ns, bool counted)
{
    int maxc = 0;
    for (int i = 0; i < ns; i++) maxc = std::max(maxc, m.s[i].nchunks);
    const int nb = c->g.nr + 1;
    const int form = m.s[0].form;
    const size_t hl = sizeof(int) * (size_t)nb;
    const dim3 cg(std::max(maxc, 1), ns), mg(maxc + 1, ns);
#define QPAD_SORT(T, PER)                                                                              \
    do {                                                                                              \
        if (maxc && !counted) hipLaunchKernelGGL((k_sort_hist<T, PER>), cg, dim3(T), hl, c->stream, m);            \
        if (form != SORT_DIRECT) QPAD_TRY(launch_sort_scan(c, m, ns, maxc));                           \
        hipLaunchKernelGGL((k_sort_scatter<T, PER>), mg, dim3(T), scatter_lds<T>(nb, form), c->stream, m); \
    } while (0)
    if (form == SORT_LARGE) QPAD_SORT(kSortThreads, kSortChunk / kSortThreads);
    else if (form == SORT_MID) QPAD_SORT(kSortThreads, kMidChunk / kSortThreads);
    else QPAD_SORT(kSortThreads, kSmallChunk / kSortThreads);
#undef QPAD_SORT
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_sort(qpad_ctx *c, int s)
{
    SortMulti m;
    memset(&m, 0, sizeof(m));
    m.s[0] = sort_args(c, s, sort_form(c, s));
    QPAD_TRY(launch_sort_list(c, m, 1, false));
    sort_swap(c->sp[s]);
    return 0;
}

}  // namespace qpad
