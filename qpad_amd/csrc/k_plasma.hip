// k_plasma.hip -- 2D plasma species on the GPU (FP64): lattice injection,
// radial-cell sort, rho - Jz deposit, the fused gather + robust predictor +
// current/acceleration/momentum-flux deposit, and the fused push_u + push_x.
//
// Particles are kept sorted by radial cell (cell c = int(r/dr), nodes c+1 and
// c+2).  A wavefront deposits a cell of ordinary size; the chunks (at most
// kDepChunk particles) of a crowded cell are each deposited by four
// wavefronts.  The partials of a cell's first chunk for node c+1 and node c+2
// go to P0/P1[c], those of its further chunks to the overflow rows O0/O1 the
// sort numbers; the field kernels add P0[i-1] + P1[i-2] per node, each with
// its cell's overflow rows in row order.  No atomics, deterministic order.
#include <algorithm>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "kernels.h"
#include "sort_config.h"
#include "epilogue.h"
#include "sort_device.h"
#include "rng.h"
#include "wave_reduce.h"
#include "conv.h"

namespace qpad {

#define FX(p, c, k, i) (p)[((size_t)(c) * nm + (size_t)(k)) * ld + (size_t)(i)]

// Radius of a deposit or a gather, contracted as the compiler likes: an ulp
// between kernels is harmless there (the cell comes from the sort or is
// clamped, the weights are linear in the position).
__device__ inline double radius(double x1, double x2)
{
    return sqrt(__dadd_rn(__dmul_rn(x1, x1), __dmul_rn(x2, x2)));
}

// ---------------------------------------------------------------------------
// injection: fdist2d_class.f03:289-357 (lattice theta).  A uniform plasma
// keeps every lattice point; a profiled one (den_perp given) keeps the points
// whose den_lon * den_perp * density reaches den_min, at the exclusive prefix
// `off` of the kept flags, so that the kept particles keep QPAD's order and
// their index (which also draws their thermal momenta) counts kept points.
// ---------------------------------------------------------------------------
struct InjArgs {
    int nr, ppc1, ppc2, nth;
    int64_t n;
    double dr, idr, edge, density, coef, qm, dtheta, den_lon, den_min;
    double uth0, uth1, uth2;
    uint64_t seed;
    const double *den;       // transverse density per lattice point (null: 1)
    const int32_t *off;      // kept points' exclusive prefix (null: all kept)
    double *x1, *x2, *p1, *p2, *p3, *q, *gamma, *psi;
    int32_t *id;
    uint32_t *key;
};

// kept flag of every lattice point, 0 in the pad entry n
__global__ void k_inject_keep(int64_t n, const double *den, double den_lon, double density, double den_min,
                              int32_t *keep)
{
    const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l > n) return;
    keep[l] = l < n ? (den_lon * den[l] * density < den_min ? 0 : 1) : 0;
}

__global__ void k_inject(InjArgs a)
{
    const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= a.n) return;
    int64_t ip = l;
    if (a.off) {
        if (a.off[l + 1] == a.off[l]) return;
        ip = a.off[l];
    }
    int64_t t = l;
    const int i2 = (int)(t % a.ppc2); t /= a.ppc2;
    const int i1 = (int)(t % a.ppc1); t /= a.ppc1;
    const int i = (int)(t % a.nr);
    const int j = (int)(t / a.nr);
    // 1-based loop indices of the reference: j+1, i+1, i1+1, i2+1
    double rn = ((double)(i1 + 1) - 0.5) / (double)a.ppc1 + (double)i;
    double theta = (((double)(i2 + 1) - 0.5) / (double)a.ppc2 + (double)(j + 1) - 1.0) * a.dtheta;
    double x1 = rn * a.dr * cos(theta), x2 = rn * a.dr * sin(theta);
    double th[4] = {0.0, 0.0, 0.0, 0.0};
    if (a.uth0 != 0.0 || a.uth1 != 0.0 || a.uth2 != 0.0) normal4(a.seed, (uint64_t)ip, 0u, th);
    double p1 = a.uth0 * th[0], p2 = a.uth1 * th[1], p3 = a.uth2 * th[2];
    double gam = sqrt(1.0 + p1 * p1 + p2 * p2 + p3 * p3);
    const double den_perp = a.den ? a.den[l] : 1.0;
    a.x1[ip] = x1;
    a.x2[ip] = x2;
    a.q[ip] = rn * den_perp * a.den_lon * a.density * a.coef;
    a.p1[ip] = p1;
    a.p2[ip] = p2;
    a.p3[ip] = p3;
    a.gamma[ip] = gam;
    a.psi[ip] = (1.0 - gam + p3) / a.qm;
    a.id[ip] = (int32_t)ip;
    a.key[ip] = cell_key(x1, x2, a.idr, a.edge, a.nr);
}

int launch_inject(qpad_ctx *c, int s)
{
    Species &sp = c->sp[s];
    const qpad_species_cfg &cf = sp.cfg;
    InjArgs a;
    a.nr = c->g.nr;
    a.ppc1 = cf.ppc1;
    a.ppc2 = cf.ppc2;
    a.nth = cf.num_theta;
    a.n = (int64_t)cf.num_theta * c->g.nr * cf.ppc1 * cf.ppc2;
    a.dr = c->g.dr;
    a.idr = 1.0 / c->g.dr;
    a.edge = (double)c->g.nr * c->g.dr;
    a.density = cf.density;
    a.coef = copysign(1.0, cf.qm) / ((double)(cf.ppc1 * cf.ppc2) * (double)cf.num_theta);
    a.qm = cf.qm;
    a.dtheta = 2.0 * (4.0 * atan(1.0)) / (double)cf.num_theta;
    a.den_lon = sp.den_perp ? sp.den_lon : 1.0;
    a.den_min = cf.den_min;
    a.uth0 = cf.uth[0];
    a.uth1 = cf.uth[1];
    a.uth2 = cf.uth[2];
    a.seed = cf.seed;
    a.den = sp.den_perp;
    a.off = nullptr;
    a.x1 = sp.x1; a.x2 = sp.x2; a.p1 = sp.p1; a.p2 = sp.p2; a.p3 = sp.p3;
    a.q = sp.q; a.gamma = sp.gamma; a.psi = sp.psi; a.id = sp.id;
    a.key = sp.key;
    int64_t kept = a.n;
    if (sp.den_perp) {
        hipLaunchKernelGGL(k_inject_keep, dim3((unsigned)((a.n + 1 + 255) / 256)), dim3(256), 0, c->stream, a.n,
                           sp.den_perp, a.den_lon, a.density, a.den_min, sp.inj_keep);
        QPAD_HIP_CHECK(hipGetLastError());
        size_t bytes = sp.inj_tmp_bytes;
        QPAD_HIP_CHECK(rocprim::exclusive_scan(sp.inj_tmp, bytes, sp.inj_keep, sp.inj_off, 0, (size_t)a.n + 1,
                                               rocprim::plus<int32_t>(), c->stream));
        QPAD_HIP_CHECK(hipMemcpyAsync(sp.inj_host, sp.inj_off + a.n, sizeof(int32_t), hipMemcpyDeviceToHost,
                                      c->stream));
        QPAD_HIP_CHECK(hipStreamSynchronize(c->stream));
        kept = *sp.inj_host;
        a.off = sp.inj_off;
    } else if (1.0 * 1.0 * cf.density < cf.den_min) {
        // den_lon * den_perp * density < den_min drops every particle
        kept = 0;
    }
    sp.npp = kept;
    if (kept > 0) {
        hipLaunchKernelGGL(k_inject, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, c->stream, a);
        QPAD_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

// scan scratch of the profiled injection of n lattice points
int inject_scan_bytes(int64_t n, size_t *bytes)
{
    int32_t *z = nullptr;
    QPAD_HIP_CHECK(rocprim::exclusive_scan(nullptr, *bytes, z, z, 0, (size_t)n + 1, rocprim::plus<int32_t>()));
    return 0;
}

// ---------------------------------------------------------------------------
// cell start offsets of sorted keys (the beam's (xi, r)-cell sort)
// ---------------------------------------------------------------------------
// cs[c] = first position p with key[p] >= c (lower bound in the sorted
// keys), for c = 0 .. ncs-1: one thread per cell, so empty runs of cells
// cost nothing extra
__global__ __launch_bounds__(256) void k_cellstart(const uint32_t *key, int64_t n, int ncs, int32_t *cs)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncs) return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = lo + ((hi - lo) >> 1);
        if (key[mid] < (uint32_t)c) lo = mid + 1;
        else hi = mid;
    }
    cs[c] = (int32_t)lo;
}

int launch_cell_start(qpad_ctx *c, const uint32_t *key, int64_t n, int ncs, int32_t *cs)
{
    hipLaunchKernelGGL(k_cellstart, dim3((unsigned)((ncs + 255) / 256)), dim3(256), 0, c->stream, key, n, ncs,
                       cs);
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

// scratch of rocPRIM's radix sort (uint32 keys and values) and exclusive scan
int sort_scratch(size_t n, int bits, size_t *bytes)
{
    size_t b1 = 0, b2 = 0;
    uint32_t *z = nullptr;
    QPAD_HIP_CHECK(rocprim::radix_sort_pairs<SortConfig>(nullptr, b1, z, z, z, z, n, 0, bits));
    QPAD_HIP_CHECK(rocprim::exclusive_scan(nullptr, b2, z, z, 0u, n, rocprim::plus<uint32_t>()));
    *bytes = std::max(b1, b2) + 256;
    return 0;
}

__global__ void k_keys(const double *x1, const double *x2, uint32_t *key, int64_t n, double idr, double edge,
                       int nr)
{
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    key[p] = cell_key(x1[p], x2[p], idr, edge, nr);
}

int launch_keys(qpad_ctx *c, int s)
{
    Species &sp = c->sp[s];
    if (sp.npp == 0) return 0;
    hipLaunchKernelGGL(k_keys, dim3((unsigned)((sp.npp + 255) / 256)), dim3(256), 0, c->stream, sp.x1, sp.x2,
                       sp.key, sp.npp, 1.0 / c->g.dr, (double)c->g.nr * c->g.dr, c->g.nr);
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------------------
// rho - Jz deposit: qdeposit_part2d (part2d_class.f03:231-359), per-cell
// partials; axis rules and 1/r are applied by the consumer
// ---------------------------------------------------------------------------
struct QDepArgs {
    int nr;
    double idr;
    const double *x1, *x2, *q;
    // susceptibility deposit (CHI): the particle's psi and q/m
    const double *psi;
    double qbm;
    const int32_t *cs;
    double *P0, *P1;
    // the crowded cells' chunks (listed by the sort) and the overflow rows
    const int32_t *os;
    const int4 *desc;
    double *O0, *O1;
    int first, n_crowd_max;
};

// What a deposit workgroup of CPW waves does.  The first ceil(nr / CPW)
// workgroups take the cells of at most `first` particles, one wave per cell
// (cell = workgroup * CPW + wave), into P0/P1.  The workgroups after them
// walk the list of crowded chunks: every chunk is cut into kDepSub parts of
// kDepChunk / kDepSub particles, one wave per part (a wave takes two parts
// where CPW = 2, a workgroup two chunks where CPW = 8), whose sums are added
// in LDS in part order into the chunk's row.  A single wave over a whole
// chunk (16 passes) would hold the launch up long after the ordinary cells
// are done.  CPW: waves per workgroup, a launch shape the tuner chooses
// (qpad_tune_launch); every part's work and the order of the sums are the
// same for every shape.
constexpr int kDepSub = 4;
constexpr int kDepPart = kDepChunk / kDepSub;
// at most this many workgroups walk the crowded list (on few cells all of
// them may be on it, and fewer would walk it in rounds: 512 per cell in 1024
// cells, M = 0, 7.2 ms with 512, 5.5 with 1024)
inline int crowd_groups(int nr) { return nr <= kDepFewCells ? kDepFewCells : 256; }

template <int CPW>
constexpr int crowd_chunks() { return CPW >= 2 * kDepSub ? CPW / kDepSub : 1; }   // chunks of a workgroup at once
template <int CPW>
constexpr int crowd_parts() { return CPW < kDepSub ? kDepSub / CPW : 1; }         // parts of a wave

struct DepRange {
    int cell, pb, pe;
};

// the cell of a wave (cells of more than `first` particles are on the
// crowded list; live false for those and past the last cell)
template <int CPW>
__device__ __forceinline__ DepRange cell_range(int nr, const int32_t *cs, int first, int wave, bool &live)
{
    const int c = blockIdx.x * CPW + wave;
    DepRange k;
    k.cell = min(c, nr - 1);
    k.pb = __builtin_amdgcn_readfirstlane(cs[k.cell]);
    k.pe = __builtin_amdgcn_readfirstlane(cs[k.cell + 1]);
    live = c < nr && k.pe - k.pb <= first;
    return k;
}

// entry o of the crowded list (uniform over the wave)
__device__ __forceinline__ int4 crowd_entry(const int4 *desc, int o)
{
    const int4 d = desc[o];
    return make_int4(__builtin_amdgcn_readfirstlane(d.x), __builtin_amdgcn_readfirstlane(d.y),
                     __builtin_amdgcn_readfirstlane(d.z), __builtin_amdgcn_readfirstlane(d.w));
}

// part `sub` of a crowded chunk (cell, first particle, end, row)
__device__ __forceinline__ DepRange part_range(const int4 &d, int sub, bool live)
{
    DepRange k;
    k.cell = d.x;
    k.pb = min(d.y + sub * kDepPart, d.z);
    k.pe = live ? min(k.pb + kDepPart, d.z) : k.pb;
    return k;
}

// workgroups of a deposit over (at most) npp particles: the cells', then the
// crowded list's (a chunk holds kDepChunk particles or closes a cell of more
// than `first`)
inline int dep_grid(int nr, int64_t npp, int first, int cpw)
{
    const int chunks = (int)std::min<int64_t>(npp / (first + 1) + npp / kDepChunk, 1 << 20);
    const int per = cpw >= 2 * kDepSub ? cpw / kDepSub : 1;
    return (nr + cpw - 1) / cpw + std::min((chunks + per - 1) / per, crowd_groups(nr));
}

// the arguments of every species of one launch (workgroup rows by species)
struct QDepMulti {
    QDepArgs s[kMaxSpecies];
};

// sums of the particles [p0, p1) of cell c over the wave: lane l ends with
// values [(l / 4) NB, (l / 4 + 1) NB) of [node][mode array] (padded to 16 NB)
// CHI: deposit_chi_part2d (part2d_class.f03:361-476) instead: each particle
// deposits -(q/m) q / (1 - (q/m) psi) in place of q
template <int M, bool CHI, int NB>
__device__ __forceinline__ void qdep_sums(const QDepArgs &a, int c, int p0, int p1, int lane, double (&acc)[16 * NB])
{
    constexpr int NM = 2 * M + 1;
#pragma unroll
    for (int v = 0; v < 16 * NB; v++) acc[v] = 0.0;
    // wave-uniform passes, software-pipelined as in k_amjdeposit; lanes past
    // the range's end deposit zero
    const int npass = __builtin_amdgcn_readfirstlane((p1 - p0 + 63) >> 6);
    const int pl = max(p1 - 1, 0);
    int p = p0 + lane;
    int pc = min(p, pl);
    double nx1 = a.x1[pc], nx2 = a.x2[pc], nq = a.q[pc];
    double npsi = CHI ? a.psi[pc] : 0.0;
    for (int k = 0; k < npass; k++, p += 64) {
        const double x1 = nx1, x2 = nx2;
        double q = p < p1 ? nq : 0.0;
        if constexpr (CHI) q = p < p1 ? -1.0 * a.qbm * nq / (1.0 - a.qbm * npsi) : 0.0;
        pc = min(p + 64, pl);
        nx1 = a.x1[pc];
        nx2 = a.x2[pc];
        nq = a.q[pc];
        if constexpr (CHI) npsi = a.psi[pc];
        double pos = __dmul_rn(radius(x1, x2), a.idr);
        double ph0r = x1 / pos * a.idr, ph0i = -x2 / pos * a.idr;
        double w1 = pos - (double)c, w0 = 1.0 - w1;
        double phr = 1.0 * q, phi = 0.0 * q;
        acc[0] += w0 * phr;
        acc[NM] += w1 * phr;
#pragma unroll
        for (int m = 1; m <= M; m++) {
            double tr = phr * ph0r - phi * ph0i, ti = phr * ph0i + phi * ph0r;
            phr = tr;
            phi = ti;
            acc[2 * m - 1] += w0 * phr;
            acc[NM + 2 * m - 1] += w1 * phr;
            acc[2 * m] += w0 * phi;
            acc[NM + 2 * m] += w1 * phi;
        }
    }
    wave_reduce_scatter<NB>(acc);
}

template <int M, int CPW, bool CHI = false>
__global__ __launch_bounds__(64 * CPW) void k_qdeposit(const QDepMulti m)
{
    const QDepArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    constexpr int NM = 2 * M + 1, NB = (2 * NM + 15) / 16;
    constexpr int CH = crowd_chunks<CPW>(), PT = crowd_parts<CPW>();
    __shared__ double comb[CH][kDepSub][2 * NM];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ncg = (a.nr + CPW - 1) / CPW;
    double acc[16 * NB];
    // value v of this lane's sums to D0[v] (node ix) or D1[v - NM] (node ix + 1)
    auto store = [&](double *D0, double *D1) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int v = (lane >> 2) * NB + i;
            if ((lane & 3) == (i & 3) && v < 2 * NM) {
                if (v < NM) D0[v] = acc[i];
                else D1[v - NM] = acc[i];
            }
        }
    };
    if ((int)blockIdx.x < ncg) {
        bool live;
        const DepRange r = cell_range<CPW>(a.nr, a.cs, a.first, wave, live);
        if (!live) return;
        qdep_sums<M, CHI, NB>(a, r.cell, r.pb, r.pe, lane, acc);
        store(a.P0 + (size_t)r.cell * NM, a.P1 + (size_t)r.cell * NM);
        return;
    }
    const int n = min(a.os[a.nr + 1], a.n_crowd_max), step = ((int)gridDim.x - ncg) * CH;
    for (int o0 = ((int)blockIdx.x - ncg) * CH; o0 < n; o0 += step) {
        const int ch = wave / (CPW / CH), o = o0 + ch;
        const bool live = o < n;
        const int4 d = crowd_entry(a.desc, min(o, n - 1));
#pragma unroll
        for (int u = 0; u < PT; u++) {
            const int sub = (wave % (CPW / CH)) * PT + u;
            const DepRange r = part_range(d, sub, live);
            qdep_sums<M, CHI, NB>(a, r.cell, r.pb, r.pe, lane, acc);
            store(comb[ch][sub], comb[ch][sub] + NM);
        }
        __syncthreads();
        for (int t = threadIdx.x; t < CH * 2 * NM; t += 64 * CPW) {
            const int q = t / (2 * NM), v = t % (2 * NM);
            if (o0 + q >= n) continue;
            const int4 e = a.desc[o0 + q];
            const double sum = ((comb[q][0][v] + comb[q][1][v]) + comb[q][2][v]) + comb[q][3][v];
            double *D = e.w < 0 ? (v < NM ? a.P0 : a.P1) + (size_t)e.x * NM : (v < NM ? a.O0 : a.O1) + (size_t)e.w * NM;
            D[v < NM ? v : v - NM] = sum;
        }
        __syncthreads();
    }
}

static QDepArgs qdep_args(qpad_ctx *c, int s)
{
    Species &sp = c->sp[s];
    QDepArgs a;
    a.nr = c->g.nr;
    a.idr = 1.0 / c->g.dr;
    a.x1 = sp.x1; a.x2 = sp.x2; a.q = sp.q;
    a.psi = sp.psi;
    a.qbm = sp.qbm;
    a.cs = sp.cell_start;
    a.P0 = sp.P0;
    a.P1 = sp.P1;
    a.os = sp.ov_start;
    a.desc = sp.ov_desc;
    a.O0 = sp.O0;
    a.O1 = sp.O1;
    a.first = sp.dep_first;
    a.n_crowd_max = sp.n_crowd_max;
    return a;
}

int launch_qdeposit(qpad_ctx *c, int s) { return launch_qdeposit_range(c, s, s + 1); }

int launch_qdeposit_all(qpad_ctx *c) { return c->nspecies ? launch_qdeposit_range(c, 0, c->nspecies) : 0; }

// the charge deposit of the species in m.s[0 .. ns-1], gx workgroups per
// species (chi: the susceptibility deposit)
static int qdeposit_launch(qpad_ctx *c, const QDepMulti &m, int ns, int gx, bool chi = false)
{
    const int cpw = c->dep_cells;
    dim3 grid((unsigned)gx, (unsigned)ns), blk(64 * cpw);
#define QPAD_QDEP(MM, CC)                                                                        \
    do {                                                                                         \
        if (chi) hipLaunchKernelGGL((k_qdeposit<MM, CC, true>), grid, blk, 0, c->stream, m);     \
        else hipLaunchKernelGGL((k_qdeposit<MM, CC, false>), grid, blk, 0, c->stream, m);        \
    } while (0)
#define QPAD_QDEP_M(MM)                              \
    do {                                             \
        if (cpw == 2) QPAD_QDEP(MM, 2);              \
        else if (cpw == 8) QPAD_QDEP(MM, 8);         \
        else QPAD_QDEP(MM, 4);                       \
    } while (0)
    switch (c->g.M) {
    case 0: QPAD_QDEP_M(0); break;
    case 1: QPAD_QDEP_M(1); break;
    case 2: QPAD_QDEP_M(2); break;
    case 3: QPAD_QDEP_M(3); break;
    default: QPAD_QDEP_M(4); break;
    }
#undef QPAD_QDEP_M
#undef QPAD_QDEP
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

// species s0 .. s1-1 in one launch
int launch_qdeposit_range(qpad_ctx *c, int s0, int s1)
{
    QDepMulti m;
    memset(&m, 0, sizeof(m));
    int gx = 1;
    for (int s = s0; s < s1; s++) {
        m.s[s - s0] = qdep_args(c, s);
        gx = std::max(gx, dep_grid(c->g.nr, c->sp[s].npp, c->sp[s].dep_first, c->dep_cells));
    }
    return qdeposit_launch(c, m, s1 - s0, gx);
}

// species s with its partial rows in caller-given memory instead of the
// species' own: rows.P0/P1 hold nr rows and rows.O0/O1 n_ov_max rows of nm
// values each.  Every row a consumer reads is written (empty cells write
// zeros), so the rows need no clearing.
int launch_qdeposit_rows(qpad_ctx *c, int s, const DepRows &rows)
{
    QDepMulti m;
    memset(&m, 0, sizeof(m));
    m.s[0] = qdep_args(c, s);
    m.s[0].P0 = rows.P0;
    m.s[0].P1 = rows.P1;
    m.s[0].O0 = rows.O0;
    m.s[0].O1 = rows.O1;
    const int gx = std::max(1, dep_grid(c->g.nr, c->sp[s].npp, c->sp[s].dep_first, c->dep_cells));
    return qdeposit_launch(c, m, 1, gx);
}

// the susceptibility deposit of species s into caller-given rows (as
// launch_qdeposit_rows)
int launch_chi_deposit_rows(qpad_ctx *c, int s, const DepRows &rows)
{
    QDepMulti m;
    memset(&m, 0, sizeof(m));
    m.s[0] = qdep_args(c, s);
    m.s[0].P0 = rows.P0;
    m.s[0].P1 = rows.P1;
    m.s[0].O0 = rows.O0;
    m.s[0].O1 = rows.O1;
    const int gx = std::max(1, dep_grid(c->g.nr, c->sp[s].npp, c->sp[s].dep_first, c->dep_cells));
    return qdeposit_launch(c, m, 1, gx, true);
}

// one species' q (axis rules, 1/r) times `scale` into out (1 x nm x ld)
__global__ void k_combine_q(const double *P0, const double *P1, const double *O0, const double *O1,
                            const int32_t *os, double *out, int nr, int nm, int ld, double scale, int accumulate)
{
    int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= (int64_t)nm * (nr + 2)) return;
    int i = (int)(tid % (nr + 2)), k = (int)(tid / (nr + 2));
    double v = 0.0;
    if (i >= 1 && i <= nr) v += cell_partial(P0, O0, os, i - 1, nm, k);
    if (i >= 2) v += cell_partial(P1, O1, os, i - 2, nm, k);
    if (i == 0) v = 0.0;
    else if (i == 1) v = (k == 0) ? 8.0 * v : 0.0;
    else v = v * (1.0 / (double)(i - 1));
    double *o = out + (size_t)k * ld + i;
    *o = accumulate ? *o + scale * v : scale * v;
}

int launch_combine_q_rows(qpad_ctx *c, int s, const DepRows &rows, double *out, double scale, bool accumulate)
{
    int64_t n = (int64_t)c->g.nm * (c->g.nr + 2);
    hipLaunchKernelGGL(k_combine_q, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, rows.P0, rows.P1,
                       rows.O0, rows.O1, c->sp[s].ov_start, out, c->g.nr, c->g.nm, c->g.ld, scale,
                       accumulate ? 1 : 0);
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_combine_q(qpad_ctx *c, int s, double *out, double scale, bool accumulate)
{
    const Species &sp = c->sp[s];
    return launch_combine_q_rows(c, s, DepRows{sp.P0, sp.P1, sp.O0, sp.O1}, out, scale, accumulate);
}

// ---------------------------------------------------------------------------
// gather of a 3-component field at nodes ix, ix+1 (interp_part2d.f03:66-110)
// ---------------------------------------------------------------------------
// f(cc, k, n): component cc of mode array k at node ix + n (n = 0, 1); NC
// components (1: interp_field_part2d_scalar, :110-153)
template <int M, int NC, class F>
__device__ __forceinline__ void gather_n(const F &f, double w0, double w1, double pc, double ps, double out[NC])
{
#pragma unroll
    for (int cc = 0; cc < NC; cc++) {
        double v = 0.0;
        v = v + f(cc, 0, 0) * w0;
        v = v + f(cc, 0, 1) * w1;
        out[cc] = v;
    }
    double phr = 1.0, phi = 0.0;
#pragma unroll
    for (int m = 1; m <= M; m++) {
        double tr = phr * pc - phi * ps, ti = phr * ps + phi * pc;
        phr = tr;
        phi = ti;
        const double ph_re = 2.0 * phr, ph_im = 2.0 * phi;
#pragma unroll
        for (int cc = 0; cc < NC; cc++) {
            out[cc] = out[cc] + (f(cc, 2 * m - 1, 0) * ph_re - f(cc, 2 * m, 0) * ph_im) * w0;
            out[cc] = out[cc] + (f(cc, 2 * m - 1, 1) * ph_re - f(cc, 2 * m, 1) * ph_im) * w1;
        }
    }
}

// E and B at a particle from the packed fields eb[node][k][e_r, e_phi, e_z,
// b_r, b_phi, b_z] (qpad_ctx::eb), p at node ix: the six sums over (node,
// mode array) of the field times w_n times the mode's cos or -sin (doubled
// above m = 0).  `fence` runs before each node's loads of a mode.
template <int M, class P, class F>
__device__ __forceinline__ void gather_eb(P p, double w0, double w1, double pc, double ps, double ep[3], double bp[3],
                                          const F &fence)
{
    constexpr int N1 = 6 * (2 * M + 1);   // one node's values
#pragma unroll
    for (int c = 0; c < 3; c++) {
        ep[c] = p[c] * w0 + p[N1 + c] * w1;
        bp[c] = p[3 + c] * w0 + p[N1 + 3 + c] * w1;
    }
    double phr = 1.0, phi = 0.0;
#pragma unroll
    for (int m = 1; m <= M; m++) {
        const double tr = phr * pc - phi * ps, ti = phr * ps + phi * pc;
        phr = tr;
        phi = ti;
        const double re = 2.0 * phr, im = -2.0 * phi;
        const int kr = 6 * (2 * m - 1), ki = 6 * (2 * m);
#pragma unroll
        for (int n = 0; n < 2; n++) {
            const double rn = re * (n ? w1 : w0), in = im * (n ? w1 : w0);
            fence(p);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                ep[c] = ep[c] + p[n * N1 + kr + c] * rn + p[n * N1 + ki + c] * in;
                bp[c] = bp[c] + p[n * N1 + kr + 3 + c] * rn + p[n * N1 + ki + 3 + c] * in;
            }
        }
    }
}

// the packed fields through the scalar cache: a wave that works on one cell
// reads its two nodes into SGPRs (one operand of every gather FMA), which
// leaves the LDS and its bandwidth to the products
typedef const double __attribute__((address_space(4))) *uniform_ptr;

// keeps one node's values of a mode in SGPRs at a time (all would not fit)
struct UniformFence {
    __device__ __forceinline__ void operator()(uniform_ptr &p) const { __asm__ volatile("" : "+s"(p)); }
};
struct NoFence {
    template <class P>
    __device__ __forceinline__ void operator()(const P &) const {}
};

// value l = n 6 NM + 6 k + q of the packed layout, for the node pair at ix of
// the slice fields e and b themselves: what a single call (species2d%amjdp,
// species2d%push) gathers, whose e and b come from separate solves.  Packing
// them first is a launch of its own (a call, MI355X: 4096 particles in 256
// cells, amjdp 22.8 us packed, 19.1 so, push 25.0 and 21.5; 524,288 in 4096,
// M = 2, 38.1 and 32.7, 63.1 and 56.1).
template <int NM>
struct SplitFields {
    const double *e, *b;
    int nm, ld, ix;
    __device__ __forceinline__ double operator[](int l) const
    {
        const int n = l / (6 * NM), k = l / 6 % NM, q = l % 6;
        return (q < 3 ? e : b)[((size_t)(q % 3) * nm + k) * ld + ix + n];
    }
};

// nodes ix, ix + 1 of a slice field in HBM
struct NodePair {
    const double *f;
    int nm, ld, ix;
    __device__ __forceinline__ double operator()(int cc, int k, int n) const
    {
        return f[((size_t)cc * nm + k) * ld + ix + n];
    }
};

// nodes ix, ix + 1 of a slice field staged in LDS as [n][cc][k] (NC
// components)
template <int NM, int NC = 3>
struct NodePairLds {
    const double *s;
    __device__ __forceinline__ double operator()(int cc, int k, int n) const { return s[(n * NC + cc) * NM + k]; }
};

// the laser envelope (ar, ai) and its gradients (ar_grad, ai_grad: r, phi,
// z) at a particle, from nodes f(field, cc, k, n) (interp_field calls of
// part2d_class.f03:1100-1105, :1406-1409, :1996-2001)
struct LaserAt {
    double apr, api, aprg[3], apig[3];
};

template <int M, class FR, class FI, class GR, class GI>
__device__ __forceinline__ LaserAt gather_laser(const FR &far, const FI &fai, const GR &gar, const GI &gai, double w0,
                                               double w1, double pc, double ps)
{
    LaserAt l;
    gather_n<M, 1>(far, w0, w1, pc, ps, &l.apr);
    gather_n<M, 1>(fai, w0, w1, pc, ps, &l.api);
    gather_n<M, 3>(gar, w0, w1, pc, ps, l.aprg);
    gather_n<M, 3>(gai, w0, w1, pc, ps, l.apig);
    return l;
}

// ---------------------------------------------------------------------------
// amjdeposit_robust_part2d (part2d_class.f03:746-1010): gather E, B; robust
// predictor on a copy of the momentum; deposit cu (3), acu (2), amu (3) per
// mode.  Value index v = comp * NM + k, comp 0..2 cu, 3..4 acu, 5..7 amu.
// ---------------------------------------------------------------------------
struct JDepArgs {
    int nr, ld, nm;
    double idr, qbm, qtmh, idt;
    const double *x1, *x2, *p1, *p2, *p3, *q;
    double *gamma, *psi;
    int store_diag;
    const int32_t *cs;
    const double *eb;   // the packed E and B of the slice (qpad_ctx::eb)
    const double *e, *b;   // the slice fields (single calls)
    // the laser envelope and its gradients of the slice (PGC pushers)
    const double *ar, *ai, *arg, *aig;
    double *P0, *P1;
    IterState *it;
    // SPEC launches: convergence of the previous iteration from the field
    // kernel's per-workgroup maxima
    const double *conv_prev;
    int nblk;
    double reltol, abstol;
    // host-visible copy of the decision (done, iterations so far) written by
    // workgroup 0 of a SPEC launch, or null
    IterState *report;
    // the crowded cells' chunks (listed by the sort) and the overflow rows
    const int32_t *os;
    const int4 *desc;
    double *O0, *O1;
    int first, n_crowd_max;
};

// What one particle deposits (robust predictor, part2d_class.f03:877-960):
// the eight deposited quantities val[comp] (cu 0..2, dcu 3..4, amu 5..7),
// the linear weights w[n] of nodes ix + n and the mode phases of mode array
// k times q / (gamma - u_z), ph[k].  Value v = n * 8NM + comp * NM + k of
// the cell's deposit is the sum over its particles of
// w[n] ph[k] val[comp].
template <int M>
struct PartTerms {
    double val[8];
    double w[2];
    double ph[2 * M + 1];
};

// the laser values a PGC deposit workgroup stages in LDS per wave: ar, ai
// ([n][k]) and ar_grad, ai_grad ([n][cc][k])
template <int NM, bool PGC>
constexpr int dep_staged() { return PGC ? 16 * NM : 1; }

// staged value l of the cell whose left node is ix
template <int NM>
__device__ __forceinline__ double dep_stage_load_pgc(const double *ar, const double *ai, const double *arg,
                                                     const double *aig, int nm, int ld, int l, int ix)
{
    const double *f;
    int nc, base;
    if (l < 4 * NM) {
        f = l < 2 * NM ? ar : ai;
        nc = 1;
        base = l < 2 * NM ? 0 : 2 * NM;
    } else {
        f = l < 10 * NM ? arg : aig;
        nc = 3;
        base = l < 10 * NM ? 4 * NM : 10 * NM;
    }
    const int r = l - base, n = r / (nc * NM), comp = (r / NM) % nc, k = r % NM;
    return f[((size_t)comp * nm + k) * ld + ix + n];
}

// gather and predictor of particle p of cell c; lanes past the chunk's end
// (valid false) deposit zero and store nothing.  STD: the standard pusher
// (amjdeposit_std_part2d, part2d_class.f03:478-744), which normalises by the
// particle's interpolated psi (psip) where the robust one uses gamma - u_z,
// and always stores the time-centred gamma.  PGC: the laser pushers
// (amjdeposit_std_pgc_part2d :1012-1308, amjdeposit_robust_pgc_part2d
// :1310-1602): every gamma carries gam_corr = (q/m)^2 |a|^2 / 2, the
// electric field the ponderomotive term -+ (q/m)/(2 gamma) a grad a
// (r, phi minus, z plus, with the initial gamma), and the robust form
// normalises its second half kick by gamma / (gamma - u_z) of the rotated
// momentum.  eb: the packed fields at the cell's left node; sf: the wave's
// staged laser values (PGC).
template <int M, bool STD, bool PGC, class P, class F>
__device__ __forceinline__ void particle_terms(const JDepArgs &a, P eb, const F &fence, const double *sf, int c, int p,
                                               bool valid,
                                               double x1, double x2, double pp1, double pp2, double pp3, double qp,
                                               double psip, PartTerms<M> &t)
{
    constexpr int NM = 2 * M + 1;
    double r = radius(x1, x2);
    const double pc = x1 / r, ps = x2 / r;
    double pos = __dmul_rn(r, a.idr);
    const double w1 = pos - (double)c, w0 = 1.0 - w1;
    double ep[3], bp[3];
    gather_eb<M>(eb, w0, w1, pc, ps, ep, bp, fence);
    double gam_corr = 0.0;
    LaserAt la;
    if constexpr (PGC) {
        la = gather_laser<M>(NodePairLds<NM, 1>{sf}, NodePairLds<NM, 1>{sf + 2 * NM}, NodePairLds<NM>{sf + 4 * NM},
                             NodePairLds<NM>{sf + 10 * NM}, w0, w1, pc, ps);
        gam_corr = 0.5 * a.qbm * a.qbm * (la.apr * la.apr + la.api * la.api);
    }
    // sqrt(1 + v^2) (+ gam_corr for the laser pushers)
    auto gamma_of = [&](const double *v) {
        double g2 = 1.0 + v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
        if constexpr (PGC) g2 = g2 + gam_corr;
        return sqrt(g2);
    };
    double wp0 = ep[0] - bp[1], wp1 = ep[1] + bp[0], wp2 = ep[2];
    double u0[3] = {pp1 * pc + pp2 * ps, pp2 * pc - pp1 * ps, pp3};
    double gam = gamma_of(u0);
    if constexpr (PGC) {
        const double tmp = 0.5 * a.qbm / gam;
        ep[0] = ep[0] - tmp * (la.apr * la.aprg[0] + la.api * la.apig[0]);
        ep[1] = ep[1] - tmp * (la.apr * la.aprg[1] + la.api * la.apig[1]);
        ep[2] = ep[2] + tmp * (la.apr * la.aprg[2] + la.api * la.apig[2]);
    }
    double ut[3], u[3];
    double qtmh2;
    if constexpr (STD) {
        qtmh2 = a.qtmh / (1.0 - a.qbm * psip);
        const double qtmh1 = qtmh2 * gam;
#pragma unroll
        for (int cc = 0; cc < 3; cc++) ut[cc] = u0[cc] + ep[cc] * qtmh1;
    } else if constexpr (PGC) {
        const double qtmh1 = a.qtmh * gam / (gam - u0[2]);
#pragma unroll
        for (int cc = 0; cc < 3; cc++) ut[cc] = u0[cc] + ep[cc] * qtmh1;
        gam = gamma_of(ut);
        qtmh2 = a.qtmh / (gam - ut[2]);
    } else {
        const double qtmh1 = a.qtmh * gam / (gam - u0[2]);
#pragma unroll
        for (int cc = 0; cc < 3; cc++) { ep[cc] = ep[cc] * qtmh1; ut[cc] = u0[cc] + ep[cc]; }
        gam = sqrt(1.0 + ut[0] * ut[0] + ut[1] * ut[1] + ut[2] * ut[2]);
        qtmh2 = a.qtmh / (gam - ut[2]);
    }
#pragma unroll
    for (int cc = 0; cc < 3; cc++) bp[cc] = bp[cc] * qtmh2;
    u[0] = ut[0] + ut[1] * bp[2] - ut[2] * bp[1];
    u[1] = ut[1] + ut[2] * bp[0] - ut[0] * bp[2];
    u[2] = ut[2] + ut[0] * bp[1] - ut[1] * bp[0];
    double ostq = 2.0 / (1.0 + bp[0] * bp[0] + bp[1] * bp[1] + bp[2] * bp[2]);
#pragma unroll
    for (int cc = 0; cc < 3; cc++) bp[cc] = bp[cc] * ostq;
    ut[0] = ut[0] + u[1] * bp[2] - u[2] * bp[1];
    ut[1] = ut[1] + u[2] * bp[0] - u[0] * bp[2];
    ut[2] = ut[2] + u[0] * bp[1] - u[1] * bp[0];
    if constexpr (STD) {
        // second half kick normalised by the gamma after the rotation
        const double qtmh1 = qtmh2 * gamma_of(ut);
#pragma unroll
        for (int cc = 0; cc < 3; cc++) u[cc] = ut[cc] + ep[cc] * qtmh1;
    } else if constexpr (PGC) {
        const double g1 = gamma_of(ut);
        const double qtmh1 = a.qtmh * g1 / (g1 - ut[2]);
#pragma unroll
        for (int cc = 0; cc < 3; cc++) u[cc] = ut[cc] + ep[cc] * qtmh1;
    } else {
#pragma unroll
        for (int cc = 0; cc < 3; cc++) u[cc] = ut[cc] + ep[cc];
    }
    double du0 = a.idt * (u[0] - u0[0]), du1 = a.idt * (u[1] - u0[1]);
#pragma unroll
    for (int cc = 0; cc < 3; cc++) u[cc] = 0.5 * (u[cc] + u0[cc]);
    double g2 = gamma_of(u);
    double ipsi;
    if constexpr (STD) {
        ipsi = 1.0 / (1.0 - a.qbm * psip);
        if (valid) a.gamma[p] = g2;
    } else {
        ipsi = 1.0 / (g2 - u[2]);
        if (a.store_diag && valid) {
            a.gamma[p] = g2;
            a.psi[p] = (1.0 - 1.0 / ipsi) / a.qbm;
        }
    }
    double dpsi = a.qbm * (wp2 - (wp0 * u[0] + wp1 * u[1]) * ipsi);
    du0 = du0 + u[0] * dpsi * ipsi;
    du1 = du1 + u[1] * dpsi * ipsi;
    t.val[0] = u[0];
    t.val[1] = u[1];
    t.val[2] = u[2];
    t.val[3] = du0;
    t.val[4] = du1;
    t.val[5] = u[0] * u[0] * ipsi;
    t.val[6] = u[0] * u[1] * ipsi;
    t.val[7] = u[1] * u[1] * ipsi;
    double phr = 1.0 * (valid ? qp : 0.0) * ipsi, phi = 0.0;
    t.w[0] = w0;
    t.w[1] = w1;
    t.ph[0] = phr;
    const double ph0r = pc, ph0i = -ps;
#pragma unroll
    for (int m = 1; m <= M; m++) {
        double tr = phr * ph0r - phi * ph0i, ti = phr * ph0i + phi * ph0r;
        phr = tr;
        phi = ti;
        t.ph[2 * m - 1] = phr;
        t.ph[2 * m] = phi;
    }
}

// The matrix form of a wave's cell deposit: the cell's values are the
// 16 x NM product D[n * 8 + comp][k] = sum_p (w[n] val[comp])_p ph[k]_p, a
// GEMM with the particles as the inner dimension, which
// v_mfma_f64_16x16x4f64 accumulates four particles at a time (FP64 on the
// matrix cores; no cross-lane reduction and four accumulators per lane
// instead of 16 NM).  Operand layout of the instruction: lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] and holds D[4 r + l / 16][l % 16]
// in its accumulator r.  The pass's particle terms reach that layout
// through the wave's own LDS rows ([particle][A 0..15, ph 0..NM-1, 0],
// stride mf_stride; lanes past the NM columns read the zero), one half-wave
// of 32 particles at a time; each half's operands are read before its eight
// instructions are issued.
typedef double dep_acc4 __attribute__((ext_vector_type(4)));

template <int NM>
constexpr int mf_stride() { return (17 + NM) | 1; }

// LDS writes of this wave visible to its other lanes (waves of a workgroup
// run different pass counts, so no workgroup barrier here)
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// one accumulator chain per wave: independent chains (summed at the end)
// would overlap the instruction's latency, but their registers cost a wave
// per SIMD, which measured slower on MI355X (C2: 25.7 against 27.5 us with
// four chains, C3: 23.7 against 18.6 us)
template <int M>
__device__ __forceinline__ void mf_accumulate(double *rows, const PartTerms<M> &t, int lane, dep_acc4 &acc)
{
    constexpr int NM = 2 * M + 1, STR = mf_stride<NM>();
    const int gi = lane >> 4, i = lane & 15;
    const int fb = 16 + min(i, NM);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if ((lane >> 5) == h) {
            double *mine = rows + (lane & 31) * STR;
#pragma unroll
            for (int n = 0; n < 2; n++)
#pragma unroll
                for (int c = 0; c < 8; c++) mine[n * 8 + c] = t.w[n] * t.val[c];
#pragma unroll
            for (int k = 0; k < NM; k++) mine[16 + k] = t.ph[k];
            mine[16 + NM] = 0.0;
        }
        wave_lds_sync();
        double av[8], bv[8];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const double *r = rows + (4 * s + gi) * STR;
            av[s] = r[i];
            bv[s] = r[fb];
        }
#pragma unroll
        for (int s = 0; s < 8; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], bv[s], acc, 0, 0, 0);
        // all sixteen reads ahead of the eight instructions
        __builtin_amdgcn_sched_group_barrier(0x0100, 16, 0);
        __builtin_amdgcn_sched_group_barrier(0x0008, 8, 0);
        wave_lds_sync();
    }
}

// The vector form of a wave's cell deposit: the same 16 x NM product as
// outer-product tiles.  Each lane writes its particle's terms into the wave's
// LDS rows ([val 0..7][ph 0..NM-1][w1], stride tile_stride); then lane
// (g, q) = (lane / 4, lane % 4) reads the particles 16 j + g and adds the
// 4 x NM products of tile q (both nodes, components 2q and 2q + 1) into its
// own accumulators.  A lane so keeps 4 NM accumulators where a lane that
// summed whole particles kept 16 NM, and the cross-lane sum at the end
// exchanges 5 NM values instead of 17 NM.  Row groups past the pass's last
// particle are skipped.
template <int M>
constexpr int tile_stride()
{
    // even (16-byte reads) and = 2 mod 4 doubles, which spreads the rows over the LDS banks
    return (10 + 2 * M) % 4 == 2 ? 10 + 2 * M : 12 + 2 * M;
}

template <int M>
__device__ __forceinline__ void tile_accumulate(double *rows, const PartTerms<M> &t, int lane, int ngroups,
                                                double (&acc)[4 * (2 * M + 1)])
{
    constexpr int NM = 2 * M + 1, STR = tile_stride<M>();
    double2 *mine = reinterpret_cast<double2 *>(rows + lane * STR);
#pragma unroll
    for (int c = 0; c < 4; c++) mine[c] = make_double2(t.val[2 * c], t.val[2 * c + 1]);
#pragma unroll
    for (int k = 0; k <= M; k++) mine[4 + k] = make_double2(t.ph[2 * k], 2 * k + 1 < NM ? t.ph[2 * k + 1] : t.w[1]);
    wave_lds_sync();
    const int g = lane >> 2, q = lane & 3;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (j >= ngroups) break;
        const double2 *r = reinterpret_cast<const double2 *>(rows + (16 * j + g) * STR);
        const double2 v = r[q];
        double ph[NM + 1];
#pragma unroll
        for (int k = 0; k <= M; k++) {
            const double2 x = r[4 + k];
            ph[2 * k] = x.x;
            ph[2 * k + 1] = x.y;
        }
        const double w1 = ph[NM], w0 = 1.0 - w1;
        const double av[4] = {w0 * v.x, w0 * v.y, w1 * v.x, w1 * v.y};
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
            for (int k = 0; k < NM; k++) acc[x * NM + k] += av[x] * ph[k];
    }
    wave_lds_sync();
}

// the 16 lane groups' tiles summed: row r of 16 lanes keeps the NM values of
// node r / 2 and component 2 q + r % 2 (q = lane % 4), in acc[0 .. NM)
template <int M>
__device__ __forceinline__ void tile_reduce(double (&acc)[4 * (2 * M + 1)])
{
    constexpr int NM = 2 * M + 1;
#pragma unroll
    for (int i = 0; i < 2 * NM; i++) acc[i] = swap32_sum(acc[i], acc[2 * NM + i]);
#pragma unroll
    for (int i = 0; i < NM; i++) {
        acc[i] = swap16_sum(acc[i], acc[NM + i]);
        acc[i] = acc[i] + dpp<kDppRowRor8>(acc[i]);
        acc[i] = acc[i] + dpp<kDppRowRor4>(acc[i]);
    }
}

// the arguments of every species of one launch; workgroup row blockIdx.y
// deposits species blockIdx.y
struct JDepMulti {
    JDepArgs s[kMaxSpecies];
};

// waves per SIMD the compiler is asked to fit, without a spill: modes 0..1 of
// the vector form take 92..128 VGPRs, modes 0..2 136.  Forced under 128, modes
// 0..2 spill 6..12 VGPRs, and four waves give what the spills take: 524,288
// particles in 4096 cells, first / later iterations, 20.4 / 14.8 us, with
// three 19.9 / 15.0; 2^20 in 8192 29.7 / 23.2 and 29.0 / 23.2.
template <int M, bool PGC, bool MF, bool SINGLE>
constexpr int dep_min_waves() { return !MF && !PGC ? (M <= 1 ? 4 : M >= 3 && SINGLE ? 2 : 3) : 1; }

// The current deposit's launch is bound by its longest wave and by the FP64
// issue rate (420 FP64 instructions per 64 particles at modes 0..2), not by
// its 48 B per particle.  MI355X, averages over the slices of a 3D step
// through the driver and the first bubble (rocprofv3), first / later
// iterations: 524,288 particles, 4096 cells, modes 0..2: 25.5 / 19.7 us with
// 16 NM accumulators per lane, fields broadcast from LDS and one wave per
// 1024-particle chunk, 20.0 / 14.6 us in this form; 2 x 131,072 particles,
// 2048 cells, modes 0..4 (matrix form): 22.4 / 17.3 and 16.3 / 13.0 us.
//
// SPEC: a speculative launch of iteration >= 2 of a slice, which returns at
// once when the iteration has already converged (a separate instance, so
// that profiles show the first-iteration launches, which always work, apart)
// MF: the matrix form of the accumulation (mf_accumulate) instead of the
// vector form (tile_accumulate); the same values up to the order of the sums
// SINGLE: species2d%amjdp, whose fields are staged in LDS from e and b
// (SplitFields) in the packed layout
template <int M, bool SPEC, int CPW, bool STD, bool PGC = false, bool MF = false, bool SINGLE = false>
__global__ __launch_bounds__(64 * CPW, (dep_min_waves<M, PGC, MF, SINGLE>())) void k_amjdeposit(const JDepMulti m)
{
    const JDepArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    constexpr int NM = 2 * M + 1;
    constexpr int NV = 8 * NM;
    constexpr int NF = dep_staged<NM, PGC>();   // staged field values per cell
    constexpr int CH = crowd_chunks<CPW>(), PT = crowd_parts<CPW>();
    constexpr int NE = SINGLE ? 12 * NM : 1;
    __shared__ double fe[CPW][NE];   // E and B at the two nodes (SINGLE)
    // the laser fields at the two nodes of each wave's cell (PGC)
    __shared__ double sf[CPW][NF];
    // the particle rows of the wave's products, per wave
    constexpr int ROWS = MF ? 32 * mf_stride<NM>() : 64 * tile_stride<M>();
    __shared__ __align__(16) double mrows[CPW * ROWS];
    // the part sums of crowded chunks
    __shared__ double comb[CH][kDepSub][2 * NV];
    static_assert(sizeof(double) * (CPW * (NE + NF + ROWS) + CH * kDepSub * 2 * NV) <= 160 * 1024, "LDS of a CU");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nm = a.nm, ld = a.ld;
    const int ncg = (a.nr + CPW - 1) / CPW;
    const bool crowd = (int)blockIdx.x >= ncg;
    const int ncrowd = crowd ? min(a.os[a.nr + 1], a.n_crowd_max) : 0;
    const int step = ((int)gridDim.x - ncg) * CH;
    int o0 = ((int)blockIdx.x - ncg) * CH;
    if (crowd && o0 >= ncrowd) return;
    // every independent load of the prologue first (one round trip): the
    // convergence state and the cell's particle range (and laser values)
    int done = 0;
    double co = 0.0, cd = 0.0;
    int iters_now = 0;
    if (SPEC) {
        done = a.it->done;
        iters_now = a.it->iters;
        conv_load(a.conv_prev, a.nblk, co, cd);
    }
    bool live = true;
    DepRange rg;
    int4 d = make_int4(0, 0, 0, 0);
    const int ch = wave / (CPW / CH);
    if (!crowd) {
        rg = cell_range<CPW>(a.nr, a.cs, a.first, wave, live);
    } else {
        d = crowd_entry(a.desc, min(o0 + ch, ncrowd - 1));
        rg.cell = d.x;
    }
    uniform_ptr eb;
    double fv[(NF + 63) / 64], ev[(NE + 63) / 64];
    auto load_fields = [&](int c) {
        eb = (uniform_ptr)(a.eb + (size_t)(c + 1) * (6 * NM));
        if constexpr (SINGLE) {
#pragma unroll
            for (int u = 0; u < (NE + 63) / 64; u++)
                ev[u] = SplitFields<NM>{a.e, a.b, nm, ld, c + 1}[min(lane + 64 * u, NE - 1)];
        }
        if constexpr (PGC) {
#pragma unroll
            for (int u = 0; u < (NF + 63) / 64; u++)
                fv[u] = dep_stage_load_pgc<NM>(a.ar, a.ai, a.arg, a.aig, nm, ld, min(lane + 64 * u, NF - 1), c + 1);
        }
    };
    load_fields(rg.cell);
    if (SPEC) {
        int stop = done;
        if (!stop) {
            // 'compare' of the previous iteration (simulation_class.f03:396):
            // every wave evaluates it (the same decision everywhere);
            // workgroup 0 records it
            double rel, ab;
            conv_finish(co, cd, rel, ab);
            stop = rel < a.reltol || ab < a.abstol;
            if (stop && blockIdx.x == 0 && threadIdx.x == 0) a.it->done = 1;
        }
        if (a.report && blockIdx.x == 0 && threadIdx.x == 0) {
            a.report->done = stop;
            a.report->iters = iters_now;
        }
        if (stop) return;
    }
    if (!live) return;
    const double *__restrict__ X1 = a.x1;
    const double *__restrict__ X2 = a.x2;
    const double *__restrict__ PP1 = a.p1;
    const double *__restrict__ PP2 = a.p2;
    const double *__restrict__ PP3 = a.p3;
    const double *__restrict__ Q = a.q;
    double acc[4 * NM];
    dep_acc4 macc;
    double *const wrows = mrows + wave * ROWS;
    auto stage_fields = [&]() {
        if constexpr (SINGLE) {
#pragma unroll
            for (int u = 0; u < (NE + 63) / 64; u++)
                if (lane + 64 * u < NE) fe[wave][lane + 64 * u] = ev[u];
        }
        if constexpr (PGC) {
#pragma unroll
            for (int u = 0; u < (NF + 63) / 64; u++) {
                const int l = lane + 64 * u;
                if (l < NF) sf[wave][l] = fv[u];
            }
        }
        if constexpr (SINGLE || PGC) wave_lds_sync();
    };
    // the wave's sums, value comp * NM + k of node ix to D0 and of node ix + 1 to D1
    auto store = [&](double *D0, double *D1) {
        if constexpr (MF) {
            // lane l holds D[4 r + l / 16][l % 16]: row = node * 8 + comp, column = mode array
            const int k = lane & 15, rb = lane >> 4;
            if (k < NM) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = 4 * r + rb;
                    (row < 8 ? D0 : D1)[(row & 7) * NM + k] = macc[r];
                }
            }
        } else {
            const int r = lane >> 4, comp = 2 * (lane & 3) + (r & 1), sub = (lane >> 2) & 3;
            double *D = (r < 2 ? D0 : D1) + comp * NM;
#pragma unroll
            for (int k = 0; k < NM; k++)
                if ((k & 3) == sub) D[k] = acc[k];
        }
    };
    stage_fields();
    const int sub0 = (wave % (CPW / CH)) * PT;
    int u = 0;
    if (crowd) rg = part_range(d, sub0, o0 + ch < ncrowd);
    for (;;) {
        // the wave's sums over the particles of the range
        const int c = rg.cell, p0 = rg.pb, p1 = rg.pe;
#pragma unroll
        for (int v = 0; v < 4 * NM; v++) acc[v] = 0.0;
        macc = dep_acc4{0.0, 0.0, 0.0, 0.0};
        // every pass has all 64 lanes active (the exchanges need them); lanes
        // past the range's end deposit zero.  Software-pipelined: the next
        // pass's particle loads are in flight while this pass computes.
        const int npass = __builtin_amdgcn_readfirstlane((p1 - p0 + 63) >> 6);
        const int pl = max(p1 - 1, 0);
        int p = p0 + lane;
        int pc = min(p, pl);
        double x1 = X1[pc], x2 = X2[pc], pp1 = PP1[pc], pp2 = PP2[pc], pp3 = PP3[pc], qp = Q[pc];
        double psip = STD ? a.psi[pc] : 0.0;
        for (int k = 0; k < npass; k++, p += 64) {
            // the fields are read anew for every pass (scalar cache or LDS)
            // rather than held in registers
            if constexpr (SINGLE) __asm__ volatile("" ::: "memory");
            else UniformFence()(eb);
            const int pn = min(p + 64, pl);
            const double nx1 = X1[pn], nx2 = X2[pn], np1 = PP1[pn], np2 = PP2[pn], np3 = PP3[pn], nq = Q[pn];
            const double npsi = STD ? a.psi[pn] : 0.0;
            PartTerms<M> pt;
            if constexpr (SINGLE) {
                particle_terms<M, STD, PGC>(a, (const double *)fe[wave], NoFence(), sf[wave], c, p, p < p1, x1, x2, pp1,
                                            pp2, pp3, qp, psip, pt);
            } else {
                particle_terms<M, STD, PGC>(a, eb, UniformFence(), sf[wave], c, p, p < p1, x1, x2, pp1, pp2, pp3, qp,
                                            psip, pt);
            }
            if constexpr (MF) {
                mf_accumulate<M>(wrows, pt, lane, macc);
            } else {
                const int left = p1 - p0 - 64 * k;
                tile_accumulate<M>(wrows, pt, lane, __builtin_amdgcn_readfirstlane((min(left, 64) + 15) >> 4), acc);
            }
            x1 = nx1; x2 = nx2; pp1 = np1; pp2 = np2; pp3 = np3; qp = nq; psip = npsi;
        }
        if constexpr (!MF) tile_reduce<M>(acc);
        if (!crowd) {
            store(a.P0 + (size_t)c * NV, a.P1 + (size_t)c * NV);
            return;
        }
        store(comb[ch][sub0 + u], comb[ch][sub0 + u] + NV);
        if (++u < PT) {
            rg = part_range(d, sub0 + u, o0 + ch < ncrowd);
            continue;
        }
        u = 0;
        __syncthreads();
        for (int t = threadIdx.x; t < CH * 2 * NV; t += 64 * CPW) {
            const int q = t / (2 * NV), v = t % (2 * NV);
            if (o0 + q >= ncrowd) continue;
            const int4 e = a.desc[o0 + q];
            const double sum = ((comb[q][0][v] + comb[q][1][v]) + comb[q][2][v]) + comb[q][3][v];
            double *D = e.w < 0 ? (v < NV ? a.P0 : a.P1) + (size_t)e.x * NV : (v < NV ? a.O0 : a.O1) + (size_t)e.w * NV;
            D[v < NV ? v : v - NV] = sum;
        }
        o0 += step;
        if (o0 >= ncrowd) return;
        __syncthreads();
        d = crowd_entry(a.desc, min(o0 + ch, ncrowd - 1));
        load_fields(d.x);
        stage_fields();
        rg = part_range(d, sub0, o0 + ch < ncrowd);
    }
}

void time_begin(qpad_ctx *c, int which, hipEvent_t *stop);
void time_end(qpad_ctx *c, int which, hipEvent_t stop);

static JDepArgs jdep_args(qpad_ctx *c, int s, int l, bool store_diag, bool report)
{
    const bool speculative = l >= 2;
    Species &sp = c->sp[s];
    JDepArgs a;
    a.nr = c->g.nr;
    a.ld = c->g.ld;
    a.nm = c->g.nm;
    a.idr = 1.0 / c->g.dr;
    a.qbm = sp.qbm;
    a.qtmh = 0.5 * sp.qbm * c->dt2d;
    a.idt = 1.0 / c->dt2d;
    a.x1 = sp.x1; a.x2 = sp.x2; a.p1 = sp.p1; a.p2 = sp.p2; a.p3 = sp.p3; a.q = sp.q;
    a.gamma = sp.gamma;
    a.psi = sp.psi;
    a.store_diag = store_diag;
    a.cs = sp.cell_start;
    a.eb = c->eb;
    a.e = c->f[QPAD_F_E];
    a.b = c->f[QPAD_F_B];
    a.ar = c->f[QPAD_F_AR];
    a.ai = c->f[QPAD_F_AI];
    a.arg = c->f[QPAD_F_AR_GRAD];
    a.aig = c->f[QPAD_F_AI_GRAD];
    a.P0 = sp.P0;
    a.P1 = sp.P1;
    a.it = c->it;
    a.nblk = conv_blocks(c->g.nr);
    a.conv_prev = c->conv_blk + (size_t)((l - 1) & 1) * 2 * a.nblk;
    a.reltol = c->g.reltol;
    a.abstol = c->g.abstol;
    a.report = (report && speculative) ? c->it_report : nullptr;
    a.os = sp.ov_start;
    a.desc = sp.ov_desc;
    a.O0 = sp.O0;
    a.O1 = sp.O1;
    a.first = sp.dep_first;
    a.n_crowd_max = sp.n_crowd_max;
    return a;
}

// the species of species-list entries in one launch (grid rows by list
// entry), all of the push type STD, PGC names; l: the iteration, 0 a single
// call (one workgroup shape: no result depends on it)
template <bool STD, bool PGC>
static int launch_jdep_list(qpad_ctx *c, const int *list, int n, int l, bool store_diag, bool timed, bool report)
{
    const bool speculative = l >= 2;
    JDepMulti m;
    memset(&m, 0, sizeof(m));
    const bool single = l == 0;
    const int cpw = single ? kDepWaves : c->dep_cells;
    int gx = 1;
    for (int i = 0; i < n; i++) {
        const int s = list[i];
        // the report (the host's copy of the decision) from the first entry only
        m.s[i] = jdep_args(c, s, l, store_diag, report && i == 0);
        gx = std::max(gx, dep_grid(c->g.nr, c->sp[s].npp, c->sp[s].dep_first, cpw));
    }
    dim3 grid((unsigned)gx, (unsigned)n), blk(64 * cpw);
    hipEvent_t stop = nullptr;
    if (timed) time_begin(c, 0, &stop);
    const bool mf = c->dep_mfma != 0;
#define QPAD_DEP3(MM, CC, MFV)                                                                                \
    do {                                                                                                      \
        if (speculative)                                                                                      \
            hipLaunchKernelGGL((k_amjdeposit<MM, true, CC, STD, PGC, MFV>), grid, blk, 0, c->stream, m);       \
        else hipLaunchKernelGGL((k_amjdeposit<MM, false, CC, STD, PGC, MFV>), grid, blk, 0, c->stream, m);     \
    } while (0)
#define QPAD_DEP2(MM, CC)                    \
    do {                                     \
        if (mf) QPAD_DEP3(MM, CC, true);     \
        else QPAD_DEP3(MM, CC, false);       \
    } while (0)
#define QPAD_DEP(MM)                                 \
    do {                                             \
        if (single) {                                                                                              \
            if (mf) hipLaunchKernelGGL((k_amjdeposit<MM, false, kDepWaves, STD, PGC, true, true>), grid, blk, 0, c->stream, m); \
            else hipLaunchKernelGGL((k_amjdeposit<MM, false, kDepWaves, STD, PGC, false, true>), grid, blk, 0, c->stream, m);   \
        } else if (cpw == 2) QPAD_DEP2(MM, 2);       \
        else if (cpw == 8) QPAD_DEP2(MM, 8);         \
        else QPAD_DEP2(MM, 4);                       \
    } while (0)
    switch (c->g.M) {
    case 0: QPAD_DEP(0); break;
    case 1: QPAD_DEP(1); break;
    case 2: QPAD_DEP(2); break;
    case 3: QPAD_DEP(3); break;
    default: QPAD_DEP(4); break;
    }
#undef QPAD_DEP
#undef QPAD_DEP2
#undef QPAD_DEP3
    QPAD_HIP_CHECK(hipGetLastError());
    if (timed) time_end(c, 0, stop);
    return 0;
}

// the four pushers in launch order: robust, standard, robust_pgc,
// standard_pgc
static int push_group(int push_type)
{
    switch (push_type) {
    case QPAD_PUSH2_STD: return 1;
    case QPAD_PUSH2_ROBUST_PGC: return 2;
    case QPAD_PUSH2_STD_PGC: return 3;
    default: return 0;
    }
}

// species s0 .. s1-1: one launch per push type present (the first launch
// carries the timing and the host report when there is one)
static int launch_jdep(qpad_ctx *c, int s0, int s1, int l, bool store_diag, bool timed, bool report)
{
    int list[4][kMaxSpecies], n[4] = {0, 0, 0, 0};
    for (int s = s0; s < s1; s++) {
        const int g = push_group(c->sp[s].cfg.push_type);
        list[g][n[g]++] = s;
    }
    bool first = true;
    int rc = 0;
    for (int g = 0; g < 4 && !rc; g++) {
        if (!n[g]) continue;
        const bool tm = timed && first, rp = report && first;
        if (g == 0) rc = launch_jdep_list<false, false>(c, list[g], n[g], l, store_diag, tm, rp);
        else if (g == 1) rc = launch_jdep_list<true, false>(c, list[g], n[g], l, store_diag, tm, rp);
        else if (g == 2) rc = launch_jdep_list<false, true>(c, list[g], n[g], l, store_diag, tm, rp);
        else rc = launch_jdep_list<true, true>(c, list[g], n[g], l, store_diag, tm, rp);
        first = false;
    }
    return rc;
}

int launch_amjdeposit(qpad_ctx *c, int s, int l, bool store_diag, bool timed, bool report)
{
    return launch_jdep(c, s, s + 1, l, store_diag, timed, report);
}

int launch_amjdeposit_all(qpad_ctx *c, int l, bool store_diag, bool timed, bool report)
{
    if (c->nspecies == 0) return 0;
    return launch_jdep(c, 0, c->nspecies, l, store_diag, timed, report);
}

// ---------------------------------------------------------------------------
// push_u_robust (part2d_class.f03:1879-1965) + push_x (:2221-2262) + the
// re-sort by the new cells (update_bound :2307-2353 is the key nr).
// Particles that already left the box (past cell_start[nr]) keep key nr.
// The push is in place, a thread per particle, and the key is the cell of the
// position it stores.  Two forms, by the form of the sort (sort_form):
// - few particles (direct): the push launch also counts its chunk's keys
//   (k_push_count) and the scattering pass follows, two launches whose
//   latencies are all that counts.  MI355X, kernel trace, push + re-sort of a
//   slice: 4096 particles in 256 cells 5.8 + 5.9 us, 21189 in 1009 cells 6.1 +
//   9.4; with a second push in the scattering pass instead of the stores here
//   5.1 + 7.1 and 6.0 + 10.5 us.
// - many: k_push, then the plain sort's passes; the direct form's sum of every
//   chunk's counts in each workgroup ends there.
// ---------------------------------------------------------------------------
struct PushArgs {
    int nr, ld, nm;
    double idr, edge, qtmh, dt, qbm;
    double clamp;        // expansion-factor clamp of a sub-cycled push (0: none)
    const double *eb;    // the packed E and B of the slice
    const double *e, *b; // the slice fields (single calls)
    const double *ar, *ai, *arg, *aig;   // laser envelope and gradients (PGC)
    double *x1, *x2, *p1, *p2, *p3, *gamma;   // pushed in place
    const double *psi;   // interpolated psi (standard pusher)
    SortArgs s;
};

constexpr int kPushThreads = 256;

// the arguments of every species of one launch (workgroup rows by species)
struct PushMulti {
    PushArgs s[kMaxSpecies];
    int n;       // species; workgroup row n is the slice's epilogue
    EpiArgs epi;
};

// STD: push_u_std_part2d (part2d_class.f03:1790-1877), normalised by the
// interpolated psi and the gamma the last current deposit stored, where
// push_u_robust_part2d (:1879-1965) uses the particle's own gamma - p_z.
// PGC: push_u_robust_pgc_part2d / push_u_std_pgc_part2d (:1967-2219, the
// same steps): the standard normalisation, the ponderomotive term in E with
// the stored gamma, and the new gamma with gam_corr extrapolated half a step
// in xi (the envelope's xi gradient).  Returns the new cell.
// SINGLE: the fields from e and b (species2d%push, SplitFields).
template <int M, bool STD, bool PGC, bool SINGLE>
__device__ __forceinline__ uint32_t push_particle(const PushArgs &a, int64_t p)
{
    const int nm = a.nm, ld = a.ld;
    double x1 = a.x1[p], x2 = a.x2[p];
    double r = radius(x1, x2);
    const double pc = x1 / r, ps = x2 / r;
    double pos = __dmul_rn(r, a.idr);
    if (!(pos >= 0.0)) pos = 0.0;   // r = 0 or NaN: keep the gather in bounds
    int ic = (int)fmin(pos, (double)(a.nr - 1));
    const int ix = ic + 1;
    const double w1 = pos - (double)ic, w0 = 1.0 - w1;
    double ep[3], bp[3];
    if constexpr (SINGLE)
        gather_eb<M>(SplitFields<2 * M + 1>{a.e, a.b, nm, ld, ix}, w0, w1, pc, ps, ep, bp, NoFence());
    else
        gather_eb<M>(a.eb + (size_t)ix * (6 * (2 * M + 1)), w0, w1, pc, ps, ep, bp, NoFence());
    double t = ep[0] * pc - ep[1] * ps;
    ep[1] = ep[0] * ps + ep[1] * pc;
    ep[0] = t;
    t = bp[0] * pc - bp[1] * ps;
    bp[1] = bp[0] * ps + bp[1] * pc;
    bp[0] = t;
    double gam_corr = 0.0, apr_z = 0.0, api_z = 0.0, apr = 0.0, api = 0.0;
    if constexpr (PGC) {
        LaserAt la = gather_laser<M>(NodePair{a.ar, nm, ld, ix}, NodePair{a.ai, nm, ld, ix},
                                     NodePair{a.arg, nm, ld, ix}, NodePair{a.aig, nm, ld, ix}, w0, w1, pc, ps);
        t = la.aprg[0] * pc - la.aprg[1] * ps;
        la.aprg[1] = la.aprg[0] * ps + la.aprg[1] * pc;
        la.aprg[0] = t;
        t = la.apig[0] * pc - la.apig[1] * ps;
        la.apig[1] = la.apig[0] * ps + la.apig[1] * pc;
        la.apig[0] = t;
        const double qbm2_hf = a.qbm * a.qbm * 0.5;
        gam_corr = qbm2_hf * (la.apr * la.apr + la.api * la.api);
        const double tmp = 0.5 * a.qbm / a.gamma[p];
        ep[0] = ep[0] - tmp * (la.apr * la.aprg[0] + la.api * la.apig[0]);
        ep[1] = ep[1] - tmp * (la.apr * la.aprg[1] + la.api * la.apig[1]);
        ep[2] = ep[2] + tmp * (la.apr * la.aprg[2] + la.api * la.apig[2]);
        apr = la.apr;
        api = la.api;
        apr_z = la.aprg[2];
        api_z = la.apig[2];
    }
    double pp[3] = {a.p1[p], a.p2[p], a.p3[p]}, ut[3];
    double qtmh1, qtmh2;
    if constexpr (STD || PGC) {
        qtmh1 = a.qtmh / (1.0 - a.qbm * a.psi[p]);
        qtmh2 = qtmh1 * a.gamma[p];
    } else {
        const double gam = sqrt(1.0 + pp[0] * pp[0] + pp[1] * pp[1] + pp[2] * pp[2]);
        qtmh1 = a.qtmh / (gam - pp[2]);
        qtmh2 = qtmh1 * gam;
    }
#pragma unroll
    for (int cc = 0; cc < 3; cc++) {
        ep[cc] = ep[cc] * qtmh2;
        bp[cc] = bp[cc] * qtmh1;
        ut[cc] = pp[cc] + ep[cc];
    }
    pp[0] = ut[0] + ut[1] * bp[2] - ut[2] * bp[1];
    pp[1] = ut[1] + ut[2] * bp[0] - ut[0] * bp[2];
    pp[2] = ut[2] + ut[0] * bp[1] - ut[1] * bp[0];
    double ostq = 2.0 / (1.0 + bp[0] * bp[0] + bp[1] * bp[1] + bp[2] * bp[2]);
#pragma unroll
    for (int cc = 0; cc < 3; cc++) bp[cc] = bp[cc] * ostq;
    ut[0] = ut[0] + pp[1] * bp[2] - pp[2] * bp[1];
    ut[1] = ut[1] + pp[2] * bp[0] - pp[0] * bp[2];
    ut[2] = ut[2] + pp[0] * bp[1] - pp[1] * bp[0];
#pragma unroll
    for (int cc = 0; cc < 3; cc++) pp[cc] = ut[cc] + ep[cc];
    double g2;
    if constexpr (PGC) {
        const double qbm2_hf = a.qbm * a.qbm * 0.5;
        double tmp = apr_z * a.dt;
        gam_corr = gam_corr + qbm2_hf * (apr + 0.25 * tmp) * tmp;
        tmp = api_z * a.dt;
        gam_corr = gam_corr + qbm2_hf * (api + 0.25 * tmp) * tmp;
        g2 = sqrt(1.0 + pp[0] * pp[0] + pp[1] * pp[1] + pp[2] * pp[2] + gam_corr);
    } else {
        g2 = sqrt(1.0 + pp[0] * pp[0] + pp[1] * pp[1] + pp[2] * pp[2]);
    }
    if (a.clamp > 0.0) {
        // clamp_exp_fac (proj_subcyc/part2d_subcyc_class.f03:46-66): the
        // momentum scaled so that gamma / (gamma - p_z) becomes the clamp
        const double F = a.clamp;
        if (g2 / (g2 - pp[2]) > F) {
            double sc = (F - 1.0) * (F - 1.0);
            sc = sc / (F * F * pp[2] * pp[2] - sc * (g2 * g2 - 1.0));
            sc = sqrt(sc);
            pp[0] = pp[0] * sc;
            pp[1] = pp[1] * sc;
            pp[2] = pp[2] * sc;
            g2 = sqrt(1.0 + pp[0] * pp[0] + pp[1] * pp[1] + pp[2] * pp[2]);
        }
    }
    double dtc = a.dt / (g2 - pp[2]);
    x1 = x1 + pp[0] * dtc;
    x2 = x2 + pp[1] * dtc;
    a.p1[p] = pp[0];
    a.p2[p] = pp[1];
    a.p3[p] = pp[2];
    a.gamma[p] = g2;
    a.x1[p] = x1;
    a.x2[p] = x2;
    const uint32_t key = cell_key(x1, x2, a.idr, a.edge, a.nr);
    a.s.key_w[p] = key;
    return key;
}

template <int M, bool STD, bool PGC, bool SINGLE>
__global__ __launch_bounds__(kSmallChunk) void k_push_count(const PushMulti m)
{
    if ((int)blockIdx.y == m.n) {
        epilogue_block<kSmallChunk>(m.epi, blockIdx.x);
        return;
    }
    const PushArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    if ((int)blockIdx.x >= a.s.nchunks) return;
    extern __shared__ __attribute__((aligned(16))) int lds[];
    const int64_t p = sort_element<kSmallChunk, 1>(0);
    uint32_t kv[1] = {(uint32_t)a.nr};
    if (p < a.s.n) {
        if (p < a.s.cs[a.nr]) kv[0] = push_particle<M, STD, PGC, SINGLE>(a, p);
        else a.s.key_w[p] = (uint32_t)a.nr;
    }
    chunk_hist<kSmallChunk, 1>(a.s, kv, lds);
}

template <int M, bool STD, bool PGC, bool SINGLE>
__global__ __launch_bounds__(kPushThreads) void k_push(const PushMulti m)
{
    if ((int)blockIdx.y == m.n) {
        epilogue_block<kPushThreads>(m.epi, blockIdx.x);
        return;
    }
    const PushArgs a = m.s[__builtin_amdgcn_readfirstlane(blockIdx.y)];
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.s.n) return;
    const int npp = a.s.cs[a.nr];
    if (p >= npp) {
        a.s.key_w[p] = (uint32_t)a.nr;
        return;
    }
    push_particle<M, STD, PGC, SINGLE>(a, p);
}

static PushArgs push_args(qpad_ctx *c, int s, int form)
{
    Species &sp = c->sp[s];
    PushArgs a;
    a.nr = c->g.nr;
    a.ld = c->g.ld;
    a.nm = c->g.nm;
    a.idr = 1.0 / c->g.dr;
    a.edge = (double)c->g.nr * c->g.dr;
    a.qtmh = sp.qbm * c->dt2d * 0.5;
    a.dt = c->dt2d;
    a.clamp = c->clamp2d;
    a.qbm = sp.qbm;
    a.eb = c->eb;
    a.e = c->f[QPAD_F_E];
    a.b = c->f[QPAD_F_B];
    a.ar = c->f[QPAD_F_AR];
    a.ai = c->f[QPAD_F_AI];
    a.arg = c->f[QPAD_F_AR_GRAD];
    a.aig = c->f[QPAD_F_AI_GRAD];
    a.x1 = sp.x1; a.x2 = sp.x2; a.p1 = sp.p1; a.p2 = sp.p2; a.p3 = sp.p3; a.gamma = sp.gamma;
    a.psi = sp.psi;
    a.s = sort_args(c, s, form);
    return a;
}

// the push of the species of list entries (all of the push type STD, PGC
// names), with their cells counted where the sort's form asks for it
template <bool STD, bool PGC, bool SINGLE>
static int launch_push_list(qpad_ctx *c, const int *list, int n, int form, int &epi)
{
    PushMulti m;
    memset(&m, 0, sizeof(m));
    int maxc = 0;
    int64_t nmax = 0;
    for (int i = 0; i < n; i++) {
        m.s[i] = push_args(c, list[i], form);
        maxc = std::max(maxc, m.s[i].s.nchunks);
        nmax = std::max(nmax, m.s[i].s.n);
    }
    if (nmax == 0) return 0;
    // the slice's epilogue (epi > 0) rides with the first launch that moves
    // particles
    unsigned rows = n, eb = 0;
    m.n = n;
    if (epi > 0) {
        m.epi = epilogue_args(c, epi);
        eb = (unsigned)(epilogue_row_blocks(c->g.nr, form == SORT_DIRECT ? kSmallChunk : kPushThreads) * c->g.nm);
        rows = n + 1;
        epi = 0;
    }
    const dim3 cg(std::max((unsigned)maxc, eb), rows), blk(kSmallChunk);
    const dim3 pg(std::max((unsigned)((nmax + kPushThreads - 1) / kPushThreads), eb), rows);
    const size_t clds = sizeof(int) * (size_t)(c->g.nr + 1);
    hipEvent_t stop = nullptr;
    time_begin(c, 1, &stop);
#define QPAD_PUSH(MM)                                                                                       \
    do {                                                                                                    \
        if (form == SORT_DIRECT)                                                                            \
            hipLaunchKernelGGL((k_push_count<MM, STD, PGC, SINGLE>), cg, blk, clds, c->stream, m);           \
        else hipLaunchKernelGGL((k_push<MM, STD, PGC, SINGLE>), pg, dim3(kPushThreads), 0, c->stream, m);    \
    } while (0)
    switch (c->g.M) {
    case 0: QPAD_PUSH(0); break;
    case 1: QPAD_PUSH(1); break;
    case 2: QPAD_PUSH(2); break;
    case 3: QPAD_PUSH(3); break;
    default: QPAD_PUSH(4); break;
    }
#undef QPAD_PUSH
    QPAD_HIP_CHECK(hipGetLastError());
    time_end(c, 1, stop);
    return 0;
}

// species s0 .. s1-1: a push launch per pusher present (the two PGC pushers
// push alike), the first with slice epi's epilogue (0: none), then one sort of
// them all in the form that the most demanding species needs (MI355X, push and
// re-sort of a slice; a set of launches for each form and pusher -> one sort:
// 96,000 electrons and 12,000 ions in 3000 cells 42 -> 28 us, 524,288 and
// 32,768 in 8192 86 -> 56)
template <bool SINGLE>
static int launch_move_range(qpad_ctx *c, int s0, int s1, int epi)
{
    if (s1 > s0) {
        int list[3][kMaxSpecies], n[3] = {0, 0, 0}, form = SORT_DIRECT;
        for (int s = s0; s < s1; s++) {
            const int g = std::min(push_group(c->sp[s].cfg.push_type), 2);
            list[g][n[g]++] = s;
            form = std::min(form, sort_form(c, s));
        }
        if (n[0]) QPAD_TRY((launch_push_list<false, false, SINGLE>(c, list[0], n[0], form, epi)));
        if (n[1]) QPAD_TRY((launch_push_list<true, false, SINGLE>(c, list[1], n[1], form, epi)));
        if (n[2]) QPAD_TRY((launch_push_list<false, true, SINGLE>(c, list[2], n[2], form, epi)));
        SortMulti m;
        memset(&m, 0, sizeof(m));
        for (int s = s0; s < s1; s++) m.s[s - s0] = sort_args(c, s, form);
        QPAD_TRY(launch_sort_list(c, m, s1 - s0, form == SORT_DIRECT));
        for (int s = s0; s < s1; s++) sort_swap(c->sp[s]);
    }
    return epi > 0 ? launch_epilogue(c, epi) : 0;   // no particles
}

int launch_move(qpad_ctx *c, int s) { return launch_move_range<true>(c, s, s + 1, 0); }

int launch_move_all(qpad_ctx *c, int epi) { return launch_move_range<false>(c, 0, c->nspecies, epi); }

// ---------------------------------------------------------------------------
// interp_psi_part2d (part2d_class.f03:2264-2305): the field psi at every
// particle of a standard-pusher species, after the slice's psi solve
// (simulation_class.f03:357-359).  Thread per particle slot; particles past
// cell_start[nr] have left the box.
// ---------------------------------------------------------------------------
struct InterpPsiArgs {
    int nr, ld;
    int64_t nslots;
    double idr;
    const double *x1, *x2, *f;
    double *psi;
    const int32_t *cs;
};

template <int M>
__global__ __launch_bounds__(256) void k_interp_psi(const InterpPsiArgs a)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.nslots || p >= a.cs[a.nr]) return;
    constexpr int NM = 2 * M + 1;
    const double x1 = a.x1[p], x2 = a.x2[p];
    const double r = radius(x1, x2);
    const double pc = x1 / r, ps = x2 / r;
    double pos = __dmul_rn(r, a.idr);
    if (!(pos >= 0.0)) pos = 0.0;
    const int ic = (int)fmin(pos, (double)(a.nr - 1));
    const int ix = ic + 1;
    const double w1 = pos - (double)ic, w0 = 1.0 - w1;
    // the gather of interp_field (interp_part2d.f03:66-110) for one
    // component, in gather_n's order of operations
    const double *f = a.f + ix;
    double v = 0.0;
    v = v + f[0] * w0;
    v = v + f[1] * w1;
    double phr = 1.0, phi = 0.0;
#pragma unroll
    for (int m = 1; m <= M; m++) {
        const double tr = phr * pc - phi * ps, ti = phr * ps + phi * pc;
        phr = tr;
        phi = ti;
        const double ph_re = 2.0 * phr, ph_im = 2.0 * phi;
        const double *fr = f + (size_t)(2 * m - 1) * a.ld, *fi = f + (size_t)(2 * m) * a.ld;
        v = v + (fr[0] * ph_re - fi[0] * ph_im) * w0;
        v = v + (fr[1] * ph_re - fi[1] * ph_im) * w1;
    }
    (void)NM;
    a.psi[p] = v;
}

int launch_interp_psi(qpad_ctx *c, int s)
{
    Species &sp = c->sp[s];
    const int pt = sp.cfg.push_type;
    if ((pt != QPAD_PUSH2_STD && pt != QPAD_PUSH2_STD_PGC) || sp.npp == 0) return 0;
    InterpPsiArgs a;
    a.nr = c->g.nr;
    a.ld = c->g.ld;
    a.nslots = sp.npp;
    a.idr = 1.0 / c->g.dr;
    a.x1 = sp.x1;
    a.x2 = sp.x2;
    a.f = c->f[QPAD_F_PSI];
    a.psi = sp.psi;
    a.cs = sp.cell_start;
    const dim3 grid((unsigned)((sp.npp + 255) / 256)), blk(256);
    switch (c->g.M) {
    case 0: hipLaunchKernelGGL(k_interp_psi<0>, grid, blk, 0, c->stream, a); break;
    case 1: hipLaunchKernelGGL(k_interp_psi<1>, grid, blk, 0, c->stream, a); break;
    case 2: hipLaunchKernelGGL(k_interp_psi<2>, grid, blk, 0, c->stream, a); break;
    case 3: hipLaunchKernelGGL(k_interp_psi<3>, grid, blk, 0, c->stream, a); break;
    default: hipLaunchKernelGGL(k_interp_psi<4>, grid, blk, 0, c->stream, a); break;
    }
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

// q_spe += qn (the neutralising background of species s)
__global__ void k_axpy(double *y, const double *x, int64_t n)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) y[t] = y[t] + x[t];
}

// ---------------------------------------------------------------------------
// species2d%q and cbq (species2d_class.f03:186-208, :396-410): the species'
// own rho - Jz (its deposit with the axis rules and 1/r; the neutralising
// background enters only the total), then J_z of its last executed current
// deposit added, and the sum copied into the species' history slice
// ---------------------------------------------------------------------------
int launch_species_q_start(qpad_ctx *c, int s)
{
    return launch_combine_q(c, s, c->sp[s].qsl, 1.0, false);
}

// thread per (node i = 0..nr+1, mode array k): q += J_z of the species
// (comp 2 of its current-deposit partials, axis x8 at m = 0 and 0 above),
// then history slice = q
__global__ void k_species_cbq(const double *P0, const double *P1, const double *O0, const double *O1,
                              const int32_t *os, double *q, double *hist, int nr, int nm, int ld)
{
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= (int64_t)nm * (nr + 2)) return;
    const int i = (int)(tid % (nr + 2)), k = (int)(tid / (nr + 2));
    const int NV = 8 * nm, v = 2 * nm + k;
    double val = 0.0;
    if (i >= 1 && i <= nr) val += cell_partial(P0, O0, os, i - 1, NV, v);
    if (i >= 2) val += cell_partial(P1, O1, os, i - 2, NV, v);
    if (i == 0) val = 0.0;
    else if (i == 1) val = (k == 0) ? 8.0 * val : 0.0;
    else val = val * (1.0 / (double)(i - 1));
    const size_t o = (size_t)k * ld + i;
    const double x = q[o] + val;
    q[o] = x;
    hist[o] = x;
}

int launch_species_cbq(qpad_ctx *c, int s, int j)
{
    const Species &sp = c->sp[s];
    const int64_t n = (int64_t)c->g.nm * (c->g.nr + 2);
    double *hist = sp.h_q + (size_t)j * c->g.nm * c->g.ld;
    hipLaunchKernelGGL(k_species_cbq, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, sp.P0, sp.P1,
                       sp.O0, sp.O1, sp.ov_start, sp.qsl, hist, c->g.nr, c->g.nm, c->g.ld);
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_add_qn_into_qspe(qpad_ctx *c, int s)
{
    int64_t n = (int64_t)c->g.nm * c->g.ld;
    hipLaunchKernelGGL(k_axpy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, c->f[QPAD_F_Q_SPE],
                       c->sp[s].qn, n);
    QPAD_HIP_CHECK(hipGetLastError());
    return 0;
}

}  // namespace qpad
