// epilogue.h -- the closing copy-out of a slice, a kernel of its own
// (k_slice.hip) or a row of workgroups of the push launch (k_plasma.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "conv.h"
#include "field_src.h"

namespace qpad {

// ---------------------------------------------------------------------------
// slice epilogue (simulation_class.f03:401-456): cbq, E of the plasma alone,
// history copies, beam fields of slice j into the slice arrays, J_perp
// predictor
// ---------------------------------------------------------------------------
struct EpiArgs {
    FieldCommon g;
    const double *e, *b, *psi, *b_spe, *q_beam_j, *b_beam_j;
    double *cu, *dcu;   // J_perp predictor in place: dcu *= dxi, cu(1:2) += dcu
    double dxi;
    double *e_spe, *q_spe;
    double *h_e, *h_b, *h_psi, *h_b_spe, *h_e_spe, *h_cu, *h_q_spe;
    double *q_beam_f1, *b_beam_f1;
    IterState *it;
    const double *conv_blk;   // both parities
    int nblk;
    int iter_max;
};

// workgroup b of T threads of the epilogue, b = 0 .. epilogue_blocks - 1: a
// thread per node i = 0..nr+1 of mode array k.  Nothing it reads or writes is
// read or written by a push or a sort, so it also runs as a row of the push
// launch (launch_move_all): 256 nodes, M = 1 3.8 + 4.9 us apart, 5.0 together;
// 4096 nodes, M = 2, 524,288 particles 5.5 + 17.3, 18.8 together
inline __host__ __device__ int epilogue_row_blocks(int nr, int T) { return (nr + 2 + T - 1) / T; }

template <int T>
__device__ __forceinline__ void epilogue_block(const EpiArgs &a, int b)
{
    const FieldCommon &g = a.g;
    const int nm = g.nm, ld = g.ld, nr = g.nr;
    const int per = epilogue_row_blocks(nr, T), k = b / per;
    const int i = (b - k * per) * T + threadIdx.x;
    if (k >= nm) return;
    if (b == 0 && threadIdx.x < 64) {
        // residuals of the last iteration executed (rel/abs of 'compare')
        const int iters = a.it->iters;
        double rel, ab;
        conv_residuals(a.conv_blk + (size_t)(iters & 1) * 2 * a.nblk, a.nblk, rel, ab);
        if (threadIdx.x == 0) {
            a.it->rel = rel;
            a.it->abs_ = ab;
            a.it->total_iters += iters;
            if (iters >= a.iter_max) a.it->at_max += 1;
        }
    }
    if (i > nr + 1) return;
    // every load first, then every store: the arrays are distinct, and
    // interleaved copies would wait for each load in turn (the compiler must
    // assume a store may alias the next load)
    double ve[3], vb[3], vcu[3], vbs[3], vbb[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        ve[c] = FX(a.e, c, k, i);
        vb[c] = FX(a.b, c, k, i);
        vcu[c] = FX(a.cu, c, k, i);
        vbs[c] = FX(a.b_spe, c, k, i);
        vbb[c] = FX(a.b_beam_j, c, k, i);
    }
    // E_perp of the plasma fields alone (e_spe, for the next slice's pipeline
    // and diagnostics)
    const bool inner = i >= 1 && i <= nr;
    double ev[2];
    if (inner) {
        et_node(g, vbs[0], vbs[1], FieldArr{a.psi, nm, ld}, k, i, ev);
    } else {
        ev[0] = FX(a.e_spe, 0, k, i);
        ev[1] = FX(a.e_spe, 1, k, i);
    }
    const double es2 = FX(a.e_spe, 2, k, i);
    const size_t o = (size_t)k * ld + i;
    const double qs = a.q_spe[o], ps = a.psi[o], qb = a.q_beam_j[o];
    const double dc0 = FX(a.dcu, 0, k, i), dc1 = FX(a.dcu, 1, k, i);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        FX(a.h_e, c, k, i) = ve[c];
        FX(a.h_b, c, k, i) = vb[c];
        FX(a.h_cu, c, k, i) = vcu[c];
        FX(a.h_b_spe, c, k, i) = vbs[c];
        FX(a.b_beam_f1, c, k, i) = vbb[c];
    }
    if (inner) {
        FX(a.e_spe, 0, k, i) = ev[0];
        FX(a.e_spe, 1, k, i) = ev[1];
    }
    FX(a.h_e_spe, 0, k, i) = ev[0];
    FX(a.h_e_spe, 1, k, i) = ev[1];
    FX(a.h_e_spe, 2, k, i) = es2;
    // q_spe = (rho - Jz) + Jz (species2d%cbq)
    const double q = qs + vcu[2];
    a.q_spe[o] = q;
    a.h_q_spe[o] = q;
    a.h_psi[o] = ps;
    a.q_beam_f1[o] = qb;
    // J_perp predictor for the next slice, after the history copy of cu
    // (simulation_class.f03:425-426)
    const double d0 = a.dxi * dc0, d1 = a.dxi * dc1;
    FX(a.dcu, 0, k, i) = d0;
    FX(a.dcu, 1, k, i) = d1;
    FX(a.cu, 0, k, i) = vcu[0] + d0;
    FX(a.cu, 1, k, i) = vcu[1] + d1;
}

EpiArgs epilogue_args(qpad_ctx *c, int j);   // k_slice.hip

}  // namespace qpad
