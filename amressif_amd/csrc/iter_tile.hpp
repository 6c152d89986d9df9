// One FP64 pseudo-iteration (four RK4 dual-time stages) of a 2D step in one
// launch (kernels_iter.hip), for wall and periodic sides and either face layout.
#pragma once

#include <hip/hip_runtime.h>

#include "internal.hpp"

namespace amr {

struct IterTile {
    const double *u, *v;    // u^k: the stages' base and the first one's stencil input
    const double *cu, *cv;  // BDF2 constant with -G p
    double *uo, *vo;        // u^{k+1}; must not alias u, v
    const double *lid;      // per-column velocity of the north side (kind 3), or null: inflow
    double *partials;       // records of `rec` doubles, the first two written: sum of the weighted change^2 of u and v
    Ctl *ctl;               // null: unguarded
    // records of the launch before, if its norm has not been taken yet: this launch then ends the loop
    // itself where k_fin_pseudo would have (null: the control block is up to date)
    const double *prev;
    int it;                 // pseudo-iterations of the step before this launch
    int n, su, sv;          // cells per side, row strides of the x- and y-faces
    int rec;
    int copy_done;  // a launch past convergence copies u^k to the output (else it writes nothing)
    int nst, expl;  // stages (4; 1 with expl: the explicit update's wall rule)
    int per[2], kind[4];  // periodic directions; wall rules W, E, S, N as gen.hpp's kinds
    double inflow[2];
    double rk[4], c15, idx[2], idx2[2], iren;
    // set by launch_iter_tile
    int ntx;
    double kq[2], kv[2], sg[4][2], ct[4][2];
};

// workgroups (partial records) of a launch at n cells per side
int iter_tile_blocks(int n);
hipError_t launch_iter_tile(IterTile a, hipStream_t s);

}  // namespace amr
