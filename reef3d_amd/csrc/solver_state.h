// The scalar state machine of bicgstab_ijk::solve (bicgstab_ijk.cpp:125-278) and of its mixed
// form, one thread per tank: what each phase's sums leave in BiState.  Shared by the
// finalize kernels of the streaming solver and the on-chip solver, so both take the same
// decisions from the same sums.
#pragma once

#include "batch.h"

namespace reef {
namespace bk {

// The tank table is never written by a kernel: reading it through the constant address
// space lets the compiler use scalar loads (the tank's pointers and sizes stay in SGPRs).
// Kernels take the tank by reference there and copy only its DevGrid: indexing a local
// copy of the pointer table with a run-time array id would keep the whole table in
// registers.
// (the host compilation pass of this file never runs device code and has no such
// address space)
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(4))) const TankDev CTank;
#else
typedef const TankDev CTank;
#endif

__device__ __forceinline__ CTank& tank_of_slot(const TankDev* tanks, int slot) { return ((CTank*)tanks)[slot]; }

// The state that a reliable update (mode 3) or restart (mode 1) of the mixed solve leaves,
// from the FP64 sums of its residual phase tot = {|r|^2, (r0, r)} (kb_mix_ru).  The phase
// has no finalize launch of its own: the blocks of the next v phase evaluate the outcome
// from the same sums (they need beta and the mode), kb_fin_v stores it, and
// kb_fin_mix_ru stores it after the last iteration of a batch, so the states the host
// reads are settled.  An idle phase then costs one launch, not two.
struct RuNext
{
    double rn, residual, r_j, norm_r0, beta;
    int iter, done, mode;
};

__device__ __forceinline__ RuNext ru_next(const BiState* st, const double (&tot)[2])
{
    RuNext n;
    n.rn = sqrt(tot[0]);
    n.residual = n.rn / double(st->ncell);
    n.iter = st->iter + (st->mode == 1 ? 1 : 0);   // a restart counts as an iteration (bicgstab_ijk.cpp:183-191)
    n.done = !((n.residual >= st->stop) && (n.iter < st->maxiter));
    n.mode = st->mode == 1 ? 2 : 0;
    n.r_j = tot[1];
    n.norm_r0 = st->norm_r0;
    n.beta = st->beta;
    if(st->mode == 1)
        n.norm_r0 = sqrt(tot[1]);
    else
    {
        const double wr = st->w * st->r_j_prev;
        n.beta = st->alpha * tot[1] / (wr == 0 ? 1.0e-15 : wr);
    }
    return n;
}

__device__ __forceinline__ void restart_store(BiState* st, double rr)
{
    st->r_j = rr;
    st->rr = rr;
    st->norm_r0 = sqrt(rr);
    st->residual = sqrt(rr) / double(st->ncell);
    st->iter += 1;
    if(!((st->residual >= st->stop) && (st->iter < st->maxiter))) st->done = 1;
    st->mode = 2;
}

// stores the outcome (one thread)
__device__ __forceinline__ void ru_store(BiState* st, const RuNext& n)
{
    st->residual = n.residual;
    st->nru += 1;
    st->pending = 1;
    st->rmax = n.rn;
    st->iter = n.iter;
    if(n.done)
    {
        st->done = 1;
        return;
    }
    st->r_j = n.r_j;
    st->norm_r0 = n.norm_r0;
    st->beta = n.beta;
    st->mode = n.mode;
}

// alpha and the restart tests from the v phase's sums: sigma = (v, r0), vv = |v|^2, rr = |r|^2
// (bicgstab_ijk.cpp:162-191); swap: the phase wrote p and v into the other halves of their
// buffers
__device__ __forceinline__ void v_store(BiState* st, double sigma, double vv, double rr, bool swap)
{
    const double norm_vj = sqrt(vv);
    const double norm_rj = sqrt(rr);
    const double alpha = st->r_j / sigma;
    st->sigma = sigma;
    st->norm_vj = norm_vj;
    st->norm_rj = norm_rj;
    st->alpha = alpha;
    if(swap) st->buf ^= 1;
    if(st->mixed) st->pending = 0;   // the fused v phase added x32
    if(fabs(sigma) <= (1.0e-12 * (norm_vj * st->norm_r0)))
        st->mode = 1;
    else if((fabs(alpha) * norm_vj / (norm_rj == 0 ? 1.0e-15 : norm_rj)) <= 0.08)
        st->mode = 1;
    else
        st->mode = 0;
}

// omega from the t phase's sums {(t, s), (t, t), (s, s)} (bicgstab_ijk.cpp:205-221)
__device__ __forceinline__ void t_store(BiState* st, const double (&tot)[3])
{
    st->w1 = tot[0];
    st->w2 = tot[1];
    st->norm_sj = sqrt(tot[2]);
    st->branch = st->norm_sj > st->stop ? 1 : 0;
    st->w = st->branch ? tot[0] / (tot[1] == 0 ? 1.0e-15 : tot[1]) : st->w;
}

// beta, residual, iteration count from the x phase's sums {(r, r0), |r|^2}; the mixed form
// asks for reliable updates instead of ending on the iterated residual
__device__ __forceinline__ void x_store(BiState* st, const double (&tot)[2])
{
    const double alpha = st->alpha, w = st->w, r_j1 = tot[0];
    st->r_j_prev = st->r_j;
    if(st->branch) st->beta = alpha * r_j1 / (w * st->r_j == 0 ? 1.0e-15 : (w * st->r_j));
    st->r_j1 = r_j1;
    st->r_j = r_j1;
    st->rr = tot[1];
    st->residual = sqrt(tot[1]) / double(st->ncell);
    st->iter += 1;
    st->mode = 0;
    if(!st->mixed)
    {
        if(!((st->residual >= st->stop) && (st->iter < st->maxiter))) st->done = 1;
        return;
    }
    const double rn = sqrt(tot[1]);
    if(rn > st->rmax) st->rmax = rn;
    if(!st->branch)
        st->mode = 1;
    else if(!(st->residual >= st->stop) || st->iter >= st->maxiter || rn < st->delta * st->rmax)
        st->mode = 3;
}

}  // namespace bk
}  // namespace reef
