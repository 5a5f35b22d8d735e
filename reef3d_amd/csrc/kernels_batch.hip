// Kernels of the batched engine.  A launch covers a set of tanks (TankSet, by value).
// Stencil and elementwise kernels run one 256-cell tile per block; the tiles of the set
// are numbered tank by tank, z fastest, and block b takes tile (b % 8) * per + b / 8, so
// the blocks the hardware sends to XCD x (b % 8 == x) work on one contiguous eighth of
// the tiles and share that XCD's L2 for their halos.  Reductions run a persistent grid
// (a multiple of 8 blocks) over the set's work items (runs of cpt tiles of one tank):
// block group x walks the x-th eighth of the item range.  Every reduction writes one
// partial per work item and a per-tank finalize block adds a tank's partials in item
// order, so a tank's arithmetic does not depend on the other tanks of a launch.
//
// The per-cell arithmetic is cell_ops.h's (the reference's operation order), so the
// stencil results are bit-identical to the reference whatever the set.
#include "batch.h"
#include "cell_ops.h"
#include "solver_state.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace reef {
namespace bk {

// ------------------------------------------------------------------ work walk
// index p with a[p] <= g < a[p + 1] in a set's prefix array a[0..n]
__device__ __forceinline__ int set_find(const int* a, int n, int g)
{
    int lo = 0, hi = n;
    while(hi - lo > 1)
    {
        const int mid = (lo + hi) >> 1;
        if(a[mid] <= g)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

__device__ __forceinline__ CTank& tank_at(const TankSet& b, int p) { return ((CTank*)b.tanks)[b.slot[p]]; }

// persistent walk over the set's work items: q the item, p its tank in the set
struct ItemIter
{
    int q, hi, step, p;
};

// items [first, first + count) of the set, split into 8 XCD groups
__device__ __forceinline__ ItemIter set_items(const TankSet& b, int first, int count)
{
    int lo, hi;
    group_range(count, (int)(blockIdx.x & 7), lo, hi);
    lo += first;
    hi += first;
    ItemIter it;
    it.q = lo + (int)(blockIdx.x >> 3);
    it.hi = hi;
    it.step = (int)(gridDim.x >> 3);
    it.p = it.q < hi ? set_find(b.item0, b.n, it.q) : 0;
    return it;
}

__device__ __forceinline__ ItemIter set_items(const TankSet& b) { return set_items(b, 0, b.nitems); }

// all blocks stride over all items, so item q runs on XCD q % 8 (blocks go to the XCDs
// in turn) and the items of any one tank spread over every XCD: for kernels without
// neighbour reuse between items, where only some tanks of the set may have work
__device__ __forceinline__ ItemIter set_items_spread(const TankSet& b)
{
    ItemIter it;
    it.q = (int)blockIdx.x;
    it.hi = b.nitems;
    it.step = (int)gridDim.x;
    it.p = it.q < it.hi ? set_find(b.item0, b.n, it.q) : 0;
    return it;
}

// the items of the class-walked tanks (a prefix of the set) or of the others
template<bool PW>
__device__ __forceinline__ ItemIter set_items_of(const TankSet& b)
{
    return PW ? set_items(b, 0, b.pw_items) : set_items(b, b.pw_items, b.nitems - b.pw_items);
}

__device__ __forceinline__ void next_item(ItemIter& it, const TankSet& b)
{
    it.q += it.step;
    if(it.q < it.hi)
        while(b.item0[it.p + 1] <= it.q) ++it.p;
}

// a tank the walk skips: go on to this block's last item of it (the tank's items are
// contiguous in the set), so the next step leaves the tank after a single state check
__device__ __forceinline__ void skip_tank(ItemIter& it, const TankSet& b)
{
    const int end = b.item0[it.p + 1];
    if(it.q < end) it.q += ((end - 1 - it.q) / it.step) * it.step;
}

// the one tile of a block of a per-tile launch
struct TileIter
{
    bool ok;
    int p, t;
};

__device__ __forceinline__ TileIter set_tile(const TankSet& b)
{
    TileIter it;
    const int per = (b.ntiles + 7) >> 3;
    const int g = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    it.ok = g < b.ntiles;
    it.p = it.ok ? set_find(b.tile0, b.n, g) : 0;
    it.t = it.ok ? g - b.tile0[it.p] : 0;
    return it;
}

// tiles [t, t1) of the walk; gi = reduction slot of an item walk
struct TileWalk
{
    int t, t1, gi;
    TileShape s;
};

__device__ __forceinline__ TileWalk item_walk(CTank& T, const TankSet& b, const ItemIter& q)
{
    const int li = item_at(T.shape, q.q - b.item0[q.p]);
    TileWalk w;
    w.s = T.shape;
    w.t = li * T.shape.cpt;
    w.t1 = min(w.t + T.shape.cpt, T.shape.ntiles);
    w.gi = T.item0 + li;
    return w;
}

// the same in item_spread order (the class phases)
__device__ __forceinline__ TileWalk class_item(CTank& T, const TankSet& b, const ItemIter& q)
{
    const int li = item_spread(T.shape, q.q - b.item0[q.p]);
    TileWalk w;
    w.s = T.shape;
    w.t = li * T.shape.cpt;
    w.t1 = min(w.t + T.shape.cpt, T.shape.ntiles);
    w.gi = T.item0 + li;
    return w;
}

// reduction slot of the current item of a persistent walk
__device__ __forceinline__ int item_slot(CTank& T, const TankSet& b, const ItemIter& q)
{
    return T.item0 + item_at(T.shape, q.q - b.item0[q.p]);
}

__device__ __forceinline__ TileWalk tile_walk(CTank& T, int t)
{
    TileWalk w;
    w.s = T.shape;
    w.t = t;
    w.t1 = t + 1;
    w.gi = -1;
    return w;
}

__device__ __forceinline__ bool tile_cell(const DevGrid& g, const TileWalk& w, int t, int& i, int& j, int& k, long& c)
{
    if(!tile_cell_of(w.s, g.nx, g.ny, g.nz, t, (int)threadIdx.x, i, j, k)) return false;
    c = g.base + i + g.sx * j + g.sxy * k;
    return true;
}

// tile_cell for the per-cell stencils: a wavefront covers one row of the tile, so j and k
// are the same in all its lanes and are made scalar; the y / z grid tables they index then
// load through the scalar unit
__device__ __forceinline__ bool tile_cell_row(const DevGrid& g, const TileWalk& w, int t, int& i, int& j, int& k,
                                              long& c)
{
    tile_cell_of(w.s, g.nx, g.ny, g.nz, t, (int)threadIdx.x, i, j, k);
    j = __builtin_amdgcn_readfirstlane(j);
    k = __builtin_amdgcn_readfirstlane(k);
    if(i >= g.nx || j >= g.ny || k >= g.nz) return false;
    c = g.base + i + g.sx * j + g.sxy * k;
    return true;
}

// block sum of M values (wavefront butterfly, lane 0's sum, 4-wave combine) into dst[0..M)
template<int M>
__device__ __forceinline__ void block_sum_to(double (&v)[M], double* __restrict__ dst)
{
    __shared__ double ws[M][NT / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for(int m = 0; m < M; ++m)
        for(int off = 32; off > 0; off >>= 1) v[m] += __shfl_xor(v[m], off);
    if(lane == 0)
        for(int m = 0; m < M; ++m) ws[m][wave] = v[m];
    __syncthreads();
    if(threadIdx.x == 0)
        for(int m = 0; m < M; ++m) dst[m] = ((ws[m][0] + ws[m][1]) + ws[m][2]) + ws[m][3];
    __syncthreads();
}

// a tank's partials: items [item0, item0 + nitems), M values each
template<int M>
__device__ __forceinline__ void tank_totals(CTank& T, const TankSet& b, double (&tot)[M])
{
    sum_partials<M>(b.partials + (size_t)T.item0 * M, T.shape.nitems, tot);
}

// the sums of a reliable-update phase (RuNext)
__device__ __forceinline__ void tank_totals_ru(CTank& T, const TankSet& b, double (&tot)[2])
{
    sum_partials<2>(b.partials_ru + (size_t)T.item0 * 2, T.shape.nitems, tot);
}

// the outcome as the v phase needs it: mode (0 or 2; 4 for done) in the high word, the FP32
// beta's bits in the low word.  Out of line, so that the walk of the calling kernel keeps
// its registers.
__device__ __noinline__ unsigned long long ru_outcome(const double* __restrict__ parts, int nitems, const BiState* st)
{
    double tot[2];
    sum_partials<2>(parts, nitems, tot);
    const RuNext n = ru_next(st, tot);
    return ((unsigned long long)(n.done ? 4u : (unsigned)n.mode) << 32) | __builtin_bit_cast(unsigned, (float)n.beta);
}

// The FP64 solve's restart (kb_bicg_p in mode 1) has no finalize launch of its own either:
// the v phase that follows it in the same iteration needs only its stop decision, taken
// from its sum |r|^2 (restart_done), and kb_fin_v stores its outcome (restart_store), as
// kb_fin_p does for the explicit-operator solve (bicgstab_ijk.cpp:183-191).
__device__ __noinline__ int restart_done(const double* __restrict__ parts, int nitems, const BiState* st)
{
    double tot[1];
    sum_partials<1>(parts, nitems, tot);
    const double residual = sqrt(tot[0]) / double(st->ncell);
    return !((residual >= st->stop) && (st->iter + 1 < st->maxiter));
}

// ------------------------------------------------------------------ per-precision views
template<class V>
struct Prec;

template<>
struct Prec<double>
{
    using Op = SolverOp64;
    __device__ static SolverOp64 op(CTank& T)
    {
        SolverOp64 o;
        o.rfx = T.f[A_RFX];
        o.rfy = T.f[A_RFY];
        o.rfz = T.f[A_RFZ];
        return o;
    }
    __device__ static BiVec<double> vec(CTank& T, int x, int rhs)
    {
        BiVec<double> v;
        v.x = T.f[x];
        v.rhs = T.f[rhs];
        v.r = T.f[A_R];
        v.r0 = T.f[A_R0];
        v.p = T.f[A_P];
        v.ph = T.f[A_PH];
        v.v = T.f[A_V];
        v.t = T.f[A_T];
        v.aii = T.f[A_AII];
        v.partials = nullptr;
        v.st = T.st;
        return v;
    }
};

template<>
struct Prec<float>
{
    using Op = SolverOp32;
    __device__ static SolverOp32 op(CTank& T)
    {
        SolverOp32 o;
        o.kx = T.s[S_KX];
        o.ky = T.s[S_KY];
        o.kz = T.s[S_KZ];
        o.iDXN = T.iDXN32;
        o.iDYN = T.iDYN32;
        o.iDZN = T.iDZN32;
        return o;
    }
    __device__ static BiVec<float> vec(CTank& T, int, int)
    {
        const int h = T.st->buf;
        BiVec<float> v;
        v.x = T.s[S_X];
        v.rhs = nullptr;
        v.r = T.s[S_R];
        v.r0 = T.s[S_R0];
        v.p = T.s[h ? S_P2 : S_P];
        v.ph = T.s[S_PH];
        v.v = T.s[h ? S_V2 : S_V];
        v.t = T.s[S_T];
        v.aii = T.s[S_AII];
        v.partials = nullptr;
        v.st = T.st;
        return v;
    }
};

// ------------------------------------------------------------------ simple kernels
__global__ void __launch_bounds__(NT) kb_copy(TankSet b, int src, int dst)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ s = T.f[src];
        double* __restrict__ d = T.f[dst];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(tile_cell(g, tw, t, i, j, k, c)) d[c] = s[c];
        }
    }
}

// every element of array id (ghosts and padding included) of every active tank
__global__ void __launch_bounds__(NT) kb_fill(TankSet b, int id, double v)
{
    for(int tk = 0; tk < b.n; ++tk)
    {
        CTank& T = tank_at(b, tk);
        double* __restrict__ f = T.f[id];
        const long n = T.g.nalloc;
        for(long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) f[q] = v;
    }
}

// compiled ghost program prog of tank blockIdx.y on array id
__global__ void __launch_bounds__(NT) kb_ghost(TankSet b, int prog, int id)
{
    CTank& T = tank_at(b, (int)blockIdx.y);
    const GhostOp* __restrict__ ops = T.gops[prog];
    const int n = T.gnops[prog];
    double* __restrict__ f = T.f[id];
    for(int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x)
    {
        const GhostOp op = ops[q];
        double val;
        if(op.src < 0)
            val = 0.0;
        else if(op.src & (1 << 30))
            val = 0.0 + op.w * f[op.src & ~(1 << 30)];
        else
            val = f[op.src];
        f[op.dst] = val;
    }
}

// ------------------------------------------------------------------ level set, reinit
// HJ-WENO transport stage fused with the TVD-RK3 combination (levelset_RK3.cpp:118-157,
// momentum_FC3.cpp:132-358); cdt = cfac * dt of the tank; stage 0 accumulates out += L
__global__ void __launch_bounds__(NT, 4) kb_hj_stage(TankSet b, int stage, int phi_s_, int phi_n_, int u_, int v_,
                                                   int w_, int out_, double cfac)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ phi_s = T.f[phi_s_];
        const double* __restrict__ phi_n = phi_n_ >= 0 ? T.f[phi_n_] : nullptr;
        const double* __restrict__ u = T.f[u_];
        const double* __restrict__ v = T.f[v_];
        const double* __restrict__ w = T.f[w_];
        double* __restrict__ out = T.f[out_];
        const double cdt = cfac * T.tstep[0];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell_row(g, tw, t, i, j, k, c)) continue;
            const double L = hj_L(g, phi_s, u, v, w, c, i, j, k);
            const double La = 0.0 + L;
            if(stage == 0)
                out[c] += L;
            else if(stage == 1)
                out[c] = phi_s[c] + cdt * La;
            else if(stage == 2)
                out[c] = 0.75 * phi_n[c] + 0.25 * phi_s[c] + cdt * La;
            else
                out[c] = (1.0 / 3.0) * phi_n[c] + (2.0 / 3.0) * phi_s[c] + cdt * La;
        }
    }
}

// reinit sub-stage (reini_RK3.cpp:114-139) with the per-cell pseudo time step
__global__ void __launch_bounds__(NT, 4) kb_reini_stage(TankSet b, int stage, int fs_, int f0_, int out_, double F43,
                                                      int fsf)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ f = T.f[fs_];
        const double* __restrict__ f0 = T.f[f0_];
        double* __restrict__ out = T.f[out_];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell_row(g, tw, t, i, j, k, c)) continue;
            const double lsv = f[c];
            const double L = reini_L(g, f, c, i, j, k, fsf);
            const double dtc = reini_dtc(g, i, j, k, F43);
            if(stage == 1)
                out[c] = f0[c] + dtc * L;
            else if(stage == 2)
                out[c] = 0.75 * f0[c] + 0.25 * lsv + 0.25 * dtc * L;
            else
                out[c] = (1.0 / 3.0) * f0[c] + (2.0 / 3.0) * lsv + (2.0 / 3.0) * dtc * L;
        }
    }
}

// ------------------------------------------------------------------ momentum
// WENO flux divergence accumulated into acc (convection::start, ipol 1..3)
__global__ void __launch_bounds__(NT, 4) kb_flux_acc(TankSet b, int ipol, int q_, int u_, int v_, int w_, int acc_)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        if(ipol == 2 && g.jdir == 0) continue;
        const double* __restrict__ qf = T.f[q_];
        const double* __restrict__ u = T.f[u_];
        const double* __restrict__ v = T.f[v_];
        const double* __restrict__ w = T.f[w_];
        double* __restrict__ acc = T.f[acc_];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell_row(g, tw, t, i, j, k, c) || !comp_cell(g, ipol, i, j, k)) continue;
            acc[c] += flux_div(g, ipol, qf, u, v, w, c, i, j, k);
        }
    }
}

// velocity predictor of one component (momentum_FC3.cpp:160-208 and the later stages);
// cdt = cfac * dt of the tank.  MODE 0: diff_void, 1: ediff2's explicit viscous terms added
// to F, 2 (idiff2_FS, D20 = 2): only F (irhs + convection) into out, the implicit solve and
// the stage combination follow (km_idiff, km_combine)
template<int comp, int MODE>
__global__ void __launch_bounds__(NT, 2) kb_momentum(TankSet b, int stage, int qin_, int qold_, int u_, int v_, int w_,
                                                   double grav, double cfac, int out_, double rw, double ra)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        if(comp == 2 && g.jdir == 0) continue;
        const double* __restrict__ qin = T.f[qin_];
        const double* __restrict__ qold = T.f[qold_];
        const double* __restrict__ u = T.f[u_];
        const double* __restrict__ v = T.f[v_];
        const double* __restrict__ w = T.f[w_];
        const double* __restrict__ press = T.f[REEF_PRESS];
        const double* __restrict__ phi = T.f[REEF_PHI];
        double* __restrict__ out = T.f[out_];
        const double cdt = cfac * T.tstep[0];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell_row(g, tw, t, i, j, k, c) || !comp_cell(g, comp, i, j, k)) continue;
            double F = momentum_F(g, comp, qin, u, v, w, press, phi, grav, rw, ra, c, i, j, k);
            if constexpr(MODE == 1) F += ediff_term(g, comp, u, v, w, T.f[REEF_VISC], c, i, j, k);
            if constexpr(MODE == 2)
            {
                out[c] = F;
                continue;
            }
            const double df = qin[c];
            if(stage == 1)
                out[c] = df + cdt * 1.0 * F;
            else if(stage == 2)
                out[c] = 0.75 * qold[c] + 0.25 * df + cdt * 1.0 * F;
            else
                out[c] = (1.0 / 3.0) * qold[c] + (2.0 / 3.0) * df + cdt * 1.0 * F;
        }
    }
}

// ------------------------------------------------------------------ fluid update
// fluid_update_fsf::start (fluid_update_fsf.cpp:39-74): rho, nu and the volume partials
__global__ void __launch_bounds__(NT) kb_heaviside(TankSet b, double rw, double vw, double ra, double va)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ phi = T.f[REEF_PHI];
        double* __restrict__ ro = T.f[REEF_RO];
        double* __restrict__ visc = T.f[REEF_VISC];
        double vals[2] = {0.0, 0.0};
        const TileWalk tw = item_walk(T, b, q);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            const double H = heaviside_H(phi[c], g.psi);
            ro[c] = rw * H + ra * (1.0 - H);
            visc[c] = vw * H + va * (1.0 - H);
            const double vol = g.DXN[i + MARGE] * g.DYN[j + MARGE] * g.DZN[k + MARGE];
            vals[0] += vol * (H - (1.0 - 1.0));
            vals[1] += vol * (1.0 - H - (1.0 - 1.0));
        }
        block_sum_to<2>(vals, b.partials + (size_t)item_slot(T, b, q) * 2);
    }
}

// volume1, volume2 of each tank of the set: into the tank's volume slot, or with out set
// into out[2 * (tank's index in the set) + 0, 1]
__global__ void __launch_bounds__(NT) kb_heaviside_fin(TankSet b, double* __restrict__ out)
{
    CTank& T = tank_at(b, blockIdx.x);
    double tot[2];
    tank_totals<2>(T, b, tot);
    double* dst = out ? out + 2 * blockIdx.x : T.vol;
    if(threadIdx.x == 0)
    {
        dst[0] = tot[0];
        dst[1] = tot[1];
    }
}

// ------------------------------------------------------------------ projection
__global__ void __launch_bounds__(NT) kb_poisson_rhs(TankSet b, int u_, int v_, int w_, double afac)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ u = T.f[u_];
        const double* __restrict__ v = T.f[v_];
        const double* __restrict__ w = T.f[w_];
        double* __restrict__ rhs = T.f[A_RHS];
        const double adt = afac * T.tstep[0];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(tile_cell(g, tw, t, i, j, k, c)) rhs[c] = poisson_rhs_cell(g, u, v, w, adt, c, i, j, k);
        }
    }
}

// the class of the wavefront's row of a tile (TankDev::cls): a wavefront holds one row of
// every tile shape, so j and k are its own; cells outside the grid count as any class
__device__ __forceinline__ void store_row_class(CTank& T, const TankSet& b, const DevGrid& g, bool in, double f0, double f1,
                                                double f2, double f3, double f4, double f5, int i, int j, int k)
{
    auto all_are = [&](double r) { return f0 == r && f1 == r && f2 == r && f3 == r && f4 == r && f5 == r; };
    const bool water = __all(!in || all_are(b.rw)), air = __all(!in || all_are(b.ra));
    if(in && (threadIdx.x & 63) == 0)
        T.cls[((long)(i / TILE_X) * g.ny + j) * g.nz + k] = water ? ROW_WATER : air ? ROW_AIR : ROW_MIXED;
}

// face densities of the "+" faces of the interior and of the -1 layer, optionally the
// Jacobi diagonal aii = -1/(M.p + 1e-19) (needs all faces: second pass)
__global__ void __launch_bounds__(NT) kb_face_rho(TankSet b, double rw, double ra)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ phi = T.f[REEF_PHI];
        double* __restrict__ rfx = T.f[A_RFX];
        double* __restrict__ rfy = T.f[A_RFY];
        double* __restrict__ rfz = T.f[A_RFZ];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            rfx[c] = roface(phi[c], phi[c + 1], g.psi, rw, ra);
            rfy[c] = roface(phi[c], phi[c + g.sx], g.psi, rw, ra);
            rfz[c] = roface(phi[c], phi[c + g.sxy], g.psi, rw, ra);
            if(i == 0) rfx[c - 1] = roface(phi[c], phi[c - 1], g.psi, rw, ra);
            if(j == 0) rfy[c - g.sx] = roface(phi[c], phi[c - g.sx], g.psi, rw, ra);
            if(k == 0) rfz[c - g.sxy] = roface(phi[c], phi[c - g.sxy], g.psi, rw, ra);
        }
    }
}

__global__ void __launch_bounds__(NT) kb_aii(TankSet b)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ rfx = T.f[A_RFX];
        const double* __restrict__ rfy = T.f[A_RFY];
        const double* __restrict__ rfz = T.f[A_RFZ];
        double* __restrict__ aii = T.f[A_AII];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            // every lane of the wavefront takes part in its row's class
            const bool in = tile_cell(g, tw, t, i, j, k, c);
            if(!in) c = g.base;
            store_row_class(T, b, g, in, rfx[c], rfx[c - 1], rfy[c], rfy[c - g.sx], rfz[c], rfz[c - g.sxy], i, j, k);
            if(!in) continue;
            const Coupling cq = couplings(g, rfx, rfy, rfz, c, i, j, k);
            aii[c] = -1.0 / (diag_of(g, cq) + 1e-19);
        }
    }
}

__global__ void __launch_bounds__(NT) kb_correct(TankSet b, double rw, double ra, double afac, int u_, int v_,
                                                  int w_)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double adt = afac * T.tstep[0];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(tile_cell(g, tw, t, i, j, k, c))
                correct_cell(g, T.f[REEF_PCORR], T.f[REEF_PHI], rw, ra, adt, T.f[u_], T.f[v_], T.f[w_],
                             T.f[REEF_PRESS], c, i, j, k);
        }
    }
}

// ------------------------------------------------------------------ BiCGStab
// Occupancy of the persistent solver kernels (waves per SIMD = blocks per CU): 8 for the
// FP32 / elementwise kernels; 5 for the kernels that apply the FP64
// operator cell by cell (about 100 registers), whose grids are sized to match.
constexpr int OCC_FULL = 8, OCC_A64 = 5;
// class walk: 4 blocks per CU (the default plan of a 3-D tank gives it one work item per
// block)
constexpr int OCC_PW = REEF_OCC_PW, OCC_CX = REEF_OCC_PW;

// The state machine of bicgstab_ijk::solve (bicgstab_ijk.cpp:125-278) per tank: mode 1 = a
// restart is pending, 2 = p and ph were just set from the residual, 3 = reliable update
// pending (mixed precision).  Dot products are accumulated in FP64 for both precisions.

// element e of an array through a 32-bit byte offset from its (uniform) base, so the load
// takes the scalar-base + 32-bit vector-offset form (a tank's arrays are below 4 GiB)
template<class T>
__device__ __forceinline__ T ld32(const T* __restrict__ p, unsigned e)
{
    return *(const T*)((const char*)p + e * (unsigned)sizeof(T));
}
template<class T>
__device__ __forceinline__ void st32(T* __restrict__ p, unsigned e, T v)
{
    *(T*)((char*)p + e * (unsigned)sizeof(T)) = v;
}

struct NoEpi
{
};

// ------------------------------------------------------------------ class walk (3-D tanks)
// Class walk of the 3-D stencil phases (tanks with 64 x 4 x 1 tiles): a block walks up the k
// planes of its item's column; the operand of plane k (rows j-1 .. j+4, columns i-1 .. i+64)
// sits in a double-buffered LDS plane (one barrier per plane), planes k-1 and k+1 of the own
// cell in registers.
//
// The operator comes from the density class of each 64-cell row (TankDev::cls): away from the
// interface band every face of a row has the density of water or of air exactly, so the six
// couplings of its cells are functions of one axis each: two table entries per axis, index and
// class (TankDev::ct, formed with the assembly's operations, so they are the same bits).  x and
// y entries stay in registers along a column, the z entries load through the scalar unit, and
// the Jacobi factor is one division of their sum.  Only rows of mixed class read the three
// face arrays and aii and form the couplings with six divisions.
// What bounds it: HBM bytes.  On the 512x64x128 wave tank 91 % of the rows have one class and
// read neither faces nor aii.

// the couplings of a row class along one axis at index ix
template<class V>
struct Pair
{
    V p, m;
};
__device__ __forceinline__ Pair<double> class_pair64(CTank& T, int axis, int n, int c, int ix)
{
    const double* t = T.ct[axis] + 2 * ((c - 1) * n + ix);
    return {t[0], t[1]};
}
template<class V>
__device__ __forceinline__ Pair<V> class_pair(CTank& T, int axis, int n, int c, int ix)
{
    const int e = 2 * ((c - 1) * n + ix);
    if constexpr(sizeof(V) == 8)
        return {T.ct[axis][e], T.ct[axis][e + 1]};
    else
        return {T.ct32[axis][e], T.ct32[axis][e + 1]};
}

// the classes of one row in up to 64 planes from k on: lane l holds plane k + l
struct RowClasses
{
    int k0, v;
    __device__ __forceinline__ void open(const unsigned char* row, int nz, int k)
    {
        k0 = k;
        v = row[min(k + (int)(threadIdx.x & 63), nz - 1)];
    }
    __device__ __forceinline__ int at(int k) const { return __builtin_amdgcn_readlane(v, k - k0); }
};

// Loads of one plane of the walk, issued D planes ahead: the operand's raw inputs at one halo
// cell of the block and at the cell above, the epilogue's inputs; of mixed rows also the
// faces, aii above and aii of the halo cell.  Halo cells are spread over the threads: thread
// h < 64 the south row (j0-1, i0+h), 64 <= h < 128 the north row (j0+TY, i0+h-64), 128 <= h <
// 132 the west column (j0+h-128, i0-1), 132 <= h < 136 the east column (j0+h-132, i0+TX).
template<class V, class R, class E>
struct ClassIn
{
    R h, xu;
    V f[6], ah, au;
    E e;
};

// Where the operand's aii comes from: none needed (the operand is stored), loaded with the
// operand (4 bytes cost less than the FP64 division), or from the row class
enum
{
    AII_NONE = 0,
    AII_LOAD = 1,
    AII_CLASS = 2
};

// For the planes of a column run and the one below and above, in LDS: the z entries of both
// classes, {water +, -, air +, -}, and the row classes (rows j0 .. j0+3, j0-1, j0+4, the west
// and the east neighbours of the first four).  They are not loaded where they are used: a
// global load in the plane loop that is used at once, on any path, waits for the loads in flight.
constexpr int ZPLANES = 66, CROWS = 2 + 3 * TY;
template<class V>
struct ClassLDS
{
    V x[2][TY + 2][TX + 2];
    double z[ZPLANES][4];
    float z32[sizeof(V) == 4 ? ZPLANES : 1][4];
    unsigned char c[CROWS][ZPLANES + 2];
    // grid factors of the mixed rows' couplings
    using AF = AxisFactor<std::conditional_t<sizeof(V) == 8, SolverOp64, SolverOp32>>;
    AF ax[TX], ay[TY], az[ZPLANES];
};

// raw(cc) -> R: the loads of the stencil operand at cc; val(R, aii, V& aux) -> V: the operand
// (aux: what the epilogue needs of the centre); pre(c) -> E: the epilogue's loads;
// post(c, Ax, aux, E): the epilogue.  Every load's address is valid (clamped) and its value
// masked afterwards.  A column run is at most 64 planes (cpt <= 64).
template<class V, int AII, int D, class Raw, class Val, class Pre, class Post>
__device__ __forceinline__ void class_walk(CTank& T, const DevGrid& g, const TileWalk& tw, Raw raw, Val val, Pre pre, Post post)
{
    using R = decltype(raw(0u));
    using E = decltype(pre(0u));
    using In = ClassIn<V, R, E>;
    constexpr bool DIV = AII == AII_CLASS, LOAD = AII == AII_LOAD;
    __shared__ ClassLDS<V> S;
    std::conditional_t<sizeof(V) == 8, SolverOp64, SolverOp32> op{};
    if constexpr(sizeof(V) == 4) op = SolverOp32{nullptr, nullptr, nullptr, T.iDXN32, T.iDYN32, T.iDZN32};
    const V *fxa, *fya, *fza, *aiia;
    if constexpr(sizeof(V) == 8)
    {
        fxa = T.f[A_RFX];
        fya = T.f[A_RFY];
        fza = T.f[A_RFZ];
        aiia = T.f[A_AII];
    }
    else
    {
        fxa = T.s[S_KX];
        fya = T.s[S_KY];
        fza = T.s[S_KZ];
        aiia = T.s[S_AII];
    }
    const int h = threadIdx.x;
    // one tile row per wavefront: the row (and with it j) is wave-uniform
    const int lane = h & (TX - 1), row = __builtin_amdgcn_readfirstlane(h >> 6);
    // halo cell relative to the tile, its LDS slot, its row's classes
    int hi = 0, hj = 0, hslot = 0, hrow = 0;
    if(h < TX)
    {
        hi = h;
        hj = -1;
        hslot = h + 1;
        hrow = TY;
    }
    else if(h < 2 * TX)
    {
        hi = h - TX;
        hj = TY;
        hslot = (TY + 1) * (TX + 2) + h - TX + 1;
        hrow = TY + 1;
    }
    else if(h < 2 * TX + TY)
    {
        hi = -1;
        hj = h - 2 * TX;
        hslot = (h - 2 * TX + 1) * (TX + 2);
        hrow = TY + 2 + hj;
    }
    else if(h < 2 * TX + 2 * TY)
    {
        hi = TX;
        hj = h - 2 * TX - TY;
        hslot = (h - 2 * TX - TY + 1) * (TX + 2) + TX + 1;
        hrow = 2 * TY + 2 + hj;
    }
    const bool has_halo = h < 2 * TX + 2 * TY;
    const unsigned sxy = (unsigned)g.sxy, sx = (unsigned)g.sx;

    // ---- column state
    int k = 0, kend = 0, zk0 = 0;   // current plane, planes [k, kend) of this run, first z plane in LDS
    int ic = 0, jc = 0;
    bool in = false, hval = false;
    unsigned coff = 0, hoff = 0;    // element offsets within plane k = 0
    auto own = [&](int kk) { return __builtin_amdgcn_readfirstlane((int)S.c[row][kk - zk0]); };
    // of the class each belongs to: the own cell's x coefficients and coupling sum over x and y,
    // the same sum for the next own cell and for the halo cell
    V cn = V(0), cs = V(0), s4 = V(0);
    double s4N = 0.0, s4H = 0.0;
    int keyC = 0, keyN = 0, keyH = 0;
    auto sum_xy = [&](int c, int ci, int cj) {
        const Pair<double> px = class_pair64(T, 0, g.nx, c, ci), py = class_pair64(T, 1, g.ny, c, cj);
        return px.p + px.m + py.p + py.m;
    };
    // aii of a cell of class c in plane kk from its x and y sum (diag_of's order)
    auto jacobi = [&](double sxy4, int c, int kk) -> V {
        const double* const z = &S.z[kk - zk0][2 * c - 2];
        return (V)(-1.0 / ((sxy4 + z[0] + z[1]) + 1e-19));
    };
    auto own_a = [&](int kk, int c, V loaded) -> V {
        if(!DIV || c == ROW_MIXED) return loaded;
        if(c != keyN)
        {
            s4N = sum_xy(c, ic, jc);
            keyN = c;
        }
        return jacobi(s4N, c, kk);
    };
    // the loads of a plane that need no class, then those that do
    auto fetch_raw = [&](int kk, In& P) {
        const unsigned c = coff + sxy * (unsigned)kk;
        P.h = raw(hoff + sxy * (unsigned)kk);
        P.xu = raw(c + sxy);   // kk + 1 <= nz: a ghost plane at worst
        P.e = pre(c);
        if(LOAD)
        {
            P.au = ld32(aiia, coff + sxy * (unsigned)min(kk + 1, g.nz - 1));
            P.ah = ld32(aiia, hoff + sxy * (unsigned)kk);
        }
    };
    auto fetch_mixed = [&](int kk, In& P) {
        const unsigned c = coff + sxy * (unsigned)kk;
        if(own(kk) == ROW_MIXED)
        {
            P.f[0] = ld32(fxa, c);
            P.f[1] = ld32(fxa, c - 1u);
            P.f[2] = ld32(fya, c);
            P.f[3] = ld32(fya, c - sx);
            P.f[4] = ld32(fza, c);
            P.f[5] = ld32(fza, c - sxy);
        }
        if(DIV)
        {
            const int ku = min(kk + 1, g.nz - 1);
            if(own(ku) == ROW_MIXED) P.au = ld32(aiia, coff + sxy * (unsigned)ku);
            if(has_halo && S.c[hrow][kk - zk0] == ROW_MIXED) P.ah = ld32(aiia, hoff + sxy * (unsigned)kk);
        }
    };
    auto fetch = [&](int kk, In& P) {
        fetch_raw(kk, P);
        fetch_mixed(kk, P);
    };
    V xd = V(0), xc = V(0), auxc = V(0);
    int t = tw.t;
    bool v1 = false;   // D = 2: the buffer after the current one holds plane k + 1
    // start of a column run at tile t
    auto start = [&](In& P0, In& P1) {
        const int col = t / tw.s.nbz;
        k = t - col * tw.s.nbz;
        const int by = col / tw.s.nbx, bx = col - by * tw.s.nbx;
        kend = min(tw.s.nbz, k + (tw.t1 - t));
        zk0 = max(k - 1, 0);
        const int i0 = bx * TX, j0 = by * TY;
        const int i = i0 + lane, j = j0 + row;
        in = i < g.nx && j < g.ny;
        ic = min(i, g.nx - 1);
        jc = min(j, g.ny - 1);
        coff = (unsigned)(g.base + ic + g.sx * jc);
        int ih = i0 + hi, jh = j0 + hj;
        hval = has_halo && ih >= 0 && ih < g.nx && jh >= 0 && jh < g.ny;
        ih = max(0, min(ih, g.nx - 1));
        jh = max(0, min(jh, g.ny - 1));
        hoff = (unsigned)(g.base + ih + g.sx * jh);
        // the operand's first loads are in flight while the tables are staged
        const unsigned c = coff + sxy * (unsigned)k;
        const R rc = raw(c), rd = raw(k > 0 ? c - sxy : c);
        V ac = V(0), ad = V(0);
        if(LOAD)
        {
            ac = ld32(aiia, c);
            ad = ld32(aiia, k > 0 ? c - sxy : c);
        }
        fetch_raw(k, P0);
        // the classes of the run's planes, one row per wavefront and load, all in flight together:
        // with 14 x 66 entries dealt to the threads in turn an item of one plane took as long to
        // set up as one of 64
        const int kl = min(kend, g.nz - 1), np = kl - zk0 + 1;
        constexpr int RW = (CROWS + TY - 1) / TY;
        auto row_of = [&](int rr) {
            const int jr = rr < TY ? j0 + rr : rr == TY ? j0 - 1 : rr == TY + 1 ? j0 + TY : j0 + (rr - 2) % TY;
            const int br = rr < TY + 2 ? bx : rr < 2 * TY + 2 ? bx - 1 : bx + 1;
            const int jq = max(0, min(jr, g.ny - 1)), bq = max(0, min(br, tw.s.nbx - 1));
            return T.cls + ((long)bq * g.ny + jq) * g.nz + zk0;
        };
        unsigned char rcl[RW];
        #pragma unroll
        for(int m = 0; m < RW; ++m) rcl[m] = row_of(min(row + m * TY, CROWS - 1))[min(lane, np - 1)];
        __syncthreads();   // the last run's entries have been read
        for(int q = h; q < 4 * np; q += NT)
        {
            const int e = 2 * (((q >> 1) & 1) * g.nz + zk0 + (q >> 2)) + (q & 1);
            S.z[q >> 2][q & 3] = T.ct[2][e];
            if constexpr(sizeof(V) == 4) S.z32[q >> 2][q & 3] = T.ct32[2][e];
        }
        #pragma unroll
        for(int m = 0; m < RW; ++m)
        {
            const int rr = row + m * TY;
            if(rr >= CROWS) continue;
            if(lane < np) S.c[rr][lane] = rcl[m];
            if(lane + TX < np) S.c[rr][lane + TX] = row_of(rr)[lane + TX];
        }
        if(h < TX)
            S.ax[h] = axis_factor(g, op, 0, min(i0 + h, g.nx - 1));
        else if(h < TX + TY)
            S.ay[h - TX] = axis_factor(g, op, 1, min(j0 + h - TX, g.ny - 1));
        else if(h >= 2 * TX && h < 2 * TX + np)
            S.az[h - 2 * TX] = axis_factor(g, op, 2, zk0 + h - 2 * TX);
        __syncthreads();
        keyC = keyN = keyH = 0;
        V d;
        xd = xc = auxc = V(0);
        const int cc = own(k), cd = own(max(k - 1, 0));
        if(DIV && cc == ROW_MIXED) ac = ld32(aiia, c);
        if(DIV && cd == ROW_MIXED) ad = ld32(aiia, k > 0 ? c - sxy : c);
        fetch_mixed(k, P0);
        v1 = false;
        if constexpr(D == 2)
            if(k + 1 < kend)
            {
                fetch(k + 1, P1);
                v1 = true;
            }
        if(k > 0)
        {
            const V x = val(rd, own_a(k - 1, cd, ad), d);
            xd = in ? x : V(0);
        }
        const V x = val(rc, own_a(k, cc, ac), auxc);
        xc = in ? x : V(0);
    };
    int buf = 0;
    // one plane: cur is plane k, nf receives plane k + D; n1: plane k + 1 (D = 2); false at the end
    auto step = [&](In& cur, In& n1, In& nf) -> bool {
        V* const P = &S.x[buf][0][0];
        const int at = (row + 1) * (TX + 2) + lane + 1;
        P[at] = xc;
        if(has_halo)
        {
            V a = cur.ah, d;
            const int ch = S.c[hrow][k - zk0];
            if(DIV && ch != ROW_MIXED)
            {
                if(ch != keyH)
                {
                    s4H = sum_xy(ch, (int)((hoff - (unsigned)g.base) % sx), (int)((hoff - (unsigned)g.base) / sx));
                    keyH = ch;
                }
                a = jacobi(s4H, ch, k);
            }
            const V hv = val(cur.h, a, d);
            P[hslot] = hval ? hv : V(0);
        }
        bool vf = false;
        if(k + D < kend && (D == 1 || v1))
        {
            fetch(k + D, nf);
            vf = true;
        }
        __syncthreads();
        V auxu = V(0), xu = V(0);
        if(k + 1 < g.nz)
        {
            const V a = own_a(k + 1, DIV ? own(k + 1) : 0, cur.au);
            const V x = val(cur.xu, a, auxu);
            xu = in ? x : V(0);
        }
        const int c = own(k);
        V Ax;
        if(c == ROW_MIXED)
        {
            const Coef<V> cf = poisson_coef(g,
                                            coupling_axes(op, cur.f[0], cur.f[1], cur.f[2], cur.f[3], cur.f[4], cur.f[5],
                                                          S.ax[lane], S.ay[row], S.az[k - zk0]),
                                            ic, jc, k);
            Ax = coef_apply(cf, true, xc, P[at + 1], P[at - 1], P[at + TX + 2], P[at - TX - 2], xu, xd);
        }
        else
        {
            const int ey = 2 * ((c - 1) * g.ny + jc);
            V yp, ym, zp, zm;
            if constexpr(sizeof(V) == 8)
            {
                yp = ((CDouble*)T.ct[1])[ey];
                ym = ((CDouble*)T.ct[1])[ey + 1];
                zp = S.z[k - zk0][2 * c - 2];
                zm = S.z[k - zk0][2 * c - 1];
            }
            else
            {
                yp = ((CFloat*)T.ct32[1])[ey];
                ym = ((CFloat*)T.ct32[1])[ey + 1];
                zp = S.z32[k - zk0][2 * c - 2];
                zm = S.z32[k - zk0][2 * c - 1];
            }
            if(c != keyC)
            {
                const Pair<V> px = class_pair<V>(T, 0, g.nx, c, ic);
                s4 = px.p + px.m + yp + ym;
                cn = ic == g.nx - 1 ? V(0) : -px.p;
                cs = ic == 0 ? V(0) : -px.m;
                keyC = c;
            }
            const Coef<V> cf{s4 + zp + zm,
                             cn,
                             cs,
                             jc == g.ny - 1 ? V(0) : -yp,
                             jc == 0 ? V(0) : -ym,
                             k == g.nz - 1 ? V(0) : -zp,
                             k == 0 ? V(0) : -zm};
            Ax = coef_apply(cf, true, xc, P[at + 1], P[at - 1], P[at + TX + 2], P[at - TX - 2], xu, xd);
        }
        if(in) post(coff + sxy * (unsigned)k, Ax, auxc, cur.e);
        buf ^= 1;
        ++t;
        if(t >= tw.t1) return false;
        if(k + 1 < kend)
        {
            ++k;
            xd = xc;
            xc = xu;
            auxc = auxu;
            v1 = vf;
        }
        else if constexpr(D == 1)
            start(nf, n1);
        else
            start(n1, nf);
        return true;
    };
    if(t >= tw.t1) return;
    In X, Y;
    if constexpr(D == 1)
    {
        start(X, Y);
        #pragma unroll 1
        for(;;)
        {
            if(!step(X, Y, Y)) break;
            if(!step(Y, X, X)) break;
        }
    }
    else
    {
        In Z;
        start(X, Y);
        #pragma unroll 1
        for(;;)
        {
            if(!step(X, Y, Z)) break;
            if(!step(Y, Z, X)) break;
            if(!step(Z, X, Y)) break;
        }
    }
}

// Elementwise pass over an item of a class-walked tank with aii from the row classes (mixed
// rows load it): load(u, c) and use(u, c, aii) for each cell, U tiles at a time so that their
// loads are in flight together; the cells of a thread come in tile order.
template<class V, int U, class Load, class Use>
__device__ __forceinline__ void class_cells(CTank& T, const DevGrid& g, const TileWalk& tw, Load load, Use use)
{
    const V* aii;
    if constexpr(sizeof(V) == 8)
        aii = T.f[A_AII];
    else
        aii = T.s[S_AII];
    const int lane = threadIdx.x & 63, row = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int t = tw.t;
    #pragma unroll 1
    while(t < tw.t1)
    {
        // a run of at most 64 tiles of one column
        const int col = t / tw.s.nbz, k0 = t - col * tw.s.nbz, by = col / tw.s.nbx, bx = col - by * tw.s.nbx;
        const int k1 = min(tw.s.nbz, k0 + (tw.t1 - t));
        const int i = bx * TX + lane, j = by * TY + row;
        const bool in = i < g.nx && j < g.ny;
        const int ic = min(i, g.nx - 1), jc = min(j, g.ny - 1);
        const unsigned c0 = (unsigned)(g.base + ic + g.sx * jc);
        RowClasses own;
        own.open(T.cls + ((long)bx * g.ny + jc) * g.nz, g.nz, k0);
        int key = 0;
        double s4 = 0.0;
        #pragma unroll 1
        for(int k = k0; k < k1; k += U)
        {
            V ae[U];
            int cl[U];
            double zs[U][2];
            #pragma unroll
            for(int u = 0; u < U; ++u)
            {
                const int kk = min(k + u, k1 - 1);
                const unsigned c = c0 + (unsigned)(g.sxy * kk);
                cl[u] = own.at(kk);
                load(u, c);
                CDouble* const z = (CDouble*)T.ct[2] + 2 * (max(cl[u] - 1, 0) * g.nz + kk);
                zs[u][0] = z[0];
                zs[u][1] = z[1];
                ae[u] = V(0);
                if(cl[u] == ROW_MIXED) ae[u] = ld32(aii, c);
            }
            #pragma unroll
            for(int u = 0; u < U; ++u)
            {
                if(k + u >= k1) break;
                if(cl[u] != ROW_MIXED)
                {
                    if(cl[u] != key)
                    {
                        const Pair<double> px = class_pair64(T, 0, g.nx, cl[u], ic), py = class_pair64(T, 1, g.ny, cl[u], jc);
                        s4 = px.p + px.m + py.p + py.m;
                        key = cl[u];
                    }
                    ae[u] = (V)(-1.0 / ((s4 + zs[u][0] + zs[u][1]) + 1e-19));
                }
                if(in) use(u, c0 + (unsigned)(g.sxy * (k + u)), ae[u]);
            }
        }
        t += k1 - k0;
    }
}

// Row walk of the 2-D (x-z) solver kernels: the item is a run of 64 x 1 x 4 tiles of one
// x-column (z rows k0 .. k0 + 4 cpt); wave w of the block walks rows
// [k0 + w cpt, k0 + (w+1) cpt) up z with the operand of rows k-1, k, k+1 in registers;
// the i+-1 neighbours come from the neighbouring lanes (wavefront shuffles), lanes 0 and
// 63 load the one outside the wavefront.  No block barrier until the item's reduction.
// The y couplings of a 2-D tank are multiplied by 0 in the operator, so they are 0 here.
__device__ __forceinline__ bool row_walk_ok(const DevGrid& g, const TileWalk& tw)
{
    return g.jdir == 0 && tw.s.ty == 1 && tw.s.tz == 4 && tw.t / tw.s.nbz == (tw.t1 - 1) / tw.s.nbz;
}

template<class V>
__device__ __forceinline__ V shfl_dn1(V x)
{
    return __shfl_down(x, 1, 64);
}
template<class V>
__device__ __forceinline__ V shfl_up1(V x)
{
    return __shfl_up(x, 1, 64);
}

template<class V, class Op, class Raw, class Val, class Pre, class Post>
__device__ __forceinline__ void row_walk(const DevGrid& g, const Op& op, const TileWalk& tw, Raw raw, Val val, Pre pre,
                                         Post post)
{
    using AF = AxisFactor<Op>;
    const V* __restrict__ fxa = face_x(op);
    const V* __restrict__ fza = face_z(op);
    const int lane = threadIdx.x & (TX - 1), wave = threadIdx.x >> 6;
    const int col = tw.t / tw.s.nbz;
    const int bz0 = tw.t - col * tw.s.nbz;
    const int per = tw.t1 - tw.t;                 // rows per wave (4 waves, 4 rows per tile)
    const int k0 = bz0 * 4 + wave * per;
    const int k1 = min(k0 + per, g.nz);
    const int i = col * TX + lane;
    const bool in = i < g.nx;
    const int ic = min(i, g.nx - 1);
    const unsigned c0 = (unsigned)(g.base + ic);   // (ic, 0, 0)
    const unsigned sxy = (unsigned)g.sxy;
    const AF ax = axis_factor(g, op, 0, ic);
    if(k0 >= k1) return;
    V d, auxc = V(0);
    unsigned c = c0 + (unsigned)k0 * sxy;
    V xd = k0 > 0 ? val(raw(c - sxy), d) : V(0);
    V xc = val(raw(c), auxc);
    V fzd = ld32(fza, c - sxy);
    #pragma unroll 1
    for(int k = k0; k < k1; ++k, c += sxy)
    {
        V auxu = V(0);
        const V xu = k + 1 < g.nz ? val(raw(c + sxy), auxu) : V(0);
        const auto e = pre(c);
        const V f0 = ld32(fxa, c), f4 = ld32(fza, c);
        // the -x face and the x neighbours: from the neighbouring lanes, the lanes at the
        // wavefront's edges load theirs
        V f1 = shfl_up1(f0), xs = shfl_up1(xc), xn = shfl_dn1(xc);
        if(lane == 0)
        {
            f1 = ld32(fxa, c - 1u);
            xs = i > 0 ? val(raw(c - 1u), d) : V(0);
        }
        if(lane == TX - 1) xn = i + 1 < g.nx ? val(raw(c + 1u), d) : V(0);
        if(in)
        {
            const AF az = axis_factor(g, op, 2, k);
            post(c, stencil5(g, coupling_xz(op, f0, f1, f4, fzd, ax, az), xc, xn, xs, xu, xd, i, k), auxc, e);
        }
        xd = xc;
        xc = xu;
        auxc = auxu;
        fzd = f4;
    }
}

__device__ __forceinline__ bool class_walk_ok(CTank& T)
{
    return T.g.jdir == 1 && T.shape.ty == TY && T.shape.tz == 1;
}

// restart / initial residual of the iterated precision: r = b - A x, r0 = p = r,
// ph = aii p (restart label, bicgstab_ijk.cpp:136-148)
template<class V, class Op>
__device__ __forceinline__ void restart_body(const DevGrid& g, const Op& op, const BiVec<V>& v, const TileWalk& tw,
                                             double& rr)
{
    #pragma unroll 1
    for(int t = tw.t; t < tw.t1; ++t)
    {
        int i, j, k;
        long c;
        if(!tile_cell(g, tw, t, i, j, k, c)) continue;
        const CouplingV<V> cq = coupling_of(g, op, c, i, j, k);
        const V rv = v.rhs[c] - (apply_A(g, cq, (const V*)v.x, c, i, j, k));
        v.r[c] = rv;
        v.r0[c] = rv;
        v.p[c] = rv;
        v.ph[c] = rv * v.aii[c];
        rr += double(rv) * double(rv);
    }
}

__global__ void kb_setup(TankSet b, double stop, int maxiter, int mixed, double delta)
{
    const int tk = blockIdx.x * blockDim.x + threadIdx.x;
    if(tk >= b.n) return;
    CTank& T = tank_at(b, tk);
    BiState* st = T.st;
    st->r_j = st->norm_r0 = st->alpha = st->w = st->beta = 0.0;
    st->sigma = st->norm_vj = st->norm_rj = st->norm_sj = st->w1 = st->w2 = st->r_j1 = 0.0;
    st->residual = 1.0e9;
    st->stop = stop;
    st->iter = 0;
    st->maxiter = maxiter;
    st->done = 0;
    st->mode = 0;
    st->branch = 0;
    st->mixed = mixed;
    st->r_j_prev = st->rmax = st->res0 = st->rr = 0.0;
    st->delta = delta;
    st->pending = 0;
    st->nru = 0;
    st->buf = 0;
    st->chip_fail = 0;
    st->ncell = (long)T.g.nx * T.g.ny * T.g.nz;
}

template<class V>
__global__ void __launch_bounds__(NT, OCC_A64) kb_bicg_init(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        double vals[1] = {0.0};
        restart_body(g, Prec<V>::op(T), Prec<V>::vec(T, x, rhs), item_walk(T, b, q), vals[0]);
        block_sum_to<1>(vals, b.partials + (size_t)item_slot(T, b, q));
    }
}

__global__ void kb_fin_init(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    double tot[1];
    tank_totals<1>(T, b, tot);
    if(threadIdx.x == 0)
    {
        st->r_j = tot[0];
        st->rr = tot[0];
        st->norm_r0 = sqrt(tot[0]);
        // a negative stop asks for ||r||_2 / N < |stop| * ||b - A x0||_2 / N
        if(st->stop < 0.0) st->stop = -st->stop * sqrt(tot[0]) / double(st->ncell);
        if(!((st->residual >= st->stop) && (st->iter < st->maxiter))) st->done = 1;
        st->mode = 2;
    }
}

// start of an iteration: the pending restart, or p = r + beta (p - w v), ph = aii p
// (bicgstab_ijk.cpp:234-235 and precon_solve).  ALL: the class-walked tanks of the set too.
template<class V, bool ALL>
__global__ void __launch_bounds__(NT, OCC_A64) kb_bicg_p(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items_spread(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 2 || (!ALL && class_walk_ok(T)))
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<V> v = Prec<V>::vec(T, x, rhs);
        const TileWalk tw = item_walk(T, b, q);
        if(st->mode == 1)
        {
            double vals[1] = {0.0};
            restart_body(g, Prec<V>::op(T), v, tw, vals[0]);
            block_sum_to<1>(vals, b.partials_ru + (size_t)item_slot(T, b, q));
            continue;
        }
        const V beta = (V)st->beta, w = (V)st->w;
        const V* __restrict__ r = v.r;
        const V* __restrict__ vv = v.v;
        const V* __restrict__ aii = v.aii;
        V* __restrict__ p = v.p;
        V* __restrict__ ph = v.ph;
        // independent tiles: unrolled so that several tiles' loads are in flight
        #pragma unroll 4
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            const V pn = r[c] + beta * (p[c] - w * vv[c]);
            p[c] = pn;
            ph[c] = pn * aii[c];
        }
    }
}

// kb_bicg_p of the class-walked tanks, aii from the row classes: 40 bytes per cell (r, p, v / p,
// ph)
__global__ void __launch_bounds__(NT, OCC_CX) kb_class_p(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b, 0, b.pw_items); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 2)
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<double> v = Prec<double>::vec(T, x, rhs);
        const TileWalk tw = class_item(T, b, q);
        if(st->mode == 1)
        {
            double vals[1] = {0.0};
            restart_body(g, Prec<double>::op(T), v, tw, vals[0]);
            block_sum_to<1>(vals, b.partials_ru + (size_t)tw.gi);
            continue;
        }
        const double beta = st->beta, w = st->w;
        const double* __restrict__ r = v.r;
        const double* __restrict__ vv = v.v;
        double* __restrict__ p = v.p;
        double* __restrict__ ph = v.ph;
        constexpr int U = 4;
        double rr[U], pp[U], ve[U];
        class_cells<double, U>(
            T, g, tw,
            [&](int u, unsigned c) {
                rr[u] = ld32(r, c);
                pp[u] = ld32(p, c);
                ve[u] = ld32(vv, c);
            },
            [&](int u, unsigned c, double a) {
                const double pn = rr[u] + beta * (pp[u] - w * ve[u]);
                st32(p, c, pn);
                st32(ph, c, pn * a);
            });
    }
}

// totals of a restart of the explicit-operator solve (km_p): ++solveriter, residual = |r|/N
// (bicgstab_ijk.cpp:183-191); the Poisson solve's restarts are finalized by its v phase
__global__ void kb_fin_p(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    if(st->done || st->mode != 1) return;
    double tot[1];
    tank_totals<1>(T, b, tot);
    if(threadIdx.x == 0)
    {
        restart_store(st, tot[0]);
    }
}

// v = A ph; sigma = (v, r0), |v|^2 (bicgstab_ijk.cpp:151-160).  |r|^2 of the same loop is
// the square norm of the residual the x phase (or the restart) has just formed and summed:
// kb_fin_v takes it from the state instead of reading r again here.
// Tanks without a class walk; kb_class_v takes the others.
template<class V>
__global__ void __launch_bounds__(NT, sizeof(V) == 4 ? OCC_FULL : OCC_A64) kb_bicg_v(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items_of<false>(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 3 || class_walk_ok(T))
        {
            skip_tank(q, b);
            continue;
        }
        // mode 1: this iteration's p phase has restarted the tank (ph = aii r, fresh)
        if(st->mode == 1
           && (sizeof(V) != 8
               || __builtin_amdgcn_readfirstlane(restart_done(b.partials_ru + (size_t)T.item0, T.shape.nitems, st))))
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<V> bv = Prec<V>::vec(T, x, rhs);
        const typename Prec<V>::Op op = Prec<V>::op(T);
        const TileWalk tw = item_walk(T, b, q);
        double vals[3] = {0.0, 0.0, 0.0};
        const V* __restrict__ ph = bv.ph;
        const V* __restrict__ r0 = bv.r0;
        V* __restrict__ vo = bv.v;
        auto epilogue = [&](long c, V v) {
            vo[c] = v;
            const double vd = v;
            vals[0] += vd * double(r0[c]);
            vals[1] += vd * vd;
        };
        if(row_walk_ok(g, tw))
        {
            struct EpiIn
            {
                V r0;
            };
            row_walk<V>(
                g, op, tw, [&](unsigned cc) { return ld32(ph, cc); }, [](V x, V&) { return x; },
                [&](unsigned c) { return EpiIn{ld32(r0, c)}; },
                [&](unsigned c, V Ax, V, const EpiIn& e) {
                    st32(vo, c, Ax);
                    const double vd = Ax;
                    vals[0] += vd * double(e.r0);
                    vals[1] += vd * vd;
                });
        }
        else
            #pragma unroll 1
            for(int t = tw.t; t < tw.t1; ++t)
            {
                int i, j, k;
                long c;
                if(!tile_cell(g, tw, t, i, j, k, c)) continue;
                const CouplingV<V> cq = coupling_of(g, op, c, i, j, k);
                epilogue(c, apply_A(g, cq, ph, c, i, j, k));
            }
        block_sum_to<3>(vals, b.partials + (size_t)item_slot(T, b, q) * 3);
    }
}

// v = A ph of the class-walked tanks (24 bytes per cell: ph, r0 / v).  The p update stays a
// pass of its own (kb_class_p): fused into this walk, as the FP32 v phase has it, the FP64
// operand needs r, p, v and aii at every stencil point, and the walk spills at 4 blocks per CU.
__global__ void __launch_bounds__(NT, OCC_PW) kb_class_v(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items_of<true>(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 3 || !class_walk_ok(T))
        {
            skip_tank(q, b);
            continue;
        }
        // mode 1: this iteration's p phase has restarted the tank (ph = aii r, fresh)
        if(st->mode == 1
           && __builtin_amdgcn_readfirstlane(restart_done(b.partials_ru + (size_t)T.item0, T.shape.nitems, st)))
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<double> bv = Prec<double>::vec(T, x, rhs);
        const TileWalk tw = class_item(T, b, q);
        double vals[3] = {0.0, 0.0, 0.0};
        const double* __restrict__ ph = bv.ph;
        const double* __restrict__ r0 = bv.r0;
        double* __restrict__ vo = bv.v;
        struct EpiIn
        {
            double r0;
        };
        class_walk<double, AII_NONE, 2>(
            T, g, tw, [&](unsigned cc) { return ld32(ph, cc); }, [](double z, double, double&) { return z; },
            [&](unsigned c) { return EpiIn{ld32(r0, c)}; },
            [&](unsigned c, double Ax, double, const EpiIn& e) {
                st32(vo, c, Ax);
                vals[0] += Ax * e.r0;
                vals[1] += Ax * Ax;
            });
        block_sum_to<3>(vals, b.partials + (size_t)tw.gi * 3);
    }
}

// Start of an FP32 iteration fused with v = A ph (mixed precision): the pending
// x64 += x32 after a reliable update, and, in mode 0, p = r + beta (p - w v), ph = aii p
// evaluated at every stencil point (the FP32 p update, bicgstab_ijk.cpp:234-235 with
// precon_solve) so that no separate p pass runs; in mode 2 (p, ph fresh from the start
// or a restart) ph is read.  The new p and v go to the other half of their double
// buffers (kb_fin_v swaps the halves), ph is written at the cell for the x phase;
// (v, r0), |v|^2, |r|^2 as kb_bicg_v.  A tank still in mode 1 / 3 has just had its
// reliable-update phase: the walk runs on that phase's outcome (RuNext).
template<bool PW>
__global__ void __launch_bounds__(NT, PW ? OCC_PW : OCC_FULL) kb_mix_v(TankSet b, int x)
{
    #pragma unroll 1
    for(ItemIter q = set_items_of<PW>(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || class_walk_ok(T) != PW)
        {
            skip_tank(q, b);
            continue;
        }
        int mode = st->mode, pend = st->pending;
        float beta = (float)st->beta;
        if(mode == 1 || mode == 3)
        {
            // the reliable-update phase ran last: its outcome from its sums (every thread
            // holds the same totals; the decisions are made scalar)
            const unsigned long long o = ru_outcome(b.partials_ru + (size_t)T.item0 * 2, T.shape.nitems, st);
            const int om = __builtin_amdgcn_readfirstlane((int)(o >> 32));
            if(om == 4)
            {
                skip_tank(q, b);
                continue;
            }
            mode = om;
            beta = __builtin_bit_cast(float, (unsigned)o);
            pend = 1;
        }
        const int upd = mode == 0, hsel = st->buf;
        const float w = (float)st->w;
        const SolverOp32 op = Prec<float>::op(T);
        const float* __restrict__ r = T.s[S_R];
        const float* __restrict__ r0 = T.s[S_R0];
        const float* __restrict__ aii = T.s[S_AII];
        const float* __restrict__ pc = T.s[hsel ? S_P2 : S_P];
        const float* __restrict__ vc = T.s[hsel ? S_V2 : S_V];
        float* __restrict__ pn = T.s[hsel ? S_P : S_P2];
        float* __restrict__ vn = T.s[hsel ? S_V : S_V2];
        float* __restrict__ ph = T.s[S_PH];
        float* __restrict__ x32 = T.s[S_X];
        double* __restrict__ x64 = T.f[x];
        const TileWalk tw = PW ? class_item(T, b, q) : item_walk(T, b, q);
        double vals[3] = {0.0, 0.0, 0.0};
        if constexpr(PW)
        {
            // the operator and aii from the row classes; ph is not stored, the x phase forms it
            struct EpiIn
            {
                float r0, r;
            };
            struct Rp
            {
                float r, p, v;
            };
            auto cpre = [&](unsigned c) { return EpiIn{ld32(r0, c), ld32(r, c)}; };
            auto cpost = [&](unsigned c, float Ax, float pv, const EpiIn& e) {
                st32(vn, c, Ax);
                st32(pn, c, pv);
                if(pend)
                {
                    st32(x64, c, ld32(x64, c) + (double)ld32(x32, c));
                    st32(x32, c, 0.0f);
                }
                const double vd = Ax, rc = e.r;
                vals[0] += vd * double(e.r0);
                vals[1] += vd * vd;
                vals[2] += rc * rc;
            };
            if(upd)
                class_walk<float, AII_LOAD, 2>(
                    T, g, tw, [&](unsigned cc) { return Rp{ld32(r, cc), ld32(pc, cc), ld32(vc, cc)}; },
                    [&](const Rp& z, float a, float& pv) {
                        pv = z.r + beta * (z.p - w * z.v);
                        return pv * a;
                    },
                    cpre, cpost);
            else
                class_walk<float, AII_LOAD, 2>(
                    T, g, tw, [&](unsigned cc) { return ld32(pc, cc); },
                    [&](float z, float a, float& pv) {
                        pv = z;
                        return z * a;
                    },
                    cpre, cpost);
            block_sum_to<3>(vals, b.partials + (size_t)tw.gi * 3);
            continue;
        }
        struct Epi
        {
            float r0, r, a, p;
        };
        auto pre = [&](unsigned c) { return Epi{ld32(r0, c), ld32(r, c), ld32(aii, c), upd ? 0.0f : ld32(pc, c)}; };
        // aux: the new p at the centre (mode 0)
        auto post = [&](unsigned c, float Ax, float pnew, const Epi& e) {
            st32(vn, c, Ax);
            if(upd)
            {
                st32(pn, c, pnew);
                st32(ph, c, pnew * e.a);
            }
            else
                st32(pn, c, e.p);
            if(pend)
            {
                st32(x64, c, ld32(x64, c) + (double)ld32(x32, c));
                st32(x32, c, 0.0f);
            }
            const double vd = Ax, rc = e.r;
            vals[0] += vd * double(e.r0);
            vals[1] += vd * vd;
            vals[2] += rc * rc;
        };
        struct Rp
        {
            float r, p, v, a;
        };
        auto raw_u = [&](unsigned cc) { return Rp{ld32(r, cc), ld32(pc, cc), ld32(vc, cc), ld32(aii, cc)}; };
        auto val_u = [&](const Rp& z, float& pnew) {
            pnew = z.r + beta * (z.p - w * z.v);
            return pnew * z.a;
        };
        auto raw_f = [&](unsigned cc) { return ld32(ph, cc); };
        auto val_f = [](float z, float&) { return z; };
        if(row_walk_ok(g, tw))
        {
            if(upd)
                row_walk<float>(g, op, tw, raw_u, val_u, pre, post);
            else
                row_walk<float>(g, op, tw, raw_f, val_f, pre, post);
        }
        else
            #pragma unroll 1
            for(int t = tw.t; t < tw.t1; ++t)
            {
                int i, j, k;
                long c;
                if(!tile_cell(g, tw, t, i, j, k, c)) continue;
                const CouplingV<float> cq = coupling_of(g, op, c, i, j, k);
                float pnew = 0.0f, d;
                float Ax;
                if(upd)
                {
                    const float phc = val_u(raw_u((unsigned)c), pnew);
                    Ax = apply_A_fn(g, cq, [&](long cc) { return cc == c ? phc : val_u(raw_u((unsigned)cc), d); }, c,
                                    i, j, k);
                }
                else
                    Ax = apply_A(g, cq, (const float*)ph, c, i, j, k);
                post((unsigned)c, Ax, pnew, pre((unsigned)c));
            }
        block_sum_to<3>(vals, b.partials + (size_t)tw.gi * 3);
    }
}

// alpha and the restart tests (bicgstab_ijk.cpp:162-191); rr_state: |r|^2 from the state
// (kb_bicg_v), else the phase's third sum (kb_mix_v, km_v).  A mixed-precision tank in
// mode 1 / 3 first takes the outcome of its reliable-update phase, as kb_mix_v did.
__global__ void kb_fin_v(TankSet b, int rr_state)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    // the partials' loads go out together with the state's (one memory latency, not two)
    const int done = st->done, mode = st->mode;
    const bool ru = st->mixed && (mode == 1 || mode == 3);
    // the FP64 Poisson solve (rr_state): mode 1 is the restart of this iteration's p phase
    const bool rs = rr_state && mode == 1;
    double tot[3];
    tank_totals<3>(T, b, tot);
    double rtot[2];
    if(ru && !done) tank_totals_ru(T, b, rtot);
    double stot[1];
    if(rs && !done) sum_partials<1>(b.partials_ru + (size_t)T.item0, T.shape.nitems, stot);
    if(done || (!ru && !rs && (mode == 1 || mode == 3))) return;
    if(threadIdx.x == 0)
    {
        if(ru)
        {
            const RuNext n = ru_next(st, rtot);
            ru_store(st, n);
            if(n.done) return;
        }
        if(rs)
        {
            restart_store(st, stot[0]);
            if(st->done) return;
        }
        v_store(st, tot[0], tot[1], rr_state ? st->rr : tot[2], st->mixed);
    }
}

// s = r - alpha v, sh = aii s, t = A sh; (t,s), (t,t), (s,s) (bicgstab_ijk.cpp:193-221)
template<class V, bool PW>
__global__ void __launch_bounds__(NT, PW ? OCC_PW : (sizeof(V) == 4 ? OCC_FULL : OCC_A64)) kb_bicg_t(TankSet b, int x,
                                                                                               int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items_of<PW>(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 1 || st->mode == 3 || class_walk_ok(T) != PW)
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<V> bv = Prec<V>::vec(T, x, rhs);
        const typename Prec<V>::Op op = Prec<V>::op(T);
        const TileWalk tw = PW ? class_item(T, b, q) : item_walk(T, b, q);
        double vals[3] = {0.0, 0.0, 0.0};
        const V alpha = (V)st->alpha;
        const V* __restrict__ r = bv.r;
        const V* __restrict__ v = bv.v;
        const V* __restrict__ a = bv.aii;
        V* __restrict__ to = bv.t;
        auto epilogue = [&](long c, V t, V s) {
            to[c] = t;
            const double td = t, sd = s;
            vals[0] += td * sd;
            vals[1] += td * td;
            vals[2] += sd * sd;
        };
        auto shv = [&](long cc, V& sv) {
            sv = r[cc] - alpha * v[cc];
            return sv * a[cc];
        };
        if constexpr(PW)
        {
            // t into the half of v's buffer that is not current
            if constexpr(sizeof(V) == 4) to = T.s[st->buf ? S_V : S_V2];
            struct Rin
            {
                V r, v;
            };
            class_walk<V, sizeof(V) == 8 ? AII_CLASS : AII_LOAD, sizeof(V) == 8 ? 1 : 2>(
                T, g, tw, [&](unsigned cc) { return Rin{ld32(r, cc), ld32(v, cc)}; },
                [&](const Rin& q, V aq, V& sv) {
                    sv = q.r - alpha * q.v;
                    return sv * aq;
                },
                [](unsigned) { return NoEpi{}; },
                [&](unsigned c, V Ax, V s, const NoEpi&) {
                    st32(to, c, Ax);
                    const double td = Ax, sd = s;
                    vals[0] += td * sd;
                    vals[1] += td * td;
                    vals[2] += sd * sd;
                });
        }
        else if(row_walk_ok(g, tw))
        {
            struct Rin
            {
                V r, v, a;
            };
            row_walk<V>(
                g, op, tw, [&](unsigned cc) { return Rin{ld32(r, cc), ld32(v, cc), ld32(a, cc)}; },
                [&](const Rin& q, V& sv) {
                    sv = q.r - alpha * q.v;
                    return sv * q.a;
                },
                [](unsigned) { return NoEpi{}; },
                [&](unsigned c, V Ax, V sc, const NoEpi&) {
                    st32(to, c, Ax);
                    const double td = Ax, sd = sc;
                    vals[0] += td * sd;
                    vals[1] += td * td;
                    vals[2] += sd * sd;
                });
        }
        else
            #pragma unroll 1
            for(int tt = tw.t; tt < tw.t1; ++tt)
            {
                int i, j, k;
                long c;
                if(!tile_cell(g, tw, tt, i, j, k, c)) continue;
                const CouplingV<V> cq = coupling_of(g, op, c, i, j, k);
                V s;
                const V shc = shv(c, s);
                V dummy;
                const V t = apply_A_fn(g, cq, [&](long cc) { return cc == c ? shc : shv(cc, dummy); }, c, i, j, k);
                epilogue(c, t, s);
            }
        block_sum_to<3>(vals, b.partials + (size_t)tw.gi * 3);
    }
}

__global__ void kb_fin_t(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    const int done = st->done, mode = st->mode;
    double tot[3];
    tank_totals<3>(T, b, tot);
    if(done || mode == 1 || mode == 3) return;
    if(threadIdx.x == 0)
    {
        t_store(st, tot);
    }
}

// x and r updates, (r, r0), |r|^2 (bicgstab_ijk.cpp:223-268).  ALL: the class-walked tanks of the
// set too, for sets that hold both kinds: with a launch of its own for each kind these tanks ran
// one after the other, and the x phase of a served stream's mixed sets took 28 us instead of 17.
template<class V, bool ALL>
__global__ void __launch_bounds__(NT, OCC_FULL) kb_bicg_x(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items_spread(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        const bool cls = class_walk_ok(T);
        if(st->done || st->mode == 1 || st->mode == 3 || (!ALL && cls))
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<V> bv = Prec<V>::vec(T, x, rhs);
        const TileWalk tw = item_walk(T, b, q);
        const V alpha = (V)st->alpha, w = (V)st->w;
        const int branch = st->branch;
        // the FP32 class walk stores no ph, and t in the other half of v's buffer (kb_bicg_t)
        const bool form_ph = ALL && sizeof(V) == 4 && cls;
        double vals[2] = {0.0, 0.0};
        V* __restrict__ xv = bv.x;
        V* __restrict__ r = bv.r;
        const V* __restrict__ vv = bv.v;
        const V* __restrict__ aii = bv.aii;
        const V* __restrict__ pv = form_ph ? bv.p : bv.ph;
        const V* __restrict__ tv = bv.t;
        if constexpr(ALL && sizeof(V) == 4)
            if(cls) tv = T.s[st->buf ? S_V : S_V2];
        const V* __restrict__ r0 = bv.r0;
        // independent tiles (the dot sums keep their order): unrolled so that several
        // tiles' loads are in flight
        #pragma unroll 4
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            const V s = r[c] - alpha * vv[c];
            V ph = pv[c];
            if(form_ph) ph = ph * aii[c];
            V rn;
            if(branch)
            {
                const V sh = s * aii[c];
                xv[c] += alpha * ph + w * sh;
                rn = s - w * tv[c];
            }
            else
            {
                xv[c] += alpha * ph;
                rn = s;
            }
            r[c] = rn;
            const double rd = rn;
            vals[0] += rd * double(r0[c]);
            vals[1] += rd * rd;
        }
        block_sum_to<2>(vals, b.partials + (size_t)item_slot(T, b, q) * 2);
    }
}

// kb_bicg_x of the class-walked tanks, aii from the row classes: 64 bytes per cell in FP64 (x,
// ph, r, v, t, r0 / x, r); FP32 forms ph = aii p from the current p
template<class V>
__global__ void __launch_bounds__(NT, OCC_CX) kb_class_x(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b, 0, b.pw_items); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 1 || st->mode == 3)
        {
            skip_tank(q, b);
            continue;
        }
        const BiVec<V> bv = Prec<V>::vec(T, x, rhs);
        const TileWalk tw = class_item(T, b, q);
        const V alpha = (V)st->alpha, w = (V)st->w;
        const int branch = st->branch;
        double vals[2] = {0.0, 0.0};
        V* __restrict__ xv = bv.x;
        V* __restrict__ r = bv.r;
        const V* __restrict__ vv = bv.v;
        const V* __restrict__ pv = sizeof(V) == 8 ? bv.ph : bv.p;
        const V* __restrict__ tv = bv.t;
        if constexpr(sizeof(V) == 4) tv = T.s[st->buf ? S_V : S_V2];
        const V* __restrict__ r0 = bv.r0;
        constexpr int U = 4;
        V xx[U], pp[U], rr[U], ve[U], te[U], r0e[U];
        class_cells<V, U>(
            T, g, tw,
            [&](int u, unsigned c) {
                xx[u] = ld32(xv, c);
                pp[u] = ld32(pv, c);
                rr[u] = ld32(r, c);
                ve[u] = ld32(vv, c);
                te[u] = ld32(tv, c);
                r0e[u] = ld32(r0, c);
            },
            [&](int u, unsigned c, V a) {
                const V ph = sizeof(V) == 8 ? pp[u] : pp[u] * a, s = rr[u] - alpha * ve[u];
                V rn;
                if(branch)
                {
                    const V sh = s * a;
                    st32(xv, c, xx[u] + (alpha * ph + w * sh));
                    rn = s - w * te[u];
                }
                else
                {
                    st32(xv, c, xx[u] + alpha * ph);
                    rn = s;
                }
                st32(r, c, rn);
                const double rd = rn;
                vals[0] += rd * double(r0e[u]);
                vals[1] += rd * rd;
            });
        block_sum_to<2>(vals, b.partials + (size_t)tw.gi * 2);
    }
}

// beta, residual, iteration count; the mixed form asks for reliable updates instead of
// ending on the iterated residual
__global__ void kb_fin_x(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    const int done = st->done, mode = st->mode;
    double tot[2];
    tank_totals<2>(T, b, tot);
    if(done || mode == 1 || mode == 3) return;
    if(threadIdx.x == 0) x_store(st, tot);
}

// ------------------------------------------------------------------ mixed precision
// FP32 face conductances kx = 1/(rho_f DXP) (+x faces of the interior and the -1 layer,
// likewise y, z) and aii = -1/(M.p + 1e-19) from the FP64 diagonal, rounded once
__global__ void __launch_bounds__(NT) kb_coef32(TankSet b)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ rfx = T.f[A_RFX];
        const double* __restrict__ rfy = T.f[A_RFY];
        const double* __restrict__ rfz = T.f[A_RFZ];
        float* __restrict__ kx = T.s[S_KX];
        float* __restrict__ ky = T.s[S_KY];
        float* __restrict__ kz = T.s[S_KZ];
        float* __restrict__ aii = T.s[S_AII];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            const bool in = tile_cell(g, tw, t, i, j, k, c);
            if(!in) c = g.base;
            store_row_class(T, b, g, in, rfx[c], rfx[c - 1], rfy[c], rfy[c - g.sx], rfz[c], rfz[c - g.sxy], i, j, k);
            if(!in) continue;
            const int ip = i + MARGE, jp = j + MARGE, kp = k + MARGE;
            kx[c] = (float)(1.0 / (rfx[c] * g.DXP[ip]));
            ky[c] = (float)(1.0 / (rfy[c] * g.DYP[jp]));
            kz[c] = (float)(1.0 / (rfz[c] * g.DZP[kp]));
            if(i == 0) kx[c - 1] = (float)(1.0 / (rfx[c - 1] * g.DXP[ip - 1]));
            if(j == 0) ky[c - g.sx] = (float)(1.0 / (rfy[c - g.sx] * g.DYP[jp - 1]));
            if(k == 0) kz[c - g.sxy] = (float)(1.0 / (rfz[c - g.sxy] * g.DZP[kp - 1]));
            const Coupling cq = couplings(g, rfx, rfy, rfz, c, i, j, k);
            aii[c] = (float)(-1.0 / (diag_of(g, cq) + 1e-19));
        }
    }
}

// initial residual in FP64: r = b - A64 x64; r0 = p = r, ph = aii r, x32 = 0
__global__ void __launch_bounds__(NT, OCC_A64) kb_mix_start(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const SolverOp64 op = Prec<double>::op(T);
        const BiVec<float> v = Prec<float>::vec(T, x, rhs);
        const double* __restrict__ x64 = T.f[x];
        const double* __restrict__ b64 = T.f[rhs];
        const TileWalk tw = item_walk(T, b, q);
        double vals[2] = {0.0, 0.0};
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            const Coupling cq = coupling_of(g, op, c, i, j, k);
            const double rv = b64[c] - apply_A(g, cq, x64, c, i, j, k);
            const float r = (float)rv;
            v.r[c] = r;
            v.r0[c] = r;
            v.p[c] = r;
            v.ph[c] = r * v.aii[c];
            v.x[c] = 0.0f;
            vals[0] += rv * rv;
            vals[1] += double(r) * double(r);
        }
        block_sum_to<2>(vals, b.partials + (size_t)item_slot(T, b, q) * 2);
    }
}

__global__ void kb_fin_mix_start(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    double tot[2];
    tank_totals<2>(T, b, tot);
    if(threadIdx.x == 0)
    {
        const double rn = sqrt(tot[0]);
        st->r_j = tot[1];
        st->norm_r0 = sqrt(tot[1]);
        if(st->stop < 0.0) st->stop = -st->stop * rn / double(st->ncell);
        st->residual = rn / double(st->ncell);
        st->rmax = rn;
        st->res0 = rn;
        if(!((st->residual >= st->stop) && (st->iter < st->maxiter))) st->done = 1;
        st->mode = 2;
    }
}

// reliable update (mode 3) or restart (mode 1): r = b - A64 (x64 + x32) in FP64, rounded to
// the FP32 residual; a restart also sets r0 = p = r, ph = aii r
__global__ void __launch_bounds__(NT, OCC_A64) kb_mix_ru(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items_spread(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const BiState* st = T.st;
        if(st->done || (st->mode != 1 && st->mode != 3))
        {
            skip_tank(q, b);
            continue;
        }
        const int restart = st->mode == 1;
        const DevGrid g = T.g;
        const SolverOp64 op = Prec<double>::op(T);
        const BiVec<float> v = Prec<float>::vec(T, x, rhs);
        const double* __restrict__ x64 = T.f[x];
        const double* __restrict__ b64 = T.f[rhs];
        const float* __restrict__ x32 = v.x;
        const TileWalk tw = item_walk(T, b, q);
        double vals[2] = {0.0, 0.0};
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            const Coupling cq = coupling_of(g, op, c, i, j, k);
            const double rv =
                b64[c] - apply_A_fn(g, cq, [&](long cc) { return x64[cc] + (double)x32[cc]; }, c, i, j, k);
            const float r = (float)rv;
            v.r[c] = r;
            float r0v;
            if(restart)
            {
                v.r0[c] = r;
                v.p[c] = r;
                v.ph[c] = r * v.aii[c];
                r0v = r;
            }
            else
                r0v = v.r0[c];
            vals[0] += rv * rv;
            vals[1] += double(r0v) * double(r);
        }
        block_sum_to<2>(vals, b.partials_ru + (size_t)item_slot(T, b, q) * 2);
    }
}

// the outcome of a reliable-update phase that no v phase has taken yet (launched after the
// last iteration of a batch)
__global__ void kb_fin_mix_ru(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    BiState* st = T.st;
    if(st->done || (st->mode != 1 && st->mode != 3)) return;
    double tot[2];
    tank_totals_ru(T, b, tot);
    if(threadIdx.x == 0) ru_store(st, ru_next(st, tot));
}

// ------------------------------------------------------------------ explicit 7-diagonal operator
// bicgstab_ijk::start / bicgstab_ijk_2D::start (bicgstab_ijk.cpp:51-123, bicgstab_ijk_2D.cpp:
// 49-94) on a caller's matrix_diag: M.p, M.n, M.s, M.w, M.e, M.t, M.b and the right-hand
// side of every FLEXLOOP cell sit in field layout in TankDev::m[0..7], the solver's private
// x in m[8].  The FLEXLOOP cells of var (looping.h:55-57,159) on a box are i < nx - ulast,
// j < ny - vlast, k < nz - wlast (ulast / vlast / wlast = 1 for var 1 / 2 / 3, whose
// flag1..3 drop the last row of their grid; var 4, 5: every interior cell).  As in the
// reference, fillxvec copies the field into the private x on those cells only: its other
// interior cells keep what the calls of other vars left there (they are read by the
// restart's A x), its ghosts stay 0.  ph and sh are 0 outside the FLEXLOOP cells (the
// reference zeroes them after every solve, bicgstab_ijk.cpp:271-275), so their neighbours
// there contribute M * 0.0 and are not read.  The iteration is the state machine of the
// Poisson solve (the same finalize kernels); 3-D tanks use the 7-point product of
// matvec_std (bicgstab_ijk.cpp:296-310), 2-D tanks the 5-point one of bicgstab_ijk_2D.cpp:
// 308-320.
struct MatMask
{
    int ie, je, ke;    // exclusive ends of the FLEXLOOP box
};

__device__ __forceinline__ MatMask mat_mask(const DevGrid& g, int var)
{
    MatMask m;
    m.ie = g.nx - (var == 1 ? 1 : 0);
    m.je = g.ny - (var == 2 ? 1 : 0);
    m.ke = g.nz - (var == 3 ? 1 : 0);
    return m;
}

struct MatOp
{
    const double *p, *n, *s, *w, *e, *t, *b;
};

// the private x of the solve: m[8] for var 1..3 (psolv, the diffusion solves), m[9] for
// var 4, 5 (ppoissonsolv, a separate bicgstab_ijk object in the driver)
__device__ __forceinline__ int mat_xslot(int var) { return var <= 3 ? 8 : 9; }

__device__ __forceinline__ MatOp mat_op(CTank& T)
{
    MatOp o;
    o.p = T.m[0];
    o.n = T.m[1];
    o.s = T.m[2];
    o.w = T.m[3];
    o.e = T.m[4];
    o.t = T.m[5];
    o.b = T.m[6];
    return o;
}

// (A y)(c); MASK: y(cc) = yv(cc) inside the FLEXLOOP box and 0 outside it (ph, sh), else
// yv(cc) everywhere (the private x)
template<bool MASK, class YV>
__device__ __forceinline__ double mat_apply(const DevGrid& g, const MatOp& M, const MatMask& mk, YV yv, long c, int i,
                                            int j, int k)
{
    const double yn = !MASK || i + 1 < mk.ie ? yv(c + 1) : 0.0;
    const double ys = !MASK || i > 0 ? yv(c - 1) : 0.0;
    const double yt = !MASK || k + 1 < mk.ke ? yv(c + g.sxy) : 0.0;
    const double yb = !MASK || k > 0 ? yv(c - g.sxy) : 0.0;
    if(g.jdir == 1)
    {
        const double yw = !MASK || j + 1 < mk.je ? yv(c + g.sx) : 0.0;
        const double ye = !MASK || j > 0 ? yv(c - g.sx) : 0.0;
        return M.p[c] * yv(c) + M.n[c] * yn + M.s[c] * ys + M.w[c] * yw + M.e[c] * ye + M.t[c] * yt + M.b[c] * yb;
    }
    return M.p[c] * yv(c) + M.n[c] * yn + M.s[c] * ys + M.t[c] * yt + M.b[c] * yb;
}

__device__ __forceinline__ bool mat_cell(const DevGrid& g, const MatMask& mk, const TileWalk& tw, int t, int& i, int& j,
                                         int& k, long& c)
{
    return tile_cell(g, tw, t, i, j, k, c) && i < mk.ie && j < mk.je && k < mk.ke;
}

// restart label (bicgstab_ijk.cpp:134-148): r = rhs - A x, r0 = p = r, ph = aii p; on the
// first pass also precon_setup (:356-364), aii = -1/(M.p + 1e-19)
__device__ __forceinline__ void mat_restart(CTank& T, const DevGrid& g, const MatMask& mk, int var,
                                            const TileWalk& tw, bool setup, double& rr)
{
    const double* __restrict__ x = T.m[mat_xslot(var)];
    const MatOp M = mat_op(T);
    const double* __restrict__ rhs = T.m[7];
    double* __restrict__ r = T.f[A_R];
    double* __restrict__ r0 = T.f[A_R0];
    double* __restrict__ p = T.f[A_P];
    double* __restrict__ ph = T.f[A_PH];
    double* __restrict__ aii = T.f[A_AII];
    #pragma unroll 1
    for(int t = tw.t; t < tw.t1; ++t)
    {
        int i, j, k;
        long c;
        if(!mat_cell(g, mk, tw, t, i, j, k, c)) continue;
        if(setup) aii[c] = -1.0 / (M.p[c] + 1.0e-19);
        const double rv = rhs[c] - (mat_apply<false>(g, M, mk, [&](long cc) { return x[cc]; }, c, i, j, k));
        r[c] = rv;
        r0[c] = rv;
        p[c] = rv;
        ph[c] = rv * aii[c];
        rr += rv * rv;
    }
}

// fillxvec (bicgstab_ijk.cpp:366-378): private x = field f on the FLEXLOOP cells (dir 0);
// finalize (:380-384): f = private x there (dir 1)
__global__ void __launch_bounds__(NT) km_copy_x(TankSet b, int f_, int var, int dir)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const MatMask mk = mat_mask(g, var);
        double* __restrict__ f = T.f[f_];
        double* __restrict__ x = T.m[mat_xslot(var)];
        const TileWalk tw = tile_walk(T, q.t);
        int i, j, k;
        long c;
        if(!mat_cell(g, mk, tw, q.t, i, j, k, c)) continue;
        if(dir == 0)
            x[c] = f[c];
        else
            f[c] = x[c];
    }
}

__global__ void __launch_bounds__(NT, OCC_A64) km_init(TankSet b, int var)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        double vals[1] = {0.0};
        mat_restart(T, g, mat_mask(g, var), var, item_walk(T, b, q), true, vals[0]);
        block_sum_to<1>(vals, b.partials + (size_t)item_slot(T, b, q));
    }
}

// the pending restart, or p = r + beta (p - w v), ph = aii p (bicgstab_ijk.cpp:234-235, 151)
__global__ void __launch_bounds__(NT, OCC_A64) km_p(TankSet b, int var)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 2)
        {
            skip_tank(q, b);
            continue;
        }
        const MatMask mk = mat_mask(g, var);
        const TileWalk tw = item_walk(T, b, q);
        if(st->mode == 1)
        {
            double vals[1] = {0.0};
            mat_restart(T, g, mk, var, tw, false, vals[0]);
            block_sum_to<1>(vals, b.partials + (size_t)item_slot(T, b, q));
            continue;
        }
        const double beta = st->beta, w = st->w;
        const double* __restrict__ r = T.f[A_R];
        const double* __restrict__ vv = T.f[A_V];
        const double* __restrict__ aii = T.f[A_AII];
        double* __restrict__ p = T.f[A_P];
        double* __restrict__ ph = T.f[A_PH];
        #pragma unroll 4
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!mat_cell(g, mk, tw, t, i, j, k, c)) continue;
            const double pn = r[c] + beta * (p[c] - w * vv[c]);
            p[c] = pn;
            ph[c] = pn * aii[c];
        }
    }
}

// v = A ph; sigma = (v, r0), |v|^2, |r|^2 (bicgstab_ijk.cpp:151-160)
__global__ void __launch_bounds__(NT, OCC_A64) km_v(TankSet b, int var)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 1 || st->mode == 3)
        {
            skip_tank(q, b);
            continue;
        }
        const MatMask mk = mat_mask(g, var);
        const MatOp M = mat_op(T);
        const TileWalk tw = item_walk(T, b, q);
        const double* __restrict__ ph = T.f[A_PH];
        const double* __restrict__ r = T.f[A_R];
        const double* __restrict__ r0 = T.f[A_R0];
        double* __restrict__ vo = T.f[A_V];
        double vals[3] = {0.0, 0.0, 0.0};
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!mat_cell(g, mk, tw, t, i, j, k, c)) continue;
            const double v = mat_apply<true>(g, M, mk, [&](long cc) { return ph[cc]; }, c, i, j, k);
            vo[c] = v;
            const double rc = r[c];
            vals[0] += v * r0[c];
            vals[1] += v * v;
            vals[2] += rc * rc;
        }
        block_sum_to<3>(vals, b.partials + (size_t)item_slot(T, b, q) * 3);
    }
}

// s = r - alpha v, sh = aii s (at the stencil points), t = A sh; (t, s), (t, t), (s, s)
// (bicgstab_ijk.cpp:193-221)
__global__ void __launch_bounds__(NT, OCC_A64) km_t(TankSet b, int var)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 1 || st->mode == 3)
        {
            skip_tank(q, b);
            continue;
        }
        const MatMask mk = mat_mask(g, var);
        const MatOp M = mat_op(T);
        const TileWalk tw = item_walk(T, b, q);
        const double alpha = st->alpha;
        const double* __restrict__ r = T.f[A_R];
        const double* __restrict__ v = T.f[A_V];
        const double* __restrict__ a = T.f[A_AII];
        double* __restrict__ to = T.f[A_T];
        double vals[3] = {0.0, 0.0, 0.0};
        #pragma unroll 1
        for(int tt = tw.t; tt < tw.t1; ++tt)
        {
            int i, j, k;
            long c;
            if(!mat_cell(g, mk, tw, tt, i, j, k, c)) continue;
            const double sc = r[c] - alpha * v[c];
            const double t =
                mat_apply<true>(g, M, mk, [&](long cc) { return (r[cc] - alpha * v[cc]) * a[cc]; }, c, i, j, k);
            to[c] = t;
            vals[0] += t * sc;
            vals[1] += t * t;
            vals[2] += sc * sc;
        }
        block_sum_to<3>(vals, b.partials + (size_t)item_slot(T, b, q) * 3);
    }
}

// x and r updates, (r, r0), |r|^2 (bicgstab_ijk.cpp:223-268)
__global__ void __launch_bounds__(NT, OCC_FULL) km_x(TankSet b, int var)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const BiState* st = T.st;
        if(st->done || st->mode == 1 || st->mode == 3)
        {
            skip_tank(q, b);
            continue;
        }
        const MatMask mk = mat_mask(g, var);
        const TileWalk tw = item_walk(T, b, q);
        const double alpha = st->alpha, w = st->w;
        const int branch = st->branch;
        double* __restrict__ xv = T.m[mat_xslot(var)];
        double* __restrict__ r = T.f[A_R];
        const double* __restrict__ vv = T.f[A_V];
        const double* __restrict__ aii = T.f[A_AII];
        const double* __restrict__ ph = T.f[A_PH];
        const double* __restrict__ tv = T.f[A_T];
        const double* __restrict__ r0 = T.f[A_R0];
        double vals[2] = {0.0, 0.0};
        #pragma unroll 4
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!mat_cell(g, mk, tw, t, i, j, k, c)) continue;
            const double sv = r[c] - alpha * vv[c];
            double rn;
            if(branch)
            {
                const double sh = sv * aii[c];
                xv[c] += alpha * ph[c] + w * sh;
                rn = sv - w * tv[c];
            }
            else
            {
                xv[c] += alpha * ph[c];
                rn = sv;
            }
            r[c] = rn;
            vals[0] += rn * r0[c];
            vals[1] += rn * rn;
        }
        block_sum_to<2>(vals, b.partials + (size_t)item_slot(T, b, q) * 2);
    }
}

// ------------------------------------------------------------------ implicit diffusion (D20 = 2)
// pdiff->diff_u / diff_v / diff_w of idiff2_FS (idiff2_FS_2D on 2-D tanks) inside a
// momentum_FC3 stage (momentum_FC3.cpp:170-204, 272-306, 370-404): the operator rows and
// right-hand side of component comp into TankDev::m[0..7], and fillxvec of the diff field
// (= u_in on the loop, idiff2_FSu.cpp:47-48) into the private x m[8].  The direct-forcing
// flags are set in TankDev::tstep[5] after the first stage-1 predictor of the run.
template<int comp>
__global__ void __launch_bounds__(NT, 2) km_idiff(TankSet b, double alpha, int qin_, int u_, int v_, int w_)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        if(comp == 2 && g.jdir == 0) continue;
        const MatMask mk = mat_mask(g, comp);
        const double* __restrict__ vin = T.f[qin_];
        const double* __restrict__ u = T.f[u_];
        const double* __restrict__ v = T.f[v_];
        const double* __restrict__ w = T.f[w_];
        const double dt = T.tstep[0];
        const bool df = T.tstep[5] != 0.0;
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell_row(g, tw, t, i, j, k, c) || !comp_cell(g, comp, i, j, k)) continue;
            const MatRow r = idiff_row(g, comp, alpha, dt, vin, u, v, w, T.f[REEF_U], T.f[REEF_V], T.f[REEF_VISC], df,
                                       mk.ie, mk.je, mk.ke, c, i, j, k);
            T.m[0][c] = r.p;
            T.m[1][c] = r.n;
            T.m[2][c] = r.s;
            T.m[3][c] = r.w;
            T.m[4][c] = r.e;
            T.m[5][c] = r.t;
            T.m[6][c] = r.b;
            T.m[7][c] = r.rhs;
            T.m[8][c] = vin[c];
        }
    }
}

// the stage combination of component comp with the solved diff (the private x, which
// finalize would copy into diff): stage 1 urk1 = udiff + dt F, stage 2 urk2 = 0.75 u +
// 0.25 udiff + 0.25 dt F, stage 3 u = u / 3 + 2/3 udiff + 2/3 dt F (momentum_FC3.cpp:
// 172-174, 274-276, 372-374); F is the component's F / G / H
template<int comp>
__global__ void __launch_bounds__(NT) km_combine(TankSet b, int stage, int qold_, int F_, double cfac, int out_)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        if(comp == 2 && g.jdir == 0) continue;
        const double* __restrict__ qold = T.f[qold_];
        const double* __restrict__ F = T.f[F_];
        const double* __restrict__ df = T.m[8];
        double* __restrict__ out = T.f[out_];
        const double cdt = cfac * T.tstep[0];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell_row(g, tw, t, i, j, k, c) || !comp_cell(g, comp, i, j, k)) continue;
            if(stage == 1)
                out[c] = df[c] + cdt * 1.0 * F[c];
            else if(stage == 2)
                out[c] = 0.75 * qold[c] + 0.25 * df[c] + cdt * 1.0 * F[c];
            else
                out[c] = (1.0 / 3.0) * qold[c] + (2.0 / 3.0) * df[c] + cdt * 1.0 * F[c];
        }
    }
}

// ghostcell::solid_forcing_flag_update at the end of momentum_forcing_start
// (momentum_forcing.cpp:102): from here on the diffusion rows fold their wall couplings
__global__ void km_df_set(TankSet b)
{
    const int tk = blockIdx.x * blockDim.x + threadIdx.x;
    if(tk >= b.n) return;
    tank_at(b, tk).tstep[5] = 1.0;
}

// ------------------------------------------------------------------ adaptive time step
// ietimestep::start (ietimestep.cpp:38-207) and ::ini (:209-304) with N50 = 1, first pass:
// per work item the largest |u| over the u loop (i < nx - 1), |v| over the v loop
// (j < ny - 1) and |w| over the w loop (k < nz - 1): ULOOP / VLOOP / WLOOP
// (looping.h:149-151) without the last rows of the staggered grids
__global__ void __launch_bounds__(NT) kb_velmax(TankSet b, int u_, int v_, int w_)
{
    __shared__ double ws[3][NT / 64];
    #pragma unroll 1
    for(ItemIter q = set_items_spread(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const double* __restrict__ u = T.f[u_];
        const double* __restrict__ v = T.f[v_];
        const double* __restrict__ w = T.f[w_];
        const TileWalk tw = item_walk(T, b, q);
        double m[3] = {0.0, 0.0, 0.0};
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            if(i < g.nx - 1) m[0] = fmax(m[0], fabs(u[c]));
            if(j < g.ny - 1) m[1] = fmax(m[1], fabs(v[c]));
            if(k < g.nz - 1) m[2] = fmax(m[2], fabs(w[c]));
        }
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        for(int a = 0; a < 3; ++a)
            for(int off = 32; off > 0; off >>= 1) m[a] = fmax(m[a], __shfl_xor(m[a], off));
        if(lane == 0)
            for(int a = 0; a < 3; ++a) ws[a][wave] = m[a];
        __syncthreads();
        if(threadIdx.x == 0)
            for(int a = 0; a < 3; ++a)
                b.partials[(size_t)item_slot(T, b, q) * 3 + a] =
                    fmax(fmax(ws[a][0], ws[a][1]), fmax(ws[a][2], ws[a][3]));
        __syncthreads();
    }
}

// second pass, one block per tank: the maxima over the tank's items, then
//   dt = N47 * MIN over cells of 2 / (|u|max / dx + sqrt(4 |maxF,G,H| / dx)), dx = MIN3(DXN,
//   DYN, DZN) of the cell, with maxF = maxG = maxH = 0 (only the EARSM closure sets them)
// (::ini: umax at least 2, dt * 0.25, at least 1e-6).  The term is monotone in dx, so the
// minimum over the cells is the term at the smallest cell width (tstep[4], from the grid).
__global__ void kb_fin_dt(TankSet b, double N47, int ini)
{
    __shared__ double sh[3][NT];
    CTank& T = tank_at(b, blockIdx.x);
    const double* __restrict__ part = b.partials + (size_t)T.item0 * 3;
    double m[3] = {0.0, 0.0, 0.0};
    for(int it = threadIdx.x; it < T.shape.nitems; it += NT)
        for(int a = 0; a < 3; ++a) m[a] = fmax(m[a], part[(size_t)it * 3 + a]);
    for(int a = 0; a < 3; ++a) sh[a][threadIdx.x] = m[a];
    __syncthreads();
    for(int s = NT / 2; s > 0; s >>= 1)
    {
        if(threadIdx.x < s)
            for(int a = 0; a < 3; ++a) sh[a][threadIdx.x] = fmax(sh[a][threadIdx.x], sh[a][threadIdx.x + s]);
        __syncthreads();
    }
    if(threadIdx.x == 0)
    {
        double umax = sh[0][0];
        const double vmax = sh[1][0], wmax = sh[2][0];
        if(ini) umax = umax > 2.0 ? umax : 2.0;
        const double dx = T.tstep[4], maxFGH = 0.0;
        const double c = 2.0 / ((sqrt(umax * umax + vmax * vmax + wmax * wmax)) / dx + sqrt((4.0 * fabs(maxFGH)) / dx));
        double cu = 1.0e10 < c ? 1.0e10 : c;
        double dt = N47 * cu;
        if(ini)
        {
            dt = N47 * cu * 0.25;
            dt = dt > 1.0e-6 ? dt : 1.0e-6;
        }
        T.tstep[0] = dt;
        T.tstep[1] = umax;
        T.tstep[2] = vmax;
        T.tstep[3] = wmax;
    }
}

// x64 += x32, x32 = 0
__global__ void __launch_bounds__(NT) kb_add32(TankSet b, int x)
{
    #pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        double* __restrict__ x64 = T.f[x];
        float* __restrict__ x32 = T.s[S_X];
        const TileWalk tw = tile_walk(T, q.t);
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            x64[c] += (double)x32[c];
            x32[c] = 0.0f;
        }
    }
}

// ||rhs - A x||_2 (res_calc, bicgstab_ijk.cpp:314-338, without 1/N)
__global__ void __launch_bounds__(NT, OCC_A64) kb_defect(TankSet b, int x, int rhs)
{
    #pragma unroll 1
    for(ItemIter q = set_items(b); q.q < q.hi; next_item(q, b))
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        const SolverOp64 op = Prec<double>::op(T);
        const double* __restrict__ xv = T.f[x];
        const double* __restrict__ bv = T.f[rhs];
        const TileWalk tw = item_walk(T, b, q);
        double vals[1] = {0.0};
        #pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            const Coupling cq = coupling_of(g, op, c, i, j, k);
            const double rv = bv[c] - apply_A(g, cq, xv, c, i, j, k);
            vals[0] += rv * rv;
        }
        block_sum_to<1>(vals, b.partials + (size_t)item_slot(T, b, q));
    }
}

__global__ void kb_fin_norm(TankSet b, double* __restrict__ norms)
{
    CTank& T = tank_at(b, blockIdx.x);
    double tot[1];
    tank_totals<1>(T, b, tot);
    if(threadIdx.x == 0) norms[b.slot[blockIdx.x]] = sqrt(tot[0]);
}

// solver states of the set's tanks into dst[slot] (one copy-out per iteration batch)
__global__ void kb_gather_states(TankSet b, BiState* __restrict__ dst)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if(p >= b.n) return;
    CTank& T = tank_at(b, p);
    dst[b.slot[p]] = *T.st;
}

// Field rows between the device (sx doubles apart) and a pinned host slot (X apart), which the
// kernel reads or writes over the bus, which bounds it (40 GB/s to the device).  The copy engine
// was no faster for 2 MB and took 50 us more to start and to wait for.
__global__ void __launch_bounds__(NT) kb_move_rows(double* __restrict__ dev, double* __restrict__ slot, long ndev, long X,
                                                   long sx, int put)
{
    for(long e = (long)blockIdx.x * NT + threadIdx.x; e < ndev; e += (long)gridDim.x * NT)
    {
        const long r = (unsigned)e / (unsigned)sx, x = e - r * sx;   // a chunk has less than 2^32 doubles
        if(put)
            dev[e] = x < X ? slot[r * X + x] : 0.0;
        else if(x < X)
            slot[r * X + x] = dev[e];
    }
}

// ------------------------------------------------------------------ level-set benchmark
// benchmark_vortex3D::start (benchmark_vortex3D.cpp:67-96): the prescribed deformation velocity
// at the face positions, at time simtime, of the three components.  The factors depend on one
// coordinate each: a block evaluates them once per x of its row, per y and per z of its tile
// (the same function calls, so the same bits) instead of eleven times per cell in three
// launches.  What bounds it is the chain of one such evaluation per block: 105 -> 23 us a step at
// 128^3 (50 MB stored).
__global__ void __launch_bounds__(NT) kb_vortex_velocity(TankSet b, double simtime, double DXM)
{
    __shared__ double X[2][TX], Y[2][TY], Z[2][TY], cts;   // pow(sin(PI (q + DXM/2)), 2) and sin(2 PI q)
    TileIter q = set_tile(b);
    if(!q.ok) return;
    CTank& T = tank_at(b, q.p);
    const DevGrid g = T.g;
    const TileWalk tw = tile_walk(T, q.t);
    const int col = q.t / tw.s.nbz, bz = q.t - col * tw.s.nbz, by = col / tw.s.nbx, bx = col - by * tw.s.nbx;
    const int h = threadIdx.x;
    auto factors = [&](double pos, double& sq, double& s2) {
        const double pc = pos + 0.5 * DXM;
        sq = pow(sin(PI_REF * pc), 2.0);
        s2 = sin(2.0 * PI_REF * pos);
    };
    if(h < TX)
        factors(g.XP[min(bx * TX + h, g.nx - 1) + MARGE], X[0][h], X[1][h]);
    else if(h < TX + tw.s.ty)
        factors(g.YP[min(by * tw.s.ty + h - TX, g.ny - 1) + MARGE], Y[0][h - TX], Y[1][h - TX]);
    else if(h >= 2 * TX && h < 2 * TX + tw.s.tz)
        factors(g.ZP[min(bz * tw.s.tz + h - 2 * TX, g.nz - 1) + MARGE], Z[0][h - 2 * TX], Z[1][h - 2 * TX]);
    else if(h == 3 * TX)
        cts = cos((PI_REF * simtime) / 3.0);
    __syncthreads();
    const double ct = cts;
    int i, j, k;
    long c;
    if(!tile_cell(g, tw, q.t, i, j, k, c)) return;
    const int lx = i - bx * TX, ly = j - by * tw.s.ty, lz = k - bz * tw.s.tz;
    if(i < g.nx - 1) T.f[REEF_U][c] = 2.0 * X[0][lx] * Y[1][ly] * Z[1][lz] * ct;
    if(j < g.ny - 1) T.f[REEF_V][c] = -X[1][lx] * Y[0][ly] * Z[1][lz] * ct;
    if(k < g.nz - 1) T.f[REEF_W][c] = -X[1][lx] * Y[1][ly] * Z[0][lz] * ct;
}

// momentum_RK3 with void convection, diffusion and pressure (momentum_RK3.cpp:70-326):
// the three stages of one component with the constant forcing Fv
__global__ void __launch_bounds__(NT) kb_void_rk3(TankSet b, int comp, int id, double Fv)
{
#pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const DevGrid g = T.g;
        double* __restrict__ qf = T.f[id];
        const double dt = T.tstep[0];
        const TileWalk tw = tile_walk(T, q.t);
#pragma unroll 1
        for(int t = tw.t; t < tw.t1; ++t)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, t, i, j, k, c)) continue;
            if((comp == 1 && i >= g.nx - 1) || (comp == 2 && j >= g.ny - 1) || (comp == 3 && k >= g.nz - 1)) continue;
            const double q0 = qf[c];
            double a1 = q0 + dt * 1.0 * Fv;
            a1 += 1.0 * dt * 1.0 * 0.0;
            double a2 = 0.75 * q0 + 0.25 * a1 + 0.25 * dt * 1.0 * Fv;
            a2 += 0.25 * dt * 1.0 * 0.0;
            double qn = (1.0 / 3.0) * q0 + (2.0 / 3.0) * a2 + (2.0 / 3.0) * dt * 1.0 * Fv;
            qn += (2.0 / 3.0) * dt * 1.0 * 0.0;
            qf[c] = qn;
        }
    }
}

// ------------------------------------------------------------------ wave generation (iowave)
// Relaxation-zone wave generation (B98 = 2) and numerical beach (B99) of linear waves.  The
// static part (zones, relaxation factors, distances along the wave) comes per column from
// the host; the kernels evaluate the wave at the tank's simtime (tstep[6]), the value
// wavegen_precalc gives at the start of the step, where a relaxation reads it.

// iowave::ramp (iowave_relax_functions.cpp:239-254); ramp_T = B102 wT (B101 = 1) or B102
__device__ __forceinline__ double wave_ramp(const WaveDev& W, double t)
{
    double f = 1.0;
    if(W.ramp_mode == 1 && t < W.ramp_T) f = t / (W.ramp_T) - (1.0 / PI_REF) * sin(PI_REF * (t / (W.ramp_T)));
    if(W.ramp_mode == 2 && t < W.ramp_T) f = t / (W.ramp_T) - (1.0 / PI_REF) * sin(PI_REF * (t / (W.ramp_T)));
    return f;
}

// wave_interface (wave_interface.cpp:137-219) over wave_lib_linear (wave_lib_linear.cpp:
// 47-85): the start and end times are 0 and 1e20, the depth clamp is wD
__device__ __forceinline__ double wave_horz(const WaveDev& W, double x, double z, double t)
{
    const double teta = W.wk * x - W.ww * (t) + W.pshift;
    return W.ww * W.wa * (cosh(W.wk * (W.wdt + z)) / sinh(W.wk * W.wdt)) * cos(teta);
}
__device__ __forceinline__ double wave_target(const WaveDev& W, int comp, double x, double z, double t)
{
    z = z > -W.wD ? z : -W.wD;
    if(!(t >= 0.0 && t <= 1.0e20)) return 0.0;
    if(comp == 1) return W.cosg * wave_horz(W, x, z, t);
    if(comp == 2) return W.sing * wave_horz(W, x, z, t);
    const double teta = W.wk * x - W.ww * (t) + W.pshift;
    return W.ww * W.wa * (sinh(W.wk * (W.wdt + z)) / sinh(W.wk * W.wdt)) * sin(teta);
}

// eta(i, j) of wavegen_precalc_relax (iowave_precalc_relax.cpp:37-48) in the generation
// zone's columns; the other columns keep 0, as the reference's slice does.  One block per
// tank of the set.
__global__ void __launch_bounds__(NT) kb_wave_eta(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    const WaveDev W = T.wave;
    if(!W.col || !W.gen) return;
    const long ncol = (long)T.g.nx * T.g.ny;
    const double t = T.tstep[6];
    const double* __restrict__ gen = W.col + WC_GEN * ncol;
    const double* __restrict__ xg = W.col + WC_XG4 * ncol;
    for(long q = threadIdx.x; q < ncol; q += NT)
        if(gen[q] != 0.0) W.eta[q] = (t >= 0.0 && t <= 1.0e20) ? W.wa * cos(W.wk * xg[q] - W.ww * (t) + W.pshift) : 0.0;
}

// iowave::u_relax, v_relax, w_relax, p_relax, phi_relax (iowave_relax.cpp:28-395) with the
// target values of wavegen_precalc_relax (iowave_precalc_relax.cpp:50-160), per cell of the
// zones' columns: velocity (u_ >= 0: the fields u_, v_, w_), pressure (p_ >= 0) and level set
// (f_ >= 0)
__global__ void __launch_bounds__(NT) kb_wave_relax(TankSet b, int u_, int v_, int w_, int p_, int f_)
{
#pragma unroll 1
    for(TileIter q = set_tile(b); q.ok; q.ok = false)
    {
        CTank& T = tank_at(b, q.p);
        const WaveDev W = T.wave;
        if(!W.col) continue;
        const DevGrid g = T.g;
        const long ncol = (long)g.nx * g.ny;
        const double t = T.tstep[6];
        const double ramp = wave_ramp(W, t);
        const double* __restrict__ phi = T.f[REEF_PHI];
        const TileWalk tw = tile_walk(T, q.t);
#pragma unroll 1
        for(int tt = tw.t; tt < tw.t1; ++tt)
        {
            int i, j, k;
            long c;
            if(!tile_cell(g, tw, tt, i, j, k, c)) continue;
            const long col = i + (long)g.nx * j;
            const bool gen = W.gen && W.col[WC_GEN * ncol + col] != 0.0;
            const bool beach = W.beach && W.col[WC_BEACH * ncol + col] != 0.0;
            if(!gen && !beach) continue;
            const double zp = g.ZP[k + MARGE];
            if(u_ >= 0)
                for(int comp = 1; comp <= 3; ++comp)
                {
                    if(!comp_cell(g, comp, i, j, k)) continue;
                    double* __restrict__ vel = T.f[comp == 1 ? u_ : comp == 2 ? v_ : w_];
                    const long off = comp == 1 ? 1 : comp == 2 ? g.sx : g.sxy;
                    const double phival = 0.5 * (phi[c] + phi[c + off]);
                    double H = 0.0, G = 0.0;
                    if(phival >= -W.psi) { H = 1.0; G = 1.0; }
                    if(phival < -W.epsi) { H = 0.0; G = 0.0; }
                    if(phival >= -W.epsi && phival < -W.psi)
                    {
                        H = 0.5 * (1.0 + phival / W.epsi + (1.0 / PI_REF) * sin((PI_REF * phival) / W.epsi));
                        G = H;
                    }
                    double v = vel[c];
                    if(gen)
                    {
                        // the target of wavegen_precalc_relax at this point
                        const double e0 = W.eta[col];
                        const double e1 = comp == 1 ? W.eta[col + 1] : comp == 2 ? W.eta[col + g.nx] : 0.0;
                        const double zloc = comp == 3 ? W.zn[k + 1 + MARGE] : zp;
                        const double emid = comp == 3 ? e0 : 0.5 * (e0 + e1);
                        const double fsfloc = emid + W.phimean;
                        const double z = zloc <= fsfloc ? zloc - W.phimean : emid;
                        const double xg = W.col[(comp == 1 ? WC_XG1 : comp == 2 ? WC_XG2 : WC_XG4) * ncol + col];
                        double val = 0.0;
                        if(zloc <= fsfloc + W.epsi) val = wave_target(W, comp, xg, z, t) + (comp == 1 ? W.Ui : 0.0);
                        const double r = W.col[(comp == 1 ? WC_R1WG : comp == 2 ? WC_R2WG : WC_R4WG) * ncol + col];
                        v = (1.0 - r) * ramp * val * H + r * H * v + (1.0 - G) * v;
                        if(comp == 1) v += (1.0 - r) * ramp * W.W50 * (1.0 - H) + r * (1.0 - H) * W.W50;
                    }
                    if(beach) v = W.col[(comp == 1 ? WC_R1NB : comp == 2 ? WC_R2NB : WC_R4NB) * ncol + col] * v;
                    vel[c] = v;
                }
            if(p_ >= 0 && beach)
            {
                double* __restrict__ press = T.f[p_];
                const double r = W.col[WC_R4NB * ncol + col];
                press[c] = (1.0 - r) * ((W.phimean - zp) * T.f[REEF_RO][c] * W.gabs) + r * press[c];
            }
            if(f_ >= 0)
            {
                double* __restrict__ f = T.f[f_];
                if(gen)
                {
                    const double r = W.col[WC_R4WG * ncol + col];
                    f[c] = (1.0 - r) * ramp * (W.eta[col] + W.phimean - zp) + r * f[c];
                }
                if(beach && W.beach_phi)
                {
                    const double r = W.col[WC_R4NB * ncol + col];
                    f[c] = (1.0 - r) * (W.phimean - zp) + r * f[c];
                }
            }
        }
    }
}

// the driver's p->simtime += p->dt after the step (driver_loop_cfd.cpp:100)
__global__ void kb_wave_time(TankSet b)
{
    CTank& T = tank_at(b, blockIdx.x);
    if(T.wave.col && threadIdx.x == 0) T.tstep[6] = T.tstep[6] + T.tstep[0];
}

}  // namespace bk

// ------------------------------------------------------------------ launchers
using namespace bk;

static inline dim3 tankgrid(const TankSet& b) { return dim3((unsigned)b.n); }
static inline dim3 setup_grid(const TankSet& b) { return dim3((unsigned)((b.n + 63) / 64)); }
// per-tile launch: 8 * ceil(tiles / 8) blocks
static inline dim3 tgrid(const TankSet& b) { return dim3((unsigned)(8 * std::max(1, (b.ntiles + 7) / 8))); }
// persistent launch over the work items: one block per work item, at most occ blocks per
// CU (the kernel's occupancy) on the 256 CUs, a multiple of 8
static inline dim3 pgrid_n(int nitems, int occ)
{
    return dim3((unsigned)std::max(8, std::min(256 * occ, (nitems + 7) / 8 * 8)));
}
static inline dim3 pgrid(const TankSet& b, int occ = OCC_FULL) { return pgrid_n(b.nitems, occ); }
// the launches of one kind of tank (set_items_of): class-walked or the others
static inline dim3 pgrid_pw(const TankSet& b, int occ) { return pgrid_n(b.pw_items, occ); }
static inline dim3 pgrid_direct(const TankSet& b, int occ) { return pgrid_n(b.nitems - b.pw_items, occ); }

hipError_t bl_move_rows(double* dev, double* pinned, long ndev, long X, long sx, bool put, hipStream_t s)
{
    const unsigned blocks = (unsigned)std::min(1024L, (ndev + NT - 1) / NT);
    int to_dev = put ? 1 : 0;
    void* args[] = {&dev, &pinned, &ndev, &X, &sx, &to_dev};
    return hipLaunchKernel(reinterpret_cast<const void*>(kb_move_rows), dim3(blocks), dim3(NT), args, 0, s);
}
void bl_copy(const TankSet& b, int src, int dst, hipStream_t s)
{
    hipLaunchKernelGGL(kb_copy, tgrid(b), dim3(NT), 0, s, b, src, dst);
}
void bl_fill(const TankSet& b, int id, double v, hipStream_t s)
{
    hipLaunchKernelGGL(kb_fill, dim3(1024), dim3(NT), 0, s, b, id, v);
}
// Two ghost operations per thread of the largest program, whose length sets the grid: 256 blocks
// whatever the size left up to 20 dependent rounds to a thread of a large tank and idle blocks
// to a small one (a fill at 512x64x128 16.0 -> 13.9 us, 128^3 6.9 -> 6.2).  Each tank has its
// own row of blocks: with every block going through the tanks one after the other the tanks'
// latencies added up (16 tanks of 700x160: 14 us with 256 blocks, 21 us with 8, now 6.7;
// 8 of 128x64 7.5, 7.9, 6.5; one tank 6.4 either way).
void bl_ghost(const TankSet& b, int prog, int id, int most, hipStream_t s)
{
    const unsigned blocks = (unsigned)std::max(8, std::min(4096, (most + 2 * NT - 1) / (2 * NT)));
    hipLaunchKernelGGL(kb_ghost, dim3(blocks, (unsigned)b.n), dim3(NT), 0, s, b, prog, id);
}
void bl_hj_stage(const TankSet& b, int stage, int phi_s, int phi_n, int u, int v, int w, int out, double cfac,
                 hipStream_t s)
{
    hipLaunchKernelGGL(kb_hj_stage, tgrid(b), dim3(NT), 0, s, b, stage, phi_s, phi_n, u, v, w, out, cfac);
}
void bl_reini_stage(const TankSet& b, int stage, int fs, int f0, int out, double F43, int fsf, hipStream_t s)
{
    hipLaunchKernelGGL(kb_reini_stage, tgrid(b), dim3(NT), 0, s, b, stage, fs, f0, out, F43, fsf);
}
void bl_flux_acc(const TankSet& b, int ipol, int q, int u, int v, int w, int acc, hipStream_t s)
{
    hipLaunchKernelGGL(kb_flux_acc, tgrid(b), dim3(NT), 0, s, b, ipol, q, u, v, w, acc);
}
void bl_momentum(const TankSet& b, int comp, int stage, int qin, int qold, int u, int v, int w, double grav,
                 double cfac, int out, double rw, double ra, int diff, hipStream_t s)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, tgrid(b), dim3(NT), 0, s, b, stage, qin, qold, u, v, w, grav, cfac, out, rw, ra);
    };
    if(comp == 1)
        diff == 2 ? go(kb_momentum<1, 2>) : diff ? go(kb_momentum<1, 1>) : go(kb_momentum<1, 0>);
    else if(comp == 2)
        diff == 2 ? go(kb_momentum<2, 2>) : diff ? go(kb_momentum<2, 1>) : go(kb_momentum<2, 0>);
    else
        diff == 2 ? go(kb_momentum<3, 2>) : diff ? go(kb_momentum<3, 1>) : go(kb_momentum<3, 0>);
}
void bl_heaviside(const TankSet& b, const double* prm4, hipStream_t s)
{
    hipLaunchKernelGGL(kb_heaviside, pgrid(b), dim3(NT), 0, s, b, prm4[0], prm4[1], prm4[2], prm4[3]);
    hipLaunchKernelGGL(kb_heaviside_fin, tankgrid(b), dim3(NT), 0, s, b, (double*)nullptr);
}

// ------------------------------------------------------------------ allocation-free scratch
// The reduction memory of the allocation-free fluid update (reef_fluid_update_noalloc): a
// file-scope device array instead of library-allocated memory.  Layout: the block partials
// (2 doubles per work item of the set, the slots kb_heaviside writes) from element 0, the
// set's volumes (2 doubles per tank) from element NOALLOC_VOL0.  Every GPU the library
// runs on holds its own copy until the process ends.  Host code never passes the array's
// name to a kernel (in host code the name is a stand-in, not a device address): it takes
// the address hipGetSymbolAddress gives for the current device, once per device.
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

namespace {
std::mutex g_scratch_mu;
double* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
}

int noalloc_scratch(double** out)
{
    int dev = 0;
    if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEVICES) return REEF_E_HIP;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if(!g_scratch_ptr[dev])
    {
        void* ptr = nullptr;
        if(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return REEF_E_HIP;
        g_scratch_ptr[dev] = (double*)ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

void bl_heaviside_noalloc(const TankSet& b, const double* prm4, double* scratch_dev, hipStream_t s)
{
    TankSet t = b;
    t.partials = scratch_dev;
    hipLaunchKernelGGL(kb_heaviside, pgrid(t), dim3(NT), 0, s, t, prm4[0], prm4[1], prm4[2], prm4[3]);
    hipLaunchKernelGGL(kb_heaviside_fin, tankgrid(t), dim3(NT), 0, s, t, scratch_dev + NOALLOC_VOL0);
}
void bl_poisson_rhs(const TankSet& b, int u, int v, int w, double afac, hipStream_t s)
{
    hipLaunchKernelGGL(kb_poisson_rhs, tgrid(b), dim3(NT), 0, s, b, u, v, w, afac);
}
void bl_face_rho(const TankSet& b, double rw, double ra, int with_aii, hipStream_t s)
{
    hipLaunchKernelGGL(kb_face_rho, tgrid(b), dim3(NT), 0, s, b, rw, ra);
    if(with_aii) hipLaunchKernelGGL(kb_aii, tgrid(b), dim3(NT), 0, s, b);
}
void bl_correct(const TankSet& b, double rw, double ra, double afac, int u, int v, int w, hipStream_t s)
{
    hipLaunchKernelGGL(kb_correct, tgrid(b), dim3(NT), 0, s, b, rw, ra, afac, u, v, w);
}

void bl_bicg_init(const TankSet& b, int x, int rhs, double stop, int maxiter, hipStream_t s)
{
    hipLaunchKernelGGL(kb_setup, setup_grid(b), dim3(64), 0, s, b, stop, maxiter, 0, 0.0);
    hipLaunchKernelGGL(kb_bicg_init<double>, pgrid(b, OCC_A64), dim3(NT), 0, s, b, x, rhs);
    hipLaunchKernelGGL(kb_fin_init, tankgrid(b), dim3(NT), 0, s, b);
}

void bl_bicg_phase(const TankSet& b, int x, int rhs, int phase, int part, hipStream_t s)
{
    const dim3 grid = pgrid(b), grid64 = pgrid(b, OCC_A64);
    if(part == 0)
    {
        switch(phase)
        {
            case 0:
                if(b.has_pw && b.has_direct)
                    hipLaunchKernelGGL((kb_bicg_p<double, true>), grid64, dim3(NT), 0, s, b, x, rhs);
                else if(b.has_pw)
                    hipLaunchKernelGGL(kb_class_p, pgrid_pw(b, OCC_CX), dim3(NT), 0, s, b, x, rhs);
                else
                    hipLaunchKernelGGL((kb_bicg_p<double, false>), grid64, dim3(NT), 0, s, b, x, rhs);
                break;
            case 1:
                if(b.has_pw) hipLaunchKernelGGL(kb_class_v, pgrid_pw(b, OCC_PW), dim3(NT), 0, s, b, x, rhs);
                if(b.has_direct)
                    hipLaunchKernelGGL(kb_bicg_v<double>, pgrid_direct(b, OCC_A64), dim3(NT), 0, s, b, x, rhs);
                break;
            case 2:
                if(b.has_pw) hipLaunchKernelGGL((kb_bicg_t<double, true>), pgrid_pw(b, OCC_PW), dim3(NT), 0, s, b, x, rhs);
                if(b.has_direct)
                    hipLaunchKernelGGL((kb_bicg_t<double, false>), pgrid_direct(b, OCC_A64), dim3(NT), 0, s, b, x, rhs);
                break;
            default:
                if(b.has_pw && b.has_direct)
                    hipLaunchKernelGGL((kb_bicg_x<double, true>), grid, dim3(NT), 0, s, b, x, rhs);
                else if(b.has_pw)
                    hipLaunchKernelGGL(kb_class_x<double>, pgrid_pw(b, OCC_CX), dim3(NT), 0, s, b, x, rhs);
                else
                    hipLaunchKernelGGL((kb_bicg_x<double, false>), grid, dim3(NT), 0, s, b, x, rhs);
                break;
        }
        return;
    }
    switch(phase)
    {
        case 0: break;   // a restart of the p phase is finalized by the v phase
        case 1: hipLaunchKernelGGL(kb_fin_v, tankgrid(b), dim3(NT), 0, s, b, 1); break;
        case 2: hipLaunchKernelGGL(kb_fin_t, tankgrid(b), dim3(NT), 0, s, b); break;
        default: hipLaunchKernelGGL(kb_fin_x, tankgrid(b), dim3(NT), 0, s, b); break;
    }
}

void bl_idiff(const TankSet& b, int comp, double alpha, int qin, int u, int v, int w, hipStream_t s)
{
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, tgrid(b), dim3(NT), 0, s, b, alpha, qin, u, v, w); };
    comp == 1 ? go(km_idiff<1>) : comp == 2 ? go(km_idiff<2>) : go(km_idiff<3>);
}

void bl_idiff_combine(const TankSet& b, int comp, int stage, int qold, int F, double cfac, int out, hipStream_t s)
{
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, tgrid(b), dim3(NT), 0, s, b, stage, qold, F, cfac, out); };
    comp == 1 ? go(km_combine<1>) : comp == 2 ? go(km_combine<2>) : go(km_combine<3>);
}

void bl_df_set(const TankSet& b, hipStream_t s)
{
    hipLaunchKernelGGL(km_df_set, setup_grid(b), dim3(64), 0, s, b);
}

void bl_mat_copy_x(const TankSet& b, int f, int var, int dir, hipStream_t s)
{
    hipLaunchKernelGGL(km_copy_x, tgrid(b), dim3(NT), 0, s, b, f, var, dir);
}

void bl_mat_init(const TankSet& b, int var, double stop, int maxiter, hipStream_t s)
{
    hipLaunchKernelGGL(kb_setup, setup_grid(b), dim3(64), 0, s, b, stop, maxiter, 0, 0.0);
    hipLaunchKernelGGL(km_init, pgrid(b, OCC_A64), dim3(NT), 0, s, b, var);
    hipLaunchKernelGGL(kb_fin_init, tankgrid(b), dim3(NT), 0, s, b);
}

void bl_mat_phase(const TankSet& b, int var, int phase, int part, hipStream_t s)
{
    const dim3 grid64 = pgrid(b, OCC_A64);
    if(part == 0)
    {
        switch(phase)
        {
            case 0: hipLaunchKernelGGL(km_p, grid64, dim3(NT), 0, s, b, var); break;
            case 1: hipLaunchKernelGGL(km_v, grid64, dim3(NT), 0, s, b, var); break;
            case 2: hipLaunchKernelGGL(km_t, grid64, dim3(NT), 0, s, b, var); break;
            default: hipLaunchKernelGGL(km_x, pgrid(b), dim3(NT), 0, s, b, var); break;
        }
        return;
    }
    switch(phase)
    {
        case 0: hipLaunchKernelGGL(kb_fin_p, tankgrid(b), dim3(NT), 0, s, b); break;
        case 1: hipLaunchKernelGGL(kb_fin_v, tankgrid(b), dim3(NT), 0, s, b, 0); break;
        case 2: hipLaunchKernelGGL(kb_fin_t, tankgrid(b), dim3(NT), 0, s, b); break;
        default: hipLaunchKernelGGL(kb_fin_x, tankgrid(b), dim3(NT), 0, s, b); break;
    }
}

void bl_coef32(const TankSet& b, hipStream_t s)
{
    hipLaunchKernelGGL(kb_coef32, tgrid(b), dim3(NT), 0, s, b);
}

void bl_mixed_init(const TankSet& b, int x, int rhs, double stop, int maxiter, double delta, hipStream_t s)
{
    hipLaunchKernelGGL(kb_setup, setup_grid(b), dim3(64), 0, s, b, stop, maxiter, 1, delta);
    hipLaunchKernelGGL(kb_mix_start, pgrid(b, OCC_A64), dim3(NT), 0, s, b, x, rhs);
    hipLaunchKernelGGL(kb_fin_mix_start, tankgrid(b), dim3(NT), 0, s, b);
}

void bl_mixed_phase(const TankSet& b, int x, int rhs, int phase, int part, hipStream_t s)
{
    const dim3 grid = pgrid(b);
    if(part == 0)
    {
        switch(phase)
        {
            case 0:
                if(b.has_pw) hipLaunchKernelGGL((kb_mix_v<true>), pgrid_pw(b, OCC_PW), dim3(NT), 0, s, b, x);
                if(b.has_direct) hipLaunchKernelGGL((kb_mix_v<false>), pgrid_direct(b, OCC_FULL), dim3(NT), 0, s, b, x);
                break;
            case 1:
                if(b.has_pw) hipLaunchKernelGGL((kb_bicg_t<float, true>), pgrid_pw(b, OCC_PW), dim3(NT), 0, s, b, x, rhs);
                if(b.has_direct)
                    hipLaunchKernelGGL((kb_bicg_t<float, false>), pgrid_direct(b, OCC_FULL), dim3(NT), 0, s, b, x, rhs);
                break;
            case 2:
                if(b.has_pw && b.has_direct)
                    hipLaunchKernelGGL((kb_bicg_x<float, true>), grid, dim3(NT), 0, s, b, x, rhs);
                else if(b.has_pw)
                    hipLaunchKernelGGL(kb_class_x<float>, pgrid_pw(b, OCC_CX), dim3(NT), 0, s, b, x, rhs);
                else
                    hipLaunchKernelGGL((kb_bicg_x<float, false>), grid, dim3(NT), 0, s, b, x, rhs);
                break;
            default: hipLaunchKernelGGL(kb_mix_ru, pgrid(b, OCC_A64), dim3(NT), 0, s, b, x, rhs); break;
        }
        return;
    }
    switch(phase)
    {
        case 0: hipLaunchKernelGGL(kb_fin_v, tankgrid(b), dim3(NT), 0, s, b, 0); break;
        case 1: hipLaunchKernelGGL(kb_fin_t, tankgrid(b), dim3(NT), 0, s, b); break;
        case 2: hipLaunchKernelGGL(kb_fin_x, tankgrid(b), dim3(NT), 0, s, b); break;
        default: break;   // the reliable-update phase is finalized by the next v phase
    }
}

void bl_mixed_settle(const TankSet& b, hipStream_t s)
{
    hipLaunchKernelGGL(kb_fin_mix_ru, tankgrid(b), dim3(NT), 0, s, b);
}

void bl_add32(const TankSet& b, int x, hipStream_t s)
{
    hipLaunchKernelGGL(kb_add32, tgrid(b), dim3(NT), 0, s, b, x);
}

void bl_timestep(const TankSet& b, int u, int v, int w, double N47, int ini, hipStream_t s)
{
    hipLaunchKernelGGL(kb_velmax, pgrid(b), dim3(NT), 0, s, b, u, v, w);
    hipLaunchKernelGGL(kb_fin_dt, tankgrid(b), dim3(NT), 0, s, b, N47, ini);
}

void bl_vortex_velocity(const TankSet& b, double simtime, double DXM, hipStream_t s)
{
    hipLaunchKernelGGL(kb_vortex_velocity, tgrid(b), dim3(NT), 0, s, b, simtime, DXM);
}
void bl_void_rk3(const TankSet& b, int comp, int id, double Fv, hipStream_t s)
{
    hipLaunchKernelGGL(kb_void_rk3, tgrid(b), dim3(NT), 0, s, b, comp, id, Fv);
}

void bl_wave_eta(const TankSet& b, hipStream_t s)
{
    hipLaunchKernelGGL(kb_wave_eta, tankgrid(b), dim3(NT), 0, s, b);
}
void bl_wave_relax(const TankSet& b, int u, int v, int w, int p, int f, hipStream_t s)
{
    hipLaunchKernelGGL(kb_wave_relax, tgrid(b), dim3(NT), 0, s, b, u, v, w, p, f);
}
void bl_wave_time(const TankSet& b, hipStream_t s)
{
    hipLaunchKernelGGL(kb_wave_time, tankgrid(b), dim3(64), 0, s, b);
}

void bl_gather_states(const TankSet& b, BiState* dst, hipStream_t s)
{
    hipLaunchKernelGGL(kb_gather_states, setup_grid(b), dim3(64), 0, s, b, dst);
}

void bl_residual(const TankSet& b, int x, int rhs, double* norms, hipStream_t s)
{
    hipLaunchKernelGGL(kb_defect, pgrid(b, OCC_A64), dim3(NT), 0, s, b, x, rhs);
    hipLaunchKernelGGL(kb_fin_norm, tankgrid(b), dim3(NT), 0, s, b, norms);
}

}  // namespace reef
