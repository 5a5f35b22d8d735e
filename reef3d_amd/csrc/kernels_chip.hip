// On-chip BiCGStab of small and mid-sized tanks: one launch runs a tank's iterations from
// start to end with every solver vector and operator coefficient in registers and the
// stencil operand in LDS.  Same arithmetic, same work items and the same order of every
// sum as the streaming phases (kernels_batch.hip), so the results are the same bits.
//
// What bounds it: a tank of up to 2048 tiles (524 288 cells) is a few hundred cells per CU,
// so the streaming solver's seven dependent launches per iteration are all latency (28 us
// per iteration on 40x8x24 cells, 40 us on 1150x157), not bytes.  Here an iteration is three
// exchanges between the tank's blocks.  Each carries the block's partial sums to every
// block of the tank and the boundary values of v or t to its neighbours in one hop:
// every 8-byte word holds 32 bits of data and a 32-bit tag (the exchange's number), written
// and polled with relaxed agent-scope atomics, so a word that carries the right tag is its
// own arrival flag and no fence or counter is needed.  Halo values of r, p, v and aii are
// kept and updated by the reader with the owner's operations, so alpha, omega and beta are
// all the halo needs beyond v and t.
//
// Blocks: NB (a power of two, at most 256, one block per CU) per tank.  Block b owns the work
// items b, b + NB, b + 2 NB, ...: sum_partials adds the items t, t + 256, ... for its thread t,
// and with NB dividing 256 a block holds whole such strided subsets, so it publishes the
// 256 / NB accumulators of its threads instead of every item's partial.
//
// Every wait is bounded (WAIT_TICKS): a block that waits too long (another process holds
// part of the GPU, so not all blocks are resident) sets the tank's abort bit, every block of
// the tank leaves, and nothing has been stored: the vectors and the state are written only
// after all blocks have arrived at the commit counter, which the abort bit shares.  The host can
// set the bit before the launch (Engine::onchip_giveup).
#include "chip.h"
#include "cell_ops.h"
#include "solver_state.h"

namespace reef {
namespace bk {

typedef unsigned long long u64;

constexpr int CG = CHIP_NT / NT;           // 256-thread groups
static_assert(CG == 2, "groups of a block");
constexpr unsigned ABORT = 0x80000000u;
// 500 ms of the 100 MHz wall clock: where a set has more blocks than the card has CUs, a tank's
// blocks can be dispatched one tank's whole solve apart
constexpr long WAIT_TICKS = 50000000;

__device__ __forceinline__ void put_word(u64* p, u64 v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get_word(const u64* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a value in tagged words: two for a double, one for a float
template<class W>
struct Wire;
template<>
struct Wire<double>
{
    u64 a, b;
    __device__ static void put(u64* p, double v, unsigned tag)
    {
        const u64 d = __builtin_bit_cast(u64, v);
        put_word(p, (d << 32) | tag);
        put_word(p + 1, (d & 0xffffffff00000000ull) | tag);
    }
    __device__ void load(const u64* p)
    {
        a = get_word(p);
        b = get_word(p + 1);
    }
    __device__ bool ready(unsigned tag) const { return (unsigned)a == tag && (unsigned)b == tag; }
    __device__ double value() const { return __builtin_bit_cast(double, (a >> 32) | (b & 0xffffffff00000000ull)); }
};
template<>
struct Wire<float>
{
    u64 a;
    __device__ static void put(u64* p, float v, unsigned tag)
    {
        put_word(p, ((u64)__builtin_bit_cast(unsigned, v) << 32) | tag);
    }
    __device__ void load(const u64* p) { a = get_word(p); }
    __device__ bool ready(unsigned tag) const { return (unsigned)a == tag; }
    __device__ float value() const { return __builtin_bit_cast(float, (unsigned)(a >> 32)); }
};

// the bound of one wait: true when it has to end (the tank's abort bit is set, by another
// block or here after WAIT_TICKS)
struct Guard
{
    unsigned* ctl;
    long t0;
    int spins;
    __device__ Guard(unsigned* c) : ctl(c), t0((long)wall_clock64()), spins(0) {}
    __device__ bool stop()
    {
        if((++spins & 63) != 0) return false;
        if(__hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ABORT) return true;
        if((long)wall_clock64() - t0 < WAIT_TICKS) return false;
        __hip_atomic_fetch_or(ctl, ABORT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
};

// wavefront sum by the butterfly off = 32, 16, .. 1 of block_sum_to and sum_partials, lane 0's
// (and every lane's) bits: the swaps give both halves to all lanes, and the rotations within
// 16 lanes reach the partner lane because the values already repeat with the previous offset
template<int CTRL>
__device__ __forceinline__ double row_ror(double v)
{
    const u64 d = __builtin_bit_cast(u64, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)d, CTRL, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(d >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (u64)lo | ((u64)hi << 32));
}
__device__ __forceinline__ double wave_sum(double v)
{
    {
        const u64 d = __builtin_bit_cast(u64, v);
        const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)d, (unsigned)d, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(d >> 32), (unsigned)(d >> 32), false, false);
        v = __builtin_bit_cast(double, (u64)lo[0] | ((u64)hi[0] << 32)) +
            __builtin_bit_cast(double, (u64)lo[1] | ((u64)hi[1] << 32));
    }
    {
        const u64 d = __builtin_bit_cast(u64, v);
        const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)d, (unsigned)d, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(d >> 32), (unsigned)(d >> 32), false, false);
        v = __builtin_bit_cast(double, (u64)lo[0] | ((u64)hi[0] << 32)) +
            __builtin_bit_cast(double, (u64)lo[1] | ((u64)hi[1] << 32));
    }
    v += row_ror<0x128>(v);
    v += row_ror<0x124>(v);
    v += row_ror<0x122>(v);
    v += row_ror<0x121>(v);
    return v;
}

// KIND: CHIP_FP64, CHIP_MIXED (V = float) or CHIP_MAT; d3: 3-D tanks; CT: tile slots a group
// uses and SL halo cells a thread keeps, at most (both set the registers a thread needs); x_
// the solution's array, rhs_ the right-hand side's (CHIP_MAT: the FLEXLOOP var)
template<class V, int KIND, bool d3, int CT, int SL>
__global__ void __launch_bounds__(CHIP_NT) kc_solve(ChipSet S, int x_, int rhs_)
{
    constexpr int CS = CG * CT;           // tile slots per group and block
    constexpr bool MIXED = KIND == CHIP_MIXED, MAT = KIND == CHIP_MAT;
    extern __shared__ __align__(16) char lds[];
    __shared__ BiState st;
    __shared__ double ws[CG][NT / 64][CT][3];      // wave sums per item
    __shared__ double wt[3][NT / 64];              // its wave sums
    __shared__ double acc1[NT][3];                 // the accumulators of a one-block tank
    __shared__ int fnb[CS][6], foff[CS][6], ftile[CS][6], stile[CS];
    __shared__ int nhalo, dead;

    // ---- which tank, which block of it
    int p = 0;
    while(p + 1 < S.n && S.blk0[p + 1] <= (int)blockIdx.x) ++p;
    const int NB = S.blk0[p + 1] - S.blk0[p], b = (int)blockIdx.x - S.blk0[p];
    CTank& T = tank_of_slot(S.tanks, S.slot[p]);
    const DevGrid g = T.g;
    const TileShape sh = T.shape;
    const int cpt = sh.cpt, nitems = sh.nitems;
    const int tid = threadIdx.x, grp = tid >> 8, ct = tid & (NT - 1), wave = ct >> 6, lane = ct & 63;
    u64* const halo0 = S.halo;
    u64* const halo1 = S.halo + S.halo_words;
    u64* const halo2 = S.halo + 2 * S.halo_words;
    u64* const accw = S.acc + (size_t)p * CHIP_ACC_WORDS;
    unsigned* const ctl = S.ctl + p;
    const int xt0 = S.tile0[p];
    const int nloc = chip_items(sh, NB, b);        // items of this block
    const int naccs = NT / NB;                     // strided subsets of this block
    const int nacc = min(NT, nitems);              // accumulators that are not 0
    const int nred = (nacc + 63) / 64;             // reducing wavefronts, one per 64 accumulators
    // few accumulators and blocks: every block adds them all itself, in one hop
    const bool direct = NB > 1 && nred == 1 && NB <= CHIP_DIRECT;
    auto red_block = [&](int w) { return NB >= 4 ? w * (NB / 4) : w % NB; };
    const int nc = ((nloc + CG - 1) / CG) * cpt;   // tile slots in use per group

    if(tid == 0)
    {
        st = *T.st;
        dead = 0;
    }
    if(tid < CS) stile[tid] = chip_slot_tile(sh, CT, NB, b, tid);
    __syncthreads();
    if(st.done) return;
    // the neighbour tile of each face (+x, -x, +y, -y, +z, -z): in this block (its slot), in
    // another (-2), none (-1)
    if(tid < CS * 6)
    {
        const int sl = tid / 6, f = tid - sl * 6, tl = stile[sl];
        int nb = -1, nt = -1;
        if(tl >= 0 && (nt = chip_face_tile(sh, tl, f)) >= 0)
        {
            nb = chip_tile_slot(sh, CT, NB, b, nt);
            if(nb < 0) nb = -2;
        }
        fnb[sl][f] = nb;
        ftile[sl][f] = nt;
    }
    __syncthreads();
    if(tid == 0)
    {
        int o = 0;
        for(int sl = 0; sl < CS; ++sl)
            for(int f = 0; f < 6; ++f)
            {
                foff[sl][f] = o;
                if(fnb[sl][f] == -2) o += chip_face_size(sh, f);
            }
        nhalo = o;
    }
    __syncthreads();
    const int H = nhalo, Hm = S.hmax;
    const int ns = (H + CHIP_NT - 1) / CHIP_NT;    // halo cells per thread
    // LDS: the stencil operand (own cells, halo cells, a zero), then r, p, v of the halo and
    // the exchange index of each halo cell.  The operand is 8 bytes wide in the mixed kernel
    // too (the FP64 residual uses it).
    constexpr int ZERO = CS * NT;
    double* const op64 = (double*)lds;
    V* const op = (V*)lds;
    char* q0 = lds + (size_t)(CS * NT + 1 + Hm) * 8;
    V* const hr = (V*)q0;
    V* const hp = hr + Hm;
    V* const hv = hp + Hm;
    int* const hsrc = (int*)(hv + Hm);
    constexpr int HALO = ZERO + 1;
    // exchange index of each halo cell: 256 * (tank's first tile + tile) + cell of the tile
    for(int sf = 0; sf < CS * 6; ++sf)
    {
        const int sl = sf / 6, f = sf - sl * 6;
        if(fnb[sl][f] != -2) continue;
        for(int q = tid; q < chip_face_size(sh, f); q += CHIP_NT)
            hsrc[foff[sl][f] + q] = (xt0 + ftile[sl][f]) * NT + chip_face_far(sh, f, q);
    }
    // ---- own cells
    const int var = MAT ? rhs_ : 0;
    const int ie = g.nx - (var == 1 ? 1 : 0), je = g.ny - (var == 2 ? 1 : 0), ke = g.nz - (var == 3 ? 1 : 0);
    const int mode0 = st.mode, hb = st.buf;
    double* const x64p = MAT ? T.m[var <= 3 ? 8 : 9] : T.f[x_];
    const double* const b64 = MAT ? T.m[7] : T.f[rhs_];
    V *gx, *gr, *gr0, *gp, *gph, *gv;
    const V* ga;
    if constexpr(MIXED)
    {
        gx = T.s[S_X];
        gr = T.s[S_R];
        gr0 = T.s[S_R0];
        gp = T.s[hb ? S_P2 : S_P];
        gph = T.s[S_PH];
        gv = T.s[hb ? S_V2 : S_V];
        ga = T.s[S_AII];
    }
    else
    {
        gx = x64p;
        gr = T.f[A_R];
        gr0 = T.f[A_R0];
        gp = T.f[A_P];
        gph = T.f[A_PH];
        gv = T.f[A_V];
        ga = T.f[A_AII];
    }
    V x[CT], r[CT], r0[CT], pv[CT], v[CT], t[CT], a[CT];
    double x64[MIXED ? CT : 1];
    Coef<V> cf[CT];
    unsigned nx01[CT], nx23[CT], nx45[CT];   // LDS indices of the six neighbours, 16 bits each
    unsigned cidx[CT];                       // element of the cell
    bool act[CT], grid[CT], pub[CT];
    auto cell_of = [&](int tl, int cell, int& i, int& j, int& k) {
        return tile_cell_of(sh, g.nx, g.ny, g.nz, tl, cell, i, j, k);
    };
    #pragma unroll
    for(int c = 0; c < CT; ++c)
    {
        x[c] = r[c] = r0[c] = pv[c] = v[c] = t[c] = a[c] = V(0);
        cf[c] = Coef<V>{V(0), V(0), V(0), V(0), V(0), V(0), V(0)};
        nx01[c] = nx23[c] = nx45[c] = (unsigned)ZERO | ((unsigned)ZERO << 16);
        act[c] = grid[c] = pub[c] = false;
        cidx[c] = 0;
        if constexpr(MIXED) x64[c] = 0.0;
        if(c >= nc) continue;
        const int sl = grp * CT + c, tl = stile[sl];
        if(tl < 0) continue;
        int i, j, k;
        if(!cell_of(tl, ct, i, j, k)) continue;
        grid[c] = true;
        const long e = g.base + i + g.sx * j + g.sxy * k;
        cidx[c] = (unsigned)e;
        x[c] = gx[e];
        act[c] = i < ie && j < je && k < ke;
        const bool in[6] = {i + 1 < g.nx, i > 0, j + 1 < g.ny, j > 0, k + 1 < g.nz, k > 0};
        unsigned nbx[6];
        bool anyr = false;
        #pragma unroll
        for(int f = 0; f < 6; ++f)
        {
            unsigned q = ZERO;
            if(in[f])
            {
                const int fp = chip_face_pos(sh, f, wave, lane);
                if(!chip_on_face(sh, f, wave, lane))
                    q = (unsigned)(sl * NT + ct + chip_face_step(sh, f));
                else if(fnb[sl][f] >= 0)
                    q = (unsigned)(fnb[sl][f] * NT + chip_face_far(sh, f, fp));
                else if(fnb[sl][f] == -2)
                {
                    q = (unsigned)(HALO + foff[sl][f] + fp);
                    anyr = true;
                }
            }
            nbx[f] = q;
        }
        pub[c] = anyr;
        nx01[c] = nbx[0] | (nbx[1] << 16);
        nx23[c] = nbx[2] | (nbx[3] << 16);
        nx45[c] = nbx[4] | (nbx[5] << 16);
        if constexpr(MIXED) x64[c] = x64p[e];
        if(!act[c]) continue;
        r[c] = gr[e];
        r0[c] = gr0[e];
        pv[c] = gp[e];
        if(mode0 != 2) v[c] = gv[e];
        a[c] = ga[e];
        if constexpr(MAT)
            cf[c] = Coef<V>{T.m[0][e], T.m[1][e], T.m[2][e], T.m[3][e], T.m[4][e], T.m[5][e], T.m[6][e]};
        else if constexpr(MIXED)
            cf[c] = poisson_coef(g, coupling_of(g, SolverOp32{T.s[S_KX], T.s[S_KY], T.s[S_KZ], T.iDXN32, T.iDYN32, T.iDZN32}, e, i, j, k), i, j, k);
        else
            cf[c] = poisson_coef(g, couplings(g, T.f[A_RFX], T.f[A_RFY], T.f[A_RFZ], e, i, j, k), i, j, k);
    }
    if(tid == 0) op64[ZERO] = 0.0;
    if(MIXED && tid == 0) op[ZERO] = V(0);
    __syncthreads();
    // ---- halo cells: thread tid keeps cells tid, tid + 512, ...; hst: a cell of the grid
    // outside the FLEXLOOP box (SOLVE_MAT), whose x is not a neighbour's to publish
    V ha[SL];
    unsigned hcell[SL];     // element of a static halo cell + 1, else 0
    #pragma unroll
    for(int s = 0; s < SL; ++s)
    {
        ha[s] = V(0);
        hcell[s] = 0;
        const int q = tid + s * CHIP_NT;
        if(q >= H) continue;
        const int ix = hsrc[q], tl = (ix >> 8) - xt0;
        int i, j, k;
        V vr = V(0), vp = V(0), vv = V(0);
        const bool ing = cell_of(tl, ix & (NT - 1), i, j, k);
        if(ing && i < ie && j < je && k < ke)
        {
            const long e = g.base + i + g.sx * j + g.sxy * k;
            vr = gr[e];
            vp = gp[e];
            if(mode0 != 2) vv = gv[e];
            ha[s] = ga[e];
        }
        else
        {
            // never waited for; its operand is 0, or the unchanging x of a restart
            if(ing) hcell[s] = (unsigned)(g.base + i + g.sx * j + g.sxy * k) + 1u;
            hsrc[q] = -1;
        }
        hr[q] = vr;
        hp[q] = vp;
        hv[q] = vv;
    }

    // Reuse of the buffers.  A block publishes exchange n before it has read exchange n, so a
    // buffer may be written again only after a later exchange of the whole tank that every
    // reader joined after reading.  v goes to halo0, t to halo1, x (or x64 + x32) of a restart
    // to halo1 and the restarted r to halo2: v, t, x phase and v, restart (x to the
    // neighbours only, then r with the totals) both keep that rule, and the accumulators
    // alternate between two buffers.
    unsigned tag = S.epoch;      // number of the next exchange
    int parity = 0;              // accumulator buffer
    // publishes one value per boundary cell
    auto publish = [&](u64* buf, auto&& val, unsigned tg) {
        #pragma unroll
        for(int c = 0; c < CT; ++c)
            if(c < nc && pub[c] && act[c])
            {
                auto w = val(c);
                Wire<decltype(w)>::put(buf + ((size_t)(xt0 + stile[grp * CT + c]) * NT + ct) * 2, w, tg);
            }
    };
    // receives the neighbours' values of this thread's halo cells: got(s, q, value)
    auto receive = [&](const u64* buf, unsigned tg, auto zero, auto&& got) {
        using W = decltype(zero);
        Wire<W> w[SL];
        int src[SL];
        #pragma unroll
        for(int s = 0; s < SL; ++s)
        {
            src[s] = -1;
            if(s < ns && tid + s * CHIP_NT < H) src[s] = hsrc[tid + s * CHIP_NT];
        }
        Guard gd(ctl);
        for(;;)
        {
            bool ok = true;
            #pragma unroll
            for(int s = 0; s < SL; ++s)
                if(s < ns && src[s] >= 0) w[s].load(buf + (size_t)src[s] * 2);
            #pragma unroll
            for(int s = 0; s < SL; ++s)
                if(s < ns && src[s] >= 0) ok = ok && w[s].ready(tg);
            if(ok) break;
            if(gd.stop())
            {
                dead = 1;
                break;
            }
        }
        #pragma unroll
        for(int s = 0; s < SL; ++s)
            if(s < ns && src[s] >= 0) got(s, tid + s * CHIP_NT, w[s].value());
    };
    // One exchange with the tank's totals.  contrib(c, s): the sums' terms of tile slot c's
    // cell; send / recv: the boundary values; store(tot): the new state, run by one thread.
    // The totals take two hops: the block publishes its accumulators, four wavefronts of the
    // tank (reducers) add 64 of them each, as the four wavefronts of sum_partials do, and
    // publish the wave sums in CHIP_COPIES places, so that 256 blocks do not poll one line.
    // Measured with 256 blocks: 3.5 us an exchange, against 6.4 us when every block polls all
    // accumulators.
    auto exchange = [&](auto M_, auto&& contrib, auto&& send, auto&& recv, auto&& store) {
        constexpr int M = decltype(M_)::value;
        const unsigned tg = tag++;
        send(tg);
        // sums of each item: the tiles of an item in order, wavefront butterfly, 4 waves
        double cur[M];
        #pragma unroll
        for(int m = 0; m < M; ++m) cur[m] = 0.0;
        #pragma unroll
        for(int c = 0; c < CT; ++c)
            if(c < nc)
            {
                double s[M];
                contrib(c, s);
                #pragma unroll
                for(int m = 0; m < M; ++m) cur[m] += s[m];
                if((c + 1) % cpt == 0)
                {
                    #pragma unroll
                    for(int m = 0; m < M; ++m)
                    {
                        const double y = wave_sum(cur[m]);
                        if(lane == 0) ws[grp][wave][c / cpt][m] = y;
                        cur[m] = 0.0;
                    }
                }
            }
        __syncthreads();
        u64* const aw = accw + (size_t)parity * CHIP_ACC_HALF;
        u64* const cw = aw + 3 * NT * 2;             // the copies of the wave sums
        for(int ix = tid; ix < naccs * M; ix += CHIP_NT)
        {
            const int q = ix / M, m = ix - q * M;
            double s = 0.0;
            for(int li = q; li < nloc; li += naccs)
            {
                const double(*w4)[CT][3] = ws[li % CG];
                const int kk = li / CG;
                s += ((w4[0][kk][m] + w4[1][kk][m]) + w4[2][kk][m]) + w4[3][kk][m];
            }
            const int ai = b + q * NB;
            if(NB == 1)
                acc1[ai][m] = s;
            else if(ai < nacc)
                Wire<double>::put(aw + (size_t)(ai * M + m) * 2, s, tg);
        }
        if(NB == 1) __syncthreads();
        // the reducing wavefronts: wave w of the last group in the block that adds part w
        if(grp == CG - 1 && wave < nred && (NB == 1 || direct || b == red_block(wave)))
        {
            const int ai = wave * 64 + lane;
            double y[M];
            #pragma unroll
            for(int m = 0; m < M; ++m) y[m] = 0.0;
            if(ai < nacc)
            {
                if(NB == 1)
                {
                    #pragma unroll
                    for(int m = 0; m < M; ++m) y[m] = acc1[ai][m];
                }
                else
                {
                    Wire<double> w[M];
                    Guard gd(ctl);
                    for(;;)
                    {
                        bool ok = true;
                        #pragma unroll
                        for(int m = 0; m < M; ++m) w[m].load(aw + (size_t)(ai * M + m) * 2);
                        #pragma unroll
                        for(int m = 0; m < M; ++m) ok = ok && w[m].ready(tg);
                        if(ok) break;
                        if(gd.stop())
                        {
                            dead = 1;
                            break;
                        }
                    }
                    #pragma unroll
                    for(int m = 0; m < M; ++m) y[m] = 0.0 + w[m].value();
                }
            }
            #pragma unroll
            for(int m = 0; m < M; ++m)
            {
                const double z = wave_sum(y[m]);
                y[m] = ((z + 0.0) + 0.0) + 0.0;   // the totals when direct
                if(NB == 1)
                {
                    if(lane == 0) wt[m][wave] = z;
                }
                else if(!direct && lane < CHIP_COPIES)
                    Wire<double>::put(cw + (size_t)(lane * CHIP_COPY_WORDS) + (wave * M + m) * 2, z, tg);
            }
            if(direct && lane == 0) store(y);
        }
        if(NB == 1) __syncthreads();
        // the totals and the state they leave: one wavefront of the first group
        if(!direct && tid >= NT - 64 && tid < NT)
        {
            double y = 0.0;
            if(lane < 4 * M)
            {
                const int w = lane / M, m = lane - w * M;
                if(NB == 1)
                    y = w < nred ? wt[m][w] : 0.0;
                else if(w < nred)
                {
                    const u64* src = cw + (size_t)((b % CHIP_COPIES) * CHIP_COPY_WORDS) + (w * M + m) * 2;
                    Wire<double> z;
                    Guard gd(ctl);
                    for(;;)
                    {
                        z.load(src);
                        if(z.ready(tg)) break;
                        if(gd.stop())
                        {
                            dead = 1;
                            break;
                        }
                    }
                    y = z.value();
                }
            }
            double tot[M];
            #pragma unroll
            for(int m = 0; m < M; ++m)
                tot[m] = ((__shfl(y, m) + __shfl(y, M + m)) + __shfl(y, 2 * M + m)) + __shfl(y, 3 * M + m);
            if(lane == 0) store(tot);
        }
        recv(tg);
        __syncthreads();
        parity ^= 1;
    };
    auto no_send = [](unsigned) {};
    auto stencil = [&](int c, const auto* o, const auto& m) {
        using W = std::remove_cv_t<std::remove_reference_t<decltype(o[0])>>;
        const int sl = grp * CT + c;
        const W yw = d3 ? o[nx23[c] & 0xffffu] : W(0), ye = d3 ? o[nx23[c] >> 16] : W(0);
        return coef_apply<W>(m, d3, o[sl * NT + ct], o[nx01[c] & 0xffffu], o[nx01[c] >> 16], yw, ye, o[nx45[c] & 0xffffu],
                             o[nx45[c] >> 16]);
    };

    bool gone = false;
    for(int it = 0; it < S.cap; ++it)
    {
        // every thread reads the state thread 0 stored before the last barrier
        if(st.done) break;
        if(!MIXED && st.mode == 1)
        {
            // restart (bicgstab_ijk.cpp:136-148): r = rhs - A x, r0 = p = r
            const unsigned tg = tag++;
            publish(halo1, [&](int c) { return x[c]; }, tg);
            #pragma unroll
            for(int c = 0; c < CT; ++c)
                if(c < nc) op[(grp * CT + c) * NT + ct] = x[c];
            receive(halo1, tg, V(0), [&](int, int q, V val) { op[HALO + q] = val; });
            #pragma unroll
            for(int s = 0; s < SL; ++s)
            {
                const int q = tid + s * CHIP_NT;
                if(q < H && hsrc[q] < 0) op[HALO + q] = MAT && hcell[s] ? (V)x64p[hcell[s] - 1u] : V(0);
            }
            __syncthreads();
            if(dead)
            {
                gone = true;
                break;
            }
            #pragma unroll
            for(int c = 0; c < CT; ++c)
                if(c < nc && act[c])
                {
                    const V rv = (V)b64[cidx[c]] - stencil(c, op, cf[c]);
                    r[c] = r0[c] = pv[c] = rv;
                }
            exchange(std::integral_constant<int, 1>(), [&](int c, double* s) { s[0] = double(r[c]) * double(r[c]); },
                     [&](unsigned tg2) { publish(halo2, [&](int c) { return r[c]; }, tg2); },
                     [&](unsigned tg2) {
                         receive(halo2, tg2, V(0), [&](int, int q, V val) {
                             hr[q] = val;
                             hp[q] = val;
                         });
                     },
                     [&](const double* tot) { restart_store(&st, tot[0]); });
            if(dead)
            {
                gone = true;
                break;
            }
            if(st.done) break;
        }
        else if(st.mode == 0)
        {
            // p = r + beta (p - w v) (bicgstab_ijk.cpp:234-235)
            const V beta = (V)st.beta, w = (V)st.w;
            #pragma unroll
            for(int c = 0; c < CT; ++c)
                if(c < nc) pv[c] = r[c] + beta * (pv[c] - w * v[c]);
            #pragma unroll
            for(int s = 0; s < SL; ++s)
            {
                const int q = tid + s * CHIP_NT;
                if(q < H) hp[q] = hr[q] + beta * (hp[q] - w * hv[q]);
            }
        }
        // v = A ph, ph = aii p
        if constexpr(MIXED)
            if(st.pending)
            {
                #pragma unroll
                for(int c = 0; c < CT; ++c)
                {
                    x64[c] += (double)x[c];
                    x[c] = V(0);
                }
            }
        #pragma unroll
        for(int c = 0; c < CT; ++c)
            if(c < nc) op[(grp * CT + c) * NT + ct] = pv[c] * a[c];
        #pragma unroll
        for(int s = 0; s < SL; ++s)
        {
            const int q = tid + s * CHIP_NT;
            if(q < H) op[HALO + q] = hp[q] * ha[s];
        }
        __syncthreads();
        #pragma unroll
        for(int c = 0; c < CT; ++c)
            if(c < nc) v[c] = stencil(c, op, cf[c]);
        auto vsums = [&](int c, double* s) {
            const double vd = v[c];
            s[0] = vd * double(r0[c]);
            s[1] = vd * vd;
        };
        auto vsend = [&](unsigned tg) { publish(halo0, [&](int c) { return v[c]; }, tg); };
        auto vrecv = [&](unsigned tg) { receive(halo0, tg, V(0), [&](int, int q, V val) { hv[q] = val; }); };
        if constexpr(KIND == CHIP_FP64)
            exchange(std::integral_constant<int, 2>(), vsums, vsend, vrecv,
                     [&](const double* tot) { v_store(&st, tot[0], tot[1], st.rr, false); });
        else
            exchange(std::integral_constant<int, 3>(),
                     [&](int c, double* s) {
                         vsums(c, s);
                         s[2] = double(r[c]) * double(r[c]);
                     },
                     vsend, vrecv, [&](const double* tot) { v_store(&st, tot[0], tot[1], tot[2], MIXED); });
        if(dead)
        {
            gone = true;
            break;
        }
        if(st.mode == 0)
        {
            // s = r - alpha v, t = A sh, sh = aii s (bicgstab_ijk.cpp:193-221)
            const V alpha = (V)st.alpha;
            #pragma unroll
            for(int c = 0; c < CT; ++c)
                if(c < nc) op[(grp * CT + c) * NT + ct] = (r[c] - alpha * v[c]) * a[c];
            #pragma unroll
            for(int s = 0; s < SL; ++s)
            {
                const int q = tid + s * CHIP_NT;
                if(q < H)
                {
                    const V sv = hr[q] - alpha * hv[q];
                    hr[q] = sv;              // s of the halo until the x phase forms r from it
                    op[HALO + q] = sv * ha[s];
                }
            }
            __syncthreads();
            #pragma unroll
            for(int c = 0; c < CT; ++c)
                if(c < nc) t[c] = stencil(c, op, cf[c]);
            V ht[SL];
            #pragma unroll
            for(int s = 0; s < SL; ++s) ht[s] = V(0);
            exchange(std::integral_constant<int, 3>(),
                     [&](int c, double* s) {
                         const double td = t[c], sd = r[c] - alpha * v[c];
                         s[0] = td * sd;
                         s[1] = td * td;
                         s[2] = sd * sd;
                     },
                     [&](unsigned tg) { publish(halo1, [&](int c) { return t[c]; }, tg); },
                     [&](unsigned tg) { receive(halo1, tg, V(0), [&](int s, int, V val) { ht[s] = val; }); },
                     [&](const double(&tot)[3]) { t_store(&st, tot); });
            if(dead)
            {
                gone = true;
                break;
            }
            // x and r (bicgstab_ijk.cpp:223-268)
            const V w = (V)st.w;
            const int branch = st.branch;
            #pragma unroll
            for(int c = 0; c < CT; ++c)
                if(c < nc)
                {
                    const V ph = pv[c] * a[c], sv = r[c] - alpha * v[c];
                    if(branch)
                    {
                        const V shv = sv * a[c];
                        if(act[c]) x[c] += alpha * ph + w * shv;
                        r[c] = sv - w * t[c];
                    }
                    else
                    {
                        if(act[c]) x[c] += alpha * ph;
                        r[c] = sv;
                    }
                }
            if(branch)
            {
                #pragma unroll
                for(int s = 0; s < SL; ++s)
                {
                    const int q = tid + s * CHIP_NT;
                    if(q < H) hr[q] = hr[q] - w * ht[s];
                }
            }
            exchange(std::integral_constant<int, 2>(),
                     [&](int c, double* s) {
                         const double rd = r[c];
                         s[0] = rd * double(r0[c]);
                         s[1] = rd * rd;
                     },
                     no_send, no_send, [&](const double(&tot)[2]) { x_store(&st, tot); });
            if(dead)
            {
                gone = true;
                break;
            }
        }
        if constexpr(MIXED)
            if(!st.done && (st.mode == 1 || st.mode == 3))
            {
                // reliable update (mode 3) or restart (mode 1): r = b - A64 (x64 + x32)
                const int restart = st.mode == 1;
                const unsigned tg = tag++;
                publish(halo1, [&](int c) { return x64[c] + (double)x[c]; }, tg);
                #pragma unroll
                for(int c = 0; c < CT; ++c)
                    if(c < nc) op64[(grp * CT + c) * NT + ct] = x64[c] + (double)x[c];
                if(tid == 0) op64[ZERO] = 0.0;
                receive(halo1, tg, 0.0, [&](int, int q, double val) { op64[HALO + q] = val; });
                #pragma unroll
                for(int s = 0; s < SL; ++s)
                {
                    const int q = tid + s * CHIP_NT;
                    if(q < H && hsrc[q] < 0) op64[HALO + q] = 0.0;
                }
                __syncthreads();
                if(dead)
                {
                    gone = true;
                    break;
                }
                double rv[CT], r0v[CT];
                #pragma unroll
                for(int c = 0; c < CT; ++c)
                {
                    rv[c] = r0v[c] = 0.0;
                    if(c >= nc || !act[c]) continue;
                    int i, j, k;
                    cell_of(stile[grp * CT + c], ct, i, j, k);
                    const Coef<double> m =
                        poisson_coef(g, couplings(g, T.f[A_RFX], T.f[A_RFY], T.f[A_RFZ], (long)cidx[c], i, j, k), i, j, k);
                    rv[c] = b64[cidx[c]] - stencil(c, op64, m);
                    r[c] = (V)rv[c];
                    if(restart) r0[c] = pv[c] = r[c];
                    r0v[c] = r0[c];
                }
                exchange(std::integral_constant<int, 2>(),
                         [&](int c, double* s) {
                             s[0] = rv[c] * rv[c];
                             s[1] = r0v[c] * double(r[c]);
                         },
                         [&](unsigned tg2) { publish(halo2, [&](int c) { return r[c]; }, tg2); },
                         [&](unsigned tg2) {
                             receive(halo2, tg2, V(0), [&](int, int q, V val) {
                                 hr[q] = val;
                                 if(restart) hp[q] = val;
                             });
                         },
                         [&](const double(&tot)[2]) {
                             ru_store(&st, ru_next(&st, tot));
                             op[ZERO] = V(0);   // the FP32 operand is next
                         });
                if(dead)
                {
                    gone = true;
                    break;
                }
            }
    }
    // ---- commit: every block arrives, or the tank's abort bit is set before the last does
    __syncthreads();
    if(tid == 0)
    {
        int ok = !gone;
        if(NB > 1)
        {
            unsigned cur = gone ? ABORT : __hip_atomic_fetch_add(ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
            const long t0 = (long)wall_clock64();
            while(!(cur & ABORT) && (int)cur < NB)
            {
                cur = __hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if(!(cur & ABORT) && (int)cur < NB && (long)wall_clock64() - t0 > WAIT_TICKS)
                {
                    // only while someone is missing: once all have arrived nobody may abort
                    unsigned want = cur;
                    if(__hip_atomic_compare_exchange_strong(ctl, &want, cur | ABORT, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT))
                        cur |= ABORT;
                    else
                        cur = want;
                }
            }
            ok = !(cur & ABORT);
        }
        dead = !ok;
        if(!ok && b == 0) T.st->chip_fail = 1;
    }
    __syncthreads();
    if(dead) return;
    const int done = st.done;
    #pragma unroll
    for(int c = 0; c < CT; ++c)
    {
        if(c >= nc || !act[c]) continue;
        const unsigned e = cidx[c];
        gx[e] = x[c];
        if constexpr(MIXED) x64p[e] = x64[c];
        if(done) continue;
        V *op_ = gp, *ov_ = gv;
        if constexpr(MIXED)
        {
            op_ = T.s[st.buf ? S_P2 : S_P];
            ov_ = T.s[st.buf ? S_V2 : S_V];
        }
        gr[e] = r[c];
        gr0[e] = r0[c];
        op_[e] = pv[c];
        ov_[e] = v[c];
        gph[e] = pv[c] * a[c];
    }
    if(b == 0 && tid == 0) *T.st = st;
}

}  // namespace bk

// the variant of the kernel for a launch (chip_geom.h: ct tile slots, chip_sl halo cells)
template<class F>
static void chip_variant(int kind, bool d3, int ct, F f)
{
    auto pick = [&](auto V_, auto K_) {
        using V = decltype(V_);
        constexpr int K = decltype(K_)::value;
        if(ct == 2)
            d3 ? f(bk::kc_solve<V, K, true, 2, chip_sl(1, 2)>) : f(bk::kc_solve<V, K, false, 2, chip_sl(0, 2)>);
        else
            d3 ? f(bk::kc_solve<V, K, true, 4, chip_sl(1, 4)>) : f(bk::kc_solve<V, K, false, 4, chip_sl(0, 4)>);
    };
    if(kind == CHIP_FP64)
        pick(0.0, std::integral_constant<int, CHIP_FP64>());
    else if(kind == CHIP_MAT)
        pick(0.0, std::integral_constant<int, CHIP_MAT>());
    else
        pick(0.0f, std::integral_constant<int, CHIP_MIXED>());
}

int chip_prepare()
{
    int bad = 0;
    for(int kind : {CHIP_FP64, CHIP_MIXED, CHIP_MAT})
        for(int d3 = 0; d3 < 2; ++d3)
            for(int ct = 2; ct <= CHIP_CT_MAX; ct *= 2)
                chip_variant(kind, d3 != 0, ct, [&](auto k) {
                    bad |= hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, CHIP_LDS_MAX) !=
                           hipSuccess;
                });
    return bad ? REEF_E_HIP : 0;
}

void bl_chip_solve(const ChipSet& S, int kind, int x, int rhs, hipStream_t s)
{
    const size_t lds = chip_lds_bytes(S.ct, kind == CHIP_MIXED ? 4 : 8, S.hmax);
    chip_variant(kind, S.d3 != 0, S.ct, [&](auto k) {
        hipLaunchKernelGGL(k, dim3((unsigned)S.blk0[S.n]), dim3(CHIP_NT), lds, s, S, x, rhs);
    });
}

}  // namespace reef
