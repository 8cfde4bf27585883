// sweep2d.hip -- 2D level-set fast sweeping on gfx950.
//
// solver2D.F90:782-978: 4 initialization sweeps (lexicographic in the
// reference, :825-867) and nsweep x 4 Gauss-Seidel sweeps over the levels
// ix+iz (:897-925).  Every sweep is evaluated here level by level -- a
// topological order of the same dependency graph, so the results equal the
// reference's bit for bit -- by one workgroup per source.  Two schedules:
// solve2d_pipe_kernel (default) pipelines one column per lane without
// barriers; solve2d_kernel (level by level, one barrier per level) is the
// cross-check, serves grids wider than kMaxStrips strips of 64 columns, and
// many sources on wide grids of short columns.
// Several sources (solveLSM) run as independent workgroups of one launch.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "stencils.h"
#include "kernels.h"

namespace fteik {

constexpr int T2 = 512;
constexpr unsigned long long kSpinLimit2D = 1ull << 24;

// localSolver.F90:160-193
__device__ __forceinline__ void signs2d(int sweep, int& sgntz, int& sgntx)
{
    sgntz = (sweep <= 2) ? 1 : -1;
    sgntx = (sweep == 1 || sweep == 3) ? 1 : -1;
}

__global__ __launch_bounds__(T2)
void solve2d_kernel(double* __restrict__ ttall, const double* __restrict__ slow,
                    int nz, int nx, double dz, double dx, double eps,
                    int nsweep, long ld_tt, const double* __restrict__ zsa_v,
                    const double* __restrict__ xsa_v,
                    const int* __restrict__ zsi_v, const int* __restrict__ xsi_v)
{
    const int src = blockIdx.x;
    double* tt = ttall + (long) src*ld_tt;
    const long ngrd = (long) nz*nx;
    __shared__ Consts<double> cs;
    if (threadIdx.x == 0) {
        // localSolver.F90:299-345
        Consts<double> c;
        c.zsa = zsa_v[src]; c.xsa = xsa_v[src]; c.ysa = 1.0;
        c.zsi = zsi_v[src]; c.xsi = xsi_v[src]; c.ysi = 1;
        c.szero = slow[(long) (c.xsi - 1)*(nz - 1) + c.zsi - 1];
        c.szero2 = c.szero*c.szero;
        c.epsSolver = eps;
        c.dz = dz; c.dx = dx; c.dy = 1.0;
        const double dz2 = dz*dz, dx2 = dx*dx;
        c.dzi = 1.0/dz; c.dxi = 1.0/dx; c.dyi = 1.0;
        c.dz2i = 1.0/dz2; c.dx2i = 1.0/dx2; c.dy2i = 1.0;
        c.dz2i_dx2i = c.dz2i*c.dx2i;
        c.dz2i_p_dx2i = c.dz2i + c.dx2i;
        c.dz2i_p_dx2i_inv = 1.0/(c.dz2i + c.dx2i);
        cs = c;
    }
    __syncthreads();
    const Consts<double> c = cs;
    for (long g = threadIdx.x; g < ngrd; g += blockDim.x) tt[g] = kHuge;
    __syncthreads();
    if (threadIdx.x < 4) {
        const int i = c.zsi + (threadIdx.x & 1), j = c.xsi + (threadIdx.x >> 1);
        tt[(long) (j - 1)*nz + i - 1] = tana2d(i, j, c);
    }
    __syncthreads();
    const int zsi = c.zsi, xsi = c.xsi;
    const int nsw = 4 + 4*nsweep;
    for (int q = 0; q < nsw; q++) {
        const bool linit = q < 4;
        const int sweep = (q & 3) + 1;
        int sgntz, sgntx;
        signs2d(sweep, sgntz, sgntx);
        // actual 1-based box (solver2D.F90:826-866 init, :377-454 iterate)
        int z0, z1, x0, x1;
        if (sgntz > 0) { z0 = linit ? max(2, zsi) : 2; z1 = nz; }
        else           { z0 = 1; z1 = linit ? zsi + 1 : nz - 1; }
        if (sgntx > 0) { x0 = linit ? max(2, xsi) : 2; x1 = nx; }
        else           { x0 = 1; x1 = linit ? xsi + 1 : nx - 1; }
        // flipped 0-based box
        const int fz0 = (sgntz > 0) ? z0 - 1 : nz - z1;
        const int fz1 = (sgntz > 0) ? z1 - 1 : nz - z0;
        const int fx0 = (sgntx > 0) ? x0 - 1 : nx - x1;
        const int fx1 = (sgntx > 0) ? x1 - 1 : nx - x0;
        if (fz0 > fz1 || fx0 > fx1) continue;
        for (int L = fz0 + fx0; L <= fz1 + fx1; L++) {
            for (int fj = fx0 + (int) threadIdx.x; fj <= fx1; fj += blockDim.x) {
                const int fi = L - fj;
                if (fi < fz0 || fi > fz1) continue;
                const int iz = (sgntz > 0) ? fi + 1 : nz - fi;
                const int ix = (sgntx > 0) ? fj + 1 : nx - fj;
                const long me = (long) (ix - 1)*nz + iz - 1;
                const double tv  = tt[(long) (ix - 1)*nz + iz - sgntz - 1];
                const double te  = tt[(long) (ix - sgntx - 1)*nz + iz - 1];
                const double tev = tt[(long) (ix - sgntx - 1)*nz + iz - sgntz - 1];
                const double t   = tt[me];
                // solver2D.F90:491-502 / localSolver.F90:222-231
                const int izc = iz - (sgntz > 0 ? 1 : 0);
                const int ixc = ix - (sgntx > 0 ? 1 : 0);
                const double s1 = rmin(slow[(long) (max(ix - 1, 1) - 1)*(nz - 1) + izc - 1],
                                       slow[(long) (min(ix, nx - 1) - 1)*(nz - 1) + izc - 1]);
                const double s2 = rmin(slow[(long) (ixc - 1)*(nz - 1) + max(iz - 1, 1) - 1],
                                       slow[(long) (ixc - 1)*(nz - 1) + min(iz, nz - 1) - 1]);
                const double s3 = slow[(long) (ixc - 1)*(nz - 1) + izc - 1];
                double tupd;
                if (linit)
                    tupd = init2d(c, sgntz, sgntx, iz, ix, tv, te, tev, t, s1,
                                  s2, s3);
                else
                    tupd = noinit2d(c, tv, te, tev, s1, s2, s3);
                tt[me] = rmin(t, tupd);
            }
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------ pipelined
// The same sweeps without a barrier per level: one workgroup per source, up
// to 8 waves, a strip of 64 flipped x columns per wave at a time (wave w
// takes strips w, w + 8, ...), one lane per column, each lane walking down
// its column one node per step (step L: node fi = L - fj of column fj), so a
// step's nodes are independent (one level).  A lane keeps its column's node
// above (fi - 1) in a register; the left column's value of the step before
// comes from lane - 1 by a wave shift, and the one of two steps before is
// the shifted value the lane received at the last step.
//
// Steps go in batches of S2.  The batch's old times and slownesses are staged
// through LDS, loaded cooperatively along the columns (a load instruction
// touches a few cache lines instead of one per lane), and the new times
// leave the same way.  Lane 0 of strip s > 0 takes the batch's S2 values of
// lane 63 of strip s - 1 from a ring in LDS after that strip's step counter
// has passed the batch; strip 0's lane 0 reads the frozen column left of the
// box.  A step itself touches registers only, so the compiler moves what
// does not depend on the step before out of the chain shift, stencil, shift:
// with the ring read, its poll, the counter and the LDS reads inside every
// step an iteration's step took 0.63 us, now 0.35 us (one source of 501 x 501
// nodes).  Values that did not change are not stored: with 256 such sources,
// whose fields do not fit the last-level cache, the stores of every value
// held a step at 0.57 us.  256 sources, 2 iterations: 9.0 -> 6.15 ms.  What
// bounds a step now is issue: about 115 instructions, two waves per SIMD.
// A strip trails the one before it by a batch: 64 of about 1,060 steps
// there.  Grids wider than the 8 waves' 512 columns had the level kernel
// before: 4 sources of 301 x 1,201 nodes 19.7 -> 8.8 ms.  (Initialization
// sweeps, whose stencil has three divisions and roots more, take about 0.8
// us a step.)
//
// The first strip of a later pass takes its left values from the field: the
// strip before it, on the last wave, stores each batch at once and then
// counts it.  With a ring there the last wave would wait for a strip that
// cannot start before the first wave has finished, which in turn waits for
// ring space along all waves.  So a strip waits for the strip before it,
// started earlier, and for ring space on the next one of its own pass, on a
// wave of its own: every wait ends, and each has a spin limit.  Rings are
// indexed by strip modulo twice the waves: a wave that starts strip s + 16
// has finished s + 8, which ended after s + 1 had read the last of strip s's
// values.
//
// The order of the node updates is a topological order of each sweep's
// dependency graph, as in the level kernel, so the results are the same bit
// for bit.
constexpr int R2D = 32;      // ring slots: strip s may lead strip s + 1 by that
constexpr int T2P = 512;     // largest workgroup (8 waves)
constexpr int S2 = 8;        // steps per batch; divides 64 and R2D
constexpr int kMaxStrips = 1024;
constexpr int NR2 = (65*S2 + 63)/64;    // old-time, and cell, pieces per lane

__device__ __forceinline__ double wave_shr1(double x)
{
    // lane i gets lane i - 1's value (lane 0 keeps its own)
    const long long b = __double_as_longlong(x);
    int lo = (int) b, hi = (int) (b >> 32);
    lo = __builtin_amdgcn_mov_dpp(lo, 0x138, 0xf, 0xf, false);
    hi = __builtin_amdgcn_mov_dpp(hi, 0x138, 0xf, 0xf, false);
    return __longlong_as_double(((long long) hi << 32) | (unsigned) lo);
}

// TMAX threads at most (TMAX/64 waves)
template <int TMAX>
__global__ __launch_bounds__(TMAX)
void solve2d_pipe_kernel(double* __restrict__ ttall,
                         const double* __restrict__ slow, int nz, int nx,
                         double dz, double dx, double eps, int nsweep,
                         long ld_tt, const double* __restrict__ zsa_v,
                         const double* __restrict__ xsa_v,
                         const int* __restrict__ zsi_v,
                         const int* __restrict__ xsi_v, int* err)
{
    const int src = blockIdx.x;
    double* tt = ttall + (long) src*ld_tt;
    const long ngrd = (long) nz*nx;
    __shared__ Consts<double> cs;
    __shared__ double ring[TMAX/32][R2D];
    __shared__ int s_done[kMaxStrips];
    // per wave: old times of a batch (64 node columns + the frozen left
    // column), its cells (65 columns), its new times;
    // rows padded against LDS bank conflicts
    __shared__ double s_t[TMAX/64][65][S2 + 1];
    __shared__ double s_c[TMAX/64][65][S2 + 1];
    __shared__ double s_o[TMAX/64][64][S2 + 1];
    __shared__ int s_fail;
    if (threadIdx.x == 0) {
        // localSolver.F90:299-345
        Consts<double> c;
        c.zsa = zsa_v[src]; c.xsa = xsa_v[src]; c.ysa = 1.0;
        c.zsi = zsi_v[src]; c.xsi = xsi_v[src]; c.ysi = 1;
        c.szero = slow[(long) (c.xsi - 1)*(nz - 1) + c.zsi - 1];
        c.szero2 = c.szero*c.szero;
        c.epsSolver = eps;
        c.dz = dz; c.dx = dx; c.dy = 1.0;
        const double dz2 = dz*dz, dx2 = dx*dx;
        c.dzi = 1.0/dz; c.dxi = 1.0/dx; c.dyi = 1.0;
        c.dz2i = 1.0/dz2; c.dx2i = 1.0/dx2; c.dy2i = 1.0;
        c.dz2i_dx2i = c.dz2i*c.dx2i;
        c.dz2i_p_dx2i = c.dz2i + c.dx2i;
        c.dz2i_p_dx2i_inv = 1.0/(c.dz2i + c.dx2i);
        cs = c;
    }
    __syncthreads();
    // (wave-uniform: to scalar registers)
    auto uni = [](double x) -> double {
        const long long b = __double_as_longlong(x);
        const int lo = __builtin_amdgcn_readfirstlane((int) b),
                  hi = __builtin_amdgcn_readfirstlane((int) (b >> 32));
        return __longlong_as_double(((long long) hi << 32) | (unsigned) lo);
    };
    Consts<double> c = cs;
    c.zsa = uni(c.zsa); c.xsa = uni(c.xsa);
    c.szero = uni(c.szero); c.szero2 = uni(c.szero2);
    c.epsSolver = uni(c.epsSolver);
    c.dz = uni(c.dz); c.dx = uni(c.dx);
    c.dzi = uni(c.dzi); c.dxi = uni(c.dxi);
    c.dz2i = uni(c.dz2i); c.dx2i = uni(c.dx2i);
    c.dz2i_dx2i = uni(c.dz2i_dx2i);
    c.dz2i_p_dx2i = uni(c.dz2i_p_dx2i);
    c.dz2i_p_dx2i_inv = uni(c.dz2i_p_dx2i_inv);
    c.zsi = __builtin_amdgcn_readfirstlane(c.zsi);
    c.xsi = __builtin_amdgcn_readfirstlane(c.xsi);
    for (long g = threadIdx.x; g < ngrd; g += blockDim.x) tt[g] = kHuge;
    __syncthreads();
    if (threadIdx.x < 4) {
        const int i = c.zsi + (threadIdx.x & 1), j = c.xsi + (threadIdx.x >> 1);
        tt[(long) (j - 1)*nz + i - 1] = tana2d(i, j, c);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int nwv = blockDim.x >> 6;
    const int zsi = c.zsi, xsi = c.xsi;
    const int nsw = 4 + 4*nsweep;
    bool fail = false;
    if (threadIdx.x == 0) s_fail = 0;
    for (int q = 0; q < nsw; q++) {
        const bool linit = q < 4;
        const int sweep = (q & 3) + 1;
        int sgntz, sgntx;
        signs2d(sweep, sgntz, sgntx);
        int z0, z1, x0, x1;
        if (sgntz > 0) { z0 = linit ? max(2, zsi) : 2; z1 = nz; }
        else           { z0 = 1; z1 = linit ? zsi + 1 : nz - 1; }
        if (sgntx > 0) { x0 = linit ? max(2, xsi) : 2; x1 = nx; }
        else           { x0 = 1; x1 = linit ? xsi + 1 : nx - 1; }
        const int fz0 = (sgntz > 0) ? z0 - 1 : nz - z1;
        const int fz1 = (sgntz > 0) ? z1 - 1 : nz - z0;
        const int fx0 = (sgntx > 0) ? x0 - 1 : nx - x1;
        const int fx1 = (sgntx > 0) ? x1 - 1 : nx - x0;
        if (fz0 > fz1 || fx0 > fx1) continue;            // uniform
        // strips of the box
        const int ns = (fx1 - fx0)/64 + 1;
        for (int i = threadIdx.x; i < ns; i += blockDim.x)
            s_done[i] = fz0 + fx0 + 64*i - 2;
        __syncthreads();
        if (s_fail) break;                                // uniform
        auto sweep_columns = [&](auto kind) {
        constexpr bool LINIT = decltype(kind)::value;
        for (int strip = wv; strip < ns && !fail; strip += nwv) {
            // first and last steps (one step early, for the left column's
            // value of two steps before)
            const int Lf = fz0 + fx0 + 64*strip - 1;
            const int Ll = fz1 + min(fx0 + 64*strip + 63, fx1);
            // This strip's columns are F .. F + 63 (flipped), lane j has
            // column fj = F + j and at step L the node on flipped row
            // fi = L - fj.  In flipped cells (cell column fj - 1 lies
            // upwind of node column fj, cell row fi - 1 upwind of node row
            // fi) a node reads the cells (fj-1, fi-1), (min(fj, nx-2),
            // fi-1) and (fj-1, min(fi, nz-2)) (solver2D.F90:491-502: slow
            // at izc over xa, xb and at ixc over max(iz-1,1), min(iz,nz-1)).
            // Per batch of S2 steps the wave loads, S2 lanes along each
            // column: the S2 old times of each of its 64 node columns (and,
            // a pass's first strip, of the column left of it) and S2 rows of
            // each of its 65 cell columns F-1 .. F+63 (cell column F-1+c
            // from row L0 - (F-1+c) - 1; a lane keeps the row above), into
            // LDS one batch ahead through registers; the new times of a
            // batch go to LDS and out to the field S2 lanes per column after
            // it.  No lane reads the field
            // values another lane of this sweep writes (old times are the
            // lane's own, ahead of its writes), so deferring the stores to
            // the end of a batch changes nothing the sweep reads.
            const int F = fx0 + 64*strip;
            const int fj = F + lane;
            const bool colA = fj <= fx1;
            const int cfj = min(fj, fx1);
            const int ix = (sgntx > 0) ? cfj + 1 : nx - cfj;
            // element offsets of the flipped columns' first nodes and cells
            auto nodecol = [&](int f) -> unsigned {         // f clamped
                f = min(f, fx1);
                return (unsigned) ((sgntx > 0) ? f : nx - 1 - f)*(unsigned) nz
                     + (sgntz > 0 ? 0u : (unsigned) nz - 1);
            };
            auto cellcol = [&](int f) -> unsigned {
                f = min(f, nx - 2);
                return (unsigned) ((sgntx > 0) ? f : nx - 2 - f)
                       *(unsigned) (nz - 1)
                     + (sgntz > 0 ? 0u : (unsigned) nz - 2);
            };
            // left values from the field; new times stored at once for the
            // next pass
            const bool field = strip % nwv == 0;
            const bool take = field && strip > 0;
            const bool hand = (strip + 1) % nwv == 0 && strip + 1 < ns;
            // node and cell of a flipped row of such a column
            auto node = [&](unsigned col, int fi) -> unsigned {
                fi = min(max(fi, fz0 - 1), fz1);
                return col + (unsigned) __mul24(fi, sgntz);
            };
            auto cell = [&](unsigned col, int fr) -> unsigned {
                fr = min(max(fr, 0), nz - 2);
                return col + (unsigned) __mul24(fr, sgntz);
            };
            double (*const st)[S2 + 1] = s_t[wv];
            double (*const sc)[S2 + 1] = s_c[wv];
            double (*const so)[S2 + 1] = s_o[wv];
            // piece i: row pe of column pc + (64/S2) i, of the node columns
            // from F (column 64: the one left of the strip) and of the cell
            // columns from F - 1; the last piece's lanes past column 64 load
            // what they do not park
            const int pe = lane % S2, pc = lane/S2;
            double rt[NR2], rc[NR2];
            unsigned ot[NR2], oc[NR2];
            #pragma unroll
            for (int i = 0; i < NR2; i++) {
                const int c = min(pc + (64/S2)*i, 64);
                ot[i] = nodecol(c < 64 ? F + c : F - 1);
                oc[i] = cellcol(F - 1 + c);
            }
            auto fetch = [&](int L0) {
                #pragma unroll
                for (int i = 0; i < NR2; i++) {
                    const int r = L0 + pe - F - pc - (64/S2)*i;
                    rt[i] = tt[node(ot[i], i < NR2 - 1 ? r
                                                       : L0 + pe - F)];
                    rc[i] = slow[cell(oc[i], r)];
                }
            };
            auto park = [&]() {                     // registers to LDS
                #pragma unroll
                for (int i = 0; i < NR2; i++) {
                    const int c = pc + (64/S2)*i;
                    if (i < NR2 - 1 || pc == 0) {
                        st[c][pe] = rt[i];
                        sc[c][pe] = rc[i];
                    }
                }
            };
            // the new times of the batch from step L0 to the field (below
            // zero: unchanged)
            auto flush = [&](int L0) {
                #pragma unroll
                for (int i = 0; i < NR2 - 1; i++) {
                    const int c = pc + (64/S2)*i, fi = L0 + pe - F - c;
                    const double v = so[c][pe];
                    if (F + c <= fx1 && fi >= fz0 && fi <= fz1 && v >= 0.0)
                        tt[ot[i] + (unsigned) __mul24(fi, sgntz)] = v;
                }
            };
            double P = tt[node(nodecol(fj), fz0 - 1)];  // node above the box
            double tep = 0.0;
            // the cell row above the batch's, of the lane's own cell column
            double cabove = slow[cell(cellcol(fj - 1), Lf - (fj - 1) - 2)];
            // waits until strip q's counter has reached `to`
            auto wait = [&](int q, int& seen, int to) {
                unsigned spins = 0;
                while (seen < to) {
                    seen = __builtin_amdgcn_readfirstlane(
                        __hip_atomic_load(&s_done[q], __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_WORKGROUP));
                    if (seen >= to) break;
                    if (++spins > kSpinLimit2D) { fail = true; break; }
                    __builtin_amdgcn_s_sleep(1);
                }
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
            };
            // the left values of the batch from step L0 are in the field
            auto wait_field = [&](int L0, int& seen) {
                wait(strip - 1, seen, min(L0 + S2 - 2, fz1 + F - 1));
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            };
            double* const rout = ring[strip % (2*nwv)];
            const double* const rin = ring[(strip + 2*nwv - 1) % (2*nwv)];
            int cl = -(1 << 30), cr = -(1 << 30);   // cached counters
            if (take) wait_field(Lf, cl);
            fetch(Lf);
            for (int L0 = Lf; L0 <= Ll; L0 += S2) {
                park();
                // (loads before stores: a wave's loads and stores are counted
                // together in order, and the next park waits for the loads)
                if (L0 + S2 <= Ll) {
                    if (take) wait_field(L0 + S2, cl);
                    fetch(L0 + S2);
                }
                if (L0 > Lf && !hand) flush(L0 - S2);
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                __builtin_amdgcn_wave_barrier();
                // lane 63 of the strip before, steps L0 - 1 .. (what lies
                // after its last step meets no node of the box)
                if (!field)
                    wait(strip - 1, cl, min(L0 + S2 - 2, fz1 + F - 1));
                auto left = [&](int k) -> double {
                    return field ? st[64][k] : rin[(L0 + k) & (R2D - 1)];
                };
                // a step, from its old time, cells (fj-1, fi-1), below it
                // and (min(fj, nx-2), fi-1), and the left value
                const int depth = colA ? L0 - fj - fz0 : -(1 << 30);
                auto step = [&](int k, double t, double cA, double cB,
                                double cC, double lft) {
                    const double sh = wave_shr1(P);
                    const double te = (lane == 0) ? lft : sh;
                    const double s1 = lmin(cA, cC);
                    const double s2 = lmin(cA, cB);
                    const bool in = (unsigned) (depth + k) <=
                                    (unsigned) (fz1 - fz0);
                    if constexpr (LINIT) {
                        if (in)
                            P = rmin(t, init2d(c, sgntz, sgntx,
                                               (sgntz > 0) ? L0 + k - fj + 1
                                                           : nz - L0 - k + fj,
                                               ix, P, te, tep, t, s1, s2, cA));
                    } else {
                        const double u = lmin(t, noinit2d_flat(
                            c, P, te, tep, s1, s2, cA));
                        P = in ? u : P;
                    }
                    tep = te;
                };
                // what the batch leaves of a node of old time t: lane 63's
                // values go to the next strip too
                auto keep = [&](double t) -> double {
                    return P != t || lane == 63 ? P : -1.0;
                };
                if constexpr (LINIT) {
                    // (unrolled it would spill)
                    #pragma unroll 1
                    for (int k = 0; k < S2; k++) {
                        const double cb = sc[lane][k];
                        step(k, st[lane][k], cabove, cb, sc[lane + 1][k],
                             left(k));
                        cabove = cb;
                        so[lane][k] = keep(st[lane][k]);
                    }
                } else {
                    double tb[S2], ca[S2], cc[S2], lf[S2];
                    #pragma unroll
                    for (int k = 0; k < S2; k++) {
                        tb[k] = st[lane][k];
                        ca[k] = sc[lane][k];
                        cc[k] = sc[lane + 1][k];
                        lf[k] = left(k);
                    }
                    #pragma unroll
                    for (int k = 0; k < S2; k++) {
                        step(k, tb[k], k ? ca[k - 1] : cabove, ca[k], cc[k],
                             lf[k]);
                        so[lane][k] = keep(tb[k]);
                    }
                    cabove = ca[S2 - 1];
                }
                // lane 63's values for steps L0 + 1 .. L0 + S2 of the next
                // strip, once it has read what the slots hold
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                __builtin_amdgcn_wave_barrier();
                if (hand) {
                    flush(L0);
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                } else if (strip + 1 < ns) {
                    wait(strip + 1, cr, L0 + S2 - R2D);
                    if (lane < S2)
                        rout[(L0 + 1 + lane) & (R2D - 1)] = so[63][lane];
                }
                if (fail) break;
                // LDS operations of one wave execute in order
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                if (lane == 0)
                    __hip_atomic_store(&s_done[strip], L0 + S2 - 1,
                                       __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
            }
            // the last batch's new times
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_wave_barrier();
            if (!fail && !hand) {
                const int nb = (Ll - Lf)/S2;
                flush(Lf + nb*S2);
            }
        }
        };
        if (linit) sweep_columns(std::true_type{});
        else sweep_columns(std::false_type{});
        if (fail && lane == 0) {
            atomicExch(err, 1);
            s_fail = 1;
        }
        __syncthreads();                  // the sweep's field is complete
    }
}

} // namespace fteik

using namespace fteik;

extern "C" int fteik_k_solve2d(double* tt, const double* slow, int nz, int nx,
                               double dz, double dx, double eps, double zsa,
                               double xsa, int zsi, int xsi, int nsweep,
                               int nsrc_batch, int ld_tt, const double* zsa_v,
                               const double* xsa_v, const int* zsi_v,
                               const int* xsi_v, int schedule, int ncu,
                               int* err, hipStream_t stream)
{
    (void) zsa; (void) xsa; (void) zsi; (void) xsi;
    // pipelined columns while every strip has a counter and rows fit 24-bit
    // products
    const int strips = (nx - 1 + 63)/64;
    // Two workgroups of the level kernel fit a CU, one of the other.  With
    // more sources than CUs on grids of several passes and short columns, of
    // which a strip's 64 skewed columns do little at a time, the level kernel
    // is the faster one: 1,024 sources of 5 x 577 nodes 8.7 ms against 11.5,
    // 40 x 1,100 22.8 against 24.7, 80 x 1,100 28.4 against 26.2, 20 x 2,000
    // 41.4 against 43.0, 40 x 2,000 48.6 against 44.3.
    const bool shortColumns = strips > T2P/64 && nsrc_batch > ncu &&
                              nz < 130 - nx/19;
    if (schedule == 0 && strips <= kMaxStrips && nz < (1 << 23) && err &&
        !shortColumns) {
        const int threads = 64*(strips < T2P/64 ? strips : T2P/64);
        hipLaunchKernelGGL((solve2d_pipe_kernel<T2P>), dim3(nsrc_batch),
                           dim3(threads), 0, stream, tt, slow, nz, nx, dz, dx,
                           eps, nsweep, (long) ld_tt, zsa_v, xsa_v, zsi_v,
                           xsi_v, err);
    } else {
        hipLaunchKernelGGL(solve2d_kernel, dim3(nsrc_batch), dim3(T2), 0,
                           stream, tt, slow, nz, nx, dz, dx, eps, nsweep,
                           (long) ld_tt, zsa_v, xsa_v, zsi_v, xsi_v);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}
