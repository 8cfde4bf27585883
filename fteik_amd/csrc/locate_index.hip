// locate_index.hip -- grid search through an index of the travel-time
// tables: the same minimum as the full search (locate.hip), found without
// evaluating most cells.
//
// For one event with weights w and residuals r = o - T(cell) the misfit is
// |u|^2/2 with u_i = w_i (r_i - t0), t0 = sum w r / sum w.  u is a linear
// projection (I - P) of w o r with |I - P| = |P| = kappa =
// sqrt(npick sum w^2) / sum w (1 for equal weights), so two cells whose
// tables differ by at most h_i satisfy
//     |u(cell)| >= |u(rep)| - kappa sqrt(sum w_i^2 h_i^2).
// The cells are grouped into blocks of 64 neighbours and the blocks into
// groups of 64; every block and group has a representative cell and the
// largest differences h from it.  A search evaluates the groups'
// representatives, then those of the blocks of the groups that can hold the
// minimum, then the cells of the blocks that can.  Every evaluation is the
// reference's expression in its order, in FP32 (locate.F90:684-705), and a
// group or block is left out only where the bound, lowered by more than
// what rounding can add, lies above an objective already found, so the
// minimum and its first cell are those of the full search bit for bit.
// Where a comparison meets a NaN nothing is left out; tables that hold
// infinities or NaN are searched without the index.
//
// 48 stations, 161 x 161 x 81 cells, 10,000 events: of 35,301 blocks and
// 726 groups an event's search evaluates the 726 representatives, about 51
// groups' blocks and 92 blocks' cells, 9,900 evaluations instead of
// 2,099,601.  The call (from 8,193 events on it keeps the full search, see
// kIndexEvents): 163 -> 4.3 ms (k_cells 1.31 ms and k_children 0.64
// ms per 5,400 events, k_group 0.09); 1500 events on 37 tables of 41 x 90 x
// 77, for which the full search makes a pass per event: 46.8 -> 0.68 ms;
// one event on the 48 tables: 336 -> 105 us.  What bounds it is latency: a
// pair's few dependent loads, then a 48-term chain of additions.
#include <hip/hip_runtime.h>
#include <float.h>
#include "kernels.h"

namespace {

using fteik::LocIndex;
using fteik::kLocLine;

constexpr int EV = fteik::kLocEv;     // events a thread carries (k_group)
constexpr float kEps = 1.1920929e-7f; // 2^-23
constexpr float kRel = 1.0e-5f;       // relative slack of the bounds
// Absolute slack: each of an objective's or a bound's at most 96 squares
// loses up to 2^-126 where it underflows, which moves its root by up to
// 1.5e-18, and kappa (below 10) multiplies the bound's.
constexpr float kTiny = 1.0e-16f;

__device__ __forceinline__ unsigned long long key_of(float obj, int cell)
{
    return ((unsigned long long) __float_as_uint(obj) << 32)
         | (unsigned long long) (unsigned) cell;
}

__device__ __forceinline__ unsigned long long wave_min64(unsigned long long k)
{
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(k, off, 64);
        k = (o < k) ? o : k;
    }
    return k;
}

__device__ __forceinline__ float wave_max(float v)
{
    for (int off = 32; off > 0; off >>= 1)
        v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// Picks are written by an earlier launch and uniform where they are used:
// read through the constant address space they are scalar operands also
// in kernels that store.
#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(4))) float* Picks;
__device__ __forceinline__ Picks picks(const float* p) { return (Picks) p; }
#else   // the host pass only parses the kernels
typedef const float* Picks;
__device__ __forceinline__ Picks picks(const float* p) { return p; }
#endif

// Lowest key so far: the word only decreases, so a stale read can only
// post or evaluate something needlessly.
__device__ __forceinline__ unsigned long long best_so_far(
    const unsigned long long* best)
{
    return __hip_atomic_load(best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void post(unsigned long long* best,
                                     unsigned long long k)
{
    if (k < best_so_far(best)) atomicMin(best, k);
}

// Norm below which a bound keeps its block: sqrt(2 objective), raised.
__device__ __forceinline__ float keep_norm(unsigned long long key)
{
    const float obj = __uint_as_float((unsigned) (key >> 32));
    return (key == ~0ull) ? __builtin_inff()
                          : sqrtf(2.0f*obj)*(1.0f + kRel);
}

// Lower bound of |u| over a block: obj at its representative, s2 =
// sum w^2 h^2; per event kap = kappa and mar, twice what rounding can move
// a computed |u|.  An objective that overflowed says that it is at least the
// largest number, not that its block holds no finite one.
__device__ __forceinline__ float low_norm(float obj, float s2, float kap,
                                          float mar)
{
    const float big = 0.5f*FLT_MAX;
    obj = obj > big ? big : obj;         // (a NaN stays one)
    return sqrtf(2.0f*obj)*(1.0f - kRel) - kap*sqrtf(s2)*(1.0f + kRel) - mar;
}

// A block stays unless its bound is certainly above: NaN keeps it.
__device__ __forceinline__ bool stays(float lb, float keep)
{
    return !(lb > keep);
}

// Cell (0-based) of position `lane` of block b, or -1 outside the grid;
// clamped: the nearest cell inside.
__device__ __forceinline__ void block_cell(const LocIndex& g, int b, int lane,
                                           int& cell, int& clamped)
{
    const int bz = b % g.nbz, bx = (b / g.nbz) % g.nbx, by = b/(g.nbz*g.nbx);
    const int z = (bz << g.lz) + (lane & ((1 << g.lz) - 1));
    const int x = (bx << g.lx) + ((lane >> g.lz) & ((1 << g.lx) - 1));
    const int y = (by << g.ly) + (lane >> (g.lz + g.lx));
    const int cz = min(z, g.nz - 1), cx = min(x, g.nx - 1),
              cy = min(y, g.ny - 1);
    clamped = (cy*g.nx + cx)*g.nz + cz;
    cell = (z == cz && x == cx && y == cy) ? clamped : -1;
}

// Block of position `lane` of group s (-1: none); the group's middle block
// is always one.
__device__ __forceinline__ int group_block(const LocIndex& g, int s, int lane)
{
    const int sz = s % g.nsz, sx = (s / g.nsz) % g.nsx, sy = s/(g.nsz*g.nsx);
    const int z = (sz << g.lz) + (lane & ((1 << g.lz) - 1));
    const int x = (sx << g.lx) + ((lane >> g.lz) & ((1 << g.lx) - 1));
    const int y = (sy << g.ly) + (lane >> (g.lz + g.lx));
    return (z < g.nbz && x < g.nbx && y < g.nby) ? (y*g.nbx + x)*g.nbz + z
                                                 : -1;
}
__device__ __forceinline__ int middle_block(const LocIndex& g, int s)
{
    const int sz = s % g.nsz, sx = (s / g.nsz) % g.nsx, sy = s/(g.nsz*g.nsx);
    const int z = min((sz << g.lz) + ((1 << g.lz) >> 1), g.nbz - 1);
    const int x = min((sx << g.lx) + ((1 << g.lx) >> 1), g.nbx - 1);
    const int y = min((sy << g.ly) + ((1 << g.ly) >> 1), g.nby - 1);
    return (y*g.nbx + x)*g.nbz + z;
}
// position of a block's representative: its middle cell (clamped)
__device__ __forceinline__ int rep_lane(const LocIndex& g)
{
    return ((1 << g.lz) >> 1) | (((1 << g.lx) >> 1) << g.lz)
         | (((1 << g.ly) >> 1) << (g.lz + g.lx));
}
__device__ __forceinline__ int rep_cell(const LocIndex& g, int b)
{
    int cell, clamped;
    block_cell(g, b, rep_lane(g), cell, clamped);
    return clamped;
}

// ------------------------------------------------------------- building
// One wave per block: the block's tables in block order (64 consecutive
// values per station, the layout k_cells reads), its representative's times
// and the largest differences from it.  HBM-bound: reads and writes the
// tables once.
__global__ __launch_bounds__(256)
void k_blocks(LocIndex g, const float* __restrict__ tab, long ldgrd)
{
    const int b = blockIdx.x*4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b >= g.nb) return;
    int cell, clamped;
    block_cell(g, b, lane, cell, clamped);
    const int rl = rep_lane(g);
    float big = 0.0f;
    bool bad = false;
    #pragma unroll 4
    for (int i = 0; i < g.ntf; i++) {
        const float v = tab[(long) i*ldgrd + clamped];
        g.perm[((long) b*g.ntf + i)*64 + lane] = v;
        const float r = __shfl(v, rl, 64);
        const float h = wave_max(fabsf(v - r));
        bad = bad || !(fabsf(v) <= FLT_MAX);
        big = fmaxf(big, fabsf(v));
        if (lane == 0) {
            g.rep[(long) i*g.nb + b] = r;
            g.h[(long) i*g.nb + b] = h;
        }
    }
    big = wave_max(big);
    if (__ballot(bad) != 0) big = __builtin_inff();
    if (lane == 0 && __float_as_uint(big) >
        __hip_atomic_load(g.tmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(g.tmax, __float_as_uint(big));
}

// Groups: the middle block's representative; h from the blocks' by the
// triangle inequality (raised for its rounding).
__global__ __launch_bounds__(256)
void k_groups(LocIndex g)
{
    const int s = blockIdx.x*blockDim.x + threadIdx.x, i = blockIdx.y;
    if (s >= g.ns) return;
    const float r = g.rep[(long) i*g.nb + middle_block(g, s)];
    float h = 0.0f;
    for (int q = 0; q < 64; q++) {
        const int b = group_block(g, s, q);
        if (b < 0) continue;
        h = fmaxf(h, fabsf(g.rep[(long) i*g.nb + b] - r)
                     + g.h[(long) i*g.nb + b]);
    }
    g.srep[(long) i*g.ns + s] = r;
    g.sh[(long) i*g.ns + s] = h*(1.0f + 4.0f*kEps);
}

// Mean |T[c + p] - T[c]| over sampled cells for candidate strides p (one
// workgroup each), to find the grid's columns in tables whose shape is not
// known: neighbouring columns have nearly the same times.
__global__ __launch_bounds__(256)
void k_stride(const float* __restrict__ tab, long ldgrd, int ntf, int ngrd,
              const int* __restrict__ p, float* __restrict__ d)
{
    __shared__ float red[4];
    const int st = p[blockIdx.x];
    float s = 0.0f;
    for (int q = threadIdx.x; q < 6144; q += 256) {
        const int i = (q % 3)*(ntf - 1)/2;
        const long c = (long) ((unsigned long long) q*2654435761ull
                               % (unsigned long long) (ngrd - st));
        s += fabsf(tab[(long) i*ldgrd + c + st] - tab[(long) i*ldgrd + c]);
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) d[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// --------------------------------------------------------------- events
// One wave per event, a lane per station: its picks as rows of nt stations
// (k_children, k_cells read them as scalars) and as station-major groups of
// EV events (k_group), skipped picks zeroed (with finite times their terms
// then add +-0, which leaves an FP32 sum unchanged), w2 = sqrt(1/2) w, the
// norm of the weights summed in index order (locate.F90:654), and the
// constants of the bounds.
__global__ __launch_bounds__(64)
void k_events(int n, int lntf, int ntf, int nt,
              const float* __restrict__ obs, const float* __restrict__ wt,
              const unsigned char* __restrict__ skip,
              const unsigned* __restrict__ tmax, fteik::LocEvents v)
{
    const int e = blockIdx.x, lane = threadIdx.x;
    const float sqrtHalf = 0.70710677f;   // SQRT(0.5) in single precision
    const long row = (long) e*lntf;
    const long base = (long) (e/EV)*ntf*EV + e % EV;
    float sw = 0.0f, sw2 = 0.0f, omax = 0.0f;
    int np = 0;
    for (int i0 = 0; i0 < nt; i0 += 64) {
        const int i = i0 + lane;
        const bool in = e < n && i < ntf, use = in && !skip[row + i];
        const float raw = in ? wt[row + i] : 0.0f;
        const float o = use ? obs[row + i] : 0.0f, w = use ? raw : 0.0f;
        const float w2 = sqrtHalf*w;
        if (i < ntf) {
            v.o8[base + (long) i*EV] = o;
            v.w8[base + (long) i*EV] = w;
            v.h8[base + (long) i*EV] = w2;
        }
        if (e < n && i < nt) {
            v.row[((long) e*nt + i)*3] = o;
            v.row[((long) e*nt + i)*3 + 1] = w;
            v.row[((long) e*nt + i)*3 + 2] = w2;
        }
        const int m = min(64, ntf - i0);
        for (int q = 0; q < m; q++)
            sw = sw + __uint_as_float(__builtin_amdgcn_readlane(
                          __float_as_uint(raw), q));
        sw2 += w*w;
        omax = fmaxf(omax, fabsf(o));
        np += __popcll(__ballot(use));
    }
    for (int off = 32; off > 0; off >>= 1) sw2 += __shfl_xor(sw2, off, 64);
    omax = wave_max(omax);
    if (lane != 0) return;
    v.xn[e] = (e < n) ? 1.0f/sw : 0.0f;
    if (e >= n) return;
    v.best[e] = ~0ull;
    v.kap[e] = sqrtf((float) np*sw2)/sw*(1.0f + kRel);
    // a computed residual is off by at most about (npick + 12) roundings of
    // the largest residual; twice that for each of the two cells compared
    const float rmax = omax + __uint_as_float(*tmax);
    v.mar[e] = 4.0f*(float) (np + 16)*kEps*rmax*sqrtf(sw2) + kTiny;
}

// --------------------------------------------------------------- search
// Objectives at the groups' representatives: a thread has one group and EV
// events, whose picks are scalar operands.
__global__ __launch_bounds__(64)
void k_group(LocIndex g, fteik::LocEvents v, int e0, int n)
{
    const int s = blockIdx.x*64 + threadIdx.x;
    const int q0 = e0 + (int) blockIdx.y*EV;
    const int cs = min(s, g.ns - 1);
    const Picks o = picks(v.o8 + (long) (q0/EV)*g.ntf*EV);
    const Picks w = picks(v.w8 + (long) (q0/EV)*g.ntf*EV);
    const Picks w2 = picks(v.h8 + (long) (q0/EV)*g.ntf*EV);
    float t0[EV], ob[EV], s2[EV], xn[EV];
    #pragma unroll
    for (int q = 0; q < EV; q++) { t0[q] = ob[q] = s2[q] = 0.0f;
                                   xn[q] = v.xn[q0 + q]; }
    #pragma unroll 8
    for (int i = 0; i < g.ntf; i++) {
        const float T = g.srep[(long) i*g.ns + cs];
        #pragma unroll
        for (int q = 0; q < EV; q++) {
            const float res = xn[q]*(o[i*EV + q] - T);
            t0[q] = t0[q] + w[i*EV + q]*res;
        }
    }
    #pragma unroll 4
    for (int i = 0; i < g.ntf; i++) {
        const float T = g.srep[(long) i*g.ns + cs];
        const float h = g.sh[(long) i*g.ns + cs];
        #pragma unroll
        for (int q = 0; q < EV; q++) {
            const float est = T + t0[q];
            const float res = w2[i*EV + q]*(o[i*EV + q] - est);
            ob[q] = ob[q] + res*res;
            const float wh = w2[i*EV + q]*h;
            s2[q] = s2[q] + wh*wh;
        }
    }
    const int cell = rep_cell(g, middle_block(g, cs));
    #pragma unroll
    for (int q = 0; q < EV; q++) {
        const int e = q0 + q;
        if (e >= e0 + n) break;                        // uniform
        const unsigned long long k = wave_min64(s < g.ns ? key_of(ob[q], cell)
                                                         : ~0ull);
        if (threadIdx.x == 0) post(v.best + e, k);
        // s2 sums w2^2 h^2 = w^2 h^2 / 2
        if (s < g.ns)
            g.lbs[(long) s*g.eb + (e - e0)] =
                low_norm(ob[q], 2.0f*s2[q], v.kap[e], v.mar[e]);
    }
}

// Objective at one cell per lane: T, the lane's times of NT stations, and
// the event's picks, NT too: those past the network are zeros, whose terms
// add +-0.
template <int NT>
__device__ __forceinline__ float misfit(Picks row, float xn,
                                        const float (&T)[NT])
{
    float t0 = 0.0f, ob = 0.0f;
    #pragma unroll
    for (int i = 0; i < NT; i++) {
        const float res = xn*(row[3*i] - T[i]);
        t0 = t0 + row[3*i + 1]*res;
    }
    #pragma unroll
    for (int i = 0; i < NT; i++) {
        const float est = T[i] + t0;
        const float res = row[3*i + 2]*(row[3*i] - est);
        ob = ob + res*res;
    }
    return ob;
}

// Blocks of the groups that stay: one wave per group and 64 events, a lane
// per block, the blocks' representatives and differences in registers.  Each
// (group, event) that stays is entered in a list with its 64 blocks' bounds;
// the list holds every pair of the batch, so it cannot overflow.
// COUNT: and counts the blocks left (the registers that takes cost 4 % of a
// search, so searches without a limit do without).
template <int NT, bool COUNT>
__global__ __launch_bounds__(64)
void k_children(LocIndex g, fteik::LocEvents v, int e0, int n)
{
    // a group's waves adjoin: they read the same blocks, and its pairs adjoin
    // in the list
    const int nc = (n + 63)/64;
    const int s = blockIdx.x / nc, lane = threadIdx.x;
    const int b = group_block(g, s, lane);
    const int cb = b < 0 ? middle_block(g, s) : b;
    const int cell = rep_cell(g, cb);
    float T[NT], H[NT];
    const int q0 = ((int) blockIdx.x - s*nc)*64, q = q0 + lane;
    unsigned long long low = ~0ull;
    float keep = 0.0f;
    bool st = false;
    if (q < n) {
        low = best_so_far(v.best + e0 + q);
        keep = keep_norm(low);
        st = stays(g.lbs[(long) s*g.eb + q], keep);
    }
    unsigned long long m = __ballot(st);
    if (m == 0) return;
    // stations past the network repeat its last (finite) times
    #pragma unroll
    for (int i = 0; i < NT; i++) {
        T[i] = g.rep[(long) min(i, g.ntf - 1)*g.nb + cb];
        H[i] = g.h[(long) min(i, g.ntf - 1)*g.nb + cb];
    }
    int at = 0, left = 0;
    if (lane == 0) at = atomicAdd(g.npair, __popcll(m));
    at = __builtin_amdgcn_readfirstlane(at);
    for (; m; m &= m - 1, at++) {
        const int w = __ffsll((long long) m) - 1, e = e0 + q0 + w;
        const Picks row = picks(v.row + (long) e*NT*3);
        const float ob = misfit<NT>(row, v.xn[e], T);
        float s2 = 0.0f;
        #pragma unroll
        for (int i = 0; i < NT; i++) {
            const float wh = row[3*i + 2]*H[i];
            s2 = s2 + wh*wh;
        }
        const unsigned long long k = wave_min64(b >= 0 ? key_of(ob, cell)
                                                       : ~0ull);
        // lane w holds the event's minimum as it was at the start
        if (lane == w && k < low) atomicMin(v.best + e, k);
        if (lane == 0) {
            g.pair[2*(long) at] = s;
            g.pair[2*(long) at + 1] = e;
        }
        const float lb = b >= 0 ? low_norm(ob, 2.0f*s2, v.kap[e], v.mar[e])
                                : __builtin_inff();
        g.lbc[(long) at*64 + lane] = lb;
        if (COUNT) {
            // (by the minimum at the wave's start: rather too many)
            const float kp = __uint_as_float((unsigned)
                __builtin_amdgcn_readlane((int) __float_as_uint(keep), w));
            left += __popcll(__ballot(b >= 0 && stays(lb, kp)));
        }
    }
    if (COUNT && lane == 0)
        atomicAdd(g.npair + (1 + (blockIdx.x & 63))*kLocLine, left);
}

// Cells of the blocks that stay: one wave per (group, event) of the list, a
// lane per cell of a block.  A block's times are 64 consecutive values per
// station, all loaded before the first is used; the kernel is bound by
// their latency and L2 traffic (256 NT bytes per block and event), so the
// launch is many waves, and each XCD (workgroups are dealt to the eight in
// turn) takes a contiguous part of the list, whose pairs share groups.
//
// With few events the list is short: `sl` waves (a power of two) share a
// pair's blocks.
//
// With more than `limit` blocks left in the batch (~0: no limit) none is
// evaluated and `over` is set: the caller searches in full.
template <int NT>
__global__ __launch_bounds__(64)
void k_cells(LocIndex g, fteik::LocEvents v, int sl, unsigned limit,
             unsigned* __restrict__ over)
{
    const int lane = threadIdx.x;
    if (limit != ~0u) {
        unsigned left = (unsigned) g.npair[(1 + lane)*kLocLine];
        for (int off = 32; off > 0; off >>= 1)
            left += __shfl_xor(left, off, 64);
        const bool up = left > limit;
        if (blockIdx.x == 0 && lane == 0) *over = up;
        if (up) return;
    }
    const int np = *g.npair*sl, per = (np + 7)/8, xcd = blockIdx.x & 7;
    const int p1 = min(np, (xcd + 1)*per);
    for (int ps = xcd*per + ((int) blockIdx.x >> 3); ps < p1;
         ps += (int) gridDim.x >> 3) {
        const int p = ps/sl;
        const int s = __builtin_amdgcn_readfirstlane(g.pair[2*(long) p]);
        const int e = __builtin_amdgcn_readfirstlane(g.pair[2*(long) p + 1]);
        const float lb = g.lbc[(long) p*64 + lane];
        const int mine = group_block(g, s, lane);
        const Picks row = picks(v.row + (long) e*NT*3);
        unsigned long long m = __ballot(mine >= 0 &&
            ((lane ^ ps) & (sl - 1)) == 0 &&
            stays(lb, keep_norm(best_so_far(v.best + e))));
        for (; m; m &= m - 1) {
            const int q = __ffsll((long long) m) - 1;
            const int b = __builtin_amdgcn_readlane(mine, q);
            const float* const t = g.perm + (long) b*g.ntf*64 + lane;
            // the minimum again, on the way with the times: a block before
            // this one, or another wave, may have lowered it
            const unsigned long long low = best_so_far(v.best + e);
            float T[NT];
            #pragma unroll
            for (int i = 0; i < NT; i++) T[i] = t[min(i, g.ntf - 1)*64];
            int cell, clamped;
            block_cell(g, b, lane, cell, clamped);
            if (!((__ballot(stays(lb, keep_norm(low))) >> q) & 1)) continue;
            const float ob = misfit<NT>(row, v.xn[e], T);
            const unsigned long long k = wave_min64(cell >= 0
                                                    ? key_of(ob, cell)
                                                    : ~0ull);
            if (lane == 0 && k < low) atomicMin(v.best + e, k);
        }
    }
}

// Origin time at each event's optimum (locate.F90:684-688): one wave per
// event, the terms a lane each, added in station order.
__global__ __launch_bounds__(64)
void k_origin(fteik::LocEvents v, const float* __restrict__ tab, int ntf,
              int nt, long ldgrd, int lntf,
              const unsigned char* __restrict__ skip)
{
    const int e = blockIdx.x, lane = threadIdx.x;
    const int c = (int) (v.best[e] & 0xffffffffull);
    const float* const row = v.row + (long) e*nt*3;
    const float xn = v.xn[e];
    float t = 0.0f;
    for (int i0 = 0; i0 < ntf; i0 += 64) {
        const int i = min(i0 + lane, ntf - 1);
        const float res = xn*(row[3*i] - tab[(long) i*ldgrd + c]);
        const float u = row[3*i + 1]*res;
        unsigned long long use = __ballot(i0 + lane < ntf &&
                                          !skip[(long) e*lntf + i]);
        for (; use; use &= use - 1)
            t = t + __uint_as_float(__builtin_amdgcn_readlane(
                        __float_as_uint(u), __ffsll((long long) use) - 1));
    }
    if (lane == 0) v.t0[e] = t;
}

inline int ok() { return hipGetLastError() == hipSuccess ? 0 : 1; }

} // namespace

extern "C" {

int fteik_k_locate_index_nt(int ntf)
{
    static const int nt[] = {8, 16, 24, 32, 40, 48, 64, 80, 96};
    for (int v : nt) if (ntf <= v) return v;
    return 0;
}

int fteik_k_locate_strides(const float* tab, long ldgrd, int ntf, int ngrd,
                           const int* p, int np, float* d, hipStream_t s)
{
    hipLaunchKernelGGL(k_stride, dim3(np), dim3(256), 0, s, tab, ldgrd, ntf,
                       ngrd, p, d);
    return ok();
}

int fteik_k_locate_index_build(const LocIndex* g, const float* tab,
                               long ldgrd, hipStream_t s)
{
    hipLaunchKernelGGL(k_blocks, dim3((g->nb + 3)/4), dim3(256), 0, s, *g,
                       tab, ldgrd);
    hipLaunchKernelGGL(k_groups, dim3((g->ns + 255)/256, g->ntf), dim3(256),
                       0, s, *g);
    return ok();
}

int fteik_k_locate_index_events(const LocIndex* g, const fteik::LocEvents* v,
                                int n, int lntf, const float* obs,
                                const float* wt, const unsigned char* skip,
                                hipStream_t s)
{
    hipLaunchKernelGGL(k_events, dim3((n + EV - 1)/EV*EV), dim3(64), 0, s, n,
                       lntf, g->ntf, g->nt, obs, wt, skip, g->tmax, *v);
    return ok();
}

int fteik_k_locate_index_search(const LocIndex* g, const fteik::LocEvents* v,
                                int e0, int n, unsigned limit,
                                unsigned* over, int ncu, hipStream_t s)
{
    if (e0 % EV != 0 || n < 1 || n > g->eb) return 2;
    if (fteik_k_fill_u64((unsigned long long*) g->npair, fteik::kLocCounts/2,
                         0ull, s)) return 1;
    hipLaunchKernelGGL(k_group, dim3((g->ns + 63)/64, (n + EV - 1)/EV),
                       dim3(64), 0, s, *g, *v, e0, n);
    const dim3 gc((unsigned) g->ns*(unsigned) ((n + 63)/64));
    // waves of k_cells: what the registers of NT times leave resident
#define LI(N) case N: \
        if (limit == ~0u) \
            hipLaunchKernelGGL((k_children<N, false>), gc, dim3(64), 0, s, \
                               *g, *v, e0, n); \
        else \
            hipLaunchKernelGGL((k_children<N, true>), gc, dim3(64), 0, s, \
                               *g, *v, e0, n); \
        hipLaunchKernelGGL(k_cells<N>, dim3((N <= 32 ? 32 : N <= 64 ? 20 : 16) \
                                            *((ncu + 7)/8*8)), \
                           dim3(64), 0, s, *g, *v, n <= 64 ? 8 : 1, limit, \
                           over); \
        break;
    switch (g->nt) {
        LI(8) LI(16) LI(24) LI(32) LI(40) LI(48) LI(64) LI(80) LI(96)
        default: return 2;
    }
#undef LI
    return ok();
}

int fteik_k_locate_index_origin(const LocIndex* g, const fteik::LocEvents* v,
                                int n, const float* tab, long ldgrd, int lntf,
                                const unsigned char* skip, hipStream_t s)
{
    hipLaunchKernelGGL(k_origin, dim3(n), dim3(64), 0, s, *v, tab, g->ntf, g->nt, ldgrd, lntf, skip);
    return ok();
}

} // extern "C"
