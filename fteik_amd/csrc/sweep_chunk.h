// sweep_chunk.h -- the chunked column-tile sweep: one wave sweeps an 8 x 8
// tile of columns, four levels (a chunk) at a time.
//
// Same dependency order as the streamed tiles of sweep_pencil.h (level t of
// the sweep's flipped frame after levels t-1 .. t-3), with another division
// of the work:
//
//   * a workgroup is one wave and owns 64 columns, one per lane; nothing in
//     a tile is handed between waves, so a step has no counters and no
//     polls, and as many compute waves share a SIMD as registers allow
//     (the streamed tiles need a halo and a store wave per compute wave,
//     which leaves one compute wave per SIMD);
//   * tiles exchange whole chunks: after a chunk a tile posts the last
//     column and the last row of its four levels to the edge-major mailbox
//     (one 16-byte tagged entry per lane), and a tile starts a chunk when
//     its upwind neighbours have posted the same four levels;
//   * old times and cell slownesses of the next chunk are loaded
//     cooperatively, four lanes along z per column, while the current chunk
//     is computed, and parked in LDS;
//   * only nodes that changed are stored.
//
// Chunk skipping (SKIP).  A node's update is a function of its seven upwind
// neighbours; its value after a sweep is the minimum of that and its own.
// If no upwind neighbour changed since the node's last pass in the same
// direction, the update gives what it gave then, and the node, which has
// been at or below that value since, cannot change.  Every change is
// recorded per node as the (cyclic) number of the sweep that made it.  A
// neighbour is "dirty" when its number lies within the last seven sweeps or
// it changed in the running one; changes that the node's last pass in this
// direction made were seen by that pass.  A chunk with no dirty node among
// those its nodes read is not computed, and nothing of it but its four
// bytes per column is read.  Mailbox entries carry the dirty bit, and a
// skipped chunk posts entries without a value: a reader that needs one
// takes it from the field, which this launch does not change there.  The
// first eight sweeps of a record (RECORD without SKIP) compute every chunk,
// and so do later ones where much is dirty (sweep_is_busy).
// Measured (one wave, batches): 16 grids of 64 .. 192 nodes per axis, 12
// iterations, 98 -> 29 ms (streamed tiles before); 48 tables of 81 x 161 x
// 161, 2 iterations, 50 -> 31 ms; 8 of the 16 grids in mixed precision 84 ->
// 40 ms.  What bounds a tile
// is the issue rate of FP64 instructions in its active chunks and, where
// little is left to do, a mailbox round trip per skipped chunk.
// Three waves, single grids: a level of a lone tile 0.48 us (streamed tiles
// 0.68), a dense 257^3 sweep 615 us (725), its solve of 19 iterations 104 ->
// 84 ms, 101^3 with 2 iterations 6.3 -> 5.1 ms.  A dense sweep is its chain
// of chunks (193 at 1.9 us) and a hop of 4 us, a chunk and the mailbox, for
// each of 62 tiles from corner to corner; a sweep with nothing left to do is
// the hops.
#pragma once
#include "sweep_pencil.h"

namespace fteik {

constexpr int CB = 8;                  // tile edge, columns
constexpr int CK = 4;                  // levels per chunk
constexpr int CROW = 84;               // LDS row: 9 x 9 columns, padded
constexpr int CTROW = 66;              // LDS row of old times, padded
constexpr int CSLOT = (CB + 1)*(CB + 1);
constexpr int CNC = (CSLOT*CK + 63)/64;          // cell pieces per lane
// Bytes of the change record before its first and after its last node: a
// lane reads the four bytes of a chunk, which may begin or end that far
// outside its column.
constexpr int kStampPad = 64;
constexpr unsigned kMbVal = 1u << 30, kMbDirty = 1u << 31,
                   kMbSerial = kMbVal - 1;

// Number of a sweep in the change record: 1 .. 255, cyclic (0: never).
__host__ __device__ inline int stamp_code(unsigned long long count)
{
    return 1 + (int) (count % 255ull);
}

typedef unsigned int U32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int U32x2 __attribute__((ext_vector_type(2)));

// Buffer accesses: 32-bit byte offsets from a base in scalar registers, and
// an offset past the end (kOut) reads zero or writes nothing, so lanes drop
// out without a branch.  The grids that get this tile keep every buffer
// below 4 GB (chunk_fits).
constexpr unsigned kOut = 0xffffffffu;
constexpr int kDeviceCoherent = 16;         // sc1
struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ Buf(const void* p, unsigned bytes)
    {
        r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                              0x00027000);
    }
    __device__ void get(unsigned o, double& v) const
    {
        const U32x2 w = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0);
        v = __longlong_as_double(((long long) w.y << 32) | w.x);
    }
    __device__ void get(unsigned o, float& v) const
    {
        v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
    }
    __device__ void put(unsigned o, double v) const
    {
        const long long b = __double_as_longlong(v);
        U32x2 w;
        w.x = (unsigned) b;
        w.y = (unsigned) (b >> 32);
        __builtin_amdgcn_raw_buffer_store_b64(w, r, o, 0, 0);
    }
    __device__ void put(unsigned o, float v) const
    {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, o, 0, 0);
    }
    __device__ int byte(unsigned o) const
    {
        return (int) __builtin_amdgcn_raw_buffer_load_b8(r, o, 0, 0);
    }
    __device__ void put_byte(unsigned o, int v) const
    {
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char) v, r, o, 0, 0);
    }
};

// ------------------------------------------------------ mailbox entries
// A value with the launch's serial and two flags in each 64-bit word, as in
// mb_put: FP64 in two words, written and read as 16 bytes, FP32 in one.
template <typename R> struct MbEntry;
template <> struct MbEntry<double> {
    U32x4 w;
    __device__ void load(const Buf& b, unsigned o)
    {
        w = __builtin_amdgcn_raw_buffer_load_b128(b.r, o, 0, kDeviceCoherent);
    }
    static __device__ void store(const Buf& b, unsigned o, double v, unsigned f)
    {
        const long long x = __double_as_longlong(v);
        U32x4 e;
        e.x = (unsigned) x; e.y = f;
        e.z = (unsigned) (x >> 32); e.w = f;
        __builtin_amdgcn_raw_buffer_store_b128(e, b.r, o, 0, kDeviceCoherent);
    }
    __device__ void clear() { w = U32x4{0, 0, 0, 0}; }
    __device__ unsigned flags() const { return w.y; }
    __device__ bool is(unsigned serial) const
    {
        return w.y == w.w && (w.y & kMbSerial) == serial;
    }
    __device__ double value() const
    {
        return __longlong_as_double(((long long) w.z << 32) | w.x);
    }
    static constexpr int bytes = 16;
};
template <> struct MbEntry<float> {
    U32x2 w;
    __device__ void load(const Buf& b, unsigned o)
    {
        w = __builtin_amdgcn_raw_buffer_load_b64(b.r, o, 0, kDeviceCoherent);
    }
    static __device__ void store(const Buf& b, unsigned o, float v, unsigned f)
    {
        U32x2 e;
        e.x = __float_as_uint(v); e.y = f;
        __builtin_amdgcn_raw_buffer_store_b64(e, b.r, o, 0, kDeviceCoherent);
    }
    __device__ void clear() { w = U32x2{0, 0}; }
    __device__ unsigned flags() const { return w.y; }
    __device__ bool is(unsigned serial) const
    {
        return (w.y & kMbSerial) == serial;
    }
    __device__ float value() const { return __uint_as_float(w.x); }
    static constexpr int bytes = 8;
};

// LDS accesses of one wave execute in order; the compiler must not reorder
// a lane's read of another lane's value before the write it follows.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Whether a grid's field, slowness and mailboxes fit 32-bit offsets, and its
// axes the 24-bit products of the address arithmetic.
__host__ __device__ inline bool chunk_fits(long nz, long nx, long ny,
                                           unsigned long long mbBytes)
{
    const unsigned long long lim = 0xfffffff0ull;
    return 8ull*(unsigned long long) nz*nx*ny < lim && mbBytes < lim &&
           nz < (1 << 17) && nx < (1 << 20) && ny < (1 << 20);
}

// Words of a grid's record: the last changing sweep, then the number of
// chunks that a sweep changed, for the last sixteen sweeps.
constexpr int kRecordWords = 32;
template <typename R>
__device__ __forceinline__ unsigned* changed_chunks(const SweepArgs<R>& a,
                                                    unsigned count)
{
    return a.lastchg + 1 + (count & 15u);
}
// One tile as a lane sees it: geometry, addresses, and the loads and stores
// of a chunk.  Fields that a wave does not use cost it nothing.
template <typename R>
struct ChunkTile {
    static constexpr int SZ = (int) sizeof(R);
    static constexpr int EB = MbEntry<R>::bytes;
    static constexpr int kNever = 1 << 28;       // diagonal of no step

    const SweepArgs<R>& a;
    const Buf btt, bsl, bmb, bst;
    int lane, fbx, fby, fj0, fk0, jhi, khi, ez0, fz1, tlo, thi;
    unsigned nzx, ncx, nbox, tag;
    int zs, z0, cz0;
    // the lane's own column: field offset, diagonal (depB: kNever where the
    // box has no such column), ring position, first cell slot
    int lj, lk, dep, depB, me, cs;
    unsigned ocol;
    // the lane's part of the cooperative loads: piece i of the old times is
    // step lane & 3 of node column (lx, ly + 2 i), piece i of the cells
    // layer lane & 3 of a cell column (slot): (lx, ly + 2 i) for i < 4, then
    // (8, 0 .. 7) and (0 .. 7, 8), then (8, 8).  Slot (x, y), 0..8, lies
    // between node columns x - 1 and x of the tile along each axis; node
    // (lj, lk) reads slots (lj, lk) .. (lj + 1, lk + 1), and at step t
    // layers f = t - dep and f + 1 of the first (autoCode.f90:407-445; the
    // clamps are those of the cell's own column)
    int lq, lc, lx, ly, tdep, cdep4, cdep5, slot4, slot5;
    unsigned toff[4], coff[CNC];
    // the lane's halo entry: step hq of a chunk of upwind column hc (lanes
    // 0..31: the row of columns before the tile in x, 32..63: in y), and on
    // lanes 0..3 also the corner column's step `lane`.  Diagonals of the
    // lanes that read an entry (M), that read the field (D: columns before
    // the box are not written in this launch and have no mailbox), and that
    // post one; hent, cent: entry offsets at t0 = 0, hstep bytes a step, a
    // tile's own post hedge further.
    int hc, hq, hdep, cdep, hdepM, cdepM, hdepD, cdepD, pdep, hpos, hn;
    bool hx, cdir;
    unsigned hfld, cfld, hent, cent, hedge;

    // steps s of a column whose node on diagonal `dep` lies in the box, the
    // frozen layer before it included
    __device__ bool in_box(int s, int dep) const
    {
        return (unsigned) (s - ez0 - dep) <= nbox;
    }
    __device__ unsigned column(int fj, int fk) const      // first byte
    {
        return ((unsigned) (unflip(fk, a.ny, a.sy) - 1)*nzx
                + (unsigned) (unflip(fj, a.nx, a.sx) - 1)*(unsigned) a.nz)*SZ;
    }
    __device__ unsigned node(unsigned col, int fi) const  // clamped to the box
    {
        fi = min(max(fi, ez0), fz1);
        return col + (unsigned) (z0 + __mul24(fi, zs));
    }
    __device__ unsigned cell_column(int sa, int sb) const
    {
        const int nx = a.nx, ny = a.ny;
        const int cx = (a.sx > 0) ? min(max(fj0 + sa, 1), nx - 1)
                                  : min(max(nx - fj0 - sa, 1), nx - 1);
        const int cy = (a.sy > 0) ? min(max(fk0 + sb, 1), ny - 1)
                                  : min(max(ny - fk0 - sb, 1), ny - 1);
        return ((unsigned) (cy - 1)*ncx + (unsigned) (cx - 1)
                *(unsigned) (a.nz - 1))*SZ;
    }

    __device__ ChunkTile(const SweepArgs<R>& a_, int wg, int ln, bool skip)
        : a(a_), btt(a_.tt, (unsigned) a_.nz*a_.nx*a_.ny*SZ),
          bsl(a_.slow, (unsigned) (a_.nz - 1)*(a_.nx - 1)*(a_.ny - 1)*SZ),
          bmb(a_.mbx, a_.mbBytes),
          bst(a_.stamp, skip ? (unsigned) a_.nz*a_.nx*a_.ny : 0u), lane(ln)
    {
        const int nz = a.nz, nx = a.nx, ny = a.ny;
        fbx = wg / a.nby; fby = wg - fbx*a.nby;
        fj0 = a.fx0 + fbx*CB; fk0 = a.fy0 + fby*CB;
        jhi = min(fj0 + CB - 1, a.fx1); khi = min(fk0 + CB - 1, a.fy1);
        ez0 = a.fz0 - 1; fz1 = a.fz1;
        tlo = ez0 + fj0 + fk0; thi = fz1 + jhi + khi;
        nzx = (unsigned) nz*nx; ncx = (unsigned) (nz - 1)*(nx - 1);
        nbox = (unsigned) (fz1 - ez0);
        tag = (unsigned) a.serial & kMbSerial;
        // byte step and origin of node fi (flipped) of a column: z0 + fi*zs;
        // the upwind cell layer of f is layer cz0 + f*zs, f in 1 .. nz - 1
        zs = (a.sz > 0) ? SZ : -SZ;
        z0 = (a.sz > 0) ? 0 : (nz - 1)*SZ;
        cz0 = (a.sz > 0) ? -SZ : (nz - 1)*SZ;
        lj = lane & 7; lk = lane >> 3;
        const bool colB = fj0 + lj <= jhi && fk0 + lk <= khi;
        ocol = column(min(fj0 + lj, jhi), min(fk0 + lk, khi));
        dep = fj0 + fk0 + lj + lk;
        depB = colB ? dep : kNever;
        me = (lk + 1)*9 + lj + 1;
        cs = lk*9 + lj;
        lq = lane & 3; lc = lane >> 2;
        lx = lc & 7; ly = lc >> 3;
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            toff[i] = column(min(fj0 + lx, jhi), min(fk0 + ly + 2*i, khi));
            coff[i] = cell_column(lx, ly + 2*i);
        }
        const int s4x = ly ? lx : 8, s4y = ly ? 8 : lx;
        coff[4] = cell_column(s4x, s4y);
        slot4 = s4y*9 + s4x;
        coff[5] = cell_column(8, 8);
        slot5 = lc == 0 ? 80 : 81;               // 81: padding
        tdep = fj0 + fk0 + lx + ly;
        cdep4 = fj0 + fk0 + s4x + s4y;
        cdep5 = fj0 + fk0 + 16;
        hc = lane & 7; hq = (lane >> 3) & 3;
        hx = lane < 32;
        const int hj = hx ? fj0 - 1 : fj0 + hc, hk = hx ? fk0 + hc : fk0 - 1;
        const bool hdir = hx ? fbx == 0 : fby == 0;
        cdir = fbx == 0 || fby == 0;
        const bool hcol = hj <= a.fx1 && hk <= a.fy1;
        hdep = hj + hk - hq;                     // at t0: fi = t0 - hdep
        cdep = fj0 + fk0 - 2 - lane;             // corner, lanes 0..3
        hdepM = hcol && !hdir ? hdep : kNever;
        cdepM = lane < 4 && !cdir ? cdep : kNever;
        hdepD = hcol && hdir ? hdep : kNever;
        cdepD = lane < 4 && cdir ? cdep : kNever;
        // is there a tile past this edge, and a column
        const bool pwant = hx ? fj0 + CB <= a.fx1 && fk0 + hc <= khi
                              : fk0 + CB <= a.fy1 && fj0 + hc <= jhi;
        pdep = pwant ? hdep + CB : kNever;
        hpos = hx ? (hc + 1)*9 : hc + 1;
        hfld = column(min(hj, a.fx1), min(hk, a.fy1));
        cfld = column(fj0 - 1, fk0 - 1);
        // entry of (edge e, step t, row or column): x edges (e*mbnt + t)*ny
        // + row, y edges after them, (e*mbnt + t)*nx + column
        const unsigned yoff = (unsigned) ((char*) a.mby - (char*) a.mbx);
        hn = hx ? ny : nx;
        hent = (hx ? 0u : yoff) +
            (((unsigned) ((hx ? fbx : fby) - 1)*a.mbnt + hq)*hn
             + (hx ? hk : hj))*EB;
        cent = (((unsigned) (fbx - 1)*a.mbnt + lane)*ny + fk0 - 1)*EB;
        hedge = (unsigned) a.mbnt*hn*EB;
    }
    __device__ bool empty() const { return fj0 > jhi || fk0 > khi; }

    // ---- old times and cells.  fetch_c(t0): layers t0 - dep + 3 + (0..3):
    // with the three before them the seven layers of chunk t0
    __device__ unsigned t_at(int i, int t0) const
    {
        return node(toff[i], t0 + lq - tdep - 2*i);
    }
    __device__ void fetch_t(int t0, R (&v)[4]) const
    {
        #pragma unroll
        for (int i = 0; i < 4; i++) btt.get(t_at(i, t0), v[i]);
    }
    __device__ void fetch_c(int t0, R (&v)[CNC]) const
    {
        #pragma unroll
        for (int i = 0; i < CNC; i++) {
            int f = t0 + 3 + lq - (i < 4 ? tdep + 2*i : i == 4 ? cdep4
                                                                 : cdep5);
            f = min(max(f, 1), a.nz - 1);
            const unsigned o = coff[i] + (unsigned) (cz0 + __mul24(f, zs));
            bsl.get(i < 5 ? o : lc == 0 ? o : kOut, v[i]);
        }
    }
    __device__ void park_t(R* tbuf, const R (&v)[4]) const
    {
        #pragma unroll
        for (int i = 0; i < 4; i++) tbuf[lq*CTROW + 16*i + lc] = v[i];
    }
    __device__ void park_c(R* rows, const R (&v)[CNC]) const
    {
        R* const p = rows + lq*CROW;
        #pragma unroll
        for (int i = 0; i < 4; i++) p[ly*9 + lx + 18*i] = v[i];
        p[slot4] = v[4];
        p[slot5] = v[5];
    }
    // own times of the three steps before t0
    __device__ void fetch_hist(int t0, R (&v)[3]) const
    {
        #pragma unroll
        for (int q = 0; q < 3; q++) btt.get(node(ocol, t0 - 3 + q - dep), v[q]);
    }

    // ---- halo
    __device__ void load_entries(int t0, MbEntry<R>& e0, MbEntry<R>& e1) const
    {
        const unsigned t = (unsigned) t0;
        e0.load(bmb, in_box(t0, hdepM) ? hent + t*hn*EB : kOut);
        e1.load(bmb, in_box(t0, cdepM) ? cent + t*a.ny*EB : kOut);
    }
    // clean: upwind tiles (bit 0 in x, 1 in y, 2 in both) whose entries for
    // the chunk need not have been posted
    __device__ bool ready(int t0, const MbEntry<R>& e0, const MbEntry<R>& e1,
                          int clean) const
    {
        return __ballot((in_box(t0, hdepM) && !e0.is(tag) &&
                         !(clean & (hx ? 1 : 2))) ||
                        (in_box(t0, cdepM) && !e1.is(tag) &&
                         !(clean & 4))) == 0;
    }
    // field values (and change bytes) of the lanes without a mailbox; only
    // tiles on the box's first row of tiles along an axis have such lanes
    __device__ void load_direct(int t0, bool stamps, R& d0, R& d1, int& b0,
                                int& b1) const
    {
        if (cdir) {
            const unsigned o0 = in_box(t0, hdepD) ? node(hfld, t0 - hdep)
                                                  : kOut;
            const unsigned o1 = in_box(t0, cdepD) ? node(cfld, t0 - cdep)
                                                  : kOut;
            btt.get(o0, d0);
            btt.get(o1, d1);
            if (stamps) {
                b0 = bst.byte(o0 == kOut ? kOut : o0/SZ);
                b1 = bst.byte(o1 == kOut ? kOut : o1/SZ);
            }
        }
    }
    // flags of an entry; none where it is not this sweep's (a chunk known
    // clean before its entries are posted)
    __device__ unsigned flags(const MbEntry<R>& e) const
    {
        return e.is(tag) ? e.flags() : 0u;
    }
    // values of a chunk's halo from its entries; those of skipped chunks
    // are read from the field
    __device__ void halo_values(int t0, const MbEntry<R>& e0,
                                const MbEntry<R>& e1, R d0, R d1, R& v0,
                                R& v1) const
    {
        const bool h0 = flags(e0) & kMbVal, h1 = flags(e1) & kMbVal;
        const bool m0 = in_box(t0, hdepM) && !h0;
        const bool m1 = in_box(t0, cdepM) && !h1;
        v0 = h0 ? e0.value() : d0;
        v1 = h1 ? e1.value() : d1;
        if (__ballot(m0 || m1) != 0) {
            R x0, x1;
            btt.get(m0 ? node(hfld, t0 - hdep) : kOut, x0);
            btt.get(m1 ? node(cfld, t0 - cdep) : kOut, x1);
            v0 = m0 ? x0 : v0;
            v1 = m1 ? x1 : v1;
        }
    }

    // ---- change record
    __device__ bool dirty_byte(int b) const
    {
        int age = a.code - b;
        age += age < 0 ? 255 : 0;
        return b != 0 && age <= 7;
    }
    // own change bytes of a chunk, step q in byte q
    __device__ unsigned load_stamp(int t0) const
    {
        const int f0 = t0 - dep;
        const long p = (long) (ocol/SZ) + ((a.sz > 0) ? f0
                                                      : a.nz - 1 - f0 - 3);
        unsigned w;
        __builtin_memcpy(&w, a.stamp + p, 4);
        return (a.sz > 0) ? w : __builtin_bswap32(w);
    }
    __device__ unsigned own_dirty(int t0, unsigned st) const
    {
        unsigned m = 0;
        #pragma unroll
        for (int q = 0; q < CK; q++)
            if (in_box(t0 + q, depB) && dirty_byte((st >> (8*q)) & 255))
                m |= 1u << q;
        return m;
    }
    // dirty halo nodes of the lane's entries: step hq (hd), lane (cd)
    __device__ void halo_dirty(int t0, const MbEntry<R>& e0,
                               const MbEntry<R>& e1, int b0, int b1, bool& hd,
                               bool& cd) const
    {
        hd = (in_box(t0, hdepM) && (flags(e0) & kMbDirty)) ||
             (in_box(t0, hdepD) && dirty_byte(b0));
        cd = (in_box(t0, cdepM) && (flags(e1) & kMbDirty)) ||
             (in_box(t0, cdepD) && dirty_byte(b1));
    }

    // Marks (in LDS, a byte per chunk) the chunks with a dirty node in the
    // tile's columns or in the upwind columns without a mailbox: columns 0
    // .. 63, then 64 .. 71 (before it in x), 72 .. 79 (in y) and 80.  A lane
    // reads 16 bytes of a column at a time, consecutive lanes consecutive
    // pieces.
    __device__ void scan(unsigned char* dirt, int ng) const
    {
        // nodes fi = ez0 .. fz1, in memory order from byte lo of a column
        const unsigned lo = (a.sz > 0) ? ez0 : a.nz - 1 - fz1;
        const int n = (int) nbox + 1, np = (n + 15)/16;
        const int total = (cdir ? 81 : 64)*np;
        #pragma unroll 4
        for (int p0 = 0; p0 < total; p0 += 64) {
            const int p = p0 + lane, col = p/np, o = (p - col*np)*16;
            const int cj = col < 64 ? fj0 + (col & 7)
                         : col < 72 || col == 80 ? fj0 - 1 : fj0 + (col & 7);
            const int ck = col < 64 ? fk0 + (col >> 3)
                         : col < 72 ? fk0 + (col & 7) : fk0 - 1;
            bool use = p < total && cj <= a.fx1 && ck <= a.fy1;
            if (col >= 64)
                use = use && (col < 72 ? fbx == 0 : col < 80 ? fby == 0 : cdir);
            const unsigned base = column(min(max(cj, 0), a.fx1),
                                         min(max(ck, 0), a.fy1))/SZ + lo;
            unsigned w[4] = {0, 0, 0, 0};
            if (use) __builtin_memcpy(w, a.stamp + base + o, 16);
            unsigned m = 0;
            #pragma unroll
            for (int q = 0; q < 16; q++)
                m |= dirty_byte((w[q >> 2] >> (8*(q & 3))) & 255) ? 1u << q
                                                                  : 0u;
            for (; m; m &= m - 1) {
                const int q = o + __ffs((int) m) - 1;
                if (q >= n) break;
                const int fi = (a.sz > 0) ? ez0 + q : fz1 - q;
                const int g = (fi + cj + ck - tlo) >> 2;      // or below 0
                if (g >= -1 && g < ng) dirt[g + 1] = 1;
            }
        }
    }
    // ---- results.  Posts the chunk's last column and last row (lanes
    // 0..31: row hc of the last column, 32..63: column hc of the last row;
    // step hq); rows: the chunk's ring rows, own: a column's dirty steps
    // (by lane of the column)
    __device__ int post_lane() const { return hx ? 8*hc + 7 : 56 + hc; }
    __device__ void post(int t0, bool val, const R* rows, unsigned own) const
    {
        const unsigned f = tag | (val ? kMbVal : 0u)
                         | (((own >> hq) & 1u) ? kMbDirty : 0u);
        R pv = R(0);
        if (val) pv = rows[hq*CROW + (hx ? (hc + 1)*9 + 8 : 73 + hc)];
        MbEntry<R>::store(bmb, in_box(t0, pdep)
                          ? hent + hedge + (unsigned) t0*hn*EB : kOut, pv, f);
    }
    // the chunk's new times, in the order of its old ones
    __device__ void collect(const R* rows, R (&out)[4]) const
    {
        const R* const p = rows + lq*CROW + (ly + 1)*9 + lx + 1;
        #pragma unroll
        for (int i = 0; i < 4; i++) out[i] = p[18*i];
    }
    // nchg: chunks that changed (uniform, with RECORD)
    template <bool RECORD>
    __device__ void store(int t0, const R (&old)[4], const R (&out)[4],
                          R& dmax, int& nchg) const
    {
        bool changed = false;
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool ch = out[i] != old[i];
            const unsigned o = ch ? t_at(i, t0) : kOut;
            btt.put(o, out[i]);
            if (RECORD) bst.put_byte(ch ? o/SZ : kOut, a.code);
            changed = changed || ch;
            dmax = ch ? rmax(dmax, old[i] - out[i]) : dmax;
        }
        if (RECORD) nchg += __ballot(changed) != 0 ? 1 : 0;
    }
    template <bool RECORD>
    __device__ void finish(R dmax, int nchg) const
    {
        if (a.maxdelta && dmax > R(0)) {
            const double dd = (double) dmax;
            atomicMax((unsigned long long*) a.maxdelta,
                      (unsigned long long) __double_as_longlong(dd));
        }
        if (RECORD && nchg > 0 && lane == 0) {
            __hip_atomic_store(a.lastchg, a.count, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            atomicAdd(changed_chunks(a, a.count), (unsigned) nchg);
        }
    }
};

// Nothing changed in the last seven sweeps: this one changes nothing (every
// tile decides alike, from launches before this one: where nothing is dirty
// no tile of this launch posts a change).
template <typename R>
__device__ __forceinline__ bool sweep_is_clean(const SweepArgs<R>& a)
{
    return __hip_atomic_load(a.lastchg, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT) + 7u < a.count;
}

// A chunk that looks for dirty nodes and has some takes longer than one that
// is computed in any case (three waves, lone tile: 2.7 against 1.95 us; one
// wave: a tenth longer), and the more tiles a sweep has to cross, the less it
// gains from a clean chunk: it waits for the tiles that have work.  So a sweep
// computes every chunk where the last seven changed more than `share` (64ths)
// of them, all seven together: about 1.2 to 1.5 times the chunks that have a
// dirty node, more on grids of few tiles, whose changes stay in one place.
// Every tile of a grid decides alike, from launches before this one.
template <typename R>
__device__ __forceinline__ bool sweep_is_busy(const SweepArgs<R>& a, int share)
{
    unsigned n = 0;
    #pragma unroll
    for (unsigned k = 1; k <= 7; k++) n += *changed_chunks(a, a.count - k);
    const int chunks = a.nbx*a.nby*((a.fz1 - a.fz0 + 2*CB)/CK + 1);
    return (long) n*64 > (long) chunks*share;
}
// Single grids.  Where a sweep that skips is as fast as one that computes
// every chunk, smooth random velocities: 25 % of the chunks at 33^3 nodes (6
// tiles to cross), 7 % at 129^3 (30), 5 % at 257^3 (62).  129 x 257 x 257
// nodes, 8 iterations, most chunks dirty in six of them: 45.0 ms skipping in
// all, 36.5 with this line (streamed tiles 39.9).
template <typename R>
__device__ __forceinline__ int single_share(const SweepArgs<R>& a)
{
    return max(4, 96/max(a.nbx + a.nby - 2, 2));
}
// Batches.  a.load: where the SIMDs have their waves of other tiles every
// clean chunk counts.  6 grids of 128^3 nodes, rough velocities, 12
// iterations: 47.3 ms skipping in all, 41 with this line (streamed 44.5); 16
// smooth ones of 64 .. 192 nodes per axis 34.9 and 34.7.  Grids of few tiles
// never compute every chunk: 256 of 200 x 20 x 20, 32.6 ms skipping, 36.5
// with a line of 3/4 of the chunks.
template <typename R>
__device__ __forceinline__ int batch_share(const SweepArgs<R>& a)
{
    const int hops = a.nbx + a.nby - 2;
    return hops < 6 ? 7*64
                    : max(max(4, a.load), max(192/hops, 1536/(hops*hops)));
}
// The grid's first tile clears the next sweep's count.
template <typename R>
__device__ __forceinline__ void clear_count(const SweepArgs<R>& a, int wg)
{
    if (wg == 0 && threadIdx.x == 0) *changed_chunks(a, a.count + 1) = 0;
}

template <typename R, bool CUBE>
__device__ __forceinline__ Consts<R> chunk_consts(const SweepArgs<R>& a)
{
    Consts<R> c = *a.cst;
    if (CUBE) {
        // equal spacings: the constants of the axes are equal bit for bit
        // (source3d_init_kernel forms them alike), and fewer of them fit the
        // scalar registers
        c.dx = c.dy = c.dz;
        c.dx2i = c.dy2i = c.dz2i;
        c.dz2dy2 = c.dx2dy2 = c.dz2dx2;
        c.dz2i_dy2i = c.dx2i_dy2i = c.dz2i_dx2i;
        c.dz2i_p_dy2i = c.dx2i_p_dy2i = c.dz2i_p_dx2i;
        c.dz2i_p_dy2i_inv = c.dx2i_p_dy2i_inv = c.dz2i_p_dx2i_inv;
    }
    return c;
}

// Times read or written one step earlier (the x, y and xy neighbours' and
// the own), which are the next step's other neighbours.
template <typename R> struct ChunkPast { R w, s, sw, v; };

// The four levels of a chunk.  rp, rc: ring rows of the chunk before and of
// this one; ch, co: cell rows of the chunk before's new layers and of this
// one's: layer t - dep + m of slot uu is row 1 + q + m of the two taken
// together; ud and du need one layer more than uu, dd two.  Returns the
// lane's changed steps (a bit each, with CHG).  mid() is called before the
// last level.
template <typename R, bool CUBE, bool CHG, typename F>
__device__ __forceinline__ unsigned chunk_levels(
    const ChunkTile<R>& T, const Consts<R>& c, int t0, const R* rp, R* rc,
    const R* ch, const R* co, const R* tbuf, ChunkPast<R>& h, F mid)
{
    const int me = T.me;
    ch += T.cs;
    co += T.cs;
    auto cell4 = [&](int m, R (&z)[4]) {
        const int o[4] = {0, 9, 1, 10}, d[4] = {0, 1, 1, 2};
        #pragma unroll
        for (int x = 0; x < 4; x++) {
            const int row = 1 + m + d[x];
            z[x] = row < 4 ? ch[row*CROW + o[x]] : co[(row - 4)*CROW + o[x]];
        }
    };
    R cu[4];
    cell4(0, cu);
    unsigned chg = 0;
    #pragma unroll
    for (int q = 0; q < CK; q++) {
        const R* const r1 = q >= 1 ? rc + (q - 1)*CROW : rp + 3*CROW;
        const R* const r2 = q >= 2 ? rc + (q - 2)*CROW : rp + (q + 2)*CROW;
        R cd[4];
        cell4(q + 1, cd);
        Slw<R> sl;
        slowness7_ud<R>(cu, cd, sl);
        #pragma unroll
        for (int x = 0; x < 4; x++) cu[x] = cd[x];
        Nbr<R> nb;
        nb.tv = h.v;
        nb.tev = h.w;
        nb.tnv = h.s;
        nb.tnve = h.sw;
        nb.te = r1[me - 1];
        nb.tn = r1[me - 9];
        nb.ten = r2[me - 10];
        const R v = tbuf[q*CTROW + T.lane];
        R vn = noinit3d<R, CUBE>(c, nb, sl, v);
        // updated: in the box past the frozen layer
        vn = (unsigned) (t0 + q - T.ez0 - 1 - T.depB) < T.nbox ? vn : v;
        if (CHG) chg |= vn != v ? 1u << q : 0u;
        rc[q*CROW + me] = vn;
        h.v = vn; h.w = nb.te; h.s = nb.tn; h.sw = nb.ten;
        wave_lds_fence();
        if (q == CK - 2) mid();
    }
    return chg;
}

// ---------------------------------------------------------- one wave
template <typename R, bool SKIP, bool RECORD, bool CUBE>
__device__ __forceinline__ void chunk_body(const SweepArgs<R>& a, const int wg)
{
    // ring[r]: times of the tile's 9 x 9 columns (the upwind column row, row
    // and corner first) at a step; rows 0..3 and 4..7 are the halves of two
    // consecutive chunks.  cbuf: cell layers, likewise.  tbuf: the chunk's
    // old times.
    __shared__ R ring[8*CROW];
    __shared__ R cbuf[8*CROW];
    __shared__ R tbuf[CK*CTROW];
    const int lane = threadIdx.x;
    const ChunkTile<R> T(a, wg, lane, RECORD);
    if (T.empty() || (SKIP && sweep_is_clean(a))) return;
    // (one body for both: the two side by side spill registers)
    const bool skip = SKIP && !sweep_is_busy(a, batch_share(a));
    const Consts<R> c = chunk_consts<R, CUBE>(a);
    // What the chunk before left: prevDirty, its steps 1..3 hold a dirty
    // node (own, halo); loaded: its times, cells and halo are in LDS.
    bool prevDirty = false, loaded = false;
    ChunkPast<R> past = {R(0), R(0), R(0), R(0)};
    MbEntry<R> e0, e1;                  // the coming chunk's entries
    R d0 = R(0), d1 = R(0);             // field values of direct lanes
    int b0 = 0, b1 = 0;                 // their change bytes
    R tnx[4], cnx[CNC];
    unsigned stn = 0;
    R dmax = R(0);
    int nchg = 0;
    int half = 0;                       // ring and cell half of the chunk
    if (skip) stn = T.load_stamp(T.tlo - CK);
    T.load_entries(T.tlo - CK, e0, e1);
    T.load_direct(T.tlo - CK, skip, d0, d1, b0, b1);
    for (int t0 = T.tlo - CK; t0 <= T.thi; t0 += CK, half ^= 4) {
        const bool more = t0 + CK <= T.thi;
        // ---- the upwind neighbours' chunk
        {
            unsigned spins = 0;
            while (!T.ready(t0, e0, e1, 0)) {
                if (++spins > kSpinLimit) {
                    if (lane == 0) atomicExch(a.err, 1);
                    return;
                }
                __builtin_amdgcn_s_sleep(1);
                T.load_entries(t0, e0, e1);
            }
        }
        // ---- dirty nodes among those the chunk reads: steps t0 - 3 .. t0
        // + 2 of the own and the halo columns
        unsigned own = 0;
        bool active = !skip && t0 >= T.tlo;
        bool nextDirty = false;
        if (skip) {
            own = T.own_dirty(t0, stn);
            if (more) stn = T.load_stamp(t0 + CK);
            bool hd, cd;
            T.halo_dirty(t0, e0, e1, b0, b1, hd, cd);
            const bool now = (own & 7u) || (hd && T.hq < 3) ||
                             (cd && lane < 3);
            nextDirty = (own & 14u) || (hd && T.hq > 0) || (cd && lane > 0);
            active = t0 >= T.tlo && (prevDirty || __ballot(now) != 0);
        }
        R* const rc = ring + half*CROW;             // rows of this chunk
        R* const rp = ring + (half ^ 4)*CROW;       // of the one before
        R* const ch = cbuf + half*CROW;
        R* const co = cbuf + (half ^ 4)*CROW;
        R tw[4];
        if (active) {
            if (!loaded) {
                // all of it at once: the chunk's old times, both parts of
                // its cell layers, the three steps before it
                R hist[3];
                T.fetch_c(t0 - CK, cnx);
                T.park_c(ch, cnx);
                T.fetch_t(t0, tnx);
                T.fetch_c(t0, cnx);
                T.fetch_hist(t0, hist);
                // the entries of the chunk before are still in the mailbox
                MbEntry<R> p0, p1;
                R x0 = R(0), x1 = R(0), pv0, pv1;
                int y0, y1;
                T.load_entries(t0 - CK, p0, p1);
                T.load_direct(t0 - CK, false, x0, x1, y0, y1);
                T.halo_values(t0 - CK, p0, p1, x0, x1, pv0, pv1);
                T.park_t(tbuf, tnx);
                T.park_c(co, cnx);
                #pragma unroll
                for (int q = 0; q < 3; q++) rp[(q + 1)*CROW + T.me] = hist[q];
                rp[T.hq*CROW + T.hpos] = pv0;
                if (lane < 4) rp[lane*CROW] = pv1;
                wave_lds_fence();
                past.w = rp[2*CROW + T.me - 1];
                past.s = rp[2*CROW + T.me - 9];
                past.sw = rp[CROW + T.me - 10];
                past.v = hist[2];
            }
            #pragma unroll
            for (int i = 0; i < 4; i++) tw[i] = tnx[i];
            R v0, v1;
            T.halo_values(t0, e0, e1, d0, d1, v0, v1);
            rc[T.hq*CROW + T.hpos] = v0;
            if (lane < 4) rc[lane*CROW] = v1;
            if (more) { T.fetch_t(t0 + CK, tnx); T.fetch_c(t0 + CK, cnx); }
            wave_lds_fence();
            const unsigned chg = chunk_levels<R, CUBE, SKIP>(
                T, c, t0, rp, rc, ch, co, tbuf, past, [&]() {
                    if (more) {
                        T.load_entries(t0 + CK, e0, e1);
                        T.load_direct(t0 + CK, skip, d0, d1, b0, b1);
                    }
                });
            own |= chg;
            if (skip) nextDirty = nextDirty || (chg & 14u);
        } else if (more) {
            T.load_entries(t0 + CK, e0, e1);
            T.load_direct(t0 + CK, skip, d0, d1, b0, b1);
        }
        if (t0 >= T.tlo)
            T.post(t0, active, rc, SKIP ? (unsigned) __shfl((int) own,
                                                            T.post_lane(), 64)
                                        : 0u);
        // ---- store what changed; the next chunk's old times and cells
        if (active) {
            R out[4];
            T.collect(rc, out);
            if (more) {
                T.park_t(tbuf, tnx);
                T.park_c(ch, cnx);
            }
            T.template store<RECORD>(t0, tw, out, dmax, nchg);
            wave_lds_fence();
        }
        loaded = active;
        prevDirty = skip && __ballot(nextDirty) != 0;
    }
    T.template finish<RECORD>(dmax, nchg);
}

// -------------------------------------------------------- three waves
// The same tile by three waves: the first computes and touches LDS only, the
// second loads (mailbox, change record, old times, cells) and decides which
// chunks are computed, the third posts and stores.  A wave's loads and
// stores are counted together and complete in order, so a wave that polls
// the mailbox after posting waits for its own stores to reach memory; here
// the polling wave stores nothing.  For single grids, whose tiles leave
// room for it; in a batch, where every SIMD has its waves of other tiles,
// one wave per tile is faster.
//
// Buffers of three chunks in turn (chunk g in part g mod 3): ring rows, old
// times, new cell layers, own dirty and changed steps.  Counters, one per
// wave: g_load, g_comp, g_store = the chunks that wave is done with.  The
// loading wave announces chunks one by one or, where nothing is dirty, a run
// at once (s_news).
//
// Runs.  a.runs has a word per tile, each in a cache line of its own (the
// tiles' polls and posts of words in shared lines got in each other's way:
// 90.6 against 84.2 ms per 257^3 solve): (serial << 32) | first << 16 | end,
// the tile's current run of chunks that it skips with no dirty node of its
// own.
// A tile whose own chunks are clean (s_dirt, from the change record, read
// once) and whose upwind tiles' runs cover the same levels skips them all at
// once, so a clean stretch costs one exchange per tile instead of one per
// chunk.  When a run ends before the tile does, its entries are posted too,
// for readers that come when a later run has replaced the word.
constexpr int kRunStride = 16;          // words
constexpr int kMaxDirt = 1024;          // chunks of s_dirt: nz up to 4000
constexpr int kNews = 64;
enum : int { kSkipClean = 0, kSkipDirty = 1, kCompute = 2 };
// A thread's index that the compiler does not know to be the same in the two
// bodies of a kernel that chooses between them: what it could form from it
// once for both would hold registers through either (20 VGPRs spilled).
__device__ __forceinline__ int own_index(int i)
{
    asm volatile("" : "+v"(i));
    return i;
}

template <typename R>
struct Chunk3Lds {
    R ring[12*CROW], cbuf[12*CROW], tbuf[3*CK*CTROW];
    unsigned char own[3][64], chg[3][64];
    // announcement k in slot k mod kNews: what becomes of the next chunks,
    // kSkipClean (nothing dirty of its own), kSkipDirty (see own) or
    // kCompute, and, from bit 2 on, how many they are; the chunk it starts
    // at; any, per part: whether the chunk changed a node on its steps 1..3
    int news[kNews], start[kNews], any[3];
    unsigned char dirt[kMaxDirt];
    int load, comp, store, abort;
};
template <typename R, bool SKIP, bool RECORD, bool CUBE>
__device__ __forceinline__ void chunk3_body(const SweepArgs<R>& a,
                                            const int wg, Chunk3Lds<R>& lds)
{
    R* const ring = lds.ring;
    R* const cbuf = lds.cbuf;
    R* const tbuf = lds.tbuf;
    unsigned char (*const s_own)[64] = lds.own;
    unsigned char (*const s_chg)[64] = lds.chg;
    int* const s_news = lds.news;
    int* const s_start = lds.start;
    int* const s_any = lds.any;
    unsigned char* const s_dirt = lds.dirt;
    int &g_load = lds.load, &g_comp = lds.comp, &g_store = lds.store,
        &s_abort = lds.abort;
    const int thread = own_index(threadIdx.x);
    const int lane = thread & 63, role = thread >> 6;
    const ChunkTile<R> T(a, wg, lane, RECORD);
    if (T.empty() || (SKIP && sweep_is_clean(a))) return;     // uniform
    if (threadIdx.x == 0) g_load = g_comp = g_store = s_abort = 0;
    __syncthreads();
    const int ng = (T.thi - T.tlo)/CK + 1;
    auto give_up = [&]() {
        if (lane == 0) {
            atomicExch(a.err, 1);
            __hip_atomic_store(&s_abort, 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    // LDS accesses of a wave are in order, and a counter is written after
    // the data it announces; a waiting wave reads it before them.  Returns
    // the count, at least g, or -1 after a failure.
    auto wait = [&](int* p, int g) -> int {
        unsigned spins = 0;
        int v;
        while ((v = __builtin_amdgcn_readfirstlane(lds_load_rx(p))) < g) {
            if (lds_load_rx(&s_abort)) return -1;
            if (++spins > kSpinLimit) { give_up(); return -1; }
            __builtin_amdgcn_s_sleep(1);
        }
        wave_lds_fence();
        return v;
    };
    auto done = [&](int* p, int g) {
        wave_lds_fence();
        if (lane == 0)
            __hip_atomic_store(p, g, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
    };
    // announcement k, of the chunks from g on
    auto news = [&](int k, int g, int& f, int& n) {
        if (!SKIP) { f = kCompute; n = 1; return; }
        const int w = __builtin_amdgcn_readfirstlane(s_news[k & (kNews - 1)]);
        f = w & 3;
        n = w >> 2;
    };
    if (role == 0) {
        // -------------------------------------------------------- compute
        const Consts<R> c = chunk_consts<R, CUBE>(a);
        ChunkPast<R> past = {R(0), R(0), R(0), R(0)};
        bool loaded = false;
        int part = 0, before = 2, avail = 0;
        for (int g = 0, k = 0; g < ng; k++) {
            if (avail <= g && (avail = wait(&g_load, g + 1)) < 0) return;
            int f, n;
            news(k, g, f, n);
            if (f == kCompute) {
                const int t0 = T.tlo + g*CK;
                R* const rc = ring + part*4*CROW;
                const R* const rp = ring + before*4*CROW;
                if (!loaded) {
                    past.w = rp[2*CROW + T.me - 1];
                    past.s = rp[2*CROW + T.me - 9];
                    past.sw = rp[CROW + T.me - 10];
                    past.v = rp[3*CROW + T.me];
                }
                const unsigned chg = chunk_levels<R, CUBE, SKIP>(
                    T, c, t0, rp, rc, cbuf + before*4*CROW,
                    cbuf + part*4*CROW, tbuf + part*CK*CTROW, past, []() {});
                if (SKIP) {
                    s_chg[part][lane] = (unsigned char) chg;
                    const bool any = __ballot(chg & 14u) != 0;
                    if (lane == 0) s_any[part] = any ? 1 : 0;
                }
            }
            loaded = f == kCompute;
            g += n;
            done(&g_comp, g);
            part = g % 3;
            before = part == 0 ? 2 : part - 1;
        }
    } else if (role == 1) {
        // ----------------------------------------------------------- load
        MbEntry<R> e0, e1;
        R d0 = R(0), d1 = R(0);
        int b0 = 0, b1 = 0;
        unsigned stn = 0;
        // runs of the upwind tiles (lanes 0, 1, 2: in x, y and both; none:
        // a tile that always covers)
        unsigned long long run = 0;
        const int ux = T.fbx - (lane == 1 ? 0 : 1),
                  uy = T.fby - (lane == 0 ? 0 : 1);
        const bool up = SKIP && lane < 3 && ux >= 0 && uy >= 0;
        const int uoff = lane == 2 ? 4 : 2;      // its chunk of our chunk 0
        const unsigned long long* const upw = a.runs + kRunStride*(up ? ux*a.nby + uy
                                                         : 0);
        // tiles have runs: the chunks of a whole tile fit s_dirt
        const bool runs = SKIP && ((int) T.nbox + 2*CB - 2)/CK < kMaxDirt - 1;
        auto load_run = [&]() {
            if (runs && up)
                run = __hip_atomic_load(upw, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        };
        // end (in this tile's chunks) of the stretch from chunk g on that the
        // upwind tiles' runs cover; g if none
        // (clean: those that do)
        int clean = 0;
        auto covered = [&](int g) -> int {
            if (!runs) return g;
            const int b = (int) (run & 0xffffu) - uoff,
                      f = (int) ((run >> 16) & 0xffffu) - uoff;
            const bool mine = (unsigned) (run >> 32) == (unsigned) a.serial &&
                              f <= g && b > g;
            clean = (int) __ballot(up && mine);
            // the box's other upwind columns have no tile: s_dirt
            int end = up ? (mine ? b : g) : 1 << 20;
            end = min(end, __shfl_xor(end, 1, 64));
            end = min(end, __shfl_xor(end, 2, 64));
            return min(__builtin_amdgcn_readfirstlane(end), ng);
        };
        // loaded: the chunk's old times and cells are on the way (tnx, cnx)
        bool prevDirty = false, loaded = false;
        int part = 2, before = 1, k = 0;
        int first = -1;              // of the run that chunk g continues
        R tnx[4], cnx[CNC];
        if (SKIP) stn = T.load_stamp(T.tlo - CK);
        T.load_entries(T.tlo - CK, e0, e1);
        T.load_direct(T.tlo - CK, SKIP, d0, d1, b0, b1);
        load_run();
        if (runs) {
            for (int i = lane; i <= ng; i += 64) s_dirt[i] = 0;
            wave_lds_fence();
            T.scan(s_dirt, ng);
            wave_lds_fence();
        }
        auto announce = [&](int g, int f, int n) -> bool {
            if (SKIP) {
                // the slots of announcements long ago have been read
                if ((k & 15) == 0 && k >= 48) {
                    const int old = __builtin_amdgcn_readfirstlane(
                        s_start[(k - 32) & (kNews - 1)]);
                    if (wait(&g_comp, old) < 0 || wait(&g_store, old) < 0)
                        return false;
                }
                if (lane == 0) {
                    s_news[k & (kNews - 1)] = f | n << 2;
                    s_start[k & (kNews - 1)] = g;
                }
            }
            k++;
            done(&g_load, g + n);
            return true;
        };
        // the run's word: chunks from .. end - 1 continue or begin it
        auto publish = [&](int from, int end) {
            if (first < 0) first = from;
            if (lane == 0)
                __hip_atomic_store(a.runs + kRunStride*wg, (a.serial << 32) |
                                   (unsigned long long) first << 16 |
                                   (unsigned long long) end,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        for (int g = -1; g < ng; ) {
            const int t0 = T.tlo + g*CK;
            // ---- what does not need the neighbours: the own dirty nodes
            // among those the chunk reads (steps t0 - 3 .. t0 + 2), and its
            // old times and cells
            unsigned own = 0;
            bool active = g >= 0;
            if (SKIP) {
                own = T.own_dirty(t0, stn);
                active = g >= 0 && (prevDirty || __ballot(own & 7u) != 0);
            }
            auto load_all = [&]() -> bool {
                // of this chunk, and the three steps before it
                R* const rp = ring + before*4*CROW;
                R hist[3], pv0, pv1, x0 = R(0), x1 = R(0), cfirst[CNC];
                int y0, y1;
                MbEntry<R> p0, p1;
                T.fetch_c(t0 - CK, cfirst);
                T.fetch_hist(t0, hist);
                T.fetch_t(t0, tnx);
                T.fetch_c(t0, cnx);
                T.load_entries(t0 - CK, p0, p1);
                T.load_direct(t0 - CK, false, x0, x1, y0, y1);
                T.halo_values(t0 - CK, p0, p1, x0, x1, pv0, pv1);
                // no chunk before this one still needs its part
                if (g > 0 && (wait(&g_store, g) < 0 || wait(&g_comp, g) < 0))
                    return false;
                T.park_c(cbuf + before*4*CROW, cfirst);
                #pragma unroll
                for (int q = 0; q < 3; q++)
                    rp[(q + 1)*CROW + T.me] = hist[q];
                rp[T.hq*CROW + T.hpos] = pv0;
                if (lane < 4) rp[lane*CROW] = pv1;
                T.park_t(tbuf + part*CK*CTROW, tnx);
                T.park_c(cbuf + part*4*CROW, cnx);
                return true;
            };
            bool parked = false;
            if (g >= 0 && loaded) {
                // this part's last chunk is stored, and the chunk before the
                // last no longer reads its cell rows
                if (wait(&g_store, g - 2) < 0 || wait(&g_comp, g - 1) < 0)
                    return;
                T.park_t(tbuf + part*CK*CTROW, tnx);
                T.park_c(cbuf + part*4*CROW, cnx);
                parked = true;
            } else if (active) {
                if (!load_all()) return;
                parked = true;
            }

            // ---- the upwind neighbours' chunk
            int end = covered(g);
            {
                unsigned spins = 0;
                if (end <= g && !T.ready(t0, e0, e1, clean)) do {
                    if (lds_load_rx(&s_abort)) return;
                    if (++spins > kSpinLimit) { give_up(); return; }
                    load_run();
                    T.load_entries(t0, e0, e1);
                    end = covered(g);
                } while (end <= g && !T.ready(t0, e0, e1, clean));
            }
            // ---- a run: the covered chunks up to the first with a dirty
            // node of its own
            if (runs && !active && !loaded && end > g) {
                int n = 0;
                for (;; n += 64) {
                    const int at = g + n + lane;
                    const unsigned long long m = __ballot(
                        at >= end || s_dirt[min(at, ng - 1) + 1]);
                    if (m == 0) continue;
                    n += __ffsll((long long) m) - 1;
                    break;
                }
                if (n > 0) {
                    const int from = max(g, 0);
                    g += n;
                    if (g > from) {
                        publish(from, g);
                        if (!announce(from, kSkipClean, g - from)) return;
                    }
                    part = g % 3;
                    before = part == 0 ? 2 : part - 1;
                    if (g < ng) {
                        stn = T.load_stamp(T.tlo + g*CK);
                        load_run();
                        T.load_entries(T.tlo + g*CK, e0, e1);
                        T.load_direct(T.tlo + g*CK, true, d0, d1, b0, b1);
                    }
                    continue;
                }
            }
            // late: the halo's dirty nodes are looked at after the chunk has
            // been announced
            bool hd = true, cd = true, nextDirty = false, late = false;
            if (SKIP) {
                if (!active) T.halo_dirty(t0, e0, e1, b0, b1, hd, cd);
                const bool known = active;
                if (!active && g >= 0) {
                    active = __ballot((hd && T.hq < 3) ||
                                      (cd && lane < 3)) != 0;
                    if (!active && loaded) {
                        // dirty only if the chunk before changed a node
                        if (wait(&g_comp, g) < 0) return;
                        active = __builtin_amdgcn_readfirstlane(s_any[before])
                                 != 0;
                    }
                }
                if (active && !parked && !load_all()) return;
                late = known;
            }
            if (active) {
                R* const rc = ring + part*4*CROW;
                R v0, v1;
                T.halo_values(t0, e0, e1, d0, d1, v0, v1);
                rc[T.hq*CROW + T.hpos] = v0;
                if (lane < 4) rc[lane*CROW] = v1;
            }
            if (g >= 0) {
                int f = kCompute;
                if (SKIP) {
                    const bool od = __ballot(own != 0) != 0;
                    if (!active) f = od || !runs ? kSkipDirty : kSkipClean;
                    if (f == kSkipDirty && wait(&g_store, g - 2) < 0) return;
                    if (f != kSkipClean)
                        s_own[part][lane] = (unsigned char) own;
                }
                if (f == kSkipClean) publish(g, g + 1);
                else first = -1;
                if (!announce(g, f, 1)) return;
            }
            if (SKIP) {
                if (late) T.halo_dirty(t0, e0, e1, b0, b1, hd, cd);
                nextDirty = (own & 14u) || (hd && T.hq > 0) ||
                            (cd && lane > 0);
            }
            if (g + 1 < ng) {
                if (SKIP) stn = T.load_stamp(t0 + CK);
                load_run();
                T.load_entries(t0 + CK, e0, e1);
                T.load_direct(t0 + CK, SKIP, d0, d1, b0, b1);
                if (active) {
                    T.fetch_t(t0 + CK, tnx);
                    T.fetch_c(t0 + CK, cnx);
                }
            }
            loaded = active;
            prevDirty = SKIP && __ballot(nextDirty) != 0;
            g++;
            before = part;
            part = part == 2 ? 0 : part + 1;
        }
    } else {
        // ---------------------------------------------------------- store
        R dmax = R(0);
        int nchg = 0;
        int part = 0, avail = 0;
        int first = -1;           // of the clean chunks not yet posted
        for (int g = 0, k = 0; g < ng; k++) {
            if (avail <= g && (avail = wait(&g_load, g + 1)) < 0) return;
            int f, n;
            news(k, g, f, n);
            const int t0 = T.tlo + g*CK;
            if (f == kSkipClean) {
                if (first < 0) first = g;
                g += n;
                done(&g_store, g);
                part = g % 3;
                continue;
            }
            if (SKIP && first >= 0) {
                for (int i = first; i < g; i++)
                    T.post(T.tlo + i*CK, false, nullptr, 0u);
                first = -1;
            }
            const bool act = f == kCompute;
            if (act && wait(&g_comp, g + 1) < 0) return;
            const R* const rc = ring + part*4*CROW;
            unsigned own = 0;
            if (SKIP) {
                own = s_own[part][T.post_lane()];
                if (act) own |= s_chg[part][T.post_lane()];
            }
            T.post(t0, act, rc, own);
            R out[4], old[4];
            if (act) {
                const R* const tb = tbuf + part*CK*CTROW;
                #pragma unroll
                for (int i = 0; i < 4; i++)
                    old[i] = tb[T.lq*CTROW + 16*i + T.lc];
                T.collect(rc, out);
            }
            done(&g_store, ++g);
            if (act) T.template store<RECORD>(t0, old, out, dmax, nchg);
            part = part == 2 ? 0 : part + 1;
        }
        T.template finish<RECORD>(dmax, nchg);
    }
}

} // namespace fteik
