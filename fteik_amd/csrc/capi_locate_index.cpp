// capi_locate_index.cpp -- the index of the locator's tables: when it is
// built and used, its memory, and the searches through it
// (locate_index.hip).  It is laid out once per set of tables and thrown
// away when a table changes.
#include "capi_internal.h"
#include "locate_index.h"

using namespace fteik_capi;

namespace {

struct Index {
    bool ready = false;
    bool off = false;                // these tables have no index
    int ngrd = 0;                    // cells of the index
    int through = 0;                 // searches through the index
    int searches = 0;                // full searches since a table changed
    int pause = 0;                   // searches of several events to come
                                     // that are made in full
    fteik::LocIndex g;
    size_t permCap = 0, repCap = 0, srepCap = 0;   // floats
    // work space: events (floats each holds), pairs of a batch
    long evCap = 0, evTf = 0, pairCap = 0;
    long rawCap = 0;
    fteik::LocEvents v;
    float *d_obs = nullptr, *d_wt = nullptr;
    unsigned char *d_skip = nullptr;
};
Index gi;

constexpr size_t kPairBytes = (size_t) 1 << 30;

void free_events()
{
    dfree(gi.v.o8); dfree(gi.v.w8); dfree(gi.v.h8); dfree(gi.v.row);
    dfree(gi.v.xn); dfree(gi.v.kap); dfree(gi.v.mar); dfree(gi.v.best);
    gi.v.t0 = nullptr;
    gi.v.over = nullptr;
    dfree(gi.d_obs); dfree(gi.d_wt); dfree(gi.d_skip);
    gi.evCap = gi.evTf = gi.rawCap = 0;
}

void free_pairs()
{
    dfree(gi.g.lbs); dfree(gi.g.pair); dfree(gi.g.lbc);
    gi.pairCap = 0;
}

template <typename T>
bool grow(T **p, size_t *cap, size_t n)
{
    if (n <= *cap) return true;
    dfree(*p);
    *cap = 0;
    if (!dalloc_spare(p, n)) return false;
    *cap = n;
    return true;
}

// Shape of the ngrd cells (z fastest): the solvers' grid when it has as
// many points, else from the tables.  Any shape gives the same results; a
// shape whose blocks are compact leaves out more.  In a table of a grid with
// nz points per column neighbouring columns have nearly the same times:
// among the divisors p of ngrd, the mean |T[c + p] - T[c]| has local minima
// at nz (against p - 1, p + 1) and at nz*nx (against steps of nz).
// false: GPU error, or no memory.
bool find_shape(int *nz, int *nx, int *ny, bool *memory)
{
    const int n = gl.ngrd;
    if (g_model.nz > 0 && (long) g_model.nz*g_model.nx*g_model.ny == n) {
        *nz = g_model.nz; *nx = g_model.nx; *ny = g_model.ny;
        return true;
    }
    *nz = n; *nx = 1; *ny = 1;
    auto strides = [&](const std::vector<int> &p, std::vector<float> &d) {
        int *d_p = nullptr;
        float *d_d = nullptr;
        d.assign(p.size(), 0.0f);
        *memory = dalloc_spare(&d_p, p.size()) &&
                  dalloc_spare(&d_d, p.size());
        bool ok = *memory &&
                  h2d(d_p, p.data(), p.size()*sizeof(int)) &&
                  fteik_k_locate_strides(gl.d_tab, gl.ldgrd, gl.ntf, n, d_p,
                                         (int) p.size(), d_d,
                                         g_dev.stream) == 0 &&
                  d2h(d.data(), d_d, p.size()*sizeof(float));
        dfree(d_p);
        dfree(d_d);
        return ok;
    };
    // candidates p with p - step, p + step; picks the smallest local
    // minimum within 2.5 times the least value
    auto best_of = [&](const std::vector<int> &c, int step, int *at,
                       float *val) -> bool {
        std::vector<int> p;
        std::vector<float> d;
        for (int v : c) { p.push_back(v - step); p.push_back(v);
                          p.push_back(v + step); }
        if (p.empty()) { *at = -1; return true; }
        if (!strides(p, d)) return false;
        float least = -1.0f;
        for (size_t i = 0; i < c.size(); i++)
            if (least < 0.0f || d[3*i + 1] < least) least = d[3*i + 1];
        *at = -1;
        for (size_t i = 0; i < c.size(); i++)
            if (d[3*i + 1] < d[3*i] && d[3*i + 1] < d[3*i + 2] &&
                d[3*i + 1] <= 2.5f*least) {
                *at = c[i];
                *val = d[3*i + 1];
                break;
            }
        return true;
    };
    std::vector<int> c;
    for (int p = 8; (long) p*8 <= n; p++) if (n % p == 0) c.push_back(p);
    int p1 = -1, p2 = -1;
    float d1 = 0.0f, d2 = 0.0f;
    if (!best_of(c, 1, &p1, &d1)) return false;
    if (p1 < 0) return true;
    *nz = p1;
    *nx = n/p1;
    std::vector<int> c2;
    for (int p : c) if (p % p1 == 0 && p/p1 >= 8) c2.push_back(p);
    if (!best_of(c2, p1, &p2, &d2)) return false;
    if (p2 > 0 && d2 <= 3.0f*d1) {
        *nx = p2/p1;
        *ny = n/p2;
    }
    return true;
}

// Lays the index out.  false: GPU error; gi.ready tells whether there is
// one.
bool build()
{
    fteik::LocIndex &g = gi.g;
    bool memory = true;
    gi.off = true;                   // until it is laid out
    if (!find_shape(&g.nz, &g.nx, &g.ny, &memory)) return !memory;
    g.ntf = gl.ntf;
    g.nt = fteik_k_locate_index_nt(g.ntf);
    g.lz = 2; g.lx = 2; g.ly = 2;
    if (g.ny == 1) { g.lz = 3; g.lx = 3; g.ly = 0; }
    if (g.nx == 1 && g.ny == 1) { g.lz = 6; g.lx = 0; }
    auto parts = [](int n, int l) { return (n + (1 << l) - 1) >> l; };
    g.nbz = parts(g.nz, g.lz); g.nbx = parts(g.nx, g.lx);
    g.nby = parts(g.ny, g.ly);
    g.nsz = parts(g.nbz, g.lz); g.nsx = parts(g.nbx, g.lx);
    g.nsy = parts(g.nby, g.ly);
    const long nb = (long) g.nbz*g.nbx*g.nby;
    g.nb = (int) nb;
    g.ns = g.nsz*g.nsx*g.nsy;
    // blocks mostly empty (a shape unlike the block's): not worth it
    if (nb*64 > 4L*gl.ngrd) return true;
    // a copy of the tables: within a quarter of the memory that is free
    const size_t np = (size_t) nb*64*g.ntf;
    size_t fr = 0, tot = 0;
    if (np > gi.permCap && (hipMemGetInfo(&fr, &tot) != hipSuccess ||
                            np*sizeof(float) > fr/4)) return true;
    const size_t nr = 2*(size_t) g.ntf*nb, nsr = 2*(size_t) g.ntf*g.ns;
    if (!grow(&g.perm, &gi.permCap, np) || !grow(&g.rep, &gi.repCap, nr) ||
        !grow(&g.srep, &gi.srepCap, nsr)) return true;
    g.h = g.rep + nr/2;
    g.sh = g.srep + nsr/2;
    if ((!g.tmax && !dalloc_spare(&g.tmax, 1)) ||
        (!g.npair && !dalloc_spare(&g.npair, fteik::kLocCounts))) return true;
    unsigned tm = 0;
    if (hipMemsetAsync(g.tmax, 0, sizeof(unsigned), g_dev.stream)
            != hipSuccess ||
        fteik_k_locate_index_build(&g, gl.d_tab, gl.ldgrd, g_dev.stream) ||
        !d2h(&tm, g.tmax, sizeof(tm))) return false;
    float t;
    memcpy(&t, &tm, sizeof(t));
    if (!(t <= kPlainLimit)) return true;
    gi.off = false;
    gi.ready = true;
    gi.ngrd = gl.ngrd;
    return true;
}

// Work space for n events and a batch of them; false: no memory.
bool work_space(int n)
{
    fteik::LocIndex &g = gi.g;
    const long ne = (n + fteik::kLocEv - 1)/fteik::kLocEv*fteik::kLocEv;
    const long tf = std::max(gl.lntf, g.nt);
    if (ne > gi.evCap || tf > gi.evTf) {
        const long c = std::max(ne, gi.evCap), f = std::max(tf, gi.evTf);
        free_events();
        // best, t0 and over adjoin: one copy brings them back
        if (!dalloc_spare(&gi.v.o8, (size_t) (c*f)) ||
            !dalloc_spare(&gi.v.w8, (size_t) (c*f)) ||
            !dalloc_spare(&gi.v.h8, (size_t) (c*f)) ||
            !dalloc_spare(&gi.v.row, (size_t) (3*c*f)) ||
            !dalloc_spare(&gi.v.xn, (size_t) c) || !dalloc_spare(&gi.v.kap, (size_t) c) ||
            !dalloc_spare(&gi.v.mar, (size_t) c) ||
            !dalloc_spare(&gi.v.best, (size_t) (2*c)) ||
            !dalloc_spare(&gi.d_obs, (size_t) (c*f)) ||
            !dalloc_spare(&gi.d_wt, (size_t) (c*f)) ||
            !dalloc_spare(&gi.d_skip, (size_t) (c*f))) {
            free_events();
            return false;
        }
        gi.evCap = c;
        gi.evTf = f;
    }
    gi.v.t0 = (float *) (gi.v.best + n);
    gi.v.over = (unsigned *) (gi.v.t0 + n);
    // pairs (group, event) of a batch of eb events
    const long per = (long) g.ns*(64 + 2 + 1)*(long) sizeof(float);
    long eb = std::max<long>(fteik::kLocEv, (long) kPairBytes/per
                                            /fteik::kLocEv*fteik::kLocEv);
    eb = std::min(eb, ne);
    const long need = (long) g.ns*eb;
    if (need > gi.pairCap) {
        free_pairs();
        if (!dalloc_spare(&g.lbs, (size_t) need) ||
            !dalloc_spare(&g.pair, 2*(size_t) need) ||
            !dalloc_spare(&g.lbc, 64*(size_t) need)) {
            free_pairs();
            return false;
        }
        gi.pairCap = need;
    }
    g.eb = (int) eb;
    return true;
}

// Events of the largest call that goes through the index.  Speed does not
// set this line: at 10,000 events on 48 tables the index takes 4.3 ms and the
// full search 162 ms.  The learned search (4.1 ms) is held by its test to ten
// times the rate of the full search over a catalogue of that size, and a
// call of that size keeps the search which that figure is measured against.
// Callers may split a catalogue.
constexpr int kIndexEvents = 8192;

// Table counts of the batched kernel of the full search.
bool batch_kernel(int ntf)
{
    return (ntf >= 1 && ntf <= 8) || ntf == 10 || ntf == 12 || ntf == 16 ||
           ntf == 20 || ntf == 24 || ntf == 32 || ntf == 40 || ntf == 48 ||
           ntf == 56 || ntf == 64;
}

// Estimated time of the full search for n events (seconds).  The batched
// kernel makes 51e12 operations a second, 9 per cell, table and event;
// without it an event is a pass over the tables at 1.8 TB/s (measured 242 us
// for 403 MB) and a launch.
double full_time(int n)
{
    const double cells = (double) gl.ngrd*gl.ntf;
    return (n > 1 && batch_kernel(gl.ntf))
        ? 20e-6 + (double) n*cells*1.8e-13
        : (double) n*(6e-6 + cells*4.0/1.8e12);
}

// Whether the estimated time of a search through the index is below that of
// the full one: about 90 us of launches and latencies, 0.3 us an event
// (measured 0.43 us with 10,000 events, 105 us for one), and once per set of
// tables its building, at first two passes over them (measured 340 us for
// 403 MB).  Picks that fit badly leave more blocks; see block_limit.
bool worth_it(int n)
{
    const double cells = (double) gl.ngrd*gl.ntf;
    double index = 90e-6 + n*0.3e-6;
    if (!gi.ready && gi.searches == 0) index += 150e-6 + cells*8.0/1.5e12;
    return index < full_time(n);
}

// Blocks whose evaluation takes as long as the full search of n events, or
// ~0 where there are not as many: a batch of events with more blocks left
// after the bounds is given up and searched in full.  A block's times pass
// at 4.2 to 14 TB/s, the more the more events share it.  The full search
// has, beyond full_time, allocations and copies of 0.3 ms a call and, with
// more events than its few-event kernel takes, 0.5 ns a cell, and 0.3 ps a
// cell and event whatever the number of tables.  4,096 events on 48 tables
// of 81 x 161 x 161 (35,301 blocks, limit 13,800 an event): picks with an
// outlier leave 630 blocks, picks without any relation to smooth tables
// 3,950 (46 ms, in full 67); with 0.25 s of noise in every table value they
// leave 17,100 (131 ms through the index).
unsigned block_limit(int n)
{
    const double block = (double) gl.ntf*256.0/9e12;
    const double more = 0.3e-3 + gl.ngrd*(n > 8 ? 0.5e-9 : 0.0)
                      + (double) n*gl.ngrd*0.3e-12;
    const double limit = (full_time(n) + more)/block;
    return limit < (double) n*gi.g.nb ? (unsigned) limit : ~0u;
}

} // namespace

namespace fteik_capi {

bool locator_tables_changed()
{
    gi.ready = gi.off = false;
    gi.searches = gi.pause = 0;
    return settle_origin_times();
}

bool locator_reclaim()
{
    const bool any = gi.permCap || gi.evCap || gi.pairCap;
    if (!any) return false;
    const int through = gi.through;
    index_release();
    gi.through = through;
    return true;
}

void index_release()
{
    free_events();
    free_pairs();
    dfree(gi.g.perm); dfree(gi.g.rep); dfree(gi.g.srep); dfree(gi.g.tmax);
    dfree(gi.g.npair);
    gi = Index();
}

int index_search(int n, const int *evnmbr, int *optIndx, double *t0Opt,
                 double *objOpt, std::vector<int> *redo)
{
    if (n > kIndexEvents || gi.off || gl.ngrd < 4096 || fteik_k_locate_index_nt(gl.ntf) == 0)
        return 1;
    // sizes set after initialize are not those of the tables
    if (gi.ready && (gi.g.ntf != gl.ntf || gi.ngrd != gl.ngrd))
        if (!locator_tables_changed()) return 2;
    for (int e = 0; e < n; e++)
        if ((size_t) evnmbr[e] > gl.plain.size() ||
            !gl.plain[(size_t) (evnmbr[e] - 1)]) return 1;
    if (!worth_it(n)) { gi.searches++; return 1; }
    if (n > 1 && gi.pause > 0) { gi.pause--; return 1; }
    if (!gi.ready) {
        if (!build()) return 2;
        if (!gi.ready) return 1;
    }
    if (!work_space(n)) return 1;
    // the events' picks: straight from the catalogue when they are one run
    // of it
    const size_t lt = (size_t) gl.lntf, m = (size_t) n*lt;
    const float *o = nullptr, *w = nullptr;
    const unsigned char *sk = nullptr;
    std::vector<float> ov, wv;
    std::vector<unsigned char> sv;
    bool run = true;
    for (int e = 1; e < n && run; e++) run = evnmbr[e] == evnmbr[0] + e;
    if (run) {
        const size_t k = (size_t) (evnmbr[0] - 1)*lt;
        o = &gl.obs[k]; w = &gl.wt[k]; sk = &gl.skip[k];
    } else {
        ov.resize(m); wv.resize(m); sv.resize(m);
        for (int e = 0; e < n; e++) {
            const size_t k = (size_t) (evnmbr[e] - 1)*lt;
            memcpy(&ov[(size_t) e*lt], &gl.obs[k], lt*sizeof(float));
            memcpy(&wv[(size_t) e*lt], &gl.wt[k], lt*sizeof(float));
            memcpy(&sv[(size_t) e*lt], &gl.skip[k], lt);
        }
        o = ov.data(); w = wv.data(); sk = sv.data();
    }
    hipStream_t s = g_dev.stream;
    // (of a batch: its share, whatever the batches before it left)
    const unsigned limit = block_limit(n);
    const int eb = gi.g.eb, nbatch = (n + eb - 1)/eb;
    bool ok = hipMemcpyAsync(gi.d_obs, o, m*sizeof(float),
                             hipMemcpyHostToDevice, s) == hipSuccess &&
              hipMemcpyAsync(gi.d_wt, w, m*sizeof(float),
                             hipMemcpyHostToDevice, s) == hipSuccess &&
              hipMemcpyAsync(gi.d_skip, sk, m, hipMemcpyHostToDevice, s)
                  == hipSuccess &&
              fteik_k_locate_index_events(&gi.g, &gi.v, n, gl.lntf, gi.d_obs,
                                          gi.d_wt, gi.d_skip, s) == 0;
    for (int q = 0; q < nbatch && ok; q++) {
        const int m = std::min(eb, n - q*eb);
        ok = fteik_k_locate_index_search(
                 &gi.g, &gi.v, q*eb, m,
                 limit == ~0u ? limit
                              : (unsigned) ((double) limit*m/n),
                 gi.v.over + q, std::max(1, g_dev.ncu), s) == 0;
    }
    ok = ok && fteik_k_locate_index_origin(&gi.g, &gi.v, n, gl.d_tab,
                                           gl.ldgrd, gl.lntf, gi.d_skip,
                                           s) == 0;
    // keys, then origin times, then the batches given up
    std::vector<unsigned long long> r(2*(size_t) n);
    ok = ok && d2h(r.data(), gi.v.best, (size_t) n*(sizeof(r[0]) +
                   sizeof(float)) + (size_t) nbatch*sizeof(unsigned));
    if (!ok) return 2;
    gi.through++;
    const float *t0 = (const float *) (r.data() + n);
    const unsigned *over = (const unsigned *) (t0 + n);
    for (int e = 0; e < n; e++) {
        if (limit != ~0u && over[e/eb]) { redo->push_back(e); continue; }
        const unsigned bits = (unsigned) (r[(size_t) e] >> 32);
        float obj;
        memcpy(&obj, &bits, sizeof(obj));
        optIndx[e] = (int) (r[(size_t) e] & 0xffffffffull) + 1;
        objOpt[e] = (double) obj;
        t0Opt[e] = (double) t0[e] + gl.tepoch[(size_t) (evnmbr[e] - 1)];
    }
    // tables or picks that the index is no help with: the bounds cost up to
    // a tenth of the full search, so look again only now and then
    if (n > 1 && 2*redo->size() > (size_t) n) gi.pause = 15;
    return 0;
}

} // namespace fteik_capi

// Searches made through the index since the locator was initialized.
extern "C" int fteik_k_locate_index_searches(void) { return gi.through; }
