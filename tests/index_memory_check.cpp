// Host check of the locator index's memory (fteik_amd/csrc/
// capi_locate_index.cpp) against stubs of the runtime and the kernels: every
// allocation of a search fails in turn.  Prints, per failing allocation, what
// the search returned (1: search in full), then what is still allocated
// after the index was given back, and whether giving it back said so.
#include <cstdio>
#include <cstdlib>
#include "../fteik_amd/csrc/capi_locate_index.cpp"

static int g_calls, g_fail, g_held;

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    if (++g_calls == g_fail) return hipErrorOutOfMemory;
    *p = malloc(n);
    g_held++;
    return hipSuccess;
}
hipError_t hipFree(void *p) { free(p); g_held--; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    *f = *t = (size_t) 1 << 40;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind,
                          hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
int fteik_k_locate_index_nt(int ntf) { return (ntf + 7)/8*8; }
int fteik_k_locate_strides(const float *, long, int, int, const int *, int,
                           float *, hipStream_t) { return 0; }
int fteik_k_locate_index_build(const fteik::LocIndex *, const float *, long,
                               hipStream_t) { return 0; }
int fteik_k_locate_index_events(const fteik::LocIndex *,
                                const fteik::LocEvents *, int, int,
                                const float *, const float *,
                                const unsigned char *, hipStream_t)
{ return 0; }
int fteik_k_locate_index_search(const fteik::LocIndex *,
                                const fteik::LocEvents *, int, int, unsigned,
                                unsigned *, int, hipStream_t) { return 0; }
int fteik_k_locate_index_origin(const fteik::LocIndex *,
                                const fteik::LocEvents *, int, const float *,
                                long, int, const unsigned char *, hipStream_t)
{ return 0; }
}

namespace fteik_capi {
Device g_dev;
ModelGeom g_model;
Locator gl;
bool settle_origin_times() { return true; }
bool h2d(void *d, const void *h, size_t n) { memcpy(d, h, n); return true; }
bool d2h(void *h, const void *d, size_t n) { memcpy(h, d, n); return true; }
}

int main()
{
    const int n = 200;
    gl.init = true;
    gl.ntf = 9;
    gl.lntf = 16;
    gl.ngrd = 40*40*40;
    gl.ldgrd = gl.ngrd;
    gl.tepoch.assign(n, 0.0);
    gl.obs.assign((size_t) n*gl.lntf, 0.0f);
    gl.wt.assign((size_t) n*gl.lntf, 1.0f);
    gl.skip.assign((size_t) n*gl.lntf, 0);
    gl.plain.assign(n, 1);
    std::vector<int> ev(n), opt(n), redo;
    std::vector<double> t0(n), obj(n);
    for (int e = 0; e < n; e++) ev[(size_t) e] = e + 1;
    auto search = [&](int fail) -> int {
        locator_tables_changed();
        g_calls = 0;
        g_fail = fail;
        redo.clear();
        return index_search(n, ev.data(), opt.data(), t0.data(), obj.data(),
                            &redo);
    };
    printf("%d", search(0));
    const int all = g_calls;
    printf(" %d", all);
    for (int f = 1; f <= all; f++) {
        index_release();
        printf(" %d", search(f));
    }
    printf(" %d", search(0));
    const bool gave = locator_reclaim();
    printf(" %d %d %d\n", gave ? 1 : 0, g_held, locator_reclaim() ? 1 : 0);
    return 0;
}
