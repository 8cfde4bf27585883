// sweep_chunk.hip -- kernels of the chunked tile (sweep_chunk.h), for one
// grid and for a batch.  No launch is cooperative: a tile waits only on
// tiles of lower-numbered workgroups and workgroups are dispatched in order,
// so the lowest unfinished tile is always resident and every wait ends; each
// wait also has a spin limit that turns a hang into a reported error.
#include <hip/hip_runtime.h>
#include "sweep_chunk.h"

namespace fteik {

template <typename R, bool SKIP, bool RECORD, bool CUBE>
__global__ __launch_bounds__(192)
__attribute__((amdgpu_waves_per_eu(3)))
void sweep3d_chunk_kernel(SweepArgs<R> a)
{
    __shared__ Chunk3Lds<R> lds;
    const int wg = tile_of_rank((int) blockIdx.x, a.nbx, a.nby);
    if (wg < 0) return;
    if (RECORD) clear_count(a, wg);
    if (SKIP && !sweep_is_busy(a, single_share(a)))
        chunk3_body<R, true, true, CUBE>(a, wg, lds);
    else
        chunk3_body<R, false, RECORD, CUBE>(a, wg, lds);
}

// Workgroup w sweeps map entry (grid, tile); args[g]: grid g's sweep
// arguments for this launch, read through the constant address space as in
// batch_mb_kernel.
template <typename R, bool SKIP, bool RECORD, bool CUBE>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(3)))
void batch_chunk_kernel(const SweepArgs<R>* __restrict__ args,
                        const int* __restrict__ map)
{
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) SweepArgs<R> CArgs;
    const SweepArgs<R> a = ((CArgs*) args)[map[2*blockIdx.x]];
#else   // the host pass only parses the kernel
    const SweepArgs<R> a = args[map[2*blockIdx.x]];
#endif
    const int wg = map[2*blockIdx.x + 1];
    if (RECORD) clear_count(a, wg);
    chunk_body<R, SKIP, RECORD, CUBE>(a, wg);
}

// kind 0: every chunk; 1: every chunk, changes recorded; 2: skipping where few
// chunks are dirty, else as 1
template <typename R, bool CUBE>
static const void* chunk_fn(int kind, bool batch)
{
#define CF(f) (kind == 0 ? (const void*) f<R, false, false, CUBE> \
               : kind == 1 ? (const void*) f<R, false, true, CUBE> \
                           : (const void*) f<R, true, true, CUBE>)
    if (batch) return CF(batch_chunk_kernel);
    return CF(sweep3d_chunk_kernel);
#undef CF
}

} // namespace fteik

using namespace fteik;

extern "C" const void* fteik_k_chunk_fn(int fp32, unsigned count, int batch,
                                        int cube)
{
    const int kind = count == 0 ? 0 : count <= 8 ? 1 : 2;
    const bool b = batch != 0;
    if (fp32) return cube ? chunk_fn<float, true>(kind, b)
                          : chunk_fn<float, false>(kind, b);
    return cube ? chunk_fn<double, true>(kind, b)
                : chunk_fn<double, false>(kind, b);
}

extern "C" int fteik_k_chunk_fits(int nz, int nx, int ny, size_t mbBytes)
{
    return chunk_fits(nz, nx, ny, mbBytes) ? 1 : 0;
}

extern "C" size_t fteik_k_run_words(int nx, int ny)
{
    return (size_t) kRunStride*((nx - 1 + CB - 1)/CB)*((ny - 1 + CB - 1)/CB);
}

extern "C" size_t fteik_k_stamp_bytes(long ngrd)
{
    return (size_t) ngrd + 2*kStampPad;
}

extern "C" long fteik_k_stamp_offset(void) { return kStampPad; }
extern "C" int fteik_k_record_words(void) { return kRecordWords; }
