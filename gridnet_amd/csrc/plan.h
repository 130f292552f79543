// Host-side launch planning shared by the tuned kernels' launchers: how many CUs the current
// device has, how the batch is dealt to workgroups, and a zero-fill that is a kernel (a
// hipMemsetAsync node in a captured graph has given wrong results on replay on this platform).
// Every translation unit that includes this gets its own copy (internal linkage).
#ifndef GRIDNET_PLAN_H
#define GRIDNET_PLAN_H

#include "common.h"

namespace gridnet {
namespace {

int plan_device_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            cus = n;
        else
            cus = 256;
    }
    return cus;
}

// The batch is dealt to workgroups in chunks, a chunk is walked `nslot` elements at a time.
// `resident` = workgroups the chip holds at once: when the blocks alone do not fill it the batch
// is split so that the grid is one full round of workgroups; `whole`: never split.
void plan_batch_chunks(int B, int nblk, int nslot, int resident, bool whole, int &nchunk, int &chunk_len) {
    nchunk = whole ? 1 : resident / nblk;
    const int max_chunks = (B + nslot - 1) / nslot;
    if (nchunk > max_chunks) nchunk = max_chunks;
    if (nchunk < 1) nchunk = 1;
    chunk_len = (B + nchunk - 1) / nchunk;
    chunk_len = (chunk_len + nslot - 1) / nslot * nslot;
    nchunk = (B + chunk_len - 1) / chunk_len;
}

// Where the chip holds fewer than two workgroups per block the rule above takes one or two chunks and
// can leave the last round of workgroups nearly empty.  Shorter chunks make that round cheaper, and
// cost a fetch of the weights each, which is worth about `fetch` turns of the walk.  Takes another number of
// chunks where rounds x (turns + fetch) says at least a tenth less, so never on grids that fill
// their rounds already.  For kernels that keep no copy of anything per chunk.  (Forward, four inner
// iterations: 80 x 80 x 72, batch 32, 129.7 us in one chunk, 116.6 in three; 96^3, batch 16, 129.1
// and 120.6.  With the rule and without over 64 random grids of 40 to 128 cells a side, batch 4 to 90, one to
// eight inner iterations, both block sizes: most the same to 2 %; forward 7 to 19 % less on four, 3 and 5 %
// more on two; backward (cross_rows) 2 to 8 % less on eight, 1.4 % more on one.)
void plan_even_rounds(int B, int ngroup, int nslot, int resident, int min_walk, int &nchunk, int &chunk_len) {
    constexpr long fetch = 3;
    if ((long)nchunk * ngroup * 10 > 9L * resident && nchunk * ngroup <= resident) return;
    auto cost = [&](int n, int len) { return ((long)n * ngroup + resident - 1) / resident * (len / nslot + fetch); };
    const long now = cost(nchunk, chunk_len);
    long best = now - now / 10;
    for (int n = 1; n <= 8 && n <= B / min_walk; ++n) {
        int len = (B + n - 1) / n;
        len = (len + nslot - 1) / nslot * nslot;
        const int m = (B + len - 1) / len;
        const long c = cost(m, len);
        if (c < best) best = c, nchunk = m, chunk_len = len;
    }
}

// As plan_batch_chunks, for the row-wise kernels: at most `resident` workgroups, none that walks fewer than
// `min_walk` elements for its one fetch of the weights.  Three keep the fetch below the walk and still
// spread a small batch over the chip (forward / second kernel of the backward; 32^3, one inner
// iteration, batch 64: 8.8 us at 3, 9.8 at 2 and 11.2 at 8; 40 x 48 x 56, batch 13: 18.6, 17.9
// and 31.9); at large batches `resident` decides.
constexpr int kRowsMinWalk = 3;
int plan_row_chunks(int B, int ntube, int resident, int min_walk, int &chunk_len) {
    int nchunk = resident / ntube;
    if (nchunk > B / min_walk) nchunk = B / min_walk;
    if (nchunk < 1) nchunk = 1;
    chunk_len = (B + nchunk - 1) / nchunk;
    return (B + chunk_len - 1) / chunk_len;
}

// Threads to a sample where the workgroups of a step merge the pairs of the step before, beside the fetch of
// their weights; 0: a kernel of its own does (4.7 us and a launch).  Every workgroup of a chunk merges the
// same pairs, so it pays as long as they are few per thread.  Forward / backward of a step with the kernel and
// without: 32^3, batch 16, 11.1 -> 9.0 / 17.4 -> 16.1 us; batch 64, 15.5 -> 13.4 / 30.7 -> 29.9; batch 256 (22 and 32
// pairs per thread) 31.0 -> 28.7 / 68.2 -> 67.3; 64^3, batch 32 (44 pairs) 30.7 -> 32.1 / 74.0 -> 74.6.  Gated, 32^3,
// batch 32, 18.1 -> 16.1 / 26.2 -> 25.8; batch 256, 56.0 -> 54.7 forward.
constexpr int kMergeMostSamples = 64, kMergeMostPairs = 32;  // per workgroup; per thread
int plan_merge_lanes(int threads, int chunk_len, int pairs) {
    if (pairs % 2 || chunk_len > kMergeMostSamples) return 0;
    int lanes = 1;
    while (2 * lanes * chunk_len <= threads && 4 * lanes <= pairs && lanes < kWave) lanes *= 2;
    return (long)chunk_len * pairs <= kMergeMostPairs * (long)threads ? lanes : 0;
}

__global__ void plan_fill_zero_f32(float *p, long n) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0.f;
}

int plan_fill_zero(float *p, long n, hipStream_t st) {
    if (n <= 0) return GRIDNET_OK;
    long blocks = (n + 1023) / 1024;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(plan_fill_zero_f32, dim3((unsigned)blocks), dim3(256), 0, st, p, n);
    return check_launch("fill_zero");
}

// ---- parameter gradients of a batch that is split over workgroups -----------------------------
// On grids with fewer blocks than the chip has CUs the batch of a block is dealt to several
// workgroups.  Each of them leaves its share of the gradient arrays in a copy of its own (a
// "slab": the arrays one behind the other, `planes` x cells floats) with plain stores, and one
// small kernel adds the copies in chunk order into the caller's arrays: no atomics, the same bits
// on every run.

// The slabs are 256-byte aligned and read as 16-byte vectors.  The caller's arrays are accessed as
// 16-byte vectors too although the C ABI asks them to be aligned to their element size only:
// gfx950 serves global accesses at any 4-byte alignment (a misaligned vector costs a second
// request, nothing else); tests/test_gpu_alignment.py runs this with arrays 4 bytes off.
constexpr int kTailAhead = 4;
// workgroup `block` of the job's; `red` is LDS, one pair of doubles per wave of the caller's workgroup
template <int THREADS>
__device__ __forceinline__ void run_tail_job(const TailJob &job, int block, int nthreads, double (*red)[2]) {
    if (block >= job.reduce_blocks) {
        finalize_sums_of_sample<THREADS>(job.sums.part, job.sums.parts, job.sums.n, job.sums.sums,
                                         block - job.reduce_blocks, red, nthreads);
        return;
    }
    long i = (long)block * nthreads + threadIdx.x;
    const long step = (long)job.reduce_blocks * nthreads;
    for (; i < job.total4; i += step) {
        const long at = 4 * i;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int q0 = 0; q0 < job.ncopies; q0 += kTailAhead) {
            // several copies requested before any is added: the kernel this runs beside leaves it few
            // waves (past the last copy the requests repeat it)
            float4 v[kTailAhead];
#pragma unroll
            for (int k = 0; k < kTailAhead; ++k)
                v[k] = *reinterpret_cast<const float4 *>(job.slabs + min(q0 + k, job.ncopies - 1) * job.stride + at);
#pragma unroll
            for (int k = 0; k < kTailAhead; ++k) {
                const bool have = q0 + k < job.ncopies;
                sum.x += have ? v[k].x : 0.f; sum.y += have ? v[k].y : 0.f;
                sum.z += have ? v[k].z : 0.f; sum.w += have ? v[k].w : 0.f;
            }
        }
        int k = 0;
        long begin = 0;
        while (k + 1 < job.t.count && at >= job.t.end[k]) begin = job.t.end[k++];
        float4 *to = reinterpret_cast<float4 *>(job.t.dst[k] + (at - begin));
        if (job.accumulate >> k & 1) {
            const float4 old = *to;
            sum.x += old.x; sum.y += old.y; sum.z += old.z; sum.w += old.w;
        }
        *to = sum;
    }
}

// how many chunks the slabs region can take (0: none)
int plan_slab_capacity(const void *slabs, size_t slab_bytes, long slab_floats) {
    if (!slabs || slab_floats <= 0) return 0;
    const size_t n = slab_bytes / ((size_t)slab_floats * sizeof(float));
    return n > 65535 ? 65535 : (int)n;
}

// A split costs a pass over a copy of the gradient arrays per chunk, but no launch: the copies are added
// up beside the second kernel of the backward (TailJob).  So the batch is split as far as it goes: 32^3,
// batch 2, ten inner iterations with normalize, forward + backward 70 us with both elements in one
// workgroup, 51 us with one in each.

// Which targets of a split backward are added to rather than written (dweight, dbias, dscale, then
// dgamma and dbeta), by the caller's flags.
int plan_accumulate_mask(int flags) {
    if (flags & GRIDNET_OVERWRITE_PARAMS) return 0;
    return (flags & GRIDNET_OVERWRITE_STEP_PARAMS) ? 8 | 16 : ~0;
}

// The same for a backward that is not split (a split one stores into its copies).
int plan_param_mode(bool split, int flags) {
    if (split || (flags & GRIDNET_OVERWRITE_PARAMS)) return kParamStore;
    return (flags & GRIDNET_OVERWRITE_STEP_PARAMS) ? kParamAddNorms : kParamAddExclusive;
}

// `nthreads`: threads per workgroup of the kernel that will run the job.  Its workgroups take as
// many vectors per thread as keeps them below the number the chip holds.
TailJob plan_tail_job(const float *slabs, int ncopies, long stride, const SlabTargets &t, int accumulate,
                      int nthreads) {
    TailJob job{};
    job.slabs = slabs;
    job.ncopies = ncopies;
    job.accumulate = accumulate;
    job.stride = stride;
    job.total4 = t.end[t.count - 1] / 4;
    job.t = t;
    const long blocks = (job.total4 + nthreads - 1) / nthreads;
    job.reduce_blocks = (int)(blocks > 4096 ? 4096 : blocks);
    return job;
}

__global__ __launch_bounds__(256) void plan_run_tail_job(TailJob job) {
    __shared__ double red[256 / kWave][2];
    run_tail_job<256>(job, blockIdx.x, 256, red);
}

// as a kernel of its own, where there is no second kernel to take it along
int plan_launch_tail_job(const TailJob &job, hipStream_t st) {
    if (job.blocks() == 0) return GRIDNET_OK;
    hipLaunchKernelGGL(plan_run_tail_job, dim3((unsigned)job.blocks()), dim3(256), 0, st, job);
    return check_launch("reduce_slabs");
}

}  // namespace
}  // namespace gridnet

#endif  // GRIDNET_PLAN_H
