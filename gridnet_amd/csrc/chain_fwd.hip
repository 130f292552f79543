// The forward of a whole chain in one launch, for problems too small to fill the chip.
//
// The loop around the step, h = LayerNorm(step(h)) `outer` times with one parameter set
// (gridnet/scripts/train_mnist.py:62-64), launch by launch costs two dependent kernels and their
// launches per step, and every step fetches its 29 parameter planes again: one 32^3 sample through 64
// steps took 826 us, 7 us of kernels and 5 us of gaps a step, for 0.4 us of arithmetic.  Here a
// workgroup takes one 8^3 block of one batch element for all steps, a thread per cell with its 27
// weights in registers (few wavefronts are the problem, so the cells are spread as thin as they go),
// and the workgroups exchange what a step needs from the one before through memory:
//   * the raw value of every cell, in a ring of four activation tensors: a reader takes the 488 cells
//     around its block from there, one per thread;
//   * (mean, M2) of either half of the block, a 64-bit word each: every workgroup merges those of all
//     blocks of its element into the statistics for itself, in the same order.
// Both kinds of word are their own flags.  They start out as a bit pattern that arithmetic does not
// produce (kEmpty, a NaN with all bits set) and a reader polls until it is gone: one trip to memory
// between writer and reader instead of store, acknowledge, flag, poll, load.  A ring slot is emptied
// by its owner two steps after it was written: by then the owner has seen every block's statistics
// of the step after, which a workgroup leaves only when it has read its neighbours' cells.  The
// emptied slot is written again, and polled, two steps later; the owner's waits at the next step's
// polls lie in between, so no reader can find the old value.
//
// Residency is guaranteed by a cooperative launch.  Every wait is bounded all the same: when a thread
// has polled `spin_limit` times in all it raises the status word and waits no more, and the kernel
// ends on whatever it read.  chain_fwd_repair, always launched behind it, returns at once unless the
// status word is raised; then it does the chain again, one workgroup per element and no waits
// between workgroups, operation by operation as chain_fwd does it: the same bits, whichever of the two they are from.  The caller
// need not look at the status and nothing synchronises.
//
// All of it is latency: one 32^3 sample, one inner iteration, 2.5 us a step, of which the arithmetic is
// 0.4 (3.6 with the taps behind the statistics, see chain_fwd); 64 steps with the MNIST model around them
// 824 -> 213 us.

#include "common.h"
#include "fast_tiles.h"
#include "launch.h"
#include "plan.h"

namespace gridnet {

namespace {

constexpr int kSide = 10, kWindow = kSide * kSide * kSide, kShellCells = 488;
constexpr int kCfThreads = 512;
constexpr int kRing = 4, kAhead = 2;
constexpr unsigned kEmpty = 0xffffffffu;

struct ChainFwdArgs {
    const float *weight, *bias, *scale, *gamma, *beta, *x0;
    float *y_all;   // [outer,B,cells] raw outputs, or null
    float *stats;   // [outer,B,2], or null
    float *saved;   // [outer,B,cells] pre-activations of the last inner iteration, or null
    float *out;     // [B,cells]: LayerNorm of the last raw output
    unsigned *status;
    unsigned long long *parts;  // [kRing][B][nblk][kGroups]: (mean, M2)
    float *ring;                // [kRing][B][cells]
    int B, M, N, K, inner, outer, nblk, spin_limit;
    double eps;
};

template <typename T> __device__ __forceinline__ T ld_agent(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void st_agent(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Where thread `tid` sits in block `blk`: its cell, and the entry of the shell around the block that
// it fetches (the first 488 threads): two full planes along i, then along j, then along k.
struct CellPlace {
    int cell, at;            // grid index of the cell, its window position
    int edge, edge_at;       // grid index of the shell entry (-1: none, or outside the grid), its position (-1: none)
    __device__ __forceinline__ CellPlace(int tid, int blk, int M, int N, int K) {
        const int kb = K / 8, nb = N / 8;
        const int p0 = blk / (kb * nb) * 8, q0 = blk / kb % nb * 8, r0 = blk % kb * 8;
        const int i = tid / 64, j = tid / 8 % 8, k = tid % 8;
        cell = ((p0 + i) * N + q0 + j) * K + r0 + k;
        at = ((i + 1) * kSide + j + 1) * kSide + k + 1;
        int wi, wj, wk;
        if (tid < 200) {
            wi = tid / 100 * 9, wj = tid % 100 / 10, wk = tid % 10;
        } else if (tid < 360) {
            const int t = tid - 200;
            wi = 1 + t / 20, wj = t % 20 / 10 * 9, wk = t % 10;
        } else {
            const int t = tid - 360;
            wi = 1 + t / 16 % 8, wj = 1 + t % 16 / 2, wk = t % 2 * 9;
        }
        const int gi = p0 + wi - 1, gj = q0 + wj - 1, gk = r0 + wk - 1;
        edge_at = tid < kShellCells ? (wi * kSide + wj) * kSide + wk : -1;
        edge = tid < kShellCells && gi >= 0 && gi < M && gj >= 0 && gj < N && gk >= 0 && gk < K
                   ? (gi * N + gj) * K + gk : -1;
    }
};

// Cells in the second half of a block's rows take the three taps along k from high to low, as in the
// kernels for 8^3 blocks (those for one inner iteration do not): their weights are kept mirrored.  Those kernels take
// the taps beyond the rows' ends first of all; a chain's last bits differ by that.
__device__ __forceinline__ int k_direction(int tid, int inner) { return inner > 1 && (tid & 4) ? -1 : 1; }
__device__ __forceinline__ void load_weights(const float *weight, int cells, int cell, int dir, float (&w)[27]) {
#pragma unroll
    for (int r = 0; r < 9; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) w[3 * r + c] = weight[(long)(3 * r + 1 + (c - 1) * dir) * cells + cell];
}

// sum + the 27 taps on a window
template <typename T>
__device__ __forceinline__ T taps(const float *win, int at, int dir, const float (&w)[27], T sum) {
    const float *row = win + at, *from[3] = {row - dir, row, row + dir};
#pragma unroll
    for (int t = 0; t < 27; ++t)
        sum = fma((T)w[t], (T)from[t % 3][(t / 9 - 1) * kSide * kSide + (t / 3 % 3 - 1) * kSide], sum);
    return sum;
}

// sum_t w_t gamma_t, and sum_t w_t beta_t + bias: see chain_fwd.  The windows are free again when it returns.
__device__ __forceinline__ void affine_sums(float (*win)[kWindow], const CellPlace &p, const float (&w)[27], float bias, float gam,
                                            float bet, float egam, float ebet, float &sum_gamma, float &bias_beta) {
    win[0][p.at] = gam;
    win[1][p.at] = bet;
    if (p.edge_at >= 0) {
        win[0][p.edge_at] = egam;
        win[1][p.edge_at] = ebet;
    }
    lds_barrier();
    sum_gamma = (float)taps(win[0], p.at, 1, w, 0.0);
    bias_beta = (float)taps(win[1], p.at, 1, w, (double)bias);
    lds_barrier();
}
// The mean of 32 of a block's values, the same in every lane.
__device__ __forceinline__ float centre_of(const float *values, int tid) {
    const float2 c = *reinterpret_cast<const float2 *>(values + 32 * (tid & 15) + (6 * tid & 30));
    return row16_sum(fmaf(1.f / 32, c.x, 1.f / 32 * c.y));
}
// The pre-activation from the taps on (y - centre) gamma; a variance beyond fp32 leaves nothing but beta.
__device__ __forceinline__ float with_statistics(float taps, float centre, float mean, float rstd, float sum_gamma, float bias_beta) {
    return rstd == 0.f ? bias_beta : fmaf(rstd, fmaf(centre - mean, sum_gamma, taps), bias_beta);
}

// All inner iterations of one block: x in, x out; the shell is in both window copies and x in the
// first.
template <int ACT>
__device__ __forceinline__ float advance(float (*win)[kWindow], int at, int dir, const float (&w)[27], float bias,
                                         float scale, float x, int inner, float &last_u) {
    for (int it = 0; it < inner; ++it) {
        const float u = taps(win[it & 1], at, dir, w, bias);
        x = fmaf(scale, Act<ACT, float>::f(u), x);
        last_u = u;
        if (it + 1 < inner) {
            win[(it + 1) & 1][at] = x;
            lds_barrier();
        }
    }
    return x;
}

// Statistics of the block's values as the kernels for 8^3 blocks leave them, bit for bit: two groups of
// 256 cells, by the first two waves, four cells of half a row per lane; (mean, M2) as one word.
constexpr int kGroups = 2, kGroupCells = 256;
__device__ __forceinline__ unsigned long long group_moments(const float *values, int tid) {
    const int half = tid % 2, i = tid / 2 % 8, j = tid / 16;
    float v[4], sum = 0.f, m2 = 0.f, mean;
    load_cells<4>(values + i * 64 + j * 8 + half * 4, v);
#pragma unroll
    for (int r = 0; r < 4; ++r) sum += half ? v[3 - r] : v[r];
    const float row_mean = row16_sum(sum) * (1.f / 64);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float d = (half ? v[3 - r] : v[r]) - row_mean;
        m2 = fmaf(d, d, m2);
    }
    const float row_m2 = row16_sum(m2);
    slot_wave_moments<64>(row_mean, row_m2, 64, mean, m2);
    return (unsigned long long)__float_as_uint(mean) | (unsigned long long)__float_as_uint(m2) << 32;
}

// Sums over the groups of an element: means, M2, squares of the means; then its statistics.
struct GroupSums {
    double m = 0.0, q = 0.0, mm = 0.0;
    __device__ __forceinline__ void add(unsigned long long word) {
        const double mean = __uint_as_float((unsigned)word);
        m += mean;
        q += (double)__uint_as_float((unsigned)(word >> 32));
        mm += mean * mean;
    }
    __device__ __forceinline__ void over_wave() {
        m = wave_sum_dpp(m);
        q = wave_sum_dpp(q);
        mm = wave_sum_dpp(mm);
    }
    __device__ __forceinline__ void finish(double inv_groups, double eps, float &mean, float &rstd) const {
        const double centre = m * inv_groups;
        const double var = fma(q * inv_groups, 1.0 / kGroupCells, fma(-centre, centre, mm * inv_groups));
        mean = (float)centre;
        rstd = (float)rsqrt_newton((var > 0.0 ? var : 0.0) + eps);
    }
};

// The wave that merges the statistics of step j - 1: every block's words, in the same order everywhere.
// `early`: its first words as they were before the taps, or null.
struct Words { unsigned long long of[kAhead]; };
__device__ __forceinline__ Words request_words(const ChainFwdArgs &a, const unsigned long long *from, int i0) {
    Words w;  // together: one trip to memory
#pragma unroll
    for (int k = 0; k < kAhead; ++k) w.of[k] = ld_agent(from + min(i0 + 64 * k, kGroups * a.nblk - 1));
    return w;
}
__device__ __forceinline__ void merge_words(const ChainFwdArgs &a, const unsigned long long *from, const Words *early, int j, int s,
                                            bool first, int &budget, float *norm) {
    const int lane = threadIdx.x & 63, nwords = kGroups * a.nblk;
    GroupSums sums;
    for (int i0 = lane; i0 < nwords; i0 += 64 * kAhead) {
        Words got = early && i0 == lane ? *early : request_words(a, from, i0);
        unsigned long long (&word)[kAhead] = got.of;
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            while (word[k] == ~0ull && budget > 0) {
                if (--budget == 0) st_agent(a.status, 1u);
                __builtin_amdgcn_s_sleep(1);
                word[k] = ld_agent(from + min(i0 + 64 * k, nwords - 1));
            }
            if (i0 + 64 * k < nwords) sums.add(word[k]);
        }
    }
    sums.over_wave();
    float mean, rstd;
    sums.finish(1.0 / nwords, a.eps, mean, rstd);
    if (lane == 0) {
        norm[0] = mean;
        norm[1] = rstd;
        if (first && a.stats) {
            a.stats[((long)(j - 1) * a.B + s) * 2] = mean;
            a.stats[((long)(j - 1) * a.B + s) * 2 + 1] = rstd;
        }
    }
}

// The statistics of a step are there half a microsecond after its cells (a reduction, another trip to memory, the merge), so
// the taps of the next step do not wait for them: with c any number near the block's values,
//   sum_t w_t LN(y_t) = rstd (S - (mean - c) G) + H,   S = sum_t w_t gamma_t (y_t - c), G = sum_t w_t gamma_t, H = sum_t w_t beta_t,
// S from the raw cells as they come in, G and H once per launch.  c is the mean of 32 of the block's values: S and
// (mean - c) G then are of the size of the normalised sum, and the result is as exact as that (errors against 64 bits over eleven
// kinds of chain, six seeds each: 1.00 times those of normalising first).  Per step of 64: 32^3, batch 1, 3.6 -> 2.5 us, batch 8,
// 5.8 -> 3.9; 64^3, batch 1, 7.5 -> 6.8.  With one inner iteration only: of more the statistics are a small part.  The backward by
// whole rows of 16, 32 or 64 cells reads the pre-activations that are kept here; the other ones form them again from the
// normalised input, with other last bits, so that a cell within rounding of a kink can have the derivative of the side that the forward
// did not take.  The value is continuous there, and against 64 bits nothing changes: with relu, 16 x 24 x 40, batch 4, eight steps,
// one chain of 200 had a cell on the wrong side, and one when the forward normalised first.  (A wave of its own for the statistics, nine to a workgroup: two workgroups no
// longer fit a CU, although the occupancy query says that they do.)
template <int ACT, bool ONE> __global__ __launch_bounds__(kCfThreads) __attribute__((amdgpu_waves_per_eu(4))) void chain_fwd(ChainFwdArgs a) {
    __shared__ float win[2][kWindow];
    __shared__ __attribute__((aligned(16))) float values[kCfThreads];
    __shared__ float norm[2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid / 64;
    const int dir = ONE ? 1 : k_direction(tid, a.inner);
    const int blk = blockIdx.x % a.nblk, s = blockIdx.x / a.nblk;
    const int cells = a.M * a.N * a.K;
    const long slot_cells = (long)a.B * cells, slot_parts = (long)kGroups * a.B * a.nblk;
    int budget = a.spin_limit < 0 ? -a.spin_limit : a.spin_limit;
    unsigned long long *parts = a.parts + (long)kGroups * s * a.nblk;
    const CellPlace p(tid, blk, a.M, a.N, a.K);
    const bool has = p.edge >= 0;
    float w[27];
    load_weights(a.weight, cells, p.cell, dir, w);
    const float bias = a.bias[p.cell], scale = a.scale[p.cell], gam = a.gamma[p.cell], bet = a.beta[p.cell];
    const float egam = has ? a.gamma[p.edge] : 0.f, ebet = has ? a.beta[p.edge] : 0.f;
    float own = a.x0[(long)s * cells + p.cell];  // this cell's raw value
    const float edge = has ? a.x0[(long)s * cells + p.edge] : 0.f;
    float *ring = a.ring + (long)s * cells;

    float sum_gamma = 0.f, bias_beta = 0.f;
    if (ONE) affine_sums(win, p, w, bias, gam, bet, egam, ebet, sum_gamma, bias_beta);
    for (int j = 0; j <= a.outer; ++j) {
        float x = own, e = edge, u, centre = 0.f;
        // what step j - 1 left: the shell's cells, and the statistics of the element
        const unsigned long long *words = parts + ((j - 1) & (kRing - 1)) * slot_parts;
        Words early;
        if (j > 0) {
            const float *from = ring + ((j - 1) & (kRing - 1)) * slot_cells;
            const bool want = j < a.outer && has;
            e = want ? ld_agent(from + p.edge) : 0.f;
            if (ONE) {
                centre = centre_of(values, tid);
                x = (own - centre) * gam;
            } else if (wave == 0) {
                merge_words(a, words, nullptr, j, s, blk == 0, budget, norm);
            }
            while (want && __float_as_uint(e) == kEmpty && budget > 0) {
                if (--budget == 0) st_agent(a.status, 1u);
                __builtin_amdgcn_s_sleep(1);
                e = ld_agent(from + p.edge);
            }
            if (ONE) e = has ? (e - centre) * egam : 0.f;
        }
        if (ONE) {
            win[0][p.at] = x;
            if (p.edge_at >= 0) win[0][p.edge_at] = e;
            lds_barrier();
            if (j > 0 && wave == 0) early = request_words(a, words, lane);
            u = taps(win[0], p.at, dir, w, j > 0 ? 0.f : bias);
            if (j > 0 && wave == 0) merge_words(a, words, &early, j, s, blk == 0, budget, norm);
        }
        if (j > 0) {
            wait_global_loads();  // and the stores before: the slot emptied a step ago is empty
            lds_barrier();        // the statistics
            const float mean = norm[0], rstd = norm[1];
            x = fmaf((own - mean) * rstd, gam, bet);
            if (j == a.outer) {
                a.out[(long)s * cells + p.cell] = x;
                break;
            }
            if (j >= 2) {  // every block has read step j - 2
                st_agent(ring + ((j - 2) & (kRing - 1)) * slot_cells + p.cell, __uint_as_float(kEmpty));
                if (tid < kGroups) st_agent(parts + ((j - 2) & (kRing - 1)) * slot_parts + kGroups * blk + tid, ~0ull);
            }
            if (ONE) u = with_statistics(u, centre, mean, rstd, sum_gamma, bias_beta);
            else e = has ? fmaf((e - mean) * rstd, egam, ebet) : 0.f;
        }
        if (ONE) {
            own = fmaf(scale, Act<ACT, float>::f(u), x);
        } else {
            win[0][p.at] = x;
            if (p.edge_at >= 0) win[0][p.edge_at] = win[1][p.edge_at] = e;
            lds_barrier();
            own = advance<ACT>(win, p.at, dir, w, bias, scale, x, a.inner, u);
        }
        st_agent(ring + (j & (kRing - 1)) * slot_cells + p.cell, own);
        values[tid] = own;
        lds_barrier();
        if (wave < kGroups) {
            const unsigned long long word = group_moments(values, tid);
            if (lane == 0 && a.spin_limit >= 0)
                st_agent(parts + (j & (kRing - 1)) * slot_parts + kGroups * blk + wave, word);
        }
        if (a.y_all) a.y_all[(long)j * slot_cells + (long)s * cells + p.cell] = own;
        if (a.saved) a.saved[(long)j * slot_cells + (long)s * cells + p.cell] = u;
    }
}

// The same chain by one workgroup per element, for the case that a wait of chain_fwd ran out.  The
// blocks of a step one after the other, raw values from one ring slot to the next; the statistics' words pass through
// memory to be merged in chain_fwd's order.
template <int ACT, bool ONE> __global__ __launch_bounds__(kCfThreads) void chain_fwd_repair(ChainFwdArgs a) {
    if (*a.status == 0) return;
    __shared__ float win[2][kWindow];
    __shared__ __attribute__((aligned(16))) float values[kCfThreads];
    __shared__ float norm[2];
    const int tid = threadIdx.x, s = blockIdx.x, dir = ONE ? 1 : k_direction(tid, a.inner);
    const int cells = a.M * a.N * a.K;
    const long slot_cells = (long)a.B * cells, mine = (long)s * cells;
    unsigned long long *words = a.parts + (long)kGroups * s * a.nblk;
    float mean = 0.f, rstd = 1.f;
    for (int j = 0; j < a.outer; ++j) {
        const float *from = j ? a.ring + ((j - 1) & 1) * slot_cells + mine : a.x0 + mine;
        float *to = a.ring + (j & 1) * slot_cells + mine;
        for (int blk = 0; blk < a.nblk; ++blk) {
            const CellPlace p(tid, blk, a.M, a.N, a.K);
            const bool has = p.edge >= 0;
            float w[27];
            load_weights(a.weight, cells, p.cell, dir, w);
            const float bias = a.bias[p.cell], scale = a.scale[p.cell], gam = a.gamma[p.cell], bet = a.beta[p.cell];
            const float egam = has ? a.gamma[p.edge] : 0.f, ebet = has ? a.beta[p.edge] : 0.f;
            const float own = from[p.cell], edge = has ? from[p.edge] : 0.f;
            float x = own, e = edge, u, y, centre = 0.f, sum_gamma = 0.f, bias_beta = 0.f;
            __syncthreads();  // the block before is done with the window and the values
            if (ONE && j) {
                values[tid] = own;
                affine_sums(win, p, w, bias, gam, bet, egam, ebet, sum_gamma, bias_beta);
                centre = centre_of(values, tid);
                x = (own - centre) * gam;
                e = has ? (edge - centre) * egam : 0.f;
            } else if (j) {
                x = fmaf((own - mean) * rstd, gam, bet);
                e = has ? fmaf((edge - mean) * rstd, egam, ebet) : 0.f;
            }
            win[0][p.at] = x;
            if (p.edge_at >= 0) win[0][p.edge_at] = win[1][p.edge_at] = e;
            __syncthreads();
            if (ONE) {
                u = taps(win[0], p.at, dir, w, j ? 0.f : bias);
                if (j) {
                    x = fmaf((own - mean) * rstd, gam, bet);
                    u = with_statistics(u, centre, mean, rstd, sum_gamma, bias_beta);
                }
                y = fmaf(scale, Act<ACT, float>::f(u), x);
            } else {
                y = advance<ACT>(win, p.at, dir, w, bias, scale, x, a.inner, u);
            }
            to[p.cell] = y;
            if (a.y_all) a.y_all[(long)j * slot_cells + mine + p.cell] = y;
            if (a.saved) a.saved[(long)j * slot_cells + mine + p.cell] = u;
            values[tid] = y;
            __syncthreads();
            if (tid / 64 < kGroups) {
                const unsigned long long word = group_moments(values, tid);
                if ((tid & 63) == 0) st_agent(words + kGroups * blk + tid / 64, word);
            }
        }
        __syncthreads();  // the step's values and words are there for every thread
        int budget = 0;   // no waits
        if (tid < 64) merge_words(a, words, nullptr, j + 1, s, true, budget, norm);
        __syncthreads();
        mean = norm[0];
        rstd = norm[1];
    }
    const float *last = a.ring + ((a.outer - 1) & 1) * slot_cells + mine;
    for (int c = tid; c < cells; c += kCfThreads)
        a.out[mine + c] = fmaf((last[c] - mean) * rstd, a.gamma[c], a.beta[c]);
}

// status word zero, everything behind it empty
__global__ __launch_bounds__(256) void chain_fwd_clear(uint4 *p, long n) {
    const long stride = (long)gridDim.x * 256;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        p[i] = i == 0 ? make_uint4(0, 0, 0, 0) : make_uint4(kEmpty, kEmpty, kEmpty, kEmpty);
}

constexpr size_t kStatusBytes = 256, kAlign = 16;  // the caller's workspace may start at any address
size_t parts_bytes(const ChainFwd &c) {
    const size_t nblk = (size_t)c.M * c.N * c.K / 512;
    return (kRing * (size_t)c.B * nblk * kGroups * 8 + 255) / 256 * 256;
}

template <int ACT> int launch_chain_fwd(const ChainFwd &c, hipStream_t st) {
    char *ws = (char *)(((uintptr_t)c.workspace + kAlign - 1) / kAlign * kAlign);
    ChainFwdArgs a{};
    a.weight = c.weight; a.bias = c.bias; a.scale = c.scale; a.gamma = c.gamma; a.beta = c.beta; a.x0 = c.x0;
    a.y_all = c.y_all; a.stats = c.stats; a.saved = c.saved; a.out = c.out;
    a.status = (unsigned *)ws;
    a.parts = (unsigned long long *)(ws + kStatusBytes);
    a.ring = (float *)(ws + kStatusBytes + parts_bytes(c));
    a.B = c.B; a.M = c.M; a.N = c.N; a.K = c.K; a.inner = c.inner; a.outer = c.outer;
    a.nblk = (int)((long)c.M * c.N * c.K / 512);
    a.spin_limit = c.spin_limit;
    a.eps = c.eps;
    const long vecs = (long)((chain_fwd_workspace(c) - kAlign) / 16);
    const long blocks = (vecs + 1023) / 1024;
    hipLaunchKernelGGL(chain_fwd_clear, dim3((unsigned)(blocks > 2048 ? 2048 : blocks)), dim3(256), 0, st, (uint4 *)ws, vecs);
    void *args[] = {&a};
    const auto chain = c.inner == 1 ? chain_fwd<ACT, true> : chain_fwd<ACT, false>;
    const auto repair = c.inner == 1 ? chain_fwd_repair<ACT, true> : chain_fwd_repair<ACT, false>;
    const hipError_t e = hipLaunchCooperativeKernel((const void *)chain, dim3((unsigned)(a.nblk * c.B)), dim3(kCfThreads), args, 0, st);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(GRIDNET_ERR_LAUNCH, "chain_fwd: cooperative launch failed: %s", hipGetErrorString(e));
    }
    hipLaunchKernelGGL(repair, dim3((unsigned)c.B), dim3(kCfThreads), 0, st, a);
    return check_launch("chain_fwd");
}

}  // namespace

bool chain_fwd_supports(int B, int M, int N, int K, int inner, int outer) {
    if (B <= 0 || M <= 0 || N <= 0 || K <= 0 || M % 8 || N % 8 || K % 8 || inner < 1 || outer < 2) return false;
    if ((long)M * N * K * 27 >= (1L << 31)) return false;
    static int per_cu = 0;
    if (per_cu == 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void *)chain_fwd<GRIDNET_ACT_TANH, true>, kCfThreads, 0) !=
                hipSuccess || n < 1)
            n = -1;
        per_cu = n;
    }
    if (per_cu < 1) return false;
    // As many as fit.  Launches included, a step of 64 against the kernel and the merge of a step launch by
    // launch (rows_fwd): 32^3, one inner iteration, batch 1, 2.5 against 6.7 us, batch 8 (two workgroups per
    // CU), 3.9 against 10.1; 64^3, batch 1, 6.8 against 10.2; four inner iterations (step_fwd_split), batch 8, 7.3 against 14.5.
    return (long)M * N * K / 512 * B <= (long)per_cu * plan_device_cus();
}

size_t chain_fwd_workspace(const ChainFwd &c) {
    return kAlign + kStatusBytes + parts_bytes(c) + kRing * (size_t)c.B * c.M * c.N * c.K * sizeof(float);
}

int chain_forward_all(const ChainFwd &c, hipStream_t st) {
    switch (c.activation) {
        case GRIDNET_ACT_RELU: return launch_chain_fwd<GRIDNET_ACT_RELU>(c, st);
        case GRIDNET_ACT_LEAKY_RELU: return launch_chain_fwd<GRIDNET_ACT_LEAKY_RELU>(c, st);
        case GRIDNET_ACT_SILU: return launch_chain_fwd<GRIDNET_ACT_SILU>(c, st);
        case GRIDNET_ACT_TANH: return launch_chain_fwd<GRIDNET_ACT_TANH>(c, st);
    }
    return fail(GRIDNET_ERR_ACTIVATION, "unknown activation function: id %d", c.activation);
}

}  // namespace gridnet
