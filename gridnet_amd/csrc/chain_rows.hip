// A chain of steps with ONE inner iteration each, h = LayerNorm(step(h)) `outer` times, by whole K-rows:
// one kernel per step and direction, for the plain update and for the gated one.
//
// With one inner iteration a step is a 27-tap stencil over the whole grid (see fwd_rows.hip) and a few
// operations per byte: what a step costs is the tensors it moves, and beside that the launches and
// small kernels between the steps.  What this file does about them:
//   * The forward of a chain that is to be differentiated keeps what the backward would recompute from
//     27 taps (plain: the pre-activation u; gated: d/d(pre), d/d(gate pre-activation) and the gate, each
//     per unit of gradient).  With it the deltas of a cell are a few operations on values of that cell
//     alone, so a workgroup forms them for its tube of 4 x 4 rows AND the rows around it, and the
//     backward of a step is one kernel: no delta tensor between two kernels, no partial dx written and
//     read back, one stencil instead of two (5 passes over activations against 8).
//   * The weight gradients come from the same stencil over delta: x[c] delta[c + off_t] is the gradient
//     of the neighbour's weight 26 - t, and no other cell contributes to it.
//   * Where the batch is split over workgroups every chunk keeps ONE copy of the gradient arrays for the
//     whole chain, each step adding its sums to what the step before left; the copies are added up once.
//   * The pairs per wave behind the LayerNorms' per-sample numbers are merged by the workgroups of the next
//     step while their weights are on their way (plan_merge_lanes says where; a small kernel between the steps
//     elsewhere, 4.7 us each).  Merged inside the walk, by one wave an element ahead, they cost the kernels
//     11 us forward and 24 us backward: everybody waits for that wave at the barrier.
// 32^3, batch 256, silu, per step: forward 27.5 us, backward 67.7, at 4.2 to 4.3 TB/s where a copy
// reaches 4.6 (with the kernel that merges 29.1 + 68.4, and with the chunks of a tube on several CUs, 30.4 and 69.0; fwd_rows, bwd_rows and cross_rows with theirs: 28.1 + 4.4,
// 59.3 + 8.0 + 23.4).  The bytes are not what binds: a fifth of the backward's taken away brought 0.7 % of the training step, two sevenths
// of the gated one's nothing; the vector ALU is 46 to 50 % busy at two waves per SIMD, and 17 and 8 us of a step do not grow with the
// batch.  Gated, tanh: 55.7 and 85.8 + 4.9 (op by op the whole training step took 21.3 ms, 9.1 now).

#include <algorithm>

#include "common.h"
#include "fast_tiles.h"
#include "launch.h"
#include "plan.h"

namespace gridnet {

namespace {

constexpr int kTube = 4, kSide = kTube + 2, kWinRows = kSide * kSide;

// Sigmoid and activation of the gated update, as gated_fast.hip.  (Shorter ones, on the hardware's exp2
// and reciprocal with one Newton step each, took 5 us off the forward; over a chain of 64 steps their
// errors, a fifth larger, left the chain's input gradient 1e-5 off where these leave 1e-6.)
template <int ACT> __device__ __forceinline__ void gate_parts(float pre, float gp, float &a, float &d, float &gate) {
    gate = sigmoid_stable(gp);
    Act<ACT, float>::fd(pre, a, d);
}

// What both kernels know about a thread's place: its row of the tube, its CPT cells of it.
template <int CPT, int K> struct RowPlace {
    static constexpr int kl = K / CPT;
    int r, ci, cj, bk, p0, q0, grow;
    bool first, last;
    __device__ __forceinline__ RowPlace(int tid, int tube, int N) {
        r = tid / kl;
        bk = tid % kl;
        ci = r / kTube;
        cj = r % kTube;
        const int nbj = N / kTube;
        p0 = tube / nbj * kTube;
        q0 = tube % nbj * kTube;
        grow = ((p0 + ci) * N + q0 + cj) * K + CPT * bk;
        first = bk == 0;
        last = bk == kl - 1;
    }
};

// CPT floats at a byte offset of this lane behind a pointer that is the same for the whole wave: an
// addressing mode; an element index per lane is widened, scaled and added in vector registers.  Both
// are opaque: the compiler otherwise widens the offset ahead of the loop, or adds to it what the tensors'
// pointers share, and is back at vector additions, one per load.
#define GRIDNET_GLOBAL __attribute__((address_space(1)))
template <int CPT> struct CellVector { typedef float type __attribute__((ext_vector_type(CPT), aligned(4))); };
template <> struct CellVector<1> { typedef float type; };
template <int CPT> __device__ __forceinline__ void load_at(const float *base, unsigned bytes, float (&v)[CPT]) {
    typedef typename CellVector<CPT>::type V;
    const GRIDNET_GLOBAL char *from = (const GRIDNET_GLOBAL char *)base;
    asm volatile("" : "+s"(from), "+v"(bytes));
    const V got = *(const GRIDNET_GLOBAL V *)(from + bytes);
    if constexpr (CPT == 1) v[0] = got;
    else
#pragma unroll
        for (int c = 0; c < CPT; ++c) v[c] = got[c];
}
template <int CPT> __device__ __forceinline__ void store_at(float *base, unsigned bytes, const float (&v)[CPT]) {
    typedef typename CellVector<CPT>::type V;
    GRIDNET_GLOBAL char *to = (GRIDNET_GLOBAL char *)base;
    asm volatile("" : "+s"(to), "+v"(bytes));
    V put;
    if constexpr (CPT == 1) put = v[0];
    else
#pragma unroll
        for (int c = 0; c < CPT; ++c) put[c] = v[c];
    *(GRIDNET_GLOBAL V *)(to + bytes) = put;
}
#undef GRIDNET_GLOBAL
// a pair of per-sample numbers, as load_ahead
__device__ __forceinline__ float2 load_pair_ahead(const float *pairs, int sample) {
    unsigned zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    float v[2];
    load_at<2>(pairs + 2L * sample, zero, v);
    return make_float2(v[0], v[1]);
}

struct RowsFwdArgs {
    const float *weight, *bias, *scale, *gamma, *beta, *x;
    const float *x_stats;   // the LayerNorm in front of the step (null: x is used as it is)
    const float *x_part;    // MERGE: the pairs that its statistics come from instead, merged by `lanes` threads each,
    float *stats_out;       // and left here for the backward (or null)
    int lanes;
    double eps;
    float *y, *y_part;
    float *saved;           // plain: [B,cells]; gated: [3][B,cells]; or null
    int B, M, N, ntube, nchunk, chunk_len;
    CuShare together;
};

// MERGE: the statistics of x from the pairs of the step before.  A kernel without it has none of that code: with
// a test instead, the gated forward took 57 -> 59 us where the pairs are merged elsewhere.
// PLAIN: four cells and 108 weights per thread; GATED: two cells and 2 x 54.  Everything else as
// fwd_rows.hip: six by six rows in LDS, two stages, one barrier per batch element.
template <int ACT, int SETS, bool SAVE, int K, bool MERGE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(SETS == 1 ? 3 : 2, 3)))
void rows_fwd(RowsFwdArgs a) {
    constexpr int CPT = 4 / SETS, RPT = 3;
    extern __shared__ __attribute__((aligned(16))) float lds[];  // [2][36][K], gamma rows, beta rows, statistics
    int tube, chunk;
    if (!split_block_id(blockIdx.x, a.ntube, a.nchunk, a.together, false, tube, chunk)) return;  // grid padding
    const int tid = threadIdx.x, M = a.M, N = a.N, nw = blockDim.x / 64, wave = tid / 64;
    const RowPlace<CPT, K> p(tid, tube, N);
    const long cells = (long)M * N * K;
    const bool ln_in = MERGE || a.x_stats != nullptr;
    const int s0 = chunk * a.chunk_len, s1 = min(a.B, s0 + a.chunk_len);
    float2 *stat = reinterpret_cast<float2 *>(lds + 4 * kWinRows * K);  // of the samples s0 ... s1, with MERGE

    float w[SETS][9][3][CPT], bv[SETS][CPT], rv[CPT];
#pragma unroll
    for (int pq = 0; pq < 9; ++pq)
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int k = 0; k < SETS; ++k) {
                load_cells<CPT>(a.weight + ((pq * 3 + cc) * SETS + k) * cells + p.grow, w[k][pq][cc]);
            }
#pragma unroll
    for (int k = 0; k < SETS; ++k) load_cells<CPT>(a.bias + k * cells + p.grow, bv[k]);
    if (SETS == 1) load_cells<CPT>(a.scale + p.grow, rv);
    if constexpr (MERGE) {  // while the parameters are on their way
        const double n = (double)a.ntube * nw, count = cells / n;
        merge_pairs<4>(a.x_part, a.ntube * nw, a.lanes, s0, s1 - s0, [&](int e, double m, double q, double mm) {
            const float2 v = merged_statistics(m, q, mm, n, count, a.eps);
            stat[e] = v;
            if (tube == 0 && a.stats_out) reinterpret_cast<float2 *>(a.stats_out)[s0 + e] = v;
        });
    }
    const float keep_first = p.first ? 0.f : 1.f, keep_last = p.last ? 0.f : 1.f;
#pragma unroll
    for (int k = 0; k < SETS; ++k)
#pragma unroll
        for (int pq = 0; pq < 9; ++pq) {
            w[k][pq][0][0] *= keep_first;
            w[k][pq][2][CPT - 1] *= keep_last;
        }

    int goff[RPT], loff[RPT];
    bool ok[RPT];
    float *gam_rows = lds + 2 * kWinRows * K, *bet_rows = gam_rows + kWinRows * K;
#pragma unroll
    for (int e = 0; e < RPT; ++e) {
        const int row = p.r + 16 * e, wi = row / kSide, wj = row % kSide;
        const int gi = p.p0 + wi - 1, gj = p.q0 + wj - 1;
        ok[e] = row < kWinRows && gi >= 0 && gi < M && gj >= 0 && gj < N;
        goff[e] = ok[e] ? (gi * N + gj) * K + CPT * p.bk : p.grow;  // anything valid when not used
        loff[e] = row * K + CPT * p.bk;
        if (ln_in && row < kWinRows) {  // zeros outside the grid: no test per element then
            float gq[CPT], bq[CPT];
            load_cells<CPT>(a.gamma + goff[e], gq);
            load_cells<CPT>(a.beta + goff[e], bq);
#pragma unroll
            for (int q = 0; q < CPT; ++q) {
                gq[q] = ok[e] ? gq[q] : 0.f;
                bq[q] = ok[e] ? bq[q] : 0.f;
            }
            store_cells<CPT>(gam_rows + loff[e], gq);
            store_cells<CPT>(bet_rows + loff[e], bq);
        }
    }
    const bool has_last = p.r + 16 * (RPT - 1) < kWinRows;
    const int own_row = (p.ci + 1) * kSide + p.cj + 1;
    wait_global_loads();
    if (MERGE) lds_barrier();  // the statistics are there

    float xbuf[RPT][CPT];
    float2 next_stat = make_float2(0.f, 1.f);
    auto fetch = [&](int s) {
        const float *x = a.x + (long)s * cells;
        if (MERGE) next_stat = stat[s - s0];
        else if (ln_in) next_stat = load_pair_ahead(a.x_stats, s);
#pragma unroll
        for (int e = 0; e < RPT; ++e) load_at<CPT>(x, 4u * (unsigned)goff[e], xbuf[e]);
    };
    if (s0 < s1) fetch(s0);
    for (int s = s0; s < s1; ++s) {
        float *stage = lds + ((s - s0) & 1) * kWinRows * K;
        const float xmean = next_stat.x, xrstd = next_stat.y;
#pragma unroll
        for (int e = 0; e < RPT; ++e) {
            if (e == RPT - 1 && !has_last) break;
            float v[CPT];
            if (ln_in) {
                float gq[CPT], bq[CPT];
                load_cells<CPT>(gam_rows + loff[e], gq);
                load_cells<CPT>(bet_rows + loff[e], bq);
#pragma unroll
                for (int q = 0; q < CPT; ++q) v[q] = fmaf((xbuf[e][q] - xmean) * xrstd, gq[q], bq[q]);
            } else {
#pragma unroll
                for (int q = 0; q < CPT; ++q) v[q] = ok[e] ? xbuf[e][q] : 0.f;
            }
            store_cells<CPT>(stage + loff[e], v);
        }
        lds_barrier();  // the stage is complete; the other one's readers are done
        fetch(min(s + 1, s1 - 1));
        __builtin_amdgcn_sched_barrier(0);  // the requests leave now, with the whole stencil in front of their use
        float u[SETS][CPT], own[CPT];
#pragma unroll
        for (int k = 0; k < SETS; ++k)
#pragma unroll
            for (int c = 0; c < CPT; ++c) u[k][c] = bv[k][c];
#pragma unroll
        for (int pq = 0; pq < 9; ++pq) {
            const int di = pq / 3 - 1, dj = pq % 3 - 1;
            float d[CPT + 2], mid[CPT];
            load_cells<CPT>(stage + (own_row + di * kSide + dj) * K + CPT * p.bk, mid);
            d[0] = lane_before(mid[CPT - 1]);
            d[CPT + 1] = lane_after(mid[0]);
#pragma unroll
            for (int c = 0; c < CPT; ++c) d[c + 1] = mid[c];
            if (pq == 4) {
#pragma unroll
                for (int c = 0; c < CPT; ++c) own[c] = mid[c];
            }
#pragma unroll
            for (int k = 0; k < SETS; ++k)
#pragma unroll
                for (int cc = 0; cc < 3; ++cc)
#pragma unroll
                    for (int c = 0; c < CPT; ++c) u[k][c] = fmaf(w[k][pq][cc][c], d[c + cc], u[k][c]);
        }
        const long at = (long)s * cells;
        const unsigned o = 4u * (unsigned)p.grow;
        float out[CPT];
        if (SETS == 1) {
#pragma unroll
            for (int c = 0; c < CPT; ++c) out[c] = fmaf(rv[c], Act<ACT, float>::f(u[0][c]), own[c]);
            if (SAVE) store_at<CPT>(a.saved + at, o, u[0]);
        } else {
            float f0[CPT], f1[CPT], gate[CPT];
#pragma unroll
            for (int c = 0; c < CPT; ++c) {
                float act, d;
                gate_parts<ACT>(u[0][c], u[SETS - 1][c], act, d, gate[c]);
                out[c] = fmaf(gate[c], own[c] - act, act);
                f0[c] = (1.f - gate[c]) * d;
                f1[c] = (own[c] - act) * gate[c] * (1.f - gate[c]);
            }
            if (SAVE) {
                store_at<CPT>(a.saved + at, o, f0);
                store_at<CPT>(a.saved + (long)a.B * cells + at, o, f1);
                store_at<CPT>(a.saved + 2L * a.B * cells + at, o, gate);
            }
        }
        store_at<CPT>(a.y + at, o, out);
        // one (mean, M2) pair per wave
        float sum = out[0];
#pragma unroll
        for (int c = 1; c < CPT; ++c) sum += out[c];
        if (CPT == 4) sum = (out[0] + out[1]) + (out[CPT - 2] + out[CPT - 1]);  // in fwd_rows' order
        const float mean = row16_sum(sum) * (1.f / (16 * CPT));
        float m2 = 0.f;
#pragma unroll
        for (int c = 0; c < CPT; ++c) m2 = fmaf(out[c] - mean, out[c] - mean, m2);
        m2 = row16_sum(m2);
        float wave_mean, wave_m2;
        slot_wave_moments<64>(mean, m2, 16 * CPT, wave_mean, wave_m2);
        if ((tid & 63) == 0) {
            float *to = a.y_part + (((long)s * a.ntube + tube) * nw + wave) * 2;
            to[0] = wave_mean;
            to[1] = wave_m2;
        }
    }
}

// One row of delta against the mirrored weights and against x: out[c] += v[t][c] d and n[t][c] += x[c] d for
// the d of the cell before (t = 0), at (1) and behind (2).  The neighbouring lanes' values are DPP
// operands of the multiply-adds; the compiler makes moves of them, a quarter of this kernel's
// instructions with one cell per thread.  A DPP operand must not be a vector ALU result of the two
// instructions before: the products that take none stand in front.
#define GRIDNET_BEFORE " wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
#define GRIDNET_BEHIND " wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
__device__ __forceinline__ void row_products(const float (&d)[1], const float (&v)[3][1], const float (&x)[1],
                                             float (&out)[1], float (&n)[3][1]) {
    asm("v_fmac_f32 %0, %4, %6\n\t"
        "v_fmac_f32 %2, %4, %8\n\t"
        "v_fmac_f32_dpp %0, %4, %5" GRIDNET_BEFORE
        "v_fmac_f32_dpp %1, %4, %8" GRIDNET_BEFORE
        "v_fmac_f32_dpp %0, %4, %7" GRIDNET_BEHIND
        "v_fmac_f32_dpp %3, %4, %8" GRIDNET_BEHIND
        : "+v"(out[0]), "+v"(n[0][0]), "+v"(n[1][0]), "+v"(n[2][0])
        : "v"(d[0]), "v"(v[0][0]), "v"(v[1][0]), "v"(v[2][0]), "v"(x[0]));
}
__device__ __forceinline__ void row_products(const float (&d)[2], const float (&v)[3][2], const float (&x)[2],
                                             float (&out)[2], float (&n)[3][2]) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        out[c] = fmaf(v[1][c], d[c], out[c]);
        n[1][c] = fmaf(x[c], d[c], n[1][c]);
    }
    n[0][1] = fmaf(x[1], d[0], n[0][1]);
    n[2][0] = fmaf(x[0], d[1], n[2][0]);
    asm("v_fmac_f32 %0, %5, %8\n\t"
        "v_fmac_f32 %1, %4, %7\n\t"
        "v_fmac_f32_dpp %0, %5, %6" GRIDNET_BEFORE
        "v_fmac_f32_dpp %2, %5, %10" GRIDNET_BEFORE
        "v_fmac_f32_dpp %1, %4, %9" GRIDNET_BEHIND
        "v_fmac_f32_dpp %3, %4, %11" GRIDNET_BEHIND
        : "+v"(out[0]), "+v"(out[1]), "+v"(n[0][0]), "+v"(n[2][1])
        : "v"(d[0]), "v"(d[1]), "v"(v[0][0]), "v"(v[0][1]), "v"(v[2][0]), "v"(v[2][1]), "v"(x[0]), "v"(x[1]));
}
#undef GRIDNET_BEFORE
#undef GRIDNET_BEHIND

struct RowsBwdArgs {
    const float *weight, *scale, *gamma, *beta;
    const float *dy;                // gradient with respect to LayerNorm(y)
    const float *y, *y_stats;
    const float *y_sums;            // the LayerNorm backward's two sums per sample,
    const float *y_part;            // MERGE: or the pairs that they come from, merged here by `lanes` threads each
    int lanes;
    const float *saved;
    const float *x, *x_stats;       // the step's input: raw, and the statistics of the LayerNorm on it (null: as it is)
    float *dx, *x_part;             // x_part: pairs for the LayerNorm on x, or null
    float *dweight, *dbias, *dscale, *dgamma, *dbeta;
    long slab_stride;               // a copy of the gradient arrays per batch chunk (0: the arrays themselves)
    int accumulate;                 // on top of what the gradient arrays hold
    int B, M, N, ntube, nchunk, chunk_len;
    CuShare together;
};

// PLAIN: two cells per thread, GATED: one; 54 mirrored weights and 54 gradient accumulators for each set
// and two cells.  A thread moves its own row and one or two of the 20 rows around the tube.
// MERGE: the merged sums go through LDS into SETS registers of every wave, which the loop takes them from with a
// readlane.  (Read from LDS by every element they cost the step 4 us of 67.)  The plain update has one register to
// spare for them, and merges for 32 samples at most: both sums of sample s0 + e in lanes 2 e and 2 e + 1.  Longer chunks,
// of over a thousand samples on fewer than 64 tubes, leave it to the kernel between the steps (16 x 16 x 32, batch 2048, 121 ->
// 123 us); the register filled again after 32 samples spilled three, and 32^3, batch 256, lost what it gains.
constexpr int bwd_merge_most(int sets) { return sets == 1 ? kWave / 2 : kWave; }
template <int ACT, int SETS, int K, bool MERGE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void rows_bwd(RowsBwdArgs a) {
    constexpr int CPT = 2 / SETS;
    extern __shared__ __attribute__((aligned(16))) float lds[];  // [2][SETS][36][K], then gamma and (plain) scale of the rows; MERGE: the sums
    int tube, chunk;
    if (!split_block_id(blockIdx.x, a.ntube, a.nchunk, a.together, false, tube, chunk)) return;  // grid padding
    const int tid = threadIdx.x, M = a.M, N = a.N, nw = blockDim.x / 64, wave = tid / 64;
    const RowPlace<CPT, K> p(tid, tube, N);
    const long cells = (long)M * N * K, tensor = (long)a.B * cells;
    const bool ln_in = a.x_stats != nullptr;
    const int s0 = chunk * a.chunk_len, s1 = min(a.B, s0 + a.chunk_len);
    const long slab = chunk * a.slab_stride;
    float *dweight = a.dweight + slab;
    float *merged = lds + (2 * SETS + 1 + (SETS == 1)) * kWinRows * K;  // of the samples s0 ... s1

    // ---- mirrored weights W[26 - t, c + off_t] and the gradients of those weights ----
    // A tap's weights for the thread's cells lie along K, one cell off its own for dk = -1 / +1: aligned
    // pieces, the missing end from the lane next door (cross_rows.hip).
    float v[SETS][9][3][CPT], nv[SETS][9][3][CPT];
    auto shift_in = [&](float (&piece)[CPT], int cc) {
        if (cc == 0) {
            const float before = lane_before(piece[CPT - 1]);
            if (CPT == 2) piece[CPT - 1] = piece[0];
            piece[0] = before;
        } else if (cc == 2) {
            const float after = lane_after(piece[0]);
            if (CPT == 2) piece[0] = piece[CPT - 1];
            piece[CPT - 1] = after;
        }
    };
    // all requests first (in one stretch: behind a test per tap each would wait for the one before)
    auto load_planes = [&](const float *planes, float (&to)[SETS][9][3][CPT]) {
#pragma unroll
        for (int pq = 0; pq < 9; ++pq) {
            const int gi = p.p0 + p.ci + pq / 3 - 1, gj = p.q0 + p.cj + pq % 3 - 1;
            const bool row_ok = gi >= 0 && gi < M && gj >= 0 && gj < N;
            const unsigned base = 4u * (unsigned)(p.grow + (row_ok ? ((pq / 3 - 1) * N + pq % 3 - 1) * K : 0));
#pragma unroll
            for (int cc = 0; cc < 3; ++cc)
#pragma unroll
                for (int k = 0; k < SETS; ++k)
                    load_at<CPT>(planes + ((26 - (pq * 3 + cc)) * SETS + k) * cells, base, to[k][pq][cc]);
        }
    };
    load_planes(a.weight, v);
    if constexpr (MERGE)  // while the weights are on their way
        merge_pairs<8>(a.y_part, a.ntube * nw, a.lanes, s0, s1 - s0, [&](int e, double t1, double t2, double) {
            reinterpret_cast<float2 *>(merged)[e] = make_float2((float)(t1 / (double)cells), (float)(t2 / (double)cells));
        });
    // a step's sums start from zero, also where there is something to add them to (see the end)
#pragma unroll
    for (int k = 0; k < SETS; ++k)
#pragma unroll
        for (int t = 0; t < 27; ++t)
#pragma unroll
            for (int c = 0; c < CPT; ++c) nv[k][t / 3][t % 3][c] = 0.f;
    float gam[CPT], bet[CPT], rv[CPT] = {}, db[SETS][CPT], dr[CPT] = {}, dgam[CPT], dbet[CPT];
    load_cells<CPT>(a.gamma + p.grow, gam);
    load_cells<CPT>(a.beta + p.grow, bet);
    if (SETS == 1) load_cells<CPT>(a.scale + p.grow, rv);
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
        dgam[c] = dbet[c] = 0.f;
#pragma unroll
        for (int k = 0; k < SETS; ++k) db[k][c] = 0.f;
    }

    // ---- the rows around the tube that this thread moves: number r and, the first four rows, 16 + r ----
    int hoff[2], hat[2];
    bool hok[2];
    // gamma and scale of a thread's rows wait in LDS (each thread reads what it wrote); the scale is zero
    // outside the grid
    float *gam_rows = lds + 2 * SETS * kWinRows * K, *scale_rows = gam_rows + kWinRows * K;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int h = min(p.r + 16 * e, 19);
        const int wi = h < 12 ? h / 6 * (kSide - 1) : 1 + (h - 12) / 2, wj = h < 12 ? h % 6 : (h - 12) % 2 * (kSide - 1);
        const int gi = p.p0 + wi - 1, gj = p.q0 + wj - 1;
        hok[e] = gi >= 0 && gi < M && gj >= 0 && gj < N;
        hoff[e] = hok[e] ? (gi * N + gj) * K + CPT * p.bk : p.grow;  // anything valid when not used
        hat[e] = (wi * kSide + wj) * K + CPT * p.bk;
        float t[CPT];
        load_cells<CPT>(a.gamma + hoff[e], t);
        if (e == 0 || p.r < 4) store_cells<CPT>(gam_rows + hat[e], t);
        if (SETS == 1) {
            load_cells<CPT>(a.scale + hoff[e], t);
#pragma unroll
            for (int c = 0; c < CPT; ++c) t[c] = hok[e] ? t[c] : 0.f;
            if (e == 0 || p.r < 4) store_cells<CPT>(scale_rows + hat[e], t);
        }
    }
    const bool second = p.r < 4;  // whole waves or parts of them
    const int own_row = (p.ci + 1) * kSide + p.cj + 1, own_at = own_row * K + CPT * p.bk;
    store_cells<CPT>(gam_rows + own_at, gam);
    if (SETS == 1) store_cells<CPT>(scale_rows + own_at, rv);
    wait_global_loads();
    const int lane = tid & 63;
    float sums[SETS] = {};
    if (MERGE) {
        lds_barrier();  // the sums are there
#pragma unroll
        for (int k = 0; k < SETS; ++k) sums[k] = merged[SETS * lane + k];  // behind the last sample: anything, not used
    }
#pragma unroll
    for (int pq = 0; pq < 9; ++pq) {
        const int gi = p.p0 + p.ci + pq / 3 - 1, gj = p.q0 + p.cj + pq % 3 - 1;
        const float keep = gi >= 0 && gi < M && gj >= 0 && gj < N ? 1.f : 0.f;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int k = 0; k < SETS; ++k) {
                shift_in(v[k][pq][cc], cc);
#pragma unroll
                for (int c = 0; c < CPT; ++c) v[k][pq][cc][c] *= keep;
                if (cc == 0 && p.first) v[k][pq][cc][0] = 0.f;
                if (cc == 2 && p.last) v[k][pq][cc][CPT - 1] = 0.f;
            }
    }

    // what an element needs, requested TWO elements ahead: dy, y and the saved factors of the cell (plain:
    // u; gated: f0, f1, and of the own cells the gate)
    constexpr int NF = SETS;
    struct Ahead {
        float dy[3][CPT], y[3][CPT], f[3][NF][CPT], gate[CPT], x[CPT];
        float numbers;  // of the sample, by lane: statistics of y, the two sums (not with MERGE), statistics of x
    };
    const unsigned own_off = 4u * (unsigned)p.grow;
    const unsigned off[3] = {own_off, 4u * (unsigned)hoff[0], 4u * (unsigned)hoff[1]};
    // MERGE: statistics of y in lanes 0 and 1, of x in 4 and 5, from one base (both are parts of one array)
    const float *number = lane < 2 ? a.y_stats + lane : lane < 4 ? a.y_sums + (lane - 2) : lane < 6 && ln_in ? a.x_stats + (lane - 4) : a.y_stats;
    const float *stats = ln_in ? a.x_stats : a.y_stats;
    const unsigned stat_at = 4u * (lane & 1) + (lane < 4 ? (unsigned)((const char *)a.y_stats - (const char *)stats) : 0u);
    auto fetch = [&](int s, Ahead &n) {
        const long at = (long)s * cells;
        if constexpr (MERGE) {
            float v[1];
            load_at<1>(stats + 2L * s, stat_at, v);
            n.numbers = v[0];
        } else {
            n.numbers = number[2 * s];
        }
        load_at<CPT>(a.x + at, own_off, n.x);
        if (SETS == 2) load_at<CPT>(a.saved + 2 * tensor + at, own_off, n.gate);
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            load_at<CPT>(a.dy + at, off[e], n.dy[e]);
            load_at<CPT>(a.y + at, off[e], n.y[e]);
#pragma unroll
            for (int k = 0; k < NF; ++k) load_at<CPT>(a.saved + k * tensor + at, off[e], n.f[e][k]);
        }
    };
    float out[CPT];
    auto element = [&](int s, float *stage, Ahead &n) {
        auto number_of = [&](int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(n.numbers), k)); };
        auto sum_of = [&](int k) {
            return __int_as_float(SETS == 1 ? __builtin_amdgcn_readlane(__float_as_int(sums[0]), 2 * (s - s0) + k)
                                            : __builtin_amdgcn_readlane(__float_as_int(sums[k * (SETS - 1)]), s - s0));
        };
        const float ymean = number_of(0), yrstd = number_of(1);
        const float c1 = MERGE ? sum_of(0) : number_of(2), c2 = MERGE ? sum_of(1) : number_of(3);
        const float xmean = number_of(4), xrstd = number_of(5);
        // through the LayerNorm's backward: the gradient with respect to the step's raw output
        auto raw_gradient = [&](float dy, float y, float gamma, float &yh) {
            yh = (y - ymean) * yrstd;
            return yrstd * (gamma * dy - c1 - yh * c2);
        };
        float direct[CPT], xh[CPT], xn[CPT];
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
            xn[c] = (n.x[c] - xmean) * xrstd;
        }
        float g_own[CPT];
        load_cells<CPT>(gam_rows + own_at, g_own);
#pragma unroll
        for (int c = 0; c < CPT; ++c) xh[c] = ln_in ? fmaf(xn[c], g_own[c], bet[c]) : n.x[c];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            if (e == 2 && !second) break;
            float delta[SETS][CPT], gq[CPT], rq[CPT];
            const int at = e == 0 ? own_at : hat[e - 1 < 0 ? 0 : e - 1];
            load_cells<CPT>(gam_rows + at, gq);
            if (SETS == 1) load_cells<CPT>(scale_rows + at, rq);
#pragma unroll
            for (int c = 0; c < CPT; ++c) {
                float yh;
                const float g = raw_gradient(n.dy[e][c], n.y[e][c], gq[c], yh);
                const bool in_grid = SETS == 1 || e == 0 || hok[e - 1 < 0 ? 0 : e - 1];
                if (SETS == 1) {
                    float f, d;
                    Act<ACT, float>::fd(n.f[e][0][c], f, d);
                    delta[0][c] = d * g * rq[c];
                    if (e == 0) dr[c] = fmaf(f, g, dr[c]);
                } else {
#pragma unroll
                    for (int k = 0; k < SETS; ++k) delta[k][c] = in_grid ? g * n.f[e][k][c] : 0.f;
                }
                if (e == 0) {
                    direct[c] = SETS == 1 ? g : n.gate[c] * g;
                    dgam[c] = fmaf(n.dy[e][c], yh, dgam[c]);
                    dbet[c] += n.dy[e][c];
#pragma unroll
                    for (int k = 0; k < SETS; ++k) db[k][c] += delta[k][c];
                }
            }
#pragma unroll
            for (int k = 0; k < SETS; ++k)
                store_cells<CPT>(stage + k * kWinRows * K + at, delta[k]);
        }
        // worked out in front of the requests that replace what they come from (behind them, the compiler
        // has to wait for the first of those)
        keep_here(xn);
        keep_here(xh);
        keep_here(direct);
        lds_barrier();  // the stage is complete; the other one's readers are done
        // The result of the element before leaves here, ahead of the requests: the memory counter is in
        // order, and a store behind them would be waited for with the last of them.
        if (s > s0) store_at<CPT>(a.dx + (long)(s - 1) * cells, own_off, out);
        fetch(min(s + 2, s1 - 1), n);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < CPT; ++c) out[c] = direct[c];
#pragma unroll
        for (int k = 0; k < SETS; ++k)
#pragma unroll
            for (int pq = 0; pq < 9; ++pq) {
                const int di = pq / 3 - 1, dj = pq % 3 - 1;
                float mid[CPT];
                load_cells<CPT>(stage + k * kWinRows * K + own_at + (di * kSide + dj) * K, mid);
                row_products(mid, v[k][pq], xh, out, nv[k][pq]);
            }
        if (a.x_part) {  // the sums of the LayerNorm on x, one pair per wave
            float t1 = 0.f, t2 = 0.f, g_own[CPT];
            load_cells<CPT>(gam_rows + own_at, g_own);
#pragma unroll
            for (int c = 0; c < CPT; ++c) {
                const float go = g_own[c] * out[c];
                t1 += go;
                t2 = fmaf(go, xn[c], t2);
            }
            t1 = slot_wave_sum<64>(t1);
            t2 = slot_wave_sum<64>(t2);
            if ((tid & 63) == 0) {
                float *to = a.x_part + (((long)s * a.ntube + tube) * nw + wave) * 2;
                to[0] = t1;
                to[1] = t2;
            }
        }
    };
    float *stages[2] = {lds, lds + SETS * kWinRows * K};
    Ahead even, odd;
    fetch(min(s0, a.B - 1), even);
    fetch(min(s0 + 1, a.B - 1), odd);
    // in pairs: with a test between the two the compiler counts on fewer requests in flight, and waits for all
    int s = s0;
    for (; s + 1 < s1; s += 2) {
        element(s, stages[0], even);
        element(s + 1, stages[1], odd);
    }
    if (s < s1) element(s, stages[0], even);
    if (s0 < s1) store_at<CPT>(a.dx + (long)(s1 - 1) * cells, own_off, out);

    // ---- parameter gradients: the shifts of the set-up back again, aligned stores of whole rows ----
    // What the arrays hold is added HERE, once, to the finished sums of this step.  Accumulators that
    // started from it would take every product of the chain into one running fp32 sum, most of them small
    // beside it: 64 elements x 64 steps at 32^3, batch 256, left dbias 8e-7 to 5e-6 off the sum in 64 bits, this
    // way 1e-7 to 5e-7, for 6.69 and 6.60 ms per training step (plain), 9.20 and 9.28 (gated).  The weights are
    // done with: their registers take the old values, requested in one stretch.
    float old_db[SETS][CPT] = {}, old_dr[CPT] = {}, old_dgam[CPT] = {}, old_dbet[CPT] = {};
    if (a.accumulate) {
        load_planes(dweight, v);
#pragma unroll
        for (int k = 0; k < SETS; ++k) load_cells<CPT>(a.dbias + slab + k * cells + p.grow, old_db[k]);
        if (SETS == 1) load_cells<CPT>(a.dscale + slab + p.grow, old_dr);
        load_cells<CPT>(a.dgamma + slab + p.grow, old_dgam);
        load_cells<CPT>(a.dbeta + slab + p.grow, old_dbet);
    } else {
#pragma unroll
        for (int k = 0; k < SETS; ++k)
#pragma unroll
            for (int t = 0; t < 27; ++t)
#pragma unroll
                for (int c = 0; c < CPT; ++c) v[k][t / 3][t % 3][c] = 0.f;
    }
#pragma unroll
    for (int pq = 0; pq < 9; ++pq) {
        const int gi = p.p0 + p.ci + pq / 3 - 1, gj = p.q0 + p.cj + pq % 3 - 1;
        const bool row_ok = gi >= 0 && gi < M && gj >= 0 && gj < N;
        const int base = (gi * N + gj) * K + CPT * p.bk;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int k = 0; k < SETS; ++k) {
                const float (&n)[CPT] = nv[k][pq][cc];
                float piece[CPT];
                if (cc == 1) {
#pragma unroll
                    for (int c = 0; c < CPT; ++c) piece[c] = n[c];
                } else if (cc == 0) {  // from the cell after; behind the row's last cell there is none
                    const float after = lane_after(n[0]);
                    if (CPT == 2) piece[0] = n[CPT - 1];
                    piece[CPT - 1] = p.last ? 0.f : after;
                } else {
                    const float before = lane_before(n[CPT - 1]);
                    if (CPT == 2) piece[CPT - 1] = n[0];
                    piece[0] = p.first ? 0.f : before;
                }
                const int t = pq * 3 + cc;
                float *to = dweight + (long)((26 - t) * SETS + k) * cells + base;
                if (row_ok) {
#pragma unroll
                    for (int c = 0; c < CPT; ++c) piece[c] += v[k][pq][cc][c];
                    store_cells<CPT>(to, piece);
                } else if (!a.accumulate) {  // the own weight of tap t reads outside the grid: no gradient
#pragma unroll
                    for (int c = 0; c < CPT; ++c) piece[c] = 0.f;
                    store_cells<CPT>(dweight + (long)(t * SETS + k) * cells + p.grow, piece);
                }
            }
    }
    auto add = [](float (&to)[CPT], const float (&more)[CPT]) {
#pragma unroll
        for (int c = 0; c < CPT; ++c) to[c] += more[c];
    };
    add(dr, old_dr);
    add(dgam, old_dgam);
    add(dbet, old_dbet);
#pragma unroll
    for (int k = 0; k < SETS; ++k) {
        add(db[k], old_db[k]);
        store_cells<CPT>(a.dbias + slab + k * cells + p.grow, db[k]);
    }
    if (SETS == 1) store_cells<CPT>(a.dscale + slab + p.grow, dr);
    store_cells<CPT>(a.dgamma + slab + p.grow, dgam);
    store_cells<CPT>(a.dbeta + slab + p.grow, dbet);
}

// ---- host side -------------------------------------------------------------------------------
int sets_of(const RowsChain &c) { return c.gated ? 2 : 1; }
long cells_of(const RowsChain &c) { return (long)c.M * c.N * c.K; }
int tubes_of(const RowsChain &c) { return c.M / kTube * (c.N / kTube); }
int fwd_threads(const RowsChain &c) { return 16 * c.K * sets_of(c) / 4; }
int bwd_threads(const RowsChain &c) { return 16 * c.K * sets_of(c) / 2; }
int fwd_pairs(const RowsChain &c) { return tubes_of(c) * fwd_threads(c) / 64; }
int bwd_pairs(const RowsChain &c) { return tubes_of(c) * bwd_threads(c) / 64; }
size_t align_up(size_t v) { return (v + 255) / 256 * 256; }
size_t part_bytes(int B, int pairs) { return align_up((size_t)B * pairs * 2 * sizeof(float)); }

template <typename K> int workgroups_per_cu(K kern, int threads, size_t lds) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void *)kern, threads, lds) != hipSuccess || n < 1) n = 1;
    return n;
}
// The chunks of a tube on one CU.  Per step, forward / backward: 32^3, batch 256, 29.1 -> 28.2 / 68.7 -> 67.0 us; batch
// 64, 13.4 -> 13.1 / 29.9 -> 29.4.  Not with rows of 64 cells: 64^3, batch 32, forward 30.8 -> 32.5.
template <int K> CuShare rows_together(int ntube, int nchunk, int per_cu) {
    return K < 64 ? cu_share(ntube, nchunk, per_cu) : CuShare{};
}

template <int ACT, int SETS, bool SAVE, int K> int run_forward(const RowsChain &c, hipStream_t st) {
    const auto kern = rows_fwd<ACT, SETS, SAVE, K, false>, merging = rows_fwd<ACT, SETS, SAVE, K, true>;
    const long cells = cells_of(c), tensor = (long)c.B * cells;
    const int ntube = tubes_of(c), nt = fwd_threads(c), pairs = fwd_pairs(c);
    const size_t lds = 4 * (size_t)kWinRows * c.K * sizeof(float) + kMergeMostSamples * sizeof(float2);
    static int per_cu = 0;  // per instantiation
    if (per_cu == 0) per_cu = workgroups_per_cu(kern, nt, lds);
    RowsFwdArgs a{};
    a.nchunk = plan_row_chunks(c.B, ntube, per_cu * plan_device_cus(), kRowsMinWalk, a.chunk_len);
    a.lanes = plan_merge_lanes(nt, a.chunk_len, pairs);
    a.together = rows_together<K>(ntube, a.nchunk, per_cu);
    a.eps = c.eps;
    a.weight = c.weight; a.bias = c.bias; a.scale = c.scale; a.gamma = c.gamma; a.beta = c.beta;
    a.B = c.B; a.M = c.M; a.N = c.N; a.ntube = ntube;
    // workspace: the pairs; and, where nothing is kept, statistics and two raw tensors
    char *ws = (char *)c.workspace;
    float *parts[2] = {(float *)ws, (float *)(ws + part_bytes(c.B, pairs))};
    ws += 2 * part_bytes(c.B, pairs);
    float *own_stats = (float *)ws, *own_y = (float *)(ws + align_up((size_t)2 * c.B * sizeof(float)));
    for (int j = 0; j < c.outer; ++j) {
        float *stats = c.stats ? c.stats + (long)j * 2 * c.B : own_stats;
        a.x = j ? a.y : c.x0;
        a.x_part = a.y_part;
        a.stats_out = c.stats ? stats - 2 * c.B : nullptr;
        a.y_part = parts[j & 1];
        a.y = c.y_raw ? c.y_raw + j * tensor : own_y + (j & 1) * tensor;
        a.saved = SAVE ? c.saved + (long)j * (SETS == 1 ? 1 : 3) * tensor : nullptr;
        hipLaunchKernelGGL(j && a.lanes ? merging : kern, dim3(padded_grid(ntube, a.nchunk)), dim3(nt), lds, st, a);
        if (int rc = check_launch("rows_fwd")) return rc;
        if (a.lanes && j + 1 < c.outer) continue;
        if (int rc = layernorm_finalize_stats(a.y_part, pairs, (int)(cells / pairs), stats, c.B, c.eps, st)) return rc;
        a.x_stats = stats;
    }
    return layernorm_apply_stats(a.y, a.x_stats, c.gamma, c.beta, c.out, c.B, cells, st);
}

// at least eight elements per copy of the gradient arrays, but where that leaves CUs without a
// workgroup, down to three (as bwd_rows.hip)
int bwd_chunks(const RowsChain &c, int per_cu, int &chunk_len) {
    const int cus = plan_device_cus(), ntube = tubes_of(c);
    const int n = plan_row_chunks(c.B, ntube, per_cu * cus, 8, chunk_len);
    return n * ntube >= cus ? n : plan_row_chunks(c.B, ntube, cus, kRowsMinWalk, chunk_len);
}
constexpr int kBwdMostPerCu = 4;
// no fewer than bwd_chunks gives, here or at any smaller batch: what the workspace is sized for
int bwd_most_chunks(const RowsChain &c) {
    const int fill = plan_device_cus() / tubes_of(c);
    const int walks = std::min(kBwdMostPerCu * plan_device_cus() / tubes_of(c), c.B / 8);
    return std::max({walks, std::min(fill, c.B / kRowsMinWalk), 1});
}
int grad_planes(const RowsChain &c) { return c.gated ? 58 : 31; }

template <int ACT, int SETS, int K> int run_backward(const RowsChain &c, hipStream_t st) {
    const auto kern = rows_bwd<ACT, SETS, K, false>, merging = rows_bwd<ACT, SETS, K, true>;
    const long cells = cells_of(c), tensor = (long)c.B * cells;
    const int ntube = tubes_of(c), nt = bwd_threads(c), pairs = bwd_pairs(c);
    const size_t lds = (2 * SETS + 1 + (SETS == 1)) * (size_t)kWinRows * K * sizeof(float) + SETS * kWave * sizeof(float);
    static int per_cu = 0;  // per instantiation
    if (per_cu == 0) {
        const int n = workgroups_per_cu(kern, nt, lds);
        per_cu = n < kBwdMostPerCu ? n : kBwdMostPerCu;
    }
    RowsBwdArgs a{};
    a.nchunk = bwd_chunks(c, per_cu, a.chunk_len);
    a.lanes = a.chunk_len <= bwd_merge_most(SETS) ? plan_merge_lanes(nt, a.chunk_len, pairs) : 0;
    a.together = rows_together<K>(ntube, a.nchunk, per_cu);
    a.weight = c.weight; a.scale = c.scale; a.gamma = c.gamma; a.beta = c.beta;
    a.B = c.B; a.M = c.M; a.N = c.N; a.ntube = ntube;
    // workspace: the pairs, the sums, scratch of the last LayerNorm's sums, a second dx, the copies
    char *ws = (char *)c.workspace;
    float *parts[2] = {(float *)ws, (float *)(ws + part_bytes(c.B, pairs))};
    ws += 2 * part_bytes(c.B, pairs);
    float *sums = (float *)ws;
    ws += align_up((size_t)2 * c.B * sizeof(float));
    float *scratch = (float *)ws;
    ws += align_up(layernorm_workspace(GRIDNET_F32, c.B, cells));
    float *other_dx = (float *)ws;
    ws += align_up((size_t)tensor * sizeof(float));
    float *slabs = (float *)ws;
    const int wplanes = 27 * SETS;
    const long slab_floats = grad_planes(c) * cells;
    const bool split = a.nchunk > 1, add = (c.flags & GRIDNET_OVERWRITE_PARAMS) == 0;
    SlabTargets t{};
    int k = 0;
    auto target = [&](float *dst, long planes) {
        t.dst[k] = dst;
        t.end[k] = (k ? t.end[k - 1] : 0) + planes * cells;
        ++k;
    };
    target(c.dweight, wplanes);
    target(c.dbias, SETS);
    if (SETS == 1) target(c.dscale, 1);
    target(c.dgamma, 1);
    target(c.dbeta, 1);
    t.count = k;
    if (split) {
        a.dweight = slabs;
        a.dbias = a.dweight + wplanes * cells;
        a.dscale = SETS == 1 ? a.dbias + cells : nullptr;
        a.dgamma = a.dbias + 2 * cells;  // plain: behind the scale; gated: behind the second bias
        a.dbeta = a.dgamma + cells;
        a.slab_stride = slab_floats;
    } else {
        a.dweight = c.dweight; a.dbias = c.dbias; a.dscale = c.dscale; a.dgamma = c.dgamma; a.dbeta = c.dbeta;
    }
    const long last = c.outer - 1;
    if (int rc = layernorm_backward_sums(c.dy, c.y_raw + last * tensor, c.stats + last * 2 * c.B, c.gamma, sums, c.B, cells,
                                         scratch, st))
        return rc;
    a.dy = c.dy;
    a.y_sums = sums;
    for (long j = last; j >= 0; --j) {
        a.y = c.y_raw + j * tensor;
        a.y_stats = c.stats + j * 2 * c.B;
        a.saved = c.saved + j * (SETS == 1 ? 1 : 3) * tensor;
        a.x = j ? c.y_raw + (j - 1) * tensor : c.x0;
        a.x_stats = j ? c.stats + (j - 1) * 2 * c.B : nullptr;
        a.y_part = parts[(j + 1) & 1];
        a.x_part = j ? parts[j & 1] : nullptr;
        a.dx = j & 1 ? other_dx : c.dx;
        a.accumulate = j < last || (!split && add);
        hipLaunchKernelGGL(j < last && a.lanes ? merging : kern, dim3(padded_grid(ntube, a.nchunk)), dim3(nt), lds, st, a);
        if (int rc = check_launch("rows_bwd")) return rc;
        a.dy = a.dx;
        if (j && !a.lanes)
            if (int rc = layernorm_finalize_sums(parts[j & 1], pairs, cells, sums, c.B, st)) return rc;
    }
    if (!split) return GRIDNET_OK;
    return plan_launch_tail_job(plan_tail_job(slabs, a.nchunk, slab_floats, t, add ? ~0 : 0, 256), st);
}

template <int ACT, int SETS, bool SAVE> int forward_rows(const RowsChain &c, hipStream_t st) {
    if (c.K == 16) return run_forward<ACT, SETS, SAVE, 16>(c, st);
    if (c.K == 32) return run_forward<ACT, SETS, SAVE, 32>(c, st);
    if constexpr (SETS == 1) return run_forward<ACT, SETS, SAVE, 64>(c, st);
    return fail(GRIDNET_ERR_ARGUMENT, "rows of %d cells", c.K);
}
template <int ACT, int SETS> int backward_rows(const RowsChain &c, hipStream_t st) {
    if (c.K == 16) return run_backward<ACT, SETS, 16>(c, st);
    if (c.K == 32) return run_backward<ACT, SETS, 32>(c, st);
    if constexpr (SETS == 1) return run_backward<ACT, SETS, 64>(c, st);
    return fail(GRIDNET_ERR_ARGUMENT, "rows of %d cells", c.K);
}
template <int SETS, bool SAVE> int forward_act(const RowsChain &c, hipStream_t st) {
    switch (c.activation) {
        case GRIDNET_ACT_RELU: return forward_rows<GRIDNET_ACT_RELU, SETS, SAVE>(c, st);
        case GRIDNET_ACT_LEAKY_RELU: return forward_rows<GRIDNET_ACT_LEAKY_RELU, SETS, SAVE>(c, st);
        case GRIDNET_ACT_SILU: return forward_rows<GRIDNET_ACT_SILU, SETS, SAVE>(c, st);
        case GRIDNET_ACT_TANH: return forward_rows<GRIDNET_ACT_TANH, SETS, SAVE>(c, st);
    }
    return fail(GRIDNET_ERR_ACTIVATION, "unknown activation function: id %d", c.activation);
}
// The gated backward works on saved factors: no activation in it.
template <int SETS> int backward_act(const RowsChain &c, hipStream_t st) {
    if constexpr (SETS == 2) {
        return backward_rows<GRIDNET_ACT_RELU, SETS>(c, st);
    } else {
        switch (c.activation) {
            case GRIDNET_ACT_RELU: return backward_rows<GRIDNET_ACT_RELU, SETS>(c, st);
            case GRIDNET_ACT_LEAKY_RELU: return backward_rows<GRIDNET_ACT_LEAKY_RELU, SETS>(c, st);
            case GRIDNET_ACT_SILU: return backward_rows<GRIDNET_ACT_SILU, SETS>(c, st);
            case GRIDNET_ACT_TANH: return backward_rows<GRIDNET_ACT_TANH, SETS>(c, st);
        }
    }
    return fail(GRIDNET_ERR_ACTIVATION, "unknown activation function: id %d", c.activation);
}

}  // namespace

// Rows that are a power of two of lanes in both kernels; with two weight sets a row of 64 cells would
// take a workgroup of 1024 threads, whose waves have half the registers this needs.
bool rows_chain_supports(int M, int N, int K, bool gated) {
    if (M <= 0 || N <= 0 || M % kTube || N % kTube || (long)M * N * K * 54 >= (1L << 31)) return false;
    return K == 16 || K == 32 || (K == 64 && !gated);
}

size_t rows_chain_workspace(const RowsChain &c, bool backward) {
    if (!backward) {
        size_t n = 2 * part_bytes(c.B, fwd_pairs(c)) + align_up((size_t)2 * c.B * sizeof(float));
        if (!c.keep) n += 2 * (size_t)c.B * cells_of(c) * sizeof(float);
        return n;
    }
    const int chunks = bwd_most_chunks(c);
    return 2 * part_bytes(c.B, bwd_pairs(c)) + align_up((size_t)2 * c.B * sizeof(float)) +
           align_up(layernorm_workspace(GRIDNET_F32, c.B, cells_of(c))) + align_up((size_t)c.B * cells_of(c) * sizeof(float)) +
           (chunks > 1 ? (size_t)chunks * grad_planes(c) * cells_of(c) * sizeof(float) : 0);
}

int rows_chain_forward(const RowsChain &c, hipStream_t st) {
    if (c.gated) return c.saved ? forward_act<2, true>(c, st) : forward_act<2, false>(c, st);
    return c.saved ? forward_act<1, true>(c, st) : forward_act<1, false>(c, st);
}

int rows_chain_backward(const RowsChain &c, hipStream_t st) {
    return c.gated ? backward_act<2>(c, st) : backward_act<1>(c, st);
}

}  // namespace gridnet
