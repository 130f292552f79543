// One step in fp64, forward and backward (gradient checks and reference runs), a thread per cell.
// Backward calls without scratch, and those that step_f64_supports leaves out, keep the scattering kernel
// of step_generic.hip.
//
// That kernel sends each of a cell's 27 products w[t] * delta to the window by an LDS atomic, every inner
// iteration, works the pre-activation out a second time on the way back, and adds dx, and where the batch
// of a block is split its parameter gradients too, by global atomics to arrays that four launches have
// zeroed.  Here
//   * a thread gathers: on the way back it holds, for every neighbour in its block, the weight that reads ITS
//     cell (V[t] = W[26-t, c+off_t]); the gradient of the cell is a sum over the deltas around it, read from a
//     window with a zero halo, and x[c] * delta[c+off_t] from the same reads is the gradient of that neighbour
//     weight: 27 reads and 54 multiply-adds, no atomics, one barrier.  Its own weights and V are fetched when
//     their turn comes (81 doubles at once do not fit beside the rest: 24 to 72 spilled registers);
//   * values, activations and their derivatives of the recompute wait in LDS;
//   * what crosses a block boundary depends on the iterations only through sums over them, because the
//     window's halo is frozen: a second kernel adds sum_(c,t)->h w[t,c] D[c], D = sum_i delta_i, to the cells h
//     around a block.  The gradient of a weight whose tap reads a halo entry is x_h D[c]; it is kept where
//     the gradient of a neighbour's weight would be if that neighbour were in the block.
// With normalisation, dz_i the gradient with respect to the normalised window, every raw entry k gets
//   inv_i (dz_i[k] - A_i / W) - C_i (x_i[k] - mean_i),  A_i = sum dz_i,  C_i ~ sum dz_i (x_i - mean_i)
// over the whole window; what the halo adds to either sum is delta[c] times a number per cell and element
// (`wh`, `sh`: the cell's weights that read the halo, and those times what they read).  A halo entry gets
// sum w D1 - x_h Q + R with D1 = sum_i inv_i delta_i, Q = sum_i C_i, R = sum_i (C_i mean_i - inv_i A_i / W),
// the gradient of a weight that reads it x_h D1 - D2, D2 = sum_i mean_i inv_i delta_i; x and the means less the
// window's shift (`shift_of`), or these differences would cancel.
// No atomics anywhere: two runs give the same bits.
//
// What bounds it: latency, at one workgroup of eight waves per CU (216 to 256 registers).  24 x 32 x 32, batch
// 6, three inner iterations: per workgroup 9 us of set-up and gradient stores and 10 us an element, of which the
// six passes over LDS take 5; backward 67 us with the scattering kernel and its fills, 39 now (forward 10.9 -> 9.0);
// 40^3, batch 12, four iterations with normalize 257 -> 182 (forward 53 -> 38).

#include "common.h"
#include "fast_tiles.h"
#include "launch.h"
#include "plan.h"

#include <type_traits>

namespace gridnet {

namespace {

// LDS row and plane strides of the window, and which way the lanes run: with the 32 lanes that a 64-bit
// access serves together on different banks.  Plain strides of S and S * S put them on the same ones two by
// two, and these kernels' time went with the LDS (a pass of 27 reads 1.0 us of 1.25).
template <int BS> struct Geo {
    static constexpr int S = BS + 2;                 // window side
    static constexpr int W = S * S * S;              // window entries
    static constexpr int NT = BS * BS * BS;          // threads = cells
    static constexpr int RS = BS == 8 ? 10 : 8;
    static constexpr int PS = BS == 8 ? 104 : 52;
    static constexpr int WIN = S * PS;               // a window in LDS
    // window position of tap t of the cell that sits at `base`
    static __device__ __forceinline__ int tap(int base, int t) { return base + t / 9 * PS + t / 3 % 3 * RS + t % 3; }
};

// A thread's cell: lanes run along k, then i with 8^3 blocks and j with 4^3, then the third axis.
template <int BS> struct Cell {
    using G = Geo<BS>;
    int p0, q0, r0, i, j, k;  // block origin in the grid, place in the block
    int gc, base, centre;     // grid index, window positions of tap 0 and of the cell itself
    int first;                // grid index of the block's first cell
    __device__ __forceinline__ Cell(int tid, int blk, int N, int K) {
        const int kb = K / BS, nb = N / BS;
        p0 = (blk / (kb * nb)) * BS, q0 = ((blk / kb) % nb) * BS, r0 = (blk % kb) * BS;
        const int b = tid / BS % BS, c = tid / (BS * BS);
        k = tid % BS, i = BS == 8 ? b : c, j = BS == 8 ? c : b;
        gc = ((p0 + i) * N + (q0 + j)) * K + (r0 + k);
        first = (p0 * N + q0) * K + r0;
        base = i * G::PS + j * G::RS + k;
        centre = G::tap(base, 13);
    }
};

template <int BS> struct Shell {
    static constexpr int S = BS + 2, kCells = S * S * S - BS * BS * BS;
    static constexpr int kPerThread = (kCells + BS * BS * BS - 1) / (BS * BS * BS);
    // window coordinates of shell entry n: two planes along i, then along j, then along k
    static __device__ __forceinline__ void at(int n, int &wi, int &wj, int &wk) {
        constexpr int planes_i = 2 * S * S, planes_j = 2 * BS * S;
        if (n < planes_i) {
            wi = n / (S * S) * (S - 1), wj = n / S % S, wk = n % S;
        } else if (n < planes_i + planes_j) {
            const int t = n - planes_i;
            wi = 1 + t / (2 * S), wj = t / S % 2 * (S - 1), wk = t % S;
        } else {
            const int t = n - planes_i - planes_j;
            wi = 1 + t / (2 * BS), wj = 1 + t / 2 % BS, wk = t % 2 * (S - 1);
        }
    }
};

constexpr int kWaveRed = 8;  // waves of the largest workgroup
constexpr size_t kF64MaxLds = 160 * 1024;
template <int BS> __host__ __device__ constexpr size_t bwd_f64_lds(int inner, int slabs) {
    return (4 * Geo<BS>::WIN + slabs * inner * Geo<BS>::NT + 4 * kWaveRed + 3 * inner) * sizeof(double);
}
// the activation and its derivative are kept where LDS has room for both (ten iterations of 8^3 blocks),
// the pre-activation otherwise
template <int BS> __host__ __device__ constexpr bool bwd_f64_keeps_act(int inner) {
    return bwd_f64_lds<BS>(inner, 3) <= kF64MaxLds;
}
template <int BS> size_t bwd_f64_lds(int inner) { return bwd_f64_lds<BS>(inner, bwd_f64_keeps_act<BS>(inner) ? 3 : 2); }

extern __shared__ __align__(16) unsigned char f64_lds[];

// The shell entries a thread looks after: window position (-1: none), grid index (-1: none, or outside)
template <int BS> struct Edges {
    using SH = Shell<BS>;
    using G = Geo<BS>;
    int at[SH::kPerThread], grid[SH::kPerThread];
    __device__ __forceinline__ Edges(int tid, const Cell<BS> &p, int M, int N, int K) {
#pragma unroll
        for (int e = 0; e < SH::kPerThread; ++e) {
            const int n = tid + e * G::NT;
            int wi, wj, wk;
            SH::at(n < SH::kCells ? n : 0, wi, wj, wk);
            const int gi = p.p0 + wi - 1, gj = p.q0 + wj - 1, gk = p.r0 + wk - 1;
            at[e] = n < SH::kCells ? wi * G::PS + wj * G::RS + wk : -1;
            grid[e] = n < SH::kCells && gi >= 0 && gi < M && gj >= 0 && gj < N && gk >= 0 && gk < K
                          ? (gi * N + gj) * K + gk : -1;
        }
    }
    // the shell of sample `xs`, less `shift`, into both window copies, and into `halo` (0 where there is no entry)
    __device__ __forceinline__ void fill(const double *xs, double shift, double *win, double (&halo)[SH::kPerThread]) const {
#pragma unroll
        for (int e = 0; e < SH::kPerThread; ++e) {
            halo[e] = (grid[e] >= 0 ? xs[grid[e]] : 0.0) - (at[e] >= 0 ? shift : 0.0);
            if (at[e] >= 0) win[at[e]] = win[G::WIN + at[e]] = halo[e];
        }
    }
};

// What a normalised window is worked on without: its block's first cell.  The result does not depend on it, and
// differences of neighbours are exact, where sums and differences of values with a large mean round at its scale.
// Error of dweight over its norm, without -> with, 24^3, three iterations, x around 100: 4e-15 -> 2e-16, 1e4: 4e-13 ->
// 2e-16, 1e6: 3e-11 -> 1e-14.  It costs the forward up to 5 %, the backward's kernels 1 to 2 and 0.3 us.
// None where squares of it leave the range: that window's variance is infinite, as it is without.
__device__ __forceinline__ double shift_of(double first) { return __builtin_fabs(first) < 1e150 ? first : 0.0; }
// (the same for the whole workgroup: in scalar registers)
__device__ __forceinline__ double shift_of_block(const double *xs, int first) {
    const double v = shift_of(xs[first]);
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)), __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Sums over the workgroup, the same bits in every thread; `red` is this call's own (two calls in a row take
// different ones), so one barrier is enough.
template <int NT, int COUNT> __device__ __forceinline__ void sum_all(double (&v)[COUNT], double *red, int tid) {
#pragma unroll
    for (int c = 0; c < COUNT; ++c) v[c] = wave_sum_dpp(v[c]);
    if constexpr (NT > kWave) {
        if ((tid & (kWave - 1)) == 0)
#pragma unroll
            for (int c = 0; c < COUNT; ++c) red[2 * (tid / kWave) + c] = v[c];
        lds_barrier();
#pragma unroll
        for (int c = 0; c < COUNT; ++c) {
            v[c] = red[c];
#pragma unroll
            for (int i = 1; i < NT / kWave; ++i) v[c] += red[2 * i + c];
        }
    }
}

// Statistics of the window: mean, population std, 1 / (std + eps), in two passes.  `red`: [2][waves][2].
template <int BS>
__device__ __forceinline__ void window_stats(double cur, const double (&halo)[Shell<BS>::kPerThread],
                                             const Edges<BS> &edges, double eps, double *red, int tid,
                                             double &mean, double &sd, double &inv) {
    double sum[1] = {cur};
#pragma unroll
    for (double h : halo) sum[0] += h;
    sum_all<Geo<BS>::NT>(sum, red, tid);
    mean = sum[0] / Geo<BS>::W;
    sum[0] = (cur - mean) * (cur - mean);
#pragma unroll
    for (int e = 0; e < Shell<BS>::kPerThread; ++e)
        sum[0] += edges.at[e] >= 0 ? (halo[e] - mean) * (halo[e] - mean) : 0.0;
    sum_all<Geo<BS>::NT>(sum, red + 2 * kWaveRed, tid);
    sd = sqrt(sum[0] / Geo<BS>::W);
    inv = 1.0 / (sd + eps);
}

// bias + sum w (v - mean) inv; a sum per plane of taps, since one chain of 27 is as long as all else
template <int BS, bool NORM>
__device__ __forceinline__ double pre_activation(const double *win, const double (&w)[27], double bias, int base,
                                                 double mean, double inv) {
    double sum[3] = {NORM ? 0.0 : bias, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < 27; ++t) {
        const double v = win[Geo<BS>::tap(base, t)];
        sum[t / 9] += w[t] * (NORM ? v - mean : v);
    }
    const double u = (sum[0] + sum[1]) + sum[2];
    return NORM ? fma(u, inv, bias) : u;
}

template <int BS, int ACT, bool NORM>
__global__ __launch_bounds__(BS *BS *BS) void step_fwd_f64(
    const double *__restrict__ weight, const double *__restrict__ bias, const double *__restrict__ scale,
    const double *__restrict__ x, double *__restrict__ y, int B, int M, int N, int K, int inner, double eps,
    int nblk, int nchunk, int chunk_len) {
    using G = Geo<BS>;
    __shared__ double win[2 * G::WIN], red[4 * kWaveRed];
    const int tid = threadIdx.x;
    int blk, chunk;
    if (!split_block_id(blockIdx.x, nblk, nchunk, blk, chunk)) return;  // grid padding
    const Cell<BS> p(tid, blk, N, K);
    const Edges<BS> edges(tid, p, M, N, K);
    const long cells = (long)M * N * K;
    double w[27];
#pragma unroll
    for (int t = 0; t < 27; ++t) w[t] = weight[t * cells + p.gc];
    const double bv = bias[p.gc], rv = scale[p.gc];
    const int s_end = min(B, (chunk + 1) * chunk_len);
    for (int s = chunk * chunk_len; s < s_end; ++s) {
        const double *xs = x + s * cells;
        const double shift = NORM ? shift_of_block(xs, p.first) : 0.0;
        double cur = NORM ? xs[p.gc] - shift : xs[p.gc], halo[Shell<BS>::kPerThread];
        edges.fill(xs, shift, win, halo);  // the element before is done with the windows: its last pass wrote none
        win[p.centre] = cur;
        lds_barrier();
        for (int it = 0; it < inner; ++it) {
            double mean = 0.0, sd, inv = 1.0;
            if (NORM) window_stats<BS>(cur, halo, edges, eps, red, tid, mean, sd, inv);
            const double u = pre_activation<BS, NORM>(win + (it & 1) * G::WIN, w, bv, p.base, mean, inv);
            cur += rv * Act<ACT, double>::f(u);
            if (it + 1 < inner) win[((it + 1) & 1) * G::WIN + p.centre] = cur;
            lds_barrier();
        }
        y[s * cells + p.gc] = NORM ? cur + shift : cur;
    }
}

// (two waves per SIMD asked for: left alone the compiler takes a few registers more with normalize and 4^3 blocks, and
// there is one; 40^3, batch 4, three iterations, 57 us instead of 47)
template <int BS, int ACT, bool NORM>
__global__ __launch_bounds__(BS *BS *BS, 2) void step_bwd_f64(
    const double *__restrict__ weight, const double *__restrict__ bias, const double *__restrict__ scale,
    const double *__restrict__ x, const double *__restrict__ dy, double *__restrict__ dweight,
    double *__restrict__ dbias, double *__restrict__ dscale, double *__restrict__ dx, double *__restrict__ dsum,
    double *__restrict__ halo_part, int B, int M, int N, int K, int inner, double eps, int nblk, int nchunk,
    int chunk_len, int add_dx, int add_params, long copy_stride) {
    using G = Geo<BS>;
    using SH = Shell<BS>;
    double *win = reinterpret_cast<double *>(f64_lds);  // two copies of the window, alternating
    double *dwin = win + 2 * G::WIN;                    // two of the deltas, their halo zero
    const bool keep_act = bwd_f64_keeps_act<BS>(inner);
    const int slabs = keep_act ? 3 : 2;
    double *hist = dwin + 2 * G::WIN;              // [inner][slabs][cells]: value; act, act' or the pre-activation
    double *red = hist + slabs * inner * G::NT;    // [2][waves][2]
    double *stat = red + 4 * kWaveRed;             // [inner][3]: mean, std, 1 / (std + eps)

    const int tid = threadIdx.x;
    int blk, chunk;
    if (!split_block_id(blockIdx.x, nblk, nchunk, blk, chunk)) return;  // grid padding
    const Cell<BS> p(tid, blk, N, K);
    const Edges<BS> edges(tid, p, M, N, K);
    const long cells = (long)M * N * K;
    const int gc = p.gc, base = p.base, centre = p.centre;

    // bit t: tap t of this thread's cell stays in the block.  Taken through `now` where it is used, or the
    // compiler keeps the 27 lane masks that follow from it in scalar registers, and those in vector ones.
    unsigned stays = 0;
#pragma unroll
    for (int t = 0; t < 27; ++t)
        if ((unsigned)(p.i + t / 9 - 1) < BS && (unsigned)(p.j + t / 3 % 3 - 1) < BS && (unsigned)(p.k + t % 3 - 1) < BS)
            stays |= 1u << t;
    const auto now = [](auto value) {
        asm volatile("" : "+v"(value));
        return value;
    };
    double dw[27];
#pragma unroll
    for (int t = 0; t < 27; ++t) dw[t] = 0.0;
    const double bv = bias[gc], rv = scale[gc];
    double db = 0.0, dr = 0.0;
    for (int idx = tid; idx < 2 * G::WIN; idx += G::NT) dwin[idx] = 0.0;

    const int s_end = min(B, (chunk + 1) * chunk_len);
    for (int s = chunk * chunk_len; s < s_end; ++s) {
        const double *xs = x + s * cells;
        const double shift = NORM ? shift_of_block(xs, p.first) : 0.0;
        double cur = NORM ? xs[gc] - shift : xs[gc], g = dy[s * cells + gc], halo[SH::kPerThread];
        lds_barrier();  // the element before is done with the windows
        edges.fill(xs, shift, win, halo);
        win[centre] = cur;
        // The cell's own weights are fetched for every element and are gone on the way back: with them the
        // 81 doubles per thread do not fit beside the rest (24 to 72 registers spilled).
        double w[27];
        {
            const int at = now(gc);
#pragma unroll
            for (int t = 0; t < 27; ++t) w[t] = weight[t * cells + at];
        }
        lds_barrier();

        double wh = 0.0, sh = 0.0;  // NORM: the cell's weights that read the halo, and those times what they read
        if (NORM) {
            const unsigned in = now(stays);
#pragma unroll
            for (int t = 0; t < 27; ++t) {
                const double h = win[G::tap(base, t)];
                wh += in >> t & 1 ? 0.0 : w[t];
                sh += in >> t & 1 ? 0.0 : w[t] * h;
            }
        }
        // recompute
        for (int it = 0; it < inner; ++it) {
            const double *from = win + (it & 1) * G::WIN;
            double mean = 0.0, inv = 1.0;
            if (NORM) {
                double sd;
                window_stats<BS>(cur, halo, edges, eps, red, tid, mean, sd, inv);
                if (tid == 0) {
                    stat[3 * it] = mean;
                    stat[3 * it + 1] = sd;
                    stat[3 * it + 2] = inv;
                }
            }
            const double u = pre_activation<BS, NORM>(from, w, bv, base, mean, inv);
            double *mine = hist + slabs * it * G::NT + tid, f, d;
            Act<ACT, double>::fd(u, f, d);
            mine[0] = cur;
            mine[G::NT] = keep_act ? f : u;
            if (keep_act) mine[2 * G::NT] = d;
            cur += rv * f;
            win[((it + 1) & 1) * G::WIN + centre] = cur;
            lds_barrier();
        }

        double v[27];
        {
            const int at = now(gc);
            const unsigned in = now(stays);
#pragma unroll
            for (int t = 0; t < 27; ++t) {
                const bool has = in >> t & 1;
                const double m =
                    weight[(26 - t) * cells + at + (has ? ((t / 9 - 1) * N + t / 3 % 3 - 1) * K + t % 3 - 1 : 0)];
                v[t] = has ? m : 0.0;
            }
        }
        double d1 = 0.0, d2 = 0.0, q = 0.0, r = 0.0;
        for (int it = inner - 1; it >= 0; --it) {
            const double *mine = hist + slabs * it * G::NT + tid;
            const double xi = mine[0], u = mine[G::NT];
            double *dwi = dwin + (it & 1) * G::WIN;
            double f = u, d;
            if (keep_act) d = mine[2 * G::NT];
            else Act<ACT, double>::fd(u, f, d);
            dr += f * g;
            const double delta = d * g * rv;
            db += delta;
            dwi[centre] = delta;
            const double mean = NORM ? stat[3 * it] : 0.0, inv = NORM ? stat[3 * it + 2] : 1.0;
            d1 += inv * delta;
            if (NORM) d2 += mean * inv * delta;
            lds_barrier();
            const double z = NORM ? (xi - mean) * inv : xi;
            double part[3] = {0.0, 0.0, 0.0};
            const auto gather = [&](auto finite) {
                const unsigned in = decltype(finite)::value ? 0u : now(stays);
#pragma unroll
                for (int t = 0; t < 27; ++t) {
                    const double dn = dwi[G::tap(base, t)];
                    part[t / 9] += v[t] * dn;
                    dw[t] += decltype(finite)::value || (in >> t & 1) ? z * dn : 0.0;
                }
            };
            // the zero of a neighbour that is not there times infinity must not reach the other gradient
            // that dw[t] holds; tested for all lanes at once, since the selects cost as much as the sum
            if (__any(!__builtin_isfinite(z))) gather(std::false_type{});
            else gather(std::true_type{});
            const double dz = (part[0] + part[1]) + part[2];
            if (NORM) {
                double sums[2] = {dz + delta * wh, dz * (xi - mean) + delta * (sh - mean * wh)};
                sum_all<G::NT>(sums, red + (it & 1) * 2 * kWaveRed, tid);
                const double mdz = sums[0] / G::W, sd = stat[3 * it + 1], tiny = 1e-30;
                const double coef = sums[1] * inv * inv / (G::W * (sd > tiny ? sd : tiny));
                g += inv * (dz - mdz) - coef * (xi - mean);
                q += coef;
                r += coef * mean - inv * mdz;
            } else {
                g += dz;
            }
        }

        // the taps that leave the block: the gradients of their weights
        {
            const unsigned in = now(stays);
#pragma unroll
            for (int t = 0; t < 27; ++t) {
                const double h = win[G::tap(base, t)];
                const double p = NORM ? h * d1 - d2 : h * d1;
                dw[t] += in >> t & 1 ? 0.0 : p;
            }
        }
        double *to = dx + s * cells + gc;
        *to = add_dx ? *to + g : g;
        dsum[s * cells + gc] = d1;
        if (NORM && tid == 0) {
            halo_part[((long)s * nblk + blk) * 2] = q;
            halo_part[((long)s * nblk + blk) * 2 + 1] = r;
        }
    }

    // dw[t] is the gradient of the neighbour's mirrored weight where that neighbour is in the block, of
    // the cell's own otherwise: every weight of the block in exactly one thread
    const auto commit = [&](double *to, double sum) {
        to += chunk * copy_stride;
        *to = add_params ? *to + sum : sum;
    };
#pragma unroll
    for (int t = 0; t < 27; ++t) {
        const bool in = stays >> t & 1;
        commit(dweight + (in ? 26 - t : t) * cells + gc + (in ? ((t / 9 - 1) * N + t / 3 % 3 - 1) * K + t % 3 - 1 : 0),
               dw[t]);
    }
    commit(dbias + gc, db);
    commit(dscale + gc, dr);
}


// What the cells of other blocks owe a cell: dx[c] += sum over the taps t that leave c's block of
// W[26-t, c+off_t] D[c+off_t], and with normalisation R - x[c] Q, x less the shift, of every block that has c in its halo.  A
// thread per cell and batch element, for the cells some tap of which leaves the block.  The workgroups behind
// those add up the copies of the parameter gradients.  Four waves per SIMD for their sake: with the weights
// in registers for several elements (two waves) the kernel took 13.2 us at 24 x 32 x 32, batch 6, now 8.3.
struct CrossF64 {
    const double *weight, *x, *dsum, *halo_part, *copies;
    double *dx, *params[3];
    int B, M, N, K, nblk, ncopies, cell_blocks, add_params;
};

template <int BS, bool NORM> __global__ __launch_bounds__(256, 4) void step_cross_f64(CrossF64 a) {
    const int cells = a.M * a.N * a.K, cell_groups = a.cell_blocks * a.B;
    if ((int)blockIdx.x >= cell_groups) {
        // two at a time: 29 * cells is a multiple of 64
        const long total = 29L * cells, step = (long)(gridDim.x - cell_groups) * 512;
        for (long i = ((long)(blockIdx.x - cell_groups) * 256 + threadIdx.x) * 2; i < total; i += step) {
            double2 sum = make_double2(0.0, 0.0);
#pragma unroll 4
            for (int n = 0; n < a.ncopies; ++n) {
                const double2 v = *reinterpret_cast<const double2 *>(a.copies + n * total + i);
                sum.x += v.x;
                sum.y += v.y;
            }
            double *to = i < 27L * cells ? a.params[0] + i
                                         : i < 28L * cells ? a.params[1] + (i - 27L * cells)
                                                           : a.params[2] + (i - 28L * cells);
            to[0] = a.add_params ? to[0] + sum.x : sum.x;
            to[1] = a.add_params ? to[1] + sum.y : sum.y;
        }
        return;
    }
    const int c = (blockIdx.x % a.cell_blocks) * 256 + threadIdx.x, s = blockIdx.x / a.cell_blocks;
    if (c >= cells) return;
    const int k = c % a.K, j = c / a.K % a.N, i = c / (a.K * a.N);
    // per axis, a bit per step by -1, 0, +1: it stays in the grid; it stays in the grid and leaves the block
    unsigned in[3] = {}, leaves[3] = {};
    const int at[3] = {i, j, k}, side[3] = {a.M, a.N, a.K};
#pragma unroll
    for (int axis = 0; axis < 3; ++axis)
#pragma unroll
        for (int o = -1; o <= 1; ++o) {
            const int to = at[axis] + o;
            if (to < 0 || to >= side[axis]) continue;
            in[axis] |= 1u << (o + 1);
            if (to / BS != at[axis] / BS) leaves[axis] |= 1u << (o + 1);
        }
    if (!(leaves[0] | leaves[1] | leaves[2])) return;
    const double *d = a.dsum + (long)s * cells + c, *w = a.weight + c;
    double *to = a.dx + (long)s * cells + c, sum = *to;
    double x = 0.0;
    if (NORM) x = a.x[(long)s * cells + c];
#pragma unroll
    for (int t = 0; t < 27; ++t) {
        const int oi = t / 9, oj = t / 3 % 3, ok = t % 3;
        const bool there = (in[0] >> oi & 1) && (in[1] >> oj & 1) && (in[2] >> ok & 1);
        const bool out = (leaves[0] >> oi & 1) || (leaves[1] >> oj & 1) || (leaves[2] >> ok & 1);
        const int off = there && out ? ((oi - 1) * a.N + oj - 1) * a.K + ok - 1 : 0;
        const double p = w[(long)(26 - t) * cells + off] * d[off];
        sum += there && out ? p : 0.0;
    }
    if (NORM) {
        const int kb = a.K / BS, nb = a.N / BS;
        // the blocks on the side of every combination of axes along which a step leaves the block
#pragma unroll
        for (int mask = 1; mask < 8; ++mask) {
            int b[3];
            bool there = true;
#pragma unroll
            for (int axis = 0; axis < 3; ++axis) {
                const bool moves = mask >> axis & 1;
                there = there && (!moves || leaves[axis]);
                b[axis] = at[axis] / BS + (moves ? (leaves[axis] & 1 ? -1 : 1) : 0);
            }
            if (there) {
                const double *qr = a.halo_part + ((long)s * a.nblk + ((long)b[0] * nb + b[1]) * kb + b[2]) * 2;
                const long first = (((long)b[0] * a.N + b[1]) * a.K + b[2]) * BS;  // of block b
                sum += qr[1] - (x - shift_of(a.x[(long)s * cells + first])) * qr[0];
            }
        }
    }
    *to = sum;
}

int blocks_of(const StepArgs &a) { return (a.M / a.block_size) * (a.N / a.block_size) * (a.K / a.block_size); }
size_t round256(size_t n) { return (n + 255) / 256 * 256; }
size_t dsum_bytes(const StepArgs &a) { return round256((size_t)a.B * a.M * a.N * a.K * sizeof(double)); }
size_t halo_bytes(const StepArgs &a) { return a.normalize ? round256((size_t)a.B * blocks_of(a) * 2 * sizeof(double)) : 0; }
size_t copy_doubles(const StepArgs &a) { return 29 * (size_t)a.M * a.N * a.K; }

// How the batch is split: a workgroup fetches and leaves parameters for about as long as it works on one
// element (9 and 10 us at three inner iterations), and the CUs hold `resident` workgroups at once.  Fewer
// chunks where the rounds come to the same.
int plan_chunks(int B, int nblk, int resident, int most) {
    int best = 1;
    long least = -1;
    for (int n = 1; n <= B && n <= most; ++n) {
        const int len = (B + n - 1) / n, m = (B + len - 1) / len;
        const long cost = (((long)nblk * m + resident - 1) / resident) * (len + 1);
        if (least < 0 || cost < least) least = cost, best = m;
        if ((long)nblk * n > 4L * resident) break;
    }
    return best;
}
// resident workgroups per CU: one of eight waves, eight of one wave (two waves per SIMD; the LDS of the
// deepest history leaves room for two)
int resident_f64(const StepArgs &a) {
    if (a.block_size == 8) return plan_device_cus();
    const size_t fit = kF64MaxLds / bwd_f64_lds<4>(a.inner);
    return plan_device_cus() * (int)(fit > 8 ? 8 : fit);
}

// The forward keeps no copy per chunk: workgroups for the chip a few times over
template <int BS, int ACT, bool NORM> int launch_fwd_f64(const StepArgs &a, hipStream_t st) {
    const int nblk = blocks_of(a);
    int nchunk = (4 * plan_device_cus() + nblk - 1) / nblk;
    if (nchunk > a.B) nchunk = a.B;
    const int chunk_len = (a.B + nchunk - 1) / nchunk;
    nchunk = (a.B + chunk_len - 1) / chunk_len;
    hipLaunchKernelGGL((step_fwd_f64<BS, ACT, NORM>), dim3(padded_grid(nblk, nchunk)), dim3(Geo<BS>::NT), 0, st,
                       (const double *)a.weight, (const double *)a.bias, (const double *)a.scale, (const double *)a.x,
                       (double *)a.y, a.B, a.M, a.N, a.K, a.inner, a.eps, nblk, nchunk, chunk_len);
    return check_launch("step_fwd_f64");
}

template <int BS, int ACT, bool NORM> int launch_bwd_f64(const StepArgs &a, hipStream_t st) {
    auto kern = step_bwd_f64<BS, ACT, NORM>;
    const size_t lds = bwd_f64_lds<BS>(a.inner);
    static bool enabled = false;  // per instantiation
    if (lds > 64 * 1024 && !enabled) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kF64MaxLds);
        if (e != hipSuccess)
            return fail(GRIDNET_ERR_LAUNCH, "cannot enable %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        enabled = true;
    }
    const int nblk = blocks_of(a);
    const long cells = (long)a.M * a.N * a.K;
    const size_t room = a.slabs ? a.slab_bytes / (copy_doubles(a) * sizeof(double)) : 0;
    const int nchunk = plan_chunks(a.B, nblk, resident_f64(a), room > 1 ? (int)(room > 65535 ? 65535 : room) : 1);
    const int chunk_len = (a.B + nchunk - 1) / nchunk;
    const bool split = nchunk > 1, add_params = !(a.flags & GRIDNET_OVERWRITE_PARAMS);
    double *dsum = (double *)a.workspace, *part = (double *)((char *)a.workspace + dsum_bytes(a));
    double *copies = (double *)a.slabs;
    double *dw = split ? copies : (double *)a.dweight;
    double *db = split ? copies + 27 * cells : (double *)a.dbias, *dr = split ? copies + 28 * cells : (double *)a.dscale;
    hipLaunchKernelGGL(kern, dim3(padded_grid(nblk, nchunk)), dim3(Geo<BS>::NT), lds, st, (const double *)a.weight,
                       (const double *)a.bias, (const double *)a.scale, (const double *)a.x, (const double *)a.dy, dw,
                       db, dr, (double *)a.dx, dsum, part, a.B, a.M, a.N, a.K, a.inner, a.eps, nblk, nchunk, chunk_len,
                       !(a.flags & GRIDNET_OVERWRITE_DX), !split && add_params, split ? (long)copy_doubles(a) : 0L);
    CrossF64 c{};
    c.weight = (const double *)a.weight; c.x = (const double *)a.x; c.dsum = dsum; c.halo_part = part; c.copies = copies;
    c.dx = (double *)a.dx;
    c.params[0] = (double *)a.dweight; c.params[1] = (double *)a.dbias; c.params[2] = (double *)a.dscale;
    c.B = a.B; c.M = a.M; c.N = a.N; c.K = a.K; c.nblk = nblk; c.ncopies = nchunk; c.add_params = add_params;
    c.cell_blocks = (int)((cells + 255) / 256);
    const long sums = split ? (29 * cells + 511) / 512 : 0;
    const long grid = (long)c.cell_blocks * a.B + (sums > 2048 ? 2048 : sums);
    hipLaunchKernelGGL((step_cross_f64<BS, NORM>), dim3((unsigned)grid), dim3(256), 0, st, c);
    return check_launch("step_bwd_f64");
}

template <int BS, bool BWD, bool NORM> int dispatch_f64(const StepArgs &a, hipStream_t st) {
#define GRIDNET_CASE(ID)                                          \
    case ID:                                                      \
        if (BWD) return launch_bwd_f64<BS, ID, NORM>(a, st);      \
        return launch_fwd_f64<BS, ID, NORM>(a, st);
    switch (a.activation) {
        GRIDNET_CASE(GRIDNET_ACT_RELU)
        GRIDNET_CASE(GRIDNET_ACT_LEAKY_RELU)
        GRIDNET_CASE(GRIDNET_ACT_SILU)
        GRIDNET_CASE(GRIDNET_ACT_TANH)
    }
#undef GRIDNET_CASE
    return fail(GRIDNET_ERR_ACTIVATION, "unknown activation function: %d", a.activation);
}

}  // namespace

// Where the scattering kernel would split the batch of a block, and add the parameter gradients by atomics:
// batches of two and more, fewer than 1024 blocks.  Elsewhere its one launch less decides.  Backward there / here
// (two inner iterations; three with normalize), 40^3, batch 4, 8^3 blocks: 82 / 47 and 106 / 69 us; 4^3 blocks:
// 78 / 50 and 91 / 67; 48^3 in 4^3 blocks (1728 of them): 56 / 62 and 86 / 114; 40^3, batch 1: 21 / 22 and 33 / 33,
// 4^3 blocks 19 / 22 and 26 / 26.  Up to 2^17 cells: gridnet_hip_backward has asked callers with larger fp64
// grids for no scratch.  No iteration at all, and histories beyond LDS (more than 15 iterations of 8^3 blocks), stay there too.
// Size queries come here with arguments that nothing has looked at: what the sums below cannot take is refused first.
bool step_f64_supports(const StepArgs &a) {
    if (a.dtype != GRIDNET_F64 || (a.block_size != 4 && a.block_size != 8) || a.inner < 1 || a.inner > kMaxBackwardIters)
        return false;
    return a.B >= 2 && a.M <= 1 << 17 && a.N <= 1 << 17 && (long)a.M * a.N <= 1L << 17 &&
           (long)a.M * a.N * a.K <= 1L << 17 && blocks_of(a) < 1024 &&
           (a.block_size == 8 ? bwd_f64_lds<8>(a.inner) : bwd_f64_lds<4>(a.inner)) <= kF64MaxLds;
}
size_t step_f64_workspace(const StepArgs &a) { return dsum_bytes(a) + halo_bytes(a); }
size_t step_f64_slab_bytes(const StepArgs &a) {
    const int n = plan_chunks(a.B, blocks_of(a), resident_f64(a), a.B);
    return n > 1 ? n * copy_doubles(a) * sizeof(double) : 0;
}
int step_forward_f64(const StepArgs &a, hipStream_t st) {
    if (a.block_size == 8) return a.normalize ? dispatch_f64<8, false, true>(a, st) : dispatch_f64<8, false, false>(a, st);
    return a.normalize ? dispatch_f64<4, false, true>(a, st) : dispatch_f64<4, false, false>(a, st);
}
int step_backward_f64(const StepArgs &a, hipStream_t st) {
    if (a.block_size == 8) return a.normalize ? dispatch_f64<8, true, true>(a, st) : dispatch_f64<8, true, false>(a, st);
    return a.normalize ? dispatch_f64<4, true, true>(a, st) : dispatch_f64<4, true, false>(a, st);
}

}  // namespace gridnet
