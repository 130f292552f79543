// The steps of a chain with 4^3 blocks: four samples of a block to a wave.  The algorithm is that of step_fast.hip (the
// halo is frozen, so what reads or leaves it needs only sums over the iterations); this file deals it differently.
//
// A row of a 4^3 block is four cells: a wave's 64 lanes are the block's 16 rows times four, and the entries of a neighbour
// row in one sample are one aligned 16-byte access.  A wave has its block to itself, so no iteration waits for another wave.
// The two entries beyond the ends of a row (k = -1 and 4) are halo whatever the row: what they add to the pre-activations
// is worked out once per sample, nothing but the row's four entries is read in an iteration.
//
// Forward (quads_fwd): lane (row, sample) has the row's 108 weights and does 90 multiply-adds for its four cells in an
// iteration, where step_fwd_fast does 108 and reads twice as much from LDS.  It is bound by the vector ALU: 102 instructions of a
// loop of 112.  A step of 64^3, batch 128, eight iterations, leaky_relu: 395 -> 243 us under the
// profiler, 392 -> 246 from a graph with the statistics.
//
// Backward (quads_bwd): there are no registers for that three times over (weights, mirrored weights and gradients).  The
// fp32 matrix instruction v_mfma_f32_4x4x1_16b does what a row sends to a row for four samples at once, sixteen products of
// a column and a row of four, one for each row of the block: entry by entry one fused multiply-add, bit for bit that of fmaf.  A
// row of weights is then in four lanes once instead of in every lane: 45 registers for the weights.  Nine neighbour rows of
// four entries are 36 instructions; the band (cell k reads entries k - 1, k, k + 1) fills ten of sixteen places, the rest multiplies
// zeros.  They run on the vector ALU's multipliers, not beside them (8 cycles each, to which a multiply-add of another wave
// adds its own), so an iteration's 108 there and back cost what the 324 multiply-adds they stand for do; what they save is half of
// the LDS traffic, half of the other instructions and all of the registers that step_bwd_fast spills in its loops.  The same step under the
// profiler: 1057 -> 875 us (903 on another box).  What bounds it: the vector ALU, by counters 44 % of the time in matrix and 18 % in
// other instructions; two waves per SIMD do not fill the waits between dependent matrix instructions; and a clock of 2.0 to 2.2 GHz.
//
// A wave's registers come in two layouts there:
//   by cell:   lane (row, k), one register per sample -- what the matrix instruction leaves when the window is its
//              first operand; bias, scale and the small gradients are one register each;
//   by sample: lane (row, sample), one register per cell of the row -- its first operand, read from LDS.
//
// In front of a LayerNorm only: the backward's zeros of the band, and of rows that are not the block's, multiply values of the same
// sample, and an infinity or a NaN there spreads to cells that do not read it.  A LayerNorm behind the step spreads what the output or
// its gradient hold of that kind over the whole sample anyway; a step on its own and the last one of the residual loop, which is
// handed its gradient as it is, keep it within the taps' reach and go to step_bwd_fast.  What is left is a gradient that overflows
// inside the sweep (or meets an infinite weight whose cell's activation is saturated): the gradients of this step's own parameters then
// are NaN in more of the block's cells than that; those of all earlier steps are for the whole sample either way.

#include <type_traits>

#include "common.h"
#include "fast_tiles.h"
#include "launch.h"
#include "plan.h"

namespace gridnet {

namespace {

typedef float quad __attribute__((ext_vector_type(4)));

constexpr int kGroup = 4;           // samples to a wave
constexpr int kWaves = 4;           // to a workgroup: neighbouring blocks of a K-row, the same samples
constexpr int kThreads = kWaves * kWave;
constexpr int kWinRows = 36;        // rows of a window, 6 x 6
// Floats of a wave's LDS.  Rows by sample, [36][4 samples][4 cells]; the floats between planes spread the backward's
// 4-byte writes by cell, or the forward's 16-byte writes, over all banks.  The entries beyond the rows' ends, [36][2][4 samples].
constexpr int kPlaneBackward = 6 * 16 + 4, kPlaneForward = 6 * 16 + 16, kSides = kWinRows * 8;
constexpr int rows_floats(int plane) { return 6 * plane; }
constexpr int window_floats(int plane) { return rows_floats(plane) + kSides; }
// the four waves' windows: 16 floats past a multiple of 64, so that the pieces of a row, one for each wave, go to different banks
constexpr int kForwardFloats = window_floats(kPlaneForward) + 16;
// The residual form, forward: h and n = LayerNorm(h) of a block's own cells, [2][row][sample][cell], for h + (result - n).  In registers
// (h requested with the window, a second time) they made 7 to 12 of them spill: 64^3, batch 128, eight iterations, 295 -> 275 us, with silu 380 -> 335.
constexpr int kBack = 512;
// gamma and beta of the workgroup's rows and of the entries beyond their ends
constexpr int kAffineRows = kWinRows * kWaves * 8, kAffine = kAffineRows + kWinRows * 4;
// Deltas by cell, [row][4 cells][4 samples], zeros around the block: row (i, j) is number 5 (i + 1) + j + 1, the row behind
// a plane's last is the one in front of the next plane's first.
constexpr int kDeltaPlane = 5 * 16, kDeltas = 6 * kDeltaPlane + 16;
constexpr int kExchange = 27 * 64 + 16;  // the weights, once at set-up
// history: u of all iterations but the last, x of those between (the first and the last stay in registers)
__host__ __device__ constexpr int history_floats(int inner) {
    return 256 * ((inner > 1 ? inner - 1 : 0) + (inner > 2 ? inner - 2 : 0));
}
__host__ __device__ constexpr int backward_floats(int inner) {
    const int run = window_floats(kPlaneBackward) + kDeltas + 40 + history_floats(inner);  // 16 past a multiple of 64, too
    return run > kExchange ? run : kExchange;
}

__device__ __forceinline__ quad mfma(float a, float b, quad c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ quad load_quad(const float *p) { return *reinterpret_cast<const quad *>(p); }
// value of lane 4 * (lane / 4) + S
template <int S> __device__ __forceinline__ float of_sample(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), S * 0x55, 0xf, 0xf, true));
}
template <typename F> __device__ __forceinline__ void for_samples(F &&f) {
    f(std::integral_constant<int, 0>());
    f(std::integral_constant<int, 1>());
    f(std::integral_constant<int, 2>());
    f(std::integral_constant<int, 3>());
}
// An offset that the compiler cannot see through: added to a uniform base where it is used (an addressing mode), instead of
// to every base in front of the loop (a pair of registers each).
__device__ __forceinline__ unsigned opaque(unsigned at) {
    asm volatile("" : "+v"(at));
    return at;
}
// p[cell], the lane's cell
__device__ __forceinline__ const float *at_cell(const float *p, int cell) {
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + opaque(4u * (unsigned)cell));
}
__device__ __forceinline__ float *at_cell(float *p, int cell) {
    return reinterpret_cast<float *>(reinterpret_cast<char *>(p) + opaque(4u * (unsigned)cell));
}
// orders a wave's LDS accesses for the compiler; the LDS itself serves a wave in order
__device__ __forceinline__ void wave_order() { slot_barrier<kWave>(); }

// What a workgroup and a wave of it work on: up to four neighbouring blocks of a K-row, a chunk of the batch.
struct QuadWork {
    int p0, q0, r0, blocks;  // the first block's origin, the number of blocks
    int chunk, first, end;   // samples
    int wave, blk;           // of the calling wave (past the last block: the last one again)
    bool active;
    __device__ __forceinline__ bool find(int wg, int M, int N, int K, int nchunk, int chunk_len, int B) {
        const int kb = K / 4, nb = N / 4, per_row = (kb + kWaves - 1) / kWaves;
        int group;
        if (!split_block_id(wg, M / 4 * nb * per_row, nchunk, group, chunk)) return false;
        const int line = group / per_row, k0 = group % per_row * kWaves;
        p0 = line / nb * 4;
        q0 = line % nb * 4;
        r0 = 4 * k0;
        blocks = min(kWaves, kb - k0);
        first = chunk * chunk_len;
        end = min(B, first + chunk_len);
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        active = wave < blocks;
        blk = line * kb + k0 + min(wave, blocks - 1);
        return true;
    }
};

// Where a lane sits in its wave's block.  The LDS serves a 16-byte read sixteen lanes at a time: lanes 0-3, 12-15, 20-23
// and 24-27 together, then the others of the lower half wave, and so on.  Those are given the four rows of a plane, which lie side by
// side.  With row = lane / 4 they came from two planes, and every read took eight cycles instead of four (counted): the LDS was
// busy for 70 % of the forward and 61 % of the backward, four tenths of it with conflicts.  Now 45 and 40 %, and a step of 64^3, batch
// 128, eight iterations is 1 to 4 % faster forward and 1 % backward: the vector ALU and its clock bind it, not the LDS.
template <int PLANE> struct QuadPlace {
    int lane, row, k;        // k is the cell or the sample
    int i, j;                // of the row in the block
    int own;                 // cell (row, k) in the grid
    int rows00, cell;        // LDS: window row (i, j) by sample k; cell (row, k) of the first sample
    int sides00;             // LDS: the end of window row (i, j) on the side of cell k, first sample
    __device__ __forceinline__ QuadPlace(const QuadWork &work, int N, int K) {
        lane = threadIdx.x & (kWave - 1);
        const int quad = lane >> 2;
        k = lane & 3;
        i = quad >> 3 << 1 | (__popc(quad & 7) & 1);
        j = quad >> 1 & 3;
        row = 4 * i + j;
        own = ((work.p0 + i) * N + work.q0 + j) * K + work.r0 + 4 * min(work.wave, work.blocks - 1) + k;
        rows00 = i * PLANE + j * 16 + 4 * k;
        cell = (i + 1) * PLANE + (j + 1) * 16 + k;
        sides00 = rows_floats(PLANE) + (i * 6 + j) * 8 + (k >> 1) * 4;
    }
    __device__ __forceinline__ bool has(int a, int c) const {  // the block has row (i + a - 1, j + c - 1)
        return (unsigned)(i + a - 1) < 4u && (unsigned)(j + c - 1) < 4u;
    }
};

// The windows of four samples, fetched by the whole workgroup: 36 rows of up to 16 cells, four lanes to a row (a wave
// that fetched its own block's pieces of 16 bytes asked the L2 for every line four times: 2.2 GB for a forward at 64^3, batch 128, 
// in which 0.13 GB are read), and one entry beyond either end.  What lies outside the grid, and threads
// without a row, read the first block's own first row and count as zero.
struct QuadFetch {
    struct Buf { quad rows[3]; float ends[2]; };
    unsigned at[5];  // byte offsets in a sample, three rows and two ends; bit 0: inside the grid
    int blocks;
    // thread = 16 row + 4 sample + block; for the ends block = 2 (row & 1) + side
    static __device__ __forceinline__ int sample() { return threadIdx.x >> 2 & 3; }
    __device__ __forceinline__ QuadFetch(const QuadWork &work, int M, int N, int K) : blocks(work.blocks) {
        const int t = threadIdx.x, m = t & 3, side = t & 1;
#pragma unroll
        for (int e = 0; e < 5; ++e) {
            const int r = e < 3 ? e * 16 + (t >> 4) : (e - 3) * 32 + (t >> 4) * 2 + (t >> 1 & 1);
            const int gi = work.p0 + r / 6 - 1, gj = work.q0 + r % 6 - 1;
            const int col = e < 3 ? work.r0 + 4 * m : side ? work.r0 + 4 * work.blocks : work.r0 - 1;
            const bool ok = r < kWinRows && (unsigned)gi < (unsigned)M && (unsigned)gj < (unsigned)N && (unsigned)col < (unsigned)K &&
                            (e >= 3 || m < work.blocks);
            at[e] = 4u * (unsigned)(ok ? (gi * N + gj) * K + col : (work.p0 * N + work.q0) * K + work.r0) | (ok ? 1u : 0u);
        }
    }
    // `lane_at`: byte offset of the thread's sample
    __device__ __forceinline__ void fetch(const float *x, unsigned lane_at, Buf &v) const {
        const char *base = reinterpret_cast<const char *>(x);
#pragma unroll
        for (int e = 0; e < 3; ++e) v.rows[e] = load_quad(reinterpret_cast<const float *>(base + opaque(lane_at + (at[e] & ~1u))));
#pragma unroll
        for (int e = 0; e < 2; ++e) v.ends[e] = *reinterpret_cast<const float *>(base + opaque(lane_at + (at[3 + e] & ~1u)));
    }
    // gamma and beta of the windows, as fetched with lane_at 0
    __device__ __forceinline__ void pack_affine(float *to, const Buf &g, const Buf &b) const {
        if (sample() == 0) {
            const int t = threadIdx.x, m = t & 3;
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const int r = e * 16 + (t >> 4);
                if (r < kWinRows) {
                    *reinterpret_cast<quad *>(to + (r * kWaves + m) * 8) = g.rows[e];
                    *reinterpret_cast<quad *>(to + (r * kWaves + m) * 8 + 4) = b.rows[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int r2 = (e * 32 + (t >> 4) * 2) * 2 + m;  // 2 * row + side
                if (r2 < 2 * kWinRows)
                    *reinterpret_cast<float2 *>(to + kAffineRows + r2 * 2) = make_float2(g.ends[e], b.ends[e]);
            }
        }
    }
    // Into the windows, `stride` floats apart: a row's four cells to their block, its first and last to the blocks beside it.
    // LN: normalised on the way, with the statistics of the thread's sample.  The LDS places are worked out here, from a thread
    // number that the compiler cannot see through: it would keep them in registers that the loops have no room for.
    // An end goes to [row][side][sample], in the forward to [row][sample][side].
    // BACK: the blocks' own cells, as they are and normalised, to back[block][2][row][sample][cell].
    template <bool LN, int PLANE, bool BACK = false>
    __device__ __forceinline__ void commit(float *windows, int stride, const Buf &v, const float *affine, float mean,
                                           float rstd, float *back = nullptr) const {
        constexpr int SIDE = PLANE == kPlaneForward ? 1 : 4, SAMPLE = PLANE == kPlaneForward ? 2 : 1;
        const int t = opaque(threadIdx.x), m = t & 3, s = t >> 2 & 3;
        float *win = windows + m * stride;
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            const int r = e * 16 + (t >> 4);
            if (e < 2 || t < 64) {
                const unsigned where = opaque(at[e]);
                quad val = v.rows[e];
                if (LN) {
                    const float *gb = affine + (r * kWaves + m) * 8;
                    const quad g = load_quad(gb), b = load_quad(gb + 4);
#pragma unroll
                    for (int q = 0; q < 4; ++q) val[q] = fmaf((val[q] - mean) * rstd, g[q], b[q]);
                }
                if (BACK) {
                    const int i = r / 6 - 1, j = r % 6 - 1;
                    if ((unsigned)i < 4u && (unsigned)j < 4u) {
                        float *to = back + m * kBack + (4 * i + j) * 16 + s * 4;
                        *reinterpret_cast<quad *>(to) = v.rows[e];
                        *reinterpret_cast<quad *>(to + 256) = val;
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) val[q] = where & 1 ? val[q] : 0.f;
                *reinterpret_cast<quad *>(win + r * 16 + r / 6 * (PLANE - 96) + s * 4) = val;
                float *sides = win + rows_floats(PLANE) + r * 8 + s * SAMPLE;
                if (m > 0 && m < blocks) sides[SIDE - stride] = val[0];
                if (m < kWaves - 1) sides[stride] = val[3];
            }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            if (e < 1 || t < 32) {
                const unsigned where = opaque(at[3 + e]);
                const int r2 = (e * 32 + (t >> 4) * 2) * 2 + m, side = m & 1;
                float val = v.ends[e];
                if (LN) {
                    const float2 gb = *reinterpret_cast<const float2 *>(affine + kAffineRows + r2 * 2);
                    val = fmaf((val - mean) * rstd, gb.x, gb.y);
                }
                const int r = e * 32 + (t >> 4) * 2 + (t >> 1 & 1);
                windows[(side ? blocks - 1 : 0) * stride + rows_floats(PLANE) + r * 8 + side * SIDE + s * SAMPLE] = where & 1 ? val : 0.f;
            }
        }
    }
};

// A cell's 27 weights as the bands of its row: W[n][h] what entry h of neighbour row n is multiplied with (zero where it
// is no neighbour), S[n] the same for the entry beyond the row's end that the cell reads (cells 0 and 3).
struct Bands {
    float w[9][4], s[9];
    __device__ __forceinline__ void take(const float *weight, long cells, int own, int k) {
#pragma unroll
        for (int n = 0; n < 9; ++n) {
            const float before = weight[(3 * n) * cells + own], at = weight[(3 * n + 1) * cells + own],
                        after = weight[(3 * n + 2) * cells + own];
#pragma unroll
            for (int h = 0; h < 4; ++h) w[n][h] = k == h ? at : k == h + 1 ? before : k == h - 1 ? after : 0.f;
            s[n] = k == 0 ? before : k == 3 ? after : 0.f;
            keep_here<4>(w[n]);
        }
        keep_here<9>(s);
    }
};

// bias and what the entries beyond the rows' ends add, by cell: the same for every iteration
__device__ __forceinline__ quad side_sums(const float *win, const QuadPlace<kPlaneBackward> &pl, const Bands &w, float bias) {
    quad u = {bias, bias, bias, bias};
#pragma unroll
    for (int n = 0; n < 9; ++n) {
        const quad v = load_quad(win + pl.sides00 + (n / 3 * 6 + n % 3) * 8);
#pragma unroll
        for (int s = 0; s < 4; ++s) u[s] = fmaf(w.s[n], v[s], u[s]);
        if (n % 3 == 2) __builtin_amdgcn_sched_barrier(0);  // not all requested at once: registers
    }
    return u;
}

// u += the 27 taps but for the rows' ends, by cell, DEPTH rows requested ahead of the arithmetic.
template <int DEPTH>
__device__ __forceinline__ quad band_sums(const float *win, const QuadPlace<kPlaneBackward> &pl, const float (&w)[9][4], quad u) {
    quad v[DEPTH];
    const auto row = [&](int n) { return load_quad(win + pl.rows00 + n / 3 * kPlaneBackward + n % 3 * 16); };
#pragma unroll
    for (int n = 0; n < DEPTH; ++n) v[n] = row(n);
#pragma unroll
    for (int n = 0; n < 9; ++n) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 4; ++h) u = mfma(v[n % DEPTH][h], w[n][h], u);
        __builtin_amdgcn_sched_barrier(0);
        if (n + DEPTH < 9) v[n % DEPTH] = row(n + DEPTH);
    }
    return u;
}

// Lane (row, sample), four cells.  Three waves per SIMD; the 18 weights that read beyond the row's ends wait in LDS.
template <int ACT, bool RES>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3)))
void quads_fwd(const float *__restrict__ weight, const float *__restrict__ bias, const float *__restrict__ scale,
               const float *__restrict__ x, float *__restrict__ y, int B, int M, int N, int K, int inner, int nblk,
               int nchunk, int chunk_len, LnFold ln) {
    constexpr int PLANE = kPlaneForward, WINDOW = kForwardFloats;
    constexpr int SIDE_WEIGHTS = 16 * 18;  // [row][neighbour row][side]
    __shared__ __attribute__((aligned(16))) float lds[kWaves * (WINDOW + SIDE_WEIGHTS + (RES ? kBack : 0)) + kAffine];
    QuadWork work;
    if (!work.find(ln.walk_reverse ? reversed_on_its_xcd(blockIdx.x, gridDim.x) : blockIdx.x, M, N, K, nchunk, chunk_len, B))
        return;
    const QuadPlace<PLANE> pl(work, N, K);
    const QuadFetch fx(work, M, N, K);
    float *win = lds + work.wave * WINDOW, *affine = lds + kWaves * WINDOW;
    float *ends = affine + kAffine + work.wave * SIDE_WEIGHTS + pl.row * 18;
    float *back = affine + kAffine + kWaves * SIDE_WEIGHTS;
    const long cells = (long)M * N * K;
    const bool ln_in = ln.x_stats != nullptr;
    const int first = pl.own - pl.k;  // cell 0 of the lane's row; pl.k is the lane's sample

    quad w[27];
#pragma unroll
    for (int t = 0; t < 27; ++t) w[t] = load_quad(weight + t * cells + first);
    const quad bv = load_quad(bias + first), rv = load_quad(scale + first);
    if (pl.k == 0) {
#pragma unroll
        for (int n = 0; n < 9; ++n) *reinterpret_cast<float2 *>(ends + 2 * n) = make_float2(w[3 * n][0], w[3 * n + 2][3]);
    }
    QuadFetch::Buf pre;
    float mean = 0.f, rstd = 1.f;
    if (ln_in) {
        QuadFetch::Buf beta;
        fx.fetch(ln.gamma, 0, pre);
        fx.fetch(ln.beta, 0, beta);
        fx.pack_affine(affine, pre, beta);
    }
    wait_global_loads();
    auto fetch_group = [&](int s) {
        const int mine = min(s + fx.sample(), work.end - 1) - s;  // past the end: the last sample again
        fx.fetch(x + s * cells, 4u * (unsigned)mine * (unsigned)cells, pre);
        if (ln_in) {
            const float2 st = *reinterpret_cast<const float2 *>(ln.x_stats + 2 * (s + mine));
            mean = st.x;
            rstd = st.y;
        }
    };
    fetch_group(work.first);
    quad cur, stored = {0.f, 0.f, 0.f, 0.f};
    int done = -1;  // the first of the samples in `stored`: a group's result leaves behind the wait for the next one's window
    const auto store_group = [&] {
        if (done >= 0 && done + pl.k < work.end)
            *reinterpret_cast<quad *>(at_cell(y + done * cells, pl.k * (int)cells + first)) = stored;
    };
    for (int s = work.first; s < work.end; s += kGroup) {
        lds_barrier();  // gamma and beta; the windows are free
        if (RES) fx.template commit<true, PLANE, true>(lds, WINDOW, pre, affine, mean, rstd, back);  // with statistics always
        else if (ln_in) fx.template commit<true, PLANE>(lds, WINDOW, pre, affine, mean, rstd);
        else fx.template commit<false, PLANE>(lds, WINDOW, pre, affine, mean, rstd);
        lds_barrier();
        if (work.active) store_group();
        if (s + kGroup < work.end) fetch_group(s + kGroup);
        if (!work.active) continue;
        float *own = win + pl.rows00 + PLANE + 16;
        cur = load_quad(own);
        quad u0 = bv;
#pragma unroll
        for (int n = 0; n < 9; ++n) {  // the entries beyond the row's ends: the same for every iteration
            const float2 v = *reinterpret_cast<const float2 *>(win + rows_floats(PLANE) + (pl.i * 6 + pl.j) * 8 + 2 * pl.k + (n / 3 * 6 + n % 3) * 8);
            const float2 e = *reinterpret_cast<const float2 *>(ends + 2 * n);
            u0[0] = fmaf(e.x, v.x, u0[0]);
            u0[3] = fmaf(e.y, v.y, u0[3]);
        }
        for (int it = 0; it < inner; ++it) {
            constexpr int DEPTH = 5;
            quad u = u0, v[DEPTH];
            const auto row = [&](int n) { return load_quad(win + pl.rows00 + n / 3 * PLANE + n % 3 * 16); };
#pragma unroll
            for (int n = 0; n < DEPTH; ++n) v[n] = row(n);
#pragma unroll
            for (int n = 0; n < 9; ++n) {
                const quad in = v[n % DEPTH];
                __builtin_amdgcn_sched_barrier(0);
                // taps in raster order, as the matrix instructions of the backward add them: the same bits
#pragma unroll
                for (int c = 1; c < 4; ++c) u[c] = fmaf(w[3 * n][c], in[c - 1], u[c]);
#pragma unroll
                for (int c = 0; c < 4; ++c) u[c] = fmaf(w[3 * n + 1][c], in[c], u[c]);
#pragma unroll
                for (int c = 0; c < 3; ++c) u[c] = fmaf(w[3 * n + 2][c], in[c + 1], u[c]);
                __builtin_amdgcn_sched_barrier(0);
                if (n + DEPTH < 9) v[n % DEPTH] = row(n + DEPTH);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) cur[c] = fmaf(rv[c], Act<ACT, float>::f(u[c]), cur[c]);
            wave_order();
            if (it + 1 < inner) *reinterpret_cast<quad *>(own) = cur;
            wave_order();
        }
        if (RES) {
            const float *from = back + work.wave * kBack + pl.row * 16 + pl.k * 4;
            cur = load_quad(from) + (cur - load_quad(from + 256));
        }
        stored = cur;
        done = s;
        if (ln.y_part) {  // (mean, M2) of the block's 64 cells, by the lanes of a sample
            const auto over_rows = [](float v) {
                v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));  // row_ror:4
                v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));  // row_ror:8
                v += __shfl_xor(v, 16);
                return v + __shfl_xor(v, 32);
            };
            const float block_mean = over_rows((cur[0] + cur[1]) + (cur[2] + cur[3])) * (1.f / kWave);
            float m2 = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) m2 = fmaf(cur[c] - block_mean, cur[c] - block_mean, m2);
            m2 = over_rows(m2);
            if (pl.row == 0 && s + pl.k < work.end)
                *reinterpret_cast<float2 *>(ln.y_part + ((long)(s + pl.k) * nblk + work.blk) * 2) = make_float2(block_mean, m2);
        }
    }
    if (work.active) store_group();
}

constexpr int kDepth = 4, kDepthPairs = 3;  // rows requested ahead in the backward

// The backward, first kernel: what step_bwd_fast does (its arguments and what it leaves are the same), four samples at
// a time.  Per neighbour row n and iteration, with the deltas of the block's cells in LDS in both layouts,
//   g += delta (by sample) x V[n]    V[n][h]: what cell (row + n, h) multiplies this cell by, zero for rows of other blocks
//   nw[n] += x (by cell) x delta (by cell) of row + n: entry (i, h) is x of cell (row, i) times delta of cell (row + n, h),
//            the gradient of the latter's weight that reads the former.  For a row of another block the deltas read as
//            zeros, and nw[n] gets D x (x of that row) at the end: the gradients of this cell's own weights there.
// The deltas by sample take the place of the block's rows in the window, which the recompute has left.
template <int ACT, bool RES>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void quads_bwd(const float *__restrict__ weight, const float *__restrict__ bias, const float *__restrict__ scale,
               const float *__restrict__ x, const float *__restrict__ dy, float *__restrict__ dweight,
               float *__restrict__ dbias, float *__restrict__ dscale, float *__restrict__ dx,
               float *__restrict__ dsum_out, int B, int M, int N, int K, int inner, int nchunk, int chunk_len, int param_mode,
               int dx_accumulate, LnFold ln, long slab_stride) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    QuadWork work;
    if (!work.find(blockIdx.x, M, N, K, nchunk, chunk_len, B)) return;
    if (slab_stride) {
        const long off = work.chunk * slab_stride;  // this chunk's copy of the gradient arrays
        dweight += off;
        dbias += off;
        dscale += off;
        ln.dgamma += off;
        ln.dbeta += off;
    }
    constexpr int PLANE = kPlaneBackward;
    const QuadPlace<PLANE> pl(work, N, K);
    const QuadFetch fx(work, M, N, K);
    const int stride = backward_floats(inner);
    float *affine = lds, *windows = lds + kAffine, *win = windows + work.wave * stride;
    float *deltas = win + window_floats(PLANE), *hist_u = deltas + kDeltas, *hist_x = hist_u + 256 * (inner - 1);
    const long cells = (long)M * N * K;
    const bool ln_in = ln.x_stats != nullptr;
    // always true, and not known to be: the residual form spills 8 registers more where these loads and what is made of them
    // are not in blocks of their own
    const bool through_ln = !RES || ln.y_raw != nullptr;

    Bands w;
    w.take(weight, cells, pl.own, pl.k);
    float v[9][4];
    {   // the neighbours' weights, exchanged through LDS
#pragma unroll
        for (int t = 0; t < 27; ++t) win[t * kWave + pl.row * 4 + pl.k] = weight[t * cells + pl.own];
        wave_order();
#pragma unroll
        for (int n = 0; n < 9; ++n)
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int a = n / 3, c = n % 3, d = pl.k - h + 1;
                const bool ok = pl.has(a, c) && (unsigned)d < 3u;
                const int at = ((8 - n) * 3 + d) * kWave + (pl.row + (a - 1) * 4 + c - 1) * 4 + h;
                const float there = win[ok ? at : 0];
                v[n][h] = ok ? there : 0.f;
            }
        wave_order();
    }
    const float bv = bias[pl.own], rv = scale[pl.own], gam = ln.gamma[pl.own];
    QuadFetch::Buf pre;
    if (ln_in) {
        QuadFetch::Buf beta;
        fx.fetch(ln.gamma, 0, pre);
        fx.fetch(ln.beta, 0, beta);
        fx.pack_affine(affine, pre, beta);
    }
    for (int at = pl.lane; at < kDeltas; at += kWave) deltas[at] = 0.f;
    const float *deltas00 = deltas + pl.i * kDeltaPlane + pl.j * 16 + pl.k * 4;  // of cell k of row (i - 1, j - 1)
    wave_order();
    wait_global_loads();

    quad nw[9];
    float ns[9], db = 0.f, dr = 0.f, dgam = 0.f, dbet = 0.f;
#pragma unroll
    for (int n = 0; n < 9; ++n) {
        nw[n] = quad{0.f, 0.f, 0.f, 0.f};
        ns[n] = 0.f;
    }
    // entry i of nw[n] is the gradient of the weight at this place, where |i - k| < 2
    auto place_of = [&](int n, int i) {
        const int a = n / 3, c = n % 3;
        return pl.has(a, c) ? ((8 - n) * 3 + i - pl.k + 1) * cells + pl.own + ((a - 1) * N + c - 1) * K
                            : (n * 3 + pl.k - i + 1) * cells + pl.own + i - pl.k;
    };
    auto is_weight = [&](int i) { return (unsigned)(i - pl.k + 1) < 3u; };
    const bool has_side = pl.k == 0 || pl.k == 3;
    auto side_of = [&](int n) { return (n * 3 + (pl.k ? 2 : 0)) * cells + pl.own; };

    float x_mean = 0.f, x_rstd = 1.f;
    float2 y_st = make_float2(0.f, 1.f), y_sm = make_float2(0.f, 0.f);
    float gnext[kGroup], ynext[kGroup], gprev[kGroup];
    auto fetch_group = [&](int s) {
        const int mine = min(s + fx.sample(), work.end - 1) - s;  // past the end: the last sample again
        fx.fetch(x + s * cells, 4u * (unsigned)mine * (unsigned)cells, pre);
        if (ln_in) {
            const float2 st = *reinterpret_cast<const float2 *>(ln.x_stats + 2 * (s + mine));
            x_mean = st.x;
            x_rstd = st.y;
        }
        if (through_ln) {
            const int at = 2 * min(s + pl.k, work.end - 1);
            y_st = *reinterpret_cast<const float2 *>(ln.y_stats + at);
            y_sm = *reinterpret_cast<const float2 *>(ln.y_sums + at);
        }
#pragma unroll
        for (int q = 0; q < kGroup; ++q) {
            const long at = min(s + q, work.end - 1) * cells;
            gnext[q] = *at_cell(dy + at, pl.own);
            if (through_ln) ynext[q] = *at_cell(ln.y_raw + at, pl.own);
            if (RES && through_ln) gprev[q] = *at_cell(ln.g_prev + at, pl.own);
        }
    };
    quad g, gin;
    auto take_group = [&](int s) {
        for_samples([&](auto sample) {
            constexpr int q = decltype(sample)::value;
            const bool in = s + q < work.end;
            const float up = in ? gnext[q] : 0.f;
            float v = up;
            if (through_ln) {
                const float rstd = of_sample<q>(y_st.y), yh = (ynext[q] - of_sample<q>(y_st.x)) * rstd;
                dgam = fmaf(up, yh, dgam);
                dbet += up;
                v = rstd * (gam * up - of_sample<q>(y_sm.x) - yh * of_sample<q>(y_sm.y));
                if (RES) v += gprev[q];
                v = in ? v : 0.f;
            }
            g[q] = v;
        });
        if (RES) gin = g;
        if (ln_in) fx.template commit<true, PLANE>(windows, stride, pre, affine, x_mean, x_rstd);
        else fx.template commit<false, PLANE>(windows, stride, pre, affine, x_mean, x_rstd);
    };
    fetch_group(work.first);
    // What leaves is stored one group late, behind the wait for the windows: loads and stores share one in-order counter.
    quad out = {0.f, 0.f, 0.f, 0.f}, dsum = out, kept = out;
    const auto store_group = [&](int s) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (s + q < work.end) {
                const long at = (s + q) * cells;
                *at_cell(dsum_out + at, pl.own) = dsum[q];
                float *to = at_cell(dx + at, pl.own);
                *to = dx_accumulate ? *to + out[q] : out[q];
                if (RES && ln.g_out) *at_cell(ln.g_out + at, pl.own) = kept[q];
            }
    };
    for (int s = work.first; s < work.end; s += kGroup) {
        lds_barrier();  // gamma and beta, the weights have been exchanged; the windows are free
        take_group(s);
        if (s > work.first && work.active) store_group(s - kGroup);
        lds_barrier();
        if (s + kGroup < work.end) fetch_group(s + kGroup);
        if (!work.active) continue;
        quad x0, cur, u;
        dsum = quad{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) x0[q] = win[pl.cell + 4 * q];
        cur = x0;
        const quad u0 = side_sums(win, pl, w, bv);
        for (int it = 0;; ++it) {
            u = band_sums<kDepth>(win, pl, w.w, u0);
            if (it + 1 == inner) break;
            *reinterpret_cast<quad *>(hist_u + it * 256 + pl.lane * 4) = u;
            wave_order();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                cur[q] = fmaf(rv, Act<ACT, float>::f(u[q]), cur[q]);
                win[pl.cell + 4 * q] = cur[q];
            }
            if (it + 2 < inner) *reinterpret_cast<quad *>(hist_x + it * 256 + pl.lane * 4) = cur;
            wave_order();
        }
        for (int it = inner - 1;; --it) {
            quad delta;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float f, d;
                Act<ACT, float>::fd(u[q], f, d);
                const float e = d * g[q];
                delta[q] = e * rv;
                // leaky_relu(u) g = u (leaky_relu'(u) g)
                dr = ACT == GRIDNET_ACT_LEAKY_RELU ? fmaf(u[q], e, dr) : fmaf(f, g[q], dr);
                win[pl.cell + 4 * q] = delta[q];
            }
            dsum += delta;
            *reinterpret_cast<quad *>(const_cast<float *>(deltas00) + kDeltaPlane + 16) = delta;
            wave_order();
            // a sum of its own, added to g once: its terms are rounded at their size and not at that of g
            quad sum = {0.f, 0.f, 0.f, 0.f}, by_sample[kDepthPairs], by_cell[kDepthPairs];
            const auto request = [&](int n) {
                by_sample[n % kDepthPairs] = load_quad(win + pl.rows00 + n / 3 * PLANE + n % 3 * 16);
                by_cell[n % kDepthPairs] = load_quad(deltas00 + n / 3 * kDeltaPlane + n % 3 * 16);
            };
#pragma unroll
            for (int n = 0; n < kDepthPairs; ++n) request(n);
#pragma unroll
            for (int n = 0; n < 9; ++n) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    sum = mfma(by_sample[n % kDepthPairs][h], v[n][h], sum);
                    nw[n] = mfma(cur[h], by_cell[n % kDepthPairs][h], nw[n]);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (n + kDepthPairs < 9) request(n + kDepthPairs);
            }
            g += sum;
            wave_order();
            if (it == 0) break;
            u = load_quad(hist_u + (it - 1) * 256 + pl.lane * 4);
            cur = it > 1 ? load_quad(hist_x + (it - 2) * 256 + pl.lane * 4) : x0;
        }
        db += (dsum[0] + dsum[1]) + (dsum[2] + dsum[3]);
        // the weights that read the halo: the window without the block
        *reinterpret_cast<quad *>(win + pl.rows00 + PLANE + 16) = quad{0.f, 0.f, 0.f, 0.f};
        wave_order();
#pragma unroll
        for (int n = 0; n < 9; ++n) {
            if (n != 4) {
                const float *row = win + pl.cell + (n / 3 - 1) * PLANE + (n % 3 - 1) * 16;
#pragma unroll
                for (int q = 0; q < 4; ++q) nw[n] = mfma(dsum[q], row[4 * q], nw[n]);
            }
            const quad end = load_quad(win + pl.sides00 + (n / 3 * 6 + n % 3) * 8);
#pragma unroll
            for (int q = 0; q < 4; ++q) ns[n] = fmaf(end[q], dsum[q], ns[n]);
            if (n % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        out = g;
        if (RES) {
            out -= gin;
            kept = gin;
        }
    }
    if (!work.active) return;
    store_group(work.first + (work.end - work.first - 1) / kGroup * kGroup);
    // What the arrays hold is added here, in one rounding.  Sums that start from it, as those of step_bwd_fast do, take all steps
    // of a chain into one running sum: 4072 of the 7 million entries of dweight were outside the tests' bar for 64^3, batch 128, 16
    // steps of eight iterations, 1541 with step_bwd_fast's two sums of half the batch.
    if (param_mode == kParamAddExclusive) {
#pragma unroll
        for (int n = 0; n < 9; ++n) {
            quad old;
#pragma unroll
            for (int i = 0; i < 4; ++i) old[i] = is_weight(i) ? dweight[place_of(n, i)] : 0.f;
            nw[n] += old;
            ns[n] += has_side ? dweight[side_of(n)] : 0.f;
        }
        db += dbias[pl.own];
        dr += dscale[pl.own];
    }
    if (param_mode != kParamStore) {
        dgam += ln.dgamma[pl.own];
        dbet += ln.dbeta[pl.own];
    }
#pragma unroll
    for (int n = 0; n < 9; ++n) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (is_weight(i)) dweight[place_of(n, i)] = nw[n][i];
        if (has_side) dweight[side_of(n)] = ns[n];
    }
    dbias[pl.own] = db;
    dscale[pl.own] = dr;
    ln.dgamma[pl.own] = dgam;
    ln.dbeta[pl.own] = dbet;
}

// workgroups of one chunk of the batch
int quad_groups(const StepArgs &a) { return (a.M / 4) * (a.N / 4) * ((a.K / 4 + kWaves - 1) / kWaves); }

template <int ACT, bool RES> int launch_fwd(const StepArgs &a, hipStream_t st) {
    auto kern = quads_fwd<ACT, RES>;
    static int per_cu = 0;
    if (per_cu == 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, kThreads, 0) != hipSuccess || n < 1) n = 1;
        per_cu = n;
    }
    const int nblk = (a.M / 4) * (a.N / 4) * (a.K / 4), groups = quad_groups(a);
    int nchunk, chunk_len;
    plan_batch_chunks(a.B, groups, kGroup, per_cu * plan_device_cus(), false, nchunk, chunk_len);
    plan_even_rounds(a.B, groups, kGroup, per_cu * plan_device_cus(), 2 * kGroup, nchunk, chunk_len);
    hipLaunchKernelGGL(kern, dim3(padded_grid(groups, nchunk)), dim3(kThreads), 0, st, (const float *)a.weight,
                       (const float *)a.bias, (const float *)a.scale, (const float *)a.x, (float *)a.y, a.B, a.M, a.N, a.K,
                       a.inner, nblk, nchunk, chunk_len, a.ln);
    return check_launch("quads_fwd");
}

constexpr size_t kMaxLds = 160 * 1024;

// The backward's chunks, two workgroups to a CU: where the blocks are fewer the batch goes in chunks with a copy of the
// gradients each, of which there is room for `room`.  Whether step_bwd_fast is left for it: where the walk pays for the
// set-up, the groups of four are nearly full, and so are the rounds of waves.  Both kernels of a chain's backward, leaky_relu, us,
// step_bwd_fast -> quads_bwd: 64^3, batch 128, eight iterations, 1162 -> 947; batch 32, four, 236 -> 207; batch 12, 123 ->
// 113; batch 16, two, 123 -> 119; batch 4, eight, 96 -> 92; but batch 8, two (a walk of 16), 83 -> 95; batch 5, four (five of eight
// places), 91 -> 96; batch 10, eight (ten of twelve), 144 -> 140, with silu 151 -> 156; 32^3, batch 64, four (chunks of
// 16), 75 -> 72; batch 8 (chunks of four), 29 -> 34; 52^3, batch 32, 192 -> 159; 44^3 (1331 blocks for 2048 places), 109 ->
// 100; but 40^3 (1000), 102 -> 132, where step_bwd_fast fills the chip with four samples of a block to a workgroup.  Where there are
// three rounds or more, seven tenths of the places: 128 x 56 x 36, batch 100, five iterations (4032 of 6144), 745 -> 827; 56 x 80 x 52,
// batch 16, six (3640), 161 -> 178; 80 x 80 x 40, batch 20, four (4000), 170 -> 183.  Over 1200 grids that it is taken on by this rule
// (half of them with silu, half in the residual form) 1.14 times as fast, on 20 of them slower, by 11 % at most: batches in
// chunks on thin rows, 16 x 56 x 36, batch 64, six, 93 -> 99, with silu 96 -> 108.
constexpr int kShortestWalk = 32, kMostIterations = 8;
bool plan_backward(const StepArgs &a, int room, int &nchunk, int &chunk_len) {
    const int groups = quad_groups(a), resident = 2 * plan_device_cus();
    plan_batch_chunks(a.B, groups, kGroup, resident, false, nchunk, chunk_len);
    if (nchunk > 1 && room < nchunk)
        plan_batch_chunks(a.B, groups, kGroup, (room < 2 ? 1 : room) * groups, room < 2, nchunk, chunk_len);
    const long waves = (long)(a.M / 4) * (a.N / 4) * (a.K / 4) * nchunk;
    const long rounds = ((long)groups * nchunk + resident - 1) / resident;
    const long places = rounds * resident * kWaves;
    return chunk_len * a.inner >= kShortestWalk && 20L * a.B >= 17L * nchunk * chunk_len &&
           (rounds < 3 ? 2 * waves > places : 10 * waves >= 7 * places);
}

template <int ACT, bool RES> int launch_bwd(const StepArgs &a, hipStream_t st) {
    auto kern = quads_bwd<ACT, RES>;
    const size_t lds = ((size_t)kWaves * backward_floats(a.inner) + kAffine) * sizeof(float);
    static bool big_lds_enabled = false;  // per instantiation
    if (lds > 64 * 1024 && !big_lds_enabled) {
        const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
        if (e != hipSuccess) return fail(GRIDNET_ERR_LAUNCH, "cannot enable %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        big_lds_enabled = true;
    }
    const long cells = (long)a.M * a.N * a.K, slab_floats = kStepSlabPlanes * cells;
    const int groups = quad_groups(a);
    int nchunk, chunk_len;
    plan_backward(a, plan_slab_capacity(a.slabs, a.slab_bytes, slab_floats), nchunk, chunk_len);
    const bool split = nchunk > 1;
    float *slab = (float *)a.slabs;
    LnFold ln = a.ln;
    if (split) {
        ln.dgamma = slab + 29 * cells;
        ln.dbeta = slab + 30 * cells;
    }
    hipLaunchKernelGGL(kern, dim3(padded_grid(groups, nchunk)), dim3(kThreads), lds, st, (const float *)a.weight,
                       (const float *)a.bias, (const float *)a.scale, (const float *)a.x, (const float *)a.dy,
                       split ? slab : (float *)a.dweight, split ? slab + 27 * cells : (float *)a.dbias,
                       split ? slab + 28 * cells : (float *)a.dscale, (float *)a.dx, (float *)a.workspace, a.B, a.M, a.N,
                       a.K, a.inner, nchunk, chunk_len, plan_param_mode(split, a.flags),
                       (a.flags & GRIDNET_OVERWRITE_DX) ? 0 : 1, ln, split ? slab_floats : 0L);
    if (int rc = check_launch("quads_bwd")) return rc;
    TailJob tail{};
    if (split) {
        SlabTargets t{};
        t.dst[0] = (float *)a.dweight; t.end[0] = 27 * cells;
        t.dst[1] = (float *)a.dbias;   t.end[1] = 28 * cells;
        t.dst[2] = (float *)a.dscale;  t.end[2] = 29 * cells;
        t.dst[3] = a.ln.dgamma;        t.end[3] = 30 * cells;
        t.dst[4] = a.ln.dbeta;         t.end[4] = 31 * cells;
        t.count = 5;
        tail = plan_tail_job(slab, nchunk, slab_floats, t, plan_accumulate_mask(a.flags), cross_rows_threads(a));
    }
    return cross_rows_launch(a, tail, st);
}

template <template <int> class Launch> int with_activation(const StepArgs &a, hipStream_t st) {
    switch (a.activation) {
        case GRIDNET_ACT_RELU: return Launch<GRIDNET_ACT_RELU>::go(a, st);
        case GRIDNET_ACT_LEAKY_RELU: return Launch<GRIDNET_ACT_LEAKY_RELU>::go(a, st);
        case GRIDNET_ACT_SILU: return Launch<GRIDNET_ACT_SILU>::go(a, st);
        case GRIDNET_ACT_TANH: return Launch<GRIDNET_ACT_TANH>::go(a, st);
    }
    return fail(GRIDNET_ERR_ACTIVATION, "unknown activation function: id %d", a.activation);
}
template <int ACT> struct Forward {
    static int go(const StepArgs &a, hipStream_t st) {
        return a.ln.residual ? launch_fwd<ACT, true>(a, st) : launch_fwd<ACT, false>(a, st);
    }
};
template <int ACT> struct Backward {
    static int go(const StepArgs &a, hipStream_t st) {
        return a.ln.residual ? launch_bwd<ACT, true>(a, st) : launch_bwd<ACT, false>(a, st);
    }
};

}  // namespace

// by what the kernels can do; byte offsets of a group's four samples have to fit 32 bits
static bool covers(const StepArgs &a) {
    return a.dtype == GRIDNET_F32 && a.block_size == 4 && !a.normalize && a.inner >= 2 && a.B >= kGroup &&
           a.ln.gamma && (long)a.M * a.N * a.K <= 1L << 26;
}
// The forward's rule.  Few samples of few blocks are left to step_fwd_fast, which spreads each over a wave with one cell per thread
// (few_for_slots).  So are rows of one block, where three waves of four have no block (with a batch that is no multiple of four
// places of the fourth are empty, too), as soon as the chip has more than a few rounds of waves -- until then idle ones cost nothing --
// and rows of two, or of more with a batch of five, where there are more rounds still and the workgroups are more than the chip holds.
// Forward of a chain's step, leaky_relu, statistics included, from a graph, us, step_fwd_fast -> quads_fwd: 16 x 16 x 4, batch 6,
// two iterations, 5.9 -> 7.9; 32 x 32 x 12, batch 7 (1344 pairs of block and sample), 7.7 -> 8.1; 16 x 16 x 64, batch 6 (1536), 9.2 ->
// 8.5; 32 x 32 x 20, batch 5 (1600), 11.4 -> 8.3; 64 x 64 x 44, batch 13, 40 -> 25; 64^3, batch 9, eight, 57 -> 37.  Rows of one block,
// 128 x 128 x 4: batch 12 (four rounds), two iterations, 23.4 -> 21.1, eight 29.2 -> 29.1; batch 13 (five and a third), 23.4 -> 24.4, eight
// 29.5 -> 35.8; batch 128, eight, 117 -> 174; 64 x 64 x 4, batch 128, 42 -> 48; batch 64 (five and a third), two, 23.4 -> 21.0.  Of
// two: 128 x 128 x 8, batch 16, eight, 42.8 -> 39.3; batch 64, two, 60 -> 65, eight 114 -> 103, with silu, batch 128, 217 -> 247; but 64 x 64 x 8, batch
// 128 (256 workgroups), 67 -> 52.  Over 2000 grids of 16 to 128 cells a side, K from 4, batch 4 to 128, two to eight iterations, the
// better kernel every time would be 0.1 % faster than the rule and quads_fwd everywhere 4 % slower; with silu and in the residual
// form the same to 0.1 %.
constexpr int kFewestPairs = 6;                    // per CU
constexpr int kForwardPerCu = 3;                   // workgroups, a wave of each on every SIMD
constexpr int kMostRoundsOfOne = 5, kMostRoundsOfTwo = 8;
static bool fills_places(const StepArgs &a) {
    const long cus = plan_device_cus(), groups = quad_groups(a), pairs = (long)(a.M / 4) * (a.N / 4) * (a.K / 4) * a.B;
    const long waves = groups * kWaves * ((a.B + kGroup - 1) / kGroup), round = kForwardPerCu * kWaves * cus;
    if (pairs <= kFewestPairs * cus) return false;
    if (10 * pairs <= 3 * waves * kGroup && waves > kMostRoundsOfOne * round) return false;
    return !(2 * pairs <= waves * kGroup && waves > kMostRoundsOfTwo * round && groups > kForwardPerCu * cus);
}
bool step_quads_supports(const StepArgs &a, bool backward) {
    if (!covers(a)) return false;
    if (!backward) return fills_places(a);
    if (!a.ln.y_raw) return false;  // no LayerNorm behind the step
    int nchunk, chunk_len;
    return a.inner <= kMostIterations && cross_rows_supports(a) &&
           plan_backward(a, plan_slab_capacity(a.slabs, a.slab_bytes, kStepSlabPlanes * (long)a.M * a.N * a.K), nchunk, chunk_len);
}
size_t step_quads_slab_bytes(const StepArgs &a) {
    int nchunk, chunk_len;
    if (!covers(a) || a.inner > kMostIterations || !cross_rows_supports(a) ||
        !plan_backward(a, a.B, nchunk, chunk_len) || nchunk < 2)
        return 0;
    return (size_t)nchunk * kStepSlabPlanes * a.M * a.N * a.K * sizeof(float);
}
int step_quads_forward(const StepArgs &a, hipStream_t st) { return with_activation<Forward>(a, st); }
int step_quads_backward(const StepArgs &a, hipStream_t st) { return with_activation<Backward>(a, st); }

}  // namespace gridnet
