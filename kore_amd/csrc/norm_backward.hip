// norm_backward.hip -- RMSNorm backward: dx and dgamma in one pass over the
// rows plus a small deterministic column reduction.
//
// Definition: crates/kore-kernels/src/cpu_fused_backward.rs:20-81
// (fused_rms_norm_backward), per row r with d = cols:
//   sum_sq = sum_i x^2;  inv = 1 / sqrt(sum_sq / d + eps)
//   dgamma[i] += (dy[i] * x[i]) * inv                 (accumulated over rows)
//   dot = sum_i (x[i] * dy[i]) * g[i]
//   coeff = (dot * inv) / (sum_sq + eps * d)
//   dx[i] = (g[i] * inv) * dy[i] - coeff * x[i]
// Sums are tree reductions (f32 tolerance; the reference has no GPU version).
//
// Roofline: HBM.  Algorithmic bytes: x and dy read once, dx written once
// (12 * rows * cols), plus gamma and dgamma.  The dgamma partials add
// 2 * P * cols * 4 bytes (P = the workgroup count, ~512 for large batches:
// 2% of the traffic at 16384 x 2048).
//
// Row pass (rms_bwd_rows_kernel, cols <= 16384, any alignment): a row is split
// over S = 1, 2, 4, 8 or 16 waves (at most 4 float4 columns per wave and
// operand); a workgroup runs several row iterations with the next row's loads
// in flight; gamma is staged in LDS; each wave's dgamma partial stays in
// registers; the row slots' partials are added in a fixed order through LDS
// and written as partial row p = the block index.  Column pass: 8 float4
// columns x 64 row slots per block; every slot adds its partial rows in order
// (16 loads in flight), then a fixed-shape tree adds the slots -> dgamma
// (deterministic).
//   * 16-byte aligned rows of whole float4, cols <= 4096: workgroups of 4
//     waves, up to 16 row iterations, the partial rows in the workspace
//     (rms_bwd_reduce_kernel).
//   * other rows: their workspace is one float per row, so the partial rows
//     wait in the last P rows of dx, and the column pass computes those rows'
//     dx after it has added them (rms_bwd_finish_kernel).
// Generic path (longer rows, few ragged or long ones): one workgroup per row writes dx
// and inv[r] to the workspace; then one thread per column folds its dgamma
// over the rows in the reference's order.
#include <mutex>

#include "common.hpp"
#include "kore_hip_internal.hpp"

namespace kore {

constexpr int kBwBlock = 256;
constexpr int kBwWaves = kBwBlock / kWave;

struct BwArgs {
    const float* dy;
    const float* x;
    const float* g;
    float* dx;
    float* dgamma;
    float* ws;    // caller's or library's scratch
    float* part;  // P partial dgamma rows of cols floats
    uint64_t rows;
    uint64_t dx_rows;  // the row pass writes dx for rows r < dx_rows
    uint64_t cols;
    float eps;
    uint32_t rpw;       // row iterations per workgroup (vector path)
    uint64_t partials;  // P
};

__device__ __forceinline__ float sum4(f32x4 a) { return (a.x + a.y) + (a.z + a.w); }

// A row is split over S waves (wave w: row slot j = w / S, column part
// q = w % S, NCHW chunks of 64 float4), so a wave holds at most 4 float4 per
// operand.  Long and ragged rows deal the chunks out in turn (k*S + q), so that
// the waves' shares differ by one chunk at most.  Iteration it of workgroup b takes row
// (it * P + b) * kSlots + j (P = the grid size), so each iteration of the grid
// sweeps one contiguous band of rows (measured 89 -> 80 us at 16384 x 2048
// against giving each workgroup a contiguous block of rows).  Per row, the S
// waves' partial sums meet in LDS (slot parity double-buffered, one barrier
// per iteration) and are added in q order (by a fixed tree for S >= 8).  Each
// wave keeps its dgamma partial in registers; at the end the row slots'
// partials are added in j order through LDS and written as partial row b.
// Rows from dx_rows on leave their inv and coeff in ws instead of writing dx.
// Ragged: rows of any length and alignment (see ld_row4).
template <int NCHW, int S, int kWaves, bool Ragged>
__global__ __launch_bounds__(kWave * kWaves) __attribute__((amdgpu_waves_per_eu(4)))
void rms_bwd_rows_kernel(BwArgs a) {
    constexpr bool kLong = kWaves != kBwWaves;
    constexpr int kThreads = kWaves * kWave;
    constexpr int kSlots = kWaves / S;
    // gamma (0 past cols), then the dgamma combine: whole chunks, so that a
    // lane's entries lie at fixed offsets
    constexpr int kGam = NCHW * S * kWave;
    __shared__ f32x4 gam[kGam];
    __shared__ float red[2][kWaves][2];
    const int lane = threadIdx.x & (kWave - 1);
    // a scalar, so that row addresses live in SGPRs
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int j = wave / S, q = wave % S;
    const uint32_t cols = (uint32_t)a.cols;
    const uint32_t cols4 = Ragged ? (cols + 3) >> 2 : cols >> 2;
    const float fcols = (float)a.cols;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // iteration it of block b: row (it * P + b) * slots + j -- the grid sweeps
    // one contiguous band of rows per iteration.
    const uint64_t rstride = (uint64_t)gridDim.x * kSlots;
    const uint64_t rbase = (uint64_t)blockIdx.x * kSlots;

    auto col4 = [&](int k) { return (uint32_t)(kLong ? k * S + q : q * NCHW + k) * kWave + lane; };

    f32x4 acc[NCHW];
#pragma unroll
    for (int k = 0; k < NCHW; ++k) acc[k] = zero;
    // Row loads are double-buffered: iteration it + 1's x and dy are in
    // flight while iteration it reduces, synchronises and stores.
    f32x4 xv[NCHW], dv[NCHW];
    auto load_row = [&](uint32_t it, f32x4* xo, f32x4* dout) {
        const uint64_t r = rbase + (uint64_t)it * rstride + j;
        const bool live = it < a.rpw && r < a.rows;
        const uint64_t rr = live ? r : 0;
        const float* xr = a.x + rr * cols;
        const float* dr = a.dy + rr * cols;
#pragma unroll
        for (int k = 0; k < NCHW; ++k) {
            const uint32_t f = col4(k);
            xo[k] = live ? ld_row4<Ragged>(xr, f, cols) : zero;
            dout[k] = live ? ld_row4<Ragged>(dr, f, cols) : zero;
        }
    };
    load_row(0, xv, dv);
    // gamma lives in LDS for the whole sweep: its reads are LDS operations,
    // so they neither hold registers nor make a wait for them also wait for
    // the prefetched row.
    for (uint32_t f = threadIdx.x; f < (uint32_t)kGam; f += kThreads) gam[f] = ld_row4<Ragged, false>(a.g, f, cols);
    __syncthreads();
    for (uint32_t it = 0; it < a.rpw; ++it) {
        const uint64_t r = rbase + (uint64_t)it * rstride + j;
        const bool live = r < a.rows;
        f32x4 xn[NCHW], dn[NCHW];
        load_row(it + 1, xn, dn);
        float ss = 0.0f, dot = 0.0f;
#pragma unroll
        for (int k = 0; k < NCHW; ++k) {
            const uint32_t f = col4(k);
            ss += sum4(xv[k] * xv[k]);
            dot += sum4((xv[k] * dv[k]) * gam[f]);
        }
        ss = wave_sum_dpp(ss);
        dot = wave_sum_dpp(dot);
        if (S > 1) {
            const int par = it & 1;
            if (lane == 0) {
                red[par][wave][0] = ss;
                red[par][wave][1] = dot;
            }
            __syncthreads();
            if (S >= 8) {  // one read a lane and a tree, instead of 2 S values in registers
                const bool mine = lane < S;
                ss = wave_sum_dpp(mine ? red[par][j * S + lane][0] : 0.0f);
                dot = wave_sum_dpp(mine ? red[par][j * S + lane][1] : 0.0f);
            } else {
                ss = red[par][j * S][0];
                dot = red[par][j * S][1];
#pragma unroll
                for (int t = 1; t < S; ++t) {
                    ss += red[par][j * S + t][0];
                    dot += red[par][j * S + t][1];
                }
            }
        }
        const float inv = 1.0f / sqrtf(ss / fcols + a.eps);
        const float coeff = (dot * inv) / (ss + a.eps * fcols);
        if (live) {
#pragma unroll
            for (int k = 0; k < NCHW; ++k) acc[k] = acc[k] + (dv[k] * xv[k]) * inv;
        }
        if (kLong && live && r >= a.dx_rows) {  // dx from rms_bwd_finish_kernel
            if (q == 0 && lane == 0) {
                a.ws[r - a.dx_rows] = inv;
                a.ws[r - a.dx_rows + (a.rows - a.dx_rows)] = coeff;
            }
        } else if (live) {
            float* orow = a.dx + r * cols;
#pragma unroll
            for (int k = 0; k < NCHW; ++k) {
                const uint32_t f = col4(k);
                st_row4<Ragged>(orow, f, cols, (gam[f] * inv) * dv[k] - coeff * xv[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < NCHW; ++k) {
            xv[k] = xn[k];
            dv[k] = dn[k];
        }
    }
    // One partial row: a single row slot's as it is, several added in j order
    // through LDS (gamma is done with).
    float* prow = a.part + (uint64_t)blockIdx.x * cols;
    if (kSlots == 1) {
#pragma unroll
        for (int k = 0; k < NCHW; ++k) st_row4<Ragged, false>(prow, col4(k), cols, acc[k]);
        return;
    }
    __syncthreads();
#pragma unroll 1
    for (int jj = 0; jj < kSlots; ++jj) {
        if (j == jj) {
#pragma unroll
            for (int k = 0; k < NCHW; ++k) {
                const uint32_t f = col4(k);
                gam[f] = (jj == 0) ? acc[k] : gam[f] + acc[k];
            }
        }
        __syncthreads();
    }
    for (uint32_t f = threadIdx.x; f < cols4; f += kThreads) st_row4<Ragged, false>(prow, f, cols, gam[f]);
}

// dgamma = sum of the P partial rows, deterministic: block = 8 float4
// columns (128 contiguous bytes of a partial row) x 64 row slots; thread
// (slot, c) adds rows slot, slot+64, ... in order, with 16 loads in flight;
// the 64 slot sums are then added by a fixed-shape tree in LDS.  The order
// depends only on P, so repeated calls give identical bits.
constexpr int kRedCols = 8;
constexpr int kRedSlots = 64;
constexpr int kRedBatch = 16;
template <bool Ragged>
__device__ __forceinline__ void reduce_partials(const BwArgs& a, int c, int slot, uint64_t col) {
    __shared__ f32x4 red[kRedSlots][kRedCols];
    const uint64_t cols4 = (a.cols + 3) >> 2;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 t = zero;
    if (col < cols4) {
        for (uint64_t p0 = slot; p0 < a.partials; p0 += kRedBatch * kRedSlots) {
            f32x4 v[kRedBatch];
#pragma unroll
            for (int u = 0; u < kRedBatch; ++u) {
                const uint64_t p = p0 + (uint64_t)u * kRedSlots;
                if (Ragged)
                    v[u] = p < a.partials
                               ? ld_row4<true, false>(a.part + p * a.cols, (uint32_t)col, (uint32_t)a.cols)
                               : zero;
                else
                    v[u] = p < a.partials ? reinterpret_cast<const f32x4*>(a.part)[p * cols4 + col] : zero;
            }
#pragma unroll
            for (int u = 0; u < kRedBatch; ++u) {
                if (p0 + (uint64_t)u * kRedSlots < a.partials) t = t + v[u];
            }
        }
    }
    red[slot][c] = t;
    __syncthreads();
#pragma unroll
    for (int w = kRedSlots / 2; w >= 1; w >>= 1) {
        if (slot < w) red[slot][c] = red[slot][c] + red[slot + w][c];
        __syncthreads();
    }
    if (slot == 0 && col < cols4)
        st_row4<Ragged, false>(a.dgamma, (uint32_t)col, (uint32_t)a.cols, red[0][c]);
}

__global__ __launch_bounds__(kRedCols * kRedSlots) void rms_bwd_reduce_kernel(BwArgs a) {
    const int c = threadIdx.x % kRedCols, slot = threadIdx.x / kRedCols;
    reduce_partials<false>(a, c, slot, (uint64_t)blockIdx.x * kRedCols + c);
}

// The same, and then dx of the last rows, which held the partials: a block
// owns its columns of all of them, so after the reduction's barriers nothing
// reads what it overwrites.  inv and coeff of those rows come from ws.
constexpr int kFinBatch = 4;  // rows a thread has in flight
template <bool Ragged>
__global__ __launch_bounds__(kRedCols * kRedSlots) void rms_bwd_finish_kernel(BwArgs a) {
    const int c = threadIdx.x % kRedCols, slot = threadIdx.x / kRedCols;
    const uint64_t col = (uint64_t)blockIdx.x * kRedCols + c;
    const uint32_t cols = (uint32_t)a.cols;
    // gamma before dgamma is written: the two may be the same buffer
    const f32x4 g = ld_row4<Ragged, false>(a.g, (uint32_t)col, cols);
    reduce_partials<Ragged>(a, c, slot, col);
    if (4 * col >= a.cols) return;
    const uint64_t tail = a.rows - a.dx_rows;
    for (uint64_t p0 = slot; p0 < tail; p0 += kFinBatch * kRedSlots) {
        f32x4 x[kFinBatch], d[kFinBatch];
#pragma unroll
        for (int u = 0; u < kFinBatch; ++u) {
            const uint64_t p = p0 + (uint64_t)u * kRedSlots;
            if (p >= tail) continue;
            x[u] = ld_row4<Ragged>(a.x + (a.dx_rows + p) * cols, (uint32_t)col, cols);
            d[u] = ld_row4<Ragged>(a.dy + (a.dx_rows + p) * cols, (uint32_t)col, cols);
        }
#pragma unroll
        for (int u = 0; u < kFinBatch; ++u) {
            const uint64_t p = p0 + (uint64_t)u * kRedSlots;
            if (p >= tail) continue;
            const float inv = a.ws[p], coeff = a.ws[p + tail];
            st_row4<Ragged>(a.dx + (a.dx_rows + p) * cols, (uint32_t)col, cols, (g * inv) * d[u] - coeff * x[u]);
        }
    }
}

// ---- generic path
__global__ __launch_bounds__(kBwBlock) void rms_bwd_row_generic_kernel(BwArgs a) {
    __shared__ float red[2][kBwWaves];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const uint64_t r = blockIdx.x;
    const float* xr = a.x + r * a.cols;
    const float* dr = a.dy + r * a.cols;
    float ss = 0.0f, dot = 0.0f;
    for (uint64_t i = threadIdx.x; i < a.cols; i += kBwBlock) {
        const float xv = xr[i];
        ss += xv * xv;
        dot += (xv * dr[i]) * a.g[i];
    }
    ss = wave_sum(ss);
    dot = wave_sum(dot);
    if (lane == 0) {
        red[0][wave] = ss;
        red[1][wave] = dot;
    }
    __syncthreads();
    ss = red[0][0];
    dot = red[1][0];
#pragma unroll
    for (int w = 1; w < kBwWaves; ++w) {
        ss += red[0][w];
        dot += red[1][w];
    }
    const float fcols = (float)a.cols;
    const float inv = 1.0f / sqrtf(ss / fcols + a.eps);
    const float coeff = (dot * inv) / (ss + a.eps * fcols);
    for (uint64_t i = threadIdx.x; i < a.cols; i += kBwBlock)
        a.dx[r * a.cols + i] = (a.g[i] * inv) * dr[i] - coeff * xr[i];
    if (threadIdx.x == 0) a.ws[r] = inv;
}

// One thread per column: dgamma[c] = sum over rows, in row order.
__global__ __launch_bounds__(kBwBlock) void rms_bwd_col_generic_kernel(BwArgs a) {
    const uint64_t c = (uint64_t)blockIdx.x * kBwBlock + threadIdx.x;
    if (c >= a.cols) return;
    float acc = 0.0f;
    for (uint64_t r = 0; r < a.rows; ++r) acc = acc + (a.dy[r * a.cols + c] * a.x[r * a.cols + c]) * a.ws[r];
    a.dgamma[c] = acc;
}

__global__ __launch_bounds__(kBwBlock) void fill_zero_kernel(float* p, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * kBwBlock + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// Waves per row: each wave holds <= 4 float4 columns.
static uint32_t bwd_split(uint64_t cols) {
    const uint64_t c4 = (cols + 3) / 4;
    return c4 <= 256 ? 1u : (c4 <= 512 ? 2u : (c4 <= 1024 ? 4u : (c4 <= 2048 ? 8u : 16u)));
}

// Row iterations per workgroup, up to 4096 columns: ~512 workgroups (4 waves
// each, two per SIMD, with the next row's loads in flight) -- measured against
// 256, 384, 768 and 1024 at 16384 x 2048: fewer partial rows to reduce, and
// enough waves to keep HBM busy (70.0 vs 72.7 us at 1024); at most 16
// iterations so that large batches keep few partial rows, and past 2^28 rows
// as many as keep it at 2^30 threads (a launch holds fewer than 2^32).
static uint32_t bwd_iters(uint64_t rows, uint32_t split) {
    const uint64_t per_iter = kBwWaves / split;
    uint64_t it = (rows + 512 * per_iter - 1) / (512 * per_iter);
    if (it < 1) it = 1;
    const uint64_t most = rows >> 22 > 16 * per_iter ? (rows >> 22) / per_iter + 1 : 16;
    if (it > most) it = most;
    return (uint32_t)it;
}

// Workspace floats: the partial rows for whole float4 rows of up to 4096
// columns, else one float per row.
static bool bwd_ws_plan(uint64_t cols) { return cols % 4 == 0 && cols / 4 <= 1024; }
static uint64_t bwd_ws_floats(uint64_t rows, uint64_t cols) {
    if (!bwd_ws_plan(cols)) return rows;
    const uint32_t split = bwd_split(cols);
    const uint64_t rpb = (uint64_t)bwd_iters(rows, split) * (kBwWaves / split);  // rows per block = per partial row
    const uint64_t vec = (rows + rpb - 1) / rpb * cols;
    return vec > rows ? vec : rows;
}

// Rows of the generic path where the workspace plan does not run: a workgroup a
// row and a thread a dgamma column, against the long path's two launches that
// few rows leave waiting on 16 waves' barriers (us, generic against long path):
// 40 x 700 9.4 against 9.9, 48 x 1021 10.6 against 10.0; 40 x 4095 12.9 against
// 12.9, 49 x 2049 12.3 against 11.5; ragged 16 x 6912 12.3 against 12.9, 24 x 6144
// 12.6 against 10.5, 20 x 8192 14.2 against 13.8; whole 8 x 5120 9.4 against 9.9, 16
// 10.4 against 10.1, 2 x 8192 11.8 against 11.0; ragged 2 x 12001 15.8 against 14.2.
// An odd row more than the partial rows leave room for takes every workgroup
// another turn: whole 3 x 6144 9.9 against 10.7, 15 11.3 against 10.6, 9 x 8192 12.5
// against 12.8; ragged 5 x 12000 16.0 against 16.4, 15 x 12001 17.4 against 16.3.
static uint64_t bwd_generic_rows(uint64_t rows, uint64_t cols, bool aligned) {
    if (cols <= 4096) return 44;
    if (!aligned && cols <= 8192) return 18;
    if (cols <= 5120) return 10;
    return rows % 2 == 1 && cols <= (aligned ? 8192u : 12288u) ? 9 : 1;
}

template <int NCHW, int S>
static void launch_rows(const BwArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((rms_bwd_rows_kernel<NCHW, S, kBwWaves, false>), dim3((uint32_t)a.partials), dim3(kBwBlock), 0,
                       s, a);
}

// Long and ragged rows (up to 16384 columns): workgroups of 16 waves, one per
// CU, so that the fewest partial rows (whose rows of dx are read and written
// again at the end) keep every SIMD at four waves.  Measured, rows x columns:
// 4096 x 8192 85.5 us (4.7 TB/s; one workgroup per row and one thread per
// dgamma column before: 1740), 4096 x 8191 108 (1753), 8000 x 2049 57 (2770),
// 2048 x 14336 82 (966); with 512 workgroups of 8 waves 90, 110, 62 and 96,
// 256 of 8 86, 117, 67 and 82, 128 of 16 110, 134, 76 and 96.  Ragged rows of
// 513-1024 columns take two waves of 2 float4, as one of 4 has more registers in
// use than four waves a SIMD leave it and spills (100 x 1001 13.9 -> 10.0, 4096 x
// 1021 28.4 -> 24.0, 16384 x 1001 58.4 -> 54.6, 16384 x 515 44.4 -> 39.4).  Whole
// float4 up to 4096 columns keep the workspace plan (8192 x 4096 74 us, 5.4
// TB/s: no row is done twice).
constexpr int kBwLongWaves = 16;
constexpr uint64_t kBwLongBlocks = 256;

template <int NCHW, int S>
static void launch_long(const BwArgs& a, bool ragged, hipStream_t s) {
    static_assert(S <= kBwLongWaves, "a workgroup holds a row");
    const dim3 grid((uint32_t)a.partials), block(kBwLongWaves * kWave);
    if constexpr (S >= 8) {  // shorter whole rows take the workspace plan
        if (!ragged) {
            hipLaunchKernelGGL((rms_bwd_rows_kernel<NCHW, S, kBwLongWaves, false>), grid, block, 0, s, a);
            return;
        }
    }
    hipLaunchKernelGGL((rms_bwd_rows_kernel<NCHW, S, kBwLongWaves, true>), grid, block, 0, s, a);
}

// Library-held scratch for the allocation-free entry point: the dgamma
// partial rows (vector path) or the per-row inv (generic path), at most
// kBwScratchBytes.  Each GPU holds its own copy for the life of the process.
// Every call fully writes the part it reads back, so nothing needs clearing;
// calls that overlap on one GPU share the array and race.
constexpr uint64_t kBwScratchBytes = 16ull << 20;
static __device__ __align__(256) float rms_bwd_scratch[kBwScratchBytes / sizeof(float)];

// Device address of rms_bwd_scratch on the current device, looked up once per
// device with that device current.  In host code the array's name is only a
// host-side stand-in; kernels get this address instead.
constexpr int kMaxScratchDevices = 64;
static std::mutex g_bw_scratch_mu;
static float* g_bw_scratch[kMaxScratchDevices];

static int bwd_scratch_ptr(float** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxScratchDevices) return KORE_HIP_ERR_BAD_DIM;
    std::lock_guard<std::mutex> lock(g_bw_scratch_mu);
    if (!g_bw_scratch[dev]) {
        // The first call on a device may come from code under stream capture.
        // The lookup enqueues nothing, but a strict capture mode can refuse
        // runtime calls it does not know to be safe: this thread switches to
        // relaxed mode for the lookup and restores its mode afterwards.
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        e = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) return (int)e;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(rms_bwd_scratch));
        const hipError_t r = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) return (int)e;
        if (r != hipSuccess) return (int)r;
        g_bw_scratch[dev] = static_cast<float*>(p);
    }
    *out = g_bw_scratch[dev];
    return KORE_HIP_OK;
}

}  // namespace kore

using namespace kore;

extern "C" uint64_t kore_hip_rms_norm_backward_workspace_bytes(uint64_t rows, uint64_t cols) {
    if (rows == 0 || cols == 0) return 0;
    uint64_t elems;
    if (!mul_ok(rows, cols, &elems) || elems > kMaxElements) return 0;
    return bwd_ws_floats(rows, cols) * sizeof(float);
}

// The whole entry point once the workspace is known.  ws == nullptr asks for
// the library's own scratch array (the allocation-free entry point); it is
// looked up only after every argument check has passed.
static int rms_bwd_run(const float* grad_out, const float* x, const float* gamma, float* grad_x,
                       float* grad_gamma, float* workspace, uint64_t workspace_bytes, bool own_scratch,
                       uint64_t rows, uint64_t cols, float eps, hipStream_t s) {
    if (cols == 0) return KORE_HIP_OK;
    if (!grad_gamma || !gamma) return KORE_HIP_ERR_NULL_PTR;
    if (rows == 0) {  // dgamma of an empty batch is zero (the reference's vec![0.0; d])
        if (cols > kMaxElements) return KORE_HIP_ERR_OVERFLOW;
        // A fill kernel rather than hipMemsetAsync, so the call can be captured in a graph.
        hipLaunchKernelGGL(fill_zero_kernel, dim3((uint32_t)((cols + kBwBlock - 1) / kBwBlock)), dim3(kBwBlock), 0, s,
                           grad_gamma, cols);
        return launch_status();
    }
    if (!grad_out || !x || !grad_x || (!own_scratch && !workspace)) return KORE_HIP_ERR_NULL_PTR;
    uint64_t elems;
    if (!mul_ok(rows, cols, &elems) || elems > kMaxElements || rows > 0x7fffffffull) return KORE_HIP_ERR_OVERFLOW;
    BwArgs a{grad_out, x, gamma, grad_x, grad_gamma, workspace, nullptr, rows, rows, cols, eps, 0, 0};
    const uint64_t need = bwd_ws_floats(rows, cols) * sizeof(float);
    if (own_scratch) {
        if (need > kBwScratchBytes) return KORE_HIP_ERR_SCRATCH;
        workspace_bytes = kBwScratchBytes;
    } else if (workspace_bytes < need) {
        return KORE_HIP_ERR_BAD_DIM;
    }
    // grad_x must not overlap the inputs (the row pass reads a row ahead).
    const char* o0 = (const char*)grad_x;
    const char* o1 = o0 + elems * sizeof(float);
    for (const float* in : {grad_out, x}) {
        const char* i0 = (const char*)in;
        if (i0 < o1 && o0 < i0 + elems * sizeof(float)) return KORE_HIP_ERR_ALIAS;
    }
    if (own_scratch) {
        const int st = bwd_scratch_ptr(&a.ws);
        if (st != KORE_HIP_OK) return st;
        workspace = a.ws;
    }
    const uint64_t cols4 = (cols + 3) / 4;
    const bool aligned = cols % 4 == 0 && aligned16(grad_out) && aligned16(x) && aligned16(gamma) &&
                         aligned16(grad_x) && aligned16(grad_gamma) && aligned16(workspace);
    const uint32_t split = bwd_split(cols);
    if (aligned && bwd_ws_plan(cols)) {
        a.rpw = bwd_iters(rows, split);
        const uint64_t rpb = (uint64_t)a.rpw * (kBwWaves / split);
        a.partials = (rows + rpb - 1) / rpb;
        a.part = a.ws;
        if (cols4 <= 64) launch_rows<1, 1>(a, s);
        else if (cols4 <= 128) launch_rows<2, 1>(a, s);
        else if (cols4 <= 256) launch_rows<4, 1>(a, s);
        else if (cols4 <= 512) launch_rows<4, 2>(a, s);
        else launch_rows<4, 4>(a, s);
        hipLaunchKernelGGL(rms_bwd_reduce_kernel, dim3((uint32_t)((cols4 + kRedCols - 1) / kRedCols)),
                           dim3(kRedCols * kRedSlots), 0, s, a);
    } else if (cols <= 16384 && rows > bwd_generic_rows(rows, cols, aligned)) {
        // The workspace of these shapes holds one float per row, so the P
        // partial rows wait in dx's last P rows until the second launch has
        // reduced them and computes those rows' dx; 2 P <= rows, the inv and
        // coeff it needs being the workspace's first 2 P floats.
        const uint64_t slots = (uint32_t)kBwLongWaves / (cols4 > 128 && cols4 <= 256 ? 2u : split);
        uint64_t rpb = (rows + kBwLongBlocks - 1) / kBwLongBlocks;
        if (rpb < 2) rpb = 2;
        rpb = (rpb + slots - 1) / slots * slots;
        a.rpw = (uint32_t)(rpb / slots);
        a.partials = (rows + rpb - 1) / rpb;
        if (2 * a.partials > rows) a.partials = rows / 2;  // one row more for some workgroup
        while (a.partials * rpb < rows) a.rpw += 1, rpb += slots;
        a.dx_rows = rows - a.partials;
        a.part = grad_x + a.dx_rows * cols;
        if (cols4 <= 64) launch_long<1, 1>(a, !aligned, s);
        else if (cols4 <= 128) launch_long<2, 1>(a, !aligned, s);
        else if (cols4 <= 256) launch_long<2, 2>(a, !aligned, s);
        else if (cols4 <= 512) launch_long<4, 2>(a, !aligned, s);
        else if (cols4 <= 1024) launch_long<4, 4>(a, !aligned, s);
        else if (cols4 <= 1536) launch_long<3, 8>(a, !aligned, s);
        else if (cols4 <= 2048) launch_long<4, 8>(a, !aligned, s);
        else if (cols4 <= 3072) launch_long<3, 16>(a, !aligned, s);
        else launch_long<4, 16>(a, !aligned, s);
        const dim3 grid((uint32_t)((cols4 + kRedCols - 1) / kRedCols)), block(kRedCols * kRedSlots);
        if (aligned)
            hipLaunchKernelGGL(rms_bwd_finish_kernel<false>, grid, block, 0, s, a);
        else
            hipLaunchKernelGGL(rms_bwd_finish_kernel<true>, grid, block, 0, s, a);
    } else {
        hipLaunchKernelGGL(rms_bwd_row_generic_kernel, dim3((uint32_t)rows), dim3(kBwBlock), 0, s, a);
        hipLaunchKernelGGL(rms_bwd_col_generic_kernel, dim3((uint32_t)((cols + kBwBlock - 1) / kBwBlock)),
                           dim3(kBwBlock), 0, s, a);
    }
    return launch_status();
}

extern "C" int kore_hip_rms_norm_backward_f32(const float* grad_out, const float* x, const float* gamma,
                                              float* grad_x, float* grad_gamma, float* workspace,
                                              uint64_t workspace_bytes, uint64_t rows, uint64_t cols, float eps,
                                              kore_stream_t stream) {
    return rms_bwd_run(grad_out, x, gamma, grad_x, grad_gamma, workspace, workspace_bytes, false, rows, cols, eps,
                       (hipStream_t)stream);
}

extern "C" uint64_t kore_hip_rms_norm_backward_noalloc_max_bytes(void) { return kBwScratchBytes; }

extern "C" int kore_hip_rms_norm_backward_noalloc_f32(const float* grad_out, const float* x, const float* gamma,
                                                      float* grad_x, float* grad_gamma, uint64_t rows,
                                                      uint64_t cols, float eps, kore_stream_t stream) {
    return rms_bwd_run(grad_out, x, gamma, grad_x, grad_gamma, nullptr, 0, true, rows, cols, eps,
                       (hipStream_t)stream);
}
