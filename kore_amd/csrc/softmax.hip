// softmax.hip -- row softmax (plain and causal) and its backward.
//
// Roofline: HBM.  Bytes per row: forward 8*cols (x read, y written);
// backward 12*cols (y and dy read, dx written).
//
// Definitions (the reference's, with the f32 tolerance of its CUDA twin):
//   forward  crates/kore-kernels/src/cpu_fused.rs:195-231 (fused_softmax):
//            m = max over the row (NaN skipped, as f32::max / fmaxf),
//            e = exp(x - m), y = e * (1 / sum(e));
//   causal   crates/kore-kernels/src/cuda/kernels/softmax.cu:88-157
//            (softmax_causal_f32): row r keeps columns c < seq_offset + r + 1
//            (r counts over all rows of the call); the rest are -inf in the
//            max and 0 in the output; inv = sum > 0 ? 1/sum : 0;
//   backward crates/kore-kernels/src/cpu_fused_backward.rs:86-115
//            (fused_softmax_backward): dx = y * (dy - sum(y * dy));
//   cross-entropy backward cpu_fused_backward.rs:130-170
//            (fused_cross_entropy_backward): g = e * (inv_sum * inv_batch),
//            inv_batch = 1 / rows, then g[t] -= inv_batch at t = targets[r]
//            cast like Rust's `as usize` (truncation, NaN and negatives -> 0);
//            a t >= cols (the reference panics) subtracts nothing.
// The sums are tree reductions (lane partials, then a wave butterfly), so
// results are within the f32 tolerance of the reference's left fold, as its
// own CUDA kernel is.  exp(d) is evaluated on the reference's d = x - m
// (rounded the same way) as the hardware exp2(d * log2(e)); see exp_diff.
//
// Shapes: a row of up to 1024 floats is held in one wave's registers (one wave
// per row, 4 rows per workgroup; two waves a row where two_waves_a_row says so);
// up to 16384 in one workgroup's (256 threads; 512 for the 1025-2048 backward of
// whole rows and for few rows of more than 8192; 2049-4096 see mid_form); up to
// 135168 (vocabularies) in the registers and LDS of a CU (forward and
// cross-entropy); still longer rows, and the backward's from 16385, stream
// through a workgroup in three passes (two), as do a backward's few short
// ragged rows.  Rows of any length and alignment take the same kernels, their
// last cols % 4 floats one by one.
// Every kernel reads a row fully before writing it, so out may alias an input.
#include <type_traits>

#include "common.hpp"
#include "kore_hip_internal.hpp"

namespace kore {

enum class SmKind : int { Fwd = 0, Causal = 1, Bwd = 2, CeBwd = 3 };

struct SmArgs {
    const float* a;  // x (forward) or y (backward)
    const float* b;  // dy (backward), targets[rows] (cross-entropy), unused otherwise
    float* out;
    uint64_t rows;
    uint64_t cols;
    uint64_t seq_offset;
    float inv_batch;  // 1 / rows of the whole call (cross-entropy)
};

constexpr int kSmBlock = 256;
constexpr int kSmWaves = kSmBlock / kWave;

__device__ __forceinline__ float f4_get(const f32x4& v, int k) {
    return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w));
}
__device__ __forceinline__ void f4_set(f32x4& v, int k, float s) {
    if (k == 0) v.x = s; else if (k == 1) v.y = s; else if (k == 2) v.z = s; else v.w = s;
}

// Rust `f32 as usize`: NaN and negatives -> 0, truncation toward zero,
// saturating; returned as a column index, or UINT64_MAX when >= cols.
__device__ __forceinline__ uint64_t target_index(float t, uint64_t cols) {
    if (!(t >= 1.0f)) return cols > 0 ? 0 : ~0ull;  // NaN, negative, [0, 1)
    if (t >= 18446744073709551616.0f) return ~0ull;
    const uint64_t i = (uint64_t)t;
    return i < cols ? i : ~0ull;
}

// exp(d) for d = x - max <= 0 as v_exp_f32(d * log2(e)): 2 VALU ops instead
// of ~12 for ocml expf.  Rounding d*log2(e) perturbs the result by at most
// |d| * 2^-24 * ln 2 relative (< 1e-6 for d >= -16, where e^d > 1e-7 still
// matters next to the row's largest term e^0 = 1); v_exp_f32 adds ~1 ulp.
// Below that the absolute error is < 1e-7 * e^d.  exp(-inf) = 0 and
// exp(NaN) = NaN as in the reference.  (Measured: 87.2 -> 85.3 us on the
// 32768 x 2048 softmax.)
__device__ __forceinline__ float exp_diff(float d) { return __builtin_amdgcn_exp2f(d * 1.44269504f); }

// Number of leading columns of `row` that take part (causal mask).
template <SmKind K>
__device__ __forceinline__ uint64_t row_limit(const SmArgs& a, uint64_t row) {
    if (K != SmKind::Causal) return a.cols;
    const uint64_t lim = a.seq_offset + row + 1;  // host checked: no overflow
    return lim < a.cols ? lim : a.cols;
}

// Block-wide reduction of one value per wave through LDS, combined in wave
// order (deterministic).  `red` holds kSmWaves floats.
template <bool IsMax, int Waves = kSmWaves>
__device__ __forceinline__ float block_combine(float v, float* red) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    __syncthreads();  // previous readers of red are done
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int w = 1; w < Waves; ++w) r = IsMax ? fmaxf(r, red[w]) : r + red[w];
    return r;
}

// Row in registers.  Wave mode (Block = false): one wave per row, element f4
// index = c*64 + lane, 4 rows per 256-thread workgroup.  Block mode: one
// workgroup of BS threads per row, index = c*BS + tid.
// Ragged: rows of any length (from 4 floats) and alignment.  Their whole float4
// are read and written at dword alignment; float4 past the last one to read
// repeat it, so that the loads go out without a branch each; the row's last
// cols % 4 floats are one float each of its first threads (a branch a float4 for
// them cost more than few rows do: backward 64 x 513 3.17 us, 2.43 here, 2.26
// in the loop kernel's one float a thread).  Causal rows read only the float4
// that hold a column they keep.  Two operands of 16 float4 keep three waves a
// SIMD.
template <SmKind K, int NCH, bool Block, bool Ragged, int BS = kSmBlock>
__global__ __launch_bounds__(BS, NCH < 16 ? 1 : K == SmKind::Bwd ? 3 : 4) void softmax_reg_kernel(SmArgs a) {
    constexpr int kWavesB = BS / kWave;
    __shared__ float red[kWavesB];
    const int lane = threadIdx.x & (kWave - 1);
    // A scalar, so that row addresses live in SGPRs; but not for the backward's
    // 2049-4096 columns, whose waves it puts in step (2048 x 2500 8.7 -> 9.7 us).
    const bool lanes = K == SmKind::Bwd && NCH == 16;
    const int wave = lanes ? (int)(threadIdx.x / kWave) : __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const uint64_t row = Block ? (uint64_t)blockIdx.x : (uint64_t)blockIdx.x * kSmWaves + wave;
    if (!Block && row >= a.rows) return;  // uniform per wave; no block barrier in wave mode
    const int step = Block ? BS : kWave;
    const int me = Block ? (int)threadIdx.x : lane;
    const uint32_t cols = (uint32_t)a.cols;               // <= 16384 here
    const uint32_t lim = (uint32_t)row_limit<K>(a, row);  // <= cols
    const uint32_t whole4 = cols >> 2;
    // float4 to read: causal rows leave out those past their last column
    const uint32_t need4 = K == SmKind::Causal && (lim + 3u) >> 2 < whole4 ? (lim + 3u) >> 2 : whole4;
    const uint32_t lim4 = Ragged && lim > 4 * whole4 ? 4 * whole4 : lim;  // columns that take part and lie in whole float4
    const float* ar = a.a + row * cols;
    const float* br = a.b + row * cols;
    float* orow = a.out + row * cols;
    auto load = [&](const float* r, uint32_t f) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        if (Ragged)
            return (f32x4)__builtin_nontemporal_load(reinterpret_cast<const f32x4_a4*>(r) +
                                                     (f < need4 ? f : need4 - 1u));
        return f < need4 ? ld_stream(reinterpret_cast<const f32x4*>(r) + f) : zero;
    };
    auto store = [&](uint32_t f, f32x4 o) {
        if (f >= whole4) return;
        if (Ragged) __builtin_nontemporal_store((f32x4_a4)o, reinterpret_cast<f32x4_a4*>(orow) + f);
        else st_stream(reinterpret_cast<f32x4*>(orow) + f, o);
    };

    f32x4 v[NCH], g[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t f = (uint32_t)(c * step + me);
        v[c] = load(ar, f);
        if (K == SmKind::Bwd) g[c] = load(br, f);
    }
    // Ragged: this thread's one of the last floats, if any.
    const uint32_t tc = 4 * whole4 + (uint32_t)me;
    float tv = 0.0f, tg = 0.0f;
    if (Ragged && tc < lim) {
        tv = ar[tc];
        if (K == SmKind::Bwd) tg = br[tc];
    }

    if (K == SmKind::Bwd) {
        // dot = sum(y * dy); dx = y * (dy - dot)
        float dot = 0.0f;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const f32x4 p = v[c] * g[c];
            const float d = (p.x + p.y) + (p.z + p.w);
            dot += !Ragged || (uint32_t)(c * step + me) < whole4 ? d : 0.0f;
        }
        if (Ragged) dot += tv * tg;
        dot = wave_sum(dot);
        if (Block) dot = block_combine<false, kWavesB>(dot, red);
        if (Ragged && tc < cols) orow[tc] = tv * (tg - dot);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const uint32_t f = (uint32_t)(c * step + me);
            store(f, v[c] * (g[c] - dot));
        }
        return;
    }

    const float ninf = -__builtin_inff();
    float m = ninf;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t f = (uint32_t)(c * step + me);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool in = 4 * f + k < lim4;
            m = fmaxf(m, in ? f4_get(v[c], k) : ninf);
        }
    }
    if (Ragged) m = fmaxf(m, tc < lim ? tv : ninf);
    m = wave_max(m);
    if (Block) m = block_combine<true, kWavesB>(m, red);
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t f = (uint32_t)(c * step + me);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool in = 4 * f + k < lim4;
            const float e = in ? exp_diff(f4_get(v[c], k) - m) : 0.0f;
            f4_set(v[c], k, e);
            s += e;
        }
    }
    if (Ragged) {
        tv = tc < lim ? exp_diff(tv - m) : 0.0f;
        s += tv;
    }
    s = wave_sum(s);
    if (Block) s = block_combine<false, kWavesB>(s, red);
    const float inv = (K == SmKind::Causal) ? (s > 0.0f ? 1.0f / s : 0.0f) : 1.0f / s;
    if (K == SmKind::CeBwd) {
        const float inv_batch = a.inv_batch;
        const float scale = inv * inv_batch;
        // Through a vector load (the index is not a scalar): a scalar one leaves
        // the waves of a full chip in step, all storing at once (8192 x 900 10.4
        // us against 8.8, x 1024 10.7 against 9.0).
        const uint64_t vrow = Block ? row : (uint64_t)blockIdx.x * kSmWaves + threadIdx.x / kWave;
        const uint32_t t = (uint32_t)target_index(a.b[vrow], a.cols);  // none: past every column
        if (Ragged && tc < cols) orow[tc] = tc == t ? tv * scale - inv_batch : tv * scale;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const uint32_t f = (uint32_t)(c * step + me);
            f32x4 o = v[c] * scale;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (4 * f + k == t) f4_set(o, k, f4_get(o, k) - inv_batch);
            store(f, o);
        }
        return;
    }
    if (Ragged && tc < cols) orow[tc] = tv * inv;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t f = (uint32_t)(c * step + me);
        store(f, v[c] * inv);
    }
}

// Rows of 16385 to kLongCols floats (vocabularies): one workgroup of 1024
// threads holds the row, R float4 a thread in registers and the rest in LDS,
// and reads it once.  A CU's registers and LDS hold one such row, so its own
// arithmetic has to hide behind its own traffic: while the loads arrive a
// thread keeps a running max m and s = sum e^(x - m) (rescaled when a group of
// float4 raises m), and the values are exponentiated a second time, against
// the row's max, between the stores.  Thread i's float4 c is c * 1024 + i of
// the row; chunks past R go to LDS, and are loaded first, through the
// registers that the first chunks' loads then take over.
// Bound by HBM: 8 bytes a float.  2048 x 128256: 767 us in the loop kernel's
// three passes, 382 here (5.5 TB/s); x 50257 421 -> 157, x 20000 98 -> 56; 64 x
// 128256 103 -> 19.
constexpr int kLongThreads = 1024;
// float4 a thread: 96 of the 128 VGPRs that 16 waves leave (the causal kernels and
// the ragged cross-entropy one spill 4-7 VGPRs besides)
constexpr int kLongRegs = 24;
constexpr int kLongLds = 9;     // float4 a thread: 144 of the 160 KB
constexpr uint64_t kLongCols = 4ull * kLongThreads * (kLongRegs + kLongLds);

// Running max and sum of a thread's values; columns that take no part are -inf
// (they add 0).  A thread that has met nothing above -inf keeps s = 0 or NaN:
// the row's own max decides then.
struct Online {
    float m = -__builtin_inff();
    float s = 0.0f;
    // N float4; those with in[c] false repeat a value of the row and only leave
    // the max as it is.
    template <int N>
    __device__ __forceinline__ void add(const f32x4* v, const bool* in) {
        float mn = m;
#pragma unroll
        for (int c = 0; c < N; ++c) mn = fmaxf(fmaxf(mn, fmaxf(v[c].x, v[c].y)), fmaxf(v[c].z, v[c].w));
        s *= m == -__builtin_inff() ? 1.0f : exp_diff(m - mn);
        m = mn;
        const float base = mn == -__builtin_inff() ? 0.0f : mn;
#pragma unroll
        for (int c = 0; c < N; ++c) {
            const float t = (exp_diff(v[c].x - base) + exp_diff(v[c].y - base)) +
                            (exp_diff(v[c].z - base) + exp_diff(v[c].w - base));
            s += in[c] ? t : 0.0f;
        }
        // Used only past the block's barriers: the compiler would sink the
        // sums there and keep every term in a register until then.
        asm volatile("" : "+v"(m), "+v"(s));
    }
};

template <SmKind K, int R, bool Lds, bool Ragged>
__global__ __launch_bounds__(kLongThreads) void softmax_long_kernel(SmArgs a) {
    constexpr int kWavesB = kLongThreads / kWave;
    constexpr int kPre = Lds ? kLongLds : 0;  // LDS chunks, through v[0 .. kPre)
    constexpr int kGrp = 4;                   // float4 a rescaling
    constexpr uint32_t kChunk = 4 * kLongThreads;
    extern __shared__ f32x4 keep[];  // [LDS chunks][thread]
    __shared__ float red[kWavesB];
    const float ninf = -__builtin_inff();
    const uint32_t tid = threadIdx.x;
    const uint64_t row = blockIdx.x;
    const uint32_t cols = (uint32_t)a.cols;
    const uint32_t lim = (uint32_t)row_limit<K>(a, row);
    const uint32_t whole = cols & ~3u;  // columns in whole float4; a ragged row's last ones are one thread's `tail`
    const uint32_t need = K == SmKind::Causal && ((lim + 3u) & ~3u) < whole ? (lim + 3u) & ~3u : whole;
    const float* ar = a.a + row * cols;
    float* orow = a.out + row * cols;
    Online o;

    // Float4 past the ones to read repeat the last of them, so that no load is
    // conditional (a branch per load costs the registers this kernel lives on).
    const uint32_t last4 = (need >> 2) - 1u;
    auto load = [&](uint32_t c) {
        const uint32_t f = c * kLongThreads + tid;
        const uint32_t off = 16u * (f < last4 ? f : last4);
        const f32x4 r = __builtin_nontemporal_load(
            reinterpret_cast<const f32x4_a4*>(reinterpret_cast<const char*>(ar) + off));
        __builtin_amdgcn_sched_barrier(0);
        return r;
    };
    auto add = [&](auto N_, uint32_t c, f32x4* v) {
        constexpr int N = decltype(N_)::value;
        bool in[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const uint32_t f = (c + u) * kLongThreads + tid;
            in[u] = f <= last4;
            if (K == SmKind::Causal) {
#pragma unroll
                for (int k = 0; k < 4; ++k) f4_set(v[u], k, 4 * f + k < lim ? f4_get(v[u], k) : ninf);
            }
        }
        o.add<N>(v, in);
        __builtin_amdgcn_sched_barrier(0);
    };
    // The target's logit, read before any store: out may be the logits.
    const uint64_t t = (K == SmKind::CeBwd) ? target_index(a.b[row], a.cols) : ~0ull;
    const float xt = t < cols ? ar[t] : 0.0f;
    f32x4 v[R];
#pragma unroll
    for (int c = 0; c < R; ++c) v[c] = load(c < kPre ? R + c : c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kPre; ++c) {
        if ((uint32_t)(R + c) * kChunk < cols) keep[(uint32_t)c * kLongThreads + tid] = v[c];  // uniform
        add(std::integral_constant<int, 1>(), R + c, &v[c]);
        v[c] = load(c);
    }
    static_assert(R % kGrp == 0, "whole groups");
#pragma unroll
    for (int g = 0; g < R / kGrp; ++g) {
        // the chunks that were loaded first come first
        constexpr int kFirst = (kPre + kGrp - 1) / kGrp;
        const int c = (g + kFirst) % (R / kGrp) * kGrp;
        add(std::integral_constant<int, kGrp>(), c, &v[c]);
    }
    f32x4 tail = {ninf, ninf, ninf, ninf};
    if (Ragged) {
        if (tid == 0) {
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (whole + k < lim) f4_set(tail, k, ar[whole + k]);
        }
        const bool in = true;
        o.add<1>(&tail, &in);
    }
    const float m = block_combine<true, kWavesB>(wave_max(o.m), red);
    o.s *= o.m == ninf ? 1.0f : exp_diff(o.m - m);
    const float s = block_combine<false, kWavesB>(wave_sum(o.s), red);
    const float inv = (K == SmKind::Causal) ? (s > 0.0f ? 1.0f / s : 0.0f) : 1.0f / s;
    const float inv_batch = a.inv_batch;
    const float scale = (K == SmKind::CeBwd) ? inv * inv_batch : inv;
    auto value = [&](uint32_t f, f32x4 x) {  // outputs of float4 f
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float e = exp_diff(f4_get(x, k) - m) * scale;
            f4_set(x, k, K != SmKind::Causal || 4 * f + k < lim ? e : 0.0f * scale);
        }
        return x;
    };
    auto store = [&](uint32_t c, f32x4 x) {
        const uint32_t first = c * kChunk;
        const uint32_t n4 = whole > first ? (whole - first) >> 2 : 0u;
        x = value(c * kLongThreads + tid, x);
        if (tid < n4) __builtin_nontemporal_store((f32x4_a4)x, reinterpret_cast<f32x4_a4*>(orow + first) + tid);
    };
#pragma unroll
    for (int c = 0; c < R; ++c) {
        store(c, v[c]);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (Lds) {
        for (uint32_t c = R; c * kChunk < whole; ++c) store(c, keep[(c - R) * kLongThreads + tid]);
    }
    if (Ragged && tid == 0) {
        tail = value(whole >> 2, tail);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (whole + k < cols) orow[whole + k] = f4_get(tail, k);
    }
    // The thread that stored the target's column stores it once more.
    if (K == SmKind::CeBwd && t < cols && tid == (t < whole ? (uint32_t)(t >> 2) % kLongThreads : 0u))
        orow[t] = exp_diff(xt - m) * scale - inv_batch;
}

// Any row length and alignment: one workgroup per row, the row streamed
// three times (max, sum, write) -- or twice for the backward.  Vec = float4
// accesses (cols % 4 == 0 and aligned views), else scalar.
template <SmKind K, bool Vec>
__global__ __launch_bounds__(kSmBlock) void softmax_loop_kernel(SmArgs a) {
    __shared__ float red[kSmWaves];
    const uint64_t row = blockIdx.x;
    const uint64_t lim = row_limit<K>(a, row);
    const float* ar = a.a + row * a.cols;
    const float* br = a.b + row * a.cols;
    float* orow = a.out + row * a.cols;
    const uint64_t n = Vec ? a.cols >> 2 : a.cols;
    const float ninf = -__builtin_inff();

    if (K == SmKind::Bwd) {
        float dot = 0.0f;
        for (uint64_t i = threadIdx.x; i < n; i += kSmBlock) {
            if (Vec) {
                const f32x4 p = reinterpret_cast<const f32x4*>(ar)[i] * reinterpret_cast<const f32x4*>(br)[i];
                dot += (p.x + p.y) + (p.z + p.w);
            } else {
                dot += ar[i] * br[i];
            }
        }
        dot = block_combine<false>(wave_sum(dot), red);
        for (uint64_t i = threadIdx.x; i < n; i += kSmBlock) {
            if (Vec) {
                const f32x4 y = reinterpret_cast<const f32x4*>(ar)[i];
                const f32x4 g = reinterpret_cast<const f32x4*>(br)[i];
                st_stream(reinterpret_cast<f32x4*>(orow) + i, y * (g - dot));
            } else {
                orow[i] = ar[i] * (br[i] - dot);
            }
        }
        return;
    }

    float m = ninf;
    for (uint64_t i = threadIdx.x; i < n; i += kSmBlock) {
        if (Vec) {
            const f32x4 v = reinterpret_cast<const f32x4*>(ar)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) m = fmaxf(m, 4 * i + k < lim ? f4_get(v, k) : ninf);
        } else {
            m = fmaxf(m, i < lim ? ar[i] : ninf);
        }
    }
    m = block_combine<true>(wave_max(m), red);
    float s = 0.0f;
    for (uint64_t i = threadIdx.x; i < n; i += kSmBlock) {
        if (Vec) {
            const f32x4 v = reinterpret_cast<const f32x4*>(ar)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) s += 4 * i + k < lim ? exp_diff(f4_get(v, k) - m) : 0.0f;
        } else {
            s += i < lim ? exp_diff(ar[i] - m) : 0.0f;
        }
    }
    s = block_combine<false>(wave_sum(s), red);
    const float inv = (K == SmKind::Causal) ? (s > 0.0f ? 1.0f / s : 0.0f) : 1.0f / s;
    const float inv_batch = a.inv_batch;
    const float scale = (K == SmKind::CeBwd) ? inv * inv_batch : inv;
    const uint64_t t = (K == SmKind::CeBwd) ? target_index(a.b[row], a.cols) : ~0ull;
    for (uint64_t i = threadIdx.x; i < n; i += kSmBlock) {
        if (Vec) {
            f32x4 v = reinterpret_cast<const f32x4*>(ar)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float o = (4 * i + k < lim ? exp_diff(f4_get(v, k) - m) : 0.0f) * scale;
                if (K == SmKind::CeBwd && 4 * i + k == t) o = o - inv_batch;
                f4_set(v, k, o);
            }
            st_stream(reinterpret_cast<f32x4*>(orow) + i, v);
        } else {
            float o = (i < lim ? exp_diff(ar[i] - m) : 0.0f) * scale;
            if (K == SmKind::CeBwd && i == t) o = o - inv_batch;
            orow[i] = o;
        }
    }
}

template <SmKind K, int NCH, bool Ragged>
static void launch_wave(const SmArgs& a, hipStream_t s) {
    const uint64_t blocks = (a.rows + kSmWaves - 1) / kSmWaves;
    hipLaunchKernelGGL((softmax_reg_kernel<K, NCH, false, Ragged>), dim3((uint32_t)blocks), dim3(kSmBlock), 0, s, a);
}

template <SmKind K, int R, bool Ragged>
static void launch_long(const SmArgs& a, hipStream_t s) {
    constexpr bool kLds = R == kLongRegs;
    const uint64_t chunks = ((a.cols + 3) / 4 + kLongThreads - 1) / kLongThreads;
    const size_t lds = chunks > (uint64_t)R ? (chunks - R) * kLongThreads * sizeof(f32x4) : 0;
    hipLaunchKernelGGL((softmax_long_kernel<K, R, kLds, Ragged>), dim3((uint32_t)a.rows), dim3(kLongThreads), lds, s, a);
}

template <SmKind K, int NCH, bool Ragged, int BS>
static void launch_block(const SmArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((softmax_reg_kernel<K, NCH, true, Ragged, BS>), dim3((uint32_t)a.rows), dim3(BS), 0, s, a);
}

template <SmKind K, bool Ragged>
static void launch_loop(const SmArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((softmax_loop_kernel<K, !Ragged>), dim3((uint32_t)a.rows), dim3(kSmBlock), 0, s, a);
}

// 513-1024 columns in a workgroup of 128 threads x 2 float4 per row instead of a
// wave x 4 of each of four rows, whose workgroup ends with its slowest row.
// Graph replays, us, wave against workgroup (so below too): ragged backward 64 x
// 767 2.27 -> 2.17, 2300 x 1023 6.2 -> 5.6 (16368 x 513 18.2 against 19.7);
// ragged forward from 769 columns, 16368 x 1023 25.7 -> 24.3, as up to 768 a
// quarter of the workgroup idles (8000 x 600 8.6 against 9.4).  Whole rows only
// where they fill it (512 x 964 3.3 against 3.5) and while its rounds are few: 64
// x 1024 2.55 -> 2.31, 2560 4.46 -> 4.31, but 3300 4.89 against 5.15 and 5120 5.7
// against 7.6 (softmax 16368 22.7 -> 21.5 again, logits 20.3 against 21.5); backward 1536 x 1024 4.25 -> 3.93, but 2048 4.9 against 5.4.
template <SmKind K, bool Ragged>
static bool two_waves_a_row(uint64_t rows, uint64_t cols4) {
    if (Ragged) return cols4 > (K == SmKind::Bwd ? 128u : 192u);
    if (cols4 != 256) return false;
    if (K == SmKind::Fwd || K == SmKind::Causal) return rows <= 2560 || rows >= 12288;
    return rows <= (K == SmKind::Bwd ? 1536u : 2560u);
}

// 2049-4096 columns.  Forward: 256 threads x 4 float4 per row (512 x 2, half of
// them idle at 2052 columns, against it: 1100 x 2052 6.2 -> 5.2, 8192 27.6 ->
// 25.3), but one wave a row where that many waves still fit the chip at once and
// the workgroups take another round (2900 x 2052 9.1 against 10.3; 1100 6.7
// against 5.2, 4500 16.0 against 14.8; ragged 2900 x 2049 9.2 against 10.6, 2048
// 7.8 against 6.9, 3300 13.1 against 11.5; whole rows to 4096 where they are
// short: 4096 x 2052 12.0 against 13.5, but x 3072 19.5 against 18.7), and 512 threads for many wide rows
// (8192 x 4096 44.4 against 46.8).  Backward: 256 threads for ragged rows (1100 x
// 3001 8.3 with 512, 7.8), 512 for whole ones (8192 x 3072 49.9 with a wave a
// row, 46.4), a wave where the rows are about one or two a SIMD (1024 x 2052
// 5.55 against 5.92, 2048 x 2052 7.0 against 8.5; 768 4.97 against 4.48, 3072
// 13.2 against 12.4).
enum class MidForm { Wave, Group256, Group512 };
template <SmKind K, bool Ragged>
static MidForm mid_form(uint64_t rows, uint64_t cols4) {
    if (K == SmKind::Bwd && !Ragged) return rows > 768 && rows < 3072 ? MidForm::Wave : MidForm::Group512;
    const uint64_t last = !Ragged && cols4 <= 640 ? 4096 : 3072;
    if (K != SmKind::Bwd && rows > (Ragged ? 2304u : 1536u) && rows <= last) return MidForm::Wave;
    return rows > 3072 && cols4 > 768 ? MidForm::Group512 : MidForm::Group256;
}

// The kernel for the row length.
template <SmKind K, bool Ragged>
static void softmax_dispatch(const SmArgs& a, hipStream_t s) {
    constexpr bool kBwd = K == SmKind::Bwd;
    const uint64_t cols4 = (a.cols + 3) / 4;
    // Ragged backward, up to 512 columns and few rows: a thread a float, the row
    // read twice from the cache (512 x 255 2.14 against 2.37, 1792 x 255 2.69
    // against 2.86; 2300 x 255 3.1 against 3.0, x 511 4.1 against 3.7).
    if (kBwd && Ragged && cols4 <= 128 && a.rows <= 1792) launch_loop<K, Ragged>(a, s);
    else if (cols4 <= 64) launch_wave<K, 1, Ragged>(a, s);
    else if (cols4 <= 128) launch_wave<K, 2, Ragged>(a, s);
    else if (cols4 <= 256 && two_waves_a_row<K, Ragged>(a.rows, cols4)) launch_block<K, 2, Ragged, 128>(a, s);
    else if (cols4 <= 256) launch_wave<K, 4, Ragged>(a, s);
    else if (cols4 <= 512) {
        // 1025-2048 columns: one workgroup per row streams faster than one
        // wave per row (measured at 32768 x 2048: forward 85.8 -> 83.3 us
        // with 256 threads x 2 float4, backward 129.3 -> 121.7 us with 512
        // threads x 1 float4 each of y and dy; ragged backward 1100 x 1025 4.0
        // with 512, 3.5 with 256)
        if constexpr (kBwd && !Ragged) launch_block<K, 1, Ragged, 512>(a, s);
        else launch_block<K, 2, Ragged, 256>(a, s);
    }
    else if (cols4 <= 1024) {
        switch (mid_form<K, Ragged>(a.rows, cols4)) {
        case MidForm::Wave:  // not for ragged backward rows
            if constexpr (!kBwd || !Ragged) return launch_wave<K, 16, Ragged>(a, s);
            [[fallthrough]];
        case MidForm::Group256:  // not for whole ones
            if constexpr (!kBwd || Ragged) return launch_block<K, 4, Ragged, 256>(a, s);
            [[fallthrough]];
        case MidForm::Group512: return launch_block<K, 2, Ragged, 512>(a, s);
        }
    }
    else if (cols4 <= 2048) launch_block<K, 8, Ragged, 256>(a, s);
    else if (cols4 <= 4096) {
        // 8193-16384 columns: 512 threads while the rows are few (512 x 16384
        // 12.0 -> 10.9 us, 300 x 9000 7.3 -> 6.7, 64 x 12345 6.6 -> 5.5; 1024 x
        // 12288 logits 18.2 against 20.2, and 300 x 9000 backward 8.2 against 8.6).
        if constexpr (!kBwd) {
            if (a.rows <= 512) return launch_block<K, 8, Ragged, 512>(a, s);
        }
        launch_block<K, 16, Ragged, 256>(a, s);
    }
    else if (!kBwd && a.cols <= kLongCols) {
        if constexpr (!kBwd) {
            if (cols4 <= 8 * kLongThreads) launch_long<K, 8, Ragged>(a, s);
            else if (cols4 <= 16 * kLongThreads) launch_long<K, 16, Ragged>(a, s);
            else launch_long<K, kLongRegs, Ragged>(a, s);
        }
    }
    else launch_loop<K, Ragged>(a, s);
}

template <SmKind K>
static int softmax_launch(const SmArgs& a, hipStream_t s) {
    if (a.rows == 0 || a.cols == 0) return KORE_HIP_OK;
    if (!a.a || !a.out || ((K == SmKind::Bwd || K == SmKind::CeBwd) && !a.b)) return KORE_HIP_ERR_NULL_PTR;
    uint64_t elems;
    if (!mul_ok(a.rows, a.cols, &elems) || elems > kMaxElements || a.rows > 0x7fffffffull)
        return KORE_HIP_ERR_OVERFLOW;
    if (K == SmKind::Causal && a.seq_offset + a.rows < a.seq_offset) return KORE_HIP_ERR_OVERFLOW;
    const bool aligned = (a.cols % 4 == 0) && aligned16(a.a) && aligned16(a.out) &&
                         (K != SmKind::Bwd || aligned16(a.b));
    SmArgs band = a;
    band.inv_batch = 1.0f / (float)a.rows;
    for (uint64_t left = a.rows; left > 0;) {
        band.rows = left < kLaunchRows ? left : kLaunchRows;
        if (aligned)
            softmax_dispatch<K, false>(band, s);
        else if (a.cols >= 4)
            softmax_dispatch<K, true>(band, s);
        else  // ragged rows are read four floats at a time
            launch_loop<K, true>(band, s);
        left -= band.rows;
        band.a += band.rows * a.cols;
        band.out += band.rows * a.cols;
        if (K == SmKind::Bwd) band.b += band.rows * a.cols;
        if (K == SmKind::CeBwd) band.b += band.rows;
        band.seq_offset += band.rows;
    }
    return launch_status();
}

}  // namespace kore

using namespace kore;

extern "C" int kore_hip_softmax_f32(const float* x, float* out, uint64_t rows, uint64_t cols,
                                    kore_stream_t stream) {
    SmArgs a{x, nullptr, out, rows, cols, 0};
    return softmax_launch<SmKind::Fwd>(a, (hipStream_t)stream);
}

extern "C" int kore_hip_softmax_causal_f32(const float* x, float* out, uint64_t rows, uint64_t cols,
                                           uint64_t seq_offset, kore_stream_t stream) {
    SmArgs a{x, nullptr, out, rows, cols, seq_offset};
    return softmax_launch<SmKind::Causal>(a, (hipStream_t)stream);
}

extern "C" int kore_hip_softmax_backward_f32(const float* grad_out, const float* out, float* grad_in,
                                             uint64_t rows, uint64_t cols, kore_stream_t stream) {
    SmArgs a{out, grad_out, grad_in, rows, cols, 0};
    return softmax_launch<SmKind::Bwd>(a, (hipStream_t)stream);
}

extern "C" int kore_hip_cross_entropy_backward_f32(const float* logits, const float* targets, float* grad_logits,
                                                   uint64_t batch, uint64_t num_classes, kore_stream_t stream) {
    SmArgs a{logits, targets, grad_logits, batch, num_classes, 0};
    return softmax_launch<SmKind::CeBwd>(a, (hipStream_t)stream);
}
