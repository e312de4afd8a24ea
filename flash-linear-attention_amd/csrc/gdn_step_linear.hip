// The projections of a decode step of the layer (fla/layers/gated_deltanet.py:246-300 at one token per sequence): up to six linear
// maps of the same few rows x [N][hidden] in one launch, y = x W^T with W [cols][hidden] as nn.Linear keeps it, each with what the
// layer does to its result next:
//   PLAIN  y in x's type                                  CONV   the causal convolution's one-token update and SiLU on top of y
//   GATE   -exp(A_log) softplus(y + dt_bias), fp32        BETA   sigmoid(y) (or twice that), fp32
// y is rounded to x's type before any of them, as the tensor it stands for is.
//
// A step reads every weight once and little else, so it is bound by how much of the weights is in flight: a workgroup takes 16 (32)
// output columns, its eight waves an eighth of the contraction each, all operand fragments straight from memory (a lane: 16 bytes of
// one row; x comes from the L2), the partial sums through LDS.  More than 128 rows are taken 128 at a time by workgroups of their own
// (a workgroup's tiles of rows share its registers with the weights' fragments); the weights then come from the L2 and the cache behind it.
// Up to 16 rows have a kernel of their own (gdn_step_linear_few_kernel).
#include "gdn_chunk_common.h"

namespace gdn {

struct StepLinearParams {
    const void* x;
    int N, hidden, nseg;
    gdn_step_segment seg[GDN_STEP_SEGMENTS];
    int first[GDN_STEP_SEGMENTS + 1];            // a segment's first workgroup
    int columns;                                 // a workgroup's output columns (gdn_step_linear_few_kernel)
};

// What becomes of y = (row n, column d) of a segment.  `old`, `wt`: the convolution's state and weights where it has four taps.
template <typename T>
__device__ __forceinline__ void step_result(const gdn_step_segment& s, int cols, int n, int d, float sum, typename Mma<T>::V4 old, typename Mma<T>::V4 wt) {
    const T yt = from_f32<T>(sum);
    const float y = to_f32(yt);
    if (s.kind == GDN_STEP_PLAIN) {
        ((T*)s.out)[(int64_t)n * cols + d] = yt;
    } else if (s.kind == GDN_STEP_CONV) {
        const int W = s.conv_size;
        T* st = (T*)s.conv_state + ((int64_t)n * cols + d) * W;
        const T* cw = (const T*)s.conv_weight + (int64_t)d * W;
        float win[8], a = 0.f;
        if (W == 4) {
            typedef typename Mma<T>::V4 V4;
#pragma unroll
            for (int e = 0; e < 3; ++e) a += to_f32(old[e + 1]) * to_f32(wt[e]);
            a += y * to_f32(wt[3]);
            *(V4*)st = V4{old[1], old[2], old[3], yt};
        } else {
            for (int e = 0; e < W; ++e) win[e & 7] = e + 1 < W ? to_f32(st[e + 1]) : y;
            for (int e = 0; e < W; ++e) { a += win[e & 7] * to_f32(cw[e]); st[e] = from_f32<T>(win[e & 7]); }
        }
        if (s.conv_bias) a += to_f32(((const T*)s.conv_bias)[d]);
        a = a * sigmoid_stream(a);
        ((T*)s.out)[(int64_t)n * cols + d] = from_f32<T>(a);
    } else if (s.kind == GDN_STEP_GATE) {
        const float A = load_scalar(s.A_log, d, s.gate_dtype), dt = s.dt_bias ? load_scalar(s.dt_bias, d, s.gate_dtype) : 0.f;
        ((float*)s.out)[(int64_t)n * cols + d] = -__expf(A) * softplus_f(y + dt);
    } else {
        ((float*)s.out)[(int64_t)n * cols + d] = (s.kind == GDN_STEP_BETA2 ? 2.f : 1.f) * sigmoid_f(y);
    }
}

// Up to 16 rows.  A workgroup of sixteen (short contractions: eight) waves takes `columns` output columns (a multiple of 8 up to 16 CT), each
// wave an equal part of the contraction, and everything that it needs from memory is requested before anything is waited for: four steps of 32 of the weights and
// of x (all of a contraction of 2048), the convolution's states and weights.  The rows of x are as many bytes as sixteen columns of
// weights, so a workgroup takes as many columns as leave every CU one (launch_step_linear).  16 rows, the six projections of the default layer
// (9228 columns of 2048: 40 columns to a workgroup): 14.3 us with 16 columns and eight waves, half of the loads at a time, 11.4 us (37.8 MB);
// its output projection (2048 columns of 3072: 8) 7.2 -> 6.8 us, the layer's step 45.1 -> 40.8 us.  The gated norm inside the output projection -
// every workgroup would bring all rows of x through it - made that 16.6 us, against 7.2 + 4.6 in a launch of its own.
// The line at 16 rows is one matrix tile of them, not a measured one: this form has not been tried with more tiles.
template <typename T, int CT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gdn_step_linear_few_kernel(StepLinearParams p) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int PITCH = 16 * CT + 4, U = 4;
    static_assert(16 * CT <= 4 * WAVES, "a thread a result");
    __shared__ __align__(16) float part[WAVES][16][PITCH];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
    int si = 0;
    while (si + 1 < p.nseg && (int)blockIdx.x >= p.first[si + 1]) ++si;
    const gdn_step_segment s = p.seg[si];
    const int TC = p.columns, col0 = ((int)blockIdx.x - p.first[si]) * TC, cols = (int)s.cols, hidden = p.hidden;

    // this thread's result: row r of x, column j of the workgroup's
    const int r = tid / TC, j = tid - r * TC, d = col0 + j;
    const bool mine = r < p.N && d < cols;                       // (p.N <= 16)
    V4 old{}, wt{};
    if (mine && s.kind == GDN_STEP_CONV && s.conv_size == 4) {
        old = *(const V4*)((const T*)s.conv_state + ((int64_t)r * cols + d) * 4);
        wt = *(const V4*)((const T*)s.conv_weight + (int64_t)d * 4);
    }
    // this wave's steps of 32
    const int steps = hidden / 32, s0 = w * steps / WAVES, s1 = (w + 1) * steps / WAVES;
    // (rows past the end repeat the last one, columns past the workgroup's its last: their results are dropped)
    const int last = min(col0 + TC, cols) - 1;
    const T* xr = (const T*)p.x + (int64_t)min(c16, p.N - 1) * hidden + 8 * g;
    const T* wr[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) wr[c] = (const T*)s.weight + (int64_t)min(col0 + 16 * c + c16, last) * hidden + 8 * g;
    f32x4 acc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = s0; k < s1; k += U) {
        V8 fw[CT][U], fx[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < s1) {                                    // (the same for the wave)
#pragma unroll
                for (int c = 0; c < CT; ++c) fw[c][u] = *(const V8*)(wr[c] + 32 * (k + u));
            }
#pragma unroll
        for (int u = 0; u < U; ++u) if (k + u < s1) fx[u] = *(const V8*)(xr + 32 * (k + u));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < s1) {
#pragma unroll
                for (int c = 0; c < CT; ++c) acc[c] = Mma<T>::run(fw[c][u], fx[u], acc[c]);
            }
    }
    // lane (c16, g): row c16, columns 4g .. 4g + 3 of each tile
#pragma unroll
    for (int c = 0; c < CT; ++c) *(f32x4*)&part[w][c16][16 * c + 4 * g] = acc[c];
    __syncthreads();
    if (!mine) return;
    float sum = 0.f;
#pragma unroll
    for (int x = 0; x < WAVES; ++x) sum += part[x][r][j];
    step_result<T>(s, cols, r, d, sum, old, wt);
}

// NT: tiles of 16 rows, CT: tiles of 16 columns per workgroup; blockIdx.y: 16 NT rows each
template <typename T, int NT, int CT>
__global__ __launch_bounds__(512) void gdn_step_linear_kernel(StepLinearParams p) {
    typedef typename Mma<T>::V8 V8;
    constexpr int WAVES = 8, PITCH = 20;
    __shared__ __align__(16) float part[WAVES][NT * 16][PITCH];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
    int si = 0;
    while (si + 1 < p.nseg && (int)blockIdx.x >= p.first[si + 1]) ++si;
    const gdn_step_segment s = p.seg[si];
    const int col0 = ((int)blockIdx.x - p.first[si]) * 16 * CT, cols = (int)s.cols;
    const int hidden = p.hidden, kw = hidden / WAVES, row0 = (int)blockIdx.y * 16 * NT;

    f32x4 acc[CT][NT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // (rows past the end repeat the last one: their results are dropped)
    const T* wr[CT]; const T* xr[NT];
#pragma unroll
    for (int c = 0; c < CT; ++c) wr[c] = (const T*)s.weight + (int64_t)min(col0 + 16 * c + c16, cols - 1) * hidden + w * kw + 8 * g;
#pragma unroll
    for (int t = 0; t < NT; ++t) xr[t] = (const T*)p.x + (int64_t)min(row0 + 16 * t + c16, p.N - 1) * hidden + w * kw + 8 * g;
    constexpr int U = NT >= 8 ? 2 : 4;           // steps of 32 requested together
    for (int k = 0; k < kw; k += 32 * U) {
        V8 fw[CT][U], fx[NT][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + 32 * u >= kw) break;         // (the same for the workgroup)
#pragma unroll
            for (int c = 0; c < CT; ++c) fw[c][u] = *(const V8*)(wr[c] + k + 32 * u);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + 32 * u >= kw) break;
#pragma unroll
            for (int t = 0; t < NT; ++t) fx[t][u] = *(const V8*)(xr[t] + k + 32 * u);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + 32 * u >= kw) break;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int c = 0; c < CT; ++c) acc[c][t] = Mma<T>::run(fw[c][u], fx[t][u], acc[c][t]);
        }
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        if (c > 0) __syncthreads();
        // lane (c16, g): row 16t + c16, columns 4g .. 4g + 3 of the tile
#pragma unroll
        for (int t = 0; t < NT; ++t) *(f32x4*)&part[w][16 * t + c16][4 * g] = acc[c][t];
        __syncthreads();
        for (int i = tid; i < NT * 256; i += 512) {
            const int r = i >> 4, n = row0 + r, j = i & 15, d = col0 + 16 * c + j;
            if (n >= p.N || d >= cols) continue;
            float sum = 0.f;
#pragma unroll
            for (int x = 0; x < WAVES; ++x) sum += part[x][r][j];
            typedef typename Mma<T>::V4 V4;
            V4 old{}, wt{};
            if (s.kind == GDN_STEP_CONV && s.conv_size == 4) {
                old = *(const V4*)((const T*)s.conv_state + ((int64_t)n * cols + d) * 4);
                wt = *(const V4*)((const T*)s.conv_weight + (int64_t)d * 4);
            }
            step_result<T>(s, cols, n, d, sum, old, wt);
        }
    }
}

template <typename T>
static int launch_step_linear(StepLinearParams& p, hipStream_t stream) {
    auto go = [&](auto kern, const char* name, int threads, int columns, int rows) {
        int at = 0;
        for (int i = 0; i < p.nseg; ++i) { p.first[i] = at; at += (int)((p.seg[i].cols + columns - 1) / columns); }
        p.first[p.nseg] = at;
        hipLaunchKernelGGL(kern, dim3((unsigned)at, (unsigned)((p.N + rows - 1) / rows)), dim3((unsigned)threads), 0, stream, p);
        return check_launch(name);
    };
    if (p.N <= 16) {
        // rounds of the chip's CUs times the bytes of a workgroup, in columns of weights
        unsigned best = 8, cost = ~0u;
        for (unsigned c = 8; c <= 48; c += 8) {
            unsigned groups = 0;
            for (int i = 0; i < p.nseg; ++i) {
                const unsigned n = (unsigned)p.seg[i].cols;
                if (n >= c) groups += (n + c - 1) / c;           // (a few columns ride along)
            }
            const unsigned x = (groups + 255) / 256 * (c + 16);
            if (x < cost) { cost = x; best = c; }
        }
        p.columns = (int)best;
        const char* name = "gdn_step_linear_few_kernel";
        if (p.hidden <= 1024 && best <= 32)
            return best <= 16 ? go(gdn_step_linear_few_kernel<T, 1, 8>, name, 512, (int)best, 16) : go(gdn_step_linear_few_kernel<T, 2, 8>, name, 512, (int)best, 16);
        return best <= 16 ? go(gdn_step_linear_few_kernel<T, 1, 16>, name, 1024, (int)best, 16) : best <= 32 ? go(gdn_step_linear_few_kernel<T, 2, 16>, name, 1024, (int)best, 16)
                                                                                                             : go(gdn_step_linear_few_kernel<T, 3, 16>, name, 1024, (int)best, 16);
    }
    const char* name = "gdn_step_linear_kernel";
    if (p.N <= 32) return go(gdn_step_linear_kernel<T, 2, 1>, name, 512, 16, 32);
    // (more rows: 32 columns, so that the rows of x are read half as often)
    if (p.N <= 64) return go(gdn_step_linear_kernel<T, 4, 2>, name, 512, 32, 64);
    return go(gdn_step_linear_kernel<T, 8, 2>, name, 512, 32, 128);
}

}  // namespace gdn

extern "C" int gdn_step_linear(const void* x, int64_t N, int64_t hidden, const gdn_step_segment* segs, int nseg, int dtype, void* stream) {
    using namespace gdn;
    const char* who = "gdn_step_linear";
    GDN_CHECK_ARG(x && segs && nseg >= 1 && nseg <= GDN_STEP_SEGMENTS, GDN_ERR_INVALID, "%s: x and 1 to %d segments are required", who, GDN_STEP_SEGMENTS);
    GDN_CHECK_ARG(N >= 1 && N <= GDN_STEP_MAX_ROWS && hidden >= 256 && hidden % 256 == 0 && hidden <= GDN_STEP_MAX_COLS, GDN_ERR_UNSUPPORTED,
                  "%s: 1 to %d rows of a multiple of 256 elements (got %lld x %lld)", who, GDN_STEP_MAX_ROWS, (long long)N, (long long)hidden);
    GDN_CHECK_ARG(dtype == GDN_DTYPE_BF16 || dtype == GDN_DTYPE_F16, GDN_ERR_UNSUPPORTED, "%s: bf16 or f16 only", who);
    StepLinearParams p;
    p.x = x; p.N = (int)N; p.hidden = (int)hidden; p.nseg = nseg;
    GDN_CHECK_ARG((uintptr_t)x % 16 == 0, GDN_ERR_INVALID, "%s: x must be 16-byte aligned", who);
    for (int i = 0; i < nseg; ++i) {
        const gdn_step_segment& s = segs[i];
        GDN_CHECK_ARG(s.weight && s.out && s.cols >= 1 && s.cols <= GDN_STEP_MAX_COLS && (uintptr_t)s.weight % 16 == 0, GDN_ERR_INVALID,
                      "%s: segment %d needs a 16-byte aligned weight and an output", who, i);
        GDN_CHECK_ARG(s.kind >= GDN_STEP_PLAIN && s.kind <= GDN_STEP_BETA2, GDN_ERR_INVALID, "%s: segment %d is of no known kind", who, i);
        GDN_CHECK_ARG(s.kind != GDN_STEP_CONV || (s.conv_weight && s.conv_state && s.conv_size >= 1 && s.conv_size <= 8 &&
                                                  ((uintptr_t)s.conv_weight | (uintptr_t)s.conv_state) % 8 == 0), GDN_ERR_INVALID,
                      "%s: segment %d needs convolution weights and a state of 1 to 8 taps, 8-byte aligned", who, i);
        GDN_CHECK_ARG(s.kind != GDN_STEP_GATE || s.A_log, GDN_ERR_INVALID, "%s: segment %d needs A_log", who, i);
        p.seg[i] = s;
    }
    return dtype == GDN_DTYPE_BF16 ? launch_step_linear<bf16_t>(p, (hipStream_t)stream) : launch_step_linear<f16_t>(p, (hipStream_t)stream);
}
