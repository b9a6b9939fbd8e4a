// y[M, N] = x[M, K] * W[N, K]^T (+ bias[N]): the linear layer of
// nanovllm/layers/linear.py:51,73,153 and the output head of embed_head.py:61, with the weight
// in its stored [out, in] layout.
//
// It is the matrix product of the 32-bit path, whose operands are read as they are stored and whose products and sums are
// float operations, and accepts any M, N, K.  Each output is one chain over k whatever M is and whichever tile shape runs:
// the result does not depend on the batch.  The result is written as elements or, for logits, as float.
//
// float32 runs on the matrix cores (below).  For bfloat16 operands this is the fallback for shapes that the other product
// kernels refuse, on the vector units: a workgroup of 256 threads takes BM rows of x and BN rows of W; a thread TM x TN
// outputs, in groups of up to four consecutive rows and columns BM / GM and BN / GN apart (the reads of LDS are then 16
// bytes per lane, neighbours side by side).  The tiles of x and W go through LDS k-major, BK columns at a time, in two
// buffers: the next tile's global loads are on their way while this one is multiplied, one barrier per tile.  Four shapes:
// 128 x 128 where that gives every CU a workgroup, else 64 x 64; for the few rows of a decode step, where W is streamed
// once, 16 x 64 with tiles of 64 columns (four rows a thread: its reads of x are one broadcast), or 16 x 16 where W has too
// few rows to give every CU a workgroup of 64 of them.
#include "common.h"

#if !defined(NVA_F32)
template <typename T>
__device__ __forceinline__ void load4(const T* __restrict__ p, bool whole, int k_left, float v[4]) {
    if (whole) {
        if (sizeof(T) == 4) {
            const float4 f = *reinterpret_cast<const float4*>(p);
            v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        } else {
            typedef __attribute__((ext_vector_type(4))) __bf16 b4;
            const b4 f = *reinterpret_cast<const b4*>(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = static_cast<float>(f[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = e < k_left ? to_float(p[e]) : 0.f;
    }
}

// R rows x BK columns of a matrix, from its row `row0` and column k0, as 4-column pieces: piece p of
// a thread is number tid + 256 p; its row is number / (BK / 4).  Rows and columns past the end are zeros.
template <typename T, int R, int BK>
struct TileLoad {
    static constexpr int PIECES = R * BK / 4 / 256;
    static_assert(R * BK / 4 % 256 == 0 && PIECES >= 1, "a tile is a whole number of pieces per thread");
    float v[PIECES][4];
    __device__ __forceinline__ void fetch(const T* __restrict__ src, int64_t stride, int rows_left, int k_left, bool vec, int tid) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int n = tid + 256 * p, r = n / (BK / 4), kq = (n % (BK / 4)) * 4;
            if (r < rows_left && kq < k_left) {
                load4<T>(src + (int64_t)r * stride + kq, vec && kq + 4 <= k_left, k_left - kq, v[p]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[p][e] = 0.f;
            }
        }
    }
    __device__ __forceinline__ void store(float (*dst)[R + 4], int tid) const {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int n = tid + 256 * p, r = n / (BK / 4), kq = (n % (BK / 4)) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[kq + e][r] = v[p][e];
        }
    }
};

template <typename T, typename OutT, int BM, int BN, int BK, int TM, int TN>
__global__ void __launch_bounds__(256, 2)
linear_tiled_kernel(const T* __restrict__ x, int64_t x_stride, const T* __restrict__ w, int64_t w_stride,
                    const T* __restrict__ bias, OutT* __restrict__ y, int64_t y_stride, int M, int N, int K,
                    int vec) {
    constexpr int VM = TM >= 4 ? 4 : TM, GM = TM / VM;       // a thread's rows: GM groups of VM consecutive ones
    constexpr int VN = TN >= 4 ? 4 : TN, GN = TN / VN;
    constexpr int TX = BN / TN;                               // threads side by side along n
    static_assert((BM / TM) * TX == 256, "256 threads cover the tile");
    __shared__ float xs[2][BK][BM + 4];
    __shared__ float ws[2][BK][BN + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int ty = tid / TX, tx = tid % TX;
    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;

    TileLoad<T, BM, BK> lx;
    TileLoad<T, BN, BK> lw;
    const T* xp = x + (int64_t)m0 * x_stride;
    const T* wp = w + (int64_t)n0 * w_stride;
    lx.fetch(xp, x_stride, M - m0, K, vec, tid);
    lw.fetch(wp, w_stride, N - n0, K, vec, tid);
    lx.store(xs[0], tid);
    lw.store(ws[0], tid);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += BK) {
        const bool more = k0 + BK < K;
        if (more) {
            lx.fetch(xp + k0 + BK, x_stride, M - m0, K - k0 - BK, vec, tid);
            lw.fetch(wp + k0 + BK, w_stride, N - n0, K - k0 - BK, vec, tid);
        }
#pragma unroll 4
        for (int k = 0; k < BK; ++k) {
            float av[TM], bv[TN];
#pragma unroll
            for (int g = 0; g < GM; ++g)
#pragma unroll
                for (int i = 0; i < VM; ++i) av[g * VM + i] = xs[buf][k][g * (BM / GM) + ty * VM + i];
#pragma unroll
            for (int g = 0; g < GN; ++g)
#pragma unroll
                for (int j = 0; j < VN; ++j) bv[g * VN + j] = ws[buf][k][g * (BN / GN) + tx * VN + j];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] += av[i] * bv[j];
        }
        if (more) {
            // the other buffer was last read before the barrier that ended the previous tile
            lx.store(xs[buf ^ 1], tid);
            lw.store(ws[buf ^ 1], tid);
        }
        __syncthreads();
        buf ^= 1;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + (i / VM) * (BM / GM) + ty * VM + i % VM;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (j / VN) * (BN / GN) + tx * VN + j % VN;
            if (n >= N) continue;
            float v = acc[i][j];
            if (bias) v += to_float(bias[n]);
            y[(int64_t)m * y_stride + n] = from_float<OutT>(v);
        }
    }
}

#endif

#if defined(NVA_F32)
// ---------------------------------------------------------------------------- float operands on the matrix cores
// The products of the 32-bit path: v_mfma_f32_16x16x4_f32, float operands and float sums.  Every output is one chain of
// such instructions over k whatever the tile: in each run of 16 columns the instruction j of four takes the columns j,
// 4 + j, 8 + j, 12 + j (a lane's four numbers of 16 bytes, so that operands are read 16 bytes at a time), the runs follow
// each other, and columns past K are zeros.  A result does not depend on the rows beside it, nor on the kernel that made it.
//
// Bound by the matrix cores (157 TFLOP/s for float operands) from some 1000 rows on, below by how few workgroups the outputs
// make (their chains are not cut), and by the weight's bytes at few rows.  us before (a multiply-add per output and column
// on the vector units) / here: 957 rows, weights 4096 x 1024 218 / 104, 6144 x 1024 227 / 133, 1024 x 2048 143 / 54, 1024 x
// 3072 203 / 77; 2048 rows, 24576 x 4096 4938 / 4218 (98 TFLOP/s); 40 rows, 4096 x 1024 69 / 20; 7 rows, 1024 x 3072 67 / 28;
// 10 rows, 151936 x 1024 221 / 154 (4.0 TB/s).  The error against 64 bits is what it was (4.0e-7 to 7.1e-7 at these sizes).
typedef __attribute__((ext_vector_type(4))) float gf_f32x4;

// Columns k .. k + 3 of a row, zeros past K.  VEC: rows of whole 16 bytes, K a multiple of 4; the load is unconditional (a
// branch around a load makes the compiler wait for all the others).
template <bool VEC>
__device__ __forceinline__ gf_f32x4 gf_load(const float* __restrict__ row, int k, int K) {
    gf_f32x4 v;
    if (VEC) {
        v = *reinterpret_cast<const gf_f32x4*>(row + min(k, K - 4));
        if (k >= K) v = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = k + e < K ? row[k + e] : 0.f;
    }
    return v;
}

__device__ __forceinline__ void gf_store(const gf_f32x4& acc, const float* __restrict__ bias, float* __restrict__ y, int64_t y_stride,
                                         int m, int n, int M, int N, bool vec_y) {
    if (m >= M) return;
    float* at = y + (int64_t)m * y_stride + n;
    if (vec_y && n + 4 <= N) {
        gf_f32x4 v = acc;
        if (bias)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += bias[n + e];
        *reinterpret_cast<gf_f32x4*>(at) = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) at[e] = acc[e] + (bias ? bias[n + e] : 0.f);
    }
}

// A workgroup of four waves takes BM rows of x and BN rows of W, 32 columns at a time through two buffers in LDS, the next
// columns' loads on their way during the products; a wave a (BM / 2) x (BN / 2) part.  Rows of LDS are 36 floats, so that
// the 16 rows of a read start in different banks.
template <int BM, int BN, bool VEC>
__global__ void __launch_bounds__(256)
linear_float_kernel(const float* __restrict__ x, int64_t x_stride, const float* __restrict__ w, int64_t w_stride,
                    const float* __restrict__ bias, float* __restrict__ y, int64_t y_stride, int M, int N, int K, int vec_y) {
    constexpr int LD = 36, TM = BM / 32, TN = BN / 32, XP = BM / 32, WP = BN / 32;     // 16-byte pieces a thread brings of each
    __shared__ __attribute__((aligned(16))) float xs[2][BM * LD], ws[2][BN * LD];
    const int tid = threadIdx.x, wave = tid / NVA_WAVE, lane = tid % NVA_WAVE;
    const int col = lane & 15, g = lane >> 4, wm = wave / 2, wn = wave % 2;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int pr = tid / 8, pk = (tid % 8) * 4;             // this thread's piece of rows pr + 32 i
    const float *xrow[XP], *wrow[WP];                       // (rows past the end: the last one again, never stored)
#pragma unroll
    for (int i = 0; i < XP; ++i) xrow[i] = x + (int64_t)min(m0 + pr + 32 * i, M - 1) * x_stride;
#pragma unroll
    for (int i = 0; i < WP; ++i) wrow[i] = w + (int64_t)min(n0 + pr + 32 * i, N - 1) * w_stride;
    gf_f32x4 xv[XP], wv[WP], acc[TN][TM];
    auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; ++i) xv[i] = gf_load<VEC>(xrow[i], k0 + pk, K);
#pragma unroll
        for (int i = 0; i < WP; ++i) wv[i] = gf_load<VEC>(wrow[i], k0 + pk, K);
    };
    auto put = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; ++i) *reinterpret_cast<gf_f32x4*>(&xs[buf][(pr + 32 * i) * LD + pk]) = xv[i];
#pragma unroll
        for (int i = 0; i < WP; ++i) *reinterpret_cast<gf_f32x4*>(&ws[buf][(pr + 32 * i) * LD + pk]) = wv[i];
    };
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(0);
    put(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += 32) {
        fetch(k0 + 32);                                     // (zeros past K)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            gf_f32x4 fa[TN], fb[TM];
#pragma unroll
            for (int a = 0; a < TN; ++a) fa[a] = *reinterpret_cast<const gf_f32x4*>(&ws[buf][(wn * (BN / 2) + 16 * a + col) * LD + 16 * s + 4 * g]);
#pragma unroll
            for (int b = 0; b < TM; ++b) fb[b] = *reinterpret_cast<const gf_f32x4*>(&xs[buf][(wm * (BM / 2) + 16 * b + col) * LD + 16 * s + 4 * g]);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int a = 0; a < TN; ++a)
#pragma unroll
                    for (int b = 0; b < TM; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[a][j], fb[b][j], acc[a][b], 0, 0, 0);
        }
        put(buf ^ 1);                                       // (last read before the barrier that ended the stage before)
        __syncthreads();
        buf ^= 1;
    }
    // acc[a][b][i] = y[row 16 b + col][16 a + 4 g + i] of the wave's part
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int a = 0; a < TN; ++a)
            gf_store(acc[a][b], bias, y, y_stride, m0 + wm * (BM / 2) + 16 * b + col, n0 + wn * (BN / 2) + 16 * a + 4 * g, M, N, vec_y);
}

// Up to 16 rows of x: one wave streams 16 rows of W, and the rows of x from the caches, straight into registers, 128 columns
// asked for ahead of the 128 that are multiplied.
template <bool VEC>
__global__ void __launch_bounds__(NVA_WAVE)
linear_float_stream_kernel(const float* __restrict__ x, int64_t x_stride, const float* __restrict__ w, int64_t w_stride,
                           const float* __restrict__ bias, float* __restrict__ y, int64_t y_stride, int M, int N, int K, int vec_y) {
    constexpr int R = 8;                                    // runs of 16 columns a set of registers holds
    const int lane = threadIdx.x, col = lane & 15, g = lane >> 4, n0 = blockIdx.x * 16;
    const float* xrow = x + (int64_t)min(col, M - 1) * x_stride;
    const float* wrow = w + (int64_t)min(n0 + col, N - 1) * w_stride;
    gf_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, w0[R], x0[R], w1[R], x1[R];
    auto fetch = [&](int k0, gf_f32x4 (&wv)[R], gf_f32x4 (&xv)[R]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < R; ++s) wv[s] = gf_load<VEC>(wrow, k0 + 16 * s + 4 * g, K);
#pragma unroll
        for (int s = 0; s < R; ++s) xv[s] = gf_load<VEC>(xrow, k0 + 16 * s + 4 * g, K);
    };
    auto multiply = [&](const gf_f32x4 (&wv)[R], const gf_f32x4 (&xv)[R]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < R; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s][j], xv[s][j], acc, 0, 0, 0);
    };
    fetch(0, w0, x0);
    for (int k0 = 0; k0 < K; k0 += 32 * R) {                // (columns past K are zeros and change nothing)
        fetch(k0 + 16 * R, w1, x1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(w0, x0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(k0 + 32 * R, w0, x0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(w1, x1);
        __builtin_amdgcn_sched_barrier(0);
    }
    gf_store(acc, bias, y, y_stride, col, n0 + 4 * g, M, N, vec_y);
}
#endif

NVA_EXPORT int NVA_NAME(nva_linear_tiled)(const void* x, int64_t x_stride, const void* w, int64_t w_stride,
                                          const void* bias, void* y, int64_t y_stride, int out_is_f32, int64_t M,
                                          int64_t N, int64_t K, hipStream_t stream) {
    if (M == 0 || N == 0) return 0;
    if (M < 0 || N < 0 || K <= 0 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff)
        return nva_fail("linear: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
    const size_t vb = 4 * sizeof(elem_t);
    const int vec = x_stride % 4 == 0 && w_stride % 4 == 0 && nva_aligned(x, vb) && nva_aligned(w, vb);
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
            cus = 0;
            return nva_fail("linear: cannot read the number of CUs");
        }
    }
#if defined(NVA_F32)
    const int vec4 = vec && K % 4 == 0, vec_y = y_stride % 4 == 0 && nva_aligned(y, 16);
#define FLOAT_ARGS (const float*)x, x_stride, (const float*)w, w_stride, (const float*)bias, (float*)y, y_stride, (int)M, (int)N, (int)K, vec_y
    if (M <= 16) {
        const auto kernel = vec4 ? linear_float_stream_kernel<true> : linear_float_stream_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)((N + 15) / 16)), dim3(NVA_WAVE), 0, stream, FLOAT_ARGS);
        return nva_check_launch("linear_tiled");
    }
    // The tile: what the most loaded CU multiplies is the number of tiles it gets times a tile's size; of shapes that give the
    // same the smaller one, two of which share a CU and fill each other's waits.
    struct Shape { int bm, bn; };
    static const Shape shapes[] = {{128, 128}, {128, 64}, {64, 64}, {64, 32}, {32, 32}};
    int best = 0;
    int64_t least = INT64_MAX;
    for (int i = 0; i < 5; ++i) {
        const int64_t tiles = ((M + shapes[i].bm - 1) / shapes[i].bm) * ((N + shapes[i].bn - 1) / shapes[i].bn);
        const int64_t load = (tiles + cus - 1) / cus * shapes[i].bm * shapes[i].bn;
        if (load < least || (load == least && i < 4)) { least = load; best = i; }
    }
    if ((M + shapes[best].bm - 1) / shapes[best].bm > 65535) return nva_fail("linear: M=%lld exceeds %d rows per call", (long long)M, 65535 * shapes[best].bm);
#define FLOAT_LAUNCH(BM, BN)                                                                                          \
    hipLaunchKernelGGL((vec4 ? linear_float_kernel<BM, BN, true> : linear_float_kernel<BM, BN, false>), dim3((unsigned)((N + BN - 1) / BN), (unsigned)((M + BM - 1) / BM)), dim3(256), 0, stream, FLOAT_ARGS)
    switch (best) {
        case 0: FLOAT_LAUNCH(128, 128); break;
        case 1: FLOAT_LAUNCH(128, 64); break;
        case 2: FLOAT_LAUNCH(64, 64); break;
        case 3: FLOAT_LAUNCH(64, 32); break;
        default: FLOAT_LAUNCH(32, 32);
    }
#undef FLOAT_LAUNCH
#undef FLOAT_ARGS
#else
#define LAUNCH_AS(OUT, BM, BN, BK, TM, TN)                                                                            \
    hipLaunchKernelGGL((linear_tiled_kernel<elem_t, OUT, BM, BN, BK, TM, TN>), grid, dim3(256), 0, stream,            \
                       (const elem_t*)x, x_stride, (const elem_t*)w, w_stride, (const elem_t*)bias, (OUT*)y, y_stride, \
                       (int)M, (int)N, (int)K, vec)
#define LAUNCH(BM, BN, BK, TM, TN)                                                                                    \
    do {                                                                                                              \
        const int64_t grid_m = (M + BM - 1) / BM, grid_n = (N + BN - 1) / BN;                                         \
        if (grid_m > 65535) return nva_fail("linear: M=%lld exceeds %d rows per call", (long long)M, 65535 * BM);     \
        dim3 grid((unsigned)grid_n, (unsigned)grid_m);                                                                \
        if (out_is_f32) LAUNCH_AS(float, BM, BN, BK, TM, TN);                                                         \
        else LAUNCH_AS(elem_t, BM, BN, BK, TM, TN);                                                                   \
    } while (0)
    if (M <= 16) {
        if (N >= 64 * (int64_t)cus) LAUNCH(16, 64, 64, 4, 1);
        else LAUNCH(16, 16, 64, 1, 1);
    } else if (((M + 127) / 128) * ((N + 127) / 128) >= cus) LAUNCH(128, 128, 16, 8, 8);
    else LAUNCH(64, 64, 16, 4, 4);
#undef LAUNCH
#undef LAUNCH_AS
#endif
    return nva_check_launch("linear_tiled");
}

NVA_DEFINE_LAST_ERROR(nva_gemm)
