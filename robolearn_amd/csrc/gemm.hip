// fp32 dense-layer GEMMs on the fp32 matrix instruction (mode 0), split-K reductions, transposes and the
// rl_gemm entry point.
//
// One row-major kernel family covers the three products of a bias-free
// Linear layer (the reference's CudaLinear plans, robolearn/cuda/linear.py:179-185):
//   forward  Y[R,N]  = X[R,K]  . W[N,K]^T     (A K-contiguous, B K-contiguous)
//   input    dX[R,K] = dY[R,N] . W[N,K]       (A K-contiguous, B N-contiguous)
//   weight   dW[N,K] = dY[R,N]^T . X[R,K]     (A M-contiguous, B N-contiguous)
// batched over a leading ensemble index (the stacked twin critics).
//
// v_mfma_f32_32x32x2_f32 is 64 cycles per 2048 MACs, so these products are
// bound by MFMA issue, not by operand traffic: what matters is that every SIMD
// has independent work.  A 256-thread workgroup owns a T x T output tile as
// 2x2 waves of (T/2) x (T/2), i.e. (T/64)^2 32x32 accumulators per wave.  T =
// 64 for the small-row-count products of the PPO update (4x the workgroups of
// T = 128, so every CU gets several), T = 128 for large ones.  Operands are
// staged through LDS in [row][k] order, 16 K per step, so each lane reads its
// K-slice with two 16-byte LDS loads; the K order inside a step is permuted
// identically for both operands, which leaves the dot products unchanged.
// Mode 2 (fp32 operands and results on the bf16 matrix cores) runs in gemm_split.hip.
#include "gemm.hpp"

#include <cmath>
#include <string>

namespace rl {
namespace gemm {

constexpr int kFp32K = 32;              // K per LDS step: two 16-K substeps
constexpr int kFp32Pitch = kFp32K + 4;  // floats per LDS row

// Loads one Rows x kFp32K operand tile into registers (Threads threads) and
// later stores it to LDS.  Element (r, k) of the operand is src[r * ld + k]
// when KContig, else src[k * ld + r].
template <bool KContig, int Rows, int Threads>
struct TileLoader {
    static constexpr int VecPerRow = kFp32K / 4;
    static constexpr int PerThread = KContig ? Rows * VecPerRow / Threads : 1;
    static constexpr int Groups = Threads / Rows;      // M/N-contiguous: k groups per tile
    static constexpr int KPer = kFp32K / Groups;        // k values per thread
    static constexpr int Count = KContig ? PerThread * 4 : KPer;
    static_assert(KContig ? PerThread >= 1 : (KPer >= 1 && kFp32K % Groups == 0), "tile/thread mismatch");
    float regs[Count];

    // A tile wholly inside the operand (rows r0 .. r0 + Rows - 1 < rows, k0 + kFp32K <= ks) and, K-contiguous,
    // with 16-byte aligned rows: the loads need no per-element checks.
    __device__ __forceinline__ void load_full(const float* src, long long ld, int r0, int k0) {
        const int t = threadIdx.x;
        if constexpr (KContig) {
#pragma unroll
            for (int i = 0; i < PerThread; ++i) {
                const int v = i * Threads + t;
                const float4 x = *reinterpret_cast<const float4*>(
                    src + static_cast<long long>(r0 + v / VecPerRow) * ld + k0 + (v % VecPerRow) * 4);
                regs[i * 4 + 0] = x.x;
                regs[i * 4 + 1] = x.y;
                regs[i * 4 + 2] = x.z;
                regs[i * 4 + 3] = x.w;
            }
        } else {
            const float* q = src + static_cast<long long>(k0 + (t / Rows) * KPer) * ld + r0 + t % Rows;
#pragma unroll
            for (int e = 0; e < KPer; ++e) regs[e] = q[e * ld];
        }
    }

    __device__ __forceinline__ void load(const float* src, long long ld, int r0, int k0, int rows, int ks, bool vec) {
        const int t = threadIdx.x;
        if constexpr (KContig) {
#pragma unroll
            for (int i = 0; i < PerThread; ++i) {
                const int v = i * Threads + t;
                const int r = r0 + v / VecPerRow;
                const int k = k0 + (v % VecPerRow) * 4;
                const float* q = src + static_cast<long long>(r) * ld + k;
                if (r < rows && vec && k + 4 <= ks) {
                    const float4 x = *reinterpret_cast<const float4*>(q);
                    regs[i * 4 + 0] = x.x;
                    regs[i * 4 + 1] = x.y;
                    regs[i * 4 + 2] = x.z;
                    regs[i * 4 + 3] = x.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) regs[i * 4 + e] = (r < rows && k + e < ks) ? q[e] : 0.0f;
                }
            }
        } else {
            const int r = r0 + t % Rows;
            const int kb = k0 + (t / Rows) * KPer;
            const bool rv = r < rows;
#pragma unroll
            for (int e = 0; e < KPer; ++e) {
                const int k = kb + e;
                regs[e] = (rv && k < ks) ? src[static_cast<long long>(k) * ld + r] : 0.0f;
            }
        }
    }

    __device__ __forceinline__ void store(float* lds) const {
        const int t = threadIdx.x;
        if constexpr (KContig) {
#pragma unroll
            for (int i = 0; i < PerThread; ++i) {
                const int v = i * Threads + t;
                *reinterpret_cast<float4*>(lds + (v / VecPerRow) * kFp32Pitch + (v % VecPerRow) * 4) =
                    make_float4(regs[i * 4 + 0], regs[i * 4 + 1], regs[i * 4 + 2], regs[i * 4 + 3]);
            }
        } else {
            float* q = lds + (t % Rows) * kFp32Pitch + (t / Rows) * KPer;
#pragma unroll
            for (int e = 0; e < KPer; ++e) q[e] = regs[e];
        }
    }
};

// Four waves own the T x T tile as 2 x 2 wave tiles of (T / 2) x (T / 2).
template <int T, bool AK, bool BK>
__global__ __launch_bounds__(kThreads) void gemm_kernel(Params p) {
    constexpr int Threads = kThreads;
    constexpr int WGN = 2, WGM = 2;
    constexpr int WTM = T / WGM, WTN = T / WGN;    // wave tile
    constexpr int WBM = WTM / 32, WBN = WTN / 32;  // 32x32 accumulator blocks per wave
    __shared__ __attribute__((aligned(16))) float sa[T * kFp32Pitch];
    __shared__ __attribute__((aligned(16))) float sb[T * kFp32Pitch];

    // XCD-aware tile order: workgroups are dispatched round-robin over the 8
    // XCDs in linear (x fastest) order, so logical tile id (w % 8) * (G / 8) +
    // w / 8 gives each XCD a contiguous range of tiles; the N tiles of one M
    // panel then share that XCD's L2 instead of fetching the panel once per XCD.
    const unsigned nx = gridDim.x, ny = gridDim.y;
    const unsigned groups = nx * ny * gridDim.z;
    unsigned w = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
    if (groups % 8 == 0) w = (w % 8) * (groups / 8) + w / 8;
    const int bx = static_cast<int>(w % nx);
    const int by = static_cast<int>((w / nx) % ny);
    const int bz = static_cast<int>(w / (nx * ny));
    const int split = bz % p.splits;
    const int batch = bz / p.splits;
    const float* A = static_cast<const float*>(p.a) + batch * p.stride_a;
    const float* B = static_cast<const float*>(p.b) + batch * p.stride_b;
    const int m0 = by * T;
    const int n0 = bx * T;
    const int k_begin = split * p.k_per_split;
    const int k_end = min(p.k, k_begin + p.k_per_split);

    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int wm = wave / WGN;
    const int wn = wave % WGN;

    f32x16_t acc[WBM][WBN];
#pragma unroll
    for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    TileLoader<AK, T, Threads> la;
    TileLoader<BK, T, Threads> lb;
    const bool avec = p.a_vec != 0;
    const bool bvec = p.b_vec != 0;
    // Row sums of op(A) over this split's K (the bias gradient of a weight-
    // gradient product), by the workgroups of the first N tile: thread t adds
    // kFp32K * T / Threads staged values of row t / (Threads / T) per step.
    constexpr int SumLanes = Threads / T;
    constexpr int SumPer = kFp32K / SumLanes;
    const bool row_sums = p.a_sums != nullptr && bx == 0;
    // compensated (Kahan) accumulation: bias gradients are sums over thousands of
    // rows whose terms largely cancel, where plain sequential fp32 sums lose digits
    float a_sum = 0.0f, a_comp = 0.0f;
    const auto add_sum = [&](float x) {
        const float y = x - a_comp;
        const float t = a_sum + y;
        a_comp = (t - a_sum) - y;
        a_sum = t;
    };

    // B is indexed (n, k) when BK else (k, n); the loader wants (row=n, k).
    const auto stage = [&]() {
        la.store(sa);
        lb.store(sb);
    };
    // K steps whose operand tiles lie wholly inside A and B (uniform per workgroup) take the unchecked loads
    const bool a_full = (!AK || avec) && m0 + T <= p.m;
    const bool b_full = (!BK || bvec) && n0 + T <= p.n;
    const auto load_step = [&](int k0) {
        if (a_full && k0 + kFp32K <= k_end) la.load_full(A, p.lda, m0, k0);
        else la.load(A, p.lda, m0, k0, p.m, k_end, avec);
        if (b_full && k0 + kFp32K <= k_end) lb.load_full(B, p.ldb, n0, k0);
        else lb.load(B, p.ldb, n0, k0, p.n, k_end, bvec);
    };
    if (k_begin < k_end) {
        load_step(k_begin);
        stage();
    }
    __syncthreads();

    for (int k0 = k_begin; k0 < k_end; k0 += kFp32K) {
        const bool more = k0 + kFp32K < k_end;
        if (more) load_step(k0 + kFp32K);
        if (row_sums) {
            const float* q = sa + (threadIdx.x / SumLanes) * kFp32Pitch + (threadIdx.x % SumLanes) * SumPer;
#pragma unroll
            for (int e = 0; e < SumPer; ++e) add_sum(q[e]);
        }
#pragma unroll
        for (int sub = 0; sub < kFp32K / 16; ++sub) {
            float4 af[WBM][2], bfr[WBN][2];
#pragma unroll
            for (int i = 0; i < WBM; ++i) {
                const float* q = sa + (wm * WTM + i * 32 + lane % 32) * kFp32Pitch + 16 * sub + (lane / 32) * 8;
                af[i][0] = *reinterpret_cast<const float4*>(q);
                af[i][1] = *reinterpret_cast<const float4*>(q + 4);
            }
#pragma unroll
            for (int j = 0; j < WBN; ++j) {
                const float* q = sb + (wn * WTN + j * 32 + lane % 32) * kFp32Pitch + 16 * sub + (lane / 32) * 8;
                bfr[j][0] = *reinterpret_cast<const float4*>(q);
                bfr[j][1] = *reinterpret_cast<const float4*>(q + 4);
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) {
#pragma unroll
                for (int i = 0; i < WBM; ++i) {
                    const float a = s < 4 ? af[i][0][s] : af[i][1][s - 4];
#pragma unroll
                    for (int j = 0; j < WBN; ++j) {
                        const float b = s < 4 ? bfr[j][0][s] : bfr[j][1][s - 4];
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i][j], 0, 0, 0);
                    }
                }
            }
        }
        __syncthreads();
        if (more) stage();
        __syncthreads();
    }

    if (row_sums) {
        // the SumLanes partial sums of a row sit in adjacent lanes: fixed-order butterfly
#pragma unroll
        for (int offset = 1; offset < SumLanes; offset <<= 1) a_sum += __shfl_xor(a_sum, offset);
        const int r = m0 + static_cast<int>(threadIdx.x) / SumLanes;
        if (threadIdx.x % SumLanes == 0 && r < p.m)
            p.a_sums[(p.splits == 1 ? batch * p.sums_stride
                                     : (static_cast<long long>(split) * p.batch + batch) * p.m) + r] = a_sum;
    }

    // Accumulator layout of a 32x32 MFMA tile: lane l holds column l % 32 and
    // rows 8 * (v / 4) + 4 * (l / 32) + v % 4 for v = 0..15.
    const bool direct = p.splits == 1;
    float* D = p.d + (direct ? batch * p.stride_d
                             : (static_cast<long long>(split) * p.batch + batch) * static_cast<long long>(p.m) * p.n);
    const long long ldd = direct ? p.ldd : p.n;
    const float* bias = p.bias ? p.bias + batch * p.stride_bias : nullptr;
    const float* C = p.c ? p.c + batch * p.stride_d : nullptr;
    // Every C value this lane needs is loaded before its first store: the compiler cannot tell C from D
    // apart, so a load left inside the store loop would wait for the stores before it and expose one
    // memory round trip per element (the ELU-gradient products of the PPO backward read C everywhere).
    const bool read_c = direct && C && (p.epilogue == kEluGrad || p.beta != 0.0f);
    float cv[WBM][WBN][16];
    if (read_c) {
#pragma unroll
        for (int i = 0; i < WBM; ++i)
#pragma unroll
            for (int j = 0; j < WBN; ++j) {
                const int col = n0 + wn * WTN + j * 32 + lane % 32;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = m0 + wm * WTM + i * 32 + 8 * (v / 4) + 4 * (lane / 32) + (v % 4);
                    cv[i][j][v] = (col < p.n && row < p.m) ? C[static_cast<long long>(row) * ldd + col] : 0.0f;
                }
            }
    }
#pragma unroll
    for (int i = 0; i < WBM; ++i) {
#pragma unroll
        for (int j = 0; j < WBN; ++j) {
            const int col = n0 + wn * WTN + j * 32 + lane % 32;
            if (col >= p.n) continue;
            const float bcol = (direct && bias) ? bias[col] : 0.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm * WTM + i * 32 + 8 * (v / 4) + 4 * (lane / 32) + (v % 4);
                if (row >= p.m) continue;
                const long long offset = static_cast<long long>(row) * ldd + col;
                float* out = D + offset;
                if (direct) {
                    float value;
                    if (p.epilogue == kEluGrad) {
                        value = acc[i][j][v] * elu_grad_from_output(cv[i][j][v]);
                    } else {
                        value = apply_epilogue(acc[i][j][v] + bcol, p.epilogue);
                        if (p.beta != 0.0f) value += p.beta * cv[i][j][v];
                    }
                    *out = value;
                    if (p.d_bf16) p.d_bf16[batch * p.stride_d + offset] = f32_to_bf16_bits(value);
                } else {
                    *out = acc[i][j][v];
                }
            }
        }
    }
}

// Fixed-order split-K reduction: D = act(sum_s W[s] + bias) + beta * C.
// p[s * step] summed over s = first, first + stride, ... < splits, in that order.  Eight loads are issued
// before the first of their adds: a plain loop waits for each load before issuing the next, one memory
// round trip per split.  The adds keep the loop's order, so the sum is the same.
__device__ __forceinline__ float ordered_sum(const float* p, long long step, int first, int stride, int splits) {
    float value = 0.0f;
    int s = first;
    for (; s + 7 * stride < splits; s += 8 * stride) {
        float w[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) w[u] = p[static_cast<long long>(s + u * stride) * step];
#pragma unroll
        for (int u = 0; u < 8; ++u) value += w[u];
    }
    for (; s < splits; s += stride) value += p[static_cast<long long>(s) * step];
    return value;
}

// The same over float4 pieces (p 16-byte aligned, step a multiple of 4).
__device__ __forceinline__ float4 ordered_sum4(const float* p, long long step, int splits) {
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int s = 0;
    for (; s + 3 < splits; s += 4) {
        float4 w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = *reinterpret_cast<const float4*>(p + static_cast<long long>(s + u) * step);
#pragma unroll
        for (int u = 0; u < 4; ++u) v = make_float4(v.x + w[u].x, v.y + w[u].y, v.z + w[u].z, v.w + w[u].w);
    }
    for (; s < splits; ++s) {
        const float4 w = *reinterpret_cast<const float4*>(p + static_cast<long long>(s) * step);
        v = make_float4(v.x + w.x, v.y + w.y, v.z + w.z, v.w + w.w);
    }
    return v;
}

__global__ void splitk_reduce(const float* work, float* d, unsigned short* d_bf16, const float* c, const float* bias,
                              long long ldd, long long stride_d, long long stride_bias, int m, int n, int batch,
                              int splits, float beta, int epilogue) {
    const long long total = static_cast<long long>(batch) * m * n;
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < total;
         idx += static_cast<long long>(gridDim.x) * blockDim.x) {
        const int col = static_cast<int>(idx % n);
        const int row = static_cast<int>((idx / n) % m);
        const int b = static_cast<int>(idx / (static_cast<long long>(m) * n));
        float value = ordered_sum(work + b * static_cast<long long>(m) * n + static_cast<long long>(row) * n + col,
                                  static_cast<long long>(batch) * m * n, 0, 1, splits);
        const long long offset = b * stride_d + static_cast<long long>(row) * ldd + col;
        if (epilogue == kEluGrad) {
            value *= elu_grad_from_output(c[offset]);
        } else {
            if (bias) value += bias[b * stride_bias + col];
            value = apply_epilogue(value, epilogue);
            if (beta != 0.0f) value += beta * c[offset];
        }
        if (d) d[offset] = value;
        if (d_bf16) d_bf16[offset] = f32_to_bf16_bits(value);
    }
}

// splitk_reduce on four consecutive outputs of a row per thread (n, ldd and the
// strides multiples of 4; d, c, bias 16-byte and d_bf16 8-byte aligned).
__global__ void splitk_reduce_vec(const float* work, float* d, unsigned short* d_bf16, const float* c,
                                  const float* bias, long long ldd, long long stride_d, long long stride_bias, int m,
                                  int n, int batch, int splits, float beta, int epilogue) {
    const int n4 = n / 4;
    const long long total = static_cast<long long>(batch) * m * n4;
    const long long plane = static_cast<long long>(m) * n;
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < total;
         idx += static_cast<long long>(gridDim.x) * blockDim.x) {
        const int col = 4 * static_cast<int>(idx % n4);
        const int row = static_cast<int>((idx / n4) % m);
        const int b = static_cast<int>(idx / (static_cast<long long>(m) * n4));
        const long long within = static_cast<long long>(row) * n + col;
        float4 v = ordered_sum4(work + b * plane + within, static_cast<long long>(batch) * plane, splits);
        const long long offset = b * stride_d + static_cast<long long>(row) * ldd + col;
        if (epilogue == kEluGrad) {
            const float4 y = *reinterpret_cast<const float4*>(c + offset);
            v = make_float4(v.x * elu_grad_from_output(y.x), v.y * elu_grad_from_output(y.y),
                            v.z * elu_grad_from_output(y.z), v.w * elu_grad_from_output(y.w));
        } else {
            if (bias) {
                const float4 bv = *reinterpret_cast<const float4*>(bias + b * stride_bias + col);
                v = make_float4(v.x + bv.x, v.y + bv.y, v.z + bv.z, v.w + bv.w);
            }
            v = make_float4(apply_epilogue(v.x, epilogue), apply_epilogue(v.y, epilogue),
                            apply_epilogue(v.z, epilogue), apply_epilogue(v.w, epilogue));
            if (beta != 0.0f) {
                const float4 cv = *reinterpret_cast<const float4*>(c + offset);
                v = make_float4(v.x + beta * cv.x, v.y + beta * cv.y, v.z + beta * cv.z, v.w + beta * cv.w);
            }
        }
        if (d) *reinterpret_cast<float4*>(d + offset) = v;
        if (d_bf16)
            *reinterpret_cast<uint2*>(d_bf16 + offset) = make_uint2(f32x2_to_bf16x2(v.x, v.y), f32x2_to_bf16x2(v.z, v.w));
    }
}

// Same reduction for many splits: a workgroup covers kReduceCols consecutive
// outputs with kReduceGroups threads each; group g adds splits g, g + G, ...
// in order and group 0 adds the group sums in order, so the result is fixed
// and each thread's chain is splits / G loads long.  With sums != nullptr the
// index space continues past D with the batch * m row sums of A
// ([splits][batch][m] partials in sums_work), written at b * sums_stride + r.
constexpr int kReduceGroups = 8;
constexpr int kReduceCols = 256 / kReduceGroups;

__global__ __launch_bounds__(256) void splitk_reduce_grouped(const float* work, float* d, unsigned short* d_bf16,
                                                             const float* c, const float* bias, long long ldd,
                                                             long long stride_d, long long stride_bias, int m, int n,
                                                             int batch, int splits, float beta, int epilogue,
                                                             const float* sums_work = nullptr, float* sums = nullptr,
                                                             long long sums_stride = 0) {
    __shared__ float part[kReduceGroups][kReduceCols];
    const long long total = static_cast<long long>(batch) * m * n;
    const long long extra = sums ? static_cast<long long>(batch) * m : 0;
    const int e = threadIdx.x % kReduceCols;
    const int g = threadIdx.x / kReduceCols;
    const long long idx = static_cast<long long>(blockIdx.x) * kReduceCols + e;
    const long long plane = static_cast<long long>(m) * n;
    float value = 0.0f;
    if (idx < total) {
        const int b = static_cast<int>(idx / plane);
        const long long within = idx - b * plane;
        value = ordered_sum(work + b * plane + within, static_cast<long long>(batch) * plane, g, kReduceGroups, splits);
    } else if (idx < total + extra) {
        const long long j = idx - total;  // b * m + r
        value = ordered_sum(sums_work + j, static_cast<long long>(batch) * m, g, kReduceGroups, splits);
    }
    part[g][e] = value;
    __syncthreads();
    if (g != 0 || idx >= total + extra) return;
    for (int k = 1; k < kReduceGroups; ++k) value += part[k][e];
    if (idx >= total) {
        const long long j = idx - total;
        sums[(j / m) * sums_stride + j % m] = value;
        return;
    }
    const int col = static_cast<int>(idx % n);
    const int row = static_cast<int>((idx / n) % m);
    const int b = static_cast<int>(idx / plane);
    const long long offset = b * stride_d + static_cast<long long>(row) * ldd + col;
    if (epilogue == kEluGrad) {
        value *= elu_grad_from_output(c[offset]);
    } else {
        if (bias) value += bias[b * stride_bias + col];
        value = apply_epilogue(value, epilogue);
        if (beta != 0.0f) value += beta * c[offset];
    }
    if (d) d[offset] = value;
    if (d_bf16) d_bf16[offset] = f32_to_bf16_bits(value);
}

// Output tile edge: 64 unless 128-wide tiles would still give every SIMD several waves of work.
int fp32_tile(const Params& p) {
    const long long big = static_cast<long long>(ceil_div(p.m, 128)) * ceil_div(p.n, 128) * p.batch * p.splits;
    return big >= 2048 ? 128 : 64;
}

const char* kernel_name(int mode, const Params& p, int a_16bit, int b_16bit, bool ak, bool bk) {
    if (mode == 0) return fp32_tile(p) == 128 ? "mfma_128x128" : "mfma_64x64";
    if (mode == 1 && big_eligible(p, a_16bit, b_16bit)) return "mfma_256x256";
    if (mode == 1 && narrow_eligible(p, a_16bit, b_16bit, ak, bk)) return "mfma_64x64";
    return "mfma_256x128";
}

template <int T, bool AK, bool BK>
void launch_fp32_tiled(const Params& p, hipStream_t stream) {
    const dim3 grid(ceil_div(p.n, T), ceil_div(p.m, T), static_cast<unsigned>(p.batch * p.splits));
    hipLaunchKernelGGL((gemm_kernel<T, AK, BK>), grid, dim3(kThreads), 0, stream, p);
}

template <bool AK, bool BK>
void launch_fp32_layout(const Params& p, hipStream_t stream) {
    if (fp32_tile(p) == 128) launch_fp32_tiled<128, AK, BK>(p, stream);
    else launch_fp32_tiled<64, AK, BK>(p, stream);
}

void launch_fp32(const Params& p, bool ak, bool bk, hipStream_t stream) {
    if (ak && bk) launch_fp32_layout<true, true>(p, stream);
    else if (ak && !bk) launch_fp32_layout<true, false>(p, stream);
    else if (!ak && bk) launch_fp32_layout<false, true>(p, stream);
    else launch_fp32_layout<false, false>(p, stream);
}

// dst[b][c][r] = src[b][r][c] for 16-bit elements: 64 x 64 tiles through LDS,
// coalesced 2-byte reads along c and writes along r.  Grid (col tiles, row
// tiles, batch).
__global__ __launch_bounds__(256) void transpose16(const unsigned short* src, unsigned short* dst, int rows, int cols) {
    __shared__ unsigned short tile[64][65];
    const long long base = static_cast<long long>(blockIdx.z) * rows * cols;
    const int r0 = static_cast<int>(blockIdx.y) * 64;
    const int c0 = static_cast<int>(blockIdx.x) * 64;
    const int t = static_cast<int>(threadIdx.x);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = i * 4 + t / 64;
        const int c = t % 64;
        if (r0 + r < rows && c0 + c < cols) tile[r][c] = src[base + static_cast<long long>(r0 + r) * cols + c0 + c];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = i * 4 + t / 64;
        const int r = t % 64;
        if (r0 + r < rows && c0 + c < cols) dst[base + static_cast<long long>(c0 + c) * rows + r0 + r] = tile[r][c];
    }
}

// transpose16 with 8-byte accesses for rows and cols in multiples of 4 and
// 8-byte aligned buffers: a load covers 4 columns of one source row, a store 4
// source rows of one column (one destination row segment).
__global__ __launch_bounds__(256) void transpose16_vec(const unsigned short* src, unsigned short* dst, int rows,
                                                       int cols) {
    __shared__ unsigned short tile[64][66];
    const long long base = static_cast<long long>(blockIdx.z) * rows * cols;
    const int r0 = static_cast<int>(blockIdx.y) * 64;
    const int c0 = static_cast<int>(blockIdx.x) * 64;
    const int t = static_cast<int>(threadIdx.x);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = i * 16 + t / 16;
        const int c = 4 * (t % 16);
        if (r0 + r < rows && c0 + c < cols) {  // cols % 4 == 0: the whole group is in range
            const uint2 v = *reinterpret_cast<const uint2*>(src + base + static_cast<long long>(r0 + r) * cols + c0 + c);
            tile[r][c] = static_cast<unsigned short>(v.x & 0xffffu);
            tile[r][c + 1] = static_cast<unsigned short>(v.x >> 16);
            tile[r][c + 2] = static_cast<unsigned short>(v.y & 0xffffu);
            tile[r][c + 3] = static_cast<unsigned short>(v.y >> 16);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = i * 16 + t / 16;
        const int r = 4 * (t % 16);
        if (r0 + r < rows && c0 + c < cols) {  // rows % 4 == 0: rows r .. r + 3 are in range
            const uint2 v = make_uint2(static_cast<unsigned>(tile[r][c]) | (static_cast<unsigned>(tile[r + 1][c]) << 16),
                                       static_cast<unsigned>(tile[r + 2][c]) | (static_cast<unsigned>(tile[r + 3][c]) << 16));
            *reinterpret_cast<uint2*>(dst + base + static_cast<long long>(c0 + c) * rows + r0 + r) = v;
        }
    }
}

// Up to kMaxTransposeJobs transposes of 16-bit [batch, rows, cols] matrices in one launch: the jobs'
// 64 x 64 tiles are numbered one after another (job j's tiles from tile_start[j]), each workgroup
// finds its job by a scan of the table held in its kernel arguments and runs transpose16_vec's body
// on that tile (rows and cols multiples of 4, 8-byte aligned buffers).
constexpr int kMaxTransposeJobs = 8;
struct TransposeJobs {
    int count;
    const unsigned short* src[kMaxTransposeJobs];
    unsigned short* dst[kMaxTransposeJobs];
    int rows[kMaxTransposeJobs], cols[kMaxTransposeJobs];
    long long tile_start[kMaxTransposeJobs + 1];
};

__global__ __launch_bounds__(256) void transpose16_jobs(TransposeJobs jobs) {
    __shared__ unsigned short tile[64][66];
    const long long id = blockIdx.x;
    int j = 0;
    while (j + 1 < jobs.count && id >= jobs.tile_start[j + 1]) ++j;
    const int rows = jobs.rows[j], cols = jobs.cols[j];
    const long long local = id - jobs.tile_start[j];
    const int col_tiles = (cols + 63) / 64, row_tiles = (rows + 63) / 64;
    const long long b = local / (static_cast<long long>(col_tiles) * row_tiles);
    const int within = static_cast<int>(local - b * col_tiles * row_tiles);
    const long long base = b * rows * cols;
    const int r0 = (within / col_tiles) * 64;
    const int c0 = (within % col_tiles) * 64;
    const unsigned short* src = jobs.src[j];
    unsigned short* dst = jobs.dst[j];
    const int t = static_cast<int>(threadIdx.x);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = i * 16 + t / 16;
        const int c = 4 * (t % 16);
        if (r0 + r < rows && c0 + c < cols) {
            const uint2 v = *reinterpret_cast<const uint2*>(src + base + static_cast<long long>(r0 + r) * cols + c0 + c);
            tile[r][c] = static_cast<unsigned short>(v.x & 0xffffu);
            tile[r][c + 1] = static_cast<unsigned short>(v.x >> 16);
            tile[r][c + 2] = static_cast<unsigned short>(v.y & 0xffffu);
            tile[r][c + 3] = static_cast<unsigned short>(v.y >> 16);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = i * 16 + t / 16;
        const int r = 4 * (t % 16);
        if (r0 + r < rows && c0 + c < cols) {
            const uint2 v = make_uint2(static_cast<unsigned>(tile[r][c]) | (static_cast<unsigned>(tile[r + 1][c]) << 16),
                                       static_cast<unsigned>(tile[r + 2][c]) | (static_cast<unsigned>(tile[r + 3][c]) << 16));
            *reinterpret_cast<uint2*>(dst + base + static_cast<long long>(c0 + c) * rows + r0 + r) = v;
        }
    }
}

}  // namespace gemm

// Row-major batched GEMM with optional split-K.  See the header for the
// argument contract.  Returns 0.
int run_gemm(int mode, int a_bf16, int b_bf16, int a_kcontig, int b_kcontig, int m, int n, int k, int batch,
             const void* a, long long lda, long long stride_a, const void* b, long long ldb, long long stride_b,
             const float* c, float* d, long long ldd, long long stride_d, const float* bias, long long stride_bias,
             float beta, int epilogue, int splits, float* workspace, std::size_t workspace_bytes, hipStream_t stream,
             unsigned short* d_bf16, float* moments, float* a_sums) {
    require(mode >= 0 && mode <= 3,
            "GEMM mode must be 0 (fp32), 1 (bf16 operands), 2 (fp32 on bf16 pieces) or 3 (fp16 operands).");
    const bool half_mode = mode == 1 || mode == 3;  // 16-bit MFMA operands, K tiles of 32
    require(half_mode || !(a_bf16 || b_bf16), "fp32 GEMM modes require fp32 operands.");
    require(m > 0 && n > 0 && k > 0 && batch > 0, "GEMM dimensions must be positive.");
    require(a && b && (d || (mode == 1 && d_bf16)),
            "GEMM operands must be nonnull (bf16 mode may write the bf16 copy alone, with d null).");
    require(mode != 3 || (!d_bf16 && !moments), "The fp16 mode writes the fp32 output only.");
    require(std::isfinite(beta) && (beta == 0.0f || c), "Nonzero beta requires C; beta must be finite.");
    require(epilogue >= 0 && epilogue <= 3, "Unknown GEMM epilogue.");
    require(epilogue != 3 || (!half_mode && c && beta == 0.0f && !bias),
            "The ELU-gradient epilogue needs fp32 mode, the ELU outputs as C, beta 0 and no bias.");
    require(splits >= 1, "GEMM split count must be positive.");
    require(static_cast<long long>(m) * n <= std::numeric_limits<int>::max(), "GEMM output exceeds 2^31 elements.");
    require(!a_sums || (!half_mode && !bias), "Row sums of A are produced by the fp32 GEMM family, without a bias.");
    // the row sums take the bias layout: member e at a_sums + e * stride_bias (m when stride_bias is 0)
    const long long sums_stride = stride_bias > 0 ? stride_bias : m;
    require(!moments || (ldd == n && aligned(moments, 16)),
            "GEMM output moments need a row-contiguous output (ldd == n) and 16-byte aligned storage.");
    gemm::Params p{};
    p.a = a;
    p.b = b;
    p.bias = bias;
    p.lda = lda;
    p.ldb = ldb;
    p.ldd = ldd;
    p.stride_a = stride_a;
    p.stride_b = stride_b;
    p.stride_d = stride_d;
    p.stride_bias = stride_bias;
    p.m = m;
    p.n = n;
    p.k = k;
    p.batch = batch;
    p.c = c;
    p.beta = beta;
    p.epilogue = epilogue;
    p.d_bf16 = d_bf16;
    p.k_per_split = gemm::split_depth(mode, k, splits);
    p.splits = splits;
    const std::size_t a_elem = a_bf16 ? 2 : 4;
    const std::size_t b_elem = b_bf16 ? 2 : 4;
    p.a_vec = aligned(a, 16) && (lda * a_elem) % 16 == 0 && (stride_a * a_elem) % 16 == 0;
    p.b_vec = aligned(b, 16) && (ldb * b_elem) % 16 == 0 && (stride_b * b_elem) % 16 == 0;
    if (splits > 1) {
        const std::size_t need = static_cast<std::size_t>(splits) * batch *
                                 (static_cast<std::size_t>(m) * n + (a_sums ? m : 0)) * sizeof(float);
        require(workspace && workspace_bytes >= need && aligned(workspace, 16),
                "Split-K GEMM workspace is null, misaligned or too small.");
        p.d = workspace;
        p.a_sums = a_sums ? workspace + static_cast<std::size_t>(splits) * batch * m * n : nullptr;
        p.c = nullptr;
        p.beta = 0.0f;
        p.epilogue = 0;
        p.d_bf16 = nullptr;
    } else {
        p.d = d;
        p.a_sums = a_sums;
        p.sums_stride = sums_stride;
    }
    p.out_vec = n % 4 == 0 && aligned(p.d, 16) && (splits > 1 || (ldd % 4 == 0 && stride_d % 4 == 0)) &&
                (splits > 1 || ((!bias || (aligned(bias, 16) && stride_bias % 4 == 0)) &&
                                (beta == 0.0f || aligned(c, 16)) && (!d_bf16 || aligned(d_bf16, 8))));
    // Column moments come from the 256x256 kernel's epilogue when it runs this
    // product in direct mode with the identity epilogue; otherwise from a pass over D.
    const bool fused_moments = moments && mode == 1 && splits == 1 && !bias && epilogue == 0 && beta == 0.0f &&
                               gemm::big_eligible(p, a_bf16, b_bf16);
    p.moments = fused_moments ? moments : nullptr;
    if (mode == 1) gemm::launch_bf16(p, a_bf16, b_bf16, a_kcontig != 0, b_kcontig != 0, stream);
    else if (mode == 3) gemm::launch_f16(p, a_bf16, b_bf16, a_kcontig != 0, b_kcontig != 0, stream);
    else if (mode == 2 && gemm::split_eligible(p, a_kcontig != 0))
        gemm::launch_split(p, a_kcontig != 0, b_kcontig != 0, stream);
    else gemm::launch_fp32(p, a_kcontig != 0, b_kcontig != 0, stream);
    check_launch("Launch GEMM");
    if (splits > 1) {
        const long long total = static_cast<long long>(batch) * m * n;
        const unsigned blocks = static_cast<unsigned>(std::min<long long>((total + 255) / 256, 4096));
        const bool grouped = splits >= 2 * gemm::kReduceGroups && total <= (1LL << 22);
        const float* sums_work = workspace + static_cast<std::size_t>(splits) * batch * m * n;
        if (grouped)  // the row sums of A ride in the same launch
            hipLaunchKernelGGL(gemm::splitk_reduce_grouped,
                               dim3(ceil_div(total + (a_sums ? static_cast<long long>(batch) * m : 0),
                                             gemm::kReduceCols)),
                               dim3(256), 0, stream, workspace, d, d_bf16, c, bias, ldd, stride_d, stride_bias, m, n,
                               batch, splits, beta, epilogue, a_sums ? sums_work : nullptr, a_sums, sums_stride);
        else if (n % 4 == 0 && ldd % 4 == 0 && stride_d % 4 == 0 && aligned(d, 16) && aligned(d_bf16, 8) &&
                 (!c || aligned(c, 16)) && (!bias || (aligned(bias, 16) && stride_bias % 4 == 0)))
            hipLaunchKernelGGL(gemm::splitk_reduce_vec,
                               dim3(static_cast<unsigned>(std::min<long long>((total / 4 + 255) / 256, 4096))),
                               dim3(256), 0, stream, workspace, d, d_bf16, c, bias, ldd, stride_d, stride_bias, m, n,
                               batch, splits, beta, epilogue);
        else
            hipLaunchKernelGGL(gemm::splitk_reduce, dim3(blocks), dim3(256), 0, stream, workspace, d, d_bf16, c, bias,
                               ldd, stride_d, stride_bias, m, n, batch, splits, beta, epilogue);
        check_launch("Launch split-K reduction");
        if (a_sums && !grouped) {
            // [splits][batch][m] partial row sums -> a_sums, fixed order
            if (splits >= 2 * gemm::kReduceGroups)
                hipLaunchKernelGGL(gemm::splitk_reduce_grouped, dim3(ceil_div(static_cast<long long>(batch) * m,
                                                                               gemm::kReduceCols)),
                                   dim3(256), 0, stream, sums_work, a_sums, nullptr, nullptr, nullptr,
                                   static_cast<long long>(m), sums_stride, 0LL, 1, m, batch, splits, 0.0f, 0, nullptr,
                                   nullptr, 0LL);
            else
                hipLaunchKernelGGL(gemm::splitk_reduce, dim3(ceil_div(static_cast<long long>(batch) * m, 256)),
                                   dim3(256), 0, stream, sums_work, a_sums, nullptr, nullptr, nullptr,
                                   static_cast<long long>(m), sums_stride, 0LL, 1, m, batch, splits, 0.0f, 0);
            check_launch("Launch row-sum reduction");
        }
    }
    if (moments && !fused_moments) {
        if (d) bn_chunk_moments(batch, d, 0, stride_d, moments, m, n, stream);
        else bn_chunk_moments(batch, d_bf16, 1, stride_d, moments, m, n, stream);
    }
    return 0;
}

}  // namespace rl

RL_API int rl_gemm(int mode, int a_bf16, int b_bf16, int a_kcontig, int b_kcontig, int m, int n, int k, int batch,
                   const void* a, long long lda, long long stride_a, const void* b, long long ldb, long long stride_b,
                   const float* c, float* d, long long ldd, long long stride_d, const float* bias,
                   long long stride_bias, float beta, int epilogue, int splits, float* workspace,
                   std::size_t workspace_bytes, void* d_bf16, float* moments, float* a_sums,
                   void* stream) noexcept {
    return rl::guarded("rl_gemm", [&] {
        rl::run_gemm(mode, a_bf16, b_bf16, a_kcontig, b_kcontig, m, n, k, batch, a, lda, stride_a, b, ldb, stride_b, c,
                     d, ldd, stride_d, bias, stride_bias, beta, epilogue, splits, workspace, workspace_bytes,
                     rl::as_stream(stream), static_cast<unsigned short*>(d_bf16), moments, a_sums);
    });
}

RL_API std::size_t rl_gemm_workspace(int mode, int m, int n, int k, int batch, int splits) noexcept {
    if (m <= 0 || n <= 0 || k <= 0 || batch <= 0 || splits <= 1) return 0;
    rl::gemm::split_depth(mode, k, splits);
    if (splits <= 1) return 0;
    // D partials plus the row-sum partials of A
    return static_cast<std::size_t>(splits) * batch * (static_cast<std::size_t>(m) * n + m) * sizeof(float);
}

// Several batched 16-bit transposes in one launch (the transposed weight copies of one parameter
// store, refreshed after each optimizer step); no reference counterpart.
RL_API int rl_transpose16_many(int count, const void* const* srcs, void* const* dsts, const int* batch,
                               const int* rows, const int* cols, void* stream) noexcept {
    return rl::guarded("rl_transpose16_many", [&] {
        rl::require(count >= 1 && count <= rl::gemm::kMaxTransposeJobs, "Transpose job count must be 1 to 8.");
        rl::require(srcs && dsts && batch && rows && cols, "Transpose jobs need every array.");
        rl::gemm::TransposeJobs jobs{};
        jobs.count = count;
        long long tiles = 0;
        for (int j = 0; j < count; ++j) {
            rl::require(srcs[j] && dsts[j] && srcs[j] != dsts[j], "Transpose needs distinct source and destination buffers.");
            rl::require(batch[j] > 0 && rows[j] > 0 && cols[j] > 0 && rows[j] % 4 == 0 && cols[j] % 4 == 0 &&
                            rl::aligned(srcs[j], 8) && rl::aligned(dsts[j], 8),
                        "Batched transpose jobs need rows and cols in multiples of 4 and 8-byte aligned buffers.");
            jobs.src[j] = static_cast<const unsigned short*>(srcs[j]);
            jobs.dst[j] = static_cast<unsigned short*>(dsts[j]);
            jobs.rows[j] = rows[j];
            jobs.cols[j] = cols[j];
            jobs.tile_start[j] = tiles;
            tiles += static_cast<long long>(batch[j]) * rl::ceil_div(rows[j], 64) * rl::ceil_div(cols[j], 64);
        }
        jobs.tile_start[count] = tiles;
        rl::require(tiles <= (1LL << 31) - 1, "Too many transpose tiles.");
        hipLaunchKernelGGL(rl::gemm::transpose16_jobs, dim3(static_cast<unsigned>(tiles)), dim3(256), 0,
                           rl::as_stream(stream), jobs);
        rl::check_launch("Launch batched transpose");
    });
}

// Batched transpose of 16-bit matrices (bf16 weight copies laid out K-contiguous
// for the input-gradient product); no reference counterpart.
RL_API int rl_transpose16(const void* src, void* dst, int batch, int rows, int cols, void* stream) noexcept {
    return rl::guarded("rl_transpose16", [&] {
        rl::require(src && dst && src != dst, "Transpose needs distinct source and destination buffers.");
        rl::require(batch > 0 && rows > 0 && cols > 0 && batch <= 65535 && (rows + 63) / 64 <= 65535,
                    "Transpose dimensions are invalid.");
        const dim3 grid(rl::ceil_div(cols, 64), rl::ceil_div(rows, 64), static_cast<unsigned>(batch));
        const bool vec = rows % 4 == 0 && cols % 4 == 0 && rl::aligned(src, 8) && rl::aligned(dst, 8);
        hipLaunchKernelGGL(vec ? rl::gemm::transpose16_vec : rl::gemm::transpose16, grid, dim3(256), 0,
                           rl::as_stream(stream), static_cast<const unsigned short*>(src),
                           static_cast<unsigned short*>(dst), rows, cols);
        rl::check_launch("Launch transpose");
    });
}
