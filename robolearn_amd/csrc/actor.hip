// Eval-mode FlashSAC actor for acting rows in one launch: input BatchNorm, embedder, residual blocks, RMSNorm,
// heads and the tanh (robolearn/flashsac/networks.py:37-61, layers.py:67-166), all in fp32.
//
// A workgroup takes 16 rows through the whole network.  The rows' activations stay in LDS; the weights stream
// from L2 straight into the B operands of v_mfma_f32_16x16x4_f32, one 16-K chunk ahead.  Sixteen waves share the
// output columns, 16 at a time.
//
// What bounds it: the weights' way into one CU, about 30 GB/s however many rows (its misses in flight; with the
// weights in L1 the 256-wide network of two blocks takes 83 instead of 134 us, at an fp32 matrix floor of 57 us).  So
// it is the faster way where the layer-by-layer path is all launches: observations to actions, one launch against the
// layers issued one by one / captured in a graph, obs 4, hidden 128, one block, 64 rows 22 us against 98 / 43; obs 17,
// hidden 64, one block, 4096 rows 13 us against 108 / 42; obs 60, hidden 200, two blocks, 64 rows 85 us against 140 /
// 90 and 4096 rows 87 us against 137 / 122; obs 123, hidden 256, two blocks, 1024 rows 134 us against 157 / 110, where
// the caller takes the layers.  Both instances use the 128 registers that sixteen waves leave each other and spill
// three (16 bytes of scratch a lane).  Eight waves and deeper prefetch (two to eight chunks, copied or in turn) were
// no faster.
#include "common.hpp"

#include <cmath>

namespace rl {
namespace actor {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));  // rows of odd length are 4-byte aligned

constexpr int kRows = 16;
constexpr int kWaves = 16;
constexpr int kThreads = kWaves * kWave;
constexpr int kMaxBlocks = 8;

struct Norm {
    const float *mean, *var, *w, *b;
};

struct Block {
    const float* w1;
    Norm n1;
    const float* w2;
    Norm n2;
};

struct Args {
    const float* obs;
    long long ld_obs;
    long long rows;
    int obs_dim, hidden, blocks, action_dim;
    Norm input;
    const float* embed;
    Block block[kMaxBlocks];
    const float *post, *head_w, *head_b;
    const float* noise;  // [rows, action_dim], null: deterministic
    float* actions;
    float bn_eps, rms_eps;
};

// One column's normalization: __fmaf_rn((x - mean) * inv, w, b), as the BatchNorm kernels form it.
struct ColumnNorm {
    float mean, inv, w, b;
    __device__ __forceinline__ ColumnNorm(const Norm& n, int c, float eps)
        : mean(n.mean[c]), inv(1.0f / sqrtf(n.var[c] + eps)), w(n.w[c]), b(n.b[c]) {}
    __device__ __forceinline__ float operator()(float x) const { return __fmaf_rn((x - mean) * inv, w, b); }
};

__device__ __forceinline__ int round16(int n) { return (n + 15) & ~15; }

// U blocks of 16 output columns, `first` and every kWaves-th after it: acc[u] = in[16, K] . W[col, K]^T.  in: LDS
// rows of `pitch` floats, zero from K to the next multiple of 16.  Lane l feeds row l % 16 of `in`, row l % 16 of
// the block's weights and the K values 16 c + 4 (l / 16) + j of chunk c to the j-th of the chunk's four
// instructions: the same permutation of K on both sides.
template <int U>
__device__ __forceinline__ void multiply(const float* in, int pitch, int k, const float* w, int n, int first,
                                         f32x4_t (&acc)[U]) {
    const int lane = static_cast<int>(threadIdx.x) % kWave;
    const int kg = 4 * (lane / 16);
    const float* a = in + (lane % 16) * pitch + kg;
    const float* rows[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        acc[u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        // columns past the end repeat the last one and are not stored
        rows[u] = w + static_cast<long long>(min(16 * (first + u * kWaves) + lane % 16, n - 1)) * k + kg;
    }
    const auto step = [&](const f32x4_t& x, const f32x4_t (&b)[U]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int u = 0; u < U; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], b[u][j], acc[u], 0, 0, 0);
    };
    const int whole = k / 16;
    f32x4_t next[U];
    const auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < U; ++u) next[u] = *reinterpret_cast<const f32x4u_t*>(rows[u] + 16 * c);
    };
    if (whole > 0) load(0);
    for (int c = 0; c < whole; ++c) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(a + 16 * c);
        f32x4_t b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) b[u] = next[u];
        if (c + 1 < whole) load(c + 1);
        step(x, b);
    }
    if (whole * 16 < k) {
        f32x4_t b[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) b[u][e] = 16 * whole + kg + e < k ? rows[u][16 * whole + e] : 0.0f;
        step(*reinterpret_cast<const f32x4_t*>(a + 16 * whole), b);
    }
}

template <int U, class Column>
__device__ __forceinline__ void product_blocks(const float* in, int pitch, int k, const float* w, int n, Column&& column) {
    const int wave = static_cast<int>(threadIdx.x) / kWave, lane = static_cast<int>(threadIdx.x) % kWave;
    const int blocks = (n + 15) / 16;
    for (int first = wave; first < blocks; first += U * kWaves) {
        f32x4_t acc[U];
        multiply<U>(in, pitch, k, w, n, first, acc);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = 16 * (first + u * kWaves) + lane % 16;
            if (first + u * kWaves < blocks) column(c, 4 * (lane / 16), acc[u]);
        }
    }
}

// column(c, first row, four consecutive rows' sums), once per column c < round16(n)
template <class Column>
__device__ __forceinline__ void product(const float* in, int pitch, int k, const float* w, int n, Column&& column) {
    const int blocks = (n + 15) / 16;
    if (blocks > 2 * kWaves) product_blocks<4>(in, pitch, k, w, n, column);
    else if (blocks > kWaves) product_blocks<2>(in, pitch, k, w, n, column);
    else product_blocks<1>(in, pitch, k, w, n, column);
}

// H: the widest hidden layer the LDS holds.
template <int H>
__global__ __launch_bounds__(kThreads) void act_kernel(Args a) {
    // pitches of 4 (mod 64) floats: the 16 rows of an operand read start 4 banks apart
    constexpr int WidePitch = 4 * H + 4, Pitch = H + 4;
    __shared__ __attribute__((aligned(16))) float wide[kRows * WidePitch];
    __shared__ __attribute__((aligned(16))) float stream[kRows * Pitch];
    const int t = static_cast<int>(threadIdx.x);
    const long long r0 = static_cast<long long>(blockIdx.x) * kRows;
    const int h = a.hidden, in_dim = a.obs_dim, in_pad = round16(in_dim), h_pad = round16(h);

    for (int i = t; i < kRows * in_pad; i += kThreads) {
        const int r = i / in_pad, c = i % in_pad;
        const long long row = min(r0 + r, a.rows - 1);
        wide[r * WidePitch + c] = c < in_dim ? ColumnNorm(a.input, c, a.bn_eps)(a.obs[row * a.ld_obs + c]) : 0.0f;
    }
    __syncthreads();
    product(wide, WidePitch, in_dim, a.embed, h, [&](int c, int r, const f32x4_t& v) {
#pragma unroll
        for (int e = 0; e < 4; ++e) stream[(r + e) * Pitch + c] = c < h ? v[e] : 0.0f;
    });
    __syncthreads();
    for (int i = 0; i < a.blocks; ++i) {
        const Block& block = a.block[i];
        product(stream, Pitch, h, block.w1, 4 * h, [&](int c, int r, const f32x4_t& v) {
            const bool in = c < 4 * h;
            const ColumnNorm norm(block.n1, in ? c : 0, a.bn_eps);
#pragma unroll
            for (int e = 0; e < 4; ++e) wide[(r + e) * WidePitch + c] = in ? fmaxf(norm(v[e]), 0.0f) : 0.0f;
        });
        __syncthreads();
        product(wide, WidePitch, 4 * h, block.w2, h, [&](int c, int r, const f32x4_t& v) {
            if (c >= h) return;  // the padding stays zero
            const ColumnNorm norm(block.n2, c, a.bn_eps);
#pragma unroll
            for (int e = 0; e < 4; ++e) stream[(r + e) * Pitch + c] += fmaxf(norm(v[e]), 0.0f);
        });
        __syncthreads();
    }
    // RMSNorm
    {
        constexpr int PerRow = kThreads / kRows;
        const int r = t / PerRow, l = t % PerRow;
        float s = 0.0f;
        for (int c = l; c < h; c += PerRow) s += stream[r * Pitch + c] * stream[r * Pitch + c];
#pragma unroll
        for (int offset = PerRow / 2; offset > 0; offset >>= 1) s += __shfl_xor(s, offset);
        const float rs = 1.0f / sqrtf(s / static_cast<float>(h) + a.rms_eps);
        for (int c = l; c < h_pad; c += PerRow) wide[r * WidePitch + c] = c < h ? stream[r * Pitch + c] * rs * a.post[c] : 0.0f;
    }
    __syncthreads();
    const int A = a.action_dim, heads = a.noise ? 2 * A : A;
    product(wide, WidePitch, h, a.head_w, heads, [&](int c, int r, const f32x4_t& v) {
        if (c >= heads) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) stream[(r + e) * Pitch + c] = v[e] + a.head_b[c];
    });
    __syncthreads();
    for (int i = t; i < kRows * A; i += kThreads) {
        const int r = i / A, j = i % A;
        if (r0 + r >= a.rows) break;
        float raw = stream[r * Pitch + j];
        if (a.noise) {
            const float log_std = -10.0f + 6.0f * (1.0f + tanhf(stream[r * Pitch + A + j]));
            raw += a.noise[(r0 + r) * A + j] * expf(log_std);
        }
        a.actions[(r0 + r) * A + j] = tanhf(raw);
    }
}

}  // namespace actor
}  // namespace rl

RL_API int rl_actor_act(long long rows, int obs_dim, int hidden, int blocks, int action_dim, const float* obs,
                        long long ld_obs, const void* const* parameters, const float* noise, float* actions,
                        float bn_eps, float rms_eps, void* stream) noexcept {
    using namespace rl::actor;
    return rl::guarded("rl_actor_act", [&] {
        rl::require(rows > 0 && obs_dim > 0 && hidden > 0 && blocks >= 0 && action_dim > 0 && ld_obs >= obs_dim,
                    "Acting needs positive dimensions.");
        rl::require(hidden <= 256 && blocks <= kMaxBlocks && obs_dim <= 1024 && 2 * action_dim <= 256,
                    "The one-launch actor takes hidden widths and 2 x actions up to 256, observations up to 1024 and 8 blocks.");
        rl::require((rows + kRows - 1) / kRows <= 0x7FFFFFFF, "Too many acting rows.");
        rl::require(obs && parameters && actions, "Acting needs observations, parameters and an output.");
        Args a{};
        a.obs = obs;
        a.ld_obs = ld_obs;
        a.rows = rows;
        a.obs_dim = obs_dim;
        a.hidden = hidden;
        a.blocks = blocks;
        a.action_dim = action_dim;
        const void* const* next = parameters;
        const auto take = [&]() {
            rl::require(*next, "Acting parameters must be nonnull.");
            return static_cast<const float*>(*next++);
        };
        const auto take_norm = [&](Norm& n) {
            n.mean = take();
            n.var = take();
            n.w = take();
            n.b = take();
        };
        take_norm(a.input);
        a.embed = take();
        for (int i = 0; i < blocks; ++i) {
            a.block[i].w1 = take();
            take_norm(a.block[i].n1);
            a.block[i].w2 = take();
            take_norm(a.block[i].n2);
        }
        a.post = take();
        a.head_w = take();
        a.head_b = take();
        a.noise = noise;
        a.actions = actions;
        a.bn_eps = bn_eps;
        a.rms_eps = rms_eps;
        const dim3 grid(static_cast<unsigned>((rows + kRows - 1) / kRows));
        if (hidden <= 128 && obs_dim <= 512 && 2 * action_dim <= 128)
            hipLaunchKernelGGL(act_kernel<128>, grid, dim3(kThreads), 0, rl::as_stream(stream), a);
        else
            hipLaunchKernelGGL(act_kernel<256>, grid, dim3(kThreads), 0, rl::as_stream(stream), a);
        rl::check_launch("Launch actor");
    });
}
