// bf16 products on 64 x 64 output tiles: embedders (K = a handful of observations), categorical and policy heads
// (N or M = bins or actions) and other shapes of few or ragged tiles.  bf16 operands, fp32 accumulation.
//
// What bounds it: at a few thousand rows the launch and one workgroup's serial chain (load, LDS, products, store), at
// many the traffic of the operands and of D.  On 256 x 128 tiles the same products ran 8 to 128 workgroups of 10 us
// plus 0.65 us per 32 of K, and read rows of odd length (39, 101, 123 values) one value at a time.  Here a thousand
// small workgroups overlap each other's chains, and rows load 16 bytes (M/N-contiguous ones, pairs of rows, 4
// bytes) at any even address.  Twin critics, 256 x 128 tiles against these, bit-identical: 4096 x 512 over K = 39
// 20.1 -> 9.7 us, 2048 x 101 over 512 with its split 21.3 -> 11.7 us, 101 x 512 over 2048 with its split 21.7 -> 11.6 us,
// 4096 x 39 over 512 23.5 -> 11.4 us; 101 x 1024 over 8192 50.5 -> 27.8 us, 16384 x 160 over 1024 52.8 -> 39.8 us; one
// member, 16384 x 256 over 123 31.3 -> 10.8 us.
#include "gemm.hpp"

namespace rl {
namespace gemm {
namespace narrow {

constexpr int kTileEdge = 64;
constexpr int kDepth = 64;  // K per LDS step
constexpr int kStagePitch = kTileEdge + 4;

// Element offset of 16-byte chunk c of LDS row r: the XOR puts the 16 rows that one phase of a ds_read_b128
// touches in 16 distinct 16-byte bank groups.
__device__ __forceinline__ int slot(int r, int c) { return r * kDepth + ((c ^ ((r >> 1) & 7)) << 3); }

// bf16 rows of odd length start at any even address; global loads need no more alignment than that.
struct __attribute__((packed, aligned(2))) Chunk {
    unsigned w[4];
};
struct __attribute__((packed, aligned(2))) Pair {
    unsigned w;
};

// One 64 x 64 (row, K) operand tile in registers.  Element (r, k) is src[r * ld + k] when KContig, else src[k *
// ld + r].  Rows past the end repeat the last row: their products land in outputs that are not written.
// Each thread holds two chunks of 8 K: KContig, of rows t / 8 and 32 + t / 8; else of rows 2 (t % 32) and the next,
// read as pairs (in the last pair of an odd row count, the row before and the row).
template <bool KContig>
struct Loader {
    uint4 chunk[2];
    unsigned offset[2];  // byte offsets in the tile
    unsigned low;        // byte selector of the first row of a pair
    int k_first;
    bool pairs;

    __device__ __forceinline__ void init(long long ld, int rows) {
        const int t = static_cast<int>(threadIdx.x);
        k_first = 8 * (KContig ? t % 8 : t / 32);
        if constexpr (KContig) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                offset[i] = 2u * (static_cast<unsigned>(min(t / 8 + 32 * i, rows - 1)) * static_cast<unsigned>(ld) + k_first);
        } else {
            const int r = min(2 * (t % 32), rows - 1);
            pairs = rows >= 2;
            const bool alone = r == rows - 1;  // read with the row before it
            offset[0] = 2u * (pairs && alone ? r - 1 : r);
            low = alone ? 0x07060302u : 0x05040100u;
        }
    }

    __device__ __forceinline__ static const char* bytes(const unsigned short* p) { return reinterpret_cast<const char*>(p); }

    // tile: the operand at the tile's first row and the step's first K, `left` values of K left
    __device__ __forceinline__ void load(const unsigned short* tile, long long ld, int left) {
        if constexpr (KContig) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const char* q = bytes(tile) + offset[i];
                if (k_first + 8 <= left) {
                    const Chunk c = *reinterpret_cast<const Chunk*>(q);
                    chunk[i] = make_uint4(c.w[0], c.w[1], c.w[2], c.w[3]);
                } else {
                    unsigned w[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const unsigned short* p = reinterpret_cast<const unsigned short*>(q) + 2 * e;
                        const unsigned lo = k_first + 2 * e < left ? p[0] : 0u;
                        const unsigned hi = k_first + 2 * e + 1 < left ? p[1] : 0u;
                        w[e] = lo | (hi << 16);
                    }
                    chunk[i] = make_uint4(w[0], w[1], w[2], w[3]);
                }
            }
        } else {
            const unsigned short* q = tile + k_first * ld;
            unsigned v[8];
            if (!pairs) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = k_first + e < left ? static_cast<unsigned>(q[e * ld]) << 16 : 0u;
            } else if (left >= kDepth) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = reinterpret_cast<const Pair*>(bytes(q + e * ld) + offset[0])->w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    v[e] = k_first + e < left ? reinterpret_cast<const Pair*>(bytes(q + e * ld) + offset[0])->w : 0u;
            }
            constexpr unsigned kHigh = 0x07060302u;  // the high halves of the second operand, then of the first
            chunk[0] = make_uint4(__builtin_amdgcn_perm(v[1], v[0], low), __builtin_amdgcn_perm(v[3], v[2], low),
                                  __builtin_amdgcn_perm(v[5], v[4], low), __builtin_amdgcn_perm(v[7], v[6], low));
            chunk[1] = make_uint4(__builtin_amdgcn_perm(v[1], v[0], kHigh), __builtin_amdgcn_perm(v[3], v[2], kHigh),
                                  __builtin_amdgcn_perm(v[5], v[4], kHigh), __builtin_amdgcn_perm(v[7], v[6], kHigh));
        }
    }

    __device__ __forceinline__ void store(unsigned short* lds) const {
        const int t = static_cast<int>(threadIdx.x);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = KContig ? t / 8 + 32 * i : 2 * (t % 32) + i;
            *reinterpret_cast<uint4*>(lds + slot(r, k_first / 8)) = chunk[i];
        }
    }
};

// 4 waves, 2 x 2, of one 32 x 32 accumulator each.
template <bool AK, bool BK>
__global__ __launch_bounds__(kThreads) void narrow_kernel(Params p) {
    // the K loop's two operand tiles; the epilogue's output tile
    __shared__ __attribute__((aligned(16))) unsigned char lds[kTileEdge * kStagePitch * 4];
    static_assert(sizeof(lds) >= 2 * kTileEdge * kDepth * 2, "the operand tiles fit");
    unsigned short* sa = reinterpret_cast<unsigned short*>(lds);
    unsigned short* sb = sa + kTileEdge * kDepth;

    // XCD-aware tile order, as in the other products: each XCD takes a contiguous range of tiles
    const unsigned nx = gridDim.x, ny = gridDim.y;
    const unsigned groups = nx * ny * gridDim.z;
    unsigned w = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
    if (groups % 8 == 0) w = (w % 8) * (groups / 8) + w / 8;
    const int m0 = static_cast<int>((w / nx) % ny) * kTileEdge, n0 = static_cast<int>(w % nx) * kTileEdge;
    const int bz = static_cast<int>(w / (nx * ny));
    const int split = bz % p.splits, batch = bz / p.splits;
    const int k_begin = split * p.k_per_split;
    int left = min(p.k, k_begin + p.k_per_split) - k_begin;
    const unsigned short* A = static_cast<const unsigned short*>(p.a) + batch * p.stride_a +
                              (AK ? m0 * p.lda + k_begin : k_begin * p.lda + m0);
    const unsigned short* B = static_cast<const unsigned short*>(p.b) + batch * p.stride_b +
                              (BK ? n0 * p.ldb + k_begin : k_begin * p.ldb + n0);
    const long long step_a = AK ? kDepth : kDepth * p.lda, step_b = BK ? kDepth : kDepth * p.ldb;

    const int t = static_cast<int>(threadIdx.x);
    const int lane = t % kWave, wave = t / kWave, wm = wave / 2, wn = wave % 2;
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    Loader<AK> la;
    Loader<BK> lb;
    la.init(p.lda, p.m - m0);
    lb.init(p.ldb, p.n - n0);
    la.load(A, p.lda, left);
    lb.load(B, p.ldb, left);
    for (;;) {
        la.store(sa);
        lb.store(sb);
        const int steps = min(left, kDepth);
        left -= kDepth;
        if (left > 0) {
            A += step_a;
            B += step_b;
            la.load(A, p.lda, left);
            lb.load(B, p.ldb, left);
        }
        __syncthreads();
        // 32 K per pair of instructions, lane l holding chunks s + 2 (l / 32) of them, as the 256 x 128 kernel
        // multiplies them: both give the same sums
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (half * 32 >= steps) break;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int c = 4 * half + s + 2 * (lane / 32);
                const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(sa + slot(wm * 32 + lane % 32, c));
                const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(sb + slot(wn * 32 + lane % 32, c));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
            }
        }
        __syncthreads();
        if (left <= 0) break;
    }

    const bool direct = p.splits == 1;
    const long long ldd = direct ? p.ldd : p.n;
    const long long tile = (direct ? batch * p.stride_d
                                   : (static_cast<long long>(split) * p.batch + batch) * static_cast<long long>(p.m) * p.n) +
                           m0 * ldd + n0;
    float* D = p.d ? p.d + tile : nullptr;  // null in direct mode: the bf16 copy alone
    unsigned short* H = direct && p.d_bf16 ? p.d_bf16 + tile : nullptr;
    const float* C = direct && p.beta != 0.0f ? p.c + tile : nullptr;
    const float* bias = direct && p.bias ? p.bias + batch * p.stride_bias + n0 : nullptr;
    const int row = wm * 32 + 4 * (lane / 32), col = wn * 32 + lane % 32;
    if (p.out_vec) {
        // through LDS, so that rows leave as 16-byte (bf16: 8-byte) pieces
        float* stage = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int v = 0; v < 16; ++v) stage[(row + 8 * (v / 4) + v % 4) * kStagePitch + col] = acc[v];
        __syncthreads();
        const int c4 = 4 * (t % 16);
        if (n0 + c4 >= p.n) return;
        float4 bias4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (bias) bias4 = *reinterpret_cast<const float4*>(bias + c4);
        float4 cv[4];
        if (C) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = t / 16 + 16 * i;
                if (m0 + r < p.m) cv[i] = *reinterpret_cast<const float4*>(C + r * ldd + c4);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = t / 16 + 16 * i;
            if (m0 + r >= p.m) break;
            float4 v = *reinterpret_cast<const float4*>(stage + r * kStagePitch + c4);
            const long long at = r * ldd + c4;
            if (direct) {
                v = make_float4(apply_epilogue(v.x + bias4.x, p.epilogue), apply_epilogue(v.y + bias4.y, p.epilogue),
                                apply_epilogue(v.z + bias4.z, p.epilogue), apply_epilogue(v.w + bias4.w, p.epilogue));
                if (C) {
                    v.x += p.beta * cv[i].x;
                    v.y += p.beta * cv[i].y;
                    v.z += p.beta * cv[i].z;
                    v.w += p.beta * cv[i].w;
                }
                if (H) *reinterpret_cast<uint2*>(H + at) = make_uint2(f32x2_to_bf16x2(v.x, v.y), f32x2_to_bf16x2(v.z, v.w));
            }
            if (D) *reinterpret_cast<float4*>(D + at) = v;
        }
        return;
    }
    if (n0 + col >= p.n) return;
    const float bcol = bias ? bias[col] : 0.0f;
    float cv[16];
    if (C) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int r = row + 8 * (v / 4) + v % 4;
            cv[v] = m0 + r < p.m ? C[r * ldd + col] : 0.0f;
        }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int r = row + 8 * (v / 4) + v % 4;
        if (m0 + r >= p.m) break;
        float value = acc[v];
        if (direct) {
            value = apply_epilogue(value + bcol, p.epilogue);
            if (C) value += p.beta * cv[v];
            if (H) H[r * ldd + col] = f32_to_bf16_bits(value);
        }
        if (D) D[r * ldd + col] = value;
    }
}

template <bool AK, bool BK>
void launch(const Params& p, hipStream_t stream) {
    const dim3 grid(ceil_div(p.n, kTileEdge), ceil_div(p.m, kTileEdge), static_cast<unsigned>(p.batch * p.splits));
    hipLaunchKernelGGL((narrow_kernel<AK, BK>), grid, dim3(kThreads), 0, stream, p);
}

}  // namespace narrow

// One round of 256 x 128 tiles (512: two workgroups per CU, however few of them the last round fills) takes about as
// long as `tiles` of the small ones, whose operand reuse is four times smaller; wide_fixed and kNarrowFixed are what a
// tile costs before and after its K loop, in K.
// The lines are fitted to 3416 products of 128 large tiles and more: 1957 random ones (24 to 20000 rows and columns, K
// from 24 to 16000, all layouts, whole and split) and 1459 heads, embedders and gradients of theirs (256 to 32768 rows).
// Of the 1976 that take the small tiles 74 are 3 to 16 % slower there and the others up to 4.5 times faster; of the 1440
// that take the large ones 857 would take up to 2.5 times as long on small ones and 338 would be 5 to 49 % faster.  With
// fewer large tiles the small ones always won (1.18 to 5.8 times faster).  Small against large tiles, twin products: 500
// x 16000 over 1000 100 and 64 us; 8192 x 101 over 1024 in four splits 27 and 40 us; 16384 x 1024 over 160 52 and 54 us;
// 4096 x 512 over 160 10 and 18 us; one member, 16400 x 400 over 8200 421 and 335 us.
// Operands that do not load 16 bytes at a time, which the large tiles read one value at a time, take the small tiles at
// any size: 1.07 to 26 times faster, 3.2 times in the middle, in 1443 random products (3190 x 4972 over 29 is 13 %
// slower); 2396 x 567 over 12951 in four splits, twin: 214 against 919 us.
struct Round {
    int tiles, wide_fixed;
};
constexpr Round kRows{1500, 500};            // both operands K-contiguous
constexpr Round kTransposed{1900, 320};      // an operand that the large tiles transpose
constexpr Round kScalarOutput{1900, 1000};   // output rows that both store one value at a time
constexpr int kWideRound = 512, kNarrowFixed = 192;

bool narrow_eligible(const Params& p, int a_bf16, int b_bf16, bool ak, bool bk) {
    const long long products = static_cast<long long>(p.batch) * p.splits;
    const long long rows = ceil_div(p.m, narrow::kTileEdge);
    // 32-bit offsets inside a tile, and the grid's limits
    if (!a_bf16 || !b_bf16 || p.lda >= (1 << 22) || p.ldb >= (1 << 22) || rows > 65535 || products > 65535) return false;
    if (!p.a_vec || !p.b_vec) return true;
    const long long tiles = rows * ceil_div(p.n, narrow::kTileEdge) * products;
    const long long wide = static_cast<long long>(ceil_div(p.m, 256)) * ceil_div(p.n, 128) * products;
    const long long rounds = (wide + kWideRound - 1) / kWideRound;
    const Round& round = !p.out_vec ? kScalarOutput : ak && bk ? kRows : kTransposed;
    return tiles * (p.k_per_split + kNarrowFixed) < rounds * round.tiles * (p.k_per_split + round.wide_fixed);
}

void launch_narrow(const Params& p, bool ak, bool bk, hipStream_t stream) {
    if (ak && bk) narrow::launch<true, true>(p, stream);
    else if (ak) narrow::launch<true, false>(p, stream);
    else if (bk) narrow::launch<false, true>(p, stream);
    else narrow::launch<false, false>(p, stream);
}

}  // namespace gemm
}  // namespace rl
