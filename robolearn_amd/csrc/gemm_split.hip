// fp32 products on the bf16 matrix cores (mode 2): fp32 operands, results and sums, fp32-accurate.
//
// Every operand value x is split exactly into three bf16 pieces x = x0 + x1 + x2 when its tile is staged in
// LDS, and each 16-K step issues six v_mfma_f32_32x32x16_bf16 for a0b0 + a0b1 + a1b0 + a0b2 + a1b1 + a2b0.  The
// pieces carry 3 x 8 significant bits and the three dropped cross terms are below 2^-26 of the product, so a
// product is as accurate as an fp32 one, at 6 x 32 matrix-core cycles per 16-K step instead of 8 x 64
// (v_mfma_f32_32x32x2_f32).
//
// What bounds it: this kernel issues 1.0 to 1.2 PFLOP/s of bf16 products on random operands and 1.3 to 1.5 on zeros
// or constants (24576 x 512 over 512 and over 2048, batch 2: 150 and 529 us against 108 and 398; the difference is
// power), and between two barriers a wave's split and its products do not overlap, so each is covered only by the
// other waves of its SIMD (three or four).  The K loop loads whole steps without bounds checks (rows past the end
// repeat the last row, the short last step is peeled off), K-contiguous operands 16 bytes at a time whatever the
// rows' alignment, M/N-contiguous ones one value per K with the lanes along the row, and stages unpadded
// XOR-swizzled rows; the epilogue branches once per block and stores through a uniform base plus a lane offset, of
// 32 bits unless the rows lie too far apart (2000 x 2048 over 2048, rows of A 2^22 values apart: 100 us).  Measured against the same tiles with
// checked loads, padded rows and an epilogue with per-element branches and addresses, batch 2, bit-identical:
// 24576 x 512 x 123 with bias and ELU 90.5 -> 63.8 us, 24576 x 256 x 512 with bias and ELU 99.3 -> 82.0 us, 24576 x
// 512 x 256 with the ELU gradient 116.6 -> 97.5 us, 4096 x 512 x 2048 127 -> 103 us, 1024 x 1024 x 256 15.6 -> 11.2
// us, and 4096 x 256 x 1024 (one member) 30.7 -> 20.1 us.  Not kept: 64 x 64 wave tiles and a second LDS buffer
// (one barrier per step), slower at two and three waves per SIMD; two fp16 pieces under per-row exponents (three
// products), a further 10-20 % faster but not the same rounding.
#include "gemm.hpp"

namespace rl {
namespace gemm {

// 16-byte loads of rows that are only 4-byte aligned (global loads need no more)
typedef float f32x4_t __attribute__((ext_vector_type(4), aligned(4)));

// x = x0 + x1 + x2 exactly in bf16 pieces, two values at a time: x0 keeps x's top 8 significant bits (bf16 by
// truncation), r1 = x - x0 is exact in fp32 (same exponent), x1 keeps r1's top 8 bits, and r2 = r1 - x1 has at
// most 8 significant bits left, so x2 = r2 is exact in bf16.  Each piece's bf16 bits are the high half of its
// fp32 bits; one byte permute packs the pieces of a and b into a plane word (a in the low half).
__device__ __forceinline__ void split3_pair(float a, float b, unsigned& p0, unsigned& p1, unsigned& p2) {
    constexpr unsigned kHigh = 0xFFFF0000u;
    constexpr unsigned kHighHalves = 0x07060302u;  // bytes 2, 3 of the second operand, then of the first
    const unsigned ua = __float_as_uint(a), ub = __float_as_uint(b);
    const float ra = a - __uint_as_float(ua & kHigh), rb = b - __uint_as_float(ub & kHigh);
    const unsigned ura = __float_as_uint(ra), urb = __float_as_uint(rb);
    const float sa = ra - __uint_as_float(ura & kHigh), sb = rb - __uint_as_float(urb & kHigh);
    p0 = __builtin_amdgcn_perm(ub, ua, kHighHalves);
    p1 = __builtin_amdgcn_perm(urb, ura, kHighHalves);
    p2 = __builtin_amdgcn_perm(__float_as_uint(sb), __float_as_uint(sa), kHighHalves);
}

// Element offset of 16-byte chunk c of LDS row r (Step bf16 values long).  The XOR puts the 16 rows that one
// phase of a ds_read_b128 touches in 16 distinct 16-byte bank groups.
template <int Step>
__device__ __forceinline__ int slot(int r, int c) {
    static_assert(Step == 32 || Step == 64, "row lengths");
    return Step == 32 ? r * 32 + ((c ^ ((r >> 2) & 3)) << 3) : r * 64 + ((c ^ ((r >> 1) & 7)) << 3);
}

// One Rows x Step operand tile, held in registers between its load and its store to LDS.  Element (r, k) of
// the operand is src[r * ld + k] when KContig, else src[k * ld + r].  Rows past the operand's end repeat its
// last row: their products land in output rows that are not written.
template <bool KContig, int Rows, int Threads, int Step, class Offset>
struct SplitLoader {
    static constexpr int Vec = Step / 4;                  // K-contiguous: float4 per row
    static constexpr int Count = Rows * Step / Threads;   // values per thread
    static constexpr int Owned = KContig ? Count / 4 : 1; // rows this thread holds values of
    float regs[Count];
    Offset offset[Owned];  // byte offset of this thread's values in the tile
    int k_first;           // M/N-contiguous: first K of this thread

    __device__ __forceinline__ int row(int i) const {
        const int t = static_cast<int>(threadIdx.x);
        return KContig ? t / Vec + i * (Threads / Vec) : t % Rows;
    }

    __device__ __forceinline__ void init(long long ld, int rows) {
        const int t = static_cast<int>(threadIdx.x);
#pragma unroll
        for (int i = 0; i < Owned; ++i) {
            const Offset r = static_cast<Offset>(min(row(i), rows - 1));
            offset[i] = KContig ? (r * static_cast<Offset>(ld) + (t % Vec) * 4u) * 4u : r * 4u;
        }
        // uniform over a wave (Rows is a multiple of 64)
        k_first = KContig ? 0 : __builtin_amdgcn_readfirstlane(t / Rows) * Count;
    }

    __device__ __forceinline__ static const float* at(const float* p, Offset bytes) {
        return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes);
    }

    // tile: the operand at the tile's first row and the step's first K; all Step values of K are in the operand
    __device__ __forceinline__ void load(const float* tile, long long ld) {
        if constexpr (KContig) {
#pragma unroll
            for (int i = 0; i < Owned; ++i) {
                const f32x4_t x = *reinterpret_cast<const f32x4_t*>(at(tile, offset[i]));
#pragma unroll
                for (int e = 0; e < 4; ++e) regs[i * 4 + e] = x[e];
            }
        } else {
            const float* q = tile + k_first * ld;
#pragma unroll
            for (int e = 0; e < Count; ++e) regs[e] = *at(q + e * ld, offset[0]);
        }
    }

    // the last, short step: K from `left` on is zero
    __device__ __forceinline__ void load_tail(const float* tile, long long ld, int left) {
        if constexpr (KContig) {
            const int k = (static_cast<int>(threadIdx.x) % Vec) * 4;
#pragma unroll
            for (int i = 0; i < Owned; ++i) {
                const float* q = at(tile, offset[i]);
#pragma unroll
                for (int e = 0; e < 4; ++e) regs[i * 4 + e] = k + e < left ? q[e] : 0.0f;
            }
        } else {
            const float* q = tile + k_first * ld;
#pragma unroll
            for (int e = 0; e < Count; ++e) regs[e] = k_first + e < left ? *at(q + e * ld, offset[0]) : 0.0f;
        }
    }

    // the three bf16 planes of the tile, plane q at lds + q * Rows * Step
    __device__ __forceinline__ void store(unsigned short* lds) const {
        constexpr int Plane = Rows * Step;
        if constexpr (KContig) {
            const int v = static_cast<int>(threadIdx.x) % Vec;
#pragma unroll
            for (int i = 0; i < Owned; ++i) {
                unsigned w[3][2];
                split3_pair(regs[i * 4], regs[i * 4 + 1], w[0][0], w[1][0], w[2][0]);
                split3_pair(regs[i * 4 + 2], regs[i * 4 + 3], w[0][1], w[1][1], w[2][1]);
                unsigned short* at = lds + slot<Step>(row(i), v / 2) + (v % 2) * 4;
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(at + q * Plane) = make_uint2(w[q][0], w[q][1]);
            }
        } else {
            static_assert(KContig || Count % 8 == 0, "whole 16-byte chunks");
#pragma unroll
            for (int c = 0; c < Count / 8; ++c) {
                unsigned w[3][4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    split3_pair(regs[c * 8 + 2 * e], regs[c * 8 + 2 * e + 1], w[0][e], w[1][e], w[2][e]);
                unsigned short* at = lds + slot<Step>(row(0), k_first / 8 + c);
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    *reinterpret_cast<uint4*>(at + q * Plane) = make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]);
            }
        }
    }
};

// TM x TN output tile of WGM x WGN waves; MinWaves: the waves per SIMD the register allocation aims at (under a
// bound of 2 the 128 x 128 kernels still take 114 to 130 registers, so four waves, or three with an M-contiguous A
// and a K-contiguous B, and have better schedules: 99.4 -> 96.3 us).
// Offset: of a value in its tile, unsigned where that holds a tile's rows at their pitch.
template <int TM, int TN, int WGM, int WGN, int Step, int MinWaves, class Offset, bool AK, bool BK>
__global__ __launch_bounds__(WGM * WGN * kWave) __attribute__((amdgpu_waves_per_eu(MinWaves))) void split_kernel(
    Params p) {
    constexpr int Threads = WGM * WGN * kWave;
    constexpr int WTM = TM / WGM, WTN = TN / WGN;  // wave tile
    constexpr int WBM = WTM / 32, WBN = WTN / 32;  // 32x32 accumulator blocks per wave
    constexpr int PlaneA = TM * Step, PlaneB = TN * Step;
    __shared__ __attribute__((aligned(16))) unsigned short sa[3 * PlaneA];
    __shared__ __attribute__((aligned(16))) unsigned short sb[3 * PlaneB];

    // XCD-aware tile order: workgroups are dispatched round-robin over the 8 XCDs in linear (x fastest) order,
    // so logical tile id (w % 8) * (G / 8) + w / 8 gives each XCD a contiguous range of tiles; the N tiles of
    // one M panel then share that XCD's L2 instead of fetching the panel once per XCD.
    const unsigned nx = gridDim.x, ny = gridDim.y;
    const unsigned groups = nx * ny * gridDim.z;
    unsigned w = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
    if (groups % 8 == 0) w = (w % 8) * (groups / 8) + w / 8;
    const int bx = static_cast<int>(w % nx);
    const int by = static_cast<int>((w / nx) % ny);
    const int bz = static_cast<int>(w / (nx * ny));
    const int split = bz % p.splits;
    const int batch = bz / p.splits;
    const int m0 = by * TM, n0 = bx * TN;
    const int k_begin = split * p.k_per_split;
    const int k_count = min(p.k, k_begin + p.k_per_split) - k_begin;
    const float* A = static_cast<const float*>(p.a) + batch * p.stride_a + (AK ? m0 * p.lda + k_begin : k_begin * p.lda + m0);
    const float* B = static_cast<const float*>(p.b) + batch * p.stride_b + (BK ? n0 * p.ldb + k_begin : k_begin * p.ldb + n0);
    const long long step_a = AK ? Step : Step * p.lda, step_b = BK ? Step : Step * p.ldb;

    const int t = static_cast<int>(threadIdx.x);
    const int lane = t % kWave, wave = t / kWave;
    const int wm = wave / WGN, wn = wave % WGN;

    f32x16_t acc[WBM][WBN];
#pragma unroll
    for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    SplitLoader<AK, TM, Threads, Step, Offset> la;
    SplitLoader<BK, TN, Threads, Step, Offset> lb;
    la.init(p.lda, p.m - m0);
    lb.init(p.ldb, p.n - n0);

    // Row sums of op(A) over this split's K (the bias gradient of a weight-gradient product), by the workgroups
    // of the first N tile, from the staged fp32 values.  Compensated (Kahan) sums per group of 8 K: bias
    // gradients add thousands of values that largely cancel, where plain fp32 sums lose digits.
    const bool row_sums = !AK && p.a_sums != nullptr && bx == 0;
    constexpr int SumGroups = AK ? 1 : decltype(la)::Count / 8;
    float a_sum[SumGroups] = {}, a_comp[SumGroups] = {};
    const auto add_sums = [&]() {
        if constexpr (!AK) {
            if (row_sums) {
#pragma unroll
                for (int g = 0; g < SumGroups; ++g) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float y = la.regs[g * 8 + e] - a_comp[g];
                        const float s = a_sum[g] + y;
                        a_comp[g] = (s - a_sum[g]) - y;
                        a_sum[g] = s;
                    }
                }
            }
        }
    };

    // a 32x32 accumulator holds, in lane l, column l % 32 of rows 8 (v / 4) + 4 (l / 32) + v % 4, v = 0 .. 15
    const int wave_row = wm * WTM + 4 * (lane / 32);

    const auto multiply = [&]() {
#pragma unroll
        for (int sub = 0; sub < Step / 16; ++sub) {
            bf16x8_t af[WBM][3], bf[WBN][3];
            const int c = 2 * sub + lane / 32;
#pragma unroll
            for (int i = 0; i < WBM; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    af[i][q] = *reinterpret_cast<const bf16x8_t*>(sa + q * PlaneA + slot<Step>(wm * WTM + i * 32 + lane % 32, c));
#pragma unroll
            for (int j = 0; j < WBN; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    bf[j][q] = *reinterpret_cast<const bf16x8_t*>(sb + q * PlaneB + slot<Step>(wn * WTN + j * 32 + lane % 32, c));
            // the six products of one accumulator are spread over the blocks, so no MFMA waits for the one before it
            constexpr int ia[6] = {0, 0, 1, 0, 1, 2}, ib[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int i = 0; i < WBM; ++i)
#pragma unroll
                    for (int j = 0; j < WBN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][ia[s]], bf[j][ib[s]], acc[i][j], 0, 0, 0);
        }
    };
    const auto stage = [&]() {
        la.store(sa);
        lb.store(sb);
        add_sums();
        A += step_a;
        B += step_b;
    };

    const int full = k_count / Step, tail = k_count % Step;
    if (full > 0) {
        la.load(A, p.lda);
        lb.load(B, p.ldb);
    } else {
        la.load_tail(A, p.lda, tail);
        lb.load_tail(B, p.ldb, tail);
    }
    stage();
    // one step in LDS, the next on its way to registers; only the last load can be short
    for (int s = 1; s < full; ++s) {
        la.load(A, p.lda);
        lb.load(B, p.ldb);
        __syncthreads();
        multiply();
        __syncthreads();
        stage();
    }
    if (full > 0 && tail > 0) {
        la.load_tail(A, p.lda, tail);
        lb.load_tail(B, p.ldb, tail);
        __syncthreads();
        multiply();
        __syncthreads();
        stage();
    }
    __syncthreads();
    multiply();

    if (row_sums) {
        // thread t holds the partial sums of row t % TM over its groups: add the groups in K order
        __syncthreads();
        float* part = reinterpret_cast<float*>(sa);
        constexpr int Groups = Step / 8;
        static_assert(Groups * TM * 4 <= 3 * PlaneA * 2, "the partial sums fit the staging area");
#pragma unroll
        for (int g = 0; g < SumGroups; ++g) part[(t / TM * SumGroups + g) * TM + t % TM] = a_sum[g];
        __syncthreads();
        if (t < TM) {
            float total = part[t];
#pragma unroll
            for (int g = 1; g < Groups; ++g) total += part[g * TM + t];
            const int r = m0 + t;
            if (r < p.m)
                p.a_sums[(p.splits == 1 ? batch * p.sums_stride
                                         : (static_cast<long long>(split) * p.batch + batch) * p.m) + r] = total;
        }
    }

    // Epilogue.  Addresses are a uniform tile base plus a 32-bit lane offset, so a store costs no vector address
    // arithmetic; whole tiles (uniform) take the stores without bounds checks.
    const bool direct = p.splits == 1;
    const long long ldd = direct ? p.ldd : p.n;
    const long long tile = (direct ? batch * p.stride_d
                                   : (static_cast<long long>(split) * p.batch + batch) * static_cast<long long>(p.m) * p.n) +
                           m0 * ldd + n0;
    float* D = p.d + tile;
    const float* C = direct && p.c && (p.epilogue == kEluGrad || p.beta != 0.0f) ? p.c + tile : nullptr;
    unsigned short* H = direct && p.d_bf16 ? p.d_bf16 + tile : nullptr;
    const float* bias = direct && p.bias ? p.bias + batch * p.stride_bias + n0 : nullptr;
    const bool whole = m0 + TM <= p.m && n0 + TN <= p.n;
#pragma unroll
    for (int i = 0; i < WBM; ++i) {
#pragma unroll
        for (int j = 0; j < WBN; ++j) {
            const int col = wn * WTN + j * 32 + lane % 32;
            const Offset offset = static_cast<Offset>(wave_row) * static_cast<Offset>(ldd) + col;
            const bool in_n = whole || n0 + col < p.n;
            const auto in = [&](int v) { return whole || (in_n && m0 + wave_row + i * 32 + 8 * (v / 4) + v % 4 < p.m); };
            // all C values are loaded before the first store: the compiler cannot tell C from D apart, and a
            // load behind a store would expose one memory round trip per element
            float cv[16];
            if (C) {
#pragma unroll
                for (int v = 0; v < 16; ++v) cv[v] = in(v) ? (C + (i * 32 + 8 * (v / 4) + v % 4) * ldd)[offset] : 0.0f;
            }
            const float bcol = bias && in_n ? bias[col] : 0.0f;
            if (direct && p.epilogue == kEluGrad) {
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] *= elu_grad_from_output(cv[v]);
            } else if (direct) {
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] += bcol;
                if (p.epilogue != kNone) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] = apply_epilogue(acc[i][j][v], p.epilogue);
                }
                if (p.beta != 0.0f) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] += p.beta * cv[v];
                }
            }
            if (H) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (in(v)) (H + (i * 32 + 8 * (v / 4) + v % 4) * ldd)[offset] = f32_to_bf16_bits(acc[i][j][v]);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (in(v)) (D + (i * 32 + 8 * (v / 4) + v % 4) * ldd)[offset] = acc[i][j][v];
        }
    }
}

// Workgroups of 128 x 128 tiles (all splits) from which a product runs them on eight waves of 64 x 32: each
// staged value then feeds twice the MFMAs of a 64 x 64 tile, and the operand reads per product halve (24576 x
// 256 x 512, batch 2: 74.6 us against 88.8 us; with 128 tiles the smaller ones reach more CUs: 1024 x 1024 x 256,
// batch 2: 15.3 us against 11.0 us).  Outputs of at most 64 rows or columns (heads) keep the 64 x 64 tiles,
// which waste less of a tile (24576 x 37 x 128, batch 2: 15.1 us against 10.1 us).
constexpr long long kWideTiles = 256;

// Row sums are those of an M-contiguous A only.
bool split_eligible(const Params& p, bool ak) { return !(p.a_sums && ak); }

template <int T, int WGM, int WGN, int MinWaves, class Offset, bool AK, bool BK>
void launch_split_tiled(const Params& p, hipStream_t stream) {
    const dim3 grid(ceil_div(p.n, T), ceil_div(p.m, T), static_cast<unsigned>(p.batch * p.splits));
    hipLaunchKernelGGL((split_kernel<T, T, WGM, WGN, 32, MinWaves, Offset, AK, BK>), grid, dim3(WGM * WGN * kWave), 0,
                       stream, p);
}

template <class Offset, bool AK, bool BK>
void launch_split_offset(const Params& p, hipStream_t stream) {
    const long long wide = static_cast<long long>(ceil_div(p.m, 128)) * ceil_div(p.n, 128) * p.batch * p.splits;
    if (p.m > 64 && p.n > 64 && wide >= kWideTiles) launch_split_tiled<128, 2, 4, 2, Offset, AK, BK>(p, stream);
    else launch_split_tiled<64, 2, 2, 4, Offset, AK, BK>(p, stream);
}

// 32-bit offsets hold 128 rows of fewer than 2^22 values in bytes (an M/N-contiguous operand's rows are adjacent
// whatever its pitch) and 128 output rows of fewer than 2^24 in values; partial sums are p.n apart.
template <bool AK, bool BK>
void launch_split_layout(const Params& p, hipStream_t stream) {
    const bool near = (!AK || p.lda < (1 << 22)) && (!BK || p.ldb < (1 << 22)) && (p.splits > 1 || p.ldd < (1 << 24));
    if (near) launch_split_offset<unsigned, AK, BK>(p, stream);
    else launch_split_offset<unsigned long long, AK, BK>(p, stream);
}

void launch_split(const Params& p, bool ak, bool bk, hipStream_t stream) {
    if (ak && bk) launch_split_layout<true, true>(p, stream);
    else if (ak) launch_split_layout<true, false>(p, stream);
    else if (bk) launch_split_layout<false, true>(p, stream);
    else launch_split_layout<false, false>(p, stream);
}

}  // namespace gemm
}  // namespace rl
