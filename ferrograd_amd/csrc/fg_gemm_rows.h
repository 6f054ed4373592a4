// fg_gemm_rows.h -- GEMMs of few output rows (a forward or a data gradient at
// a small batch), for fp32, fp16 and bf16, NN and NT, any alignment.
//
// What bounds it: reading B (the weights) once from HBM; the products are a
// few per cent of the matrix units' time.  So the tiles are cut for the reads:
// a workgroup owns 32 columns of C and all of K, its NW waves take the K steps
// in turn, and every wave loads its operands straight into the MFMA registers,
// several steps ahead, with no LDS and no barrier on the way.  The waves'
// sums are added through LDS at the end, in wave order (deterministic), and
// finished by the GEMM's own epilogue, so there are no K slices in memory and
// there is no second launch.
//   * A lane of a 16x16 MFMA supplies E consecutive k (8 of 16 bits, 4 of fp32)
//     of one row of A and of one column of B.  A rows and NT's B rows hold them
//     as 16 bytes.  NN's B has them in E rows: a lane loads two adjacent
//     columns of each (64 or 128 bytes a row across the lanes), whose even and
//     odd columns make two MFMA operands.
//   * Rows of any length and alignment take these loads: 4-byte aligned ones
//     cost 16-byte loads nothing, and 16-bit rows that start on odd elements
//     (ODD) are read from the 4-byte boundary below and shifted into place (a
//     16-byte load off a 4-byte boundary took two to three times as long: 64 x
//     1000 x 2049 NT bf16 24.8 us, 10.9 for K = 2048).  The K step past the
//     last whole one is read one element at a time, from clamped addresses.
#pragma once

#include <hip/hip_runtime.h>

#include "fg_gemm16_kernel.h"
#include "fg_gemm_kernel.h"
#include "fg_half.h"

namespace fg {
namespace rows {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kCols = 32;   // columns of a workgroup
constexpr int kWaves = 8;   // 4 to 16 measured within 5 %
constexpr int kMaxRows = 64;

template <int DT>
struct Elem {  // 16-bit types
    using T = uint16_t;
    using Args = gemm16::Args;
    typedef u32x4 V __attribute__((aligned(2)));      // E elements
    typedef uint32_t Pair;                            // two adjacent columns
    typedef uint32_t PairU __attribute__((aligned(2)));
    static constexpr int E = 8;
    static __device__ __forceinline__ T zero() { return 0; }
};
template <>
struct Elem<kF32> {
    using T = float;
    using Args = gemm::GemmArgs;
    typedef u32x4 V __attribute__((aligned(4)));
    typedef u32x2 Pair;
    typedef u32x2 PairU __attribute__((aligned(4)));
    static constexpr int E = 4;
};

// E elements of a row from p on, in one 16-byte load.
template <int DT, bool ODD>
__device__ __forceinline__ u32x4 load_row(const typename Elem<DT>::T *p) {
    if constexpr (!ODD) {
        return static_cast<u32x4>(*reinterpret_cast<const typename Elem<DT>::V *>(p));
    } else {
        // The 4-byte words that hold the elements: four, and a fifth where the
        // first starts with the element before p.
        typedef u32x4 V4 __attribute__((aligned(4)));
        const uint32_t sh = ((uintptr_t)p & 2u) * 8u;
        const uint32_t *w = reinterpret_cast<const uint32_t *>(p - ((uintptr_t)p >> 1 & 1u));
        const u32x4 v = *reinterpret_cast<const V4 *>(w);
        const uint32_t v4 = w[sh ? 4 : 3];
        u32x4 r;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            r[q] = __builtin_amdgcn_alignbit(q < 3 ? v[q + 1] : v4, v[q], sh);
        return r;
    }
}

// One K step's operands of a wave: MB row blocks of A and 32 columns of B.
template <int DT, bool BNC, int MB, bool ODD>
struct Step {
    using El = Elem<DT>;
    using T = typename El::T;
    static constexpr int E = El::E, kStep = 4 * E;
    u32x4 a[MB];
    typename El::Pair bp[BNC ? E : 1];
    u32x4 bv[BNC ? 1 : 2];

    // EDGE: the step holds k past K (zeros), or B's last row where a pair of
    // columns there would end past N (elsewhere such a pair reads into the
    // next row, for an output that nothing stores).
    template <bool EDGE>
    __device__ __forceinline__ void load(const typename El::Args &p, int k0, int n0, int lane) {
        const int l16 = lane & 15, k = k0 + E * (lane >> 4);
        auto eight = [&](const T *row) {  // k .. k + E - 1 of a row
            if constexpr (!EDGE) {
                return load_row<DT, ODD>(row + k);
            } else {
                T e[E];
#pragma unroll
                for (int t = 0; t < E; ++t) {
                    e[t] = row[min(k + t, p.K - 1)];
                    if (k + t >= p.K) e[t] = 0;
                }
                u32x4 v;
                __builtin_memcpy(&v, e, 16);
                return v;
            }
        };
#pragma unroll
        for (int i = 0; i < MB; ++i)
            a[i] = eight(p.A + (size_t)min(16 * i + l16, p.M - 1) * p.lda);
        if constexpr (!BNC) {
#pragma unroll
            for (int f = 0; f < 2; ++f)
                bv[f] = eight(p.B + (size_t)min(n0 + 16 * f + l16, p.N - 1) * p.ldb);
        } else {
            const int n = n0 + 2 * l16;
#pragma unroll
            for (int t = 0; t < E; ++t) {
                if constexpr (!EDGE) {
                    bp[t] = *reinterpret_cast<const typename El::PairU *>(
                        p.B + (size_t)(k + t) * p.ldb + min(n, p.N - 1));
                } else {
                    const T *row = p.B + (size_t)min(k + t, p.K - 1) * p.ldb;
                    T e[2] = {row[min(n, p.N - 1)], row[min(n + 1, p.N - 1)]};
                    if (k + t >= p.K) e[0] = e[1] = 0;
                    __builtin_memcpy(&bp[t], e, sizeof e);
                }
            }
        }
    }

    // acc[i][f]: columns 2c + f (NN) or c + 16f (NT) of the lane's column c.
    __device__ __forceinline__ void multiply(f32x4 (&acc)[MB][2]) const {
        if constexpr (DT == kF32) {
#pragma unroll
            for (int t = 0; t < E; ++t)
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    const float b = __uint_as_float(BNC ? bp[t][f] : bv[f][t]);
#pragma unroll
                    for (int i = 0; i < MB; ++i)
                        acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i][t]),
                                                                        b, acc[i][f], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                u32x4 b;
                if constexpr (BNC) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        b[q] = __builtin_amdgcn_perm(bp[2 * q + 1], bp[2 * q],
                                                     f ? 0x07060302u : 0x05040100u);
                } else {
                    b = bv[f];
                }
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    if constexpr (DT == kBF16)
                        acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(gemm16::bf16x8, a[i]),
                            __builtin_bit_cast(gemm16::bf16x8, b), acc[i][f], 0, 0, 0);
                    else
                        acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(gemm16::f16x8, a[i]),
                            __builtin_bit_cast(gemm16::f16x8, b), acc[i][f], 0, 0, 0);
                }
            }
        }
    }
};

// U K steps of a wave, in pairs of adjacent steps (whole 128-byte lines of
// k-contiguous rows) NW pairs apart, from step s on: all loads, then the
// products.
template <int DT, bool BNC, int MB, bool ODD, int NW, int U, bool EDGE>
__device__ __forceinline__ void run_steps(const typename Elem<DT>::Args &p, int s, int n0, int lane,
                                          f32x4 (&acc)[MB][2]) {
    Step<DT, BNC, MB, ODD> st[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
        st[u].template load<EDGE>(p, (s + (u & 1) + (u >> 1) * 2 * NW) * Step<DT, BNC, MB, ODD>::kStep, n0,
                               lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) st[u].multiply(acc);
}

template <int DT, bool BNC, int MB, bool ODD>
__global__ __launch_bounds__(64 * kWaves) void gemm_rows(typename Elem<DT>::Args p) {
    constexpr int NW = kWaves;
    constexpr int kStep = Step<DT, BNC, MB, ODD>::kStep, kRows = 16 * MB, kLd = kCols + 1;
    // Steps in flight, by the registers that their operands take.
    constexpr int U = MB == 1 ? 4 : 2;
    __shared__ float red[NW * kRows * kLd];
    const int nt = gridDim.x;
    // Pairs of adjacent column blocks, which share 128-byte lines of B, on one
    // XCD (workgroup b runs on XCD b % 8); whole runs of blocks on one XCD
    // kept power-of-two row strides on few of its L2's channels.
    int bid = blockIdx.x;
    if ((nt & 15) == 0) bid = ((bid >> 4) * 8 + (bid & 7)) * 2 + ((bid >> 3) & 1);
    const int n0 = bid * kCols;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 acc[MB][2];
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    float *slot = nullptr;
    bool last = true;  // holds B's last row
    if (p.ksplit > 0) {  // K slice y, whole pairs of steps, its raw sums to slot y
        const int kb = blockIdx.y * p.ksplit;
        p.A += kb;
        p.B += BNC ? (size_t)kb * p.ldb : (size_t)kb;
        last = kb + p.ksplit >= p.K;
        p.K = min(p.ksplit, p.K - kb);
        slot = p.partial + (size_t)blockIdx.y * p.M * p.N;
    }
    const int whole = (p.K - (BNC && last && n0 + kCols > p.N ? 1 : 0)) / kStep;
    int s = 2 * wave;
    for (; s + (U - 2) * NW + 1 < whole; s += U * NW)
        run_steps<DT, BNC, MB, ODD, NW, U, false>(p, s, n0, lane, acc);
    for (; s + 1 < whole; s += 2 * NW) run_steps<DT, BNC, MB, ODD, NW, 2, false>(p, s, n0, lane, acc);
    if (s < whole) run_steps<DT, BNC, MB, ODD, NW, 1, false>(p, s++, n0, lane, acc);
    if (s == whole && s * kStep < p.K) run_steps<DT, BNC, MB, ODD, NW, 1, true>(p, s, n0, lane, acc);
    // Lane (c, g) holds rows 4g .. 4g+3 of its column of each block.
    const int c = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[(wave * kRows + 16 * i + 4 * g + r) * kLd + (BNC ? 2 * c + f : c + 16 * f)] =
                    acc[i][f][r];
    __syncthreads();
    for (int q = threadIdx.x; q < kRows * kCols; q += 64 * NW) {
        const int row = q / kCols, cc = q % kCols, col = n0 + cc;
        if (row >= p.M || col >= p.N) continue;
        float v = red[row * kLd + cc];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[(w * kRows + row) * kLd + cc];
        if (slot) {
            slot[(size_t)row * p.N + col] = v;
            continue;
        }
        const auto *bias = p.mode == 0 ? p.bias : nullptr;
        auto *dst = p.C + (size_t)row * p.ldc + col;
        if constexpr (DT == kF32) {
            float z;
            float o = gemm::epi_value(p, v, bias ? bias[col] : 0.0f, row, col, &z);
            if (p.mode == 0 && p.Z) p.Z[(size_t)row * p.ldz + col] = z;
            if (p.accumulate) o += *dst;
            *dst = o;
        } else {
            using X = gemm16::T16<DT == kBF16>;
            float z;
            float o = gemm16::epi16<DT == kBF16>(p, v, bias, row, col, &z);
            if (p.mode == 0 && p.Z) p.Z[(size_t)row * p.ldz + col] = X::from_f(z);
            if (p.accumulate) o += X::to_f(*dst);
            *dst = X::from_f(o);
        }
    }
}

// The call takes this kernel: few rows, K and N enough for its loads.
inline bool applies(int layout, int M, int N, int K) {
    return layout != 2 && M > 0 && M <= kMaxRows && N >= 2 && K > 0;
}
// K slices (1: none) for workgroups of `cus` CUs and a workspace of ws_bytes;
// their depth in ks.  esz: bytes of an element.
int split_of(int cus, int esz, int M, int N, int K, uint64_t ws_bytes, int &ks);
// layout: FG_NN or FG_NT; a.ksplit as split_of says (0: unsplit; the slices
// are left for the caller to sum).
void launch_f32(int layout, const gemm::GemmArgs &a, hipStream_t st);
void launch_16(bool bf16, int layout, const gemm16::Args &a, hipStream_t st);

}  // namespace rows
}  // namespace fg
