// k_gemm_rows.hip -- launches of the few-row GEMM kernel (fg_gemm_rows.h).
#include "fg_gemm_rows.h"

#include <algorithm>

namespace fg {
namespace rows {
namespace {

template <int DT, bool BNC, bool ODD>
void launch(const typename Elem<DT>::Args &a, hipStream_t st) {
    const dim3 grid((a.N + kCols - 1) / kCols, a.ksplit > 0 ? (a.K + a.ksplit - 1) / a.ksplit : 1);
    if (a.M <= 16)
        gemm_rows<DT, BNC, 1, ODD><<<grid, 64 * kWaves, 0, st>>>(a);
    else if (a.M <= 32)
        gemm_rows<DT, BNC, 2, ODD><<<grid, 64 * kWaves, 0, st>>>(a);
    else
        gemm_rows<DT, BNC, 4, ODD><<<grid, 64 * kWaves, 0, st>>>(a);
}

template <int DT>
void launch_type(int layout, const gemm16::Args &a, hipStream_t st) {
    // k-contiguous rows that start on odd elements (NN's B is read in pairs).
    auto odd = [](const void *q, int ld) { return ((uintptr_t)q & 3u) != 0 || (ld & 1) != 0; };
    const bool o = odd(a.A, a.lda) || (layout == 1 && odd(a.B, a.ldb));
    if (layout == 0)
        o ? launch<DT, true, true>(a, st) : launch<DT, true, false>(a, st);
    else
        o ? launch<DT, false, true>(a, st) : launch<DT, false, false>(a, st);
}

}  // namespace

int split_of(int cus, int esz, int M, int N, int K, uint64_t ws_bytes, int &ks) {
    ks = 0;
    // One workgroup per CU, of at least 2 KiB of each column: what a CU reads
    // bounds the kernel, and the summing launch costs about 2 us.  16 x 4096 x
    // 4096 bf16 13.5 us unsplit, 11.8 / 12.5 / 12.6 with 256 / 512 / 1024
    // workgroups; 16 x 1000 x 4096 13.3, 9.0 / 8.9 / 8.9; fp32 32 x 4096 x
    // 4096 37.5, 24.3 / 25.4 / 26.8.
    const int pair = 2 * 4 * (16 / esz);  // k of a pair of steps
    int s = std::min(cus / ((N + kCols - 1) / kCols), K / (2048 / esz));
    s = std::min(s, K / (pair * kWaves));
    if (s < 2) return 1;
    int d = (K + s - 1) / s;
    d = (d + pair - 1) / pair * pair;
    s = (K + d - 1) / d;
    if (s < 2 || (uint64_t)s * M * N * sizeof(float) > ws_bytes) return 1;
    ks = d;
    return s;
}

void launch_f32(int layout, const gemm::GemmArgs &a, hipStream_t st) {
    if (layout == 0)
        launch<kF32, true, false>(a, st);
    else
        launch<kF32, false, false>(a, st);
}

void launch_16(bool bf16, int layout, const gemm16::Args &a, hipStream_t st) {
    if (bf16)
        launch_type<kBF16>(layout, a, st);
    else
        launch_type<kF16>(layout, a, st);
}

}  // namespace rows
}  // namespace fg
