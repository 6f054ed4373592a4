// k_gemm16.hip -- host dispatch of the 16-bit (bf16 / fp16) MFMA GEMM:
// argument checks, alignment decisions and the tile-configuration choice.
// The kernel is in fg_gemm16_kernel.h, instantiated in k_gemm16_{bf16,f16}.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <iterator>

#include "fg_gemm16_kernel.h"
#include "fg_gemm_rows.h"
#include "fg_internal.h"

namespace {

using fg::gemm16::Args;

int tiles(int M, int N, int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); }

// How a call's rows lie: whole 16-byte chunks on 16-byte boundaries, on
// 4-byte ones, or on odd elements.
enum Rows { kRowsWhole = 0, kRowsEven = 1, kRowsOdd = 2 };
// Of operands given by address and leading dimension (multiples of 8 with
// aligned bases, and row-contiguous operands' row lengths too, are whole).
Rows rows_of(int layout, int M, int N, const void *A, int lda, const void *B, int ldb) {
    const uintptr_t ab = (uintptr_t)A | (uintptr_t)B;
    const int ld = lda | ldb;
    if ((ab & 3u) || (ld & 1)) return kRowsOdd;
    const bool rc = (layout == FG_NT || N % 8 == 0) && (layout != FG_TN || M % 8 == 0);
    return (ab & 15u) == 0 && ld % 8 == 0 && rc ? kRowsWhole : kRowsEven;
}

// Tile configuration and K slices of a call (M, N >= 8) by a model of its time,
// measured on MI355X (256 CUs, bf16, N(0,1) operands, HIP events, K from 1 to
// 4096).  Pipelined tiles: a CU with n workgroups takes n tiles' time, a tile its
// k times kRate (us per k per 64x64 of output), a fixed part that grows with it
// (pipeline fill, output), its K tail, and more where its output has edges; slices
// cut the depth for a summing launch and the slots' traffic.  That a CU's
// workgroups take their tiles one after the other is how the matrix units' time
// adds up; tiles of unaligned rows, which wait for loads, overlap more than that,
// so their kRate is a mean over the sizes.  With the fused column sums each slice
// also leaves N fp32 sums, after the output slots.  Modelled against measured (us,
// NN): 2048 x 1000 x 4096 on 128x128 tiles in two slices 33 / 33, on 256x128 in
// four 36 / 37; 2046 x 4094 x 4094 on 256x256 in two 100 / 100, unsplit 131 / 127.
// The candidates' order settles ties: the larger tiles first.
//
// Rows that are not whole chunks took one element a lane before (us): 2047 x
// 4095 x 4093 NN 975 -> 116, NT 1363 -> 121, 777 x 1333 x 2049 120 -> 27, 300^3
// 16.1 -> 10.8; 1000^3 (K not whole tiles) NN / NT / TN 58 / 35 / 102 -> 17 / 15 / 18.
// Of the whole-row calls, those with under a 256x128 tile per CU changed tiles:
// 1024^3 20.5 / 19.8 / 21.1 -> 15.4 / 13.2 / 17.2, 128 x 4096 x 4096 NN 87 -> 19.
struct Rate16 {
    int cfg;
    float nn, nt, tn;
};
constexpr Rate16 kWhole[] = {{fg::gemm16::kCfgBig, 0.0017f, 0.0017f, 0.0017f},
                             {fg::gemm16::kCfgMid, 0.0021f, 0.0021f, 0.0021f},
                             {fg::gemm16::kCfgMidTail, 0.0022f, 0.0022f, 0.0022f},
                             {fg::gemm16::kCfg256, 0.0018f, 0.0019f, 0.0024f},
                             {fg::gemm16::kCfg128, 0.0026f, 0.0023f, 0.0032f},
                             {fg::gemm16::kCfgAny256, 0.0018f, 0.0019f, 0.0024f},
                             {fg::gemm16::kCfgAny128, 0.0026f, 0.0023f, 0.0032f}};
constexpr Rate16 kEven[] = {{fg::gemm16::kCfgAny256, 0.0018f, 0.0020f, 0.0025f},
                            {fg::gemm16::kCfgAny128, 0.0033f, 0.0036f, 0.0030f}};
constexpr Rate16 kOdd[] = {{fg::gemm16::kCfgOdd256, 0.0024f, 0.0026f, 0.0030f},
                           {fg::gemm16::kCfgOdd128, 0.0041f, 0.0047f, 0.0037f}};
constexpr float kTileUs = 1.5f, kTileUnitUs = 0.4f;  // fixed, and per 64x64
constexpr float kSumUs16 = 2.0f, kSumBytesPerUs16 = 6.0e6f;

// A pipelined tile's K tail of r elements, which is loaded one element at a time:
// where rows are odd and k-contiguous it shows (1023 x 1021 NN, 128x128 tiles:
// 12.2 us for K = 2, 15.8 for 32, 14.4 for 33).
float tail_us(int layout, Rows rows, int units, int r) {
    const float per_k = rows != kRowsOdd || layout == FG_TN ? 0.006f : 0.03f;
    return r > 0 ? 0.5f + per_k * units * r : 0.0f;
}
// What the last of a launch's tiles take longer where the row length is not whole
// groups of four (written one element at a time, by rows: 1024 x 1024 x 64 NN 7.2
// us, 1023 x 1021 x 65 14.9) or a tile reaches past the output.  A slice's fp32
// sums have no such edges, the summing launch's are spread over all CUs.
float edge_us(int M, int N, int bm, int bn, int units) {
    if (N % 4 != 0)
        return (units == 4 ? 7.5f : units == 16 ? 16.0f : 8.0f) * std::min(M, bm) / bm;
    return M % bm != 0 || N % bn != 0 ? 0.3f * units : 0.0f;
}
// The 64x64 tiles that are not pipelined (kCfgSmall; n a CU, several of them at
// once), without slices; K up to 512, from where the others were faster.  The column
// sums are a reduction of their own then.  They win where K is too short for a
// pipeline to pay (us, against 128x128 tiles): TN 297 x 407 x 32 10 / 26, 512 x
// 57 x 11 9.4 / 16.9, NN 1146 x 137 x 128 13.8 / 24.7, 1024 x 1024 x 64 5.3 /
// 7.2; at K = 256 NN / TN 1024^2 8.3 / 8.8, 10.7 / 8.8.
float small_us(int layout, int M, int N, int K, Rows rows, int64_t n, bool colsum) {
    const bool vec = rows == kRowsWhole;
    const bool whole = vec && M % 64 == 0 && N % 64 == 0;
    float one, many;  // us per k: a CU's only tile, and each of several
    if (layout == FG_NT) {
        one = vec ? 0.008f : 0.034f;
        many = vec ? 0.006f : 0.034f;
    } else if (layout == FG_NN) {
        one = vec && N % 64 == 0 ? 0.012f : 0.036f;
        many = vec && N % 64 == 0 ? 0.010f : 0.034f;
    } else {
        one = whole ? 0.030f : 0.042f;
        many = whole ? 0.012f : 0.032f;
    }
    // (TN's operands are both transposed; partial tiles show from a third K tile on.)
    const float tn = whole || (vec && K <= 64) ? 1.0f : vec ? 3.0f : 2.0f;
    return std::max(0, K - 32) * std::max(one, n * many) + 0.2f + 1.2f * n +
           (layout == FG_TN ? tn : 0.0f) + (colsum ? 5.0f : 0.0f);
}

struct Choice16 {
    int cfg = fg::gemm16::kCfgSmall, splits = 1, ks = 0;
    float us = 1e30f;
};
Choice16 choose16(int layout, int M, int N, int K, int cus, Rows rows, bool colsum,
                  uint64_t ws_bytes) {
    using namespace fg::gemm16;
    Choice16 best;
    const Rate16 *r = rows == kRowsWhole ? kWhole : rows == kRowsEven ? kEven : kOdd;
    const Rate16 *end = rows == kRowsWhole  ? std::end(kWhole)
                        : rows == kRowsEven ? std::end(kEven)
                                            : std::end(kOdd);
    // A row-contiguous operand of ragged rows leaves its last row to the tail.
    const bool ragged = rows != kRowsWhole &&
                        ((layout == FG_TN && M % 8 != 0) || (layout != FG_NT && N % 8 != 0));
    for (; r != end; ++r) {
        // Whole K tiles, but for the tails': that of 256x128 takes k-contiguous
        // rows eight at a time.
        const int bk = cfg_bk16(r->cfg);
        if (r->cfg == kCfgMidTail) {
            if (K % bk == 0 || (layout != FG_TN && K % 8 != 0)) continue;
        } else if (r->cfg < kCfgMidTail) {
            if (K % bk != 0) continue;
        }
        int bm, bn;
        cfg_tile16(r->cfg, bm, bn);
        const int64_t t = tiles(M, N, bm, bn);
        const int units = (bm / 64) * (bn / 64);
        const float rate = (layout == FG_NN ? r->nn : layout == FG_NT ? r->nt : r->tn) * units;
        const int tail = K - (K - (ragged ? 1 : 0)) / bk * bk;
        const float fixed = kTileUs + kTileUnitUs * units + tail_us(layout, rows, units, tail);
        for (int s = 1; s <= 16; ++s) {
            int ks = K;
            if (s > 1) {
                // At least eight K tiles in all and four a slice, whole ones;
                // slices only while the CUs have under two tiles each.
                if (K < 8 * bk || s > K / (4 * bk) || t * s > 2 * (int64_t)cus) break;
                ks = ((K + s - 1) / s + bk - 1) / bk * bk;
                if ((K + ks - 1) / ks != s) continue;
                if ((uint64_t)s * ((uint64_t)M * N + (colsum ? N : 0)) * sizeof(float) > ws_bytes)
                    break;
            }
            const int k = s > 1 ? ks : K - tail;  // (a slice has a tail only if it is the last)
            float us = (float)((t * s + cus - 1) / cus) * (k * rate + fixed);
            us += s > 1 ? kSumUs16 + (2 * s + 1) * (float)M * N * 4.0f / kSumBytesPerUs16
                        : edge_us(M, N, bm, bn, units);
            if (us < 0.99f * best.us) best = Choice16{r->cfg, s, s > 1 ? ks : 0, us};
        }
    }
    // Its column sums only where the workspace holds their partial sums already:
    // a call never grows it for a choice that it need not make.
    if (K <= 512 && (!colsum || fg::bias_grad_ws_bytes(cus, K, N) <= ws_bytes)) {
        const float us = small_us(layout, M, N, K, rows, (tiles(M, N, 64, 64) + cus - 1) / cus,
                                  colsum);
        if (us < 0.99f * best.us) best = Choice16{kCfgSmall, 1, 0, us};
    }
    return best;
}

// The kernel choices of one call (operands as passed, colsum included).
struct Plan16 {
    bool rows = false;  // the few-row kernel (fg_gemm_rows.h); then only splits and ks apply
    bool pipe = false;  // else gemm16_mfma, with 16-byte operand loads (vec) or not
    bool vec = false;
    int cfg = fg::gemm16::kCfgSmall, splits = 1, ks = 0;
};
Plan16 plan16(const fg_ctx *ctx, int layout, const Args &a) {
    Plan16 q;
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    // K slices go into the context's workspace when what is reserved holds
    // them (it is never grown for this), summed by a second kernel in slot
    // order -- deterministic, within the GEMM tolerance of the unsplit sum.
    const uint64_t ws = ctx->ws ? ctx->ws_bytes : 0;
    // Few rows (up to 64), any alignment: bf16 16 x 4096 x 4096 97.5 -> 11.8 us,
    // 64 x 4096 x 4096 98.7 -> 17.0, 64 x 1000 x 2048 94.3 -> 12.2, 64 x 1001 x
    // 2049 99.8 -> 13.8, 40 x 300 x 333 19 -> 5.8 against the tiles below.
    if (!a.colsum && fg::rows::applies(layout, a.M, a.N, a.K)) {
        q.rows = true;
        q.splits = fg::rows::split_of(cus, 2, a.M, a.N, a.K, ws, q.ks);
        return q;
    }
    const Rows rows = rows_of(layout, a.M, a.N, a.A, a.lda, a.B, a.ldb);
    q.vec = rows == kRowsWhole;
    if (a.K <= 0 || a.M < 8 || a.N < 8) return q;
    const Choice16 ch = choose16(layout, a.M, a.N, a.K, cus, rows, a.colsum != nullptr, ws);
    q.pipe = ch.cfg != fg::gemm16::kCfgSmall;
    q.cfg = ch.cfg;
    q.splits = ch.splits;
    q.ks = ch.ks;
    return q;
}

// Argument checks of one call with M, N > 0 (nothing launched).
int gemm16_check(fg_ctx *ctx, int dtype, int layout, const Args &a, const char *who) {
    FG_REQUIRE(ctx, FG_ERR_INVALID_ARGUMENT, "%s: ctx is NULL", who);
    FG_REQUIRE(dtype == FG_DTYPE_F16 || dtype == FG_DTYPE_BF16, FG_ERR_UNSUPPORTED,
               "%s: dtype %d is not a 16-bit type (use fg_gemm_f32 for fp32)", who, dtype);
    FG_REQUIRE(a.M > 0 && a.N > 0 && a.K >= 0, FG_ERR_SHAPE, "%s: empty or negative shape", who);
    FG_REQUIRE(a.act >= 0 && a.act <= 2, FG_ERR_INVALID_ARGUMENT, "%s: bad act %d", who, a.act);
    FG_REQUIRE(a.A && a.B && a.C, FG_ERR_INVALID_ARGUMENT, "%s: NULL operand", who);
    const int a_cols = layout == FG_TN ? a.M : a.K;
    const int b_cols = layout == FG_NT ? a.K : a.N;
    FG_REQUIRE(a.lda >= std::max(a_cols, 1) && a.ldb >= std::max(b_cols, 1) && a.ldc >= a.N,
               FG_ERR_SHAPE, "%s: leading dimension too small", who);
    return FG_OK;
}

int gemm16_common(fg_ctx *ctx, int dtype, int layout, Args &a, const char *who) {
    FG_REQUIRE(ctx, FG_ERR_INVALID_ARGUMENT, "%s: ctx is NULL", who);
    FG_REQUIRE(dtype == FG_DTYPE_F16 || dtype == FG_DTYPE_BF16, FG_ERR_UNSUPPORTED,
               "%s: dtype %d is not a 16-bit type (use fg_gemm_f32 for fp32)", who, dtype);
    FG_REQUIRE(layout >= FG_NN && layout <= FG_TN, FG_ERR_INVALID_ARGUMENT, "%s: bad layout %d",
               who, layout);
    FG_REQUIRE(a.M >= 0 && a.N >= 0 && a.K >= 0, FG_ERR_SHAPE, "%s: negative dimension", who);
    FG_REQUIRE(a.act >= 0 && a.act <= 2, FG_ERR_INVALID_ARGUMENT, "%s: bad act %d", who, a.act);
    FG_REQUIRE(!a.colsum || layout == FG_TN, FG_ERR_INVALID_ARGUMENT,
               "%s: column sums need the TN layout", who);
    if (a.N == 0) return FG_OK;
    if (a.M == 0) {  // no output rows, but the column sums of B still run
        if (!a.colsum) return FG_OK;
        FG_REQUIRE(a.B && a.ldb >= a.N, FG_ERR_INVALID_ARGUMENT, "%s: bad B", who);
        return fg_bias_grad(ctx, dtype, a.K, a.N, a.B, a.ldb, a.colsum, a.colsum_accumulate);
    }
    FG_REQUIRE(a.A && a.B && a.C, FG_ERR_INVALID_ARGUMENT, "%s: NULL operand", who);
    const int a_cols = layout == FG_TN ? a.M : a.K;
    const int b_cols = layout == FG_NT ? a.K : a.N;
    FG_REQUIRE(a.lda >= std::max(a_cols, 1) && a.ldb >= std::max(b_cols, 1) && a.ldc >= a.N,
               FG_ERR_SHAPE, "%s: leading dimension too small (lda=%d ldb=%d ldc=%d)", who, a.lda,
               a.ldb, a.ldc);
    FG_HIP(hipSetDevice(ctx->device));
    uint16_t *colsum = a.colsum;  // the bias gradient of fg_gemm_dw_x16, if any
    if (a.K == 0) a.A = a.B;  // loads are all masked; K=0 yields the epilogue of zero
    const Plan16 q = plan16(ctx, layout, a);
    // Only the pipelined kernel sums B's columns; elsewhere the separate
    // reduction runs after the GEMM (same result up to the order of the
    // fp32 sums).
    if (colsum && !q.pipe) a.colsum = nullptr;
    a.partial = q.splits > 1 ? static_cast<float *>(ctx->ws) : nullptr;
    a.ksplit = q.splits > 1 ? q.ks : 0;
    a.colsum_partial =
        q.splits > 1 && a.colsum ? a.partial + (size_t)q.splits * a.M * a.N : nullptr;
    if (q.rows) {
        fg::rows::launch_16(dtype == FG_DTYPE_BF16, layout, a, ctx->stream);
        if (q.splits > 1) {
            if (dtype == FG_DTYPE_BF16)
                fg::gemm16::launch_sum_bf16(a, q.splits, ctx->stream);
            else
                fg::gemm16::launch_sum_f16(a, q.splits, ctx->stream);
        }
    } else if (dtype == FG_DTYPE_BF16)
        fg::gemm16::launch_bf16(layout, a, q.vec, q.cfg, ctx->stream);
    else
        fg::gemm16::launch_f16(layout, a, q.vec, q.cfg, ctx->stream);
    FG_LAUNCH_CHECK(who);
    if (colsum && !q.pipe)
        return fg_bias_grad(ctx, dtype, a.K, a.N, a.B, a.ldb, colsum, a.colsum_accumulate);
    return FG_OK;
}

// A layer's dW (TN, with the fused column sums) and dX (NT, act' of Zs)
// arguments, as fg_gemm_dw_x16 and fg_gemm_bwd_x16 take them.
Args dw_args16(int M, int N, int K, const void *A, int lda, const void *B, int ldb, void *C,
               int ldc, int acc, void *colsum, int colsum_acc) {
    Args a{};
    a.A = static_cast<const uint16_t *>(A);
    a.B = static_cast<const uint16_t *>(B);
    a.C = static_cast<uint16_t *>(C);
    a.M = M;
    a.N = N;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.act = FG_ACT_NONE;
    a.mode = 0;
    a.accumulate = acc ? 1 : 0;
    a.colsum = static_cast<uint16_t *>(colsum);
    a.colsum_accumulate = colsum_acc ? 1 : 0;
    return a;
}
Args dx_args16(int M, int N, int K, const void *A, int lda, const void *B, int ldb, int act,
               const void *Zs, int ldzs, void *C, int ldc, int acc) {
    Args a{};
    a.A = static_cast<const uint16_t *>(A);
    a.B = static_cast<const uint16_t *>(B);
    a.C = static_cast<uint16_t *>(C);
    a.Zs = static_cast<const uint16_t *>(Zs);
    a.M = M;
    a.N = N;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.ldzs = ldzs;
    a.act = act;
    a.mode = 1;
    a.accumulate = acc ? 1 : 0;
    return a;
}
// Both pipelined on the pair's configurations, neither split.
bool pairable16(fg_ctx *ctx, Args &w, Args &x) {
    if (w.M <= 0 || w.N <= 0 || w.K <= 0 || x.M <= 0 || x.N <= 0 || x.K <= 0) return false;
    const Plan16 qw = plan16(ctx, FG_TN, w), qx = plan16(ctx, FG_NT, x);
    return qw.pipe && qx.pipe && qw.splits == 1 && qx.splits == 1 &&
           qw.cfg == fg::gemm16::kCfgBig && qx.cfg == fg::gemm16::kCfgMid;
}

}  // namespace

namespace fg {
// A layer's two gradient GEMMs with 16-bit tensors: one launch
// (gemm16_pair_big) when both take the large tiles' pipelined kernels
// unsplit, else fg_gemm_dw_x16 then fg_gemm_bwd_x16.  Each part runs
// exactly as its own call.
int gemm16_dw_dx(fg_ctx *ctx, int dtype, int M1, int N1, int K1, const void *A1, int lda1,
                 const void *B1, int ldb1, void *C1, int ldc1, int acc1, void *colsum,
                 int colsum_acc, int M2, int N2, int K2, const void *A2, int lda2,
                 const void *B2, int ldb2, int act, const void *Zs, int ldzs, void *C2, int ldc2,
                 int acc2) {
    Args w = dw_args16(M1, N1, K1, A1, lda1, B1, ldb1, C1, ldc1, acc1, colsum, colsum_acc);
    Args x = dx_args16(M2, N2, K2, A2, lda2, B2, ldb2, act, Zs, ldzs, C2, ldc2, acc2);
    const bool checked = M1 > 0 && N1 > 0 && M2 > 0 && N2 > 0 &&
                         gemm16_check(ctx, dtype, FG_TN, w, "fg_gemm_dw_x16") == FG_OK &&
                         gemm16_check(ctx, dtype, FG_NT, x, "fg_gemm_bwd_x16") == FG_OK &&
                         (act == FG_ACT_NONE || (Zs && ldzs >= N2));
    if (!checked || !pairable16(ctx, w, x)) {
        fg::clear_error();  // the calls below report any error themselves
        const int rc = fg_gemm_dw_x16(ctx, dtype, M1, N1, K1, A1, lda1, B1, ldb1, C1, ldc1, acc1,
                                      colsum, colsum_acc);
        if (rc) return rc;
        return fg_gemm_bwd_x16(ctx, dtype, FG_NT, M2, N2, K2, A2, lda2, B2, ldb2, act, Zs, ldzs,
                               C2, ldc2, acc2);
    }
    FG_HIP(hipSetDevice(ctx->device));
    if (dtype == FG_DTYPE_BF16)
        fg::gemm16::launch_pair_bf16(w, x, ctx->stream);
    else
        fg::gemm16::launch_pair_f16(w, x, ctx->stream);
    FG_LAUNCH_CHECK("gemm16_dw_dx");
    return FG_OK;
}

// Dispatches of gemm16_dw_dx for these operands (no launch).
int gemm16_dw_dx_dispatches(fg_ctx *ctx, int M1, int N1, int K1, const void *A1, int lda1,
                            const void *B1, int ldb1, int M2, int N2, int K2, const void *A2,
                            int lda2, const void *B2, int ldb2) {
    const int sep = gemm16_dispatches(ctx, FG_TN, M1, N1, K1, A1, lda1, B1, ldb1, true) +
                    gemm16_dispatches(ctx, FG_NT, M2, N2, K2, A2, lda2, B2, ldb2, false);
    if (!ctx) return sep;
    void *c = reinterpret_cast<void *>(256);  // only the operands' alignment enters the choice
    Args w = dw_args16(M1, N1, K1, A1, lda1, B1, ldb1, c, N1, 0, c, 0);
    Args x = dx_args16(M2, N2, K2, A2, lda2, B2, ldb2, FG_ACT_NONE, nullptr, 0, c, N2, 0);
    return pairable16(ctx, w, x) ? 1 : sep;
}

// Dispatches of one 16-bit GEMM call with these operands (no launch): the
// GEMM, its summing kernel when it splits K, the column-sum reduction's two
// when colsum is asked off the pipelined kernel.
int gemm16_dispatches(fg_ctx *ctx, int layout, int M, int N, int K, const void *A, int lda,
                      const void *B, int ldb, bool colsum) {
    if (!ctx || M <= 0 || N <= 0 || K <= 0) return 1;
    Args a{};
    a.A = static_cast<const uint16_t *>(A);
    a.B = static_cast<const uint16_t *>(B);
    a.M = M;
    a.N = N;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.colsum = colsum ? reinterpret_cast<uint16_t *>(256) : nullptr;
    const Plan16 q = plan16(ctx, layout, a);
    if (colsum && !q.pipe) return 3;
    return q.splits > 1 ? 2 : 1;
}

// Workspace bytes a 16-bit GEMM of this shape uses when the workspace holds
// them (its K slices, or the column sums' partial sums off the pipelined kernel;
// 0: none), for planners that size a workspace ahead.
uint64_t gemm16_split_ws_bytes(int cus, int layout, int M, int N, int K, bool colsum) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    cus = cus > 0 ? cus : 256;
    if (!colsum && fg::rows::applies(layout, M, N, K)) {
        int ks;
        const int sl = fg::rows::split_of(cus, 2, M, N, K, ~0ull, ks);
        return sl > 1 ? (uint64_t)sl * M * N * sizeof(float) : 0;
    }
    // Off the pipelined kernel the column sums are a reduction of their own.
    const uint64_t reduce = colsum ? bias_grad_ws_bytes(cus, K, N) : 0;
    if (M < 8 || N < 8) return reduce;
    // Dense rows from aligned bases.
    const int lda = layout == FG_TN ? M : K, ldb = layout == FG_NT ? K : N;
    const Choice16 ch = choose16(layout, M, N, K, cus, rows_of(layout, M, N, nullptr, lda, nullptr, ldb),
                                 colsum, ~0ull);
    if (ch.cfg == fg::gemm16::kCfgSmall) return reduce;
    return ch.splits > 1 ? (uint64_t)ch.splits * ((uint64_t)M * N + (colsum ? N : 0)) * sizeof(float)
                         : 0;
}
}  // namespace fg

FG_API int fg_gemm_x16(fg_ctx *ctx, int dtype, int layout, int M, int N, int K, const void *d_A,
                       int lda, const void *d_B, int ldb, const void *d_bias, int act, void *d_C,
                       int ldc, void *d_Z, int ldz, int accumulate) {
    Args a{};
    a.A = static_cast<const uint16_t *>(d_A);
    a.B = static_cast<const uint16_t *>(d_B);
    a.C = static_cast<uint16_t *>(d_C);
    a.Z = static_cast<uint16_t *>(d_Z);
    a.bias = static_cast<const uint16_t *>(d_bias);
    a.M = M;
    a.N = N;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.ldz = d_Z ? ldz : 0;
    a.act = act;
    a.mode = 0;
    a.accumulate = accumulate ? 1 : 0;
    FG_REQUIRE(!d_Z || ldz >= N, FG_ERR_SHAPE, "fg_gemm_x16: ldz=%d < N=%d", ldz, N);
    FG_REQUIRE(!(accumulate && act != FG_ACT_NONE), FG_ERR_INVALID_ARGUMENT,
               "fg_gemm_x16: accumulate requires act NONE");
    return gemm16_common(ctx, dtype, layout, a, "fg_gemm_x16");
}

FG_API int fg_gemm_dw_x16(fg_ctx *ctx, int dtype, int M, int N, int K, const void *d_A, int lda,
                          const void *d_B, int ldb, void *d_C, int ldc, int accumulate,
                          void *d_colsum, int colsum_accumulate) {
    Args a{};
    a.A = static_cast<const uint16_t *>(d_A);
    a.B = static_cast<const uint16_t *>(d_B);
    a.C = static_cast<uint16_t *>(d_C);
    a.M = M;
    a.N = N;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.act = FG_ACT_NONE;
    a.mode = 0;
    a.accumulate = accumulate ? 1 : 0;
    a.colsum = static_cast<uint16_t *>(d_colsum);
    a.colsum_accumulate = colsum_accumulate ? 1 : 0;
    return gemm16_common(ctx, dtype, FG_TN, a, "fg_gemm_dw_x16");
}

FG_API int fg_gemm_bwd_x16(fg_ctx *ctx, int dtype, int layout, int M, int N, int K,
                           const void *d_A, int lda, const void *d_B, int ldb, int act,
                           const void *d_Zs, int ldzs, void *d_C, int ldc, int accumulate) {
    Args a{};
    a.A = static_cast<const uint16_t *>(d_A);
    a.B = static_cast<const uint16_t *>(d_B);
    a.C = static_cast<uint16_t *>(d_C);
    a.Zs = static_cast<const uint16_t *>(d_Zs);
    a.M = M;
    a.N = N;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.ldzs = ldzs;
    a.act = act;
    a.mode = 1;
    a.accumulate = accumulate ? 1 : 0;
    FG_REQUIRE(act == FG_ACT_NONE || (d_Zs && ldzs >= N), FG_ERR_INVALID_ARGUMENT,
               "fg_gemm_bwd_x16: act %d needs Zs with ldzs >= N", act);
    return gemm16_common(ctx, dtype, layout, a, "fg_gemm_bwd_x16");
}

FG_API int fg_matmul_bwd_x16(fg_ctx *ctx, int dtype, int M, int N, int K, const void *d_X,
                             int ldx, const void *d_W, int ldw, const void *d_dZ, int lddz,
                             int act, const void *d_Zs, int ldzs, void *d_dX, int lddx,
                             void *d_dW, int lddw, void *d_dbias, int accumulate) {
    const char *who = "fg_matmul_bwd_x16";
    FG_REQUIRE(ctx, FG_ERR_INVALID_ARGUMENT, "%s: ctx is NULL", who);
    FG_REQUIRE(act >= FG_ACT_NONE && act <= FG_ACT_GELU, FG_ERR_INVALID_ARGUMENT,
               "%s: bad act %d", who, act);
    FG_REQUIRE(M >= 0 && N >= 0 && K >= 0, FG_ERR_SHAPE, "%s: negative dimension", who);
    FG_REQUIRE(d_X && d_W && d_dZ && d_dX && d_dW, FG_ERR_INVALID_ARGUMENT,
               "%s: NULL operand or output", who);
    FG_REQUIRE(ldx >= K && ldw >= N && lddz >= N && lddx >= K && lddw >= N,
               FG_ERR_INVALID_ARGUMENT, "%s: a leading dimension is below its row length", who);
    FG_REQUIRE(act == FG_ACT_NONE || (d_Zs && ldzs >= K), FG_ERR_INVALID_ARGUMENT,
               "%s: act %d needs Zs with ldzs >= K", who, act);
    // dW: TN K x N over M; dX: NT M x K over N.
    return fg::gemm16_dw_dx(ctx, dtype, K, N, M, d_X, ldx, d_dZ, lddz, d_dW, lddw, accumulate,
                            d_dbias, accumulate, M, K, N, d_dZ, lddz, d_W, ldw, act, d_Zs, ldzs,
                            d_dX, lddx, accumulate);
}
