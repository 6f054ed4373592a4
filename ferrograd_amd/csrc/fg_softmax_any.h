// fg_softmax_any.h -- row softmax (+ cross-entropy) and its backward for rows
// of any element type, length and alignment, read and written 16 bytes a lane.
//
// A row of C elements that starts anywhere is split into a head (up to the
// first 16-byte boundary), whole 16-byte chunks and a tail; head and tail
// (fewer than a chunk each) are one element of their own per thread, in the
// row's first threads.  Every wide access is aligned, whatever the row's
// start.  The output rows must have the input rows' phase (address modulo
// 16), as rows of equal length and equally aligned tensors do.  Outputs may
// be the inputs themselves.
//
// What bounds it: HBM in fp32, the vector unit in 16 bits from where a row's
// exponentials are taken twice (NV > 4), by holding a row in registers so that it
// is read and written once.  Waves per row and chunks per thread (with_kind in
// k_softmax.hip, measured over 1, 2, 4, 8 and 16 chunks on 1, 4, 8 and 16 waves,
// HIP events): the fewest waves that hold the row in the registers that let two
// rows share a CU, one wave a row up to 256 chunks (no workgroup barrier; 16384 x
// 1000 fp32 24.2 us against 27.5 on four waves and 31.7 for the 256-thread kernel
// before).  8 chunks on 16 waves need 1 (fp32) and 3 (16 bits) registers more than
// that and spill them, which costs less than a row alone on its CU: 16 chunks on 16
// waves read and wrote at 3.1-4.4 TB/s against 4.3-4.5 for the two-pass kernel below.
// Against the kernels before (float4 rows aligned and in whole chunks; one
// element a lane, two passes and two expf an element otherwise), us:
//   CE fp32  2048 x 2048   7.8 -> 6.9     2000 x 10001   58.6 -> 29.6
//            2000 x 50257  358 -> 187
//   CE bf16  2048 x 50257  292 -> 87      8192 x 32000   465 -> 182
//            4000 x 10001  99.4 -> 32     1500 x 131072  721 -> 179
//   backward fp32 8192 x 32000 1063 -> 521  bf16 2048 x 50257 455 -> 113
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fg_half.h"

namespace fg {
namespace smany {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kNone = 0x7fffffff;  // no column

// Chunks of 16 bytes of element type DT.
template <int DT>
struct Io {
    static constexpr int E = DT == kF32 ? 4 : 8;  // elements of a chunk
    using T = typename std::conditional<DT == kF32, float, uint16_t>::type;
    static __device__ __forceinline__ float get(u32x4 w, int e) {
        if constexpr (DT == kF32) return __uint_as_float(w[e]);
        else if constexpr (DT == kBF16)
            return __uint_as_float((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
        else return f16_to_f((uint16_t)(w[e >> 1] >> (16 * (e & 1))));
    }
    static __device__ __forceinline__ u32x4 pack(const float (&v)[E]) {
        u32x4 w;
        if constexpr (DT == kF32) {
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = __float_as_uint(v[e]);
        } else if constexpr (DT == kBF16) {  // (two in one conversion: 4000 x 10001 33.4 -> 31.9 us)
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int q = 0; q < 4; ++q)
                w[q] = __builtin_bit_cast(
                    uint32_t, __builtin_convertvector((f32x2{v[2 * q], v[2 * q + 1]}), bf16x2));
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                w[q] = (uint32_t)f_to_f16(v[2 * q]) | ((uint32_t)f_to_f16(v[2 * q + 1]) << 16);
        }
        return w;
    }
    static __device__ __forceinline__ float load1(const T *p, int i) {
        if constexpr (DT == kF32) return p[i];
        else return h16_to_f(DT, p[i]);
    }
    static __device__ __forceinline__ void store1(T *p, int i, float v) {
        if constexpr (DT == kF32) p[i] = v;
        else p[i] = f_to_h16(DT, v);
    }
    // A chunk of -inf: what a chunk past the row's end holds.
    static __device__ __forceinline__ u32x4 minus_inf() {
        constexpr uint32_t w = DT == kF32 ? 0xff800000u : DT == kBF16 ? 0xff80ff80u : 0xfc00fc00u;
        return u32x4{w, w, w, w};
    }
};

// exp(x - m), x <= m (or NaN).  16-bit rows are bound by the vector unit where
// they take it twice an element, so they take it without expf's range checks: by
// the remainder of x - m to the nearest power of two, in two parts of log2(e),
// and the hardware's base-2 exponential of it.  Measured over [-79, 0], units of
// 2^-24: at most 1.37 off, 0.45 rms, as expf (1.35, 0.44); the exponential of
// (x - m) log2(e) rounded to fp32 is 2.7 off at -2, 8 at -8, 16 at -20, which
// shows in the fp32 row loss and below 2^-126 gives zeros.  2048 x 50257 CE bf16 /
// f16: 81 us with that, 87 / 92, with expf 111 / 128.
//
// The power is bounded, so that -inf leaves a remainder of -inf, and NaN stays in
// the remainder: by the conversion, which saturates, or in its own step where the
// exponentials are HELD (the conversion's form took 101 registers for 61 there: CE
// 8192 x 2048 bf16 14.7 us for 12.0; elsewhere 4 % less time).
template <int DT, bool HELD = false>
__device__ __forceinline__ float exp_below(float x, float m) {
    if constexpr (DT == kF32) {
        return expf(x - m);
    } else {
        constexpr float kLog2e = 1.44269502e+00f, kLog2eLow = 1.92596303e-08f;
        const float d = x - m;
        int k;
        float e;
        if constexpr (HELD) {
            e = fmaxf(__builtin_rintf(d * kLog2e), -200.0f);
            k = (int)e;
        } else {
            asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(k) : "v"(d * kLog2e));
            e = (float)k;
        }
        const float f = __builtin_fmaf(d, kLog2eLow, __builtin_fmaf(d, kLog2e, -e));
        return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), k);
    }
}

// Chunk j of a row, by an unsigned 32-bit offset from its (uniform) base,
// which keeps 64-bit addresses out of the vector registers.
__device__ __forceinline__ const u32x4 *at16(const u32x4 *base, int j) {
    return reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(base) +
                                           (uint32_t)j * 16u);
}
__device__ __forceinline__ u32x4 *at16(u32x4 *base, int j) {
    return reinterpret_cast<u32x4 *>(reinterpret_cast<char *>(base) + (uint32_t)j * 16u);
}

// How a row lies: elements before its first 16-byte boundary, whole chunks
// after it, elements after those; and the element outside the chunks that
// thread t holds (-1: none).
template <int DT>
struct Span {
    int head, nb, tail;
    __device__ __forceinline__ Span(const void *row, int C) {
        constexpr int E = Io<DT>::E, kSize = 16 / E;
        head = min((int)((16u - (uint32_t)((uintptr_t)row & 15u)) & 15u) / kSize, C);
        nb = (C - head) / E;
        tail = C - head - nb * E;
    }
    __device__ __forceinline__ int single(int t) const {
        constexpr int E = Io<DT>::E;
        if (t < head) return t;
        return t >= E && t < E + tail ? head + nb * E + t - E : -1;
    }
    // The thread of NT that holds column c: its single element, or one of its
    // chunks (chunk j is thread j % NT's).
    __device__ __forceinline__ int owner(int c, int NT) const {
        constexpr int E = Io<DT>::E;
        if (c < head) return c;
        const int k = c - head;
        return k < nb * E ? (k / E) & (NT - 1) : E + k - nb * E;
    }
};

// Makes packed values new to the compiler, which would otherwise keep every
// unpacked (and exponentiated) element of one pass for the next, twice or
// four times the registers.
template <int NV>
__device__ __forceinline__ void repack(u32x4 (&w)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(w[i]));
}

template <int NW>
__device__ __forceinline__ float max_over(float v, float *sm) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    if constexpr (NW > 1) {
        if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
        __syncthreads();
        v = sm[0];
#pragma unroll
        for (int k = 1; k < NW; ++k) v = fmaxf(v, sm[k]);
    }
    return v;
}
template <int NW>
__device__ __forceinline__ float sum_over(float v, float *sm) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if constexpr (NW > 1) {
        if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
        __syncthreads();
        v = sm[0];
#pragma unroll
        for (int k = 1; k < NW; ++k) v += sm[k];
    }
    return v;
}

// The sum over a wave's row of per-lane sums part[i] (those of the lane's i-th
// chunk): each of the NV added over the lanes, then the NV in order, as NV waves
// of one chunk a thread add them -- chains of a chunk, the six steps and NV, not of
// a lane's whole share of the row.  With NV > 1 the first steps halve the values a
// lane carries (lanes of bit 32, then 16, keep the upper ones).
template <int NV>
__device__ __forceinline__ float sum_chunks(const float (&part)[NV]) {
    static_assert(NV == 1 || NV == 2 || NV == 4, "one-wave rows");
    const int lane = threadIdx.x & 63;
    float v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = part[i];
    int o = 32;
#pragma unroll
    for (int n = NV / 2; n > 0; n /= 2, o >>= 1) {
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const float keep = up ? v[i + n] : v[i], give = up ? v[i] : v[i + n];
            v[i] = keep + __shfl_xor(give, o);
        }
    }
#pragma unroll
    for (; o > 0; o >>= 1) v[0] += __shfl_xor(v[0], o);
    if constexpr (NV == 1) return v[0];
    auto of = [&](int i) {  // the i-th chunks' sum
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[0]), i * (64 / NV)));
    };
    float s = of(0);
#pragma unroll
    for (int i = 1; i < NV; ++i) s += of(i);
    return s;
}

// A row's sum over the NV chunks a thread of NW waves holds, added an element at a
// time: a sum per chunk (in two halves where a chunk has eight elements), on one
// wave, which holds a larger share of the row a lane, added by sum_chunks, else by
// the thread.  fp32 on four waves: one running sum a thread.  In fp32 rows of up
// to 8192 columns on 16-byte boundaries are so added in the order of one float4 a
// thread on four waves.
template <int DT, int NV, int NW>
struct RowSum {
    static constexpr bool kEach = NW == 1, kRunning = DT == kF32 && NW == 4;
    float s[kEach ? NV : 1], lo = 0.0f, hi = 0.0f;
    __device__ __forceinline__ explicit RowSum(float first) {
#pragma unroll
        for (int i = 1; i < (kEach ? NV : 1); ++i) s[i] = 0.0f;
        s[0] = first;
    }
    __device__ __forceinline__ void add(int i, int e, float v) {
        if constexpr (kRunning || (kEach && DT == kF32)) {
            s[kEach ? i : 0] += v;
        } else {
            if (e % 4 == 0) (e ? hi : lo) = v;
            else (e > 4 ? hi : lo) += v;
            if (e == Io<DT>::E - 1) s[kEach ? i : 0] += Io<DT>::E > 4 ? lo + hi : lo;
        }
    }
    __device__ __forceinline__ float over(float *sm) {
        if constexpr (kEach) return sum_chunks<NV>(s);
        else return sum_over<NW>(s[0], sm);
    }
};

// What a label's column gets: the probability rounded, then less one.
__device__ __forceinline__ float label_grad(float scale, float e, float inv) {
#pragma clang fp contract(off)
    const float p = e * inv;
    return scale * (p - 1.0f);
}

// Threads of a workgroup whose rows take NW waves each (one wave a row:
// four rows a workgroup).
constexpr int threads_of(int NW) { return NW == 1 ? 256 : NW * 64; }
// Waves per SIMD the register budget is set for: two 1024-thread workgroups
// on a CU (64 VGPRs) where the row leaves room, so that one row's reductions
// overlap the other's memory traffic.
constexpr int waves_of(int NV, int NW) { return NW >= 16 ? (NV <= 8 ? 8 : 4) : 1; }

// The register-resident row: NV chunks a thread on NW waves, read once and
// written once.  16-bit rows stay packed (NV <= 4: their exponentials are
// kept; else they are taken again from the packed values for the output,
// which leaves room for a second row on the CU).
template <int DT, int NV, int NW>
__global__ __launch_bounds__(threads_of(NW)) __attribute__((amdgpu_waves_per_eu(waves_of(NV, NW))))
void softmax_any(const typename Io<DT>::T *x, int ldx,
                 const uint32_t *__restrict__ labels, int R, int C, float scale,
                 float *__restrict__ row_loss, typename Io<DT>::T *out, int ldo,
                 uint32_t *__restrict__ argmax, typename Io<DT>::T *probs, int ldp) {
    using IO = Io<DT>;
    constexpr int E = IO::E, NT = NW * 64;
    constexpr bool kHold = DT == kF32 || NV <= 4;
    __shared__ float smax[NW], ssum[NW];
    __shared__ int sarg;
    const int r = NW == 1 ? (int)(blockIdx.x * 4 + (threadIdx.x >> 6)) : (int)blockIdx.x;
    if (NW == 1 && r >= R) return;
    const int t = NW == 1 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
    const auto *xr = x + (size_t)r * ldx;
    const Span<DT> sp(xr, C);
    const u32x4 *xb = reinterpret_cast<const u32x4 *>(xr + sp.head);
    u32x4 w[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = t + i * NT;
        w[i] = j < sp.nb ? __builtin_nontemporal_load(at16(xb, j)) : IO::minus_inf();
    }
    float vs = sp.single(t) >= 0 ? IO::load1(xr, sp.single(t)) : -INFINITY;
    const uint32_t lab = labels ? labels[r] : 0xffffffffu;
    const int tc = lab < (uint32_t)C ? (int)lab : -1;
    if (NW > 1 && t == 0) sarg = kNone;
    float lm = vs;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) lm = fmaxf(lm, IO::get(w[i], e));
    const float m = max_over<NW>(lm, smax);
    if constexpr (!kHold) repack(w);
    if (argmax) {  // the lowest column holding the maximum
        int am = kNone;
        if (lm == m) {
            if (sp.single(t) >= 0 && vs == m) am = sp.single(t);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int j = t + i * NT;
                if (j >= sp.nb) continue;
#pragma unroll
                for (int e = 0; e < E; ++e)
                    if (IO::get(w[i], e) == m) am = min(am, sp.head + j * E + e);
            }
        }
        if constexpr (NW == 1) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) am = min(am, __shfl_xor(am, o));
            if (t == 0) argmax[r] = (uint32_t)am;
        } else if (am != kNone) {
            atomicMin(&sarg, am);
        }
    }
    if constexpr (!kHold) repack(w);
    float ex[kHold ? NV * E : 1];
    vs = sp.single(t) >= 0 ? exp_below<DT, kHold>(vs, m) : 0.0f;
    RowSum<DT, NV, NW> sum(vs);
    // Where exponentials are taken twice, a wave leaves out the chunks of which it
    // holds none: 4000 x 10001 bf16 / f16 42 / 49 us, now 34 / 40.  (Held ones: no
    // faster, 8192 x 2048 12.6 / 14.4 against 16.)
    const int first = __builtin_amdgcn_readfirstlane(t) & ~63;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if (!kHold && first + i * NT >= sp.nb) break;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float p = exp_below<DT, kHold>(IO::get(w[i], e), m);
            if constexpr (kHold) ex[i * E + e] = p;
            sum.add(i, e, p);
        }
    }
    // The label's logit, in the thread that writes its column and before any
    // thread stores (out may be x).
    const bool mine = tc >= 0 && t == sp.owner(tc, NT);
    float xt = 0.0f;
    if (mine) xt = IO::load1(xr, tc);
    const float s = sum.over(ssum);
    if (t == 0) {
        if (NW > 1 && argmax) argmax[r] = (uint32_t)sarg;
        // A label outside [0, C) has no logit; report NaN rather than read.
        if (row_loss && tc < 0) row_loss[r] = __builtin_nanf("");
    }
    if (row_loss && mine) row_loss[r] = (m + logf(s)) - xt;
    const float inv = 1.0f / s;
    auto write = [&](typename IO::T *dst, float g) {  // dst = g * softmax
        u32x4 *db = reinterpret_cast<u32x4 *>(dst + sp.head);
        const int cs = sp.single(t);
        if (cs >= 0) IO::store1(dst, cs, g * (vs * inv));
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int j = t + i * NT;
            if (j >= sp.nb) continue;
            if constexpr (!kHold) asm volatile("" : "+v"(w[i]));
            float d[E];
#pragma unroll
            for (int e = 0; e < E; ++e)
                d[e] = g * ((kHold ? ex[i * E + e] : exp_below<DT, kHold>(IO::get(w[i], e), m)) * inv);
            __builtin_nontemporal_store(IO::pack(d), at16(db, j));
        }
    };
    if (out) {
        auto *orow = out + (size_t)r * ldo;
        write(orow, scale);
        // Then, over it, the label's column.
        if (mine) IO::store1(orow, tc, label_grad(scale, exp_below<DT, kHold>(xt, m), inv));
    }
    if (probs) write(probs + (size_t)r * ldp, 1.0f);
}

// Rows too long for the registers: pass 1 keeps an online (max, sum) per
// thread, rescaled at most once per kStep chunks; pass 2 reads the row again
// (from the caches) and writes.  One 1024-thread workgroup a row.
constexpr int kLongNW = 16, kStep = 4;
template <int DT>
__global__ __launch_bounds__(kLongNW * 64) void softmax_long(
    const typename Io<DT>::T *x, int ldx, const uint32_t *__restrict__ labels, int C,
    float scale, float *__restrict__ row_loss, typename Io<DT>::T *out, int ldo,
    uint32_t *__restrict__ argmax, typename Io<DT>::T *probs, int ldp) {
    using IO = Io<DT>;
    constexpr int E = IO::E, NT = kLongNW * 64;
    __shared__ float smax[kLongNW], ssum[kLongNW];
    __shared__ int sarg;
    const int r = blockIdx.x, t = threadIdx.x;
    const auto *xr = x + (size_t)r * ldx;
    const Span<DT> sp(xr, C);
    const u32x4 *xb = reinterpret_cast<const u32x4 *>(xr + sp.head);
    const int cs = sp.single(t);
    const float vs = cs >= 0 ? IO::load1(xr, cs) : -INFINITY;
    const uint32_t lab = labels ? labels[r] : 0xffffffffu;
    const int tc = lab < (uint32_t)C ? (int)lab : -1;
    const bool mine = tc >= 0 && t == sp.owner(tc, NT);
    const float xt = mine ? IO::load1(xr, tc) : 0.0f;  // before any store: out may be x
    if (t == 0) sarg = kNone;
    float m = -INFINITY, s = 0.0f;
    int jm = -1;  // the step that raised the maximum last
    for (int j0 = t; j0 < sp.nb; j0 += NT * kStep) {
        u32x4 w[kStep];
#pragma unroll
        for (int i = 0; i < kStep; ++i)
            w[i] = j0 + i * NT < sp.nb ? xb[j0 + i * NT] : IO::minus_inf();
        float bm = -INFINITY;
#pragma unroll
        for (int i = 0; i < kStep; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) bm = fmaxf(bm, IO::get(w[i], e));
        if (bm > m) {
            s *= exp_below<DT>(m, bm);  // m = -inf: s is 0 or NaN
            m = bm;
            jm = j0;
        }
        // Nothing above -inf yet: only a NaN counts.
        const float base = m == -INFINITY ? 0.0f : m;
        float step = 0.0f;
#pragma unroll
        for (int i = 0; i < kStep; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) step += exp_below<DT>(IO::get(w[i], e), base);
        s += step;
    }
    const float lm = fmaxf(m, vs);
    const float mr = max_over<kLongNW>(lm, smax);
    if (argmax && lm == mr) {
        int am = kNone;
        if (cs >= 0 && vs == mr) am = cs;
        // A thread whose maximum is -inf has raised it in no step: its
        // first chunk holds its lowest column.
        const int j0 = m == -INFINITY ? t : jm;
        if (m == mr)
            for (int i = 0; i < kStep; ++i) {
                const int j = j0 + i * NT;
                if (j >= sp.nb) break;
                const u32x4 w = xb[j];
#pragma unroll
                for (int e = 0; e < E; ++e)
                    if (IO::get(w, e) == mr) am = min(am, sp.head + j * E + e);
            }
        if (am != kNone) atomicMin(&sarg, am);
    }
    // A thread that saw nothing above -inf adds its (zero or NaN) sum as is.
    float part = m == -INFINITY ? s : s * exp_below<DT>(m, mr);
    float es = cs >= 0 ? exp_below<DT>(vs, mr) : 0.0f;
    s = sum_over<kLongNW>(part + es, ssum);
    if (t == 0) {
        if (argmax) argmax[r] = (uint32_t)sarg;
        if (row_loss && tc < 0) row_loss[r] = __builtin_nanf("");
    }
    if (row_loss && mine) row_loss[r] = (mr + logf(s)) - xt;
    if (!out && !probs) return;
    const float inv = 1.0f / s;
    auto *orow = out ? out + (size_t)r * ldo : nullptr;
    auto *prow = probs ? probs + (size_t)r * ldp : nullptr;
    if (cs >= 0) {
        const float p = es * inv;
        if (out) IO::store1(orow, cs, scale * p);
        if (probs) IO::store1(prow, cs, p);
    }
    for (int j0 = t; j0 < sp.nb; j0 += NT * kStep) {
        u32x4 w[kStep];
#pragma unroll
        for (int i = 0; i < kStep; ++i)
            w[i] = j0 + i * NT < sp.nb ? xb[j0 + i * NT] : IO::minus_inf();
#pragma unroll
        for (int i = 0; i < kStep; ++i) {
            const int j = j0 + i * NT;
            if (j >= sp.nb) continue;
            float p[E], d[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                p[e] = exp_below<DT>(IO::get(w[i], e), mr) * inv;
                d[e] = scale * p[e];
            }
            if (out)
                __builtin_nontemporal_store(IO::pack(d),
                                            reinterpret_cast<u32x4 *>(orow + sp.head) + j);
            if (probs)
                __builtin_nontemporal_store(IO::pack(p),
                                            reinterpret_cast<u32x4 *>(prow + sp.head) + j);
        }
    }
    if (out && mine) IO::store1(orow, tc, label_grad(scale, exp_below<DT>(xt, mr), inv));
}

// dx (=|+=) y * (dy - sum(dy * y)), y and dy held in registers.
template <int DT, int NV, int NW>
__global__ __launch_bounds__(threads_of(NW)) void softmax_bwd_any(
    const typename Io<DT>::T *y, const typename Io<DT>::T *dy, int R,
    int C, typename Io<DT>::T *dx, int accumulate) {
    using IO = Io<DT>;
    constexpr int E = IO::E, NT = NW * 64;
    __shared__ float ssum[NW];
    const int r = NW == 1 ? (int)(blockIdx.x * 4 + (threadIdx.x >> 6)) : (int)blockIdx.x;
    if (NW == 1 && r >= R) return;
    const int t = NW == 1 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
    const size_t base = (size_t)r * C;
    const Span<DT> sp(y + base, C);
    const u32x4 *yb = reinterpret_cast<const u32x4 *>(y + base + sp.head);
    const u32x4 *db = reinterpret_cast<const u32x4 *>(dy + base + sp.head);
    u32x4 wy[NV], wd[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = t + i * NT;
        wy[i] = j < sp.nb ? __builtin_nontemporal_load(yb + j) : u32x4{0, 0, 0, 0};
        wd[i] = j < sp.nb ? __builtin_nontemporal_load(db + j) : u32x4{0, 0, 0, 0};
    }
    const int cs = sp.single(t);
    const float ys = cs >= 0 ? IO::load1(y + base, cs) : 0.0f;
    const float ds = cs >= 0 ? IO::load1(dy + base, cs) : 0.0f;
    RowSum<DT, NV, NW> sum(ds * ys);
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) sum.add(i, e, IO::get(wd[i], e) * IO::get(wy[i], e));
    const float dot = sum.over(ssum);
    if constexpr (DT != kF32) {
        repack(wy);
        repack(wd);
    }
    auto *xr = dx + base;
    if (cs >= 0) {
        const float g = ys * (ds - dot);
        IO::store1(xr, cs, accumulate ? IO::load1(xr, cs) + g : g);
    }
    u32x4 *xb = reinterpret_cast<u32x4 *>(xr + sp.head);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = t + i * NT;
        if (j >= sp.nb) continue;
        float g[E];
#pragma unroll
        for (int e = 0; e < E; ++e) g[e] = IO::get(wy[i], e) * (IO::get(wd[i], e) - dot);
        if (accumulate) {
            const u32x4 old = xb[j];
#pragma unroll
            for (int e = 0; e < E; ++e) g[e] = IO::get(old, e) + g[e];
        }
        __builtin_nontemporal_store(IO::pack(g), xb + j);
    }
}

// The same for rows too long for the registers: the row is read twice.
template <int DT>
__global__ __launch_bounds__(kLongNW * 64) void softmax_bwd_long(
    const typename Io<DT>::T *y, const typename Io<DT>::T *dy, int C,
    typename Io<DT>::T *dx, int accumulate) {
    using IO = Io<DT>;
    constexpr int E = IO::E, NT = kLongNW * 64;
    __shared__ float ssum[kLongNW];
    const int t = threadIdx.x;
    const size_t base = (size_t)blockIdx.x * C;
    const Span<DT> sp(y + base, C);
    const u32x4 *yb = reinterpret_cast<const u32x4 *>(y + base + sp.head);
    const u32x4 *db = reinterpret_cast<const u32x4 *>(dy + base + sp.head);
    const int cs = sp.single(t);
    const float ys = cs >= 0 ? IO::load1(y + base, cs) : 0.0f;
    const float ds = cs >= 0 ? IO::load1(dy + base, cs) : 0.0f;
    float dot = ds * ys;
#pragma unroll 2
    for (int j = t; j < sp.nb; j += NT) {
        const u32x4 wy = yb[j], wd = db[j];
        float chunk = 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) chunk += IO::get(wd, e) * IO::get(wy, e);
        dot += chunk;
    }
    dot = sum_over<kLongNW>(dot, ssum);
    auto *xr = dx + base;
    if (cs >= 0) {
        const float g = ys * (ds - dot);
        IO::store1(xr, cs, accumulate ? IO::load1(xr, cs) + g : g);
    }
    u32x4 *xb = reinterpret_cast<u32x4 *>(xr + sp.head);
#pragma unroll 2
    for (int j = t; j < sp.nb; j += NT) {
        const u32x4 wy = yb[j], wd = db[j];
        float g[E];
#pragma unroll
        for (int e = 0; e < E; ++e) g[e] = IO::get(wy, e) * (IO::get(wd, e) - dot);
        if (accumulate) {
            const u32x4 old = xb[j];
#pragma unroll
            for (int e = 0; e < E; ++e) g[e] = IO::get(old, e) + g[e];
        }
        __builtin_nontemporal_store(IO::pack(g), xb + j);
    }
}

}  // namespace smany
}  // namespace fg
