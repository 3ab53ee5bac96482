// elementwise.hpp -- N-d elementwise engine for gfx950 (binary, scalar, unary, relu, clip, copy,
// broadcast).
//
// One Matrix-level call of the reference (add_array, mul_scalar, exp_array, relu, copy_from ...,
// zenu-matrix/src/operation/basic_operations.rs:278-381,512-611, relu.rs:169-242,
// copy_from.rs:211-267) becomes ONE launch here instead of one 1-D launch per row
// (zenu-matrix/src/with_clousers.rs:180-223).  After the host has folded the operands into a
// common iteration space (shape.cpp) one of four kernels runs:
//
//   contig : every operand is one contiguous run.  128-bit loads/stores; 64 threads x one vector
//            when one input streams (the shape that moves load + store traffic fastest), 256
//            threads x two vectors for two inputs and for tanh / sigmoid.           [HBM bound]
//   rows   : the innermost dim is contiguous (stride 1) or broadcast (stride 0) in every operand;
//            outer dims are arbitrary.  Covers row / column broadcast and row-sliced views.  The
//            outer index is decomposed once per thread, the inner dim is walked with 128-bit
//            accesses; a broadcast row stays in L2.                                   [HBM bound]
//   tile   : some input is contiguous along a different dim than the output (a transposed
//            operand).  64x64 tiles walked along diagonals, one thread per vector: the transposed
//            input is read along ITS contiguous dim with 128-bit loads in 128-byte segments,
//            turned through LDS (pitch 65 words, eight lanes per segment: no bank conflicts in
//            either direction, checked with the hardware counter), and every HBM access stays
//            coalesced.                                                               [HBM bound]
//   strided: anything else (a strided destination, gathers, views without a unit-stride dim):
//            lanes along the innermost dim whatever its stride, the outer index decomposed once
//            per thread, four elements per thread with the loads issued first.
//
// Arithmetic is plain IEEE with contraction off; + - * / sqrt are correctly rounded on gfx950,
// so results are bit-identical to the CPU loops of basic_operations.rs:93-181.
// This header holds the functors, the kernels and the launch logic; the entry points are spread over
// ew_binary.hip, ew_unary.hip, ew_unary_trig.hip and ew_misc.hip so that their template
// instantiations compile in parallel.
#pragma once
#include <math.h>

#include "common.hpp"
#include "vecmem.hpp"
#include "zmath.hpp"

#include <type_traits>

namespace zenu {
namespace {

constexpr int kBlock = 256;
#ifndef ZENU_EW_UNROLL
#define ZENU_EW_UNROLL 2
#endif
constexpr int kUnroll = ZENU_EW_UNROLL;
#ifndef ZENU_EW1_BLOCK
#define ZENU_EW1_BLOCK 64
#endif
#ifndef ZENU_EW1_UNROLL
#define ZENU_EW1_UNROLL 1
#endif

// ---- functors -----------------------------------------------------------------------------------

template <typename T, int OP> __device__ __forceinline__ T bin_apply(T a, T b)
{
    if constexpr (OP == ZENU_ADD) return a + b;
    else if constexpr (OP == ZENU_SUB) return a - b;
    else if constexpr (OP == ZENU_MUL) return a * b;
    else return a / b;
}

template <typename T, int OP> struct BinF {
    static constexpr int NIN = 2;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T a, T b) const { return bin_apply<T, OP>(a, b); }
};

// a op s; the scalar comes by value or from device memory (0-d tensor operand)
template <typename T, int OP> struct ScalarF {
    static constexpr int NIN = 1;
    T s;
    const T *sp;
    __device__ __forceinline__ void init() { if (sp) s = *sp; }
    __device__ __forceinline__ T operator()(T a, T) const { return bin_apply<T, OP>(a, s); }
};

__device__ __forceinline__ float dev_tanh(float x, const zmath::TanhRegs &rg) { return zmath::tanhf_simd(x, rg); }
__device__ __forceinline__ double dev_tanh(double x, const zmath::TanhRegs &) { return zmath::tanh_simd(x); }
__device__ __forceinline__ float dev_asin(float x) { return zmath::asinf_fdlibm(x); }
__device__ __forceinline__ double dev_asin(double x) { return asin(x); }
__device__ __forceinline__ float dev_acos(float x) { return zmath::acosf_fdlibm(x); }
__device__ __forceinline__ double dev_acos(double x) { return acos(x); }
__device__ __forceinline__ float dev_atan(float x) { return zmath::atanf_fdlibm(x); }
__device__ __forceinline__ double dev_atan(double x) { return atan(x); }
__device__ __forceinline__ float dev_sigmoid(float x, const zmath::TanhRegs &rg) { return zmath::sigmoidf_zenu(x, rg); }
__device__ __forceinline__ double dev_sigmoid(double x, const zmath::TanhRegs &) { return zmath::sigmoid_zenu(x); }

// what single functions carry besides: the f64 constants of the sine / cosine / tangent (in the functor, a
// kernel argument), the tables of the f64 sine / cosine and of the f32 arc tangent (in LDS); every other function nothing
template <typename T, int FN> struct UnaryExtra {
    __device__ __forceinline__ void init() {}
};
template <> struct UnaryExtra<float, ZENU_SIN> {
    zmath::SinCosCoef k;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ float sin(float x) const { return zmath::sinf_glibc(x, k); }
};
template <> struct UnaryExtra<float, ZENU_COS> {
    zmath::SinCosCoef k;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ float cos(float x) const { return zmath::cosf_glibc(x, k); }
};
template <> struct UnaryExtra<double, ZENU_SIN> {
    zmath::SinCos64Coef k;
    zmath::SinCos64Lds t;
    __device__ __forceinline__ void init() { t.init(); }
    __device__ __forceinline__ double sin(double x) const { return zmath::sin_glibc(x, t.tab, k); }
};
template <> struct UnaryExtra<double, ZENU_COS> {
    zmath::SinCos64Coef k;
    zmath::SinCos64Lds t;
    __device__ __forceinline__ void init() { t.init(); }
    __device__ __forceinline__ double cos(double x) const { return zmath::cos_glibc(x, t.tab, k); }
};
template <> struct UnaryExtra<float, ZENU_TAN> {
    zmath::TanfCoef tk;
    __device__ __forceinline__ void init() {}
};
template <> struct UnaryExtra<float, ZENU_ATAN> {
    zmath::AtanfLds t;
    __device__ __forceinline__ void init() { t.init(); }
};

template <typename T, int FN> struct UnaryF {
    static constexpr int NIN = 1;
    zmath::ExpLog<T> m;     // exp / log state (f32: tables in LDS)
    zmath::TanhRegs tr;     // f32 tanh / sigmoid / sinh / cosh: two constants held in vector registers
    UnaryExtra<T, FN> sc;   // f32 sin / cos / tan: the f64 constants, as data; f32 atan: its table
    __device__ __forceinline__ void init()
    {
        if constexpr (FN == ZENU_EXP || FN == ZENU_LOG || FN == ZENU_SINH || FN == ZENU_COSH)
            m.init(FN != ZENU_LOG, FN == ZENU_LOG);
        if constexpr (FN == ZENU_TANH || FN == ZENU_SIGMOID || FN == ZENU_SINH || FN == ZENU_COSH) tr.pin();
        sc.init();
    }
    __device__ __forceinline__ T operator()(T a, T) const
    {
        if constexpr (FN == ZENU_EXP) return m.exp(a);
        else if constexpr (FN == ZENU_LOG) return m.log(a);
        else if constexpr (FN == ZENU_TANH) return m.tanh(a, tr);
        else if constexpr (FN == ZENU_SQRT) return sqrt(a);
        else if constexpr (FN == ZENU_ABS) return fabs(a);
        else if constexpr (FN == ZENU_SIN) return sc.sin(a);
        else if constexpr (FN == ZENU_COS) return sc.cos(a);
        else if constexpr (FN == ZENU_TAN) {
            if constexpr (sizeof(T) == 4) return zmath::tanf_glibc(a, sc.tk);
            else return tan(a);
        }
        else if constexpr (FN == ZENU_ASIN) return dev_asin(a);
        else if constexpr (FN == ZENU_ACOS) return dev_acos(a);
        else if constexpr (FN == ZENU_ATAN) {
            if constexpr (sizeof(T) == 4) return zmath::atanf_fdlibm(a, sc.t.tab);
            else return dev_atan(a);
        }
        else if constexpr (FN == ZENU_SINH) return m.sinh(a, tr);
        else if constexpr (FN == ZENU_COSH) return m.cosh(a, tr);
        else return m.sigmoid(a, tr);
    }
};

// f32 tanh within 2 units in the last place of the host library's, evaluated in f64 (no
// counterpart in the reference; f64 goes to the exact tanh instead)
struct TanhUlp2F {
    static constexpr int NIN = 1;
    zmath::TanhUlp2Coef q;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ float operator()(float a, float) const { return zmath::tanhf_ulp2(a, q); }
};

template <typename T> struct PowF {
    static constexpr int NIN = 1;
    T s;
    zmath::Pow<T> m;        // f32: tables in LDS
    __device__ __forceinline__ void init() { m.init(); }
    __device__ __forceinline__ T operator()(T a, T) const { return m.pow(a, s); }
};

// relu.rs:44-48: the non-positive branch returns the PRODUCT alpha*x (-0.0 for alpha = 0)
template <typename T> struct ReluF {
    static constexpr int NIN = 1;
    T alpha;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T a, T) const { return (a > (T)0) ? a : alpha * a; }
};
// relu.rs:74-78
template <typename T> struct ReluMaskF {
    static constexpr int NIN = 1;
    T alpha;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T a, T) const { return (a > (T)0) ? (T)1 : alpha * (T)-1; }
};
// relu.rs backward: gx = gy * mask(x), the mask of ReluMaskF (zenu-autograd/src/activation/relu.rs:35-44)
template <typename T> struct ReluBwdF {
    static constexpr int NIN = 2;
    T alpha;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T gy, T x) const { return gy * ((x > (T)0) ? (T)1 : alpha * (T)-1); }
};
// backward of tanh (zenu-autograd/src/functions/tanh.rs:30-37): cosh(x), its square, gy / square --
// three ops there, each rounded once; the same roundings here in one pass
template <typename T> struct TanhBwdF {
    static constexpr int NIN = 2;
    zmath::ExpLog<T> m;
    __device__ __forceinline__ void init() { m.init(true, false); }
    __device__ __forceinline__ T operator()(T gy, T x) const
    {
        const T c = m.cosh(x);
        const T c2 = c * c;
        return gy / c2;
    }
};
// backward of the sigmoid composite (zenu-autograd/src/activation/sigmoid.rs:7-15) through its add,
// mul, tanh and mul nodes (functions/mul.rs:35-44): ((0.5 gy) / cosh(0.5 x)^2) 0.5, every step rounded
template <typename T> struct SigmoidBwdF {
    static constexpr int NIN = 2;
    zmath::ExpLog<T> m;
    __device__ __forceinline__ void init() { m.init(true, false); }
    __device__ __forceinline__ T operator()(T gy, T x) const
    {
        const T half = (T)0.5;
        const T xh = x * half;
        const T c = m.cosh(xh);
        const T c2 = c * c;
        const T g1 = half * gy;
        const T g2 = g1 / c2;
        return g2 * half;
    }
};
// clip.rs:50-57: below min -> min, above max -> max, NaN passes through
template <typename T> struct ClipF {
    static constexpr int NIN = 1;
    T lo, hi;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T a, T) const { return a < lo ? lo : (a > hi ? hi : a); }
};
// clip.rs:90-96: 0 outside [min, max], 1 inside (and for NaN)
template <typename T> struct ClipMaskF {
    static constexpr int NIN = 1;
    T lo, hi;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T a, T) const { return (a < lo || a > hi) ? (T)0 : (T)1; }
};
template <typename T> struct CopyF {
    static constexpr int NIN = 1;
    __device__ __forceinline__ void init() {}
    __device__ __forceinline__ T operator()(T a, T) const { return a; }
};

// ---- how a kernel's operands pass the caches --------------------------------------------------------
// Below kStreamBytes: no hints.  Above, stores stream (a store that allocates pushes out what the next call reads), and
//   kMemKeep    inputs are loaded plainly while those of full size are below kKeepInputs: they are often read again, a data
//               matrix by the next statistic, a forward input by the backward pass.
//   kMemFeed    a layer's own step, whose result is what the next call reads: ReLU, its backward pass, a bias per channel
//               or row.  Written through without the hint, it waits in the memory-side cache; the inputs stream.
//   kMemStream  beyond that everything streams.
// us, plain loads / streaming, f32, operands used once and by three calls in turn: a + b of 36 MB 7.7 / 7.5, 4.7 / 7.2; 64 MB
// 12.5 / 12.0, 11.0 / 11.7; 96 MB 17.7 / 16.9, 15.5 / 16.5; 128 MB 22.9 / 21.5, 20.2 / 21.2; 201 MB 34.9 / 32.2, 30.4 / 31.8; copy of 64 MB
// 11.5 / 11.2, 9.3 / 9.9; 128 MB 21.5 / 20.7, 19.5 / 20.4; 160 MB 26.5 / 25.2, 24.0 / 25.1; 250 MB 40.4 / 38.3, 36.5 / 38.0; a + b^T 64 MB
// 13.7 / 13.2, 11.7 / 12.9; 195 MB 35.0 / 32.9, 31.1 / 32.7.  Above 72 MB of inputs what is lost by the first use is more than a later one gains.
// us with everything streaming / by these rules: bias, ReLU, NCHW -> NHWC, ReLU backward, bias gradient of [64,512,14,14]
// f32 53.5 / 47.7 (257 MB moved), [64,256,28,28] 95.8 / 88.2, f64 [16,64,56,56] 54.8 / 49.5; a + row, a * column, a + b^T, 0.5 a
// of [3001,2047] f32 45.5 / 42.5, [2000,4000] 54.6 / 49.3, [4096,4096] 102.4 / 92.8; ReLU and its backward pass of 8 million 27.9 / 25.7.
// Feeding from the 201 MB of a ReLU backward of 2^24 on loses, 31.7 / 33.6; at 154 MB 24.9 / 24.1.
enum { kMemCached, kMemKeep, kMemFeed, kMemStream };
constexpr int64_t kKeepInputs = 72ll << 20, kFeedBytes = 6 * kStreamBytes;
constexpr bool streams_loads(int mem) { return mem == kMemStream || mem == kMemFeed; }

// ONE_IN: one input streams beside the output (the written-through streaming store, vecmem.hpp)
template <typename T, int VEC, int MEM, bool ONE_IN> __device__ __forceinline__ void store_mem(T *p, const Pack<T, VEC> &r)
{
    if constexpr (VEC == 1 || MEM == kMemCached) store_pack<T, VEC, false>(p, r);
    else if constexpr (MEM == kMemFeed) store_pack_through<T, VEC>(p, r);
    else if constexpr (ONE_IN) store_pack_wt<T, VEC>(p, r);
    else store_pack<T, VEC, true>(p, r);
}

template <typename F> struct IsLayerStep { static constexpr bool value = false; };
template <typename T> struct IsLayerStep<ReluF<T>> { static constexpr bool value = true; };
template <typename T> struct IsLayerStep<ReluBwdF<T>> { static constexpr bool value = true; };
template <typename F> struct IsCopy { static constexpr bool value = false; };
template <typename T> struct IsCopy<CopyF<T>> { static constexpr bool value = true; };
template <typename F> struct IsAdd { static constexpr bool value = false; };
template <typename T> struct IsAdd<BinF<T, ZENU_ADD>> { static constexpr bool value = true; };

template <typename T, int N, typename F>
__device__ __forceinline__ Pack<T, N> apply_pack(const F &f, const Pack<T, N> &a, const Pack<T, N> &b)
{
    Pack<T, N> r;
#pragma unroll
    for (int i = 0; i < N; i++) r.v[i] = f(a.v[i], b.v[i]);
    return r;
}

// ---- kernel 1: contiguous ------------------------------------------------------------------------

// Workgroup shape per stream count (measured on 2^24 f32): two-stream ops (one load, one store)
// run best as many small workgroups with one vector per lane (copy: 6.26 TB/s at 64 x 1 against
// 5.92 at 256 x 2); three-stream ops are flat across shapes and keep 256 x 2.
// The VALU-bound functors (tanh, sigmoid) prefer the larger shape too.
template <typename F> struct IsValuBound { static constexpr bool value = false; };
template <typename T> struct IsValuBound<UnaryF<T, ZENU_TANH>> { static constexpr bool value = true; };
template <typename T> struct IsValuBound<UnaryF<T, ZENU_SIGMOID>> { static constexpr bool value = true; };
template <> struct IsValuBound<TanhUlp2F> { static constexpr bool value = true; };   // 24.4 us against 27.1 at 64 x 1
// f64 sine / cosine: a 3.5 KiB table per workgroup, and 60 f64 operations per element
template <> struct IsValuBound<UnaryF<double, ZENU_SIN>> { static constexpr bool value = true; };
template <> struct IsValuBound<UnaryF<double, ZENU_COS>> { static constexpr bool value = true; };
// measured on 2^24 elements (us at 64 x 1 -> at 256 x 2): f32 sin 25.6 -> 23.8, cos 25.9 -> 23.8, asin 25.4 -> 24.0,
// sinh 25.7 -> 25.2, cosh 26.4 -> 25.0; f64 sinh 63.9 -> 61.6, cosh 62.4 -> 55.4, sin 88.4 -> 49.8, cos 86.4 -> 49.6.
// (f32 acos 25.0 -> 26.3 and atan 23.5 -> 24.7 prefer the small shape, tan does not care.)
template <typename T> struct IsValuBound<UnaryF<T, ZENU_SINH>> { static constexpr bool value = true; };
template <typename T> struct IsValuBound<UnaryF<T, ZENU_COSH>> { static constexpr bool value = true; };
template <> struct IsValuBound<UnaryF<float, ZENU_SIN>> { static constexpr bool value = true; };
template <> struct IsValuBound<UnaryF<float, ZENU_COS>> { static constexpr bool value = true; };
template <> struct IsValuBound<UnaryF<float, ZENU_ASIN>> { static constexpr bool value = true; };
// f64 powf: 5 KiB of tables per workgroup (89 us at 64 x 1)
template <> struct IsValuBound<PowF<double>> { static constexpr bool value = true; };
template <typename T> struct IsValuBound<TanhBwdF<T>> { static constexpr bool value = true; };
template <typename T> struct IsValuBound<SigmoidBwdF<T>> { static constexpr bool value = true; };

// Largest tensor, in elements per CU, that goes one element per lane instead of as vectors.  A transcendental functor
// makes a lane's VEC * kUnroll elements a long chain; while the vectors leave SIMDs without work, four times the
// wavefronts with a quarter of the chain are faster.  us as vectors / one per lane, by number of elements: f32 sigmoid
// 10007: 4.1 / 2.4, 100003: 3.4 / 2.4, 600000: 3.9 / 3.3, 2^20: 4.2 / 4.1, 2^21: 6.2 / 6.1; f64 sigmoid 100003:
// 3.3 / 2.7, 600000: 5.3 / 4.8, 2^20: 6.8 / 6.6; f32 exp 10007: 3.0 / 2.3, 100003: 3.0 / 2.4, 200000: 2.8 / 2.8,
// 300001: 2.7 / 3.1.  Light functors (add, relu, copy) gain nothing.
template <typename F> struct IsTranscendental { static constexpr bool value = IsValuBound<F>::value; };
template <typename T, int FN> struct IsTranscendental<UnaryF<T, FN>> { static constexpr bool value = FN != ZENU_SQRT && FN != ZENU_ABS; };
template <typename T> struct IsTranscendental<PowF<T>> { static constexpr bool value = true; };
template <typename F> constexpr int64_t kSinglesPerCu = IsValuBound<F>::value ? 4096 : IsTranscendental<F>::value ? 512 : 0;

template <typename F> struct ContigShape {
    static constexpr bool kSmall = F::NIN == 1 && !IsValuBound<F>::value;
    static constexpr int kBlock = kSmall ? ZENU_EW1_BLOCK : 256;
    static constexpr int kUnroll = kSmall ? ZENU_EW1_UNROLL : zenu::kUnroll;
};

template <typename T, int VEC, int MEM, typename F>
__global__ __launch_bounds__(ContigShape<F>::kBlock) void ew_contig_kernel(T *out, const T *a, const T *b,
                                                                         int64_t n, F f)
{
    constexpr int kBlock = ContigShape<F>::kBlock;
    constexpr int kUnroll = ContigShape<F>::kUnroll;
    constexpr int64_t kTile = (int64_t)kBlock * VEC * kUnroll;
    const int64_t base = (int64_t)blockIdx.x * kTile;
    const int tid = threadIdx.x;
    if (base + kTile <= n) {
        Pack<T, VEC> va[kUnroll], vb[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            int64_t i = base + ((int64_t)u * kBlock + tid) * VEC;
            va[u] = load_pack<T, VEC, streams_loads(MEM)>(a + i);
            if constexpr (F::NIN == 2) vb[u] = load_pack<T, VEC, streams_loads(MEM)>(b + i);
            else vb[u] = va[u];
        }
        f.init();   // after the loads are issued: what it fetches (a device scalar, a table) overlaps them
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            int64_t i = base + ((int64_t)u * kBlock + tid) * VEC;
            const Pack<T, VEC> r = apply_pack<T, VEC, F>(f, va[u], vb[u]);
            store_mem<T, VEC, MEM, ContigShape<F>::kSmall>(out + i, r);
        }
    } else {   // the last tile: whole vectors while they last, then the remaining elements one by one
        f.init();
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            int64_t i = base + ((int64_t)u * kBlock + tid) * VEC;
            if (i + VEC <= n) {
                const Pack<T, VEC> x = load_pack<T, VEC, false>(a + i);
                const Pack<T, VEC> y = (F::NIN == 2) ? load_pack<T, VEC, false>(b + i) : x;
                store_pack<T, VEC, false>(out + i, apply_pack<T, VEC, F>(f, x, y));
            } else {
                for (int j = 0; j < VEC; j++) {
                    if (i + j < n) {
                        T x = a[i + j];
                        T y = (F::NIN == 2) ? b[i + j] : x;
                        out[i + j] = f(x, y);
                    }
                }
            }
        }
    }
}

// ---- kernel 1b: flat, one operand periodic ---------------------------------------------------------
// The output and one input are contiguous and of full size; the other input varies along ONE of the
// (collapsed) dims only, where it is contiguous: a bias [1,C,1,1] on [N,C,H,W], a row [1,n] on
// [m,n], a column [m,1] on [m,n].  Flat index i reads y[(i / inner) % mid].  Indices are 32-bit
// (checked at launch).  With a one-input functor there is no x: the output is f(y) spread over the
// other dims (broadcast of a row, a column, a bias).  MODE 0: inner == 1 and mid % VEC == 0, y is read as vectors; MODE 1:
// inner % VEC == 0, one y per vector; MODE 2: inner >= VEC, a vector spans at most two y; MODE 3: inner == 1 and
// any mid, y is read as vectors except where one runs past the end of the period.  (MODE 3 keeps x and the output
// flat and aligned however long the row is: [3001,2047] + [2047] f32 takes 9.9 us (5.0 TB/s), 24.4 us when rows of
// odd length were walked one by one with scalar accesses.)

template <typename T, int VEC, int MEM, typename F, bool Y_FIRST, int MODE, int kBlock, int kUnroll>
__global__ __launch_bounds__(kBlock) void ew_periodic_kernel(T *out, const T *x, const T *y, uint32_t n,
                                                             uint32_t inner, uint32_t mid, F f)
{
    f.init();
    const uint32_t base = blockIdx.x * (uint32_t)(kBlock * VEC * kUnroll);
    auto y_of = [&](uint32_t i0) {
        Pack<T, VEC> yv;
        if constexpr (MODE == 0) {
            yv = load_pack<T, VEC, false>(y + i0 % mid);
        } else if constexpr (MODE == 1) {
            yv = splat<T, VEC>(y[(i0 / inner) % mid]);
        } else if constexpr (MODE == 3) {
            const uint32_t c = i0 % mid;
            if (c + VEC <= mid) {
                yv = load_pack<T, VEC, false>(y + c);
            } else {
                uint32_t cj = c;
#pragma unroll
                for (int j = 0; j < VEC; j++) {
                    yv.v[j] = y[cj];
                    cj = cj + 1 == mid ? 0 : cj + 1;
                }
            }
        } else {
            const uint32_t q0 = i0 / inner, rem = i0 - q0 * inner, c0 = q0 % mid;
            const uint32_t c1 = c0 + 1 == mid ? 0 : c0 + 1;
            const T y0 = y[c0], y1 = y[c1];
#pragma unroll
            for (int j = 0; j < VEC; j++) yv.v[j] = rem + j >= inner ? y1 : y0;
        }
        return yv;
    };
    if (base + (uint32_t)(kBlock * VEC * kUnroll) <= n && base + (uint32_t)(kBlock * VEC * kUnroll) > base) {
        Pack<T, VEC> xv[kUnroll], yv[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint32_t i0 = base + (uint32_t)(u * kBlock + threadIdx.x) * VEC;
            yv[u] = y_of(i0);
            if constexpr (F::NIN == 2) xv[u] = load_pack<T, VEC, streams_loads(MEM)>(x + i0);
            else xv[u] = yv[u];
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint32_t i0 = base + (uint32_t)(u * kBlock + threadIdx.x) * VEC;
            const Pack<T, VEC> r = Y_FIRST ? apply_pack<T, VEC, F>(f, yv[u], xv[u]) : apply_pack<T, VEC, F>(f, xv[u], yv[u]);
            store_mem<T, VEC, MEM, true>(out + i0, r);   // at most one streamed input beside the output
        }
    } else {
        for (int u = 0; u < kUnroll; u++) {
            const uint64_t i0 = (uint64_t)base + (uint64_t)(u * kBlock + threadIdx.x) * VEC;
            for (int j = 0; j < VEC; j++) {
                const uint64_t i = i0 + j;
                if (i < n) {
                    const T ys = y[((uint32_t)i / inner) % mid];
                    const T xs = (F::NIN == 2) ? x[i] : ys;
                    out[i] = Y_FIRST ? f(ys, xs) : f(xs, ys);
                }
            }
        }
    }
}

// ---- shared index descriptor ---------------------------------------------------------------------

struct OuterDesc {
    int nouter;                          // number of outer dims (0..5)
    int64_t shape[kMaxDim];              // outer dims, slowest first
    int64_t stride[kMaxOperands][kMaxDim];
};

__device__ __forceinline__ void decompose(const OuterDesc &d, int64_t lin, int64_t &o0, int64_t &o1,
                                          int64_t &o2)
{
    o0 = o1 = o2 = 0;
    for (int k = d.nouter - 1; k >= 0; k--) {
        int64_t q, r;
        if (k == 0) {                 // the slowest dim takes what is left: no division
            q = 0;
            r = lin;
        } else if (lin < 0x7fffffffLL && d.shape[k] < 0x7fffffffLL) {
            uint32_t l32 = (uint32_t)lin, s32 = (uint32_t)d.shape[k];
            q = l32 / s32;
            r = l32 - (uint32_t)q * s32;
        } else {
            q = lin / d.shape[k];
            r = lin - q * d.shape[k];
        }
        o0 += r * d.stride[0][k];
        o1 += r * d.stride[1][k];
        o2 += r * d.stride[2][k];
        lin = q;
    }
}

// the same for an index that is known to fit 32 bits (then every dim does): no 64-bit division
__device__ __forceinline__ void decompose32(const OuterDesc &d, uint32_t lin, int64_t &o0, int64_t &o1,
                                            int64_t &o2)
{
    o0 = o1 = o2 = 0;
    for (int k = d.nouter - 1; k >= 0; k--) {
        uint32_t q = 0, r = lin;
        if (k != 0) {
            const uint32_t s32 = (uint32_t)d.shape[k];
            q = lin / s32;
            r = lin - q * s32;
        }
        o0 += (int64_t)r * d.stride[0][k];
        o1 += (int64_t)r * d.stride[1][k];
        o2 += (int64_t)r * d.stride[2][k];
        lin = q;
    }
}

// ---- kernel 2: rows (inner dim contiguous or broadcast) -------------------------------------------

struct RowsParams {
    OuterDesc outer;
    int64_t nrows;     // product of outer dims
    int64_t ncols;     // inner length
    int inner_a;       // inner stride of input a: 1 or 0
    int inner_b;       // inner stride of input b: 1 or 0
    int tx_shift;      // threads along the row = 1 << tx_shift (<= 256)
    int64_t col_tiles; // column tiles per row
    int grid2d;        // the grid is (column tiles, row blocks); else linear, column tiles fastest
};

// NTA / NTB: input a / b is streamed once (not broadcast along an outer dim); the output is
// streamed when either is.  Template parameters, because a run-time choice between a hinted and
// a plain load is merged by the compiler into one plain load.
template <typename T, int VEC, bool NTA, bool NTB, typename F, int kBlock, int kUnroll>
__global__ __launch_bounds__(kBlock) void ew_rows_kernel(T *out, const T *a, const T *b,
                                                         RowsParams p, F f)
{
    f.init();
    // The workgroups are short-lived, so the scalar work before the first load counts: every field
    // of the argument block that the common case needs is read here, together (one wait instead of
    // one per branch), and a 2-d grid spares the division of the workgroup index.
    int tx_shift = p.tx_shift, inner_a = p.inner_a, inner_b = p.inner_b, nouter = p.outer.nouter, grid2d = p.grid2d;
    int64_t nrows = p.nrows, ncols = p.ncols;
    int64_t so0 = p.outer.stride[0][0], sa0 = p.outer.stride[1][0], sb0 = p.outer.stride[2][0];
    asm volatile("" : : "s"(tx_shift), "s"(inner_a), "s"(inner_b), "s"(nouter), "s"(grid2d), "s"(nrows),
                      "s"(ncols), "s"(so0), "s"(sa0), "s"(sb0), "s"(out), "s"(a), "s"(b));
    const int tx_n = 1 << tx_shift;
    const int ty_n = kBlock >> tx_shift;
    const int tx = threadIdx.x & (tx_n - 1);
    const int ty = threadIdx.x >> tx_shift;
    uint32_t row_blk32, col_tile32;
    if (grid2d) {
        col_tile32 = blockIdx.x;
        row_blk32 = blockIdx.y;
    } else {
        // grid and col_tiles fit 32 bits (checked at launch)
        row_blk32 = blockIdx.x / (uint32_t)p.col_tiles;
        col_tile32 = blockIdx.x - row_blk32 * (uint32_t)p.col_tiles;
    }
    const int64_t col_tile = col_tile32;
    const int64_t row = (int64_t)row_blk32 * ty_n + ty;
    if (row >= nrows) return;
    int64_t oo, oa, ob;
    if (nouter == 1) {            // one outer dim: the row index is its coordinate
        oo = row * so0;
        oa = row * sa0;
        ob = row * sb0;
    } else {
        decompose(p.outer, row, oo, oa, ob);
    }
    T *orow = out + oo;
    const T *arow = a + oa;
    const T *brow = (F::NIN == 2) ? b + ob : arow;

    const int64_t cols_per_tile = (int64_t)tx_n * VEC * kUnroll;
    const int64_t c0 = col_tile * cols_per_tile;
    Pack<T, VEC> sa, sb;
    if (inner_a == 0) sa = splat<T, VEC>(arow[0]);
    if (F::NIN == 2 && inner_b == 0) sb = splat<T, VEC>(brow[0]);

    if (c0 + cols_per_tile <= ncols) {
        Pack<T, VEC> va[kUnroll], vb[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            int64_t c = c0 + ((int64_t)u * tx_n + tx) * VEC;
            va[u] = inner_a ? load_pack<T, VEC, NTA>(arow + c) : sa;
            if constexpr (F::NIN == 2) vb[u] = inner_b ? load_pack<T, VEC, NTB>(brow + c) : sb;
            else vb[u] = va[u];
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            int64_t c = c0 + ((int64_t)u * tx_n + tx) * VEC;
            const Pack<T, VEC> r = apply_pack<T, VEC, F>(f, va[u], vb[u]);
            if constexpr ((NTA != NTB || (F::NIN == 1 && NTA)) && VEC > 1) store_pack_wt<T, VEC>(orow + c, r);   // one streamed input
            else store_pack<T, VEC, (NTA || NTB)>(orow + c, r);
        }
    } else {
        for (int u = 0; u < kUnroll; u++) {
            int64_t c = c0 + ((int64_t)u * tx_n + tx) * VEC;
            if (c + VEC <= ncols) {
                Pack<T, VEC> x = inner_a ? load_pack<T, VEC, false>(arow + c) : sa;
                Pack<T, VEC> y = x;
                if constexpr (F::NIN == 2) y = inner_b ? load_pack<T, VEC, false>(brow + c) : sb;
                store_pack<T, VEC, false>(orow + c, apply_pack<T, VEC, F>(f, x, y));
            } else {
                for (int j = 0; j < VEC; j++) {
                    if (c + j < ncols) {
                        T x = inner_a ? arow[c + j] : sa.v[0];
                        T y = x;
                        if constexpr (F::NIN == 2) y = inner_b ? brow[c + j] : sb.v[0];
                        orow[c + j] = f(x, y);
                    }
                }
            }
        }
    }
}

// ---- kernel 3: 64x64 tiles with an LDS turn for transposed inputs ----------------------------------

// 64x64 tiles for f32 (16.6 KB of LDS per staged input), 32x32 for f64 (8.4 KB).  With one input
// (a transposed or permuted copy, a unary op on such a view) one thread per 16-byte vector of the
// tile (1024 / 512 threads): ONE vector per thread is the shape that streams one load and one
// store stream fastest here, as for the contiguous kernels.  Transposed copy of [4096,4096] f32 in
// a stand-alone probe, tiles walked along diagonals: 23.9 us, against 25.2 us with 256 threads and
// four vectors each; 32x32 tiles with 256 threads copy as fast (24.1 us) but leave operands that
// are not transposed with 128-byte row pieces.
// SMALL halves the edge (32 / 16): few tiles of a small matrix leave most CUs idle and make each workgroup a
// long chain; with a quarter of the tile per workgroup a transposed copy of [256,512] f32 takes 2.8 us
// against 3.3 us, of [784,512] 3.4 against 3.6 (the MLP step of a 512-wide layer issues eleven of them).
// Operands that stay in the caches take them at every size, see launch_ew.
// Tile shapes: whole tiles, small ones, and small ones with two vectors per thread for copies of up to 96 MB, which wait for
// the loads that are in flight: half the threads per workgroup, twice as many workgroups on a CU, two loads in each
// thread.  us with one vector / two: [1500,1433] f32 5.2 / 4.9, [1500,1000] 4.2 / 4.0, NCHW -> NHWC [64,512,14,14] 9.6 / 9.0,
// [4,166,75,76] 8.7 / 7.1, [40,124,29,30] 9.2 / 7.3, [92,51,22,22] 7.4 / 6.1; f64 [1500,1500] 7.8 / 7.2 (5.0 TB/s), [40,124,29,30]
// 17.2 / 16.1.  Not other functions of one input (sine of a transposed [500,500] 2.7 / 3.1), two inputs (a + b^T
// [3001,2047] 12.6 / 12.9) nor larger copies ([4099,4097] 31 / 33, f64 65 / 71).
enum { kTileWhole, kTileSmall, kTileSmallPairs };
template <typename T, int SMALL = kTileWhole> struct TileOf { static constexpr int N = (sizeof(T) == 4 ? 64 : 32) / (SMALL ? 2 : 1); };
// With two inputs (three streams, a + b^T) two vectors per thread and operand at 512 threads are the
// fastest (stand-alone probe: 36.2 us with four at 256 threads, 35.5 us with two at 512, 35.7 us with
// one at 1024).
template <typename T, typename F, int SMALL = kTileWhole> struct TileThreads {
    static constexpr int kVecs = TileOf<T, SMALL>::N * TileOf<T, SMALL>::N / VecOf<T>::N;   // vectors per tile and operand
    static constexpr int value = SMALL == kTileSmallPairs ? kVecs / 2 : (F::NIN == 1 || kVecs < 512) ? kVecs : 512;
};

enum { kWalkRows = 0, kWalkCols = 1, kWalkDiagonal = 2, kWalkBands = 3 };

struct TileParams {
    OuterDesc outer;      // batch dims (everything except the two tile dims)
    int64_t nbatch;
    int64_t R, C;         // tile dims: R = dim where transposed inputs are contiguous, C = output inner dim
    int64_t ldr[kMaxOperands];  // stride along R per operand
    int64_t ldc[kMaxOperands];  // stride along C per operand (1 for out; 0/1 direct; ld for transposed)
    int trans_a, trans_b;       // input goes through LDS
    int vec_ok;                 // every operand can be read as vectors
    int grid3d;                 // the grid is (tiles_c, tiles_r, nbatch); else linear, tiles_c fastest
    int walk;                   // order of the tiles: kWalkRows, kWalkDiagonal, or (3-d grids only) kWalkCols, kWalkBands
    int64_t tiles_r, tiles_c;
    uint32_t tiles_r_magic;     // min(floor(2^32 / tiles_r), 2^32 - 1): x mod tiles_r from one high multiply and a fix-up
};

template <typename T, int MEM, typename F, int SMALL = kTileWhole>
__global__ __launch_bounds__((TileThreads<T, F, SMALL>::value)) void ew_tile_kernel(T *out, const T *a, const T *b,
                                                                                  TileParams p, F f)
{
    constexpr int VEC = VecOf<T>::N;
    constexpr int kTile = TileOf<T, SMALL>::N;
    constexpr int kBlock = TileThreads<T, F, SMALL>::value;   // shadows the engine-wide 256
    constexpr int kPitch = kTile + 1;
    // Eight lanes cover one 128-byte segment of a tile row; 32 segments per pass.  With eight (not
    // sixteen) lanes along the vector dim the 32 lanes that the LDS serves together -- eight
    // vector positions x four rows -- fall into 32 different banks in the scatter (one element of
    // each lane's vector per instruction, rows one pitch apart) and in the gather alike; sixteen
    // lanes per row alias pairwise (4 m and 4 (m + 8) share a bank) whatever the pitch.
    constexpr int VPS = 8;                  // vectors per segment
    constexpr int SEG = kTile / (VPS * VEC);// segments per tile row (2)
    static_assert(SEG >= 1 && (kTile * SEG * VPS) % kBlock == 0, "tile geometry");
    // One staging tile per TRANSPOSED input, sized at launch: with a static tile per input, `a + b^T`
    // held 33 KB of LDS per workgroup for the one tile it uses, and four workgroups fit a CU instead
    // of eight (on a [4096,4096] f32 view of pitch 4160: 37.6 us against 36.0 us).
    extern __shared__ __align__(16) unsigned char lds_raw[];
    T *const lds_a = reinterpret_cast<T *>(lds_raw);
    f.init();

    // The order in which the tiles are walked decides which addresses the workgroups that run
    // together touch.  Row by row (consecutive workgroups along the output's rows) they read pieces
    // of a transposed input that lie a tile's height times ITS pitch apart; column by column they
    // write pieces (and read those of the other inputs) that far apart by the output's pitch; along
    // diagonals consecutive workgroups differ in both tile coordinates.  A distance that is a
    // multiple of 4 KiB lands on few memory channels, so the host picks the walk by the pitches
    // (transposed copy of 4096 x 4096 f32, pitch of the output / of the input in elements, us row by
    // row / column by column / diagonally: 4096 / 4096: 26.3 / 27.6 / 24.0; 4096 / 4352: 24.1 / 28.5 /
    // 26.7; 4352 / 4096: 26.4 / 24.9 / 28.3; 4352 / 4352: 24.1 / 25.3 / 31.2; 5120 / 5120: 26.6 / 29.4 / 25.8).
    // The grid is (column tiles, row tiles, batch) when that fits the grid limits, so that no
    // workgroup starts with a chain of integer divisions (in 64 bits they were most of this kernel's
    // instructions); otherwise a linear grid below 2^31, decomposed in 32 bits.
    // Every wave of the workgroup runs this scalar prologue, and nothing is in flight before it ends:
    // the fields it needs are read from the argument block together (one wait, not one per branch),
    // and the diagonal's remainder comes from a multiplier that the host prepared, not from a division.
    int grid3d = p.grid3d, vec_ok = p.vec_ok, nouter = p.outer.nouter, walk = p.walk;
    uint32_t ntr = (uint32_t)p.tiles_r, magic = p.tiles_r_magic;
    int64_t R = p.R, C = p.C;
    int64_t ldr0 = p.ldr[0], ldr1 = p.ldr[1], ldr2 = p.ldr[2], ldc1 = p.ldc[1], ldc2 = p.ldc[2];
    int trans_a = p.trans_a, trans_b = p.trans_b;
    asm volatile("" : : "s"(grid3d), "s"(vec_ok), "s"(nouter), "s"(walk), "s"(ntr), "s"(magic), "s"(R), "s"(C),
                      "s"(ldr0), "s"(ldr1), "s"(ldr2), "s"(ldc1), "s"(ldc2), "s"(trans_a), "s"(trans_b),
                      "s"(out), "s"(a), "s"(b));
    T *const lds_b = lds_a + ((F::NIN == 2 && trans_a) ? kTile * kPitch : 0);
    uint32_t tc32, tr32, batch32;
    if (grid3d) {
        const bool by_cols = walk == kWalkCols;       // then the grid is (row tiles, column tiles, batch)
        tc32 = by_cols ? blockIdx.y : blockIdx.x;
        tr32 = by_cols ? blockIdx.x : blockIdx.y;
        batch32 = blockIdx.z;
    } else {
        const uint32_t ntc = (uint32_t)p.tiles_c;
        const uint32_t q = blockIdx.x / ntc;
        tc32 = blockIdx.x - q * ntc;
        batch32 = q / ntr;
        tr32 = q - batch32 * ntr;
    }
    if (walk == kWalkDiagonal) {
        // (tr + tc) mod tiles_r: the multiplier is floor(2^32 / tiles_r) (2^32 - 1 for one tile row),
        // which is less than 1 below 2^32 / tiles_r, so for every 32-bit argument the quotient is
        // exact or one too small (the sum is below 2^32: both grids are)
        const uint32_t x = tr32 + tc32;
        const uint32_t q = __umulhi(x, magic);
        const uint32_t r = x - q * ntr;
        tr32 = r >= ntr ? r - ntr : r;
    }
    if (walk == kWalkBands) {
        // Workgroup i runs on XCD i mod 8; each XCD gets one run of consecutive tiles, row by row.  Where the
        // output's rows do not start at cache lines, neighbouring tiles share the lines at their border, and
        // with the neighbours on one XCD its L2 puts the two halves together.
        const uint32_t gx = gridDim.x, gxy = gx * gridDim.y, total = gxy * gridDim.z;
        const uint32_t wg = batch32 * gxy + tr32 * gx + tc32;
        const uint32_t share = total >> 3, rest = total & 7, xcd = wg & 7;
        uint32_t t = xcd * share + (xcd < rest ? xcd : rest) + (wg >> 3);
        batch32 = t / gxy;
        t -= batch32 * gxy;
        tr32 = t / gx;
        tc32 = t - tr32 * gx;
    }
    const int64_t tc = tc32, tr = tr32;
    int64_t oo = 0, oa = 0, ob = 0;
    if (nouter > 0) decompose32(p.outer, batch32, oo, oa, ob);
    const int64_t r0 = tr * kTile, c0 = tc * kTile;
    const int64_t nr = (R - r0 < kTile) ? R - r0 : kTile;
    const int64_t nc = (C - c0 < kTile) ? C - c0 : kTile;
    const bool full = (nr == kTile) & (nc == kTile);
    const int tid = threadIdx.x;

    T *obase = out + oo + r0 * ldr0 + c0;
    const T *abase = a + oa + r0 * ldr1 + c0 * ldc1;
    const T *bbase = (F::NIN == 2) ? b + ob + r0 * ldr2 + c0 * ldc2 : abase;

    // All global loads of the tile are issued first -- the transposed inputs along R (their
    // contiguous dim), the others along C -- so both streams are in flight together; then the
    // transposed ones are turned through LDS.
    // EDGE: a tile that the matrix ends in.  The vectors that would run past the end are moved back to end with
    // it (two lanes then load, and scatter to LDS, the same elements) and positions past the end of the other
    // dim repeat its last one, so the loads stay vectors without a branch between them; every element is stored
    // by one thread only, the moved-back vectors element by element.  a + b^T of [3001,2047] f32 15.6 us,
    // 19.2 us when operands of odd pitch were accessed element by element; the transposed copies of a [1000,999]
    // head and of [1500,1433] weights 4.6 - 4.9 / 6.6 us, 5.2 - 5.8 / 8.4 us before.
    auto tile_by_vectors = [&](auto edge_c) {
        constexpr bool EDGE = decltype(edge_c)::value;
        // vector e = k * kBlock + tid of the tile: eight consecutive ones form a segment, the segments
        // of one segment column follow each other along the other dim
        constexpr int K = kTile * SEG * VPS / kBlock;   // vectors per thread and operand (1 or 2)
        const int seg_v = (tid % VPS) * VEC;            // vector position inside the segment
        auto other_of = [&](int k) { return ((k * kBlock + tid) / VPS) % kTile; };                  // position along the other dim
        auto vec_of = [&](int k) { return seg_v + (((k * kBlock + tid) / VPS) / kTile) * VPS * VEC; };  // element position along the vector dim
        const bool ta = trans_a != 0;
        const bool tb = (F::NIN == 2) && trans_b != 0;
        // where the vectors of an input, or of the output, start and lie in an edge tile
        auto clip_vec = [&](int v, bool t) { return EDGE ? min(v, (int)(t ? nr : nc) - VEC) : v; };
        auto clip_other = [&](int o, bool t) { return EDGE ? min(o, (int)(t ? nc : nr) - 1) : o; };
        // A transposed input is read along R with its pitch ldc between the vectors, any other along C
        // with its pitch ldr: the same expression with the pitch selected, so the loads of one thread
        // follow each other without a branch between them.  (With a branch per load the compiler put a
        // wait for all earlier loads in front of each one: `a + b^T` 38.9 us instead of 36 us.)
        const int64_t pitch_a = ta ? ldc1 : ldr1;
        const int64_t pitch_b = tb ? ldc2 : ldr2;
        Pack<T, VEC> xa[K], xb[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int o = other_of(k);
            const int lane_v = vec_of(k);
            xa[k] = load_pack<T, VEC, streams_loads(MEM)>(abase + clip_vec(lane_v, ta) + (int64_t)clip_other(o, ta) * pitch_a);
            if constexpr (F::NIN == 2) xb[k] = load_pack<T, VEC, streams_loads(MEM)>(bbase + clip_vec(lane_v, tb) + (int64_t)clip_other(o, tb) * pitch_b);
        }
        if (ta) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const int c = clip_other(other_of(k), true);        // the loaded vector holds rows lane_v.. of column c
                const int lane_v = clip_vec(vec_of(k), true);
#pragma unroll
                for (int j = 0; j < VEC; j++) lds_a[(lane_v + j) * kPitch + c] = xa[k].v[j];
            }
        }
        if constexpr (F::NIN == 2) {
            if (tb) {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int c = clip_other(other_of(k), true);
                    const int lane_v = clip_vec(vec_of(k), true);
#pragma unroll
                    for (int j = 0; j < VEC; j++) lds_b[(lane_v + j) * kPitch + c] = xb[k].v[j];
                }
            }
        }
        __syncthreads();                                 // at least one input is transposed
        if (ta) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const int r = clip_other(other_of(k), false);
                const int lane_v = clip_vec(vec_of(k), false);
#pragma unroll
                for (int j = 0; j < VEC; j++) xa[k].v[j] = lds_a[r * kPitch + lane_v + j];
            }
        }
        if constexpr (F::NIN == 2) {
            if (tb) {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int r = clip_other(other_of(k), false);
                    const int lane_v = clip_vec(vec_of(k), false);
#pragma unroll
                    for (int j = 0; j < VEC; j++) xb[k].v[j] = lds_b[r * kPitch + lane_v + j];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int r = other_of(k);
            const int lane_v = vec_of(k);
            Pack<T, VEC> y = xa[k];
            if constexpr (F::NIN == 2) y = xb[k];
            const Pack<T, VEC> z = apply_pack<T, VEC, F>(f, xa[k], y);
            if constexpr (EDGE) {
                if ((r < nr) & (lane_v < nc)) {
                    T *const orow = obase + (int64_t)r * ldr0;
                    if (lane_v + VEC <= nc) {
                        store_mem<T, VEC, MEM, false>(orow + lane_v, z);
                    } else {
                        const int c = clip_vec(lane_v, false);
#pragma unroll
                        for (int j = 0; j < VEC; j++)
                            if (c + j >= lane_v) orow[c + j] = z.v[j];
                    }
                }
            } else {
                store_mem<T, VEC, MEM, false>(obase + (int64_t)r * ldr0 + lane_v, z);
            }
        }
    };

    if (vec_ok && full) {
        tile_by_vectors(std::false_type());
    } else if (vec_ok && nr >= VEC && nc >= VEC) {
        tile_by_vectors(std::true_type());
    } else {
        // Tiles narrower than a vector, and inputs broadcast along the row: element by element with bounds checks.  All loads of a
        // phase are issued before the first use (an element outside the tile reads the tile's first
        // one again and is dropped): with the loads inside the bounds check the compiler waits for each
        // before it issues the next, and a small matrix made of edge tiles only (the [512,10] weights of a
        // classifier head) took four memory round trips per phase instead of one.
        constexpr int E = kTile * kTile / kBlock;
        const bool ta = trans_a != 0;
        const bool tb = (F::NIN == 2) && trans_b != 0;
        if (ta || tb) {
            T va[E], vb[E];
#pragma unroll
            for (int i = 0; i < E; i++) {
                const int e = tid + i * kBlock;
                const int r = e % kTile, c = e / kTile;
                const bool ok = (r < nr) & (c < nc);
                const int64_t off_r = ok ? r : 0, off_c = ok ? c : 0;
                if (ta) va[i] = abase[off_r + off_c * ldc1];
                if constexpr (F::NIN == 2) {
                    if (tb) vb[i] = bbase[off_r + off_c * ldc2];
                }
            }
#pragma unroll
            for (int i = 0; i < E; i++) {
                const int e = tid + i * kBlock;
                const int r = e % kTile, c = e / kTile;
                if ((r < nr) & (c < nc)) {
                    if (ta) lds_a[r * kPitch + c] = va[i];
                    if constexpr (F::NIN == 2) {
                        if (tb) lds_b[r * kPitch + c] = vb[i];
                    }
                }
            }
            __syncthreads();
        }
        T x[E], y[E];
#pragma unroll
        for (int i = 0; i < E; i++) {
            const int e = tid + i * kBlock;
            const int c = e % kTile, r = e / kTile;
            const bool ok = (r < nr) & (c < nc);
            const int64_t off_r = ok ? r : 0, off_c = ok ? c : 0;
            if (!ta) x[i] = abase[off_r * ldr1 + off_c * ldc1];
            if constexpr (F::NIN == 2) {
                if (!tb) y[i] = bbase[off_r * ldr2 + off_c * ldc2];
            }
        }
#pragma unroll
        for (int i = 0; i < E; i++) {
            const int e = tid + i * kBlock;
            const int c = e % kTile, r = e / kTile;
            if ((r < nr) & (c < nc)) {
                if (ta) x[i] = lds_a[r * kPitch + c];
                if constexpr (F::NIN == 2) {
                    if (tb) y[i] = lds_b[r * kPitch + c];
                } else {
                    y[i] = x[i];
                }
                obase[(int64_t)r * ldr0 + c] = f(x[i], y[i]);
            }
        }
    }
}

// ---- kernel 3b: transposed copies with one short side ------------------------------------------------
// Images with few channels between NCHW and NHWC, the weights of a small head: a [long][short] matrix without gaps on
// one side, `nshort` runs of it `pitch` apart on the other.  Square tiles are mostly padding there (3 of 32 columns) and
// their accesses single elements.  Here a workgroup takes 2^log_run positions of all runs, 16 KB: vectors on both sides,
// turned in LDS, where run s starts at s * lds_pitch: 64 / nshort banks (rounded to whole vectors) from the one before,
// so that the elements of a wavefront's vectors, nshort runs by 64 / nshort positions, lie in different banks.
// THIN_OUT: the side without gaps is the output.
struct ThinParams {
    OuterDesc outer;
    int64_t nlong, pitch;
    int nshort, log_run, lds_pitch;
    uint32_t magic;             // ceil(2^20 / nshort): e / nshort = e * magic >> 20 where e * nshort <= 2^20
};
constexpr int kThinBytes = 16384, kThinVecs = kThinBytes / 16 / kBlock;   // per workgroup; vectors per thread
// us of square tiles / this kernel, into [long][short] and out of it, f32: [128,3,12544] 59 / 7.2 and 53 / 7.4 (39 MB,
// 5.3 TB/s), [64,8,3136] 8.5 / 4.2 and 8.4 / 4.8, [32,16,3136] 5.9 / 4.2 and 5.7 / 4.7, [8,24,12544] 6.1 / 5.1 and 6.1 /
// 5.7; f64: [128,3,12544] 50 / 12.4 (77 MB, 6.2 TB/s), [8,24,12544] 11.4 / 7.2.  From runs of 28 on they are level, whole
// tiles of 32 are faster (f64 [64,32,784] 6.0 / 6.8), and so are tiles of a few thousand positions, where the divisions
// show: [10,4096] 2.2 / 2.6, [14,1497] 2.3 / 2.6.
constexpr int64_t kThinMax = 24, kThinPositions = 8192;

template <typename T, int MEM, bool THIN_OUT>
__global__ __launch_bounds__(kBlock) void ew_thin_kernel(T *out, const T *in, ThinParams p)
{
    constexpr int VEC = VecOf<T>::N, LV = VEC == 4 ? 2 : 1;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    T *const lds = reinterpret_cast<T *>(lds_raw);
    const int tid = threadIdx.x, S = p.nshort, run = 1 << p.log_run, K = p.lds_pitch;
    int64_t oo, oi, unused;
    decompose32(p.outer, blockIdx.y, oo, oi, unused);
    const int64_t p0 = (int64_t)blockIdx.x << p.log_run;
    const int n = p.nlong - p0 < run ? (int)(p.nlong - p0) : run;   // positions of this workgroup
    const int vecs = S << (p.log_run - LV);
    const int flat = n * S;                                         // elements of the side without gaps
    const int64_t gapless = p0 * S;
    auto run_of = [&](int v) { return v >> (p.log_run - LV); };
    auto pos_of = [&](int v) { return (v << LV) & (run - 1); };
    auto spot = [&](int e) {                                        // element e of the side without gaps
        const int at = (int)(((uint32_t)e * p.magic) >> 20);
        return (e - at * S) * K + at;
    };
    Pack<T, VEC> x[kThinVecs];
    if constexpr (THIN_OUT) {
        // a vector past the end of its run is moved back to end with it (nlong >= VEC)
        const T *const src = in + oi + p0;
        const int64_t last = p.nlong - VEC - p0;
#pragma unroll
        for (int k = 0; k < kThinVecs; k++) {
            const int v = k * kBlock + tid;
            if (v < vecs) x[k] = load_pack<T, VEC, streams_loads(MEM)>(src + run_of(v) * p.pitch + (pos_of(v) < last ? pos_of(v) : last));
        }
#pragma unroll
        for (int k = 0; k < kThinVecs; k++) {
            const int v = k * kBlock + tid;
            if (v >= vecs) continue;
            T *const row = lds + run_of(v) * K;
            if (pos_of(v) <= last) {
                store_pack<T, VEC, false>(row + pos_of(v), x[k]);
            } else {
#pragma unroll
                for (int j = 0; j < VEC; j++)
                    if (last + j >= 0) row[(int)last + j] = x[k].v[j];
            }
        }
        __syncthreads();
        T *const dst = out + oo + gapless;
#pragma unroll
        for (int k = 0; k < kThinVecs; k++) {
            const int e = (k * kBlock + tid) * VEC;
            if (e >= flat) continue;
#pragma unroll
            for (int j = 0; j < VEC; j++) x[k].v[j] = lds[spot(e + j < flat ? e + j : e)];
            if (e + VEC <= flat) {
                store_mem<T, VEC, MEM, true>(dst + e, x[k]);
            } else {
#pragma unroll
                for (int j = 0; j < VEC; j++)
                    if (e + j < flat) dst[e + j] = x[k].v[j];
            }
        }
    } else {
        const T *const src = in + oi + gapless;
#pragma unroll
        for (int k = 0; k < kThinVecs; k++) {
            const int e = (k * kBlock + tid) * VEC;
            if (e + VEC <= flat) {
                x[k] = load_pack<T, VEC, streams_loads(MEM)>(src + e);
            } else if (e < flat) {
#pragma unroll
                for (int j = 0; j < VEC; j++) x[k].v[j] = src[e + j < flat ? e + j : e];
            }
        }
#pragma unroll
        for (int k = 0; k < kThinVecs; k++) {
            const int e = (k * kBlock + tid) * VEC;
#pragma unroll
            for (int j = 0; j < VEC; j++)
                if (e + j < flat) lds[spot(e + j)] = x[k].v[j];
        }
        __syncthreads();
        T *const dst = out + oo + p0;
#pragma unroll
        for (int k = 0; k < kThinVecs; k++) {
            const int v = k * kBlock + tid;
            if (v >= vecs || pos_of(v) >= n) continue;
            const Pack<T, VEC> z = load_pack<T, VEC, false>(lds + run_of(v) * K + pos_of(v));
            T *const row = dst + run_of(v) * p.pitch + pos_of(v);
            if (pos_of(v) + VEC <= n) {
                store_mem<T, VEC, MEM, true>(row, z);
            } else {
#pragma unroll
                for (int j = 0; j < VEC; j++)
                    if (pos_of(v) + j < n) row[j] = z.v[j];
            }
        }
    }
}

// ---- kernel 4: strided rows (anything else) ----------------------------------------------------------
// Operands whose innermost (collapsed) dim has any stride: a strided destination (out[:, ::2] = ...),
// gathers (a[:, ::2] + b), views without a unit-stride dim.  The threads of a workgroup form
// (ty rows) x (tx columns) with the columns along the innermost dim, so consecutive lanes touch
// addresses one inner stride apart (as coalesced as the view allows); the outer index is
// decomposed once per thread, not per element, and an element's offset is column * stride.

struct StridedRowsParams {
    OuterDesc outer;
    int64_t nrows, ncols;
    int64_t inner[kMaxOperands];   // stride along the innermost dim per operand (any value)
    int tx_shift;
    int64_t col_tiles;
    int grid2d;        // the grid is (column tiles, row blocks); else linear, column tiles fastest
};

template <typename T, typename F, int kUnroll, bool NT>
__global__ __launch_bounds__(kBlock) void ew_strided_rows_kernel(T *out, const T *a, const T *b,
                                                                 StridedRowsParams p, F f)
{
    f.init();
    // as in the rows kernel: the argument block is read once, at the top, and a 2-d grid spares the division
    int tx_shift = p.tx_shift, nouter = p.outer.nouter, grid2d = p.grid2d;
    int64_t nrows = p.nrows, ncols = p.ncols;
    int64_t so0 = p.outer.stride[0][0], sa0 = p.outer.stride[1][0], sb0 = p.outer.stride[2][0];
    int64_t so = p.inner[0], sa = p.inner[1], sb = p.inner[2];
    asm volatile("" : : "s"(tx_shift), "s"(nouter), "s"(grid2d), "s"(nrows), "s"(ncols), "s"(so0), "s"(sa0),
                      "s"(sb0), "s"(so), "s"(sa), "s"(sb), "s"(out), "s"(a), "s"(b));
    const int tx_n = 1 << tx_shift;
    const int ty_n = kBlock >> tx_shift;
    const int tx = threadIdx.x & (tx_n - 1);
    const int ty = threadIdx.x >> tx_shift;
    uint32_t row_blk32, col_tile32;
    if (grid2d) {
        col_tile32 = blockIdx.x;
        row_blk32 = blockIdx.y;
    } else {
        row_blk32 = blockIdx.x / (uint32_t)p.col_tiles;   // grid and col_tiles fit 32 bits (checked at launch)
        col_tile32 = blockIdx.x - row_blk32 * (uint32_t)p.col_tiles;
    }
    const int64_t col_tile = col_tile32;
    const int64_t row = (int64_t)row_blk32 * ty_n + ty;
    if (row >= nrows) return;
    int64_t oo, oa, ob;
    if (nouter == 1) {
        oo = row * so0;
        oa = row * sa0;
        ob = row * sb0;
    } else {
        decompose(p.outer, row, oo, oa, ob);
    }
    T *orow = out + oo;
    const T *arow = a + oa;
    const T *brow = (F::NIN == 2) ? b + ob : arow;
    const int64_t c0 = col_tile * ((int64_t)tx_n * kUnroll) + tx;
    T x[kUnroll], y[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {          // all loads of the thread first
        // A column past the end reads the last one again (and stores nothing): with the loads under
        // the bounds check the compiler waits for the first before it issues the others.
        const int64_t c = c0 + (int64_t)u * tx_n;
        const int64_t cl = c < ncols ? c : ncols - 1;
        x[u] = load_pack<T, 1, NT>(arow + cl * sa).v[0];
        if constexpr (F::NIN == 2) y[u] = load_pack<T, 1, NT>(brow + cl * sb).v[0];
        else y[u] = x[u];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
        const int64_t c = c0 + (int64_t)u * tx_n;
        if (c < ncols) {
            Pack<T, 1> r;
            r.v[0] = f(x[u], y[u]);
            store_pack<T, 1, NT>(orow + c * so, r);
        }
    }
}

// ---- host dispatch ---------------------------------------------------------------------------------

template <typename T, typename F> int launch_ew(EwProblem &p, F f, hipStream_t stream)
{
    constexpr int VEC = VecOf<T>::N;
    ew_collapse(p);
    if (p.numel == 0) return ZENU_OK;
    if (int rc = ew_check_alias(p, sizeof(T))) return rc;
    T *out = static_cast<T *>(p.ptr[0]);
    const T *a = static_cast<const T *>(p.ptr[1]);
    const T *b = (F::NIN == 2) ? static_cast<const T *>(p.ptr[2]) : a;
    const int nin = F::NIN;
    const int64_t moved = p.numel * (int64_t)sizeof(T) * (nin + 1);
    const bool nt = moved >= kStreamBytes;
    // whether inputs of which `full` have the size of the output stay in the caches, see kMemKeep
    auto keeps = [&](int full) { return p.numel * (int64_t)sizeof(T) * full < kKeepInputs; };
    // calls go(mem) with the way past the caches as a constant; feed: see kMemFeed
    auto with_mem = [&](auto feed, int full, auto go) {
        constexpr bool FEED = decltype(feed)::value;
        if (!nt) go(std::integral_constant<int, kMemCached>());
        else if (FEED ? moved < kFeedBytes : keeps(full)) go(std::integral_constant<int, FEED ? kMemFeed : kMemKeep>());
        else go(std::integral_constant<int, kMemStream>());
    };
    if (p.ndim == 0) {  // a single element
        p.ndim = 1;
        p.shape[0] = 1;
        for (int o = 0; o < p.nops; o++) p.stride[o][0] = 1;
    }
    const int last = p.ndim - 1;

    // contig
    bool all_unit = p.ndim == 1;
    for (int o = 0; o <= nin && all_unit; o++)
        if (p.stride[o][0] != 1) all_unit = false;
    if (all_unit) {
        const int64_t n = p.numel;
        constexpr int cb = ContigShape<F>::kBlock, cu = ContigShape<F>::kUnroll;
        if constexpr (kSinglesPerCu<F> > 0) {
            if (n <= kSinglesPerCu<F> * device_info().num_cus) {
                constexpr int64_t singles = (int64_t)cb * cu;
                ew_contig_kernel<T, 1, kMemCached, F><<<(unsigned)((n + singles - 1) / singles), cb, 0, stream>>>(out, a, b, n, f);
                ZENU_LAUNCH_CHECK();
                return ZENU_OK;
            }
        }
        int64_t tile = (int64_t)cb * VEC * cu;
        int64_t grid = (n + tile - 1) / tile;
        if (grid > 0x7fffffffLL) return ZENU_ERR_UNSUPPORTED;
        with_mem(std::integral_constant<bool, IsLayerStep<F>::value>(), nin, [&](auto mem) {
            ew_contig_kernel<T, VEC, decltype(mem)::value, F><<<(unsigned)grid, cb, 0, stream>>>(out, a, b, n, f);
        });
        ZENU_LAUNCH_CHECK();
        return ZENU_OK;
    }

    // flat with one periodic operand (bias over channels, a row or a column over a matrix)
    {
        if (p.numel < ((int64_t)1 << 32) - 65536) {
            auto flat = [&](int o) {
                int64_t want = 1;
                for (int d = p.ndim - 1; d >= 0; d--) {
                    if (p.stride[o][d] != want) return false;
                    want *= p.shape[d];
                }
                return true;
            };
            auto period_dim = [&](int o) {   // the one dim along which operand o varies (stride 1), else -1
                int m = -1;
                for (int d = 0; d < p.ndim; d++) {
                    if (p.stride[o][d] == 0) continue;
                    if (p.stride[o][d] != 1 || m >= 0) return -1;
                    m = d;
                }
                return m;
            };
            int yo = 0, m = -1;
            if (nin == 1) {
                if (flat(0) && !flat(1) && (m = period_dim(1)) >= 0) yo = 1;
            } else if (flat(0) && flat(1) && (m = period_dim(2)) >= 0) yo = 2;
            else if (flat(0) && flat(2) && (m = period_dim(1)) >= 0) yo = 1;
            if (yo) {
                const T *x = yo == 2 ? a : b, *y = yo == 2 ? b : a;   // one input: x == y == a, x is not read
                int64_t inner = 1;
                for (int d = m + 1; d < p.ndim; d++) inner *= p.shape[d];
                const int64_t mid = p.shape[m];
                // (one input with a period shorter than a vector: the rows path, [10000,3] f32 2.4 us against 3.2)
                const int mode = inner == 1 ? (mid % VEC == 0 ? 0 : F::NIN == 1 && mid < VEC ? -1 : 3)
                                 : inner % VEC == 0 ? 1 : inner >= VEC ? 2 : -1;
                if (mode >= 0) {
                    // one load and one store stream: the small workgroup shape of the unary ops when y comes as
                    // vectors (22.4 against 23.5 us on [4096,4096] + [1,4096]); with the index divisions of
                    // the other modes the larger shape is the better one (16.4 against 17.0 us on a
                    // [64,256,28,28] bias add)
                    const uint32_t n32 = (uint32_t)p.numel, in32 = (uint32_t)inner, mid32 = (uint32_t)mid;
                    auto go = [&](auto yfirst_c, auto mode_c) {
                        constexpr bool YF = decltype(yfirst_c)::value;
                        constexpr int MODE = decltype(mode_c)::value;
                        // a lone store stream (one-input functor) keeps the larger shape, like the fill kernel
                        constexpr bool small = (MODE == 0 || MODE == 3) && !IsValuBound<F>::value && F::NIN == 2;
                        constexpr int B = small ? ZENU_EW1_BLOCK : 256, U = small ? ZENU_EW1_UNROLL : 2;
                        const int64_t tile = (int64_t)B * VEC * U;
                        const unsigned grid = (unsigned)((p.numel + tile - 1) / tile);
                        with_mem(std::integral_constant<bool, IsAdd<F>::value && (MODE == 1 || MODE == 2)>(), nin - 1, [&](auto mem) {
                            ew_periodic_kernel<T, VEC, decltype(mem)::value, F, YF, MODE, B, U><<<grid, B, 0, stream>>>(out, x, y, n32, in32, mid32, f);
                        });
                    };
                    auto by_mode = [&](auto yfirst_c) {
                        if (mode == 0) go(yfirst_c, std::integral_constant<int, 0>());
                        else if (mode == 1) go(yfirst_c, std::integral_constant<int, 1>());
                        else if (mode == 2) go(yfirst_c, std::integral_constant<int, 2>());
                        else go(yfirst_c, std::integral_constant<int, 3>());
                    };
                    if (yo == 1) by_mode(std::true_type());
                    else by_mode(std::false_type());
                    ZENU_LAUNCH_CHECK();
                    return ZENU_OK;
                }
            }
        }
    }

    const bool out_inner_unit = p.stride[0][last] == 1;
    bool inner_01 = out_inner_unit;
    for (int o = 1; o <= nin && inner_01; o++)
        if (p.stride[o][last] != 0 && p.stride[o][last] != 1) inner_01 = false;

    if (inner_01) {
        RowsParams rp;
        rp.outer.nouter = p.ndim - 1;
        for (int d = 0; d < kMaxDim; d++) {
            rp.outer.shape[d] = d < p.ndim - 1 ? p.shape[d] : 1;
            for (int o = 0; o < kMaxOperands; o++)
                rp.outer.stride[o][d] = (d < p.ndim - 1 && o < p.nops) ? p.stride[o][d] : 0;
        }
        rp.ncols = p.shape[last];
        rp.nrows = p.numel / rp.ncols;
        rp.inner_a = (int)p.stride[1][last];
        rp.inner_b = nin == 2 ? (int)p.stride[2][last] : 1;
        bool nta = nt && rp.inner_a == 1, ntb = nt && nin == 2 && rp.inner_b == 1;
        for (int d = 0; d < p.ndim - 1; d++) {
            if (p.stride[1][d] == 0) nta = false;   // re-read for every outer index: keep it cached
            if (nin == 2 && p.stride[2][d] == 0) ntb = false;
        }
        // Vectors whatever the alignment; a short row that is no whole number of vectors leaves a lane with up to
        // VEC - 1 single elements one after the other, so it takes one element per lane.
        const bool vec = rp.ncols % VEC == 0 || rp.ncols >= 4 * VEC;
        const int v = vec ? VEC : 1;
        const int64_t vcols = (rp.ncols + v - 1) / v;
        // full-size streams of this launch: the output plus every input that is neither a scalar
        // per row nor re-read for every outer index; exactly two of them (one load, one store per
        // element) take the small workgroup shape.  A lone store stream (broadcast of a row) does
        // not: measured 13.0 us at 256 threads x 2 vectors against 18.7 us at 64 x 1 for 64 MiB
        int streams = 1;
        for (int o = 1; o <= nin; o++) {
            bool full = p.stride[o][last] == 1;
            for (int d = 0; d < p.ndim - 1; d++)
                if (p.stride[o][d] == 0 && p.shape[d] > 1) full = false;
            if (full) streams++;
        }
        const bool small = streams == 2 && !IsValuBound<F>::value;
        auto launch = [&](auto block_c, auto unroll_c) -> int {
            constexpr int B = decltype(block_c)::value, U = decltype(unroll_c)::value;
            int shift = 0;
            while ((1 << shift) < B && ((int64_t)1 << shift) < vcols) shift++;
            rp.tx_shift = shift;
            int64_t cols_per_tile = ((int64_t)1 << shift) * v * U;
            rp.col_tiles = (rp.ncols + cols_per_tile - 1) / cols_per_tile;
            int64_t rows_per_blk = B >> shift;
            const int64_t row_blks = (rp.nrows + rows_per_blk - 1) / rows_per_blk;
            if (row_blks * rp.col_tiles > 0x7fffffffLL) return ZENU_ERR_UNSUPPORTED;
            rp.grid2d = row_blks <= 65535 ? 1 : 0;
            const dim3 grid = rp.grid2d ? dim3((unsigned)rp.col_tiles, (unsigned)row_blks) : dim3((unsigned)(row_blks * rp.col_tiles));
            if (!vec)            ew_rows_kernel<T, 1, false, false, F, B, U><<<grid, B, 0, stream>>>(out, a, b, rp, f);
            else if (nta && ntb) ew_rows_kernel<T, VEC, true, true, F, B, U><<<grid, B, 0, stream>>>(out, a, b, rp, f);
            else if (nta)        ew_rows_kernel<T, VEC, true, false, F, B, U><<<grid, B, 0, stream>>>(out, a, b, rp, f);
            else if (ntb)        ew_rows_kernel<T, VEC, false, true, F, B, U><<<grid, B, 0, stream>>>(out, a, b, rp, f);
            else                 ew_rows_kernel<T, VEC, false, false, F, B, U><<<grid, B, 0, stream>>>(out, a, b, rp, f);
            return ZENU_OK;
        };
        int rc = small ? launch(std::integral_constant<int, ZENU_EW1_BLOCK>(), std::integral_constant<int, ZENU_EW1_UNROLL>())
                       : launch(std::integral_constant<int, kBlock>(), std::integral_constant<int, kUnroll>());
        if (rc) return rc;
        ZENU_LAUNCH_CHECK();
        return ZENU_OK;
    }

    // tile: every input is either inner-{0,1} or unit-stride along one common other dim `ri`
    if (out_inner_unit && p.ndim >= 2) {
        int ri = -1;
        bool ok = true;
        int trans[kMaxOperands] = {0, 0, 0};
        for (int o = 1; o <= nin && ok; o++) {
            int64_t s = p.stride[o][last];
            if (s == 0 || s == 1) continue;
            int found = -1;
            for (int d = 0; d < last; d++)
                if (p.stride[o][d] == 1) { found = d; break; }
            if (found < 0 || (ri >= 0 && ri != found)) ok = false;
            else { ri = found; trans[o] = 1; }
        }
        if (ok && ri >= 0) {
            TileParams tp;
            int k = 0;
            for (int d = 0; d < kMaxDim; d++) {
                tp.outer.shape[d] = 1;
                for (int o = 0; o < kMaxOperands; o++) tp.outer.stride[o][d] = 0;
            }
            for (int d = 0; d < last; d++) {
                if (d == ri) continue;
                tp.outer.shape[k] = p.shape[d];
                for (int o = 0; o < p.nops; o++) tp.outer.stride[o][k] = p.stride[o][d];
                k++;
            }
            tp.outer.nouter = k;
            tp.R = p.shape[ri];
            tp.C = p.shape[last];
            tp.nbatch = p.numel / (tp.R * tp.C);
            for (int o = 0; o < kMaxOperands; o++) {
                tp.ldr[o] = o < p.nops ? p.stride[o][ri] : 0;
                tp.ldc[o] = o < p.nops ? p.stride[o][last] : 0;
            }
            tp.trans_a = trans[1];
            tp.trans_b = nin == 2 ? trans[2] : 0;
            // a short side, the output's rows or the input's: see ew_thin_kernel
            if constexpr (IsCopy<F>::value) {
                const bool thin_out = tp.C <= kThinMax && tp.ldr[0] == tp.C && tp.R >= 64;
                const bool thin_in = tp.R <= kThinMax && tp.ldc[1] == tp.R && tp.C >= 64;
                if ((thin_out || thin_in) && tp.nbatch <= 65535 && tp.nbatch * (thin_out ? tp.R : tp.C) > kThinPositions) {
                    ThinParams q;
                    q.outer = tp.outer;
                    q.nlong = thin_out ? tp.R : tp.C;
                    q.pitch = thin_out ? tp.ldc[1] : tp.ldr[0];
                    q.nshort = (int)(thin_out ? tp.C : tp.R);
                    q.magic = ((1u << 20) + (uint32_t)q.nshort - 1) / (uint32_t)q.nshort;
                    // positions per workgroup: what fills its 16 KB, less where the chip would stay empty
                    q.log_run = 6;
                    while ((int64_t)q.nshort * (int64_t)sizeof(T) << (q.log_run + 1) <= kThinBytes) q.log_run++;
                    while (q.log_run > 6 && tp.nbatch * ((q.nlong + ((int64_t)1 << q.log_run) - 1) >> q.log_run) < 4 * (int64_t)device_info().num_cus) q.log_run--;
                    const int64_t tiles = (q.nlong + ((int64_t)1 << q.log_run) - 1) >> q.log_run;
                    q.lds_pitch = (1 << q.log_run) + ((64 / q.nshort + 3) & ~3);
                    if (tiles <= 0x7fffffffLL) {
                        const dim3 g((unsigned)tiles, (unsigned)tp.nbatch);
                        const size_t lds = (size_t)q.nshort * q.lds_pitch * sizeof(T);
                        with_mem(std::false_type(), 1, [&](auto mem) {
                            if (thin_out) ew_thin_kernel<T, decltype(mem)::value, true><<<g, kBlock, lds, stream>>>(out, a, q);
                            else          ew_thin_kernel<T, decltype(mem)::value, false><<<g, kBlock, lds, stream>>>(out, a, q);
                        });
                        ZENU_LAUNCH_CHECK();
                        return ZENU_OK;
                    }
                }
            }
            bool vec = true;
            // the vector path reads whole vectors along C from the inputs that are not transposed: one
            // that is broadcast along C (a column beside a transposed operand) takes the element path
            for (int o = 1; o <= nin; o++)
                if (!trans[o] && tp.ldc[o] == 0) vec = false;
            tp.vec_ok = vec ? 1 : 0;
            // Rows of the output that do not start at 128-byte lines: every border between two column tiles
            // is a line that both write in part.  Streaming accesses then cost a second transfer of that line
            // and are not used; small tiles in one band per XCD are the fastest (us of the four combinations
            // of tile edge 64 / 32 and walk rows / bands, without the hint, and of 64 / rows with it): a + b^T
            // [3001,2047] f32 20.9 / 17.7 / 21.7 / 16.8, 21.7; [4099,4097] 53.8 / 47.4 / 60.2 / 46.3, 64.0;
            // transposed copy [1500,1433] 6.2 / 5.9 / 6.1 / 4.8, 7.6.
            bool rows_split_lines = reinterpret_cast<uintptr_t>(out) % 128 != 0;
            for (int d = 0; d < last; d++)
                if (p.stride[0][d] * (int64_t)sizeof(T) % 128) rows_split_lines = true;
            // Otherwise: two inputs stream from kStreamBytes on, as the other kernels do; one input (us with the
            // small tiles and no hint / large tiles and hint: NCHW -> NHWC of [64,512,14,14] f32, 51 MB,
            // 10.5 / 13.7; transposed [2048,2048], 34 MB, 6.0 / 8.2; [4096,4096], 134 MB, 27.4 / 23.9) from three
            // times that.  The large tiles' longer row pieces pay only when streaming, with enough tiles and
            // little padding ([64,256,28,28] NCHW -> NHWC, 784 = 12.25 tiles: 19.2 small, 21.4 large).
            const int64_t bytes = p.numel * (int64_t)sizeof(T) * (nin + 1);
            const bool stream_tiles = nt && !rows_split_lines && (nin == 2 || bytes >= 3 * kStreamBytes);
            constexpr int kFullTile = TileOf<T>::N;
            const int64_t full_tiles = tp.nbatch * ((tp.R + kFullTile - 1) / kFullTile) * ((tp.C + kFullTile - 1) / kFullTile);
            const bool large = stream_tiles && full_tiles >= 2 * (int64_t)device_info().num_cus &&
                               full_tiles * (kFullTile * kFullTile) <= p.numel + p.numel / 25;
            auto launch_tiles = [&](auto small_c, auto nt_c) -> int {
                constexpr int SMALL = decltype(small_c)::value;
                constexpr bool NT = decltype(nt_c)::value;
                constexpr int kTile = TileOf<T, SMALL>::N;
                tp.tiles_r = (tp.R + kTile - 1) / kTile;
                tp.tiles_c = (tp.C + kTile - 1) / kTile;
                {
                    const uint64_t m = (1ull << 32) / (uint64_t)tp.tiles_r;
                    tp.tiles_r_magic = m > 0xffffffffull ? 0xffffffffu : (uint32_t)m;
                }
                int64_t grid = tp.nbatch * tp.tiles_r * tp.tiles_c;
                if (grid > 0x7fffffffLL) return ZENU_ERR_UNSUPPORTED;
                tp.grid3d = (tp.tiles_r <= 65535 && tp.nbatch <= 65535) ? 1 : 0;
                // Row by row unless a transposed input's pitch is within one row piece of a multiple of
                // 4 KiB; then column by column if no other operand's pitch is, else along diagonals.
                auto near_4k = [](int64_t elems) {
                    const int64_t r = ((elems < 0 ? -elems : elems) * (int64_t)sizeof(T)) % 4096;
                    return (r < 4096 - r ? r : 4096 - r) < kTile * (int64_t)sizeof(T);
                };
                bool trans_near = false, direct_near = near_4k(tp.ldr[0]);
                for (int o = 1; o <= nin; o++) {
                    if (trans[o]) trans_near = trans_near || near_4k(tp.ldc[o]);
                    else if (tp.ldc[o] == 1) direct_near = direct_near || near_4k(tp.ldr[o]);
                }
                tp.walk = (rows_split_lines && tp.grid3d && tp.tiles_c > 1) ? kWalkBands
                          : !trans_near                                     ? kWalkRows
                          : (!direct_near && tp.grid3d && tp.tiles_c <= 65535) ? kWalkCols : kWalkDiagonal;
                const bool by_cols = tp.walk == kWalkCols;
                const dim3 g = !tp.grid3d ? dim3((unsigned)grid)
                               : by_cols ? dim3((unsigned)tp.tiles_r, (unsigned)tp.tiles_c, (unsigned)tp.nbatch)
                                         : dim3((unsigned)tp.tiles_c, (unsigned)tp.tiles_r, (unsigned)tp.nbatch);
                const size_t lds = (size_t)(tp.trans_a + tp.trans_b) * kTile * (kTile + 1) * sizeof(T);
                constexpr int kThreads = TileThreads<T, F, SMALL>::value;
                if constexpr (!NT) ew_tile_kernel<T, kMemCached, F, SMALL><<<g, kThreads, lds, stream>>>(out, a, b, tp, f);
                else if (keeps(nin)) ew_tile_kernel<T, kMemKeep, F, SMALL><<<g, kThreads, lds, stream>>>(out, a, b, tp, f);
                else ew_tile_kernel<T, kMemStream, F, SMALL><<<g, kThreads, lds, stream>>>(out, a, b, tp, f);
                return ZENU_OK;
            };
            typedef std::integral_constant<int, kTileWhole> Whole;
            typedef std::integral_constant<int, kTileSmall> Small;
            // (copies have the pairs in place of the small tiles without the hint, but for those that are too large)
            const bool pairs = IsCopy<F>::value && bytes < 3 * kStreamBytes;
            const int rc_tiles = large          ? launch_tiles(Whole(), std::true_type())
                                 : stream_tiles ? launch_tiles(Small(), std::true_type())
                                 : pairs        ? launch_tiles(std::integral_constant<int, IsCopy<F>::value ? kTileSmallPairs : kTileSmall>(), std::false_type())
                                                : launch_tiles(Small(), std::false_type());
            if (rc_tiles) return rc_tiles;
            ZENU_LAUNCH_CHECK();
            return ZENU_OK;
        }
    }

    // strided rows: rows = everything but the innermost dim
    StridedRowsParams sp;
    sp.outer.nouter = p.ndim - 1;
    for (int d = 0; d < kMaxDim; d++) {
        sp.outer.shape[d] = d < p.ndim - 1 ? p.shape[d] : 1;
        for (int o = 0; o < kMaxOperands; o++)
            sp.outer.stride[o][d] = (d < p.ndim - 1 && o < p.nops) ? p.stride[o][d] : 0;
    }
    sp.ncols = p.shape[last];
    sp.nrows = p.numel / sp.ncols;
    for (int o = 0; o < kMaxOperands; o++) sp.inner[o] = o < p.nops ? p.stride[o][last] : 0;
    constexpr int kStridedUnroll = 4;
    int shift = 0;
    while ((1 << shift) < kBlock && ((int64_t)1 << shift) < sp.ncols) shift++;
    sp.tx_shift = shift;
    const int64_t cols_per_tile = ((int64_t)1 << shift) * kStridedUnroll;
    sp.col_tiles = (sp.ncols + cols_per_tile - 1) / cols_per_tile;
    const int64_t rows_per_blk = kBlock >> shift;
    const int64_t row_blks = (sp.nrows + rows_per_blk - 1) / rows_per_blk;
    if (row_blks * sp.col_tiles > 0x7fffffffLL || sp.col_tiles > 0x7fffffffLL) return ZENU_ERR_UNSUPPORTED;
    sp.grid2d = row_blks <= 65535 ? 1 : 0;
    const dim3 grid = sp.grid2d ? dim3((unsigned)sp.col_tiles, (unsigned)row_blks) : dim3((unsigned)(row_blks * sp.col_tiles));
    // streaming hint only when every cache line an access touches is used up by the same wavefront
    // (small inner strides); with large strides the neighbours of an element belong to other rows
    bool snt = nt;
    for (int o = 0; o <= nin; o++)
        if (sp.inner[o] > 4) snt = false;
    if (snt) ew_strided_rows_kernel<T, F, kStridedUnroll, true><<<grid, kBlock, 0, stream>>>(out, a, b, sp, f);
    else     ew_strided_rows_kernel<T, F, kStridedUnroll, false><<<grid, kBlock, 0, stream>>>(out, a, b, sp, f);
    ZENU_LAUNCH_CHECK();
    return ZENU_OK;
}

// problem builders -----------------------------------------------------------------------------------

void init_problem(EwProblem &p, const zenu_tensor_t &to, int nops)
{
    p.nops = nops;
    p.ndim = to.ndim;
    for (int d = 0; d < to.ndim; d++) p.shape[d] = to.shape[d];
    for (int d = to.ndim; d < kMaxDim; d++) p.shape[d] = 1;
    for (int o = 0; o < kMaxOperands; o++) {
        p.ptr[o] = nullptr;
        for (int d = 0; d < kMaxDim; d++) p.stride[o][d] = 0;
    }
    ew_set_operand(p, 0, to, to.ndim, to.shape);
    // the output is never broadcast: keep its own strides even on size-1 dims
    for (int d = 0; d < to.ndim; d++) p.stride[0][d] = to.stride[d];
}

template <typename T, typename F>
int run1(const zenu_tensor_t &to, const zenu_tensor_t &in, F f, hipStream_t s)
{
    EwProblem p;
    init_problem(p, to, 2);
    ew_set_operand(p, 1, in, to.ndim, to.shape);
    return launch_ew<T, F>(p, f, s);
}

template <typename T, typename F>
int run2(const zenu_tensor_t &to, const zenu_tensor_t &x, const zenu_tensor_t &y, F f, hipStream_t s)
{
    EwProblem p;
    init_problem(p, to, 3);
    ew_set_operand(p, 1, x, to.ndim, to.shape);
    ew_set_operand(p, 2, y, to.ndim, to.shape);
    return launch_ew<T, F>(p, f, s);
}

int check2(const zenu_tensor_t *a, const zenu_tensor_t *b)
{
    int rc = validate_tensor(a);
    if (rc) return rc;
    return validate_tensor(b);
}

}  // namespace
}  // namespace zenu
