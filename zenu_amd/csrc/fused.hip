// fused.hip -- single-launch forms of the op chains ZeNu issues around a classifier head:
//   softmax_assign                  zenu-matrix/src/operation/softmax.rs:10-25
//                                   (x - max_axis(keep) ; exp ; sum(axis, keep) ; /= ; copy_from)
//   SoftMax::backward               zenu-autograd/src/loss/softmax.rs:33-40
//                                   (gx = y*gy ; sum(gx, axis, keep) ; gx - y*sum)
//   cross_entropy (+ its backward)  zenu-autograd/src/loss/cross_entropy.rs:12-23
//                                   (softmax(pred,1) ; log ; * ans ; sum_to([]) ; / -N)
//   Linear bias add + ReLU          zenu-layer/src/layers/linear.rs:27-31, zenu-autograd/src/activation/relu.rs:24-33
//
// Every element goes through the same sequence of individually rounded operations as in the
// chain (no contraction; f32 exp/log are the host libm's algorithm, zmath.hpp), so the fused results differ
// from the chain only where the chain itself is order dependent: the sums.  The "lines" kernels
// (one thread per softmax line) add in index order, exactly like sum.rs:20-25; the
// workgroup-per-row kernels add in a fixed tree.
//
// Geometry: operands are row-major [outer, R, inner] with the softmax axis R in the middle;
// views that are not in default stride are staged through a contiguous temporary.
#include <type_traits>
#include <math.h>

#include "common.hpp"
#include "vecmem.hpp"
#include "zmath.hpp"

namespace zenu {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kWholePacks = 4;  // vectors per thread of softmax_whole_rows_kernel
constexpr int kLineMaxR = 64;   // rows up to this length: a lane per row, on one or several wavefronts

// ---- workgroup reductions in a fixed order ------------------------------------------------------------

template <typename T, bool MAX> __device__ __forceinline__ T combine(T a, T b)
{
    if (MAX) return b > a ? b : a;   // a NaN never replaces (max.rs:27)
    return a + b;
}

template <typename T, bool MAX, int BLOCK = kBlock> __device__ __forceinline__ T block_red(T v, T *lds)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = combine<T, MAX>(v, __shfl_xor(v, o));
    if (BLOCK == 64) return v;   // one wavefront: every lane already holds the result
    __syncthreads();   // lds may still be read from the previous reduction
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    T r = lds[0];
#pragma unroll
    for (int w = 1; w < BLOCK / 64; w++) r = combine<T, MAX>(r, lds[w]);
    return r;
}

// ---- forward ---------------------------------------------------------------------------------------------
// CE: additionally rowloss[line] = sum_r target * log(softmax)   (inner == 1 only)

constexpr int kLineRegs = 16;   // classes of the one-workgroup classifier head kernels below
constexpr int kLineWaves = 16;  // wavefronts that can share the lines of a workgroup

// Every quotient of a softmax line has the same divisor.  With r = RN(1 / sum): q0 = RN(a r), the
// exact remainder a - sum q0 (one fma) and q = fma(remainder, r, q0) is the correctly rounded
// a / sum (Markstein) unless the divisor's mantissa is all ones, as long as nothing underflows:
// three instructions per element instead of the division's eleven.  A thread takes that road
// when its terms are zero (the quotient is, too) or at least 2^-64 and the sum lies in [1, 2^23) (quotient
// and remainder stay normal); otherwise it divides.  On 9.6e9 random pairs from those ranges (terms down to
// 2^-80) the host finds no quotient that differs from the division's.  f32 only.
// least: the smallest of the thread's terms above zero, as its bits less one (all ones before the first)
template <typename T> __device__ __forceinline__ uint32_t least_term(uint32_t least, T a)
{
    if constexpr (sizeof(T) == 4) return min(least, __float_as_uint(a) - 1u);
    return least;
}
template <typename T> __device__ __forceinline__ bool divides_by_reciprocal(uint32_t least, T sum)
{
    if constexpr (sizeof(T) == 4)
        return least >= __float_as_uint(0x1p-64f) - 1u && sum >= (T)1 && sum < (T)0x1p23f &&
               (__float_as_uint(sum) & 0x7fffffu) != 0x7fffffu;
    return false;
}
template <typename T> __device__ __forceinline__ T quotient(T a, T sum, T rcp)
{
    if constexpr (sizeof(T) == 4) {
        const float q0 = a * rcp;
        return __builtin_fmaf(__builtin_fmaf(-sum, q0, a), rcp, q0);
    }
    return a / sum;
}

// Where a wavefront of the two lines kernels stands: a workgroup has `waves` wavefronts along R for every 64
// lines, wavefront w of them holds elements [w OWN, (w + 1) OWN) of each of its lines in registers.
struct LineSpot {
    int64_t line, base;   // base: offset of the line's element 0 (of line 0 past the end)
    int64_t first;        // the workgroup's first line
    int w, group, lines_here;
    bool active;
    __device__ __forceinline__ LineSpot(int64_t lines, int64_t R, int64_t inner, int waves)
    {
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        group = wave / waves;
        w = wave - group * waves;
        const int groups = (int)(blockDim.x >> 6) / waves;
        first = (int64_t)blockIdx.x * groups * 64;
        lines_here = (int)min((int64_t)groups * 64, lines - first);
        line = first + group * 64 + (threadIdx.x & 63);
        active = line < lines;
        const int64_t l = active ? line : 0;
        if (inner == 1) {
            base = l * R;
        } else {
            const int64_t q = l / inner;
            base = q * R * inner + (l - q * inner);
        }
    }
};

// `x[i]`, i = 0 .. valid - 1, added to a running sum in index order over the wavefronts of a line: each takes the
// sum over from the one before it.  carry: one value per line of the workgroup.  Every thread calls it.
template <typename T, int OWN>
__device__ __forceinline__ T sum_in_order(const T (&x)[OWN], int valid, const LineSpot &at, int waves, T *carry)
{
    T *const mine = carry + at.group * 64 + (threadIdx.x & 63);
    T sum = (T)0;
    for (int turn = 0; turn < waves; turn++) {
        if (at.w == turn) {
            if (turn) sum = *mine;
#pragma unroll
            for (int i = 0; i < OWN; i++)
                if (i < valid) sum = sum + x[i];
            if (waves > 1) *mine = sum;
        }
        if (waves > 1) __syncthreads();
    }
    return waves > 1 ? *mine : sum;
}

// Rows of the last axis with a lane per row: a wavefront's accesses would lie a row apart, 64 lines of the cache for 4
// or 8 bytes each.  The rows of a workgroup are one piece of memory: it is read and written in vectors, OWN elements
// per thread, and turned in LDS, where rows start an odd number of elements apart.
template <typename T, int OWN> struct StagedRows {
    static constexpr int VEC = VecOf<T>::N;
    Pack<T, VEC> x[OWN / VEC];
    int n, even;
    uint32_t magic;     // ceil(2^20 / R), as n R <= 2^20: 256 rows of 64 elements
    static __host__ __device__ __forceinline__ int pitch(int R) { return R | 1; }
    __device__ __forceinline__ StagedRows(int rows, int R) : n(rows * R), even(~R & 1), magic(((1u << 20) + R - 1) / R) {}
    __device__ __forceinline__ int first(int k) const { return (k * (int)blockDim.x + (int)threadIdx.x) * VEC; }
    __device__ __forceinline__ int spot(int e) const { return even ? e + (int)(((uint32_t)e * magic) >> 20) : e; }
    __device__ __forceinline__ void load(const T *p)
    {
#pragma unroll
        for (int k = 0; k < OWN / VEC; k++) {
            const int e = first(k);
            if (e + VEC <= n) {
                x[k] = load_pack<T, VEC, false>(p + e);
            } else if (e < n) {
#pragma unroll
                for (int j = 0; j < VEC; j++) x[k].v[j] = p[e + j < n ? e + j : e];
            }
        }
    }
    __device__ __forceinline__ void put(T *lds) const
    {
#pragma unroll
        for (int k = 0; k < OWN / VEC; k++) {
            const int e = first(k);
#pragma unroll
            for (int j = 0; j < VEC; j++)
                if (e + j < n) lds[spot(e + j)] = x[k].v[j];
        }
    }
    __device__ __forceinline__ void store(T *p, const T *lds)
    {
#pragma unroll
        for (int k = 0; k < OWN / VEC; k++) {
            const int e = first(k);
            if (e >= n) continue;
#pragma unroll
            for (int j = 0; j < VEC; j++) x[k].v[j] = lds[spot(e + j < n ? e + j : e)];
            if (e + VEC <= n) {
                store_pack_through<T, VEC>(p + e, x[k]);
            } else {
#pragma unroll
                for (int j = 0; j < VEC; j++)
                    if (e + j < n) p[e + j] = x[k].v[j];
            }
        }
    }
};
extern __shared__ __align__(16) unsigned char staged_raw[];

// The softmax axis is not the last one, or is short: a lane per line, and as many wavefronts along the line as it
// takes to hold it in registers, so that it is read and written once with all its loads in flight together.  The
// sums run over the line in index order exactly as sum.rs:20-25 adds (they are handed from wavefront to wavefront).
// Bound by the passes over memory and the f64 arithmetic of the exact exp between them: [16,21,16384] f32 (22 MB each way,
// cached) 12.5 us, 26.1 when one thread walked a line three times, one load in flight; its backward pass 10.9 us, 20.5.
// With `loss` set (cross-entropy, every line in this one workgroup) the kernel also folds the row
// terms and divides by -N, in the order of ce_finalize_kernel: the whole loss in one launch.
// MODE: kLinesStaged (inner == 1) through StagedRows; kLinesThrough writes the result through, see line_mode.
enum { kLinesDirect, kLinesThrough, kLinesStaged };
template <typename T, int MODE> __device__ __forceinline__ void store_line(T *p, T v)
{
    if constexpr (MODE == kLinesThrough) store_through<T>(p, v);
    else *p = v;
}
template <typename T, bool CE, int OWN, int MODE>
__global__ __launch_bounds__(kLineWaves * 64) void softmax_lines_kernel(const T *x, T *y, int64_t lines, int R,
                                                                         int64_t inner, int waves, const T *target,
                                                                         T *rowloss, T *loss, T neg_n)
{
    __shared__ T shared[kLineWaves * 64];
    const LineSpot at(lines, R, inner, waves);
    const int lane = threadIdx.x & 63;
    const int r0 = at.w * OWN;
    const int valid = R - r0;              // uniform; at least 1
    constexpr bool STAGED = MODE == kLinesStaged;
    zmath::ExpLog<T> ml;
    StagedRows<T, OWN> rows(at.lines_here, R);
    T *const staged = reinterpret_cast<T *>(staged_raw);
    T *const row = staged + (at.active ? at.group * 64 + lane : 0) * rows.pitch(R);
    if constexpr (STAGED) {
        rows.load(x + at.first * R);
        ml.init(true, CE);
        rows.put(staged);
        __syncthreads();
    }
    const int64_t step = STAGED ? 1 : inner;
    const T *const xl = STAGED ? row + r0 : x + at.base + r0 * inner;
    T *const yl = STAGED ? row + r0 : y + at.base + r0 * inner;
    T v[OWN];
#pragma unroll
    for (int i = 0; i < OWN; i += 4) {
        if (i < valid) {
#pragma unroll
            for (int j = i; j < i + 4; j++) v[j] = xl[(j < valid ? j : 0) * step];
        }
    }
    const T x0 = waves > 1 ? (STAGED ? row[0] : x[at.base]) : v[0];
    if constexpr (!STAGED) ml.init(true, CE);
    // max_axis: strict '>' from element 0 (max.rs:19-34): a NaN there stays, a NaN elsewhere never replaces
    T m = -INFINITY;
#pragma unroll
    for (int i = 0; i < OWN; i++)
        if (i < valid) m = combine<T, true>(m, v[i]);
    if (waves > 1) {
        shared[threadIdx.x] = m;
        __syncthreads();
        for (int w = 0; w < waves; w++) m = combine<T, true>(m, shared[(at.group * waves + w) * 64 + lane]);
        __syncthreads();
    }
    m = combine<T, true>(x0, m);
    uint32_t least = ~0u;
#pragma unroll
    for (int i = 0; i < OWN; i++) {
        if (i < valid) {
            v[i] = ml.exp_flat(v[i] - m);
            least = least_term<T>(least, v[i]);
        }
    }
    const T sum = sum_in_order<T, OWN>(v, valid, at, waves, shared);
    auto finish = [&](auto by_reciprocal) {
        const T rcp = decltype(by_reciprocal)::value ? (T)1 / sum : (T)0;
#pragma unroll
        for (int i = 0; i < OWN; i++) {
            if (i < valid) {
                const T s = decltype(by_reciprocal)::value ? quotient<T>(v[i], sum, rcp) : v[i] / sum;
                if (at.active) store_line<T, MODE>(yl + i * step, s);
                if constexpr (CE) v[i] = target[at.base + r0 + i] * ml.log(s);
            }
        }
    };
    if (divides_by_reciprocal<T>(least, sum)) finish(std::true_type());
    else finish(std::false_type());
    if constexpr (STAGED) {
        __syncthreads();
        rows.store(y + at.first * R, staged);
    }
    if constexpr (CE) {
        if (waves > 1) __syncthreads();        // the sum of the exponentials has been read
        const T term = sum_in_order<T, OWN>(v, valid, at, waves, shared);
        if (loss) {     // uniform; one workgroup of at most four groups of 64 lines
            __shared__ T lds[4];
            T acc = at.active ? (T)0 + term : (T)0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) acc = acc + __shfl_xor(acc, o);
            if (threadIdx.x < 4) lds[threadIdx.x] = (T)0;
            __syncthreads();
            if (at.w == 0 && lane == 0) lds[at.group] = acc;
            __syncthreads();
            if (threadIdx.x == 0) *loss = (((lds[0] + lds[1]) + lds[2]) + lds[3]) / neg_n;
        } else if (at.active && at.w == 0) {
            rowloss[at.line] = term;
        }
    }
}

// lines longer than kLineWaves wavefronts hold, the softmax axis not the last one: one thread walks its line
template <typename T>
__global__ __launch_bounds__(kBlock) void softmax_long_lines_kernel(const T *x, T *y, int64_t lines, int64_t R, int64_t inner)
{
    zmath::ExpLog<T> ml;
    ml.init(true, false);
    const int64_t line = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (line >= lines) return;
    const int64_t q = line / inner;
    const int64_t base = q * R * inner + (line - q * inner);
    const T *xl = x + base;
    T *yl = y + base;
    // max_axis: strict '>' from element 0 (max.rs:19-34)
    T m = xl[0];
    for (int64_t r = 1; r < R; r++) {
        const T v = xl[r * inner];
        if (v > m) m = v;
    }
    // exp(x - max), summed in index order starting from zero (sum.rs:20-25)
    T sum = (T)0;
    for (int64_t r = 0; r < R; r++) {
        const T e = ml.exp(xl[r * inner] - m);
        yl[r * inner] = e;
        sum = sum + e;
    }
    for (int64_t r = 0; r < R; r++) yl[r * inner] = yl[r * inner] / sum;
}

// A row in vectors of any alignment.  Slot k of a thread is the vector at r = tid VEC + k step - head; a slot that
// sticks out of the row at either end loads the nearest whole vector instead (the load needs no branch) and owns
// only those of its elements that lie in the slot.
template <int VEC> struct RowSlot {
    int at;      // first element loaded
    int lo, hi;  // elements [lo, hi) of the loaded vector are the slot's own; lo >= VEC or hi <= 0: none
    __device__ __forceinline__ RowSlot(int r, int R)
    {
        at = min(max(r, 0), R - VEC);
        lo = r - at;
        hi = VEC + r - at;
    }
    __device__ __forceinline__ bool any() const { return lo < VEC && hi > 0; }
    __device__ __forceinline__ bool own(int j) const { return j >= lo && j < hi; }
    __device__ __forceinline__ bool full() const { return lo == 0; }
};
template <typename T, int VEC, typename Store>
__device__ __forceinline__ void store_slot(T *row, const RowSlot<VEC> &s, const Pack<T, VEC> &v, Store store)
{
    if (s.full()) {
        store(row, s.at, v);
    } else {
#pragma unroll
        for (int j = 0; j < VEC; j++)
            if (s.own(j)) row[s.at + j] = v.v[j];
    }
}
// Elements from the row's start to the 128-byte line that it starts in.  Streaming rows are cut into vectors
// there: wavefronts then write whole lines.
template <typename T> __device__ __forceinline__ int line_head(const T *row)
{
    return (int)((reinterpret_cast<uintptr_t>(row) & 127) / sizeof(T));
}
constexpr int kMaxHead = 32;   // elements, at most

// the vectors of a row from element `from` on, `step` apart, four loads in flight; the row's last, partial
// vector comes as single elements.  fn(r, n, load): n elements at r
template <typename T, int VEC, typename Fn> __device__ __forceinline__ void stream_row(int64_t from, int64_t step, int64_t R, Fn fn)
{
    int64_t r = from;
    for (; r + 3 * step + VEC <= R; r += 4 * step) fn(r, std::integral_constant<int, 4>(), VEC);
    for (; r + VEC <= R; r += step) fn(r, std::integral_constant<int, 1>(), VEC);
    if (r < R) fn(r, std::integral_constant<int, 1>(), (int)(R - r));
}
template <typename T, int VEC> __device__ __forceinline__ Pack<T, VEC> load_some(const T *p, int n, T fill)
{
    if (n == VEC) return load_pack<T, VEC, false>(p);
    Pack<T, VEC> v = splat<T, VEC>(fill);
#pragma unroll
    for (int j = 0; j < VEC; j++)
        if (j < n) v.v[j] = p[j];
    return v;
}
template <typename T, int VEC> __device__ __forceinline__ void store_some(T *p, int n, const Pack<T, VEC> &v)
{
    if (n == VEC) {
        store_pack<T, VEC, false>(p, v);
        return;
    }
#pragma unroll
    for (int j = 0; j < VEC; j++)
        if (j < n) p[j] = v.v[j];
}

// Rows that 256 threads hold in four vectors each, single elements with VEC == 1: without the slots of the general
// kernel below, whose bookkeeping costs 5 - 9 % on long rows (both with streaming stores: f32 [8192,4096] 46.5 against 48.7 us, [16384,2048]
// 44.7 / 48.7; even at [32768,1024], 61 - 63) and more where a launch is a few microseconds; whole_row_vector says which rows come here.
// NT: streamed loads; the result is written through and not past the caches ([8192,4096] 43.8 us against 45.8, the
// backward pass that reads it 58.9 against 65.2).
template <typename T, bool CE, bool NT, int VEC>
__global__ __launch_bounds__(kBlock) void softmax_whole_rows_kernel(const T *x, T *y, int64_t R, const T *target, T *rowloss,
                                                                     zmath::ExpLog<T> ml)
{
    __shared__ T lds[kWaves];
    const int64_t row = blockIdx.x;
    const T *xr = x + row * R;
    T *yr = y + row * R;
    const int64_t first = (int64_t)threadIdx.x * VEC;
    constexpr int64_t step = (int64_t)kBlock * VEC;
    const T x0 = xr[0];
    Pack<T, VEC> v[kWholePacks];
    T m = -INFINITY;
#pragma unroll
    for (int k = 0; k < kWholePacks; k++) {
        const int64_t r = first + k * step;
        v[k] = r < R ? load_pack<T, VEC, NT>(xr + r) : splat<T, VEC>(-INFINITY);
#pragma unroll
        for (int j = 0; j < VEC; j++) m = combine<T, true>(m, v[k].v[j]);
    }
    Pack<T, VEC> tg[kWholePacks];
    if (CE) {
#pragma unroll
        for (int k = 0; k < kWholePacks; k++) {
            const int64_t r = first + k * step;
            if (r < R) tg[k] = load_pack<T, VEC, NT>(target + row * R + r);
        }
    }
    ml.init(true, CE);   // after the row's loads are issued: the table fetch overlaps them
    m = block_red<T, true, kBlock>(m, lds);
    if (x0 != x0) m = x0;   // a NaN in position 0 is never replaced
    T sum = (T)0;
    uint32_t least = ~0u;
#pragma unroll
    for (int k = 0; k < kWholePacks; k++) {
        if (first + k * step < R) {
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                v[k].v[j] = ml.exp_flat(v[k].v[j] - m);
                sum = sum + v[k].v[j];
                least = least_term<T>(least, v[k].v[j]);
            }
        }
    }
    sum = block_red<T, false, kBlock>(sum, lds);
    T acc = (T)0;
    auto finish = [&](auto by_reciprocal) {
        const T rcp = decltype(by_reciprocal)::value ? (T)1 / sum : (T)0;
#pragma unroll
        for (int k = 0; k < kWholePacks; k++) {
            const int64_t r = first + k * step;
            if (r < R) {
#pragma unroll
                for (int j = 0; j < VEC; j++) {
                    v[k].v[j] = decltype(by_reciprocal)::value ? quotient<T>(v[k].v[j], sum, rcp) : v[k].v[j] / sum;
                    if (CE) acc = acc + tg[k].v[j] * ml.log(v[k].v[j]);
                }
                if constexpr (NT && !CE) store_pack_through<T, VEC>(yr + r, v[k]);
                else store_pack<T, VEC, false>(yr + r, v[k]);
            }
        }
    };
    if (divides_by_reciprocal<T>(least, sum)) finish(std::true_type());
    else finish(std::false_type());
    if (CE) {
        acc = block_red<T, false, kBlock>(acc, lds);
        if (threadIdx.x == 0) rowloss[row] = acc;
    }
}

// The softmax axis is the last one: LANES threads hold a row in registers, EPT elements each, and read and write
// it once (a wavefront takes a row of its own when LANES == 64).  LONG: the row is longer than that; what is
// beyond the registers is read three times and its exponentials are computed twice, from and into the same place.
// Bound by memory and, f32, by the 11 f64 operations of an exp: [2048,32003] f32 106 us (524 MB, 4.9 TB/s), 329 when
// the row was walked three times with scalar accesses.  One workgroup of 1024 threads per CU takes 146 us: loading,
// exp and storing follow each other; two of 512 threads with 64 elements each overlap theirs.
template <typename T, bool CE, bool NT, int STORE, bool LONG, int LANES, int EPT>
__global__ __launch_bounds__(LANES < 256 ? 256 : LANES, EPT == 64 ? 4 : 1) void softmax_rows_kernel(const T *x, T *y, int64_t rows, int64_t R,
                                                                                  const T *target, T *rowloss,
                                                                                  zmath::ExpLog<T> ml)
{
    // STORE: how the rows are written, see softmax_forward_launch
    // (ml arrives as an argument so that the f64 constants of exp / log sit in scalar registers; written
    // as literals each is copied into a register pair per use, and this kernel is bound by its scalar
    // instructions: the branch-free exp for the same reason)
    constexpr int VEC = VecOf<T>::N;
    constexpr int kPacks = EPT / VEC;
    constexpr int kRows = LANES < 256 ? 256 / LANES : 1;
    constexpr int step = LANES * VEC;
    __shared__ T lds[LANES / 64];
    const int tid = threadIdx.x % LANES;
    const int64_t row0 = (int64_t)blockIdx.x * kRows + (kRows > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / LANES)) : 0);
    const bool active = kRows == 1 || row0 < rows;     // uniform per wavefront
    const int64_t row = active ? row0 : 0;
    const T *xr = x + row * R;
    T *yr = y + row * R;
    const T *tr = CE ? target + row * R : nullptr;
    const int head = (NT && !LONG && R + kMaxHead <= LANES * EPT) ? line_head(yr) : 0;
    int first = tid * VEC - head;
    const int Rr = LONG ? LANES * EPT : (int)R;        // the part in registers
    // slots that every thread has whole, or no thread has: uniform, so that a row shorter than the registers costs
    // neither loads nor masks for what it lacks
    auto inner = [&](int k) { return LONG || (k * step >= head && (k + 1) * step - head <= Rr); };
    auto beyond = [&](int k) { return !LONG && k * step - head >= Rr; };
    const T x0 = xr[0];
    T acc = (T)0;

    Pack<T, VEC> v[kPacks];
#pragma unroll
    for (int k = 0; k < kPacks; k++) {
        v[k] = splat<T, VEC>(-(T)INFINITY);
        if (!beyond(k)) v[k] = load_pack<T, VEC, NT>(xr + RowSlot<VEC>(first + k * step, Rr).at);
    }
    // the targets of the cross-entropy terms travel with the row: loaded where they are used, each
    // pack cost the end of the kernel a round trip of its own
    Pack<T, VEC> tg[kPacks];
    if (CE) {
#pragma unroll
        for (int k = 0; k < kPacks; k++)
            if (!beyond(k)) tg[k] = load_pack<T, VEC, NT>(tr + RowSlot<VEC>(first + k * step, Rr).at);
    }
    ml.init(true, CE);      // after the row's loads are issued: the table fetch overlaps them
    asm volatile("" : "+v"(first));   // the slots are computed anew in every phase: kept, they take more registers than the row
    T m = -INFINITY;
#pragma unroll
    for (int k = 0; k < kPacks; k++) {
        if (!inner(k) && !beyond(k)) {
            const RowSlot<VEC> s(first + k * step, Rr);
#pragma unroll
            for (int j = 0; j < VEC; j++) v[k].v[j] = s.own(j) ? v[k].v[j] : -(T)INFINITY;
        }
        if (!beyond(k)) {
#pragma unroll
            for (int j = 0; j < VEC; j++) m = combine<T, true>(m, v[k].v[j]);
        }
    }
    if constexpr (LONG) {
        stream_row<T, VEC>(Rr + first, step, R, [&](int64_t r, auto count, int n) {
            constexpr int U = decltype(count)::value;
            Pack<T, VEC> p[U];
#pragma unroll
            for (int u = 0; u < U; u++) p[u] = load_some<T, VEC>(xr + r + u * step, n, -(T)INFINITY);
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int j = 0; j < VEC; j++) m = combine<T, true>(m, p[u].v[j]);
        });
    }
    m = block_red<T, true, LANES>(m, lds);
    if (x0 != x0) m = x0;   // a NaN in position 0 is never replaced
    asm volatile("" : "+v"(first));
    T sum = (T)0;
    uint32_t least = ~0u;   // f32: the smallest of this thread's terms above zero, as its bits less one
#pragma unroll
    for (int k = 0; k < kPacks; k++) {
        if (inner(k) || (!beyond(k) && RowSlot<VEC>(first + k * step, Rr).any())) {
#pragma unroll
            for (int j = 0; j < VEC; j++) {      // an element that is not the slot's own is exp(-inf), zero
                v[k].v[j] = ml.exp_flat(v[k].v[j] - m);
                sum = sum + v[k].v[j];
                least = least_term<T>(least, v[k].v[j]);
            }
        }
    }
    if constexpr (LONG) {
        stream_row<T, VEC>(Rr + first, step, R, [&](int64_t r, auto count, int n) {
            constexpr int U = decltype(count)::value;
            Pack<T, VEC> p[U];
#pragma unroll
            for (int u = 0; u < U; u++) p[u] = load_some<T, VEC>(xr + r + u * step, n, -(T)INFINITY);
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int j = 0; j < VEC; j++) sum = sum + ml.exp_flat(p[u].v[j] - m);
        });
    }
    sum = block_red<T, false, LANES>(sum, lds);
    const bool shared_divisor = divides_by_reciprocal<T>(least, sum);
    asm volatile("" : "+v"(first));
    auto finish = [&](auto by_reciprocal) {
        const T rcp = decltype(by_reciprocal)::value ? (T)1 / sum : (T)0;
#pragma unroll
        for (int k = 0; k < kPacks; k++) {
            const RowSlot<VEC> slot(first + k * step, Rr);
            if (inner(k) || (!beyond(k) && slot.any())) {
                const Pack<T, VEC> t = tg[k];
#pragma unroll
                for (int j = 0; j < VEC; j++) {
                    const T s = decltype(by_reciprocal)::value ? quotient<T>(v[k].v[j], sum, rcp) : v[k].v[j] / sum;
                    v[k].v[j] = s;
                    if (CE) acc = (LONG || slot.own(j)) ? acc + t.v[j] * ml.log(s) : acc;
                }
                // the CE output is read again by the backward pass; plain softmax is one stream in, one out
                if (active)
                    store_slot<T, VEC>(yr, slot, v[k], [](T *row, int at, const Pack<T, VEC> &z) {
                        if constexpr (STORE == kStorePlain) store_pack<T, VEC, false>(row + at, z);
                        else store_pack_wt_at<T, VEC, STORE == kStoreStream>(row, at, z);
                    });
            }
        }
    };
    if (shared_divisor) finish(std::true_type());
    else finish(std::false_type());
    if constexpr (LONG) {       // each thread re-reads the elements that it writes
        stream_row<T, VEC>(Rr + first, step, R, [&](int64_t r, auto count, int n) {
            constexpr int U = decltype(count)::value;
            Pack<T, VEC> p[U];
#pragma unroll
            for (int u = 0; u < U; u++) p[u] = load_some<T, VEC>(xr + r + u * step, n, -(T)INFINITY);
#pragma unroll
            for (int u = 0; u < U; u++) {
                Pack<T, VEC> t;
                if (CE) t = load_some<T, VEC>(tr + r + u * step, n, (T)0);
#pragma unroll
                for (int j = 0; j < VEC; j++) {
                    p[u].v[j] = ml.exp_flat(p[u].v[j] - m) / sum;
                    if (CE) acc = j < n ? acc + t.v[j] * ml.log(p[u].v[j]) : acc;
                }
                store_some<T, VEC>(yr + r + u * step, n, p[u]);
            }
        });
    }
    if (CE) {
        acc = block_red<T, false, LANES>(acc, lds);
        if (active && tid == 0) rowloss[row] = acc;
    }
}

// loss = (sum of the row terms) / (-N), one workgroup
template <typename T>
__global__ __launch_bounds__(kBlock) void ce_finalize_kernel(const T *rowloss, int64_t n, T *loss, T neg_n)
{
    __shared__ T lds[kWaves];
    T acc = (T)0;
    int64_t i = threadIdx.x;
    for (; i + 7 * kBlock < n; i += 8 * kBlock) {       // eight loads in flight, added in index order
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = rowloss[i + u * kBlock];
#pragma unroll
        for (int u = 0; u < 8; u++) acc = acc + v[u];
    }
    for (; i < n; i += kBlock) acc = acc + rowloss[i];
    acc = block_red<T, false>(acc, lds);
    if (threadIdx.x == 0) *loss = acc / neg_n;
}

// ---- backward --------------------------------------------------------------------------------------------
// elements per thread of the largest workgroups, which leave a thread 128 registers: y and t of the backward pass, or
// the terms of the forward pass with the constants of exp, in 64 of them (f64 with 32 elements spills)
template <typename T> constexpr int kMost = 128 / (int)sizeof(T);

// gx = t - y * sum(t), t = y * gy.  CE: gy = (target * g_total) / y with g_total = gout / (-N), the
// chain div -> sum_to -> mul -> log backward of cross_entropy.rs:18-22.

// lines in registers, as in softmax_lines_kernel; the sum of t in index order.  Where t alone fills the registers of a
// workgroup of 1024 threads (f64 lines of 257 - 512 elements), y is read a second time.
template <typename T, bool CE, int OWN, int MODE>
__global__ __launch_bounds__(kLineWaves * 64) void softmax_bwd_lines_kernel(const T *y, const T *gy_or_target, T *gx,
                                                                             int64_t lines, int R, int64_t inner,
                                                                             int waves, const T *gout, T neg_n)
{
    __shared__ T carry[kLineWaves * 64];
    const LineSpot at(lines, R, inner, waves);
    const T g_total = CE ? (gout ? *gout : (T)1) / neg_n : (T)0;
    const int r0 = at.w * OWN;
    const int valid = R - r0;
    const int64_t base = at.base + r0 * inner;
    constexpr bool kHold = OWN <= kMost<T>, STAGED = MODE == kLinesStaged;
    T yv[kHold ? OWN : 1], t[OWN];
    StagedRows<T, OWN> rows(at.lines_here, R);
    T *const staged = reinterpret_cast<T *>(staged_raw);
    T *const mine = staged + (at.active ? at.group * 64 + (threadIdx.x & 63) : 0) * rows.pitch(R) + r0;
    auto product = [&](T yj, T g) { return yj * (CE ? (g * g_total) / yj : g); };
    if constexpr (STAGED) {
        static_assert(kHold, "short rows");
        StagedRows<T, OWN> second(at.lines_here, R);
        rows.load(y + at.first * R);
        second.load(gy_or_target + at.first * R);
        rows.put(staged);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < OWN; i++)
            if (i < valid) yv[i] = mine[i];
        __syncthreads();
        second.put(staged);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < OWN; i++)
            if (i < valid) t[i] = product(yv[i], mine[i]);
    } else {
        T once[OWN];
#pragma unroll
        for (int i = 0; i < OWN; i += 4) {
            if (i < valid) {
#pragma unroll
                for (int j = i; j < i + 4; j++) {
                    const int64_t off = base + (j < valid ? j : 0) * inner;
                    once[j] = y[off];
                    t[j] = gy_or_target[off];
                }
                if constexpr (!kHold) {
#pragma unroll
                    for (int j = i; j < i + 4; j++) t[j] = product(once[j], t[j]);
                }
            }
        }
        if constexpr (kHold) {
#pragma unroll
            for (int i = 0; i < OWN; i++) {
                if (i < valid) {
                    yv[i] = once[i];
                    t[i] = product(yv[i], t[i]);
                }
            }
        }
    }
    const T sum = sum_in_order<T, OWN>(t, valid, at, waves, carry);
    if constexpr (STAGED) {
        if (waves == 1) __syncthreads();       // every row has been read (sum_in_order's barriers, otherwise)
        if (at.active) {
#pragma unroll
            for (int i = 0; i < OWN; i++)
                if (i < valid) mine[i] = t[i] - yv[i] * sum;
        }
        __syncthreads();
        rows.store(gx + at.first * R, staged);
    } else if (at.active) {
#pragma unroll
        for (int i = 0; i < OWN; i += 4) {
            if (i < valid) {
                T again[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if constexpr (kHold) again[j] = yv[i + j];
                    else again[j] = y[base + (i + j < valid ? i + j : 0) * inner];
                }
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (i + j < valid) {
                        store_line<T, MODE>(gx + base + (i + j) * inner, t[i + j] - again[j] * sum);
                    }
            }
        }
    }
}

// lines longer than that, the softmax axis not the last one
template <typename T>
__global__ __launch_bounds__(kBlock) void softmax_bwd_long_lines_kernel(const T *y, const T *gy, T *gx, int64_t lines,
                                                                         int64_t R, int64_t inner)
{
    const int64_t line = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (line >= lines) return;
    const int64_t q = line / inner;
    const int64_t base = q * R * inner + (line - q * inner);
    T sum = (T)0;
    for (int64_t r = 0; r < R; r++) {
        const int64_t off = base + r * inner;
        sum = sum + y[off] * gy[off];
    }
    for (int64_t r = 0; r < R; r++) {
        const int64_t off = base + r * inner;
        const T yv = y[off];
        gx[off] = yv * gy[off] - yv * sum;
    }
}

// Rows in registers, as in softmax_rows_kernel: y and y * gy are held, two reads and one write.  LONG: what is
// beyond the registers is read twice.  [2048,32003] f32 126 us (787 MB, 6.2 TB/s; 137 when y had been written past the
// caches), 311 with scalar accesses
// and t written out and read back.
template <typename T, bool CE, bool NT, bool LONG, int LANES, int EPT>
__global__ __launch_bounds__(LANES < 256 ? 256 : LANES) void softmax_bwd_rows_kernel(const T *y, const T *gy_or_target, T *gx,
                                                                                      int64_t rows, int64_t R,
                                                                                      const T *gout, T neg_n)
{
    constexpr int VEC = VecOf<T>::N;
    constexpr int kPacks = EPT / VEC;
    constexpr int kRows = LANES < 256 ? 256 / LANES : 1;
    constexpr int step = LANES * VEC;
    __shared__ T lds[LANES / 64];
    const T g_total = CE ? (gout ? *gout : (T)1) / neg_n : (T)0;
    const int tid = threadIdx.x % LANES;
    const int64_t row = (int64_t)blockIdx.x * kRows + (kRows > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / LANES)) : 0);
    if (kRows > 1 && row >= rows) return;      // a wavefront per row: no barrier follows
    const int64_t base = row * R;
    const T *yr = y + base;
    const T *sr = gy_or_target + base;
    T *gr = gx + base;
    const int head = (NT && !LONG && R + kMaxHead <= LANES * EPT) ? line_head(gr) : 0;
    const int first = tid * VEC - head;
    const int Rr = LONG ? LANES * EPT : (int)R;
    auto product = [&](T yv, T g) { return yv * (CE ? (g * g_total) / yv : g); };
    auto inner = [&](int k) { return LONG || (k * step >= head && (k + 1) * step - head <= Rr); };   // as in the forward pass
    auto beyond = [&](int k) { return !LONG && k * step - head >= Rr; };
    T sum = (T)0;
    Pack<T, VEC> yv[kPacks], t[kPacks];
    // all loads of the thread first: with the loads inside a bounds check the compiler waits for each pair
    // before it issues the next, because the running sum orders the blocks
#pragma unroll
    for (int k = 0; k < kPacks; k++) {
        if (!beyond(k)) {
            const RowSlot<VEC> s(first + k * step, Rr);
            yv[k] = load_pack<T, VEC, NT && !CE>(yr + s.at);
            t[k] = load_pack<T, VEC, NT>(sr + s.at);
        }
    }
#pragma unroll
    for (int k = 0; k < kPacks; k++) {
        const RowSlot<VEC> s(first + k * step, Rr);
        if (inner(k)) {
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                t[k].v[j] = product(yv[k].v[j], t[k].v[j]);
                sum = sum + t[k].v[j];
            }
        } else if (!beyond(k) && s.any()) {
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                t[k].v[j] = product(yv[k].v[j], t[k].v[j]);
                sum = s.own(j) ? sum + t[k].v[j] : sum;
            }
        }
    }
    if constexpr (LONG) {
        stream_row<T, VEC>(Rr + first, step, R, [&](int64_t r, auto count, int n) {
            constexpr int U = decltype(count)::value;
            Pack<T, VEC> a[U], b[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                a[u] = load_some<T, VEC>(yr + r + u * step, n, (T)1);
                b[u] = load_some<T, VEC>(sr + r + u * step, n, (T)0);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int j = 0; j < VEC; j++) sum = j < n ? sum + product(a[u].v[j], b[u].v[j]) : sum;
        });
    }
    sum = block_red<T, false, LANES>(sum, lds);
#pragma unroll
    for (int k = 0; k < kPacks; k++) {
        const RowSlot<VEC> s(first + k * step, Rr);
        if (inner(k) || (!beyond(k) && s.any())) {
#pragma unroll
            for (int j = 0; j < VEC; j++) t[k].v[j] = t[k].v[j] - yv[k].v[j] * sum;
            store_slot<T, VEC>(gr, s, t[k], [](T *row, int at, const Pack<T, VEC> &z) { store_pack<T, VEC, NT>(row + at, z); });
        }
    }
    if constexpr (LONG) {       // each thread re-reads the elements that it writes
        stream_row<T, VEC>(Rr + first, step, R, [&](int64_t r, auto count, int n) {
            constexpr int U = decltype(count)::value;
            Pack<T, VEC> a[U], b[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                a[u] = load_some<T, VEC>(yr + r + u * step, n, (T)1);
                b[u] = load_some<T, VEC>(sr + r + u * step, n, (T)0);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int j = 0; j < VEC; j++) b[u].v[j] = product(a[u].v[j], b[u].v[j]) - a[u].v[j] * sum;
                store_some<T, VEC>(gr + r + u * step, n, b[u]);
            }
        });
    }
}

// ---- a classifier head's batch in ONE workgroup, four lanes per line -------------------------------------------
// lines <= 256 of R <= 16 elements, contiguous (inner == 1).  One thread per line (the lines kernels
// above) is a single wavefront per SIMD walking through 16 unrolled copies of exp / log / division:
// 7-8 us for [256,10], most of it instruction fetch and dependent latencies that nothing overlaps.
// Here a quad of lanes owns a line -- lane q holds elements q, q + 4, q + 8, q + 12 -- in a workgroup
// of 1024 threads: four copies of the transcendental code, sixteen wavefronts.  Everything that the
// one-thread form does in index order (the max scan, the sum of the exponentials, the sum of the
// cross-entropy terms, the sum of t) is still done in index order, by every lane of the quad on
// values gathered from its neighbours, so the bits are the same.
constexpr int kHeadBlock = 1024;
constexpr int kHeadLines = kHeadBlock / 4;
constexpr int kHeadOwn = kLineRegs / 4;

// full[r] for r = 4 i + q is own[i] of lane q of the quad
template <typename T> __device__ __forceinline__ void quad_gather(const T (&own)[kHeadOwn], T (&full)[kLineRegs])
{
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) {
#pragma unroll
        for (int q = 0; q < 4; q++) full[4 * i + q] = __shfl(own[i], q, 4);
    }
}

// Forward: y = softmax(x) per line, *loss = sum over lines of (sum_r target * log y) / neg_n, the row
// terms folded as ce_finalize_kernel folds them (256 lanes: butterfly per wavefront, wavefronts in order).
template <typename T>
__global__ __launch_bounds__(kHeadBlock) void ce_head_forward_kernel(const T *x, T *y, int64_t lines, int64_t R,
                                                                      const T *target, T *loss, T neg_n)
{
    __shared__ T terms[kHeadLines];
    __shared__ T wave_sum[kHeadLines / 64];
    const int q = threadIdx.x & 3;
    const int64_t line = threadIdx.x >> 2;
    const bool active = line < lines;
    const int64_t base = (active ? line : 0) * R;
    T v[kHeadOwn], tg[kHeadOwn];
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) {
        const int r = 4 * i + q;
        const int64_t off = base + (r < R ? r : 0);
        v[i] = x[off];
        tg[i] = target[off];
    }
    zmath::ExpLog<T> ml;
    ml.init(true, true);
    T full[kLineRegs];
    quad_gather<T>(v, full);
    T m = full[0];                       // max_axis: strict '>' from element 0 (max.rs:19-34)
#pragma unroll
    for (int r = 1; r < kLineRegs; r++)
        if (r < R && full[r] > m) m = full[r];
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) v[i] = ml.exp(v[i] - m);
    quad_gather<T>(v, full);
    T sum = (T)0;                        // in index order from zero (sum.rs:20-25)
#pragma unroll
    for (int r = 0; r < kLineRegs; r++)
        if (r < R) sum = sum + full[r];
    T term[kHeadOwn];
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) {
        const int r = 4 * i + q;
        const T sm = v[i] / sum;
        if (active && r < R) y[base + r] = sm;
        term[i] = r < R ? tg[i] * ml.log(sm) : (T)0;
    }
    quad_gather<T>(term, full);
    T acc = (T)0;
#pragma unroll
    for (int r = 0; r < kLineRegs; r++)
        if (r < R) acc = acc + full[r];
    if (q == 0) terms[line] = active ? (T)0 + acc : (T)0;
    __syncthreads();
    if (threadIdx.x < kHeadLines) {      // uniform per wavefront
        T a = terms[threadIdx.x];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) a = a + __shfl_xor(a, o);
        if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = a;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        T a = wave_sum[0];
#pragma unroll
        for (int w = 1; w < kHeadLines / 64; w++) a = a + wave_sum[w];
        *loss = a / neg_n;
    }
}

// Backward: gx = t - y * sum(t) with t = y * ((target * g_total) / y), and colsum[r] = the sum of gx over
// the lines (when set), each column folded as block_red folds 256 lanes.
template <typename T>
__global__ __launch_bounds__(kHeadBlock) void ce_head_backward_kernel(const T *y, const T *target, T *gx, int64_t lines,
                                                                       int64_t R, const T *gout, T neg_n, T *colsum)
{
    __shared__ T cols[kLineRegs][kHeadLines];      // gx by column, for the column sums
    const int q = threadIdx.x & 3;
    const int64_t line = threadIdx.x >> 2;
    const bool active = line < lines;
    const int64_t base = (active ? line : 0) * R;
    const T g_total = (gout ? *gout : (T)1) / neg_n;
    T yv[kHeadOwn], t[kHeadOwn];
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) {
        const int r = 4 * i + q;
        const int64_t off = base + (r < R ? r : 0);
        yv[i] = y[off];
        t[i] = target[off];
    }
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) t[i] = yv[i] * ((t[i] * g_total) / yv[i]);
    T full[kLineRegs];
    quad_gather<T>(t, full);
    T sum = (T)0;
#pragma unroll
    for (int r = 0; r < kLineRegs; r++)
        if (r < R) sum = sum + full[r];
#pragma unroll
    for (int i = 0; i < kHeadOwn; i++) {
        const int r = 4 * i + q;
        const T g = t[i] - yv[i] * sum;
        if (active && r < R) gx[base + r] = g;
        if (colsum && r < R) cols[r][line] = active ? (T)0 + g : (T)0;
    }
    if (!colsum) return;                 // uniform
    __syncthreads();
    // wavefront w folds column w: four runs of 64 lines, each with the butterfly, then the runs in order
    const int64_t col = threadIdx.x >> 6;
    if (col < R) {
        const int lane = threadIdx.x & 63;
        T total = (T)0;
#pragma unroll
        for (int w = 0; w < kHeadLines / 64; w++) {
            T c = cols[col][w * 64 + lane];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) c = c + __shfl_xor(c, o);
            total = w == 0 ? c : total + c;
        }
        if (lane == 0) colsum[col] = total;
    }
}

// ---- bias add + ReLU ----------------------------------------------------------------------------------------
// pre = z + bias (broadcast over rows), act = pre > 0 ? pre : alpha * pre  (relu.rs:44-48)

// Any row length, any alignment: the tensor as one run of vectors, one per lane of a 64-thread workgroup; a vector
// that spans two rows gathers its bias.  [1000,1500] f32 4.85 us (18 MB), 5.2 with a 64-bit division per vector
// in a grid-stride loop.
constexpr int kTileLanes = 64;
template <typename T, int VEC, bool NT, typename Index>
__global__ __launch_bounds__(kTileLanes) void bias_relu_kernel(const T *z, const T *bias, T *pre, T *act, Index n,
                                                               Index F, T alpha)
{
    const Index off = ((Index)blockIdx.x * kTileLanes + threadIdx.x) * VEC;
    const Index col = off % F;
    if (off + VEC <= n) {
        const Pack<T, VEC> v = load_pack<T, VEC, NT>(z + off);
        Pack<T, VEC> b;
        if (col + VEC <= F) {
            b = load_pack<T, VEC, false>(bias + col);
        } else {
            Index c = col;
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                b.v[j] = bias[c];
                c = c + 1 == F ? 0 : c + 1;
            }
        }
        Pack<T, VEC> a, h;
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            a.v[j] = v.v[j] + b.v[j];
            h.v[j] = a.v[j] > (T)0 ? a.v[j] : alpha * a.v[j];
        }
        if (pre) store_pack<T, VEC, NT>(pre + off, a);
        store_pack<T, VEC, NT>(act + off, h);
    } else {
        Index c = col;
        for (Index i = off; i < n; i++) {
            const T a = z[i] + bias[c];
            if (pre) pre[i] = a;
            act[i] = a > (T)0 ? a : alpha * a;
            c = c + 1 == F ? 0 : c + 1;
        }
    }
}

// Rows that are a whole number of 64-lane vectors: a 64-thread workgroup per contiguous piece of a
// row, one vector per lane (the shape that streams best when most of the traffic is stores); the
// row / column split is one 32-bit division per workgroup on the scalar unit.
template <typename T, int VEC, bool NT>
__global__ __launch_bounds__(kTileLanes) void bias_relu_tile_kernel(const T *z, const T *bias, T *pre, T *act,
                                                                     uint32_t tiles_per_row, T alpha)
{
    const uint32_t row = blockIdx.x / tiles_per_row;
    const uint32_t tile = blockIdx.x - row * tiles_per_row;
    const int64_t col = ((int64_t)tile * kTileLanes + threadIdx.x) * VEC;
    const int64_t off = (int64_t)blockIdx.x * kTileLanes * VEC + (int64_t)threadIdx.x * VEC;
    const Pack<T, VEC> v = load_pack<T, VEC, NT>(z + off);
    const Pack<T, VEC> b = load_pack<T, VEC, false>(bias + col);
    Pack<T, VEC> a, h;
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        a.v[j] = v.v[j] + b.v[j];
        h.v[j] = a.v[j] > (T)0 ? a.v[j] : alpha * a.v[j];
    }
    if constexpr (NT && VEC > 1) {
        if (pre) store_pack_wt<T, VEC>(pre + off, a);
        store_pack_wt<T, VEC>(act + off, h);
    } else {
        if (pre) store_pack<T, VEC, NT>(pre + off, a);
        store_pack<T, VEC, NT>(act + off, h);
    }
}

// ---- host side ------------------------------------------------------------------------------------------------

// a tensor as a contiguous device buffer: itself, or a temporary copy
template <typename T> struct ContigIn {
    Workspace ws;
    const T *ptr;
    int status;
    ContigIn(const zenu_tensor_t &t, int dtype, hipStream_t s)
        : ws(is_default_stride_strict(t) ? 0 : (size_t)num_elm(t) * sizeof(T), s),
          ptr(static_cast<const T *>(t.ptr)), status(ws.status)
    {
        if (is_default_stride_strict(t) || status) return;
        zenu_tensor_t tmp = default_view(ws.ptr, t.ndim, t.shape);
        status = zenu_hip_copy(dtype, &tmp, &t, reinterpret_cast<zenu_stream_t>(s));
        ptr = static_cast<const T *>(ws.ptr);
    }
};

// a contiguous buffer to write into: the tensor itself, or a temporary that finish() copies out
template <typename T> struct ContigOut {
    Workspace ws;
    const zenu_tensor_t &t;
    T *ptr;
    int status;
    int dtype;
    bool temp;
    ContigOut(const zenu_tensor_t &t_, int dtype_, hipStream_t s)
        : ws(is_default_stride_strict(t_) ? 0 : (size_t)num_elm(t_) * sizeof(T), s), t(t_),
          ptr(static_cast<T *>(t_.ptr)), status(ws.status), dtype(dtype_), temp(!is_default_stride_strict(t_))
    {
        if (temp && !status) ptr = static_cast<T *>(ws.ptr);
    }
    int finish()
    {
        if (!temp) return ZENU_OK;
        zenu_tensor_t tmp = default_view(ws.ptr, t.ndim, t.shape);
        return zenu_hip_copy(dtype, &t, &tmp, reinterpret_cast<zenu_stream_t>(ws.stream));
    }
};

struct Geometry { int64_t outer, R, inner; };

Geometry geometry(const zenu_tensor_t &t, int axis)
{
    Geometry g = {1, t.shape[axis], 1};
    for (int i = 0; i < axis; i++) g.outer *= t.shape[i];
    for (int i = axis + 1; i < t.ndim; i++) g.inner *= t.shape[i];
    return g;
}

inline bool grid_ok(int64_t blocks) { return blocks > 0 && blocks <= 0x7fffffffLL; }

// true when the cross-entropy forward of this geometry is one workgroup of the lines kernel, which
// then also produces the loss (no row terms in memory, no second launch)
inline bool ce_single_workgroup(const Geometry &g)
{
    return g.inner == 1 && g.R <= kLineMaxR && g.outer <= kBlock;
}

// How many elements of a line a thread of the lines kernels holds: as many as leave every SIMD two wavefronts, so
// that a large tensor needs no hand-over of sums and a small one is not a single thread's long chain; never so few
// that the line needs more than kLineWaves wavefronts.  0: the line is too long for them.
inline int line_own(int64_t lines, int64_t R, int most)
{
    const int64_t groups = (lines + 63) / 64;
    const int64_t want = 8 * (int64_t)device_info().num_cus;
    while (most > 8 && most / 2 >= R) most /= 2;   // (no registers for elements that no line has: [128,5,12544] f32 25.8 -> 16.0 us)
    for (int own = most; own >= 8; own /= 2) {
        if (R > (int64_t)own * kLineWaves) return own == most ? 0 : 2 * own;
        if (groups * ((R + own - 1) / own) >= want) return own;
    }
    return 8;
}
// The most elements a thread of the forward pass holds.  Rows of the last axis (R <= 64) need no more than eight
// wavefronts of 8, and the loss takes those: with a logarithm per element its constants spill at 16 and 32 elements (f32
// [65536,64] 93.8 us at 32, 51.8 at 8; f64 110 / 77.5); plain f64 takes 16 (96 -> 38 us).  Plain f32 and other axes
// hold up to 32.
template <typename T, bool CE> inline int line_most(const Geometry &g)
{
    if (g.inner > 1 || g.R <= 16) return 32;
    return CE ? 8 : sizeof(T) == 8 ? 16 : 32;
}
// Rows that go through StagedRows (us without / with, softmax and its backward pass): f32 [60000,33] 15.6 / 8.2 and 19.6 / 7.4,
// [65536,64] 31 / 14 and 40 / 14, [65536,16] 10.1 / 5.1 and 10.0 / 4.5, [300,50] 6.3 / 5.2 and 5.4 / 4.5, [20000,21] 6.4 / 5.1 and
// 5.4 / 4.4; f64 [65536,64] 36 / 23 and 50 / 19.  Short rows of a small tensor, which the first cache holds, lose by the turn in
// LDS ([5000,10] 4.1 / 4.3 and 3.0 / 3.9), very short ones always ([65536,2] 2.7 / 3.3).
inline bool staged_rows(const Geometry &g)
{
    return g.inner == 1 && g.R <= kLineMaxR && (g.R > 32 || (g.R >= 8 && g.outer * g.R >= 1 << 18));
}
// How the lines kernels write (us, left in the L2 / written through): all wavefronts of a launch store at about the same
// time, and what is dirty in the L2 then is written back behind the last of them.  Softmax [16,21,16384] f32 14.8 / 12.5,
// [2,32,16083] 5.4 / 4.7, [32,120,3136] 25.9 / 23.7, f64 [16,21,8000] 15.6 / 13.7; backward 11.4 / 10.9, 4.1 / 3.6, f64 11.4 /
// 10.9, but a larger result of the same operands again and again streams better through the L2 ([8,21,50000] 17.5 / 17.8).  Forward
// there is no such size; operands used once, softmax alone and with its backward pass behind it: f32 [32,21,65536] (176 MB)
// 67.7 / 65.7 and 163.5 / 160.9, [2048,5,12544] (514 MB) 222 / 215 and 489 / 484, [16,150,65536] (629 MB) 257 / 255 and 632 / 630, f64
// [32,21,65536] 130.1 / 128.6 and 319 / 317.  Staged rows: [65536,64] 16.3 / 14.1 and 15.8 / 13.6, used once [1048576,64] (268 MB)
// 113.0 / 112.7 and, backward, 153.8 / 153.6.  Where neighbouring lanes do not write neighbouring elements the L2 has to collect them ([65536,3] 3.0 / 3.2).
inline int line_mode(const Geometry &g, bool forward, size_t size)
{
    if (staged_rows(g)) return kLinesStaged;
    return g.inner >= 32 && (forward || g.outer * g.R * g.inner * (int64_t)size < kStreamBytes) ? kLinesThrough : kLinesDirect;
}
template <bool MAY_STAGE, typename Go> void with_line_mode(int mode, Go go)
{
    if constexpr (MAY_STAGE)
        if (mode == kLinesStaged) return go(std::integral_constant<int, kLinesStaged>());
    if (mode == kLinesThrough) go(std::integral_constant<int, kLinesThrough>());
    else go(std::integral_constant<int, kLinesDirect>());
}
// calls go(own) with `own` as a constant
template <int MOST, typename Go> int with_own(int own, Go go)
{
    if constexpr (MOST >= 32)
        if (own == 32) return go(std::integral_constant<int, 32>());
    if (own == 16) return go(std::integral_constant<int, 16>());
    return go(std::integral_constant<int, 8>());
}
// wavefronts along a line, and lines in groups of 64 that fill a workgroup of about four wavefronts
struct LineGrid {
    int waves, groups;
    int64_t blocks;
    LineGrid(int64_t lines, int64_t R, int own, bool one_workgroup)
    {
        const int64_t all = (lines + 63) / 64;
        waves = (int)((R + own - 1) / own);
        groups = waves >= 4 ? 1 : 4 / waves;
        if (one_workgroup || groups > all) groups = (int)all;
        blocks = (all + groups - 1) / groups;
    }
    unsigned threads() const { return (unsigned)(64 * waves * groups); }
    template <typename T, int OWN> size_t staged_bytes(int64_t R) const
    {
        return (size_t)(64 * groups) * StagedRows<T, OWN>::pitch((int)R) * sizeof(T);   // at most 35 KB: four groups only where R <= OWN
    }
};

// Threads per row and elements per thread of the rows kernels by row length (a streaming row
// is cut at cache lines where the registers leave room for it).  go(lanes, elements, long) gets constants.
template <int VEC, int EPT_LONG, typename Go> int with_row_shape(int64_t R, Go go)
{
    typedef std::integral_constant<int, 64> L64;
    typedef std::integral_constant<int, 256> L256;
    typedef std::integral_constant<int, 512> L512;
    typedef std::integral_constant<int, 1024> L1024;
    typedef std::integral_constant<int, EPT_LONG> Long;
    if (R <= 512) return go(L64(), std::integral_constant<int, 8>(), std::false_type());
    if (R <= 1024) return go(L256(), std::integral_constant<int, 4>(), std::false_type());
    if (R <= 1024 * VEC) return go(L256(), std::integral_constant<int, 4 * VEC>(), std::false_type());
    if (R <= 4096) return go(L256(), std::integral_constant<int, 16>(), std::false_type());
    if (R <= 512 * EPT_LONG) return go(L512(), Long(), std::false_type());
    if (R <= 1024 * EPT_LONG) return go(L1024(), Long(), std::false_type());
    return go(L1024(), Long(), std::true_type());
}

template <typename T> inline bool whole_rows(int64_t R, const T *in, const T *out)
{
    return R % VecOf<T>::N == 0 && aligned16(in) && aligned16(out);
}
// Vector width with which softmax_whole_rows_kernel takes rows of R > kLineMaxR elements; 0: the general kernel does.
// Single elements: few rows (four per CU, in f64 up to 256 elements two), as long as a wavefront would hold a long row
// or one with ragged ends: the shorter chain counts (f32 [100,301] 3.3 us against 4.2 in the general kernel, f64 [100,512]
// 3.8 / 5.2, its loss [100,256] 5.9 / 7.0; but f64 loss [1000,127] 8.2 / 7.2); and ragged rows beyond a wavefront's 512,
// [32768,513] f32 39.6 / 47 us, f64 62 / 65 (the loss to 768: [32768,641] 67 / 80 us, [32768,1001] 95 / 90 after writes).
// Vectors: plain rows beyond 512 (those of a wavefront are faster: [65536,512] 92 / 47 us), the loss beyond one
// vector per thread ([32768,1100] f32 108 / 123 us, [4096,1100] f64 30 / 41; [4096,1024] f32 18.8 / 17.9).
template <typename T, bool CE> inline int whole_row_vector(int64_t lines, int64_t R, bool whole)
{
    constexpr int VEC = VecOf<T>::N;
    const int64_t cus = device_info().num_cus;
    const bool few = lines <= (sizeof(T) == 8 && R <= 256 ? 2 : 4) * cus;
    if (R <= kWholePacks * kBlock) {
        if (few && (!whole || R > 256 || sizeof(T) == 8)) return 1;
        if (!whole && R > 512 && (!CE || R <= 768)) return 1;
    }
    return whole && R > (CE ? kBlock * VEC : 512) && R <= kWholePacks * kBlock * VEC ? VEC : 0;
}

template <typename T, bool CE>
int softmax_forward_launch(const T *x, T *y, Geometry g, const T *target, T *rowloss, hipStream_t s,
                           T *loss = nullptr, T neg_n = (T)0)
{
    const int64_t lines = g.outer * g.inner;
    if constexpr (CE) {
        if (loss && g.inner == 1 && g.R <= kLineRegs && lines <= kHeadLines) {   // a classifier head: four lanes per line
            ce_head_forward_kernel<T><<<1, kHeadBlock, 0, s>>>(x, y, lines, g.R, target, loss, neg_n);
            ZENU_LAUNCH_CHECK();
            return ZENU_OK;
        }
    }
    if (g.inner != 1 || g.R <= kLineMaxR) {
        // (16 elements at most where the whole loss is one workgroup: 16 wavefronts hold 256 lines of 64)
        int own = line_own(lines, g.R, line_most<T, CE>(g));
        if (CE && loss && own < 16 && (lines + 63) / 64 * ((g.R + own - 1) / own) > kLineWaves) own = 16;
        if (own == 0) {
            const int64_t blocks = (lines + kBlock - 1) / kBlock;
            if (!grid_ok(blocks)) return ZENU_ERR_UNSUPPORTED;
            softmax_long_lines_kernel<T><<<(unsigned)blocks, kBlock, 0, s>>>(x, y, lines, g.R, g.inner);
        } else {
            const LineGrid lg(lines, g.R, own, CE && loss);
            if (!grid_ok(lg.blocks)) return ZENU_ERR_UNSUPPORTED;
            with_own<32>(own, [&](auto o) {
                constexpr int OWN = decltype(o)::value;
                auto go = [&](auto mode_c) {
                    constexpr int MODE = decltype(mode_c)::value;
                    softmax_lines_kernel<T, CE, OWN, MODE><<<(unsigned)lg.blocks, lg.threads(), MODE == kLinesStaged ? lg.template staged_bytes<T, OWN>(g.R) : 0, s>>>(
                        x, y, lines, (int)g.R, g.inner, lg.waves, target, rowloss, loss, neg_n);
                };
                if constexpr (CE) go(std::integral_constant<int, kLinesDirect>());   // (the loss: inner == 1)
                else with_line_mode<true>(line_mode(g, true, sizeof(T)), go);
                return 0;
            });
        }
    } else {
        const bool whole = whole_rows<T>(g.R, x, y);
        // ragged rows of a wavefront share their first and last lines with other rows: written past the cache, softmax of
        // [32768,255] f32 takes 53 us, 19 without the hint.  The loss keeps its probabilities cached in any case.
        const bool nt = lines * g.R * (int64_t)sizeof(T) * 2 >= kStreamBytes && (CE || whole || g.R > 1024);
        constexpr int VEC = VecOf<T>::N;
        const int vec = whole_row_vector<T, CE>(lines, g.R, whole);
        if (vec) {
            if (!grid_ok(lines)) return ZENU_ERR_UNSUPPORTED;
            const unsigned grid = (unsigned)lines;
            if (vec == 1) softmax_whole_rows_kernel<T, CE, false, 1><<<grid, kBlock, 0, s>>>(x, y, g.R, target, rowloss, zmath::ExpLog<T>());
            else if (nt)  softmax_whole_rows_kernel<T, CE, true, VEC><<<grid, kBlock, 0, s>>>(x, y, g.R, target, rowloss, zmath::ExpLog<T>());
            else          softmax_whole_rows_kernel<T, CE, false, VEC><<<grid, kBlock, 0, s>>>(x, y, g.R, target, rowloss, zmath::ExpLog<T>());
            ZENU_LAUNCH_CHECK();
            return ZENU_OK;
        }
        const int rc = with_row_shape<VecOf<T>::N, kMost<T>>(g.R, [&](auto lanes, auto ept, auto is_long) -> int {
            constexpr bool LONG = decltype(is_long)::value;
            // f32: two workgroups of 512 threads on a CU instead of one of 1024, see softmax_rows_kernel
            constexpr bool two = decltype(lanes)::value == 1024 && decltype(ept)::value == 32 && !LONG && !CE;
            constexpr int L = two ? 512 : decltype(lanes)::value, E = two ? 64 : decltype(ept)::value;
            constexpr int B = L < 256 ? 256 : L;
            const int64_t grid = (lines + B / L - 1) / (B / L);
            if (!grid_ok(grid)) return ZENU_ERR_UNSUPPORTED;
            auto go = [&](auto nt_c, auto store_c) {
                softmax_rows_kernel<T, CE, decltype(nt_c)::value, decltype(store_c)::value, LONG, L, E><<<(unsigned)grid, B, 0, s>>>(
                    x, y, lines, g.R, target, rowloss, zmath::ExpLog<T>());
            };
            if (!nt) {
                go(std::false_type(), std::integral_constant<int, kStorePlain>());
            } else if constexpr (CE || LONG) {   // (the loss's probabilities are read again by its backward pass; a long row's by itself)
                go(std::true_type(), std::integral_constant<int, kStorePlain>());
            } else {
                // How a streamed row is stored (us, softmax / the backward pass that reads it again): past the caches (`sc1
                // nt`) the ragged ends of rows, lines that two rows share, are written in part, and a burst of whole rows
                // meets a busy memory.  Plainly [4096,4003] f32 takes 28 / 32 (35 / 34 past the caches, 35 / 31 written
                // through), [2048,32003] 106 / 126 (112 / 137), [2048,4003] f64 27 / 32 (32 / 34).  Whole rows are written
                // through: [4096,16384] 91 / 119 (99 / 134; 89 / 126 plainly), [1024,16000] 25 / 32 (24 / 35; 26 / 32).  A
                // small result, or one batch of workgroups, still waits at its end for what is dirty in the L2 then:
                // [300,32003] 27 us plainly, 25 past the caches, [16384,300] 15.8 and 14.2.
                if (L >= 512 && whole) go(std::true_type(), std::integral_constant<int, L >= 512 ? kStoreThrough : kStorePlain>());
                else if (lines >= 4 * (int64_t)device_info().num_cus && lines * g.R * (int64_t)sizeof(T) >= kStreamBytes)
                    go(std::true_type(), std::integral_constant<int, kStorePlain>());
                else go(std::true_type(), std::integral_constant<int, kStoreStream>());
            }
            return ZENU_OK;
        });
        if (rc) return rc;
    }
    ZENU_LAUNCH_CHECK();
    return ZENU_OK;
}

template <typename T, bool CE>
int softmax_backward_launch(const T *y, const T *gy_or_target, T *gx, Geometry g, const T *gout, T neg_n,
                            hipStream_t s, T *colsum = nullptr)
{
    const int64_t lines = g.outer * g.inner;
    if (colsum && !(g.inner == 1 && g.R <= kLineRegs && lines <= kHeadLines)) return ZENU_ERR_UNSUPPORTED;
    if constexpr (CE) {
        if (g.inner == 1 && g.R <= kLineRegs && lines <= kHeadLines) {           // a classifier head: four lanes per line
            ce_head_backward_kernel<T><<<1, kHeadBlock, 0, s>>>(y, gy_or_target, gx, lines, g.R, gout, neg_n, colsum);
            ZENU_LAUNCH_CHECK();
            return ZENU_OK;
        }
    }
    if (g.inner != 1 || g.R <= kLineMaxR) {
        int own = line_own(lines, g.R, kMost<T>);
        if (own == 0) own = line_own(lines, g.R, 32);
        if (own == 0) {
            const int64_t blocks = (lines + kBlock - 1) / kBlock;
            if (!grid_ok(blocks)) return ZENU_ERR_UNSUPPORTED;
            softmax_bwd_long_lines_kernel<T><<<(unsigned)blocks, kBlock, 0, s>>>(y, gy_or_target, gx, lines, g.R, g.inner);
        } else {
            const LineGrid lg(lines, g.R, own, false);
            if (!grid_ok(lg.blocks)) return ZENU_ERR_UNSUPPORTED;
            with_own<32>(own, [&](auto o) {
                constexpr int OWN = decltype(o)::value;
                auto go = [&](auto mode_c) {
                    constexpr int MODE = decltype(mode_c)::value;
                    softmax_bwd_lines_kernel<T, CE, OWN, MODE><<<(unsigned)lg.blocks, lg.threads(), MODE == kLinesStaged ? lg.template staged_bytes<T, OWN>(g.R) : 0, s>>>(
                        y, gy_or_target, gx, lines, (int)g.R, g.inner, lg.waves, gout, neg_n);
                };
                if constexpr (CE) go(std::integral_constant<int, kLinesDirect>());
                else with_line_mode<OWN <= kMost<T>>(line_mode(g, false, sizeof(T)), go);   // (staged rows are short)
                return 0;
            });
        }
    } else {
        // y was written just before: loads without the hint find what the caches still hold of it ([4096,1000] f32 10.3 us
        // with the hint, 8.9 without; [16384,300] 11.9 / 9.7; level at 33 MB a tensor)
        const bool nt = lines * g.R * (int64_t)sizeof(T) >= kStreamBytes;
        const int rc = with_row_shape<VecOf<T>::N, kMost<T>>(g.R, [&](auto lanes, auto ept, auto is_long) -> int {
            constexpr int L = decltype(lanes)::value, E = decltype(ept)::value;
            constexpr bool LONG = decltype(is_long)::value;
            constexpr int B = L < 256 ? 256 : L;
            const int64_t grid = (lines + B / L - 1) / (B / L);
            if (!grid_ok(grid)) return ZENU_ERR_UNSUPPORTED;
            if (nt) softmax_bwd_rows_kernel<T, CE, true, LONG, L, E><<<(unsigned)grid, B, 0, s>>>(y, gy_or_target, gx, lines, g.R, gout, neg_n);
            else    softmax_bwd_rows_kernel<T, CE, false, LONG, L, E><<<(unsigned)grid, B, 0, s>>>(y, gy_or_target, gx, lines, g.R, gout, neg_n);
            return ZENU_OK;
        });
        if (rc) return rc;
    }
    ZENU_LAUNCH_CHECK();
    return ZENU_OK;
}

template <typename T>
int softmax_t(int dtype, const zenu_tensor_t &to, const zenu_tensor_t &src, int axis, hipStream_t s)
{
    if (num_elm(src) == 0) return ZENU_OK;
    ContigIn<T> in(src, dtype, s);
    if (in.status) return in.status;
    ContigOut<T> out(to, dtype, s);
    if (out.status) return out.status;
    int rc = softmax_forward_launch<T, false>(in.ptr, out.ptr, geometry(src, axis), nullptr, nullptr, s);
    return rc ? rc : out.finish();
}

template <typename T>
int softmax_backward_t(int dtype, const zenu_tensor_t &gx, const zenu_tensor_t &y, const zenu_tensor_t &gy,
                       int axis, hipStream_t s)
{
    if (num_elm(y) == 0) return ZENU_OK;
    ContigIn<T> yin(y, dtype, s);
    if (yin.status) return yin.status;
    ContigIn<T> gin(gy, dtype, s);
    if (gin.status) return gin.status;
    ContigOut<T> out(gx, dtype, s);
    if (out.status) return out.status;
    int rc = softmax_backward_launch<T, false>(yin.ptr, gin.ptr, out.ptr, geometry(y, axis), nullptr, (T)0, s);
    return rc ? rc : out.finish();
}

template <typename T>
int cross_entropy_t(int dtype, const zenu_tensor_t &loss, const zenu_tensor_t &prob, const zenu_tensor_t &pred,
                    const zenu_tensor_t &ans, hipStream_t s)
{
    const int64_t n = pred.shape[0];
    if (num_elm(pred) == 0) return ZENU_ERR_SHAPE;
    ContigIn<T> in(pred, dtype, s);
    if (in.status) return in.status;
    ContigIn<T> tin(ans, dtype, s);
    if (tin.status) return tin.status;
    ContigOut<T> out(prob, dtype, s);
    if (out.status) return out.status;
    // n = T::from_usize(rows); Variable::from(-n)  (cross_entropy.rs:20-21)
    const T neg_n = -(T)n;
    if (ce_single_workgroup(geometry(pred, 1))) {   // a classifier head's batch: probabilities and loss in one launch
        int rc1 = softmax_forward_launch<T, true>(in.ptr, out.ptr, geometry(pred, 1), tin.ptr, nullptr, s,
                                                  static_cast<T *>(loss.ptr), neg_n);
        return rc1 ? rc1 : out.finish();
    }
    Workspace rows((size_t)n * sizeof(T), s);
    if (rows.status) return rows.status;
    T *rowloss = static_cast<T *>(rows.ptr);
    int rc = softmax_forward_launch<T, true>(in.ptr, out.ptr, geometry(pred, 1), tin.ptr, rowloss, s);
    if (rc) return rc;
    if (n <= 65536) {
        ce_finalize_kernel<T><<<1, kBlock, 0, s>>>(rowloss, n, static_cast<T *>(loss.ptr), neg_n);
        ZENU_LAUNCH_CHECK();
    } else {
        Workspace tot(sizeof(T), s);
        if (tot.status) return tot.status;
        const int64_t shape1[1] = {n};
        zenu_tensor_t rv = default_view(rowloss, 1, shape1);
        zenu_tensor_t tv = default_view(tot.ptr, 0, nullptr);
        rc = zenu_hip_sum_all(dtype, tot.ptr, &rv, reinterpret_cast<zenu_stream_t>(s));
        if (!rc) rc = zenu_hip_binary_scalar(ZENU_DIV, dtype, &loss, &tv, (double)neg_n, reinterpret_cast<zenu_stream_t>(s));
        if (rc) return rc;
    }
    return out.finish();
}

template <typename T>
int cross_entropy_backward_t(int dtype, const zenu_tensor_t &gpred, const zenu_tensor_t &prob,
                             const zenu_tensor_t &ans, const zenu_tensor_t *gloss, hipStream_t s,
                             const zenu_tensor_t *gbias = nullptr)
{
    if (num_elm(prob) == 0) return gbias ? ZENU_ERR_SHAPE : ZENU_OK;
    ContigIn<T> yin(prob, dtype, s);
    if (yin.status) return yin.status;
    ContigIn<T> tin(ans, dtype, s);
    if (tin.status) return tin.status;
    ContigOut<T> out(gpred, dtype, s);
    if (out.status) return out.status;
    const T neg_n = -(T)prob.shape[0];
    const T *gout = gloss ? static_cast<const T *>(gloss->ptr) : nullptr;
    T *colsum = gbias ? static_cast<T *>(gbias->ptr) : nullptr;
    int rc = softmax_backward_launch<T, true>(yin.ptr, tin.ptr, out.ptr, geometry(prob, 1), gout, neg_n, s, colsum);
    return rc ? rc : out.finish();
}

template <typename T>
int bias_relu_t(int dtype, const zenu_tensor_t *pre, const zenu_tensor_t &act, const zenu_tensor_t &z,
                const zenu_tensor_t &bias, double alpha, hipStream_t s)
{
    constexpr int VEC = VecOf<T>::N;
    const int64_t n = num_elm(z);
    if (n == 0) return ZENU_OK;
    const int64_t F = bias.shape[0];
    ContigIn<T> zin(z, dtype, s);
    if (zin.status) return zin.status;
    ContigIn<T> bin(bias, dtype, s);
    if (bin.status) return bin.status;
    ContigOut<T> aout(act, dtype, s);
    if (aout.status) return aout.status;
    // `pre` is optional; when absent its ContigOut wraps `act` and is never written or finished
    ContigOut<T> pout(pre ? *pre : act, dtype, s);
    if (pre && pout.status) return pout.status;
    T *pp = pre ? pout.ptr : nullptr;
    const bool nt = n * (int64_t)sizeof(T) * (pp ? 3 : 2) >= kStreamBytes;
    const int64_t packs = F / VEC;
    const T al = (T)alpha;
    const int64_t grid = (n + kTileLanes * VEC - 1) / (kTileLanes * VEC);
    if (grid > 0x7fffffffLL) return ZENU_ERR_UNSUPPORTED;
    const unsigned g = (unsigned)grid;
    if (F % (VEC * kTileLanes) == 0) {
        const uint32_t tiles = (uint32_t)(packs / kTileLanes);
        if (nt) bias_relu_tile_kernel<T, VEC, true><<<g, kTileLanes, 0, s>>>(zin.ptr, bin.ptr, pp, aout.ptr, tiles, al);
        else    bias_relu_tile_kernel<T, VEC, false><<<g, kTileLanes, 0, s>>>(zin.ptr, bin.ptr, pp, aout.ptr, tiles, al);
    } else if (n < ((int64_t)1 << 32) - 65536) {
        const uint32_t n32 = (uint32_t)n, f32 = (uint32_t)F;
        if (nt) bias_relu_kernel<T, VEC, true, uint32_t><<<g, kTileLanes, 0, s>>>(zin.ptr, bin.ptr, pp, aout.ptr, n32, f32, al);
        else    bias_relu_kernel<T, VEC, false, uint32_t><<<g, kTileLanes, 0, s>>>(zin.ptr, bin.ptr, pp, aout.ptr, n32, f32, al);
    } else {
        bias_relu_kernel<T, VEC, true, uint64_t><<<g, kTileLanes, 0, s>>>(zin.ptr, bin.ptr, pp, aout.ptr, (uint64_t)n, (uint64_t)F, al);
    }
    ZENU_LAUNCH_CHECK();
    int rc = aout.finish();
    if (!rc && pre) rc = pout.finish();
    return rc;
}

int check_all(const zenu_tensor_t *const *ts, int n)
{
    for (int i = 0; i < n; i++) {
        if (!ts[i]) return ZENU_ERR_ARG;
        int rc = validate_tensor(ts[i]);
        if (rc) return rc;
    }
    return ensure_init();
}

}  // namespace
}  // namespace zenu

using namespace zenu;

extern "C" {

int zenu_hip_softmax(int dtype, const zenu_tensor_t *to, const zenu_tensor_t *src, int axis, zenu_stream_t stream)
{
    const zenu_tensor_t *ts[] = {to, src};
    int rc = check_all(ts, 2);
    if (rc) return rc;
    if (axis < 0 || axis >= src->ndim) return ZENU_ERR_ARG;      // "axis must be less than the number of dimensions"
    if (!same_shape(*to, *src)) return ZENU_ERR_SHAPE;           // "softmax shape mismatch"
    if (dtype == ZENU_F32) return softmax_t<float>(dtype, *to, *src, axis, as_stream(stream));
    if (dtype == ZENU_F64) return softmax_t<double>(dtype, *to, *src, axis, as_stream(stream));
    return ZENU_ERR_ARG;
}

int zenu_hip_softmax_backward(int dtype, const zenu_tensor_t *gx, const zenu_tensor_t *y, const zenu_tensor_t *gy,
                              int axis, zenu_stream_t stream)
{
    const zenu_tensor_t *ts[] = {gx, y, gy};
    int rc = check_all(ts, 3);
    if (rc) return rc;
    if (axis < 0 || axis >= y->ndim) return ZENU_ERR_ARG;
    if (!same_shape(*gx, *y) || !same_shape(*gy, *y)) return ZENU_ERR_SHAPE;
    if (dtype == ZENU_F32) return softmax_backward_t<float>(dtype, *gx, *y, *gy, axis, as_stream(stream));
    if (dtype == ZENU_F64) return softmax_backward_t<double>(dtype, *gx, *y, *gy, axis, as_stream(stream));
    return ZENU_ERR_ARG;
}

int zenu_hip_softmax_cross_entropy(int dtype, const zenu_tensor_t *loss, const zenu_tensor_t *prob,
                                   const zenu_tensor_t *pred, const zenu_tensor_t *ans, zenu_stream_t stream)
{
    const zenu_tensor_t *ts[] = {loss, prob, pred, ans};
    int rc = check_all(ts, 4);
    if (rc) return rc;
    if (pred->ndim != 2 || loss->ndim != 0) return ZENU_ERR_SHAPE;   // softmax(pred, 1), sum_to(.., [])
    if (!same_shape(*prob, *pred) || !same_shape(*ans, *pred)) return ZENU_ERR_SHAPE;
    if (dtype == ZENU_F32) return cross_entropy_t<float>(dtype, *loss, *prob, *pred, *ans, as_stream(stream));
    if (dtype == ZENU_F64) return cross_entropy_t<double>(dtype, *loss, *prob, *pred, *ans, as_stream(stream));
    return ZENU_ERR_ARG;
}

int zenu_hip_softmax_cross_entropy_backward(int dtype, const zenu_tensor_t *gpred, const zenu_tensor_t *prob,
                                            const zenu_tensor_t *ans, const zenu_tensor_t *gloss,
                                            zenu_stream_t stream)
{
    const zenu_tensor_t *ts[] = {gpred, prob, ans};
    int rc = check_all(ts, 3);
    if (rc) return rc;
    if (gloss && (validate_tensor(gloss) || gloss->ndim != 0)) return ZENU_ERR_SHAPE;
    if (prob->ndim != 2) return ZENU_ERR_SHAPE;
    if (!same_shape(*gpred, *prob) || !same_shape(*ans, *prob)) return ZENU_ERR_SHAPE;
    if (dtype == ZENU_F32) return cross_entropy_backward_t<float>(dtype, *gpred, *prob, *ans, gloss, as_stream(stream));
    if (dtype == ZENU_F64) return cross_entropy_backward_t<double>(dtype, *gpred, *prob, *ans, gloss, as_stream(stream));
    return ZENU_ERR_ARG;
}

int zenu_hip_softmax_cross_entropy_backward_bias_grad(int dtype, const zenu_tensor_t *gpred, const zenu_tensor_t *gbias,
                                                      const zenu_tensor_t *prob, const zenu_tensor_t *ans,
                                                      const zenu_tensor_t *gloss, zenu_stream_t stream)
{
    const zenu_tensor_t *ts[] = {gpred, gbias, prob, ans};
    int rc = check_all(ts, 4);
    if (rc) return rc;
    if (gloss && (validate_tensor(gloss) || gloss->ndim != 0)) return ZENU_ERR_SHAPE;
    if (prob->ndim != 2) return ZENU_ERR_SHAPE;
    if (!same_shape(*gpred, *prob) || !same_shape(*ans, *prob)) return ZENU_ERR_SHAPE;
    if (gbias->ndim < 1 || gbias->shape[gbias->ndim - 1] != prob->shape[1] || num_elm(*gbias) != prob->shape[1])
        return ZENU_ERR_SHAPE;
    if (dtype != ZENU_F32 && dtype != ZENU_F64) return ZENU_ERR_ARG;
    const size_t esz = dtype == ZENU_F32 ? 4 : 8;
    const size_t gb_bytes = (size_t)num_elm(*gbias) * esz;
    if (view_overlaps(*gpred, esz, gbias->ptr, gb_bytes) || view_overlaps(*prob, esz, gbias->ptr, gb_bytes) ||
        view_overlaps(*ans, esz, gbias->ptr, gb_bytes))
        return ZENU_ERR_ARG;
    // a classifier head's batch (every line in one workgroup, at most 16 classes): gradient and its column
    // sums in one launch; anything else is the two calls it stands for
    if (prob->shape[0] <= kBlock && prob->shape[1] <= kLineRegs && is_default_stride_strict(*gbias)) {
        rc = dtype == ZENU_F32
                 ? cross_entropy_backward_t<float>(dtype, *gpred, *prob, *ans, gloss, as_stream(stream), gbias)
                 : cross_entropy_backward_t<double>(dtype, *gpred, *prob, *ans, gloss, as_stream(stream), gbias);
        if (rc != ZENU_ERR_UNSUPPORTED) return rc;
    }
    rc = zenu_hip_softmax_cross_entropy_backward(dtype, gpred, prob, ans, gloss, stream);
    if (rc) return rc;
    return zenu_hip_sum_to(dtype, gbias, gpred, stream);
}

int zenu_hip_bias_add_relu(int dtype, const zenu_tensor_t *pre, const zenu_tensor_t *act, const zenu_tensor_t *z,
                           const zenu_tensor_t *bias, double alpha, zenu_stream_t stream)
{
    const zenu_tensor_t *ts[] = {act, z, bias};
    int rc = check_all(ts, 3);
    if (rc) return rc;
    if (pre && validate_tensor(pre)) return ZENU_ERR_ARG;
    if (z->ndim < 1 || bias->ndim != 1 || bias->shape[0] != z->shape[z->ndim - 1]) return ZENU_ERR_SHAPE;
    if (!same_shape(*act, *z) || (pre && !same_shape(*pre, *z))) return ZENU_ERR_SHAPE;
    if (dtype == ZENU_F32) return bias_relu_t<float>(dtype, pre, *act, *z, *bias, alpha, as_stream(stream));
    if (dtype == ZENU_F64) return bias_relu_t<double>(dtype, pre, *act, *z, *bias, alpha, as_stream(stream));
    return ZENU_ERR_ARG;
}

}  // extern "C"
