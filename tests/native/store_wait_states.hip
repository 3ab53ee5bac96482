// Compiled by tests/test_host_native.py to assembly, never run: the written-out stores of vecmem.hpp with a scalar
// base address that a vector instruction produces just before.
#include "vecmem.hpp"

using namespace zenu;

template <typename T, int N> __global__ void store_at_read_lane(T *const *rows, const T *x)
{
    const Pack<T, N> v = load_pack<T, N, false>(x + threadIdx.x * N);
    const uint64_t a = reinterpret_cast<uint64_t>(rows[threadIdx.x]);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    store_pack_wt_at<T, N>(reinterpret_cast<T *>(((uint64_t)hi << 32) | lo), (int)threadIdx.x * N, v);
}
template __global__ void store_at_read_lane<float, 4>(float *const *, const float *);
template __global__ void store_at_read_lane<double, 2>(double *const *, const double *);
