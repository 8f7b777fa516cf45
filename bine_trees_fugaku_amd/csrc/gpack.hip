// gpack.hip -- short copies, many to a workgroup: the alltoall of small messages, and scatters and gathers of short
// blocks, or of blocks up to 20 KiB that are no whole number of vectors.
//
// An item is a grid of t1 x t2 copies of one length whose source and destination both advance by a fixed (rank, offset)
// step along either axis (GredItem), so no pool entry is read per copy: an alltoall is one such grid of P x P copies, a
// transpose of blocks.  The lanes of a workgroup run over (copy along t1, units of the copy), so that consecutive lanes
// write consecutive destination blocks; a grid is about as long along each axis, so that the lines it reads are used
// whole too.  A unit is 16, 8, 4 or 1 bytes at any address; a copy's last unit starts early so that it ends at the
// copy's end.
//
// What bounds it: at 64 bytes a pair on 512 ranks (33.6 MB moved) it runs at 4.3 TB/s, 7.8 us of GPU time against 241
// when every two copies had a workgroup of their own, with 64 bytes of work items and pool entries for them; below
// that, the latency of one load and store.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gred_dev.hpp"

namespace bine {

namespace {

typedef unsigned int u2w __attribute__((ext_vector_type(2)));
template <int N>
struct UnitOf;
template <>
struct UnitOf<16> {
    typedef u4 type;
    typedef u4b mem;
};
template <>
struct UnitOf<8> {
    typedef u2w type;
    typedef u2w mem __attribute__((aligned(1)));
};
template <>
struct UnitOf<4> {
    typedef uint32_t type;
    typedef uint32_t mem __attribute__((aligned(1)));
};
template <>
struct UnitOf<1> {
    typedef uint8_t type;
    typedef uint8_t mem;
};

template <int N>
__device__ __forceinline__ void pack_item(const GredItem& it, const Table& t, const PoolEntry* pool, uint32_t esize) {
    typedef typename UnitOf<N>::type U;
    typedef typename UnitOf<N>::mem M;
    const BINE_CONST PoolEntry* rec = cptr(pool + it.leaf_off);
    const PoolEntry l0 = cload(rec), o0 = cload(rec + 1), l1 = cload(rec + 2), o1 = cload(rec + 3), l2 = cload(rec + 4),
                    o2 = cload(rec + 5);
    const uint32_t bytes = it.n * esize, upc = (bytes + N - 1) / N;
    const uint32_t t1 = it.pad & 0xFFFFu, t2 = it.pad >> 16, total = upc * t1 * t2;
    constexpr int V = 4;  // units per lane in flight
    for (uint32_t base = 0; base < total; base += V * blockDim.x) {
        U x[V];
        char* dst[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t q = base + v * blockDim.x + threadIdx.x;
            if (q < total) {
                const uint32_t j = q / upc, u = q - j * upc, j2 = j / t1, j1 = j - j2 * t1;
                const uint32_t at = (u + 1) * N <= bytes ? u * N : bytes - N;
                // 32-bit sums: a step backwards is held modulo 2^32
                const char* src = t.at(l0.rb + l1.rb * j1 + l2.rb * j2, l0.off + l1.off * j1 + l2.off * j2, esize) + at;
                dst[v] = t.at(o0.rb + o1.rb * j1 + o2.rb * j2, o0.off + o1.off * j1 + o2.off * j2, esize) + at;
                x[v] = *gptr<const M>(src);
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (base + v * blockDim.x + threadIdx.x < total) *gptr<M>(dst[v]) = x[v];
    }
}

template <bool BATCH>
__global__ void __launch_bounds__(256) gpack_kernel(const GredItem* __restrict__ items, const PoolEntry* __restrict__ pool,
                                                    BufTable tab, const BufTable* __restrict__ tabs, uint32_t esize) {
    const GredItem it = cload(cptr(items + blockIdx.x));
    Table t;
    if (BATCH) {
        const BINE_CONST BufTable* bt = cptr(tabs + it.bucket);
        t = Table{bt->base[0], bt->base[1], bt->base[2], bt->base[3], bt->stride[0], bt->stride[1], bt->stride[2], bt->stride[3]};
    } else {
        t = Table{tab.base[0], tab.base[1], tab.base[2], tab.base[3], tab.stride[0], tab.stride[1], tab.stride[2], tab.stride[3]};
    }
    const uint32_t bytes = it.n * esize;
    if (bytes >= 16) pack_item<16>(it, t, pool, esize);
    else if (bytes >= 8) pack_item<8>(it, t, pool, esize);
    else if (bytes >= 4) pack_item<4>(it, t, pool, esize);
    else pack_item<1>(it, t, pool, esize);
}

}  // namespace

// One workgroup per item.
hipError_t launch_gpack(uint32_t esize, const GredItem* items, uint32_t n, const PoolEntry* pool, const BufTable& tab,
                        const BufTable* tabs, bool batch, hipStream_t st) {
    if (n == 0) return hipSuccess;
    if (batch)
        hipLaunchKernelGGL(gpack_kernel<true>, dim3(n), dim3(256), 0, st, items, pool, tab, tabs, esize);
    else
        hipLaunchKernelGGL(gpack_kernel<false>, dim3(n), dim3(256), 0, st, items, pool, tab, tabs, esize);
    return hipGetLastError();
}

}  // namespace bine
