// gnarrow.hip -- the gather-reduce kernel of small lists.
//
// gred_kernel gives a tile's elements to lanes and walks the tile's leaves (or its outputs) one after the other on
// every lane.  A block of ten elements with 512 leaves then keeps ten lanes busy for 64 dependent rounds of loads, and
// a 16 KiB broadcast to 511 partitions runs on five workgroups.  Here the lanes of a workgroup form a grid of W units
// (W the tile's units rounded up to a power of two) by S = threads / W segments: segment s reduces the s-th contiguous
// range of leaves, a whole subtree of the balanced tree, the subtree sums are joined pairwise in tree order (lane
// exchanges inside a wave, then LDS across the waves), and segment s stores the sum to the outputs s, s + S, ...
// The association is the tree's, element for element, as in gred_kernel.
//
// What bounds it is latency (work item, pool entry, leaf and store, one after the other), not bandwidth: eight loads in
// flight per lane and about eight stores keep each of these one round.  On one MI355X, GPU time per launch against
// gred_kernel's: allreduce of 5003 fp32 elements on 512 ranks (20.5 MB) 285 -> 13.2 us, bcast of 4099 on 512 ranks
// 169 -> 7 us, reduce 98 -> 7.5 us, allgather of 129 on 512 ranks 200 -> 39 us, allreduce of 1024 on 8 ranks
// 4.5 -> 2.9 us.  No scratch; 94 VGPRs.
//
// A unit is a 16-byte vector at whatever byte address its element falls on (the global memory serves any alignment);
// the last vector of a tile starts early so that it ends at the tile's end, and the elements it shares with the vector
// before it are computed twice and stored twice with the same bits.  Tiles shorter than one vector use single elements.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gred_dev.hpp"

namespace bine {

namespace {

// the value of lane (lane xor mask)
template <typename T>
__device__ __forceinline__ Vec<T> lane_xor(const Vec<T>& v, int mask) {
    Vec<T> r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.raw[i] = (unsigned)__shfl_xor((int)v.raw[i], mask, 64);
    return r;
}
template <typename T>
__device__ __forceinline__ T lane_xor(T v, int mask) {
    constexpr int N = sizeof(T) < 4 ? 1 : sizeof(T) / 4;
    int w[N] = {};
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = __shfl_xor(w[i], mask, 64);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// One item, U = Vec<T> or T; `units` <= blockDim.x, `step` elements per unit.
template <typename T, typename U, bool NT>
__device__ __forceinline__ void narrow_item(const GredItem& it, const Table& t, const PoolEntry* pool, uint32_t units,
                                            uint32_t step, U* lds) {
    const uint32_t lgT = 31u - (uint32_t)__builtin_clz(blockDim.x);
    const uint32_t lgW = units <= 1 ? 0 : 32u - (uint32_t)__builtin_clz(units - 1);
    const uint32_t W = 1u << lgW, lgS = lgT - lgW, S = 1u << lgS;
    const uint32_t lg = it.lg, nouts = it.nouts;
    const uint32_t u = threadIdx.x & (W - 1), seg = threadIdx.x >> lgW;
    // a lane past the last unit loads that unit again and stores nothing
    const uint32_t uu = u < units ? u : units - 1;
    const uint32_t first = step == 1 || uu + 1 < units ? uu * step : it.n - step;
    const uint64_t at = (uint64_t)it.delta + first;
    const BINE_CONST PoolEntry* leaves = cptr(pool + it.leaf_off);
    const BINE_CONST PoolEntry* outs = cptr(pool + it.out_off);
    constexpr int K = 4;  // output entries fetched together, the first ones before the leaves
    PoolEntry oe[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const uint32_t o = seg + j * S;
        oe[j] = cload(outs + (o < nouts ? o : 0));
    }
    auto load = [&](uint32_t k) __attribute__((always_inline)) {
        const PoolEntry e = cload(leaves + k);
        return load_unit<NT>(t.at(e.rb, (uint64_t)e.off + at, sizeof(T)), (U*)nullptr);
    };
    auto add = [](const U& a, const U& b) __attribute__((always_inline)) { return add_unit(a, b); };
    U v{};
    if (lg == 0) {
        v = load(0);
    } else {
        const uint32_t ls = lgS < lg ? lgS : lg;  // segments that hold leaves: 2^ls
        const uint32_t lgs = lg - ls;
        if (seg < (1u << ls)) v = tree_eval<U, 6, 8>(lgs, add, [&](uint32_t k) __attribute__((always_inline)) { return load((seg << lgs) + k); });
        const uint32_t q = lgW >= 6 ? 0 : (ls < 6 - lgW ? ls : 6 - lgW);  // tree levels joined inside a wave
        for (uint32_t l = 0; l < q; ++l) v = add(v, lane_xor(v, (int)(W << l)));
        if (seg < (1u << ls) && (seg & ((1u << q) - 1)) == 0) lds[((seg >> q) << lgW) + u] = v;
        __syncthreads();
        v = tree_eval<U, 2, 8>(ls - q, add, [&](uint32_t k) __attribute__((always_inline)) { return lds[(k << lgW) + u]; });
    }
    if (u >= units) return;
    for (uint32_t o = seg; o < nouts;) {
#pragma unroll
        for (int j = 0; j < K; ++j)
            if (o + j * S < nouts) store_unit<NT>(t.at(oe[j].rb, (uint64_t)oe[j].off + at, sizeof(T)), v);
        o += K * S;
#pragma unroll
        for (int j = 0; j < K; ++j)
            if (o + j * S < nouts) oe[j] = cload(outs + o + j * S);
    }
}

template <typename T, bool BATCH, bool NT>
__global__ void __launch_bounds__(1024) gnarrow_kernel(const GredItem* __restrict__ items,
                                                       const PoolEntry* __restrict__ pool, BufTable tab,
                                                       const BufTable* __restrict__ tabs) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const GredItem it = cload(cptr(items + blockIdx.x));
    Table t;
    if (BATCH) {
        const BINE_CONST BufTable* bt = cptr(tabs + it.bucket);
        t = Table{bt->base[0], bt->base[1], bt->base[2], bt->base[3], bt->stride[0], bt->stride[1], bt->stride[2], bt->stride[3]};
    } else {
        t = Table{tab.base[0], tab.base[1], tab.base[2], tab.base[3], tab.stride[0], tab.stride[1], tab.stride[2], tab.stride[3]};
    }
    constexpr uint32_t VE = Vec<T>::N;
    if (it.n >= VE)
        narrow_item<T, Vec<T>, NT>(it, t, pool, (it.n + VE - 1) / VE, VE, reinterpret_cast<Vec<T>*>(lds_raw));
    else
        narrow_item<T, T, false>(it, t, pool, it.n, 1, reinterpret_cast<T*>(lds_raw));
}

template <typename T, bool NT>
hipError_t launch_t(const GredItem* items, uint32_t n, const PoolEntry* pool, const BufTable& tab,
                    const BufTable* tabs, bool batch, int threads, hipStream_t st) {
    const size_t lds = (size_t)threads * 16;
    if (batch)
        hipLaunchKernelGGL((gnarrow_kernel<T, true, NT>), dim3(n), dim3(threads), lds, st, items, pool, tab, tabs);
    else
        hipLaunchKernelGGL((gnarrow_kernel<T, false, NT>), dim3(n), dim3(threads), lds, st, items, pool, tab, tabs);
    return hipGetLastError();
}

}  // namespace

// stream: vectors are loaded and stored past the caches.  One workgroup of `threads` lanes per item; every item's units must fit the workgroup (lower_narrow).
hipError_t launch_gnarrow(int dtype, const GredItem* items, uint32_t n, const PoolEntry* pool, const BufTable& tab,
                          const BufTable* tabs, bool batch, int threads, bool stream, hipStream_t st) {
    if (n == 0) return hipSuccess;
    if (threads < 64 || threads > 1024 || (threads & (threads - 1))) return hipErrorInvalidValue;
#define BINE_NARROW(T)                                                                \
    return stream ? launch_t<T, true>(items, n, pool, tab, tabs, batch, threads, st)  \
                  : launch_t<T, false>(items, n, pool, tab, tabs, batch, threads, st)
    switch (dtype) {
    case 0: BINE_NARROW(int32_t);
    case 1: BINE_NARROW(int64_t);
    case 2: BINE_NARROW(float);
    case 3: BINE_NARROW(double);
    case 4: BINE_NARROW(int8_t);
    default: return hipErrorInvalidValue;
    }
#undef BINE_NARROW
}

}  // namespace bine
