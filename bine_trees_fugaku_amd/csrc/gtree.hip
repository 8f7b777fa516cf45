// gtree.hip -- gather-reduce over general trees: the schedules of tori that are no powers of two.
//
// An item's tree comes as its leaves in postfix order, each with the number of additions that follow it, cut into one
// subtree per wave.  A wave loads eight leaves at a time and evaluates them on a stack; the subtree sums meet in LDS,
// where every wave joins them in tree order, and the waves share the outputs.  Every addition is one of the schedule's,
// so the bits are those of its steps.  Units and overlapping ends are those of the narrow kernel; each wave holds the
// whole tile, one unit per lane, so all of an item's loads are done before its first store (in-place lists rely on it).
//
// What bounds it: at small sizes the latency of two rounds of loads and the instructions of the stack, which is why
// the topmost value stays apart (half the leaves are added to it at once and touch no level) and the levels are
// registers picked by uniform branches; selects over all levels took twice the time (100 ranks of 1000 elements 23.0
// against 13.0 us with four waves).  At large sizes memory: 100 ranks of 2097152 fp32 elements (1.7 GB) move at 4.5
// TB/s.  Against the schedule's steps, GPU time per call, fp32: 36 ranks of 131072 84.8 -> 12.8 us, of 2097152
// 423 -> 138; 100 ranks of 32768 109 -> 12.9; 12 ranks of 1000 25 -> 4.0.  Stacks of more than six values run an
// instantiation of their own, whose code no longer fits the instruction cache: 0.66 us for each leaf of a wave (a ring of
// 400 ranks of 403 262 -> 83).  Evaluated with the levels by lane address it takes half of that at small sizes and 5 to
// 20 % more at middle and large ones.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gred_dev.hpp"

namespace bine {

namespace {

// D values in registers.  Every access names its level at compile time, chosen by branches on counts that are the same
// for the whole wave.  The empty asm keeps those branches apart: merged, they would index the levels, in memory.
template <typename T, int D, int L = 0>
struct Slots {
    Vec<T> x;
    Slots<T, D, L + 1> above;
    __device__ __forceinline__ void put(const Vec<T>& v, uint32_t level) {
        if (level == L) {
            x = v;
            asm volatile("" : "+v"(x.raw));
        } else {
            above.put(v, level);
        }
    }
    // add the values of levels [low, high) to v, the highest first
    __device__ __forceinline__ void take(Vec<T>& v, uint32_t low, uint32_t high) const {
        if (high > L + 1) above.take(v, low, high);
        if (L >= low && L < high) v = vadd<T>(x, v);
    }
};
template <typename T, int D>
struct Slots<T, D, D> {
    __device__ __forceinline__ void put(const Vec<T>&, uint32_t) {}
    __device__ __forceinline__ void take(Vec<T>&, uint32_t, uint32_t) const {}
};

// Push x on a stack of `held` values (the topmost in v, the others in the slots) and make `pops` additions of the two
// topmost values.
template <typename T, int D>
__device__ __forceinline__ void stack_step(Slots<T, D>& s, Vec<T>& v, uint32_t& held, const Vec<T>& x, uint32_t pops) {
    if (pops == 0) {
        if (held) s.put(v, held - 1);
        v = x;
    } else {
        v = vadd<T>(v, x);
        if (pops > 1) s.take(v, held - pops, held - 1);
    }
    held += 1 - pops;
}

// One item: `units` lanes of each wave hold a vector, or a single element where the block is shorter than one (ONE).
template <typename T, bool ONE, int D>
__device__ __forceinline__ void tree_item(const GredItem& it, const Table& t, const PoolEntry* pool, Vec<T>* lds) {
    constexpr uint32_t VE = Vec<T>::N;
    const uint32_t units = ONE ? it.n : (it.n + VE - 1) / VE;
    const uint32_t nw = blockDim.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t parts = it.lg;
    const BINE_CONST PoolEntry* cut = cptr(pool + it.leaf_off);
    const BINE_CONST PoolEntry* outs = cptr(pool + it.out_off);
    const bool ok = lane < units;
    const uint32_t uu = ok ? lane : units - 1;
    const uint32_t off = (ONE ? uu : uu + 1 < units ? uu * VE : it.n - VE) * (uint32_t)sizeof(T);
    const uint64_t delta = it.delta;
    auto load = [&](const PoolEntry& e) __attribute__((always_inline)) {
        const char* p = t.at(e.rb & 0xF0FFFFFFu, (uint64_t)e.off + delta, sizeof(T)) + off;
        if (!ONE) return load_unit(p, (Vec<T>*)nullptr);
        Vec<T> r{};
        const T x = load_unit(p, (T*)nullptr);
        __builtin_memcpy(&r.raw, &x, sizeof(T));
        return r;
    };
    Vec<T> v{};
    if (wave < parts) {
        uint32_t first = parts;
        for (uint32_t w = 0; w < wave; ++w) first += (cload(cut + w).rb + 7) & ~7u;
        const BINE_CONST PoolEntry* my = cut + first;
        const uint32_t n = cload(cut + wave).rb;
        Slots<T, D> slots;
        uint32_t held = 0;
        PoolEntry next[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) next[i] = cload(my + i);
        for (uint32_t k = 0; k < n; k += 8) {  // the pool holds whole groups of eight; those past the end are unused
            PoolEntry e[8];
            Vec<T> x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] = next[i];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = load(e[i]);
            if (k + 4 < n) {
#pragma unroll
                for (int i = 4; i < 8; ++i) x[i] = load(e[i]);
            }
            if (k + 8 < n) {  // fetched while this group's values are on their way
#pragma unroll
                for (int i = 0; i < 8; ++i) next[i] = cload(my + k + 8 + i);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (k + i < n) stack_step(slots, v, held, x[i], (e[i].rb >> 24) & 15u);
        }
        if (nw > 1) lds[wave * 64 + lane] = v;
    }
    if (nw > 1) {
        __syncthreads();
        Slots<T, D> slots;
        uint32_t held = 0;
        for (uint32_t w = 0; w < parts; w += 4) {
            Vec<T> x[4];
            uint32_t pops[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t k = w + i < parts ? w + i : w;
                x[i] = lds[k * 64 + lane];
                pops[i] = cload(cut + k).off;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (w + i < parts) stack_step(slots, v, held, x[i], pops[i]);
        }
    }
    for (uint32_t o = wave; o < it.nouts; o += nw) {
        const PoolEntry e = cload(outs + o);
        char* p = t.at(e.rb, (uint64_t)e.off + delta, sizeof(T)) + off;
        if (!ok) continue;
        if (ONE) {
            T x;
            __builtin_memcpy(&x, &v.raw, sizeof(T));
            store_unit(p, x);
        } else {
            store_unit(p, v);
        }
    }
}

template <typename T, int D, bool BATCH>
__global__ void __launch_bounds__(512) gtree_kernel(const GredItem* __restrict__ items, const PoolEntry* __restrict__ pool,
                                                    BufTable tab, const BufTable* __restrict__ tabs) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const GredItem it = cload(cptr(items + blockIdx.x));
    Table t;
    if (BATCH) {
        const BINE_CONST BufTable* bt = cptr(tabs + it.bucket);
        t = Table{bt->base[0], bt->base[1], bt->base[2], bt->base[3], bt->stride[0], bt->stride[1], bt->stride[2], bt->stride[3]};
    } else {
        t = Table{tab.base[0], tab.base[1], tab.base[2], tab.base[3], tab.stride[0], tab.stride[1], tab.stride[2], tab.stride[3]};
    }
    Vec<T>* lds = reinterpret_cast<Vec<T>*>(lds_raw);
    if (it.n >= Vec<T>::N)
        tree_item<T, false, D>(it, t, pool, lds);
    else
        tree_item<T, true, D>(it, t, pool, lds);
}

template <typename T, int D>
hipError_t launch_d(const GredItem* items, uint32_t n, const PoolEntry* pool, const BufTable& tab, const BufTable* tabs,
                    bool batch, int waves, hipStream_t st) {
    const size_t lds = (size_t)waves * 64 * 16;
    if (batch)
        hipLaunchKernelGGL((gtree_kernel<T, D, true>), dim3(n), dim3(64 * waves), lds, st, items, pool, tab, tabs);
    else
        hipLaunchKernelGGL((gtree_kernel<T, D, false>), dim3(n), dim3(64 * waves), lds, st, items, pool, tab, tabs);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_t(const GredItem* items, uint32_t n, const PoolEntry* pool, const BufTable& tab, const BufTable* tabs,
                    bool batch, int waves, int stack, hipStream_t st) {
    return stack <= kShallowStack ? launch_d<T, kShallowStack - 1>(items, n, pool, tab, tabs, batch, waves, st)
                                  : launch_d<T, kMaxTreeStack - 1>(items, n, pool, tab, tabs, batch, waves, st);
}

}  // namespace

// One workgroup per item; up to 8 waves; stack: the deepest that a subtree's evaluation needs (lower_trees).
hipError_t launch_gtree(int dtype, const GredItem* items, uint32_t n, const PoolEntry* pool, const BufTable& tab,
                        const BufTable* tabs, bool batch, int waves, int stack, hipStream_t st) {
    if (n == 0) return hipSuccess;
    if (waves < 1 || waves > 8 || stack > kMaxTreeStack) return hipErrorInvalidValue;
    switch (dtype) {
    case 0: return launch_t<int32_t>(items, n, pool, tab, tabs, batch, waves, stack, st);
    case 1: return launch_t<int64_t>(items, n, pool, tab, tabs, batch, waves, stack, st);
    case 2: return launch_t<float>(items, n, pool, tab, tabs, batch, waves, stack, st);
    case 3: return launch_t<double>(items, n, pool, tab, tabs, batch, waves, stack, st);
    case 4: return launch_t<int8_t>(items, n, pool, tab, tabs, batch, waves, stack, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace bine
