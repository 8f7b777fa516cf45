// sim.hip -- link counting for the torus traffic simulation.
//
// Under dimension-ordered minimal routing a message crosses, per dimension,
// one contiguous run of links on one ring (the nodes that differ from its
// position only in that dimension), all in one direction.  So instead of one
// atomic add per hop, a run adds +1 at its first link and -1 just past its
// last (one more +1 at the ring's start when the run wraps round), in a
// difference array; a prefix sum along every ring and direction then turns the
// differences into the number of messages crossing each directed link.  The
// counts are the same integers a per-hop count gives (wrapping arithmetic
// modulo 2^32 cancels in the sums).
//
// A class's counters are counted and summed in LDS where they fit (sim_class); the passes over device memory below
// it serve larger tori.  Grids are sized per class: a table maps every workgroup to its class and to
// its block within the class, so small tori do not launch the largest torus's
// grid.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "sim_dest.hpp"
#include "sim_launch.hpp"

namespace bine {

using simd::SimCaseRec;
using simd::SimClassRec;

namespace {

// Node stride of dimension d (row-major, last dimension fastest).
__device__ __forceinline__ uint32_t dim_stride(const simd::TorusD& t, uint32_t d) {
    uint32_t s = 1;
#pragma unroll
    for (uint32_t i = 1; i < 3; ++i)
        if (i > d && i < t.nd) s *= t.dims[i];
    return s;
}

}  // namespace

// blocks of counters, and the statistics of all classes
__global__ void sim_zero(uint32_t* __restrict__ p, uint64_t n, uint32_t* __restrict__ hops, uint32_t* __restrict__ mx,
                         unsigned long long* __restrict__ sum, uint32_t ncls) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) p[i] = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ncls; i += (uint64_t)gridDim.x * blockDim.x) {
        hops[i] = 0;
        mx[i] = 0;
        sum[i] = 0;
    }
}

// Rank r's message of a class as difference updates: add(dd, node, dir, value) for every end of a run of links (node:
// the run's ring position, dd: its dimension, dir: 1 for the negative way).  Returns the length of the route.
template <typename Add>
__device__ __forceinline__ uint32_t route(const SimCaseRec& cs, const SimClassRec& c, uint32_t r, Add add) {
    uint32_t dst = simd::dest(cs.t, c.kind, c.d, c.k, r, cs.L);
    if (dst == 0xFFFFFFFFu || dst >= cs.t.size) return 0;
    uint32_t src = r;
    if (c.kind == 10) {  // simulator.py ids -> torus coordinates
        int a[3], b[3];
        simd::simpy_coords(cs.t, src, a);
        simd::simpy_coords(cs.t, dst, b);
        src = simd::ident(cs.t, a);
        dst = simd::ident(cs.t, b);
    }
    if (src == dst) return 0;
    int s[3], d[3];
    simd::coords(cs.t, src, s);
    simd::coords(cs.t, dst, d);
    const uint32_t nd = cs.t.nd;  // node strides as shifts; the last dimension's is 0
    const uint32_t t0 = simd::lg2(dim_stride(cs.t, 0)), t1 = simd::lg2(dim_stride(cs.t, 1));
    uint32_t hops = 0;
    // along dimension dd from position p to q; base: the ring's position 0, its nodes 2^stride apart
    auto leg = [&](uint32_t dd, int n, int p, int q, uint32_t base, uint32_t stride) __attribute__((always_inline)) {
        const int delta = simd::pm(q - p, n);
        if (!delta) return;
        const bool neg = 2 * delta > n;
        const int h = neg ? n - delta : delta;
        auto at = [&](int j, uint32_t v) __attribute__((always_inline)) { add(dd, base + ((uint32_t)j << stride), neg ? 1u : 0u, v); };
        // the run covers ring positions [lo, lo + h) (mod n): from p upwards, or the h positions ending at p
        const int lo = neg ? p - h + 1 : p;
        if (lo >= 0 && lo + h <= n) {
            at(lo, 1u);
            if (lo + h < n) at(lo + h, 0xFFFFFFFFu);
        } else {  // wraps: [lo mod n, n) and [0, (lo + h) mod n)
            at(lo < 0 ? lo + n : lo, 1u);
            at(0, 1u);
            at(lo + h - (lo < 0 ? 0 : n), 0xFFFFFFFFu);
        }
        hops += (uint32_t)h;
    };
    // dimension order: the dimensions before this one are at the destination, those after it still at the source
    leg(0, (int)cs.t.dims[0], s[0], d[0], ((uint32_t)s[1] << t1) + (uint32_t)s[2], t0);
    if (nd > 1) leg(1, (int)cs.t.dims[1], s[1], d[1], ((uint32_t)d[0] << t0) + (uint32_t)s[2], t1);
    if (nd > 2) leg(2, (int)cs.t.dims[2], s[2], d[2], ((uint32_t)d[0] << t0) + ((uint32_t)d[1] << t1), 0);
    return hops;
}

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

// A class in one workgroup: its counters, or those of one dimension where a class's do not fit (slices[b] = class,
// first dimension | last + 1 << 8), are cleared, counted and summed in LDS and written out once.  The counters of the
// five tori of the selector's held-out set (52 MB) took a clearing pass, two or three L2 atomics per message and
// dimension, and a strided read-modify-write pass over memory: 250 us per run, now 61 (one launch for each size of LDS
// need).  What is left is instructions: routing takes about half of it, the sums along rings a quarter (a dimension
// whose ring positions lie 64 nodes apart reads one bank with all lanes), clearing and writing the rest.
// Rings shorter than a wave are summed one to a lane, longer ones one to a wave, 64 positions at a time.
__global__ void __launch_bounds__(1024) sim_class(const SimCaseRec* __restrict__ cases, const SimClassRec* __restrict__ classes,
                          const uint2* __restrict__ slices, uint32_t* __restrict__ mult, uint32_t* __restrict__ max_hops,
                          uint32_t* __restrict__ max_mult, unsigned long long* __restrict__ sum_mult) {
    extern __shared__ __align__(16) uint32_t cnt[];
    __shared__ uint32_t s_max[16], s_hops[16];
    __shared__ unsigned long long s_sum[16];
    const uint2 sl = slices[blockIdx.x];
    const SimClassRec c = classes[sl.x];
    const SimCaseRec& cs = cases[c.case_idx];
    const simd::TorusD& t = cs.t;
    const uint32_t d0 = sl.y & 0xFFu, d1 = sl.y >> 8, w = d1 - d0, len = t.size * w * 2;
    const bool whole = w == t.nd;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, nw = blockDim.x >> 6;
    for (uint32_t i = tid; i < len; i += blockDim.x) cnt[i] = 0;
    __syncthreads();
    uint32_t hops = 0, mx = 0;
    unsigned long long sm = 0;
    for (uint32_t r = tid; r < t.size; r += blockDim.x) {
        const uint32_t h = route(cs, c, r, [&](uint32_t dd, uint32_t node, uint32_t dir, uint32_t v) {
            if (dd >= d0 && dd < d1) atomicAdd(&cnt[(__umul24(node, w) + dd - d0) * 2 + dir], v);
        });
        hops = h > hops ? h : hops;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t dd = 0; dd < 3; ++dd) {
        if (dd < d0 || dd >= d1) continue;
        const uint32_t n = t.dims[dd], stride = dim_stride(t, dd), lines = 2 * (t.size >> simd::lg2(n)), ls = simd::lg2(stride);  // rings x directions
        const bool long_ring = n >= 64;
        for (uint32_t q = long_ring ? wave : tid; q < lines; q += long_ring ? nw : blockDim.x) {
            const uint32_t ring = q >> 1, hi = ring >> ls, lo = ring & (stride - 1);
            uint32_t* x = cnt + ((hi * n * stride + lo) * w + dd - d0) * 2 + (q & 1u);
            const uint32_t step = stride * w * 2;
            uint32_t acc = 0;
            if (long_ring) {
                for (uint32_t j = lane; j < n; j += 64) {  // n is a multiple of 64 here (all dimensions powers of two)
                    const uint32_t v = wave_scan(x[j * step]) + acc;
                    x[j * step] = v;
                    mx = v > mx ? v : mx;
                    sm += v;
                    acc = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
                }
            } else {
                for (uint32_t j = 0; j < n; ++j) {
                    acc += x[j * step];
                    x[j * step] = acc;
                    mx = acc > mx ? acc : mx;
                    sm += acc;
                }
            }
        }
    }
    __syncthreads();
    uint32_t* m = mult + c.mult_off;
    if (whole) {
        for (uint32_t i = tid; i < len / 4; i += blockDim.x)
            reinterpret_cast<uint4*>(m)[i] = reinterpret_cast<const uint4*>(cnt)[i];
    } else {  // one dimension: two counters per node
        for (uint32_t i = tid; i < t.size; i += blockDim.x)
            *reinterpret_cast<uint2*>(m + ((uint64_t)i * t.nd + d0) * 2) = reinterpret_cast<const uint2*>(cnt)[i];
    }
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t a = (uint32_t)__shfl_xor((int)mx, o, 64), b = (uint32_t)__shfl_xor((int)hops, o, 64);
        mx = a > mx ? a : mx;
        hops = b > hops ? b : hops;
        sm += __shfl_xor(sm, o, 64);
    }
    if (lane == 0) {
        s_max[wave] = mx;
        s_hops[wave] = hops;
        s_sum[wave] = sm;
    }
    __syncthreads();
    if (tid == 0) {
        for (uint32_t i = 1; i < nw; ++i) {
            mx = s_max[i] > mx ? s_max[i] : mx;
            hops = s_hops[i] > hops ? s_hops[i] : hops;
            sm += s_sum[i];
        }
        if (whole) {
            max_mult[sl.x] = mx;
            sum_mult[sl.x] = sm;
        } else {
            atomicMax(max_mult + sl.x, mx);
            atomicAdd(sum_mult + sl.x, sm);
        }
        if (d0 == 0) max_hops[sl.x] = hops;
    }
}

// The same for classes whose counters exceed LDS even one dimension at a time, in device memory.
// One thread per (class, rank): the rank's message, as difference updates on the rings it crosses.
// blocks[b] = (class, first rank of the block).
__global__ void sim_count(const SimCaseRec* __restrict__ cases, const SimClassRec* __restrict__ classes,
                          const uint2* __restrict__ blocks, uint32_t* __restrict__ diff, uint32_t* __restrict__ max_hops) {
    const uint2 bk = blocks[blockIdx.x];
    const SimClassRec c = classes[bk.x];
    const SimCaseRec cs = cases[c.case_idx];
    const uint32_t r = bk.y + threadIdx.x;
    if (r >= cs.t.size) return;
    uint32_t* m = diff + c.mult_off;
    const uint32_t hops = route(cs, c, r, [&](uint32_t dd, uint32_t node, uint32_t dir, uint32_t v) {
        atomicAdd(m + ((uint64_t)node * cs.t.nd + dd) * 2 + dir, v);
    });
    if (hops) atomicMax(max_hops + bk.x, hops);
}

// One thread per (class, ring, direction): prefix sum along the ring, then the class's most loaded link and
// its total link crossings.  blocks[b] = (class, first ring-direction of the block).
__global__ void sim_scan(const SimCaseRec* __restrict__ cases, const SimClassRec* __restrict__ classes,
                         const uint2* __restrict__ blocks, uint32_t* __restrict__ mult, uint32_t* __restrict__ max_mult,
                         unsigned long long* __restrict__ sum_mult) {
    const uint2 bk = blocks[blockIdx.x];
    const SimClassRec c = classes[bk.x];
    const SimCaseRec cs = cases[c.case_idx];
    const simd::TorusD& t = cs.t;
    uint32_t q = bk.y + threadIdx.x;  // ring-direction index within the class
    uint32_t mx = 0;
    unsigned long long sm = 0;
    uint32_t dd = 0;
    for (; dd < t.nd; ++dd) {  // rings of dimension dd: 2 * size / dims[dd] of them (two directions)
        const uint32_t nr = 2 * (t.size >> simd::lg2(t.dims[dd]));
        if (q < nr) break;
        q -= nr;
    }
    if (dd < t.nd) {
        const uint32_t dir = q & 1u, ring = q >> 1;
        const uint32_t stride = dim_stride(t, dd), n = t.dims[dd];
        // ring -> its position-0 node: the other coordinates enumerate the rings, dimension dd is held at 0
        const uint32_t hi = ring >> simd::lg2(stride), lo = ring & (stride - 1);
        const uint32_t base = hi * n * stride + lo;
        uint32_t* m = mult + c.mult_off;
        uint32_t acc = 0;
        for (uint32_t j = 0; j < n; ++j) {
            uint32_t* x = m + ((uint64_t)(base + j * stride) * t.nd + dd) * 2 + dir;
            acc += *x;
            *x = acc;
            mx = acc > mx ? acc : mx;
            sm += acc;
        }
    }
    // workgroup reduction, then one atomic per workgroup and class
    __shared__ uint32_t smax[256];
    __shared__ unsigned long long ssum[256];
    smax[threadIdx.x] = mx;
    ssum[threadIdx.x] = sm;
    __syncthreads();
    for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            smax[threadIdx.x] = smax[threadIdx.x] > smax[threadIdx.x + st] ? smax[threadIdx.x] : smax[threadIdx.x + st];
            ssum[threadIdx.x] += ssum[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicMax(max_mult + bk.x, smax[0]);
        atomicAdd(sum_mult + bk.x, ssum[0]);
    }
}

// Device memory a class's workgroup can hold its counters in.
hipError_t sim_lds_limit(int device, uint32_t* bytes) {
    int v = 0;
    hipError_t e = hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device);
    if (e != hipSuccess) return e;
    constexpr uint32_t fixed = 16 * (4 + 4 + 8);  // the reduction's arrays
    *bytes = (uint32_t)v > fixed ? (uint32_t)v - fixed : 0;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(sim_class), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)*bytes);
    if (e != hipSuccess) {  // what every launch may use
        (void)hipGetLastError();
        *bytes = std::min(*bytes, 65536u - fixed);
    }
    return hipSuccess;
}

// bins: the slices in runs of like LDS need, each one launch of workgroups of `threads` lanes.
// counts in device memory: blocks of the classes that have no slices.
hipError_t launch_sim(const SimLaunch& a, hipStream_t st) {
    if (a.zero)
        hipLaunchKernelGGL(sim_zero, dim3(a.n_count_blocks ? 4096 : 16), dim3(256), 0, st, a.mult,
                           a.n_count_blocks ? a.mult_len : 0, a.max_hops, a.max_mult, (unsigned long long*)a.sum_mult,
                           a.ncls);
    if (a.n_count_blocks) {
        hipLaunchKernelGGL(sim_count, dim3(a.n_count_blocks), dim3(256), 0, st, (const SimCaseRec*)a.cases,
                           (const SimClassRec*)a.classes, (const uint2*)a.count_blocks, a.mult, a.max_hops);
        hipLaunchKernelGGL(sim_scan, dim3(a.n_scan_blocks), dim3(256), 0, st, (const SimCaseRec*)a.cases,
                           (const SimClassRec*)a.classes, (const uint2*)a.scan_blocks, a.mult, a.max_mult,
                           (unsigned long long*)a.sum_mult);
    }
    for (uint32_t i = 0; i < a.n_bins; ++i)
        hipLaunchKernelGGL(sim_class, dim3(a.bins[i].count), dim3(a.bins[i].threads), a.bins[i].lds, st,
                           (const SimCaseRec*)a.cases, (const SimClassRec*)a.classes,
                           (const uint2*)a.slices + a.bins[i].first, a.mult, a.max_hops, a.max_mult,
                           (unsigned long long*)a.sum_mult);
    return hipGetLastError();
}

}  // namespace bine
