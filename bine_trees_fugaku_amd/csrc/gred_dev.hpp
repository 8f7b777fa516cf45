// gred_dev.hpp -- device helpers shared by the gather-reduce kernels: address-space views, 16-byte vectors and
// their additions, work-item addressing and the pairwise tree.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gred.hpp"

namespace bine {

typedef unsigned int u4 __attribute__((ext_vector_type(4)));

// Address-space views.  Data goes through global (address space 1) pointers, so loads and stores issue
// as global_* instructions, which count against the vector-memory counter only; generic pointers would
// give flat_* instructions, which also hold the scalar/LDS counter, so that every wait for a scalar load
// would drain the data loads in flight as well.  Work items, pool entries and buffer tables are read
// through constant (address space 4) pointers with a wave-uniform address, so they issue as scalar loads
// (one s_load_dwordx8 for four consecutive pool entries) that never wait on the data loads.
#define BINE_GLOBAL __attribute__((address_space(1)))
#define BINE_CONST __attribute__((address_space(4)))
typedef u4 u4b __attribute__((aligned(1)));  // 16 bytes at any byte address (global memory runs in the unaligned mode)

template <typename X>
__device__ __forceinline__ BINE_GLOBAL X* gptr(const void* p) {
    return (BINE_GLOBAL X*)(uintptr_t)p;
}

// p must be the same for every lane of the wave
template <typename X>
__device__ __forceinline__ const BINE_CONST X* cptr(const X* p) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return (const BINE_CONST X*)(((uint64_t)hi << 32) | lo);
}

// A struct read word by word through a constant pointer (a plain copy would need a copy constructor that
// takes the generic address space).
template <typename X>
__device__ __forceinline__ X cload(const BINE_CONST X* p) {
    static_assert(sizeof(X) % 4 == 0, "struct of whole words");
    const BINE_CONST uint32_t* q = (const BINE_CONST uint32_t*)p;
    uint32_t w[sizeof(X) / 4];
#pragma unroll
    for (unsigned i = 0; i < sizeof(X) / 4; ++i) w[i] = q[i];
    X r;
    __builtin_memcpy(&r, w, sizeof(X));
    return r;
}

// 16 bytes of elements of type T, held as one 128-bit register quad.
template <typename T>
struct Vec {
    static constexpr int N = 16 / sizeof(T);
    u4 raw;
};

template <typename T>
__device__ __forceinline__ T add1(T a, T b) {
    return a + b;
}
template <>
__device__ __forceinline__ int32_t add1<int32_t>(int32_t a, int32_t b) {
    return (int32_t)((uint32_t)a + (uint32_t)b);
}
template <>
__device__ __forceinline__ int64_t add1<int64_t>(int64_t a, int64_t b) {
    return (int64_t)((uint64_t)a + (uint64_t)b);
}
template <>
__device__ __forceinline__ int8_t add1<int8_t>(int8_t a, int8_t b) {
    return (int8_t)((uint8_t)a + (uint8_t)b);
}

template <typename T>
__device__ __forceinline__ Vec<T> vadd(const Vec<T>& a, const Vec<T>& b) {
    T x[Vec<T>::N], y[Vec<T>::N];
    __builtin_memcpy(x, &a.raw, 16);
    __builtin_memcpy(y, &b.raw, 16);
#pragma unroll
    for (int i = 0; i < Vec<T>::N; ++i) x[i] = add1<T>(x[i], y[i]);
    Vec<T> r;
    __builtin_memcpy(&r.raw, x, 16);
    return r;
}

// 16 bytes added lane by lane (mod 256) on four 32-bit words: the low seven
// bits of each byte cannot carry out of the byte, the top bit is the xor of
// the carry into it with both operands' top bits.
template <>
__device__ __forceinline__ Vec<int8_t> vadd<int8_t>(const Vec<int8_t>& a, const Vec<int8_t>& b) {
    const u4 x = a.raw, y = b.raw;
    Vec<int8_t> r;
    r.raw = ((x & 0x7F7F7F7Fu) + (y & 0x7F7F7F7Fu)) ^ ((x ^ y) & 0x80808080u);
    return r;
}

template <typename T, bool NT>
__device__ __forceinline__ Vec<T> vload(const char* p) {
    Vec<T> r;
    if (NT) r.raw = __builtin_nontemporal_load(gptr<const u4b>(p));
    else r.raw = *gptr<const u4b>(p);
    return r;
}

template <typename T, bool NT>
__device__ __forceinline__ void vstore(char* p, const Vec<T>& v) {
    if (NT) __builtin_nontemporal_store(v.raw, gptr<u4b>(p));
    else *gptr<u4b>(p) = v.raw;
}

// Units of the narrow and tree kernels: a 16-byte vector at any byte address, or one element.
template <bool NT = false, typename T>
__device__ __forceinline__ Vec<T> load_unit(const char* p, Vec<T>*) {
    return vload<T, NT>(p);
}
template <bool NT = false, typename T>
__device__ __forceinline__ T load_unit(const char* p, T*) {
    return *gptr<const T>(p);
}
template <bool NT = false, typename T>
__device__ __forceinline__ void store_unit(char* p, const Vec<T>& v) {
    vstore<T, NT>(p, v);
}
template <bool NT = false, typename T>
__device__ __forceinline__ void store_unit(char* p, T v) {
    *gptr<T>(p) = v;
}
template <typename T>
__device__ __forceinline__ Vec<T> add_unit(const Vec<T>& a, const Vec<T>& b) {
    return vadd<T>(a, b);
}
template <typename T>
__device__ __forceinline__ T add_unit(T a, T b) {
    return add1<T>(a, b);
}

// Buffer address of a (buffer, rank, element offset) entry.  The buffer is
// picked with masks rather than an indexed or selected load so the table stays
// in scalar registers.
struct Table {
    uint64_t b0, b1, b2, b3, s0, s1, s2, s3;
    __device__ __forceinline__ char* at(uint32_t rb, uint64_t elem_off, uint32_t tsize) const {
        const uint32_t buf = rb >> 28, rank = rb & 0x0FFFFFFFu;
        const uint64_t m0 = 0ull - (uint64_t)(buf == 0), m1 = 0ull - (uint64_t)(buf == 1);
        const uint64_t m2 = 0ull - (uint64_t)(buf == 2), m3 = 0ull - (uint64_t)(buf == 3);
        const uint64_t base = (b0 & m0) | (b1 & m1) | (b2 & m2) | (b3 & m3);
        const uint64_t stride = (s0 & m0) | (s1 & m1) | (s2 & m2) | (s3 & m3);
        return reinterpret_cast<char*>(base + (uint64_t)rank * stride + elem_off * tsize);
    }
};

// Evaluate the balanced tree over 2^lg leaves; `load(k)` fetches leaf k.
// Leaves are taken in groups of G (4 or 8), each reduced pairwise, and the
// group sums are folded with a binary counter: the association is the same
// balanced tree for either G; G = 4 halves the loads in flight per thread.
template <typename W, int MAXS, int G, typename AddF, typename LoadF>
__device__ __forceinline__ W tree_eval(uint32_t lg, AddF add, LoadF load) {
    if (lg == 0) return load(0);
    if (lg == 1) return add(load(0), load(1));
    if (lg == 2) return add(add(load(0), load(1)), add(load(2), load(3)));
    W stk[MAXS];
    const uint32_t S = lg - (G == 8 ? 3 : 2);
    const uint32_t ngroups = 1u << S;
    W res;
    for (uint32_t j = 0; j < ngroups; ++j) {
        const uint32_t k = j * G;
        W v;
        if (G == 8) {
            W x0 = load(k + 0), x1 = load(k + 1), x2 = load(k + 2), x3 = load(k + 3);
            W x4 = load(k + 4), x5 = load(k + 5), x6 = load(k + 6), x7 = load(k + 7);
            v = add(add(add(x0, x1), add(x2, x3)), add(add(x4, x5), add(x6, x7)));
        } else {
            W x0 = load(k + 0), x1 = load(k + 1), x2 = load(k + 2), x3 = load(k + 3);
            v = add(add(x0, x1), add(x2, x3));
        }
        // binary-counter carry: level l holds the sum of the previous 2^l groups
        bool carry = true;
#pragma unroll
        for (int l = 0; l < MAXS; ++l) {
            if (carry && l < (int)S) {
                if ((j >> l) & 1u) {
                    v = add(stk[l], v);
                } else {
                    stk[l] = v;
                    carry = false;
                }
            }
        }
        res = v;
    }
    return res;
}

}  // namespace bine
