// sim_dest.hpp -- destination of one rank's message in a simulation step
// class; shared by the host reference and the GPU kernel.
#pragma once

#include <cstdint>

#ifndef BINE_HD
#if defined(__HIPCC__)
#define BINE_HD __host__ __device__
#else
#define BINE_HD
#endif
#endif

namespace bine {
namespace simd {

struct TorusD {
    uint32_t dims[3];
    uint32_t nd, size;
};

// Device records of the simulation (one per case, one per step class).
struct SimCaseRec {
    TorusD t;
    uint32_t L, nlinks;
    uint64_t pad;
};
struct SimClassRec {
    uint32_t kind, d, k, case_idx;
    uint64_t mult_off;  // first link counter of the class
};

// Every simulated torus has dimensions that are powers of two (sim_build_case refuses others), so remainders are masks
// and quotients shifts; a kernel that divides spends most of its time there.
BINE_HD inline int pm(int a, int b) { return a & (b - 1); }
BINE_HD inline uint32_t lg2(uint32_t x) { return (uint32_t)__builtin_ctz(x); }
BINE_HD inline uint32_t to_nb(int32_t v) { return (0xAAAAAAAAu + (uint32_t)v) ^ 0xAAAAAAAAu; }
BINE_HD inline int32_t from_nb(uint32_t n) { return (int32_t)((0xAAAAAAAAu ^ n) - 0xAAAAAAAAu); }
BINE_HD inline int rho(uint32_t k) {
    int64_t p = 1;
    for (uint32_t i = 0; i <= k; ++i) p *= -2;
    return (int)((1 - p) / 3);
}
// Coordinates are taken one by one: an indexed array would live in memory on the GPU.
BINE_HD inline void coords(const TorusD& t, uint32_t id, int* c) {
    c[1] = c[2] = 0;
    if (t.nd > 2) {
        c[2] = pm((int)id, (int)t.dims[2]);
        id >>= lg2(t.dims[2]);
    }
    if (t.nd > 1) {
        c[1] = pm((int)id, (int)t.dims[1]);
        id >>= lg2(t.dims[1]);
    }
    c[0] = pm((int)id, (int)t.dims[0]);
}
BINE_HD inline uint32_t ident(const TorusD& t, const int* c) {
    uint32_t r = (uint32_t)pm(c[0], (int)t.dims[0]);
    if (t.nd > 1) r = (r << lg2(t.dims[1])) + (uint32_t)pm(c[1], (int)t.dims[1]);
    if (t.nd > 2) r = (r << lg2(t.dims[2])) + (uint32_t)pm(c[2], (int)t.dims[2]);
    return r;
}
BINE_HD inline int get(const int* c, uint32_t d) { return d == 0 ? c[0] : d == 1 ? c[1] : c[2]; }
BINE_HD inline void put(int* c, uint32_t d, int v) {
    c[0] = d == 0 ? v : c[0];
    c[1] = d == 1 ? v : c[1];
    c[2] = d == 2 ? v : c[2];
}
// simulation/simulator.py:11-26 (for 3D: x varies with id / d1 mod d0, y fastest, z slowest)
BINE_HD inline void simpy_coords(const TorusD& t, uint32_t id, int* c) {
    if (t.nd == 1) {
        c[0] = (int)id;
    } else if (t.nd == 2) {
        c[0] = (int)(id >> lg2(t.dims[1]));
        c[1] = pm((int)id, (int)t.dims[1]);
    } else {
        c[0] = pm((int)(id >> lg2(t.dims[1])), (int)t.dims[0]);
        c[1] = pm((int)id, (int)t.dims[1]);
        c[2] = (int)(id >> lg2(t.dims[0] * t.dims[1]));
    }
}
BINE_HD inline uint32_t simpy_ident(const TorusD& t, const int* c) {
    if (t.nd == 1) return (uint32_t)c[0];
    if (t.nd == 2) return (uint32_t)(c[0] * (int)t.dims[1] + c[1]);
    return (uint32_t)(c[2] * (int)(t.dims[0] * t.dims[1]) + c[0] * (int)t.dims[1] + c[1]);
}

// Bine tree tests (lib/libbine_coll_bcast.cc:645-663, lib/libbine_coll_reduce.cc:587-611), root 0
BINE_HD inline bool equal_lsbs(uint32_t v, uint32_t mask_lsbs) {
    uint32_t l = to_nb((int32_t)v) & mask_lsbs;
    return l == 0 || l == mask_lsbs;
}
BINE_HD inline uint32_t tree_partner(uint32_t r, uint32_t mask, uint32_t P) {
    return (uint32_t)pm(from_nb(to_nb((int32_t)r) ^ ((mask << 1) - 1)), (int)P);
}

// Destination of rank r (library rank order) or 0xFFFFFFFF when r is silent.
// L = log2(P) for the 1D kinds.
BINE_HD inline uint32_t dest(const TorusD& t, uint32_t kind, uint32_t d, uint32_t k, uint32_t r, uint32_t L) {
    const uint32_t P = t.size;
    switch (kind) {
    case 0:
    case 1: {  // torus peer on dimension d, step k of that dimension
        int c[3];
        coords(t, r, c);
        int dist;
        if (kind == 0) {
            dist = rho(k);
            if (get(c, d) & 1) dist = -dist;
        } else {
            dist = (get(c, d) ^ (1 << k)) - get(c, d);
        }
        put(c, d, pm(get(c, d) + dist, (int)t.dims[d]));
        return ident(t, c);
    }
    case 2: return (r + 1) & (P - 1);
    case 3: {
        int dist = from_nb((2u << k) - 1);
        return (uint32_t)((r % 2 == 0) ? pm((int)r + dist, (int)P) : pm((int)r - dist, (int)P));
    }
    case 4: return r ^ (1u << k);
    case 5: return (r + (1u << k)) & (P - 1);
    // Equal low bits of a number are equal in every shorter run, so the first mask at which a rank is reached (or
    // sends) is told from the two runs around it.
    case 6: {  // bcast order: masks 2^(L-1) .. 1; r sends at mask m if it was reached at a larger mask
        const uint32_t m = 1u << k;
        return r == 0 || (k + 1 < L && equal_lsbs(r, (m << 2) - 1)) ? tree_partner(r, m, P) : 0xFFFFFFFFu;
    }
    case 7: {  // reduce order: masks 1 .. 2^(L-1); r sends at the first mask where it stops receiving
        const uint32_t m = 1u << k;
        const bool before = k == 0 || equal_lsbs(r, (m << 1) - 1);
        const bool now = !equal_lsbs(r, (m << 2) - 1) || ((m << 1) >= P && r != 0);
        return before && now ? tree_partner(r, m, P) : 0xFFFFFFFFu;
    }
    case 8: {
        const uint32_t m = 1u << k;
        return ((r & (2 * m - 1)) == 0 && r + m < P) ? r + m : 0xFFFFFFFFu;
    }
    case 9: {
        const uint32_t m = 1u << k;
        return ((r & (2 * m - 1)) == m) ? r - m : 0xFFFFFFFFu;
    }
    case 10: {  // simulator.py: r's peer at step k; ranks are read in simulator.py's id order
        int c[3] = {0, 0, 0};
        simpy_coords(t, r, c);
        const uint32_t dim = k % t.nd, rel = k / t.nd;
        if (rel >= 10) return 0xFFFFFFFFu;  // beyond simulator.py's table; such cases are refused when built
        int sgn = (rel % 2 == 0) ? 1 : -1;
        const int hop = ((2 << rel) + sgn) / 3;  // its table: 1, 1, 3, 5, 11, 21, 43, 85, 171, 341
        if (get(c, dim) % 2) sgn = -sgn;
        put(c, dim, pm(get(c, dim) + sgn * hop, (int)t.dims[dim]));
        return simpy_ident(t, c);
    }
    default: return 0xFFFFFFFFu;
    }
}

}  // namespace simd
}  // namespace bine
