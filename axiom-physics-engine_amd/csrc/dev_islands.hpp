// Union-find over the bodies of a step and the island of a manifold.
#pragma once
#include "launch.hpp"

namespace axm {

// Union-find over body indices.  Every link points from a larger root to a smaller one
// (compare-and-swap on the root), so the root of a finished component is its smallest
// body index whatever the order of the links (lock-free union-find with path halving:
// Jaiganesh & Burtscher 2018, ECL-CC).  The parents are shared between workgroups, so
// they move through agent-scope atomics.
__device__ __forceinline__ uint32_t uf_load(uint32_t* p, uint32_t x) {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t uf_find(uint32_t* par, uint32_t x) {
    uint32_t cur = uf_load(par, x);
    if (cur != x) {
        uint32_t prev = x, next;
        while (cur > (next = uf_load(par, cur))) {
            __hip_atomic_store(par + prev, next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            prev = cur;
            cur = next;
        }
    }
    return cur;
}
// Root of x in the finished forest (after the union kernel, which no later kernel of the
// step changes): the union's coherent loads, without its path-halving stores (in one giant
// island every walk ends on the same root word, which stores would keep contended).
__device__ __forceinline__ uint32_t uf_root(uint32_t* par, uint32_t x) {
    uint32_t p;
    while ((p = uf_load(par, x)) != x) x = p;
    return x;
}
// Island (union-find root) of a manifold: that of its dynamic body, UNSET with none.
__device__ __forceinline__ uint32_t man_root(const Bodies& B, uint2 ab) {
    const bool plane = (ab.y & PLANE_BIT) != 0u;
    const uint32_t d = B.sv[ab.x].w > 0.0f ? ab.x : (!plane && B.sv[ab.y].w > 0.0f ? ab.y : UNSET);
    return d == UNSET ? UNSET : uf_root(B.upar, d);
}

}  // namespace axm
