// Body sets between the host's arrays and the device layout.  The host's arrays cross the link
// as they are; checking them and converting to and from the float4 arrays of Bodies is one
// thread per body here, so neither direction has a host loop over the bodies.  Both kernels are
// bound by HBM and far below the transfer (156 MB of poses and velocities of 3M bodies: 2.8 ms
// over the link at 57 GB/s from pinned memory; the pack kernel reads 192 MB and writes 156 MB).
#include "dev_geom.hpp"
#include "k_bodies.hpp"

namespace axm {

// The first fault of body i in the order they are looked for, 0 when it has none.
__device__ __forceinline__ uint32_t body_fault(const BodyIn& in, uint32_t i, float& radius, uint32_t& world) {
    auto fin3 = [](const float* p) { return isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]); };
    const float* p = in.pos + 3 * (size_t)i;
    const float* q = in.quat + 4 * (size_t)i;
    const float* lv = in.lin + 3 * (size_t)i;
    const float* av = in.ang + 3 * (size_t)i;
    const float* iv = in.inertia + 3 * (size_t)i;
    const float* pr = in.params + 3 * (size_t)i;
    const float im = in.mass[i];
    const uint32_t t = in.type[i];
    if (!fin3(p) || !fin3(lv) || !fin3(av) || !fin3(iv) || !isfinite(im) || im < 0.0f || !fin3(q) || !isfinite(q[3]) ||
        iv[0] < 0.0f || iv[1] < 0.0f || iv[2] < 0.0f)
        return BODY_BAD;
    const float ql = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
    if (!(ql > 0.5f && ql < 1.5f)) return BODY_BAD;
    if (t > SHAPE_CAPSULE || !fin3(pr)) return BODY_BAD_SHAPE;
    if (t == SHAPE_SPHERE) {
        if (!(pr[0] > 0.0f)) return BODY_BAD_SHAPE;
        radius = pr[0];
    } else if (t == SHAPE_BOX) {
        if (!(pr[0] > 0.0f && pr[1] > 0.0f && pr[2] > 0.0f)) return BODY_BAD_SHAPE;
        radius = sqrtf(pr[0] * pr[0] + pr[1] * pr[1] + pr[2] * pr[2]);
    } else {
        if (!(pr[0] > 0.0f && pr[1] >= 0.0f)) return BODY_BAD_SHAPE;
        radius = pr[0] + pr[1];
    }
    world = in.world ? in.world[i] : 0u;
    if (i > 0u && in.world && world < in.world[i - 1u]) return BODY_BAD_WORLD;  // worlds are contiguous
    if (in.material) {
        const float* m = in.material + 4 * (size_t)i;
        if (!isfinite(m[0]) || m[0] < 0.0f || !isfinite(m[1]) || m[1] < 0.0f || !isfinite(m[2]) || !isfinite(m[3]))
            return BODY_BAD;
    }
    if (in.flags && (in.flags[i] & BODY_KINEMATIC) && im != 0.0f) return BODY_BAD;  // kinematic bodies have no mass
    return 0u;
}
// A workgroup takes bodies in a stride and adds what it found once: an addition per wave and 64
// bodies queued up on the result's words (3M bodies: 1.08 ms, so 0.14).
__global__ void __launch_bounds__(256) k_bodies_check(BodyIn in, uint32_t n, BodyCheck* out) {
    __shared__ uint32_t s_r[4], s_w[4];
    uint32_t r = 0u, worlds = 0u;  // radii are positive: bit order is value order
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float radius = 0.0f;
        uint32_t world = 0u;
        const uint32_t fault = body_fault(in, i, radius, world);
        if (fault) {
            atomicMin(&out->fault, (unsigned long long)i << 32 | fault);
        } else {
            r = max(r, __float_as_uint(radius));
            worlds = max(worlds, world == 0xFFFFFFFFu ? world : world + 1u);  // no id wraps to none
        }
    }
    for (int o = 32; o >= 1; o >>= 1) {
        r = max(r, (uint32_t)__shfl_xor((int)r, o, 64));
        worlds = max(worlds, (uint32_t)__shfl_xor((int)worlds, o, 64));
    }
    if ((threadIdx.x & 63u) == 0u) {
        s_r[threadIdx.x >> 6] = r;
        s_w[threadIdx.x >> 6] = worlds;
    }
    __syncthreads();
    if (threadIdx.x == 0u) {
        atomicMax(&out->radius_bits, max(max(s_r[0], s_r[1]), max(s_r[2], s_r[3])));
        atomicMax(&out->worlds, max(max(s_w[0], s_w[1]), max(s_w[2], s_w[3])));
    }
}
__global__ void __launch_bounds__(256) k_bodies_install(BodyIn in, uint32_t n, Bodies B, float4 mat) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float* p = in.pos + 3 * (size_t)i;
    const float* q = in.quat + 4 * (size_t)i;
    const float* lv = in.lin + 3 * (size_t)i;
    const float* av = in.ang + 3 * (size_t)i;
    const float* iv = in.inertia + 3 * (size_t)i;
    const float* pr = in.params + 3 * (size_t)i;
    const float im = in.mass[i];
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    B.x[i] = make_float4(p[0], p[1], p[2], 0.0f);
    B.q[i] = make_float4(q[0], q[1], q[2], q[3]);
    B.vel[i] = make_float4(lv[0], lv[1], lv[2], im);
    B.angv[i] = make_float4(av[0], av[1], av[2], 0.0f);
    B.ii[i] = im == 0.0f ? zero : make_float4(iv[0], iv[1], iv[2], 0.0f);
    B.shape[i] = make_float4(pr[0], pr[1], pr[2], __uint_as_float(in.type[i]));
    if (in.material) {
        const float* m = in.material + 4 * (size_t)i;
        mat = make_float4(m[0], m[1], m[2], m[3]);
    }
    B.mat[i] = make_float4(mat.x, mat.y, 1.0f - mat.z, 1.0f - mat.w);
    const uint32_t fl = in.flags ? in.flags[i] : 0u;
    const uint32_t* f = in.filter + 3 * (size_t)i;
    B.bfl[i] = in.filter ? make_uint4(fl, f[0], f[1], f[2]) : make_uint4(fl, 1u, 0xFFFFFFFFu, 0u);
    const uint32_t world = in.world ? in.world[i] : 0u;
    B.world[i] = world;
    if ((i == 0u || (in.world && in.world[i - 1u] != world))) B.world_first[world] = i;
    // every body starts awake with no rest time and no island; no island has a wake request
    B.slp[i] = make_uint2(0u, LABEL_NONE);
    B.wake[i] = 0xFFFFFFFFu;
}
__global__ void __launch_bounds__(256) k_bodies_pack(Bodies B, uint32_t n, float* pos, float* quat, float* lin, float* ang) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    auto put3 = [&](float* o, const float4* a) {
        if (!o) return;
        const float4 v = a[i];
        o += 3 * (size_t)i;
        o[0] = v.x;
        o[1] = v.y;
        o[2] = v.z;
    };
    put3(pos, B.x);
    if (quat) {
        const float4 v = B.q[i];
        float* o = quat + 4 * (size_t)i;
        o[0] = v.x;
        o[1] = v.y;
        o[2] = v.z;
        o[3] = v.w;
    }
    put3(lin, B.vel);
    put3(ang, B.angv);
}

static inline dim3 blocks(uint32_t n) { return dim3((n + 255u) / 256u); }
void launch_bodies_check(const BodyIn& in, uint32_t n, BodyCheck* out, hipStream_t s) {
    const uint32_t g = (n + 255u) / 256u;
    if (n) hipLaunchKernelGGL(k_bodies_check, dim3(g < 1024u ? g : 1024u), dim3(256), 0, s, in, n, out);
}
void launch_bodies_install(const BodyIn& in, uint32_t n, const Bodies& B, float4 mat, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_bodies_install, blocks(n), dim3(256), 0, s, in, n, B, mat);
}
void launch_bodies_pack(const Bodies& B, uint32_t n, float* pos, float* quat, float* lin, float* ang, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_bodies_pack, blocks(n), dim3(256), 0, s, B, n, pos, quat, lin, ang);
}

}  // namespace axm
