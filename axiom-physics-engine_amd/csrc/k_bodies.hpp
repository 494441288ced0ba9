// Launch wrappers of the body set conversions (k_bodies.hip).
#pragma once
#include "launch.hpp"

namespace axm {

// A body set in the host's layout (axm_body_soa), on the device; world, material, flags and
// filter may be null.
struct BodyIn {
    const float *pos, *quat, *lin, *ang, *mass, *inertia, *params;
    const uint32_t *type, *world;
    const float* material;
    const uint32_t *flags, *filter;
};
// What is wrong with a body.
enum : uint32_t { BODY_BAD = 1u, BODY_BAD_SHAPE = 2u, BODY_BAD_WORLD = 3u };
// The first faulty body (index << 32 | fault; all ones: none), the largest bounding radius and
// the number of worlds (the last two of the bodies without fault).
struct BodyCheck {
    unsigned long long fault;
    uint32_t radius_bits, worlds;
};
// Adds the body set to *out (which starts as no fault, 0, 0).
void launch_bodies_check(const BodyIn& in, uint32_t n, BodyCheck* out, hipStream_t s);
// Writes a checked body set into the device layout; mat: friction, restitution and the two
// dampings of a body without material.  world_first (an entry per world) starts as zeros.
void launch_bodies_install(const BodyIn& in, uint32_t n, const Bodies& B, float4 mat, hipStream_t s);
// The bodies' state as 3, 4, 3 and 3 floats each (null: not wanted).
void launch_bodies_pack(const Bodies& B, uint32_t n, float* pos, float* quat, float* lin, float* ang, hipStream_t s);

}  // namespace axm
