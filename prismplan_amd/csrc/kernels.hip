// kernels.hip -- gfx950 kernels of the collision-kinematics substrate.
//
// Execution model (wave64, CDNA4):
//  * a workgroup is one wavefront; it walks chunks of robot states
//    (configurations, edge states or waypoints) in a static, XCD-aware order
//    (chunks never span two problems, so each wave sees one OBB set at a
//    time), with 1 to 16 lanes per state by the kernel and the launch's size;
//  * the problem's enabled OBBs are re-packed into LDS records once per
//    problem switch, or tile by tile where one staging does not hold them;
//  * FK walks the DFS-ordered joint table with wave-uniform (scalar) loads and
//    the live 3x4 transforms in VGPRs, or, with 16 lanes per state, composes
//    one joint per lane by pointer jumping through LDS;
//  * the any-collision predicate narrows each joint's boxes by rows of 16
//    states, then by each state's approximate sphere, and tests the exact
//    spheres of the (state, box) pairs left in full waves;
//  * the summed-hinge cost tests a sphere cluster's candidate boxes only; its
//    adjoint differentiates through the argmin OBB of each active sphere in
//    the same pass and sums the wrenches over the joint tree;
//  * self collision goes by blocks of sphere-cluster pairs, large
//    any-collision sets by rough distances first.
#include "ppl_internal.hpp"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <mutex>

namespace ppl {
namespace {

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

__device__ __forceinline__ bool wave_any(bool p) { return __ballot(p) != 0ull; }

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// Wave-uniform reads of tables that no launch writes (robot tables, layer
// parameters), through the constant address space: they become scalar loads
// into SGPRs. A plain read after a barrier or an LDS write is a vector load
// per lane instead, since the compiler cannot tell that the table stays.
typedef float f4u __attribute__((ext_vector_type(4)));
typedef float f4s __attribute__((ext_vector_type(4), aligned(4)));   // of a caller's floats, which lie at any float
typedef int i4u __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ T uload(const void* p, int i) {
    return reinterpret_cast<const __attribute__((address_space(4))) T*>(reinterpret_cast<uintptr_t>(p))[i];
}
template <typename V = f4u>
__device__ __forceinline__ float4 uload4(const void* p, int i) {
    const V v = uload<V>(p, i);
    return make_float4(v.x, v.y, v.z, v.w);
}

// ---------------------------------------------------------------------------
// 3x4 affine helpers (row-major, implicit last row 0 0 0 1)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void aff_identity(float* T) {
#pragma unroll
    for (int i = 0; i < 12; ++i) T[i] = 0.0f;
    T[0] = T[5] = T[10] = 1.0f;
}

// S = FT * M(q) for a joint that is the same in every lane, restating xrot_fn /
// yrot_fn / zrot_fn / prism_fn (planning/utils.cuh:560-702); FIXED or unknown
// types move nothing. tab: [J][12] rows of the fixed transforms, by scalar
// loads; s, c: sine and cosine of q (revolute joints).
template <int A, int B>
__device__ __forceinline__ void rot_cols(float s, float c, float* S) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const float fa = S[r * 4 + A], fb = S[r * 4 + B];
        S[r * 4 + A] = fmaf(fa, c, fb * s);
        S[r * 4 + B] = fmaf(fb, c, -fa * s);
    }
}
__device__ __forceinline__ void joint_step_u(const float* tab, int jj, int type, float q, float s, float c, float* S) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const f4u f = uload<f4u>(tab, 3 * jj + r);
        S[r * 4] = f.x; S[r * 4 + 1] = f.y; S[r * 4 + 2] = f.z; S[r * 4 + 3] = f.w;
    }
    if (type == kXRot) rot_cols<1, 2>(s, c, S);
    else if (type == kYRot) rot_cols<2, 0>(s, c, S);
    else if (type == kZRot) rot_cols<0, 1>(s, c, S);
    else if (type >= kXPrism) {
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const float f = type == kXPrism ? S[r * 4] : type == kYPrism ? S[r * 4 + 1] : S[r * 4 + 2];
            S[r * 4 + 3] = fmaf(f, q, S[r * 4 + 3]);
        }
    }
}

// T = P * S
__device__ __forceinline__ void aff_compose(const float* P, const float* S, float* T) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float acc = fmaf(P[r * 4 + 2], S[8 + c], fmaf(P[r * 4 + 1], S[4 + c], P[r * 4 + 0] * S[c]));
            if (c == 3) acc += P[r * 4 + 3];
            T[r * 4 + c] = acc;
        }
    }
}

__device__ __forceinline__ void aff_point(const float* T, float x, float y, float z, float& px, float& py, float& pz) {
    px = fmaf(T[0], x, fmaf(T[1], y, fmaf(T[2], z, T[3])));
    py = fmaf(T[4], x, fmaf(T[5], y, fmaf(T[6], z, T[7])));
    pz = fmaf(T[8], x, fmaf(T[9], y, fmaf(T[10], z, T[11])));
}

// Transform slots (the reference's t_memory_idx scratch), kept in VGPRs. The
// slot index is wave-uniform, so the switch compiles to scalar branches.
struct Slots {
    float s[kMaxSlots][12];
    __device__ __forceinline__ void load(int i, float* T) const {
        if (i == 0) {
#pragma unroll
            for (int k = 0; k < 12; ++k) T[k] = s[0][k];
        } else {
#pragma unroll
            for (int k = 0; k < 12; ++k) T[k] = s[1][k];
        }
    }
    __device__ __forceinline__ void store(int i, const float* T) {
        if (i == 0) {
#pragma unroll
            for (int k = 0; k < 12; ++k) s[0][k] = T[k];
        } else {
#pragma unroll
            for (int k = 0; k < 12; ++k) s[1][k] = T[k];
        }
    }
};

// Transform of DFS position jj: identity at the root, parent * step otherwise.
// APPROX walks the approximate spheres' own chain (R.aft / R.atype, set when
// the model has one): same tree, dofs and slots, its own fixed transforms and
// joint types.
template <bool APPROX = false>
__device__ __forceinline__ void fk_joint(const DRobot& R, int jj, const float* s_q, Slots& sl, float* T, int4& meta) {
    const i4u m = uload<i4u>(R.jmeta, jj);
    meta = make_int4(m.x, m.y, m.z, m.w);
    if (jj == 0) {
        aff_identity(T);
    } else {
        float P[12], S[12];
        sl.load(meta.w, P);
        const float q = meta.y >= 0 ? s_q[meta.y * kWave] : 0.0f;
        const int type = APPROX ? uload<int>(R.atype, jj) : meta.x;
        float s = 0.0f, c = 0.0f;
        if (type >= kXRot) sincosf(q, &s, &c);
        joint_step_u(APPROX ? R.aft : R.ft, jj, type, q, s, c, S);
        aff_compose(P, S, T);
    }
    sl.store(meta.z, T);
}

// The same walk for a model whose joints each hang on the joint before them in
// DFS order or on the root (DRobot::line; arms of a torso are such lines): the
// parent's frame is the last one, or the root's identity, so T itself carries
// the state from joint to joint and no slots are held. The compositions are
// fk_joint's, so the frames have the same bits.
template <bool LINE>
struct FkWalk {
    Slots sl;
    __device__ __forceinline__ void step(const DRobot& R, int jj, const float* s_q, float* T, int4& meta) {
        fk_joint(R, jj, s_q, sl, T, meta);
    }
};
template <>
struct FkWalk<true> {
    __device__ __forceinline__ void step(const DRobot& R, int jj, const float* s_q, float* T, int4& meta) {
        const i4u m = uload<i4u>(R.jmeta, jj);
        meta = make_int4(m.x, m.y, m.z, m.w);
        if (jj == 0) {
            aff_identity(T);
            return;
        }
        float P[12], S[12];
        if (uload<int>(R.parent, jj) == 0) {
            aff_identity(P);
        } else {
#pragma unroll
            for (int k = 0; k < 12; ++k) P[k] = T[k];
        }
        const float q = meta.y >= 0 ? s_q[meta.y * kWave] : 0.0f;
        float s = 0.0f, c = 0.0f;
        if (meta.x >= kXRot) sincosf(q, &s, &c);
        joint_step_u(R.ft, jj, meta.x, q, s, c, S);
        aff_compose(P, S, T);
    }
};

// ---------------------------------------------------------------------------
// OBB staging: enabled OBBs of [o0, o1) -> LDS records (see ppl_internal.hpp)
// ---------------------------------------------------------------------------
// Record of OBB o from its stored inverse pose and full extents.
__device__ __forceinline__ void obb_record(const float4& d4, const float4& p0, const float4& p1, int o, float4* rec) {
    const float w = p0.w, x = p1.x, y = p1.y, z = p1.z;
    // Matrix of v -> v + w t + u x t, t = 2 u x v (scene_collision.cuh:36-45).
    const float r00 = 1.0f - 2.0f * (y * y + z * z), r01 = 2.0f * (x * y - w * z), r02 = 2.0f * (x * z + w * y);
    const float r10 = 2.0f * (x * y + w * z), r11 = 1.0f - 2.0f * (x * x + z * z), r12 = 2.0f * (y * z - w * x);
    const float r20 = 2.0f * (x * z - w * y), r21 = 2.0f * (y * z + w * x), r22 = 1.0f - 2.0f * (x * x + y * y);
    rec[0] = make_float4(r00, r01, r02, p0.x);
    rec[1] = make_float4(r10, r11, r12, p0.y);
    rec[2] = make_float4(r20, r21, r22, p0.z);
    rec[3] = make_float4(0.5f * d4.x, 0.5f * d4.y, 0.5f * d4.z, __int_as_float(o));
}

__device__ __forceinline__ void obb_record(const DScene& S, int o, float4* rec) {
    obb_record(*reinterpret_cast<const float4*>(S.obb_dims + 4 * (size_t)o),
               *reinterpret_cast<const float4*>(S.obb_pose + 8 * (size_t)o),
               *reinterpret_cast<const float4*>(S.obb_pose + 8 * (size_t)o + 4), o, rec);
}

// Stages the enabled OBBs of [o0, o1) (at most cap of them: callers pass
// ranges of at most cap OBBs) and returns their count. STRIDE: float4s from one
// record to the next.
template <int STRIDE = 4>
__device__ int stage_obbs(const DScene& S, int o0, int o1, float4* s_obb, int cap) {
    const int lane = lane_id();
    int n = 0;
    for (int base = o0; base < o1; base += kWave) {
        const int o = base + lane;
        // enable flag, extents and pose in one round trip, then compaction
        float4 d4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), p0 = d4, p1 = d4;
        bool ok = false;
        if (o < o1) {
            ok = S.obb_enable[o] != 0;
            d4 = *reinterpret_cast<const float4*>(S.obb_dims + 4 * (size_t)o);
            p0 = *reinterpret_cast<const float4*>(S.obb_pose + 8 * (size_t)o);
            p1 = *reinterpret_cast<const float4*>(S.obb_pose + 8 * (size_t)o + 4);
        }
        const unsigned long long m = __ballot(ok);
        if (ok) {
            const int pos = n + __popcll(m & ((1ull << lane) - 1ull));
            if (pos < cap) obb_record(d4, p0, p1, o, s_obb + STRIDE * pos);
        }
        n += __popcll(m);
    }
    __syncthreads();
    return n < cap ? n : cap;
}

// OBB tiles of a problem's range [o0, o1): ranges of at most `cap` OBBs
// (cap >= 1), one LDS staging each.
__device__ __forceinline__ int obb_tiles(int o0, int o1, int cap) {
    return o1 - o0 <= cap ? 1 : (o1 - o0 + cap - 1) / cap;
}

__device__ __forceinline__ void to_box(const float4& r0, const float4& r1, const float4& r2, float px, float py, float pz,
                                       float& lx, float& ly, float& lz) {
    lx = fmaf(r0.x, px, fmaf(r0.y, py, fmaf(r0.z, pz, r0.w)));
    ly = fmaf(r1.x, px, fmaf(r1.y, py, fmaf(r1.z, pz, r1.w)));
    lz = fmaf(r2.x, px, fmaf(r2.y, py, fmaf(r2.z, pz, r2.w)));
}

// Squared distance to the box.
__device__ __forceinline__ float box_dist2(float lx, float ly, float lz, const float4& h) {
    const float cx = fmaxf(fabsf(lx) - h.x, 0.0f);
    const float cy = fmaxf(fabsf(ly) - h.y, 0.0f);
    const float cz = fmaxf(fabsf(lz) - h.z, 0.0f);
    return fmaf(cz, cz, fmaf(cy, cy, cx * cx));
}

// Collision iff squared distance to the box < r^2 (scene_collision.cuh:59-78).
__device__ __forceinline__ bool box_hit(float lx, float ly, float lz, const float4& h, float r2) {
    return box_dist2(lx, ly, lz, h) < r2;
}

// Order-preserving key of the box signed distance (Quilez form,
// scene_collision.cuh:88-112): key = |max(q,0)|^2 - min(max q, 0)^2 is
// sdf*|sdf|, so the minimum needs no square root per pair.
__device__ __forceinline__ float box_key(float lx, float ly, float lz, const float4& h) {
    const float qx = fabsf(lx) - h.x, qy = fabsf(ly) - h.y, qz = fabsf(lz) - h.z;
    const float ox = fmaxf(qx, 0.0f), oy = fmaxf(qy, 0.0f), oz = fmaxf(qz, 0.0f);
    const float in = fminf(fmaxf(qx, fmaxf(qy, qz)), 0.0f);
    return fmaf(-in, in, fmaf(oz, oz, fmaf(oy, oy, ox * ox)));
}

__device__ __forceinline__ float key_to_sdf(float k) { return k >= 0.0f ? sqrtf(k) : -sqrtf(-k); }

// World-frame gradient of the box signed distance at world point p.
__device__ __forceinline__ void box_sdf_grad(const float4& r0, const float4& r1, const float4& r2, const float4& h,
                                             float px, float py, float pz, float& gx, float& gy, float& gz) {
    float lx, ly, lz;
    to_box(r0, r1, r2, px, py, pz, lx, ly, lz);
    const float sx = lx >= 0.0f ? 1.0f : -1.0f, sy = ly >= 0.0f ? 1.0f : -1.0f, sz = lz >= 0.0f ? 1.0f : -1.0f;
    const float qx = fabsf(lx) - h.x, qy = fabsf(ly) - h.y, qz = fabsf(lz) - h.z;
    float ax, ay, az;
    if (fmaxf(qx, fmaxf(qy, qz)) > 0.0f) {
        const float ox = fmaxf(qx, 0.0f), oy = fmaxf(qy, 0.0f), oz = fmaxf(qz, 0.0f);
        const float inv = 1.0f / sqrtf(fmaf(oz, oz, fmaf(oy, oy, ox * ox)));
        ax = ox * inv * sx; ay = oy * inv * sy; az = oz * inv * sz;
    } else {
        const bool xb = qx >= qy && qx >= qz;
        const bool yb = !xb && qy >= qz;
        ax = xb ? sx : 0.0f; ay = yb ? sy : 0.0f; az = (!xb && !yb) ? sz : 0.0f;
    }
    // d/dp = R^T d/dl
    gx = fmaf(r0.x, ax, fmaf(r1.x, ay, r2.x * az));
    gy = fmaf(r0.y, ax, fmaf(r1.y, ay, r2.y * az));
    gz = fmaf(r0.z, ax, fmaf(r1.z, ay, r2.z * az));
}

// ---------------------------------------------------------------------------
// ESDF (scene_collision.cuh:186-331); trilinear mode adds value + gradient
// ---------------------------------------------------------------------------
__device__ __forceinline__ int robust_floor(float x) {
    const float nearest = roundf(x);
    if (x - nearest >= 1e-4f) return (int)floorf(x);
    return (int)nearest;
}

// Stored inverse pose (t, qw | qx, qy, qz, pad) applied to a world point.
__device__ __forceinline__ void quat_local(const float4& p0, const float4& p1, float sx, float sy, float sz, float& lx,
                                           float& ly, float& lz) {
    const float qw = p0.w, qx = p1.x, qy = p1.y, qz = p1.z;
    const float tx = 2.0f * (qy * sz - qz * sy);
    const float ty = 2.0f * (qz * sx - qx * sz);
    const float tz = 2.0f * (qx * sy - qy * sx);
    lx = sx + qw * tx + (qy * tz - qz * ty) + p0.x;
    ly = sy + qw * ty + (qz * tx - qx * tz) + p0.y;
    lz = sz + qw * tz + (qx * ty - qy * tx) + p0.z;
}

// Minimum ESDF clearance (-dist - r) over enabled layers, 1000 when none
// applies. With `want_grad` (trilinear only) returns d dist / d p (world)
// of the winning layer in g*.
__device__ float esdf_clearance(const DScene& S, float px, float py, float pz, float r, int sph_orig, bool want_grad,
                                float& gx, float& gy, float& gz) {
    float best = 1000.0f;
    gx = gy = gz = 0.0f;
    for (int layer = 0; layer < S.n_voxel_layers; ++layer) {
        if (S.voxel_enable[layer] == 0) continue;
        if (sph_orig >= 0 && S.sphere_acm && S.sphere_acm[sph_orig * S.n_voxel_layers + layer] == 0) continue;
        const float* prm = S.voxel_params + 4 * layer;
        const float* pose = S.voxel_pose + 8 * layer;
        const float vs = prm[3];
        if (vs <= 0.0f) continue;
        const float inv_vs = 1.0f / vs;
        const int nx = robust_floor(prm[0] * inv_vs) + 1;
        const int ny = robust_floor(prm[1] * inv_vs) + 1;
        const int nz = robust_floor(prm[2] * inv_vs) + 1;
        float lx, ly, lz;
        quat_local(make_float4(pose[0], pose[1], pose[2], pose[3]), make_float4(pose[4], pose[5], pose[6], pose[7]), px, py, pz,
                   lx, ly, lz);
        const float ux = (lx + prm[0] * 0.5f) * inv_vs, uy = (ly + prm[1] * 0.5f) * inv_vs, uz = (lz + prm[2] * 0.5f) * inv_vs;
        const float* feat = S.voxel_features + (size_t)layer * S.max_voxels_per_layer;
        if (S.esdf_interp == 0) {
            const int ix = (int)ux, iy = (int)uy, iz = (int)uz;
            if (ix >= nx - 2 || iy >= ny - 2 || iz >= nz - 2 || ix <= 2 || iy <= 2 || iz <= 2) continue;
            const long lin = (long)ix * ny * nz + (long)iy * nz + iz;
            if (lin >= S.max_voxels_per_layer) continue;
            const float d = feat[lin];
            if (d <= -999.0f) continue;
            const float c = -d - r;
            if (c < best) { best = c; gx = gy = gz = 0.0f; }
        } else {
            const float fx0 = floorf(ux), fy0 = floorf(uy), fz0 = floorf(uz);
            const int ix = (int)fx0, iy = (int)fy0, iz = (int)fz0;
            if (ix >= nx - 2 || iy >= ny - 2 || iz >= nz - 2 || ix <= 2 || iy <= 2 || iz <= 2) continue;
            const long base = (long)ix * ny * nz + (long)iy * nz + iz;
            if (base + (long)ny * nz + nz + 1 >= S.max_voxels_per_layer) continue;
            const long sx = (long)ny * nz, sy = nz;
            const float c000 = feat[base], c001 = feat[base + 1], c010 = feat[base + sy], c011 = feat[base + sy + 1];
            const float c100 = feat[base + sx], c101 = feat[base + sx + 1], c110 = feat[base + sx + sy], c111 = feat[base + sx + sy + 1];
            const float mn = fminf(fminf(fminf(c000, c001), fminf(c010, c011)), fminf(fminf(c100, c101), fminf(c110, c111)));
            if (mn <= -999.0f) continue;
            const float fx = ux - fx0, fy = uy - fy0, fz = uz - fz0;
            const float c00 = fmaf(c100 - c000, fx, c000), c01 = fmaf(c101 - c001, fx, c001);
            const float c10 = fmaf(c110 - c010, fx, c010), c11 = fmaf(c111 - c011, fx, c011);
            const float c0 = fmaf(c10 - c00, fy, c00), c1 = fmaf(c11 - c01, fy, c01);
            const float d = fmaf(c1 - c0, fz, c0);
            const float c = -d - r;
            if (c < best) {
                best = c;
                if (want_grad) {
                    const float ofy = 1.0f - fy, ofz = 1.0f - fz;
                    const float dx = ((c100 - c000) * ofy * ofz + (c101 - c001) * ofy * fz + (c110 - c010) * fy * ofz +
                                      (c111 - c011) * fy * fz) * inv_vs;
                    const float dy = ((c10 - c00) * ofz + (c11 - c01) * fz) * inv_vs;
                    const float dz = (c1 - c0) * inv_vs;
                    // grid-local -> world: inverse quaternion rotation
                    const float qw = pose[3], qx = -pose[4], qy = -pose[5], qz = -pose[6];
                    const float tx = 2.0f * (qy * dz - qz * dy), ty = 2.0f * (qz * dx - qx * dz), tz = 2.0f * (qx * dy - qy * dx);
                    gx = dx + qw * tx + (qy * tz - qz * ty);
                    gy = dy + qw * ty + (qz * tx - qx * tz);
                    gz = dz + qw * tz + (qx * ty - qy * tx);
                }
            }
        }
    }
    return best;
}

__device__ __forceinline__ bool esdf_hit(const DScene& S, float px, float py, float pz, float r, int sph_orig) {
    float gx, gy, gz;
    // min clearance < 0  <=>  some layer has dist > -r
    return esdf_clearance(S, px, py, pz, r, sph_orig, false, gx, gy, gz) < 0.0f;
}

// A single trilinear layer without masks, the usual world: its parameters once
// per wave instead of once per lookup, and the lookup split in two so that two
// spheres' grid loads can be in flight together. Values and gradients equal
// esdf_clearance's.
__host__ __device__ inline bool esdf_single(const DScene& S) {
    return S.n_voxel_layers == 1 && S.esdf_interp != 0 && !S.sphere_acm;
}
struct EsdfLayer {
    float4 prm, p0, p1;
    float inv_vs;
    int nx, ny, nz, max_lin;
    bool on;   // enabled, with a voxel size: else it has no inside
    const float* feat;
    EsdfLayer() = default;
    __device__ __forceinline__ explicit EsdfLayer(const DScene& S)
        : prm(uload4<f4s>(S.voxel_params, 0)), p0(uload4<f4s>(S.voxel_pose, 0)), p1(uload4<f4s>(S.voxel_pose, 1)) {
        on = S.voxel_enable[0] != 0 && prm.w > 0.0f;
        inv_vs = uniform(1.0f / prm.w);
        nx = uniform(robust_floor(prm.x * inv_vs) + 1);
        ny = uniform(robust_floor(prm.y * inv_vs) + 1);
        nz = uniform(robust_floor(prm.z * inv_vs) + 1);
        feat = S.voxel_features;
        max_lin = S.max_voxels_per_layer;
    }
};
struct EsdfTap {
    float fx, fy, fz;
    bool ok;
    float c000, c001, c010, c011, c100, c101, c110, c111;
    __device__ __forceinline__ void load(const EsdfLayer& L, float px, float py, float pz, bool on) {
        float lx, ly, lz;
        quat_local(L.p0, L.p1, px, py, pz, lx, ly, lz);
        const float ux = (lx + L.prm.x * 0.5f) * L.inv_vs, uy = (ly + L.prm.y * 0.5f) * L.inv_vs,
                    uz = (lz + L.prm.z * 0.5f) * L.inv_vs;
        const float fx0 = floorf(ux), fy0 = floorf(uy), fz0 = floorf(uz);
        const int ix = (int)fx0, iy = (int)fy0, iz = (int)fz0;
        fx = ux - fx0; fy = uy - fy0; fz = uz - fz0;
        ok = on && L.on && !(ix >= L.nx - 2 || iy >= L.ny - 2 || iz >= L.nz - 2 || ix <= 2 || iy <= 2 || iz <= 2);
        const long sx = (long)L.ny * L.nz, sy = L.nz;
        const long base = ok ? (long)ix * sx + (long)iy * sy + iz : 0;
        ok = ok && base + sx + sy + 1 < L.max_lin;
        if (ok) {
            const float* f = L.feat + base;
            c000 = f[0]; c001 = f[1]; c010 = f[sy]; c011 = f[sy + 1];
            c100 = f[sx]; c101 = f[sx + 1]; c110 = f[sx + sy]; c111 = f[sx + sy + 1];
        }
    }
    __device__ __forceinline__ float value(float r) const {
        if (!ok) return 1000.0f;
        const float mn = fminf(fminf(fminf(c000, c001), fminf(c010, c011)), fminf(fminf(c100, c101), fminf(c110, c111)));
        if (mn <= -999.0f) return 1000.0f;
        const float c00 = fmaf(c100 - c000, fx, c000), c01 = fmaf(c101 - c001, fx, c001);
        const float c10 = fmaf(c110 - c010, fx, c010), c11 = fmaf(c111 - c011, fx, c011);
        const float c0 = fmaf(c10 - c00, fy, c00), c1 = fmaf(c11 - c01, fy, c01);
        const float d = fmaf(c1 - c0, fz, c0);
        const float c = -d - r;
        return c < 1000.0f ? c : 1000.0f;
    }
    // d dist / d p (world); only where value() is below its 1000
    __device__ __forceinline__ void grad(const EsdfLayer& L, float& gx, float& gy, float& gz) const {
        const float c00 = fmaf(c100 - c000, fx, c000), c01 = fmaf(c101 - c001, fx, c001);
        const float c10 = fmaf(c110 - c010, fx, c010), c11 = fmaf(c111 - c011, fx, c011);
        const float c0 = fmaf(c10 - c00, fy, c00), c1 = fmaf(c11 - c01, fy, c01);
        const float ofy = 1.0f - fy, ofz = 1.0f - fz;
        const float dx = ((c100 - c000) * ofy * ofz + (c101 - c001) * ofy * fz + (c110 - c010) * fy * ofz +
                          (c111 - c011) * fy * fz) * L.inv_vs;
        const float dy = ((c10 - c00) * ofz + (c11 - c01) * fz) * L.inv_vs;
        const float dz = (c1 - c0) * L.inv_vs;
        const float qw = L.p0.w, qx = -L.p1.x, qy = -L.p1.y, qz = -L.p1.z;
        const float tx = 2.0f * (qy * dz - qz * dy), ty = 2.0f * (qz * dx - qx * dz), tz = 2.0f * (qx * dy - qy * dx);
        gx = dx + qw * tx + (qy * tz - qz * ty);
        gy = dy + qw * ty + (qz * tx - qx * tz);
        gz = dz + qw * tz + (qx * ty - qy * tx);
    }
};


// ---------------------------------------------------------------------------
// State resolution: flattened state index -> per-lane q in LDS
// ---------------------------------------------------------------------------
__device__ __forceinline__ int upper_bound_idx(const int* off, int n, long g) {
    // largest e in [0, n) with off[e] <= g
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= g) lo = mid; else hi = mid;
    }
    return lo;
}

struct StateRef {
    int unit;      // config / edge / trajectory index
    int k;         // edge state index or waypoint index
    int n;         // edge states (incl. skipped) or trajectory length
    long u0;       // plan-order index of the unit's first state
    long gs;       // plan-order index of the state (differs from the chunk index when waypoint-major)
};

// State ranges of units u0 .. u0+63 into LDS: s_end[i] = off[u0+i+1] and
// s_end[64+i] = off[u0+i] (whole wave; no-op for configuration sources or
// when the chunk's first unit is unknown, u0 < 0).
__device__ __forceinline__ void stage_unit_ends(const DStates& X, int u0, int* s_end) {
    if (X.source == kSrcConfig || u0 < 0) return;
    const bool dense = X.source == kSrcDense || X.source == kSrcBfs;
    const int* off = X.source == kSrcEdge ? X.edge_off : dense ? X.dense_off : X.traj_off;
    const int n = X.source == kSrcEdge ? X.n_edges : X.n_traj;
    const int u = u0 + lane_id();
    const bool in = u < n;
    s_end[lane_id()] = in ? off[u + 1] : INT_MAX;
    s_end[kWave + lane_id()] = in ? off[u] : INT_MAX;
}

// The same two loads into registers, for a chunk ahead.
__device__ __forceinline__ void prefetch_unit_ends(const DStates& X, int u0, int& e_end, int& e_beg) {
    if (X.source == kSrcConfig || u0 < 0) return;
    const bool dense = X.source == kSrcDense || X.source == kSrcBfs;
    const int* off = X.source == kSrcEdge ? X.edge_off : dense ? X.dense_off : X.traj_off;
    const int n = X.source == kSrcEdge ? X.n_edges : X.n_traj;
    const int u = u0 + lane_id();
    const bool in = u < n;
    e_end = in ? off[u + 1] : INT_MAX;
    e_beg = in ? off[u] : INT_MAX;
}

// Unit holding state g and its state range [*u_begin, *u_end): the first of
// units u0 .. u0+63 whose end exceeds g (bisection over the staged ends),
// else a binary search over the offset table.
__device__ __forceinline__ int find_unit(const int* off, int n, long g, int u0, const int* s_end, int* u_begin,
                                         int* u_end) {
    if (u0 >= 0 && s_end[kWave - 1] > g) {
        int lo = 0, hi = kWave - 1;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (s_end[mid] > g) hi = mid; else lo = mid + 1;
        }
        *u_begin = s_end[kWave + lo];
        *u_end = s_end[lo];
        return u0 + lo;
    }
    const int u = upper_bound_idx(off, n, g);
    *u_begin = off[u];
    *u_end = off[u + 1];
    return u;
}

// out(d, get(d)) for d < n, eight loads in flight at a time (a plain loop waits
// for each one; past the end the last is loaded and written again).
template <class Get, class Out>
__device__ __forceinline__ void each_dof(int n, const Get& get, const Out& out) {
    for (int d0 = 0; d0 < n; d0 += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = get(min(d0 + k, n - 1));
#pragma unroll
        for (int k = 0; k < 8; ++k) out(min(d0 + k, n - 1), v[k]);
    }
}

// Writes q_d into s_q[d * 64 + lane] for d < D (inactive lanes write nothing).
// g is the chunk-order index; prob the chunk's problem (waypoint-major plans).
// qcol / qstride: where q_d goes, s_q[d * qstride + qcol] (default: the
// lane's own column of a [D][64] array).
// store = false resolves the state without writing q (lanes that share a
// column with a storing lane).
__device__ __forceinline__ StateRef load_state(const DStates& X, int D, long g, bool active, float* s_q,
                                               int u0 = -1, const int* s_end = nullptr, int prob = 0,
                                               int qcol = -1, int qstride = kWave, bool store = true) {
    StateRef ref{0, 0, 0, 0, g};
    const int lane = qcol >= 0 ? qcol : lane_id();
    const int nd = store ? D : 0;   // dimensions to write
    if (!active) return ref;
    auto put = [&](int d, float v) { s_q[d * qstride + lane] = v; };
    if (X.source == kSrcDense) {
        int d0, d1;
        const int b = find_unit(X.dense_off, X.n_traj, g, u0, s_end, &d0, &d1);
        const int t0 = X.traj_off[b], T = X.traj_off[b + 1] - t0;
        const int ns = X.nsub[b];
        const int f = (int)(g - d0);
        ref.unit = b;
        ref.k = f;
        ref.n = (T - 1) * ns + 1;
        ref.u0 = d0;
        const float* th = X.theta + (size_t)t0 * D;
        if (f >= (T - 1) * ns) {
            each_dof(nd, [&](int d) { return th[(size_t)d * T + T - 1]; }, put);
        } else {
            const int seg = f / ns, sub = f - seg * ns;
            const float frac = __fdiv_rn((float)sub, (float)ns);
            each_dof(nd, [&](int d) {
                const float x0 = th[(size_t)d * T + seg], x1 = th[(size_t)d * T + seg + 1];
                return __fadd_rn(x0, __fmul_rn(__fsub_rn(x1, x0), frac));
            }, put);
        }
        return ref;
    }
    if (X.source == kSrcBfs) {
        // MIT*'s edge midpoints (MITStar.cu:938-965, 1316-1330): level
        // L = floor(log2(k + 1)), t = (2 (k + 1 - 2^L) + 1) / 2^(L + 1), and
        // q = q_src (1 - t) + q_dst t as written (no contraction)
        int e0, e1;
        const int e = find_unit(X.dense_off, X.n_traj, g, u0, s_end, &e0, &e1);
        const int f = (int)(g - e0);
        const int k = X.bfs_k0[e] + f;
        ref.unit = e;
        ref.k = f;
        ref.n = e1 - e0;
        ref.u0 = e0;
        const int kk = k + 1;
        const int lvl = 31 - __clz(kk);
        const float t = __fdiv_rn((float)(2 * (kk - (1 << lvl)) + 1), (float)(1 << (lvl + 1)));
        const float* a = X.cfg + (size_t)X.node_src[e] * X.cfg_stride;
        const float* b = X.cfg + (size_t)X.node_dst[e] * X.cfg_stride;
        each_dof(nd, [&](int d) { return __fadd_rn(__fmul_rn(a[d], 1.0f - t), __fmul_rn(b[d], t)); }, put);
        return ref;
    }
    if (X.source == kSrcTraj && X.wmajor) {
        const int4 pr = X.prob[prob];
        const int v = (int)(g - pr.w);
        const int t = v / pr.y, r = v - t * pr.y;
        ref.unit = pr.x + r;
        ref.k = t;
        ref.n = pr.z;
        ref.u0 = (long)pr.w + (long)r * pr.z;
        ref.gs = ref.u0 + t;
        const float* th = X.theta + (size_t)ref.u0 * D;
        each_dof(nd, [&](int d) { return th[(size_t)d * pr.z + t]; }, put);
        return ref;
    }
    if (X.source == kSrcConfig) {
        ref.unit = (int)g;
        ref.u0 = g;
        const float* q = X.cfg + (size_t)g * X.cfg_stride;
        each_dof(nd, [&](int d) { return q[d]; }, put);
    } else if (X.source == kSrcEdge) {
        int b0, b1;
        const int e = find_unit(X.edge_off, X.n_edges, g, u0, s_end, &b0, &b1);
        const int cnt = b1 - b0;
        ref.unit = e;
        ref.u0 = b0;
        ref.k = (int)(g - b0) + X.k0;
        ref.n = cnt + X.k0;
        const float t = ref.n > 1 ? (float)ref.k / (float)(ref.n - 1) : 0.0f;
        const float* a = X.from + (size_t)e * D;
        const float* b = X.to + (size_t)e * D;
        each_dof(nd, [&](int d) { return fmaf(t, b[d] - a[d], a[d]); }, put);
    } else {
        int t0, t1;
        const int b = find_unit(X.traj_off, X.n_traj, g, u0, s_end, &t0, &t1);
        const int Tn = t1 - t0;
        ref.unit = b;
        ref.u0 = t0;
        ref.k = (int)(g - t0);
        ref.n = Tn;
        const float* th = X.theta + (size_t)t0 * D;
        each_dof(nd, [&](int d) { return th[(size_t)d * Tn + ref.k]; }, put);
    }
    return ref;
}

// Static, XCD-aware chunk schedule (no atomics). Workgroups are dispatched
// round-robin over the 8 XCDs, so workgroup w runs on XCD w % 8; its logical
// rank puts every XCD on a contiguous block of chunks in each sweep, which
// keeps neighbouring states (shared edge endpoints, trajectories, OBB sets)
// in one L2. Chunk c = rank + k * grid for k = 0, 1, ...: every wave reaches
// the end of the table, and chunks are visited roughly in table order.
struct ChunkCursor {
    int next;
    int stride;
};

__device__ __forceinline__ ChunkCursor chunk_cursor() {
    const int W = gridDim.x, w = blockIdx.x;
    constexpr int kXcds = 8;
    const int rank = (W % kXcds == 0) ? (w % kXcds) * (W / kXcds) + w / kXcds : w;
    return ChunkCursor{rank, W};
}

// Chunk count of a launch: the table's, or ceil(states / chunk) for implicit
// chunks (the state count may come from device memory).
__device__ __forceinline__ int chunk_count(const DChunks& C, long n_states) {
    return C.tab ? C.n_chunks : (int)((n_states + C.chunk - 1) / C.chunk);
}

__device__ __forceinline__ long state_count(const DStates& X) { return X.n_dyn ? (long)uniform(*X.n_dyn) : X.n_states; }

__device__ __forceinline__ bool next_chunk(const DChunks& C, long n_states, int n_chunks, ChunkCursor& cur, int4& ch) {
    int c = cur.next;
    if (C.spread) {
        // a bijection of [0, 2^m) >= n_chunks that sends neighbours far apart
        // (odd multiplier near 2^32 over the golden ratio)
        const unsigned mask = n_chunks > 1 ? 0xFFFFFFFFu >> __builtin_clz((unsigned)(n_chunks - 1)) : 0u;
        for (;;) {
            if ((unsigned)cur.next > mask || n_chunks <= 0) return false;
            c = (int)(((unsigned)cur.next * 0x9E3779B1u) & mask);
            cur.next += cur.stride;
            if (c < n_chunks) break;
        }
    } else {
        if (c >= n_chunks) return false;
        cur.next += cur.stride;
    }
    if (C.tab) {
        ch = C.tab[c];
        ch.x = uniform(ch.x); ch.y = uniform(ch.y); ch.z = uniform(ch.z); ch.w = uniform(ch.w);
    } else {
        const long b = (long)c * C.chunk;
        const int u = C.unit_hint ? uniform(C.unit_hint[b >> 6]) : -1;
        ch = make_int4(0, (int)b, (int)(b + C.chunk < n_states ? b + C.chunk : n_states), u);
    }
    return true;
}

__device__ __forceinline__ void problem_obbs(const DChunks& C, const DScene& S, int prob, int& o0, int& o1) {
    if (C.obb_off) { o0 = C.obb_off[prob]; o1 = C.obb_off[prob + 1]; }
    else { o0 = 0; o1 = S.n_obbs; }
}

// Wave-uniform OBB candidate set: bit o set for OBB o (up to kMaxObbLds).
constexpr int kMaskWords = kMaxObbLds / 64;

struct ObbMask {
    unsigned long long w[kMaskWords];
};

__device__ __forceinline__ float read_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Over the 16 lanes of a row (lanes 16 k .. 16 k + 15), by row rotations.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_sum(float v) {
    v += dpp<0x128>(v);
    v += dpp<0x124>(v);
    v += dpp<0x122>(v);
    return v + dpp<0x121>(v);
}

// Maximum of values that are not negative, in which a NaN stays (fmaxf drops
// it): their bits order as unsigned numbers, NaN above infinity. For bounds that
// a lane which is no number must not pass; a test against one keeps what it
// cannot rule out.
__device__ __forceinline__ float max_nan(float a, float b) {
    return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
}
__device__ __forceinline__ float row_max_nan(float v) {
    v = max_nan(v, dpp<0x128>(v));
    v = max_nan(v, dpp<0x124>(v));
    v = max_nan(v, dpp<0x122>(v));
    return max_nan(v, dpp<0x121>(v));
}

// Whether a place may enter a mean: finite, and 64 of them sum and square
// within FP32. (With none, the mean is NaN.)
__device__ __forceinline__ bool usable(float x, float y, float z) {
    return fabsf(x) + fabsf(y) + fabsf(z) < 1e16f;
}

// A row's 16 bits of a ballot (row: its first lane).
__device__ __forceinline__ unsigned row_bits(unsigned long long m, int row) {
    const unsigned w = row >= 32 ? (unsigned)(m >> 32) : (unsigned)m;
    return (w >> (row & 16)) & 0xFFFFu;
}

// Lanes below this one set in a ballot.
__device__ __forceinline__ int rank_below(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// ===========================================================================
// Any-collision: two-phase gate semantics (two_phase_cc.cuh:57-138 with the
// check kernel's environment pass, pRRTC.cu:2337-2386).
// ===========================================================================
// A lane per state walks the joints; per joint, three steps narrow the (state,
// box) pairs down to the exact sphere tests:
//  1. each row of 16 lanes holds 16 consecutive states, whose approximate
//     spheres lie within rw of a middle one's centre c0: every box one of them
//     overlaps lies within rw + r of c0 (slack covers rounding). The row's
//     lanes test 16 boxes at once;
//  2. each lane tests its own approximate sphere against its row's candidates;
//  3. the pairs that hit are queued in LDS and taken 64 at a time, one pair
//     per lane (fewer pairs: several lanes share one, each a part of the
//     joint's spheres), with the frame out of the state's own lane.
// Bound by VALU and SALU issue. With one candidate set for the whole wave, and
// the exact spheres of a pair tested in all lanes as soon as one lane has it, a
// wave goes through 100 candidates and 12 exact boxes on 16,384 edges among 64
// boxes, of which its states need 2.7 x 64 pairs; on uncorrelated
// configurations (20 boxes) 89 and 31, needing 1.4 x 64. Together with the
// scalar table loads and the grid (kCollideWaves): the edges 321 -> 179 us a
// call, 262,144 configurations of 64 requests 135 -> 48 us, 11 densified
// validity passes of 256 trajectories 258 -> 170 us each.
// Records lie five float4s apart: the 16 boxes that a row's lanes read at once
// then start in different LDS banks (four apart they shared four of them, and
// conflicts took 53 us of the CU's LDS time on the edges above).
constexpr int kObbRec = 5;

// ESDF: the scene has voxel layers (a variant of its own: the lookups cost the
// box-only kernel registers).
// LINE: the model is a line of joints (FkWalk), which saves the slots' registers.
// P: lanes per state. With 4 each row holds the chunk's same 16 states and takes
// every fourth box (where: kCollideSplit): uncorrelated states have most boxes
// among their candidates, which one lane takes one after the other; 256 Panda
// configurations among 20 boxes 35 -> 21 us, 52.9 -> 39.6 us a call from the host.
template <bool ESDF, bool LINE, int P>
__global__ __launch_bounds__(64, 4) void k_collide(CollideArgs a) {
    static_assert(P == 1 || P == 4, "a row of 16 lanes per part");
    constexpr bool SPLIT = P == 4;
    constexpr int kStates = kWave / P;
    extern __shared__ float4 s_lds[];
    float4* s_obb = s_lds;
    float4* s_sph = s_lds + kObbRec * a.C.obb_cap;                    // [S]
    float* s_q = reinterpret_cast<float*>(s_sph + a.R.n_sph);
    const DRobot& R = a.R;
    const int lane = lane_id();
    const int J = R.n_joints, D = R.n_dof;
    int* s_end = reinterpret_cast<int*>(s_q + D * kWave);       // [2][64] unit ends, then
    int* s_queue = s_end;                                       // [128] pairs: lane | box << 8
    int* s_hit = s_end + 2 * kWave;                             // [64] states hit in a flush
    const int row = lane & 48;                                  // the lane's row of 16
    const int part = SPLIT ? lane >> 4 : 0, slot = lane & (kStates - 1);
    for (int k = lane; k < R.n_sph; k += kWave) s_sph[k] = R.sph[k];
    const uint8_t* acm = a.S.sphere_obb_acm;
    const int cap = a.C.obb_cap;
    int cur_prob = -1, n_obb = 0, o0 = 0, o1 = 0, n_tiles = 1;
    int4 ch;
    ChunkCursor cur = chunk_cursor();
    const long n_states = state_count(a.X);
    const int n_chunks = chunk_count(a.C, n_states);
    // the next chunk's table entry is loaded at the top of each round and its
    // unit ends once this chunk's states are in, so both arrive during the
    // joint loop instead of heading the next round's chain of loads
    bool have = next_chunk(a.C, n_states, n_chunks, cur, ch);
    int pf_end = 0, pf_beg = 0;
    if (have) prefetch_unit_ends(a.X, ch.w, pf_end, pf_beg);
    while (have) {
        int4 chn;
        const bool have_n = next_chunk(a.C, n_states, n_chunks, cur, chn);
        // a chunk inside one unit that already has its hit (read past the
        // caches, which would keep an old entry for the whole launch)
        if (a.any && ch.w >= 0 && __builtin_amdgcn_readlane(pf_end, 0) >= ch.z &&
            __hip_atomic_load(a.first_hit + ch.w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= 0) {
            if (have_n) prefetch_unit_ends(a.X, chn.w, pf_end, pf_beg);
            ch = chn;
            have = have_n;
            continue;
        }
        if (ch.x != cur_prob) {
            problem_obbs(a.C, a.S, ch.x, o0, o1);
            n_tiles = uniform(obb_tiles(o0, o1, cap));
            if (n_tiles == 1) {
                __syncthreads();
                n_obb = uniform(stage_obbs<kObbRec>(a.S, o0, o1, s_obb, cap));
            }
            cur_prob = ch.x;
        }
        const long g = (long)ch.y + slot;
        bool active = g < ch.z;
        if (a.X.source != kSrcConfig && ch.w >= 0) {
            s_end[lane] = pf_end;
            s_end[kWave + lane] = pf_beg;
        }
        __syncthreads();
        StateRef ref = load_state(a.X, D, g, active, s_q, ch.w, s_end, ch.x);
        bool hit = false;
        if (active && a.self_hit && a.self_hit[ref.gs]) { hit = true; active = false; }
        if (active && a.mode == 1 && a.skip_resolved) {
            const unsigned fh = (unsigned)a.first_hit[ref.unit];
            if (a.any ? fh != ~0u : fh < (unsigned)ref.k) active = false;
        }
        if (have_n) prefetch_unit_ends(a.X, chn.w, pf_end, pf_beg);
        __syncthreads();
        s_hit[lane] = 0;
        // A problem with more OBBs than one staging holds is checked tile by
        // tile (FK redone per tile); bit jj of `flagged`: joint jj's
        // approximate spheres hit an OBB of an earlier tile, which the ESDF
        // pass of the last tile counts as the joint's flag.
        unsigned flagged = 0u;
        for (int t = 0; t < n_tiles && wave_any(active); ++t) {
            const bool last = t == n_tiles - 1;
            if (n_tiles > 1) {
                const int t0 = o0 + t * cap;
                __syncthreads();
                n_obb = uniform(stage_obbs<kObbRec>(a.S, t0, min(o1, t0 + cap), s_obb, cap));
            }
            FkWalk<LINE> fk;
            float T[12];
            for (int jj = 0; jj < J && wave_any(active); ++jj) {
                int4 meta;
                fk.step(R, jj, s_q + lane, T, meta);
                const int s0 = uload<int>(R.sph_off, jj), s1 = uload<int>(R.sph_off, jj + 1);
                const int a0 = uload<int>(R.apx_off, jj), a1 = uload<int>(R.apx_off, jj + 1);
                if (s1 == s0 || a1 == a0) continue;
                bool flag = false;
                int qn = 0;              // pairs queued
                // 3. exact tests of the queued pairs; states found to collide leave `active`
                auto flush = [&]() {
                    __syncthreads();
                    const int ns = s1 - s0;
                    for (int q0 = 0; q0 < qn; q0 += kWave) {
                        const int n = min(kWave, qn - q0);
                        const int sh = n <= 8 ? 3 : n <= 16 ? 2 : n <= 32 ? 1 : 0;   // 2^sh lanes per pair
                        const int i = lane >> sh, k0 = lane & ((1 << sh) - 1);
                        const bool on = i < n;
                        const int item = s_queue[q0 + (on ? i : 0)];
                        const int l = item & 0xFF, o = item >> 8;
                        const float4 r0 = s_obb[kObbRec * o], r1 = s_obb[kObbRec * o + 1], r2 = s_obb[kObbRec * o + 2], h = s_obb[kObbRec * o + 3];
                        float Tl[12];   // the state's frame, from its own lane
#pragma unroll
                        for (int c = 0; c < 12; ++c) Tl[c] = __shfl(T[c], l);
                        // M = R_o * T_j: sphere-local -> box-local in one affine map.
                        float M[12];
#pragma unroll
                        for (int rr = 0; rr < 3; ++rr) {
                            const float4 rw = rr == 0 ? r0 : (rr == 1 ? r1 : r2);
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                float v = fmaf(rw.z, Tl[8 + c], fmaf(rw.y, Tl[4 + c], rw.x * Tl[c]));
                                if (c == 3) v += rw.w;
                                M[rr * 4 + c] = v;
                            }
                        }
                        bool h_any = false;
                        for (int k = k0; k < ns; k += 1 << sh) {
                            const float4 sp = s_sph[s0 + k];
                            float x, y, z;
                            aff_point(M, sp.x, sp.y, sp.z, x, y, z);
                            const float rr = sp.w + a.margin;
                            bool hs = box_hit(x, y, z, h, rr * rr);
                            if (acm) hs = hs && acm[(size_t)R.sph_id[s0 + k] * a.S.n_obbs + __float_as_int(h.w)] != 0;
                            h_any = h_any || hs;
                        }
                        if (on && h_any) s_hit[l & (kStates - 1)] = 1;
                    }
                    __syncthreads();
                    hit = hit || (active && s_hit[slot] != 0);
                    active = active && !hit;
                    qn = 0;
                };
                // each approximate sphere of the joint (usually one)
                for (int ai = a0; ai < a1; ++ai) {
                    const float4 as = uload4(R.apx, ai);
                    float px, py, pz;
                    aff_point(T, as.x, as.y, as.z, px, py, pz);
                    const float rr = as.w + a.margin;
                    const float apr2 = rr * rr;
                    // 1. the row's centre state (a middle one) and its spread
                    const unsigned in_row = row_bits(__ballot(active), row);
                    const int l0 = row + (in_row >> 8 ? 7 + __ffs(in_row >> 8) : in_row ? __ffs(in_row) - 1 : 0);
                    const float cx = __shfl(px, l0), cy = __shfl(py, l0), cz = __shfl(pz, l0);
                    const float dx = px - cx, dy = py - cy, dz = pz - cz;
                    // (a state that is not finite, at the centre or beside it,
                    // makes the spread no number or infinite, and every box a candidate)
                    const float d2 = row_max_nan(active ? fmaf(dz, dz, fmaf(dy, dy, dx * dx)) : 0.0f);
                    const float reach = __builtin_amdgcn_sqrtf(d2) * 1.0001f + fabsf(rr) + 1e-5f;
                    const float reach2 = reach * reach;
                    for (int base = 0; base < n_obb; base += kWave) {
                        const int m = min(kWave, n_obb - base);
                        unsigned long long todo = 0ull;   // the lane's candidates
#pragma unroll
                        for (int r = 0; r < (SPLIT ? 1 : 4); ++r) {
                            if (16 * r >= m) break;
                            // past the last box: its record again, masked off
                            const int k = SPLIT ? 4 * (lane & 15) + part : 16 * r + (lane & 15), o = base + min(k, m - 1);
                            float lx, ly, lz;
                            to_box(s_obb[kObbRec * o], s_obb[kObbRec * o + 1], s_obb[kObbRec * o + 2], cx, cy, cz, lx, ly, lz);
                            const bool c = k < m && !(box_dist2(lx, ly, lz, s_obb[kObbRec * o + 3]) > reach2);
                            todo |= (unsigned long long)row_bits(__ballot(c), row) << (16 * r);
                        }
                        if (!active) todo = 0ull;
                        while (wave_any(todo != 0ull)) {
                            // 2. the lane's own approximate sphere against its next candidate
                            const bool on = todo != 0ull;
                            const int o = base + (on ? P * (__ffsll(todo) - 1) + part : 0);
                            todo &= todo - 1ull;
                            float lx, ly, lz;
                            to_box(s_obb[kObbRec * o], s_obb[kObbRec * o + 1], s_obb[kObbRec * o + 2], px, py, pz, lx, ly, lz);
                            const bool ah = box_hit(lx, ly, lz, s_obb[kObbRec * o + 3], apr2) && on;
                            flag = flag || ah;
                            const unsigned long long push = __ballot(ah);
                            if (push == 0ull) continue;
                            if (ah) s_queue[qn + rank_below(push)] = lane | (o << 8);
                            qn += __popcll(push);
                            if (qn >= kWave) {
                                flush();
                                if (!active) todo = 0ull;
                            }
                        }
                    }
                }
                if (qn > 0) flush();
                if (!last) {
                    if (flag) flagged |= 1u << jj;
                    continue;
                }
                flag = flag || ((flagged >> jj) & 1u) != 0u;
                if (ESDF) {
                    if (SPLIT) {   // some part's
                        const unsigned long long fm = __ballot(flag);
                        flag = (((fm | fm >> 32) | (fm | fm >> 32) >> 16) >> slot & 1u) != 0u;
                    }
                    // Approx ESDF pass (ACM disabled, scene_collision.cuh:574-582),
                    // then the joint's exact spheres when it is flagged.
                    for (int ai = a0; ai < a1; ++ai) {
                        const float4 as = uload4(R.apx, ai);
                        float x, y, z;
                        aff_point(T, as.x, as.y, as.z, x, y, z);
                        flag = flag || (active && esdf_hit(a.S, x, y, z, as.w + a.margin, -1));
                    }
                    if (wave_any(flag && active)) {
                        for (int s = s0; s < s1; ++s) {
                            const float4 sp = uload4(R.sph, s);
                            float x, y, z;
                            aff_point(T, sp.x, sp.y, sp.z, x, y, z);
                            const bool hs = flag && active && esdf_hit(a.S, x, y, z, sp.w + a.margin, R.sph_id[s]);
                            hit = hit || hs;
                        }
                        active = active && !hit;
                    }
                }
            }
        }
        if (part == 0 && g < ch.z && a.out) a.out[ref.gs] = hit ? 1 : 0;
        if (a.mode == 1) {
            // One atomic per (chunk, edge): a hit lane reports only when no
            // lower lane of the same edge hit (lanes hold consecutive states).
            const bool rep = part == 0 && hit && g < ch.z;
            const unsigned long long hm = __ballot(rep);
            if (rep) {
                const int l_e0 = ref.u0 > ch.y ? (int)(ref.u0 - ch.y) : 0;
                const unsigned long long same = ((1ull << lane) - 1ull) & ~((1ull << l_e0) - 1ull);
                if ((hm & same) == 0ull) atomicMin((unsigned*)&a.first_hit[ref.unit], (unsigned)ref.k);
            }
        }
        ch = chn;
        have = have_n;
    }
}

// ===========================================================================
// Any-collision in the gated two-phase form (two_phase_cc.cuh:57-104,
// scene_collision.cuh:519-628), for models whose exact (sphere, box) hits
// need not imply the approximate hit of the same box: approximate spheres
// that do not enclose the exact ones, or that ride a chain of their own.
// The approximate pass flags joints over the whole scene (every enabled box,
// no ACM, then the ESDF layers), then the exact spheres of flagged joints are
// checked against the whole scene (box and layer ACMs). One lane per state,
// OBBs in LDS tiles as in k_collide.
// ===========================================================================
__global__ __launch_bounds__(64) void k_collide_gated(CollideArgs a) {
    extern __shared__ float4 s_lds[];
    float4* s_obb = s_lds;
    float* s_q = reinterpret_cast<float*>(s_lds + 4 * a.C.obb_cap);
    const DRobot& R = a.R;
    const int lane = lane_id();
    const int J = R.n_joints, D = R.n_dof;
    int* s_end = reinterpret_cast<int*>(s_q + D * kWave);
    const bool has_esdf = a.S.n_voxel_layers > 0;
    const bool own_chain = R.aft != nullptr;
    const uint8_t* acm = a.S.sphere_obb_acm;
    const int cap = a.C.obb_cap;
    int cur_prob = -1, n_obb = 0, o0 = 0, o1 = 0, n_tiles = 1;
    int4 ch;
    ChunkCursor cur = chunk_cursor();
    const long n_states = state_count(a.X);
    const int n_chunks = chunk_count(a.C, n_states);
    while (next_chunk(a.C, n_states, n_chunks, cur, ch)) {
        if (ch.x != cur_prob) {
            problem_obbs(a.C, a.S, ch.x, o0, o1);
            n_tiles = uniform(obb_tiles(o0, o1, cap));
            if (n_tiles == 1) {
                __syncthreads();
                n_obb = uniform(stage_obbs(a.S, o0, o1, s_obb, cap));
            }
            cur_prob = ch.x;
        }
        const long g = (long)ch.y + lane;
        bool active = g < ch.z;
        stage_unit_ends(a.X, ch.w, s_end);
        __syncthreads();
        StateRef ref = load_state(a.X, D, g, active, s_q, ch.w, s_end, ch.x);
        bool hit = false;
        if (active && a.self_hit && a.self_hit[ref.gs]) { hit = true; active = false; }
        if (active && a.mode == 1 && a.skip_resolved) {
            const unsigned fh = (unsigned)a.first_hit[ref.unit];
            if (a.any ? fh != ~0u : fh < (unsigned)ref.k) active = false;
        }
        __syncthreads();
        // 1. approximate pass: bit jj of `flagged` once an approximate sphere
        // of joint jj (its own chain's frame) hits an enabled box or a layer
        unsigned flagged = 0u;
        for (int t = 0; t < n_tiles && wave_any(active); ++t) {
            if (n_tiles > 1) {
                const int t0 = o0 + t * cap;
                __syncthreads();
                n_obb = uniform(stage_obbs(a.S, t0, min(o1, t0 + cap), s_obb, cap));
            }
            const bool last = t == n_tiles - 1;
            Slots sl;
            for (int jj = 0; jj < J; ++jj) {
                float T[12];
                int4 meta;
                if (own_chain) fk_joint<true>(R, jj, s_q + lane, sl, T, meta);
                else fk_joint(R, jj, s_q + lane, sl, T, meta);
                for (int ai = R.apx_off[jj]; ai < R.apx_off[jj + 1]; ++ai) {
                    const float4 as = R.apx[ai];
                    float x, y, z;
                    aff_point(T, as.x, as.y, as.z, x, y, z);
                    const float rr = as.w + a.margin;
                    bool f = !active || ((flagged >> jj) & 1u) != 0u;   // nothing left to find
                    for (int o = 0; o < n_obb && wave_any(!f); ++o) {
                        float lx, ly, lz;
                        to_box(s_obb[4 * o], s_obb[4 * o + 1], s_obb[4 * o + 2], x, y, z, lx, ly, lz);
                        f = f || box_hit(lx, ly, lz, s_obb[4 * o + 3], rr * rr);
                    }
                    if (last && has_esdf && !f) f = esdf_hit(a.S, x, y, z, rr, -1);
                    if (active && f) flagged |= 1u << jj;
                }
            }
        }
        // 2. exact pass over the flagged joints' spheres
        for (int t = 0; t < n_tiles && wave_any(active && flagged != 0u); ++t) {
            if (n_tiles > 1) {
                const int t0 = o0 + t * cap;
                __syncthreads();
                n_obb = uniform(stage_obbs(a.S, t0, min(o1, t0 + cap), s_obb, cap));
            }
            const bool last = t == n_tiles - 1;
            Slots sl;
            for (int jj = 0; jj < J && wave_any(active); ++jj) {
                float T[12];
                int4 meta;
                fk_joint(R, jj, s_q + lane, sl, T, meta);
                const bool fj = active && ((flagged >> jj) & 1u) != 0u;
                if (!wave_any(fj)) continue;
                for (int s = R.sph_off[jj]; s < R.sph_off[jj + 1]; ++s) {
                    const float4 sp = R.sph[s];
                    float x, y, z;
                    aff_point(T, sp.x, sp.y, sp.z, x, y, z);
                    const float rr = sp.w + a.margin;
                    const uint8_t* acm_row = acm ? acm + (size_t)R.sph_id[s] * a.S.n_obbs : nullptr;
                    bool hs = false;
                    for (int o = 0; o < n_obb && wave_any(fj && !hs); ++o) {
                        const float4 h = s_obb[4 * o + 3];
                        if (acm_row && acm_row[__float_as_int(h.w)] == 0) continue;
                        float lx, ly, lz;
                        to_box(s_obb[4 * o], s_obb[4 * o + 1], s_obb[4 * o + 2], x, y, z, lx, ly, lz);
                        hs = hs || (fj && box_hit(lx, ly, lz, h, rr * rr));
                    }
                    if (last && has_esdf && fj && !hs) hs = esdf_hit(a.S, x, y, z, rr, R.sph_id[s]);
                    hit = hit || hs;
                }
                active = active && !hit;
            }
        }
        if (g < ch.z && a.out) a.out[ref.gs] = hit ? 1 : 0;
        if (a.mode == 1) {
            const bool rep = hit && g < ch.z;
            const unsigned long long hm = __ballot(rep);
            if (rep) {
                const int l_e0 = ref.u0 > ch.y ? (int)(ref.u0 - ch.y) : 0;
                const unsigned long long same = ((1ull << lane) - 1ull) & ~((1ull << l_e0) - 1ull);
                if ((hm & same) == 0ull) atomicMin((unsigned*)&a.first_hit[ref.unit], (unsigned)ref.k);
            }
        }
    }
}

// ===========================================================================
// Summed-hinge state cost (+ adjoint). chomp.cu:151-188 / stomp.cu:206-246
// cost = w * (sum_s relu(m - min_o clr(s,o)) + sum_s relu(m - esdf clr(s))
//             + relu(m_self - min_pairs clr)), raw radii.
// Gradient: every sphere s with a non-zero point gradient g_s adds, for each
// ancestor joint j of its link, g_s . (z_j x (p_s - o_j)) (revolute) or
// g_s . z_j (prismatic), with z_j, o_j the joint's world axis and origin
// recorded during the forward walk. Lever arms are taken relative to each
// joint, so no large world-origin moments are summed and subtracted.
// ===========================================================================
// Candidate OBBs of one sphere cluster for the hinge: a wave-uniform bitmask
// of the OBBs some active lane's spheres of the cluster can come within the
// hinge band of. Every sphere s of the cluster lies inside its enclosing
// sphere `as` (centre a, radius R; DRobot::clu_enc), so clr(s, o) >=
// sdf_o(a) - R; the active lanes' centres lie within rw of c0, the mean of
// those at usable places (another one makes rw infinite or no number), so
// sdf_o(a) >= sdf_o(c0) - rw. An OBB with sdf_o(c0) >= band + R + rw therefore
// has clearance >= band from every sphere: it cannot change a hinge, its argmin
// or its gradient. One pass per 64 OBBs (lane i tests OBB base + i).
template <int STRIDE>
__device__ __forceinline__ void near_obbs(const float4* __restrict__ s_obb, int n_obb, const float* T, const float4& as,
                                          float band, bool active, unsigned long long* w) {
    float ax, ay, az;
    aff_point(T, as.x, as.y, as.z, ax, ay, az);
    auto wave = [](float v) {   // a row's value in each of its lanes -> the four rows'
        return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
    };
    const bool in = active && usable(ax, ay, az);
    const float inv_n = __builtin_amdgcn_rcpf((float)__popcll(__ballot(in)));
    const float cx = wave(row_sum(in ? ax : 0.0f)) * inv_n, cy = wave(row_sum(in ? ay : 0.0f)) * inv_n,
                cz = wave(row_sum(in ? az : 0.0f)) * inv_n;
    const float dx = ax - cx, dy = ay - cy, dz = az - cz;
    const float v = row_max_nan(active ? fmaf(dz, dz, fmaf(dy, dy, dx * dx)) : 0.0f);
    const float d2 = max_nan(max_nan(read_lane(v, 0), read_lane(v, 16)), max_nan(read_lane(v, 32), read_lane(v, 48)));
    // sdf(c0) < reach  <=>  key(c0) < reach * |reach|; slack covers rounding
    const float reach = band + as.w + __builtin_amdgcn_sqrtf(d2) * 1.0001f + 1e-5f;
    const float thr = reach * fabsf(reach);
#pragma unroll
    for (int k = 0; k < kMaskWords; ++k) {
        if (k * 64 >= n_obb) break;
        // past the last OBB: its record again, masked off
        const int o = min(k * 64 + lane_id(), n_obb - 1);
        float lx, ly, lz;
        to_box(s_obb[STRIDE * o], s_obb[STRIDE * o + 1], s_obb[STRIDE * o + 2], cx, cy, cz, lx, ly, lz);
        w[k] = __ballot(k * 64 + lane_id() < n_obb && !(box_key(lx, ly, lz, s_obb[STRIDE * o + 3]) >= thr));
    }
}

// Smallest box key over the candidate OBBs of `mk` at world point p, and its
// OBB (LDS record index; -1 when there is none). Ties keep the lowest index.
// A (sphere, OBB) pair the scene's ACM masks out is skipped
// (collision/scene_collision.cuh:140-167: sphere_obb_clearance by sphere index).
__device__ __forceinline__ void obb_argmin(const float4* __restrict__ s_obb, const ObbMask& mk, float px, float py,
                                           float pz, const uint8_t* __restrict__ acm_row, float& best, int& arg) {
    best = FLT_MAX;
    arg = -1;
#pragma unroll
    for (int k = 0; k < kMaskWords; ++k) {
        unsigned long long bits = mk.w[k];
        while (bits) {
            const int o = k * 64 + (__ffsll(bits) - 1);
            bits &= bits - 1ull;
            if (acm_row && acm_row[__float_as_int(s_obb[4 * o + 3].w)] == 0) continue;
            float lx, ly, lz;
            to_box(s_obb[4 * o], s_obb[4 * o + 1], s_obb[4 * o + 2], px, py, pz, lx, ly, lz);
            const float key = box_key(lx, ly, lz, s_obb[4 * o + 3]);
            if (key < best) { best = key; arg = o; }
        }
    }
}

// Hinge terms of one sphere at world position p given its OBB argmin (best
// key; has_arg: there is one; rec(r0, r1, r2, r3) fetches the argmin OBB's
// record, called only for the gradient of an active hinge): the summed hinge
// (OBB + ESDF) and its point gradient d hinge / d p in g*.
template <bool GRAD, bool ONE, class Rec>
__device__ __forceinline__ float sphere_hinge_at(const CostArgs& a, const EsdfLayer& layer, bool has_arg, const Rec& rec, float best, float px,
                                                 float py, float pz, float r, int sph_id, bool use_obb, bool use_esdf,
                                                 float& gx, float& gy, float& gz) {
    const float m = a.P.world_margin;
    float world = 0.0f;
    gx = gy = gz = 0.0f;
    if (use_obb) {
        const float clr = has_arg ? key_to_sdf(best) - r : 1000.0f;
        const float hh = m - clr;
        if (hh > 0.0f) {
            world += hh;
            if (GRAD) {
                float dx, dy, dz;
                float4 r0, r1, r2, r3;
                rec(r0, r1, r2, r3);
                box_sdf_grad(r0, r1, r2, r3, px, py, pz, dx, dy, dz);
                gx -= dx; gy -= dy; gz -= dz;
            }
        }
    }
    if (use_esdf) {
        float dx, dy, dz;
        if (ONE) {
            EsdfTap t;
            t.load(layer, px, py, pz, true);
            const float c = t.value(r), hh = m - c;
            if (hh > 0.0f) world += hh;
            if (GRAD && hh > 0.0f && c < 1000.0f) {   // 1000: not from the grid, no gradient
                t.grad(layer, dx, dy, dz);
                gx += dx; gy += dy; gz += dz;
            }
        } else {
            const float c = esdf_clearance(a.S, px, py, pz, r, sph_id, GRAD, dx, dy, dz);
            const float hh = m - c;
            if (hh > 0.0f) {
                world += hh;
                if (GRAD) { gx += dx; gy += dy; gz += dz; }
            }
        }
    }
    return world;
}

// Sum over the G lanes of a state group (G a power of two <= 64; the
// groups are aligned, so xor offsets below G stay inside the group).
__device__ __forceinline__ float group_sum(float v, int G) {
    for (int o = 1; o < G; o <<= 1) v += __shfl_xor(v, o);
    return v;
}

// Spheres of a lane that k_state_cost takes through the boxes together.
constexpr int kSphRun = 4;

// Cost and adjoint, G lanes per state, joint by joint.
__global__ __launch_bounds__(64, 4) void k_cost_grad(CostArgs a) {
    extern __shared__ float4 s_lds[];
    float4* s_obb = s_lds;
    float* s_q = reinterpret_cast<float*>(s_lds + 4 * a.C.obb_cap);
    const DRobot& R = a.R;
    const int lane = lane_id();
    const int G = a.group;                    // lanes per state
    const int sub = lane & (G - 1);
    const int slot = lane / G;                // state slot of this lane group
    const int J = R.n_joints, D = R.n_dof;
    // Adjoint records: per state slot and joint, the joint origin o,
    // axis z, and the force f / moment tau (about o) of its own spheres'
    // hinge gradients; then d cost / d q per dof.
    int* s_end = reinterpret_cast<int*>(s_q + D * kWave);
    const int rs = rec_stride(J), ds = dq_stride(D);
    float* rec = s_q + (D + 2) * kWave + slot * rs;
    float* dqs = s_q + (D + 2) * kWave + (kWave / G) * rs + slot * ds;
    const bool use_obb = a.P.use_obb != 0;
    const bool use_esdf = a.P.use_esdf != 0 && a.S.n_voxel_layers > 0;
    const float wt = a.P.weight;
    int cur_prob = -1, n_obb = 0;
    int4 ch;
    ChunkCursor cur = chunk_cursor();
    const long n_states = state_count(a.X);
    const int n_chunks = chunk_count(a.C, n_states);
    while (next_chunk(a.C, n_states, n_chunks, cur, ch)) {
        if (ch.x != cur_prob) {
            int o0, o1;
            problem_obbs(a.C, a.S, ch.x, o0, o1);
            __syncthreads();
            n_obb = uniform(stage_obbs(a.S, o0, o1, s_obb, a.C.obb_cap));
            cur_prob = ch.x;
        }
        const long g = (long)ch.y + slot;
        const bool active = g < ch.z;
        stage_unit_ends(a.X, ch.w, s_end);
        __syncthreads();
        StateRef ref = load_state(a.X, D, g, active, s_q, ch.w, s_end, ch.x);
        __syncthreads();
        // Self term from the self pass: hinge and its two point gradients.
        float self_h = 0.0f, snx = 0.0f, sny = 0.0f, snz = 0.0f;
        int si = -1, sj = -1;
        if (a.self_in && active) {
            const float* so = a.self_in + 8 * (size_t)ref.gs;
            self_h = fmaxf(a.P.self_margin - so[0], 0.0f);
            if (self_h > 0.0f) { si = __float_as_int(so[1]); sj = __float_as_int(so[2]); snx = so[3]; sny = so[4]; snz = so[5]; }
        }
        float world = 0.0f;
        Slots sl;
        for (int jj = 0; jj < J; ++jj) {
            float T[12];
            int4 meta;
            fk_joint(R, jj, s_q + lane, sl, T, meta);
            float fx = 0.0f, fy = 0.0f, fz = 0.0f, tx = 0.0f, ty = 0.0f, tz = 0.0f;
            const bool any = uload<int>(R.sph_off, jj + 1) > uload<int>(R.sph_off, jj);
            const int c1 = any ? uload<int>(R.clu_off, jj + 1) : 0;
            // one candidate mask per sphere cluster of the joint
            for (int c = any ? uload<int>(R.clu_off, jj) : 0; c < c1; ++c) {
                ObbMask mk{};
                if (use_obb) near_obbs<4>(s_obb, n_obb, T, uload4(R.clu_enc, c), a.P.world_margin, active, mk.w);
                const int b1 = uload<int>(R.clu_beg, c + 1);
                for (int s = uload<int>(R.clu_beg, c) + sub; s < b1; s += G) {
                    const float4 sp = R.sph[s];
                    float px, py, pz;
                    aff_point(T, sp.x, sp.y, sp.z, px, py, pz);
                    float best = FLT_MAX;
                    int arg = -1;
                    const uint8_t* acm_row =
                        a.S.sphere_obb_acm ? a.S.sphere_obb_acm + (size_t)R.sph_id[s] * a.S.n_obbs : nullptr;
                    if (use_obb) obb_argmin(s_obb, mk, px, py, pz, acm_row, best, arg);
                    float gx, gy, gz;
                    auto rec = [&](float4& r0, float4& r1, float4& r2, float4& r3) {
                        r0 = s_obb[4 * arg]; r1 = s_obb[4 * arg + 1]; r2 = s_obb[4 * arg + 2]; r3 = s_obb[4 * arg + 3];
                    };
                    const float hs = sphere_hinge_at<true, false>(a, EsdfLayer(), arg >= 0, rec, best, px, py, pz, sp.w, R.sph_id[s],
                                                           use_obb, use_esdf, gx, gy, gz);
                    world += hs;
                    if (si >= 0) {
                        const int id = R.sph_id[s];
                        if (id == si) { gx -= snx; gy -= sny; gz -= snz; }
                        if (id == sj) { gx += snx; gy += sny; gz += snz; }
                    }
                    // wrench about the joint origin: f += g, tau += (p - o) x g
                    const float rx = px - T[3], ry = py - T[7], rz = pz - T[11];
                    fx += gx; fy += gy; fz += gz;
                    tx = fmaf(ry, gz, fmaf(-rz, gy, tx));
                    ty = fmaf(rz, gx, fmaf(-rx, gz, ty));
                    tz = fmaf(rx, gy, fmaf(-ry, gx, tz));
                }
            }
            const bool nz = fx != 0.0f || fy != 0.0f || fz != 0.0f || tx != 0.0f || ty != 0.0f || tz != 0.0f;
            if (G > 1 && wave_any(nz)) {
                fx = group_sum(fx, G); fy = group_sum(fy, G); fz = group_sum(fz, G);
                tx = group_sum(tx, G); ty = group_sum(ty, G); tz = group_sum(tz, G);
            }
            if (sub == 0) {
                const int type = meta.x;
                const int ax = type >= kXRot ? type - kXRot : (type >= 0 ? type : 0);
                float* r = rec + 12 * jj;
                r[0] = T[3]; r[1] = T[7]; r[2] = T[11];
                r[3] = T[ax]; r[4] = T[4 + ax]; r[5] = T[8 + ax];
                r[6] = fx; r[7] = fy; r[8] = fz;
                r[9] = tx; r[10] = ty; r[11] = tz;
            }
        }
        if (sub == 0 && active) {
            // Reverse DFS sweep: every joint's subtree wrench is complete once
            // its descendants (higher DFS positions) have been folded in.
            for (int d = 0; d < D; ++d) dqs[d] = 0.0f;
            for (int jj = J - 1; jj >= 1; --jj) {
                const float* r = rec + 12 * jj;
                const float ox = r[0], oy = r[1], oz = r[2];
                const float fx = r[6], fy = r[7], fz = r[8];
                const float tx = r[9], ty = r[10], tz = r[11];
                const int4 meta = R.jmeta[jj];
                if (meta.y >= 0 && meta.x >= 0) {
                    const float dq = meta.x >= kXRot ? fmaf(r[3], tx, fmaf(r[4], ty, r[5] * tz))
                                                     : fmaf(r[3], fx, fmaf(r[4], fy, r[5] * fz));
                    dqs[meta.y] += dq;
                }
                float* q = rec + 12 * R.parent[jj];
                const float lx = ox - q[0], ly = oy - q[1], lz = oz - q[2];
                q[6] += fx; q[7] += fy; q[8] += fz;
                q[9] += tx + (ly * fz - lz * fy);
                q[10] += ty + (lz * fx - lx * fz);
                q[11] += tz + (lx * fy - ly * fx);
            }
            bool endpoint = false;
            size_t base = (size_t)ref.gs * D, stride = 1;
            if (a.X.source == kSrcTraj) {
                endpoint = (ref.k == 0 || ref.k == ref.n - 1);
                base = (size_t)a.X.traj_off[ref.unit] * D + ref.k;
                stride = ref.n;
            }
            for (int d = 0; d < D; ++d) a.grad_out[base + (size_t)d * stride] = endpoint ? 0.0f : wt * dqs[d];
        }
        world = group_sum(world, G);
        if (active && sub == 0 && a.cost_out) a.cost_out[ref.gs] = wt * (world + self_h);
        __syncthreads();   // records and q of this chunk are dead before the next load_state
    }
}

// The cost alone: as above, but a cluster's spheres meet a candidate box
// together, up to four of a lane at a time, so a record is read once for all of
// them and their tests do not wait for one another; the bound on the cluster is
// taken around the mean of the wave's centres. A cluster that no box comes near
// adds nothing and is left; so is the exact distance of a sphere that no lane
// has within the hinge band. Bound by VALU issue (16,000 instructions a wave of
// 64 states), at 64 % of it; a wave takes long enough that the last ones of a
// launch show. 325,152 Fetch rollout states, 30 to 80 boxes a problem: 396 us
// -> 210 with one kernel for cost and adjoint before, box by box for each
// sphere; 239 around the first lane's centre; runs of 4, 3 and 2 spheres 211,
// 213 and 220; at the waves that the chip holds at once 268.
template <bool ESDF, bool LINE>
__global__ __launch_bounds__(64, 4) void k_state_cost(CostArgs a) {
    extern __shared__ float4 s_lds[];
    float4* s_obb = s_lds;
    float* s_q = reinterpret_cast<float*>(s_lds + kObbRec * a.C.obb_cap);
    const DRobot& R = a.R;
    const int lane = lane_id();
    const int G = a.group, sub = lane & (G - 1), slot = lane / G;
    const int lg = __ffs(G) - 1;
    const int J = R.n_joints, D = R.n_dof;
    int* s_end = reinterpret_cast<int*>(s_q + D * kWave);
    const bool use_obb = a.P.use_obb != 0;
    const bool use_esdf = ESDF && a.P.use_esdf != 0;
    const float wt = a.P.weight, m = a.P.world_margin;
    const bool quiet = m <= 1000.0f;   // no box near (clearance 1000): no hinge
    const uint8_t* acm = a.S.sphere_obb_acm;
    int cur_prob = -1, n_obb = 0;
    int4 ch;
    ChunkCursor cur = chunk_cursor();
    const long n_states = state_count(a.X);
    const int n_chunks = chunk_count(a.C, n_states);
    while (next_chunk(a.C, n_states, n_chunks, cur, ch)) {
        if (ch.x != cur_prob) {
            int o0, o1;
            problem_obbs(a.C, a.S, ch.x, o0, o1);
            __syncthreads();
            n_obb = uniform(stage_obbs<kObbRec>(a.S, o0, o1, s_obb, a.C.obb_cap));
            cur_prob = ch.x;
        }
        const long g = (long)ch.y + slot;
        const bool active = g < ch.z;
        stage_unit_ends(a.X, ch.w, s_end);
        __syncthreads();
        StateRef ref = load_state(a.X, D, g, active, s_q, ch.w, s_end, ch.x);
        __syncthreads();
        const float self_h =
            a.self_in && active ? fmaxf(a.P.self_margin - a.self_in[8 * (size_t)ref.gs], 0.0f) : 0.0f;
        float world = 0.0f;
        FkWalk<LINE> fk;
        float T[12];
        for (int jj = 0; jj < J; ++jj) {
            int4 meta;
            fk.step(R, jj, s_q + lane, T, meta);
            if (uload<int>(R.sph_off, jj) == uload<int>(R.sph_off, jj + 1)) continue;
            const int c1 = uload<int>(R.clu_off, jj + 1);
            for (int c = uload<int>(R.clu_off, jj); c < c1; ++c) {
                unsigned long long w[kMaskWords] = {};
                if (use_obb) near_obbs<kObbRec>(s_obb, n_obb, T, uload4(R.clu_enc, c), m, active, w);
                if (!use_esdf && quiet && (w[0] | w[1] | w[2] | w[3]) == 0ull) continue;
                const int b1 = uload<int>(R.clu_beg, c + 1);
                for (int b = uload<int>(R.clu_beg, c); b < b1; b += kSphRun * G) {
                    const int n = min(kSphRun, (b1 - b + G - 1) >> lg);   // rounds of this run
                    float4 p[kSphRun];
                    float best[kSphRun];
                    int id[kSphRun];   // for the ACM
#pragma unroll
                    for (int k = 0; k < kSphRun; ++k) {
                        // past the cluster's end: its last sphere again
                        const int s = min(b + k * G + sub, b1 - 1);
                        const float4 sp = G == 1 ? uload4(R.sph, min(b + k, b1 - 1)) : R.sph[s];
                        aff_point(T, sp.x, sp.y, sp.z, p[k].x, p[k].y, p[k].z);
                        p[k].w = sp.w;
                        best[k] = FLT_MAX;
                        id[k] = acm ? R.sph_id[s] : 0;
                    }
                    unsigned long long v[kMaskWords];
#pragma unroll
                    for (int k = 0; k < kMaskWords; ++k) v[k] = w[k];
                    for (int o0 = 0; o0 < n_obb; o0 += 64) {
                        while (v[0]) {
                            const int o = o0 + __ffsll(v[0]) - 1;
                            v[0] &= v[0] - 1ull;
                            const float4 r0 = s_obb[kObbRec * o], r1 = s_obb[kObbRec * o + 1],
                                         r2 = s_obb[kObbRec * o + 2], h = s_obb[kObbRec * o + 3];
#pragma unroll
                            for (int k = 0; k < kSphRun; ++k) {
                                if (k >= n) break;
                                float lx, ly, lz;
                                to_box(r0, r1, r2, p[k].x, p[k].y, p[k].z, lx, ly, lz);
                                float key = box_key(lx, ly, lz, h);
                                if (acm && acm[(size_t)id[k] * a.S.n_obbs + __float_as_int(h.w)] == 0) key = FLT_MAX;
                                best[k] = fminf(best[k], key);
                            }
                        }
#pragma unroll
                        for (int k = 0; k + 1 < kMaskWords; ++k) v[k] = v[k + 1];
                    }
#pragma unroll
                    for (int k = 0; k < kSphRun; ++k) {
                        if (k >= n) break;
                        const int s = b + k * G + sub;
                        const float r = p[k].w;
                        float hs = 0.0f;
                        if (use_obb) {
                            // sdf < m + r <=> key < (m + r) |m + r|; slack covers rounding
                            const float reach = fmaf(fabsf(m) + fabsf(r), 1e-5f, m + r) + 1e-6f;
                            if (!quiet || wave_any(best[k] < reach * fabsf(reach))) {
                                const float clr = best[k] < FLT_MAX ? key_to_sdf(best[k]) - r : 1000.0f;
                                const float hh = m - clr;
                                if (hh > 0.0f) hs += hh;
                            }
                        }
                        if (ESDF && use_esdf) {
                            float gx, gy, gz;
                            const float hh = m - esdf_clearance(a.S, p[k].x, p[k].y, p[k].z, r,
                                                                R.sph_id[min(s, b1 - 1)], false, gx, gy, gz);
                            if (hh > 0.0f) hs += hh;
                        }
                        if (s < b1) world += hs;
                    }
                }
            }
        }
        world = group_sum(world, G);
        if (active && sub == 0 && a.cost_out) a.cost_out[ref.gs] = wt * (world + self_h);
        __syncthreads();   // the states of this chunk are read
    }
}

// ===========================================================================
// Grouped summed-hinge cost (+ adjoint): one state per aligned group of
// kGrp = 16 lanes, four states per wave, with the state's spheres spread over
// the group's lanes across joints instead of joint by joint.
//  1. Forward kinematics in parallel: lane jj of the group computes joint
//     jj's step (one sin/cos per lane) and the frames are composed by
//     pointer jumping over the DFS tree in ceil(log2(depth)) rounds through
//     LDS. Then every sphere cluster's enclosing sphere is placed at once
//     and one wave pass per cluster over the OBBs gives its candidate mask
//     (the broad phase of near_obbs over the wave's four states).
//  2. Sphere pass: emission slot k (spheres are emitted joint by joint,
//     cluster by cluster) goes to lane k mod 16, which reads its joint's
//     frame and its cluster's mask from LDS,
//     finds the argmin OBB and the hinge terms. Panda's 59 spheres take four
//     rounds instead of one round per joint with most lanes idle.
//  3. Adjoint: every sphere's point gradient g gives a force g and a moment
//     (p - o_j) x g about its joint's origin o_j. Each round's 16 of them pass
//     through LDS to the joints' lanes, which add up their own spheres' in
//     emission order. A prefix scan over the group's lanes (one joint per lane)
//     sums each joint's DFS subtree -- a contiguous run of positions -- into a
//     total wrench about o_jj, and lane jj reads d cost / d q = z . tau
//     (revolute) or z . f (prismatic).
// Results equal k_cost_grad's up to FP32 summation order.
// Bound by latency: 16,384 Panda states are 4,096 waves, one round of the chip,
// each a chain of loads, frames, masks and four sphere rounds, with VALU issue
// at 0.45. 256 trajectories of 64 waypoints among 40 boxes: 45.5 us -> 31.7, of
// which 6 by the masks' reach about the states' mean instead of the first
// state's place (fewer candidates) with the reaches computed a lane each, and by
// loads that start together, and 8 by the wrenches: six LDS atomics a sphere, up
// to sixteen to one address, kept the CU's LDS unit busy. The same in CHOMP's
// iterations 60 -> 48, and over an ESDF (71,000 Baxter states) 82 -> 78; there
// VALU issue is at 0.62.
// ===========================================================================
// Joint frames of the state of a 16-lane group (one state per group, a
// 1-wave workgroup), DFS positions 0..J-1, into F (12 floats each, row-major
// 3x4), by pointer jumping over the DFS tree: lane jj of the group starts
// from its joint step A = S_jj (the root's is the identity) and its parent
// link P; each round composes the frame of link P onto A and jumps P to P's
// link, until P is the root. Then A is the product of the steps from the root
// down to jj: the frame. ceil(log2(depth)) rounds through LDS. qs: the
// state's q (q_d = qs[d * qstride]); par: J ints of LDS for the links.
// Contains block barriers: every lane of the workgroup must call it.
// jt: the lane's joint (DFS position `sub`), in registers, so that a caller with
// several rounds loads it once.
struct JointRegs {
    float ft[12];
    int type, dof, parent;
    template <bool APPROX = false>
    __device__ __forceinline__ void load(const DRobot& R, int sub) {
        type = dof = -1;
        parent = 0;
#pragma unroll
        for (int k = 0; k < 12; ++k) ft[k] = 0.0f;
        if (sub == 0) {
            ft[0] = ft[5] = ft[10] = 1.0f;
        } else if (sub < R.n_joints) {
            const int4 meta = R.jmeta[sub];
            const float4* f = reinterpret_cast<const float4*>((APPROX ? R.aft : R.ft) + 12 * sub);
            const float4 f0 = f[0], f1 = f[1], f2 = f[2];
            ft[0] = f0.x; ft[1] = f0.y; ft[2] = f0.z; ft[3] = f0.w;
            ft[4] = f1.x; ft[5] = f1.y; ft[6] = f1.z; ft[7] = f1.w;
            ft[8] = f2.x; ft[9] = f2.y; ft[10] = f2.z; ft[11] = f2.w;
            type = APPROX ? R.atype[sub] : meta.x;
            dof = meta.y;
            parent = R.parent[sub];
        }
    }
    // joint_step_u of the lane's joint, its columns picked by selects
    __device__ __forceinline__ void step(float q, float* S) const {
#pragma unroll
        for (int k = 0; k < 12; ++k) S[k] = ft[k];
        if (type >= kXRot) {
            float s, c;
            sincosf(q, &s, &c);
            const bool x = type == kXRot, y = type == kYRot;
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const float f0 = ft[r * 4], f1 = ft[r * 4 + 1], f2 = ft[r * 4 + 2];
                const float fa = x ? f1 : y ? f2 : f0, fb = x ? f2 : y ? f0 : f1;
                const float na = fmaf(fa, c, fb * s), nb = fmaf(fb, c, -fa * s);
                S[r * 4] = x ? f0 : y ? nb : na;
                S[r * 4 + 1] = x ? na : y ? f1 : nb;
                S[r * 4 + 2] = x ? nb : y ? na : f2;
            }
        } else if (type >= kXPrism) {
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const float f = type == kXPrism ? ft[r * 4] : type == kYPrism ? ft[r * 4 + 1] : ft[r * 4 + 2];
                S[r * 4 + 3] = fmaf(f, q, ft[r * 4 + 3]);
            }
        }
    }
};

__device__ __forceinline__ void group_frames(const JointRegs& jt, int J, const float* qs, int qstride, float* F,
                                             int* par, int sub) {
    const bool own = sub < J;
    int P = 0;
    if (own) {
        float A[12];
        jt.step(jt.dof >= 0 ? qs[jt.dof * qstride] : 0.0f, A);
        P = jt.parent;
        float4* d = reinterpret_cast<float4*>(F + 12 * sub);
        d[0] = make_float4(A[0], A[1], A[2], A[3]);
        d[1] = make_float4(A[4], A[5], A[6], A[7]);
        d[2] = make_float4(A[8], A[9], A[10], A[11]);
        par[sub] = P;
    }
    __syncthreads();
    while (wave_any(own && P != 0)) {
        const bool jump = own && P != 0;
        float4 c0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), c1 = c0, c2 = c0;
        int PP = 0;
        if (jump) {
            const float4* b = reinterpret_cast<const float4*>(F + 12 * P);
            const float4* m = reinterpret_cast<const float4*>(F + 12 * sub);
            const float4 m0 = m[0], m1 = m[1], m2 = m[2];
            auto row = [&](const float4 br) {
                return make_float4(fmaf(br.z, m2.x, fmaf(br.y, m1.x, br.x * m0.x)),
                                   fmaf(br.z, m2.y, fmaf(br.y, m1.y, br.x * m0.y)),
                                   fmaf(br.z, m2.z, fmaf(br.y, m1.z, br.x * m0.z)),
                                   fmaf(br.z, m2.w, fmaf(br.y, m1.w, br.x * m0.w)) + br.w);
            };
            c0 = row(b[0]);
            c1 = row(b[1]);
            c2 = row(b[2]);
            PP = par[P];
        }
        __syncthreads();
        if (jump) {
            float4* d = reinterpret_cast<float4*>(F + 12 * sub);
            d[0] = c0;
            d[1] = c1;
            d[2] = c2;
            P = PP;
            par[sub] = P;
        }
        __syncthreads();
    }
}

static_assert(kGrp >= kMaxJoints, "the grouped kernel gives every joint its own lane of the group");

// Floats of a state's 16 sphere wrenches of one round (6 each; the four states'
// start in different LDS banks).
constexpr int kGrpWrench = kGrp * 6 + 4;

size_t lds_floats_grp(int obb_cap, int n_dof, int n_joints, int n_sph, int n_clu, bool grad, bool tiled) {
    size_t f = (size_t)obb_cap * 16 + (size_t)n_clu * kMaskWords * 2 +
               (((size_t)n_dof * kGrpStates + 3) & ~(size_t)3) + 2 * kWave + (size_t)kGrpStates * (n_joints * 13 + 4);
    if (grad) f += (size_t)kGrpStates * (kGrpWrench + kMaxDof + 1);
    if (tiled) f += (size_t)kGrpStates * n_sph * 2;
    return f;
}

// Candidate masks of every sphere cluster of the wave's four states over the
// staged OBBs (the broad phase of near_obbs, all clusters' enclosing spheres
// placed at once, 16 clusters per pass): lane k of each group places cluster
// c0 + k's enclosing sphere; the four states' spread about their mean sets the
// cluster's reach; one pass of 64 lanes over the OBBs per cluster gives its
// mask (words past the staged OBBs are neither written nor read).
__device__ __forceinline__ void grp_masks(const DRobot& R, const float4* __restrict__ s_obb, int n_obb, const float* Ts,
                                          float band, bool active, int sub, unsigned long long* s_mask) {
    const int C = R.n_clu, lane = lane_id();
    auto slots = [](float v) {   // sum over the four states
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    for (int c0 = 0; c0 < C; c0 += kGrp) {
        const int cl = c0 + sub;
        float4 ce = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        if (cl < C && active) {
            ce = R.clu_enc[cl];
            const float4* t = reinterpret_cast<const float4*>(Ts + 12 * R.clu_jnt[cl]);
            const float4 t0 = t[0], t1 = t[1], t2 = t[2];
            ax = fmaf(t0.x, ce.x, fmaf(t0.y, ce.y, fmaf(t0.z, ce.z, t0.w)));
            ay = fmaf(t1.x, ce.x, fmaf(t1.y, ce.y, fmaf(t1.z, ce.z, t1.w)));
            az = fmaf(t2.x, ce.x, fmaf(t2.y, ce.y, fmaf(t2.z, ce.z, t2.w)));
        }
        const bool in = cl < C && active && usable(ax, ay, az);
        const float inv_n = __builtin_amdgcn_rcpf(slots(in ? 1.0f : 0.0f));
        const float cx = slots(in ? ax : 0.0f) * inv_n, cy = slots(in ? ay : 0.0f) * inv_n,
                    cz = slots(in ? az : 0.0f) * inv_n;
        const float dx = ax - cx, dy = ay - cy, dz = az - cz;
        float d2 = (cl < C && active) ? fmaf(dz, dz, fmaf(dy, dy, dx * dx)) : 0.0f;
        d2 = max_nan(d2, __shfl_xor(d2, 16));
        d2 = max_nan(d2, __shfl_xor(d2, 32));
        const float reach = band + ce.w + __builtin_amdgcn_sqrtf(d2) * 1.0001f + 1e-5f;
        const float thr = reach * fabsf(reach);
        const int nk = min(kGrp, C - c0);
        if (n_obb <= 64) {
            // each lane reads its box's record once for every cluster of the pass
            float4 q0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), q1 = q0, q2 = q0, qh = q0;
            if (lane < n_obb) {
                q0 = s_obb[4 * lane]; q1 = s_obb[4 * lane + 1]; q2 = s_obb[4 * lane + 2]; qh = s_obb[4 * lane + 3];
            }
            unsigned long long mine = 0ull;   // cluster c0 + lane's
            for (int k = 0; k < nk; ++k) {
                float lx, ly, lz;
                to_box(q0, q1, q2, read_lane(cx, k), read_lane(cy, k), read_lane(cz, k), lx, ly, lz);
                const unsigned long long m = __ballot(lane < n_obb && !(box_key(lx, ly, lz, qh) >= read_lane(thr, k)));
                if (lane == k) mine = m;
            }
            if (lane < nk) s_mask[(c0 + lane) * kMaskWords] = mine;
        } else {
            for (int k = 0; k < nk; ++k) {
                const float c0x = read_lane(cx, k), c0y = read_lane(cy, k), c0z = read_lane(cz, k), t = read_lane(thr, k);
                for (int w = 0; w * 64 < n_obb; ++w) {
                    const int o = w * 64 + lane;
                    bool c = false;
                    if (o < n_obb) {
                        float lx, ly, lz;
                        to_box(s_obb[4 * o], s_obb[4 * o + 1], s_obb[4 * o + 2], c0x, c0y, c0z, lx, ly, lz);
                        c = !(box_key(lx, ly, lz, s_obb[4 * o + 3]) >= t);
                    }
                    const unsigned long long m = __ballot(c);
                    if (lane == 0) s_mask[(c0 + k) * kMaskWords + w] = m;
                }
            }
        }
    }
}

// Smallest box key at p over the candidate OBBs of `own` (a joint's mask in
// LDS) and its LDS record index (-1: none). Two candidates per step: both
// records are read before either test, so the LDS latency of one hides the
// other's. Ties keep the lower index.
__device__ __forceinline__ void grp_argmin(const float4* __restrict__ s_obb, int n_obb, const unsigned long long* own, bool valid,
                                           float px, float py, float pz, const uint8_t* __restrict__ acm_row,
                                           float& best, int& arg) {
    best = FLT_MAX;
    arg = -1;
    for (int k = 0; k * 64 < n_obb; ++k) {
        unsigned long long bits = valid ? own[k] : 0ull;
        while (bits) {
            const int oa = k * 64 + (__ffsll(bits) - 1);
            bits &= bits - 1ull;
            const bool two = bits != 0ull;
            const int ob = two ? k * 64 + (__ffsll(bits) - 1) : oa;
            if (two) bits &= bits - 1ull;
            const float4 a0 = s_obb[4 * oa], a1 = s_obb[4 * oa + 1], a2 = s_obb[4 * oa + 2], ah = s_obb[4 * oa + 3];
            const float4 b0 = s_obb[4 * ob], b1 = s_obb[4 * ob + 1], b2 = s_obb[4 * ob + 2], bh = s_obb[4 * ob + 3];
            float lx, ly, lz;
            to_box(a0, a1, a2, px, py, pz, lx, ly, lz);
            float ka = box_key(lx, ly, lz, ah);
            to_box(b0, b1, b2, px, py, pz, lx, ly, lz);
            float kb = box_key(lx, ly, lz, bh);
            if (acm_row) {
                if (acm_row[__float_as_int(ah.w)] == 0) ka = FLT_MAX;
                if (acm_row[__float_as_int(bh.w)] == 0) kb = FLT_MAX;
            }
            if (ka < best) { best = ka; arg = oa; }        // oa < ob: ties keep the lower index
            if (two && kb < best) { best = kb; arg = ob; }
        }
    }
}

// WORLD: bit 0 the scene's boxes may enter (OBB hinge / argmin), bit 1 its
// ESDF layers may; the launch picks the smallest variant the call needs, which
// keeps the other path's registers out of the sphere pass. TILED: some
// problem's OBBs pass through LDS in tiles (a variant of its own, so the
// folding across tiles costs the one-staging kernels no registers).
// ONE: the scene is a single trilinear ESDF layer without masks (esdf_single).
template <bool GRAD, int WORLD, bool TILED, bool ONE = false>
__device__ __forceinline__ void cost_grp(const CostArgs& a) {
    extern __shared__ float4 s_lds[];
    const DRobot& R = a.R;
    const int J = R.n_joints, D = R.n_dof, S = R.n_sph;
    float4* s_obb = s_lds;
    unsigned long long* s_mask = reinterpret_cast<unsigned long long*>(s_lds + 4 * a.C.obb_cap);
    float* s_q = reinterpret_cast<float*>(s_mask + (size_t)R.n_clu * kMaskWords);
    int* s_end = reinterpret_cast<int*>(s_q + D * kGrpStates);   // s_q: [D][slot]
    // frames [slot][J][12], slot stride padded by 4 floats so the four
    // slots' frames of one joint start in different LDS banks
    const int fstride = J * 12 + 4;
    float* s_T = reinterpret_cast<float*>(s_end + 2 * kWave);
    int* s_par = reinterpret_cast<int*>(s_T + kGrpStates * fstride);   // [slot][J] pointer-jumping links
    float* s_w = reinterpret_cast<float*>(s_par + kGrpStates * J);    // GRAD: [slot][kGrpWrench]
    float* s_dq = s_w + kGrpStates * kGrpWrench;                  // GRAD: [slot][kMaxDof + 1]
    // tiled problems: per state slot and emission slot, the smallest box key
    // over the tiles so far and its OBB (original index, -1: none)
    float* s_best = GRAD ? s_dq + kGrpStates * (kMaxDof + 1) : s_w;
    int* s_barg = reinterpret_cast<int*>(s_best + kGrpStates * S);
    const int lane = lane_id();
    const int sub = lane & (kGrp - 1);
    const int slot = lane / kGrp;
    float* Ts = s_T + slot * fstride;
    const bool use_obb = (WORLD & 1) && a.P.use_obb != 0;
    const bool use_esdf = (WORLD & 2) && a.P.use_esdf != 0 && a.S.n_voxel_layers > 0;
    const float wt = a.P.weight;
    const int cap = a.C.obb_cap;
    const EsdfLayer layer = ONE ? EsdfLayer(a.S) : EsdfLayer();
    int cur_prob = -1, n_obb = 0, o0 = 0, o1 = 0, n_tiles = 1;
    int4 ch;
    ChunkCursor cur = chunk_cursor();
    const long n_states = state_count(a.X);
    const int n_chunks = chunk_count(a.C, n_states);
    while (next_chunk(a.C, n_states, n_chunks, cur, ch)) {
        // loads that wait for nothing else, in flight together
        int u_end = 0, u_beg = 0;
        prefetch_unit_ends(a.X, ch.w, u_end, u_beg);
        JointRegs jt;
        if (WORLD & 1) jt.load(R, sub);
        if ((WORLD & 1) && ch.x != cur_prob) {
            problem_obbs(a.C, a.S, ch.x, o0, o1);
            n_tiles = TILED ? uniform(obb_tiles(o0, o1, cap)) : 1;
            if (n_tiles == 1) {
                __syncthreads();
                n_obb = uniform(stage_obbs(a.S, o0, o1, s_obb, cap));
            }
            cur_prob = ch.x;
        }
        const bool tiled = TILED && use_obb && n_tiles > 1;
        const long g = (long)ch.y + slot;
        const bool active = g < ch.z;
        s_end[lane] = u_end;
        s_end[kWave + lane] = u_beg;
        if (GRAD)
            for (int i = lane; i < kGrpStates * (kMaxDof + 1); i += kWave) s_dq[i] = 0.0f;
        __syncthreads();
        StateRef ref = load_state(a.X, D, g, active, s_q, ch.w, s_end, ch.x, slot, kGrpStates, sub == 0);
        __syncthreads();
        // 1a. joint frames (pointer jumping over the DFS tree)
        if (!(WORLD & 1)) jt.load(R, sub);   // no registers to hold it from the start
        group_frames(jt, J, s_q + slot, kGrpStates, Ts, s_par + slot * J, sub);
        // 1b. candidate masks per sphere cluster; a tiled problem's OBBs pass through
        // LDS tile by tile, each tile's argmins folded into s_best / s_barg
        // (tiles in index order and a strict < keep the lowest index on ties)
        if (use_obb && !tiled) grp_masks(R, s_obb, n_obb, Ts, a.P.world_margin, active, sub, s_mask);
        for (int t = 0; tiled && t < n_tiles; ++t) {
            const int t0 = o0 + t * cap;
            __syncthreads();
            n_obb = uniform(stage_obbs(a.S, t0, min(o1, t0 + cap), s_obb, cap));
            grp_masks(R, s_obb, n_obb, Ts, a.P.world_margin, active, sub, s_mask);
            __syncthreads();
            for (int r0 = 0; r0 < S; r0 += kGrp) {
                const int s = r0 + sub;
                const bool valid = active && s < S;
                const int sc = valid ? s : r0;
                const int jj = R.sph_jnt[sc];
                const float4* Tq = reinterpret_cast<const float4*>(Ts + 12 * jj);
                const float4 t0q = Tq[0], t1q = Tq[1], t2q = Tq[2];
                const float4 sp = R.sph[sc];
                const int sid = R.sph_id[sc];
                const float px = fmaf(t0q.x, sp.x, fmaf(t0q.y, sp.y, fmaf(t0q.z, sp.z, t0q.w)));
                const float py = fmaf(t1q.x, sp.x, fmaf(t1q.y, sp.y, fmaf(t1q.z, sp.z, t1q.w)));
                const float pz = fmaf(t2q.x, sp.x, fmaf(t2q.y, sp.y, fmaf(t2q.z, sp.z, t2q.w)));
                const uint8_t* acm_row = a.S.sphere_obb_acm ? a.S.sphere_obb_acm + (size_t)sid * a.S.n_obbs : nullptr;
                float best;
                int arg;
                grp_argmin(s_obb, n_obb, s_mask + R.sph_clu[sc] * kMaskWords, valid, px, py, pz, acm_row, best, arg);
                if (valid) {
                    float* bk = s_best + slot * S + s;
                    int* ba = s_barg + slot * S + s;
                    if (t == 0 || best < *bk) {
                        *bk = best;
                        *ba = arg >= 0 ? __float_as_int(s_obb[4 * arg + 3].w) : -1;
                    }
                }
            }
        }
        float self_h = 0.0f, snx = 0.0f, sny = 0.0f, snz = 0.0f;
        int si = -1, sj = -1;
        if (a.self_in && active) {
            const float* so = a.self_in + 8 * (size_t)ref.gs;
            self_h = fmaxf(a.P.self_margin - so[0], 0.0f);
            if (self_h > 0.0f) { si = __float_as_int(so[1]); sj = __float_as_int(so[2]); snx = so[3]; sny = so[4]; snz = so[5]; }
        }
        // 2. sphere pass, in rounds of 16 emission slots per state: each lane
        // places its sphere with its joint's frame and walks its cluster's
        // candidate mask for the argmin box (tiled: reads the folded argmin
        // and rebuilds its record from the scene when the gradient needs it).
        float world = 0.0f;
        // In this pass lane = 4 * sphere slot + state: the four states of a
        // sphere walk its cluster's mask together, so each quarter-wave of an
        // LDS record read touches 4 records (broadcast) instead of 16 (bank
        // conflicts). Each state's spheres keep their lanes' relative order,
        // so sums run in the same order as with lane = 16 * state + slot.
        const int rslot = lane & (kGrpStates - 1), rsub = lane >> 2;
        const bool ractive = (long)ch.y + rslot < ch.z;
        const float* Tr = s_T + rslot * fstride;
        const int r_si = __shfl(si, rslot * kGrp), r_sj = __shfl(sj, rslot * kGrp);
        const float r_snx = __shfl(snx, rslot * kGrp), r_sny = __shfl(sny, rslot * kGrp), r_snz = __shfl(snz, rslot * kGrp);
        // Joint `sub` of state `slot`: the force and the moment about its
        // origin of its spheres' point gradients so far (GRAD).
        float f0 = 0.0f, f1 = 0.0f, f2 = 0.0f, m0 = 0.0f, m1 = 0.0f, m2 = 0.0f;
        const int js0 = GRAD && sub < J ? R.sph_off[sub] : 0, js1 = GRAD && sub < J ? R.sph_off[sub + 1] : 0;
        for (int r0 = 0; r0 < S; r0 += kGrp) {
            const int s = r0 + rsub;
            const bool valid = ractive && s < S;
            const int sc = valid ? s : r0;
            const int jj = R.sph_jnt[sc];
            const float4* Tq = reinterpret_cast<const float4*>(Tr + 12 * jj);
            const float4 t0 = Tq[0], t1 = Tq[1], t2 = Tq[2];
            const float4 sp = R.sph[sc];
            const int sid = R.sph_id[sc];
            const float px = fmaf(t0.x, sp.x, fmaf(t0.y, sp.y, fmaf(t0.z, sp.z, t0.w)));
            const float py = fmaf(t1.x, sp.x, fmaf(t1.y, sp.y, fmaf(t1.z, sp.z, t1.w)));
            const float pz = fmaf(t2.x, sp.x, fmaf(t2.y, sp.y, fmaf(t2.z, sp.z, t2.w)));
            float best = FLT_MAX;
            int arg = -1;   // tiled: the argmin's original OBB index; else its LDS record
            if (tiled) {
                if (valid) {
                    best = s_best[rslot * S + s];
                    arg = s_barg[rslot * S + s];
                }
            } else if (use_obb) {
                const uint8_t* acm_row = a.S.sphere_obb_acm ? a.S.sphere_obb_acm + (size_t)sid * a.S.n_obbs : nullptr;
                grp_argmin(s_obb, n_obb, s_mask + R.sph_clu[sc] * kMaskWords, valid, px, py, pz, acm_row, best, arg);
            }
            auto rec = [&](float4& r0, float4& r1, float4& r2, float4& r3) {
                if (tiled) {
                    float4 t[4];
                    obb_record(a.S, arg, t);
                    r0 = t[0]; r1 = t[1]; r2 = t[2]; r3 = t[3];
                } else {
                    r0 = s_obb[4 * arg]; r1 = s_obb[4 * arg + 1]; r2 = s_obb[4 * arg + 2]; r3 = s_obb[4 * arg + 3];
                }
            };
            float gx = 0.0f, gy = 0.0f, gz = 0.0f;
            if (valid)
                world += sphere_hinge_at<GRAD, ONE>(a, layer, arg >= 0, rec, best, px, py, pz, sp.w, sid, use_obb,
                                                    use_esdf, gx, gy, gz);
            if (GRAD) {
                if (valid && r_si >= 0) {
                    if (sid == r_si) { gx -= r_snx; gy -= r_sny; gz -= r_snz; }
                    if (sid == r_sj) { gx += r_snx; gy += r_sny; gz += r_snz; }
                }
                const bool nz = gx != 0.0f || gy != 0.0f || gz != 0.0f;
                if (!wave_any(nz)) continue;
                // The round's wrenches (g and (p - o) x g about the joint's origin
                // o) through LDS to their joints' lanes, added in emission order.
                __syncthreads();
                const float rx = px - t0.w, ry = py - t1.w, rz = pz - t2.w;
                float2* w = reinterpret_cast<float2*>(s_w + rslot * kGrpWrench + rsub * 6);
                w[0] = make_float2(gx, gy);
                w[1] = make_float2(gz, nz ? ry * gz - rz * gy : 0.0f);
                w[2] = nz ? make_float2(rz * gx - rx * gz, rx * gy - ry * gx) : make_float2(0.0f, 0.0f);
                __syncthreads();
                const int k1 = min(js1 - r0, kGrp);
                for (int k = max(js0 - r0, 0); k < k1; k += 2) {
                    const float2* u = reinterpret_cast<const float2*>(s_w + slot * kGrpWrench + k * 6);
                    const bool two = k + 1 < k1;
                    const float2* v = two ? u + 3 : u;
                    const float2 u0 = u[0], u1 = u[1], u2 = u[2], v0 = v[0], v1 = v[1], v2 = v[2];
                    f0 += u0.x; f1 += u0.y; f2 += u1.x; m0 += u1.y; m1 += u2.x; m2 += u2.y;
                    if (two) { f0 += v0.x; f1 += v0.y; f2 += v1.x; m0 += v1.y; m1 += v2.x; m2 += v2.y; }
                }
            }
        }
        // each state's partial sums sit in the lanes with its lane & 3; the
        // pairwise tree matches a 16-lane group sum's
        for (int o = kGrpStates; o < kWave; o <<= 1) world += __shfl_xor(world, o);
        world = __shfl(world, slot);
        // 3. adjoint: subtree wrench of joint `sub` -> d cost / d q
        if (GRAD) {
            __syncthreads();
            float* dq = s_dq + slot * (kMaxDof + 1);
            // Subtree sums by one prefix scan over the group's lanes: lane
            // i holds joint i's force f_i and its moment about the world
            // origin m_i = tau_i + o_i x f_i; DFS subtrees are contiguous, so
            // joint j's subtree force and moment are P(jend[j] - 1) -
            // P(j - 1), and its moment about o_j is M - o_j x F.
            float ox = 0.0f, oy = 0.0f, oz = 0.0f;
            if (sub < J) {
                const float* Tj = Ts + 12 * sub;
                ox = Tj[3]; oy = Tj[7]; oz = Tj[11];
                m0 += oy * f2 - oz * f1;
                m1 += oz * f0 - ox * f2;
                m2 += ox * f1 - oy * f0;
            }
#pragma unroll
            for (int off = 1; off < kGrp; off <<= 1) {
                const float u0 = __shfl_up(f0, off, kGrp), u1 = __shfl_up(f1, off, kGrp), u2 = __shfl_up(f2, off, kGrp);
                const float u3 = __shfl_up(m0, off, kGrp), u4 = __shfl_up(m1, off, kGrp), u5 = __shfl_up(m2, off, kGrp);
                if (sub >= off) { f0 += u0; f1 += u1; f2 += u2; m0 += u3; m1 += u4; m2 += u5; }
            }
            const int gbase = lane - sub;
            const int e = sub < J ? R.jend[sub] : sub + 1;
            const int hi = gbase + e - 1, lo = gbase + (sub > 0 ? sub - 1 : 0);
            float F0 = __shfl(f0, hi), F1 = __shfl(f1, hi), F2 = __shfl(f2, hi);
            float M0 = __shfl(m0, hi), M1 = __shfl(m1, hi), M2 = __shfl(m2, hi);
            const float l0 = __shfl(f0, lo), l1 = __shfl(f1, lo), l2 = __shfl(f2, lo);
            const float l3 = __shfl(m0, lo), l4 = __shfl(m1, lo), l5 = __shfl(m2, lo);
            if (sub > 0) { F0 -= l0; F1 -= l1; F2 -= l2; M0 -= l3; M1 -= l4; M2 -= l5; }
            if (active && sub >= 1 && sub < J) {
                const int4 meta = R.jmeta[sub];
                if (meta.y >= 0 && meta.x >= 0) {
                    const float* Tj = Ts + 12 * sub;
                    const float tx = M0 - (oy * F2 - oz * F1), ty = M1 - (oz * F0 - ox * F2), tz = M2 - (ox * F1 - oy * F0);
                    const int type = meta.x;
                    const int ax = type >= kXRot ? type - kXRot : type;
                    const float zx = Tj[ax], zy = Tj[4 + ax], zz = Tj[8 + ax];
                    const float v = type >= kXRot ? fmaf(zx, tx, fmaf(zy, ty, zz * tz)) : fmaf(zx, F0, fmaf(zy, F1, zz * F2));
                    atomicAdd(dq + meta.y, v);
                }
            }
            __syncthreads();
            if (active && sub < D) {
                bool endpoint = false;
                size_t base = (size_t)ref.gs * D, stride = 1;
                if (a.X.source == kSrcTraj) {
                    endpoint = (ref.k == 0 || ref.k == ref.n - 1);
                    base = (size_t)a.X.traj_off[ref.unit] * D + ref.k;
                    stride = ref.n;
                }
                a.grad_out[base + (size_t)sub * stride] = endpoint ? 0.0f : wt * dq[sub];
            }
        }
        if (active && sub == 0 && a.cost_out) a.cost_out[ref.gs] = wt * (world + self_h);
        __syncthreads();   // frames, masks and wrenches of this chunk are dead before the next one
    }
}

// Four waves per SIMD for the one-staging variants (the adjoint's 128 VGPRs);
// the tiled ones would spill there.
template <bool GRAD, int WORLD, bool TILED>
__global__ __launch_bounds__(64, TILED ? 1 : 4) void k_cost_grp(CostArgs a) {
    cost_grp<GRAD, WORLD, TILED>(a);
}

// ESDF-only launches (no OBB path): five waves per SIMD fit in the register
// budget, which the lookups' memory latency rewards.
template <bool GRAD, bool ONE>
__global__ __launch_bounds__(64, 5) void k_cost_grp_esdf(CostArgs a) {
    cost_grp<GRAD, 2, false, ONE>(a);
}

// ===========================================================================
// Minimum ESDF clearance (radius + margin; 1000 without a layer) of every
// state, scene_min_clearance_runtime semantics (scene_collision.cuh:339-384).
//
// Bound by latency: a lane per state is too few waves (782 of them for 50,001
// Baxter configurations, 121.5 us a call, and 96 us for 256), each one chain of
// 15 joints and 75 lookups. So G lanes share a state: they take its joints'
// sines in turn, walk the tree in step (every frame has the same bits as a lane
// on its own gives it), leave the frames in LDS and take every G-th sphere each,
// two of them with their grid loads in flight together: 49 us, and 14 for 256.
// ONE: the scene is a single trilinear layer without masks (esdf_single).
// ===========================================================================
template <int G, bool ONE>
__global__ __launch_bounds__(64, 4) void k_clear(ClearArgs a) {
    extern __shared__ float s_clr[];
    constexpr int kN = kWave / G;             // states of the wave
    const DRobot& R = a.R;
    const int lane = lane_id(), sub = lane & (G - 1), slot = lane / G;
    const int J = R.n_joints, D = R.n_dof, S = R.n_sph;
    const int fstride = J * 12;
    // [slot][J][12] frames; a joint's first two floats hold its sine and cosine until its frame is there
    float* s_T = s_clr + slot * fstride;
    float* s_q = s_clr + kN * fstride;   // [D][kN]
    const long n = a.X.n_states;
    const EsdfLayer layer = ONE ? EsdfLayer(a.S) : EsdfLayer();
    for (long base = (long)blockIdx.x * kN; base < n; base += (long)gridDim.x * kN) {
        const long g = base + slot;
        const bool active = g < n;
        load_state(a.X, D, active ? g : base, true, s_q, -1, nullptr, 0, slot, kN, sub == 0);
        __syncthreads();
        float best = 1000.0f;
        float gx, gy, gz;
        Slots sl;
        for (int jj = sub; jj < J; jj += G) {
            const int4 meta = R.jmeta[jj];
            float sn = 0.0f, cs = 1.0f;
            if (meta.x >= kXRot) sincosf(meta.y >= 0 ? s_q[meta.y * kN + slot] : 0.0f, &sn, &cs);
            *reinterpret_cast<float2*>(s_T + 12 * jj) = make_float2(sn, cs);
        }
        __syncthreads();
        for (int jj = 0; jj < J; ++jj) {
            float T[12];
            const i4u meta = uload<i4u>(R.jmeta, jj);
            if (jj == 0) {
                aff_identity(T);
            } else {
                float P[12], A[12];
                sl.load(meta.w, P);
                const float2 sc = *reinterpret_cast<const float2*>(s_T + 12 * jj);
                joint_step_u(R.ft, jj, meta.x, meta.y >= 0 ? s_q[meta.y * kN + slot] : 0.0f, sc.x, sc.y, A);
                aff_compose(P, A, T);
            }
            sl.store(meta.z, T);
            if (sub == (jj & (G - 1))) {
                float4* d = reinterpret_cast<float4*>(s_T + 12 * jj);
                d[0] = make_float4(T[0], T[1], T[2], T[3]);
                d[1] = make_float4(T[4], T[5], T[6], T[7]);
                d[2] = make_float4(T[8], T[9], T[10], T[11]);
            }
        }
        __syncthreads();
        auto place = [&](const float4& sp, int jj, float& px, float& py, float& pz) {
            const float4* Tq = reinterpret_cast<const float4*>(s_T + 12 * jj);
            const float4 t0 = Tq[0], t1 = Tq[1], t2 = Tq[2];
            px = fmaf(t0.x, sp.x, fmaf(t0.y, sp.y, fmaf(t0.z, sp.z, t0.w)));
            py = fmaf(t1.x, sp.x, fmaf(t1.y, sp.y, fmaf(t1.z, sp.z, t1.w)));
            pz = fmaf(t2.x, sp.x, fmaf(t2.y, sp.y, fmaf(t2.z, sp.z, t2.w)));
        };
        if (ONE) {
            for (int s = sub; s < S; s += 2 * G) {
                const bool two = s + G < S;
                const int s2 = two ? s + G : s;
                const float4 spa = R.sph[s], spb = R.sph[s2];
                const int ja = R.sph_jnt[s], jb = R.sph_jnt[s2];
                EsdfTap ta, tb;
                float px, py, pz;
                place(spa, ja, px, py, pz);
                ta.load(layer, px, py, pz, true);
                place(spb, jb, px, py, pz);
                tb.load(layer, px, py, pz, two);
                best = fminf(best, ta.value(spa.w + a.margin));
                best = fminf(best, tb.value(spb.w + a.margin));
            }
        } else {
            for (int s = sub; s < S; s += G) {
                const float4 sp = R.sph[s];
                float px, py, pz;
                place(sp, R.sph_jnt[s], px, py, pz);
                best = fminf(best, esdf_clearance(a.S, px, py, pz, sp.w + a.margin, R.sph_id[s], false, gx, gy, gz));
            }
        }
#pragma unroll
        for (int o = 1; o < G; o <<= 1) best = fminf(best, __shfl_xor(best, o));
        if (active && sub == 0) a.out[g] = best;
        __syncthreads();   // q and the frames are read before the next round's
    }
}

// ===========================================================================
// Self collision: 16 lanes per state, sphere positions in LDS.
// mode 0: any pair with |d|^2 - (ri+rj)^2 < 0 (utils.cuh:239-267,
//         runtime_kinematics.cuh:248-283);
// mode 1: min over pairs of |d| - ri - rj with argmin pair and unit normal
//         (runtime_kinematics.cuh:294-329).
// Bound by VALU and SALU issue and the chain of a chunk's loads. Per chunk of
// four Fetch states: 1,850 VALU and 970 SALU instructions before, 1,445 and
// 640 now, with the gates and the far pairs told without square roots, the
// pairs of full blocks numbered instead of listed, the table entries in flight
// together and one kernel per mode: 325,152 rollout states 394 -> 290 us.
// ===========================================================================
constexpr int kSelfStates = kWave / kSelfGroup;
static_assert(kSelfGroup >= kMaxJoints, "the self pass composes frames with one joint per lane of a state group");

// LDS of the exact pass over four states, 16 lanes each.
struct SelfLds {
    float4* pos;    // [kSelfStates][S] (x, y, z, r)
    float4* cenc;   // [kSelfStates][NC] cluster enclosing spheres
    float* T;       // [kSelfStates][J][12] joint frames, padded
    int* par;       // [kSelfStates][J] pointer-jumping links
    static __host__ __device__ size_t bytes(int S, int NC, int J) {
        return kSelfStates * (sizeof(float4) * (size_t)(S + NC) + sizeof(float) * (size_t)(J * 12 + 4) +
                              sizeof(int) * (size_t)J);
    }
    __device__ __forceinline__ SelfLds(void* base, int S, int NC, int J) {
        pos = static_cast<float4*>(base);
        cenc = pos + kSelfStates * S;
        T = reinterpret_cast<float*>(cenc + kSelfStates * NC);
        par = reinterpret_cast<int*>(T + kSelfStates * (J * 12 + 4));
    }
};

// Sphere centres and cluster enclosing spheres of the four states from their
// frames (whole wave).
__device__ __forceinline__ void self_place(const DRobot& R, const SelfLds& L, int st, int sub) {
    const int S = R.n_sph, NC = R.n_clu;
    float4* pos = L.pos + st * S;
    float4* cenc = L.cenc + st * NC;
    const float* Ts = L.T + st * (R.n_joints * 12 + 4);
    // sphere centres (emission slot k: a joint's spheres are contiguous) and
    // each sphere cluster's enclosing sphere, from the frames
    // (each lane's table entries four at a time, before the first is used)
    auto put = [&](const float4& sp, int jj, float4* out) {
        const float4* Tq = reinterpret_cast<const float4*>(Ts + 12 * jj);
        const float4 t0 = Tq[0], t1 = Tq[1], t2 = Tq[2];
        *out = make_float4(fmaf(t0.x, sp.x, fmaf(t0.y, sp.y, fmaf(t0.z, sp.z, t0.w))),
                           fmaf(t1.x, sp.x, fmaf(t1.y, sp.y, fmaf(t1.z, sp.z, t1.w))),
                           fmaf(t2.x, sp.x, fmaf(t2.y, sp.y, fmaf(t2.z, sp.z, t2.w))), sp.w);
    };
    for (int k0 = sub; k0 < S; k0 += 4 * kSelfGroup) {
        float4 sp[4];
        int jj[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = min(k0 + e * kSelfGroup, S - 1);
            sp[e] = R.sph[k];
            jj[e] = R.sph_jnt[k];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (k0 + e * kSelfGroup < S) put(sp[e], jj[e], pos + k0 + e * kSelfGroup);
    }
    for (int c = sub; c < NC; c += kSelfGroup) put(R.clu_enc[c], R.clu_jnt[c], cenc + c);
}

// Exact self check of the four states (16 lanes each) from their sphere
// centres: the pairs of every block whose clusters are near, the outputs of
// states with `active`. live: states whose pairs are checked. MODE: the pass's.
template <int MODE>
__device__ __forceinline__ void self_pairs(const SelfArgs& a, const SelfLds& L, int st, int sub, bool active, bool live,
                                           long gs, int unit, int kstate) {
    const DRobot& R = a.R;
    const float4* pos = L.pos + st * R.n_sph;
    const float4* cenc = L.cenc + st * R.n_clu;
    // Pairs come in blocks by the sphere clusters of their two spheres; a
    // cluster's enclosing sphere contains all of its spheres, so a block
    // whose two enclosing spheres are at clearance >= band holds no pair
    // below band (band = 0 for the any-collision check, where "below" is the
    // strict d^2 < (r_i + r_j)^2 test). The 16 lanes of a state test 16
    // blocks at once; then every block that passes for some state of the
    // wave has its pair list walked, 16 pairs per step.
    const float band = MODE == 0 ? 0.0f : a.band;
    auto near = [&](float4 e, float4 f) {
        const float dx = e.x - f.x, dy = e.y - f.y, dz = e.z - f.z;
        const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        // (mode 1: |d| - rs < band, squared; the enclosing spheres' padding covers the rounding)
        const float rs = MODE == 0 ? e.w + f.w : fmaxf(e.w + f.w + band, 0.0f);
        return d2 < rs * rs;
    };
    float best = 1000.0f;
    int bkey = INT_MAX;   // (block << 16 | pair) of the best pair: ties go to the first
    bool hit = false;
    // lane sub holds the entry of block b0 + sub (DRobot::cpx), the next pass's
    // loaded ahead; a walked block's comes from its lane in the first state
    // group. A block of all pairs of its clusters, nearly every one, gives pair k's
    // slots by a division, without a look at the list.
    int4 nb4 = sub < R.n_cpb ? R.cpx[sub] : make_int4(0, 0, 0, 0);
    for (int b0 = 0; b0 < R.n_cpb; b0 += kSelfGroup) {
        const int bb = b0 + sub;
        const int4 hb = nb4;
        if (bb + kSelfGroup < R.n_cpb) nb4 = R.cpx[bb + kSelfGroup];
        const bool g = live && !hit && bb < R.n_cpb && near(cenc[hb.x & 0xFF], cenc[(hb.x >> 8) & 0xFF]);
        const unsigned long long bal = __ballot(g);
        const unsigned mine = (unsigned)(bal >> (st * kSelfGroup)) & 0xFFFFu;
        unsigned todo = (unsigned)(bal | (bal >> 16) | (bal >> 32) | (bal >> 48)) & 0xFFFFu;   // wave-uniform
        while (todo) {
            const int t = __builtin_ctz(todo);
            todo &= todo - 1u;
            const int b = b0 + t;
            const int first = __builtin_amdgcn_readlane(hb.z, t), nm = __builtin_amdgcn_readlane(hb.w, t);
            const int n = nm & 0xFFFF, inv = nm >> 16;   // inv: ceil(4096 / spheres of B), exact below 256
            const int nb = __builtin_amdgcn_readlane(hb.x, t) >> 16, ab = __builtin_amdgcn_readlane(hb.y, t);
            const bool on = ((mine >> t) & 1u) != 0u && !hit;
            for (int k0 = 0; k0 < n; k0 += kSelfGroup) {
                // (branch-free up to the rare pair that counts: lanes without
                // one take the block's last pair along)
                const int k = min(k0 + sub, n - 1);
                const bool valid = on && k0 + sub < n;
                unsigned pr;
                if (nb) {
                    const int i = (k * inv) >> 12;
                    pr = (unsigned)(ab + i + ((k - i * nb) << 16));
                } else {
                    pr = R.cpl[first + k];
                }
                const float4 u = pos[pr & 0xFFFFu], v = pos[pr >> 16];
                const float ux = u.x - v.x, uy = u.y - v.y, uz = u.z - v.z;
                const float e2 = fmaf(uz, uz, fmaf(uy, uy, ux * ux));
                const float rs = u.w + v.w;
                if (MODE == 0) {
                    hit = hit || (valid && e2 - rs * rs < 0.0f);
                } else {
                    // only a pair below the band and no farther than the best
                    // so far counts: the others are told without the root
                    // (with room for its rounding)
                    const float lim = fmaxf(fminf(best, band) + rs, 0.0f);
                    if (valid && e2 <= fmaf(lim * lim, 1.00001f, 1e-12f)) {
                        const float cl = sqrtf(e2) - rs;
                        const int key = (b << 16) | k;
                        if (cl < best || (cl == best && key < bkey)) {
                            best = cl;
                            bkey = key;
                        }
                    }
                }
            }
            if (MODE == 0) {
                // share the state's verdict so its lanes stop
                hit = ((__ballot(hit) >> (st * kSelfGroup)) & 0xFFFFull) != 0ull;
            }
        }
        if (MODE == 0 && __ballot(live && !hit) == 0ull) break;
    }
    if (MODE == 0) {
        if (active && sub == 0) {
            if (a.unit_first_hit) {
                if (hit) atomicMin((unsigned*)&a.unit_first_hit[unit], (unsigned)kstate);
            } else {
                a.hit_out[gs] = hit ? 1 : 0;
            }
        }
    } else {
#pragma unroll
        for (int off = 1; off < kSelfGroup; off <<= 1) {
            const float ob = __shfl_xor(best, off, kSelfGroup);
            const int ok = __shfl_xor(bkey, off, kSelfGroup);
            if (ob < best || (ob == best && ok < bkey)) {
                best = ob;
                bkey = ok;
            }
        }
        if (active && sub == 0) {
            float* o = a.out + 8 * (size_t)gs;
            o[0] = best;
            if (bkey != INT_MAX) {
                const unsigned pr = R.cpl[R.cpb[bkey >> 16].z + (bkey & 0xFFFF)];
                const int si = (int)(pr & 0xFFFFu), sj = (int)(pr >> 16);
                const float4 u = pos[si], v = pos[sj];
                const float dx = u.x - v.x, dy = u.y - v.y, dz = u.z - v.z;
                const float inv = 1.0f / sqrtf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
                o[1] = __int_as_float(R.sph_id[si]); o[2] = __int_as_float(R.sph_id[sj]);
                o[3] = dx * inv; o[4] = dy * inv; o[5] = dz * inv;
            } else {
                o[1] = __int_as_float(-1); o[2] = __int_as_float(-1);
                o[3] = o[4] = o[5] = 0.0f;
            }
            o[6] = o[7] = 0.0f;
        }
    }
}

// Whether a state can no longer change its unit's first hit: an edge's states
// past its known hit, every state of another unit that has one.
__device__ __forceinline__ bool unit_settled(const SelfArgs& a, const StateRef& ref) {
    const int fh = a.unit_first_hit[ref.unit];
    return a.X.source == kSrcEdge ? (unsigned)fh <= (unsigned)ref.k : fh >= 0;
}

// GATED: mode 0 of a model whose exact pairs do not decide alone.
template <int MODE, bool GATED>
__global__ __launch_bounds__(64, 4) void k_self(SelfArgs a) {
    extern __shared__ float4 s_dyn4[];
    const DRobot& R = a.R;
    const int lane = lane_id();
    const int sub = lane & (kSelfGroup - 1);
    const int st = lane / kSelfGroup;
    const int S = R.n_sph, D = R.n_dof, J = R.n_joints;
    const SelfLds L(s_dyn4, S, R.n_clu, J);
    const int fstride = J * 12 + 4;
    float* s_q = reinterpret_cast<float*>(reinterpret_cast<char*>(s_dyn4) + SelfLds::bytes(S, R.n_clu, J));   // [kMaxDof][kSelfStates]
    int* s_end = reinterpret_cast<int*>(s_q + kMaxDof * kSelfStates); // [2][64] unit ends / starts of a chunk
    float4* s_apos = reinterpret_cast<float4*>(s_end + 2 * kWave);    // gated mode 0: [kSelfStates][A] approx spheres
    const long n_states = state_count(a.X);
    // With the plan's chunk table a chunk names its first unit (staged unit
    // ends make the state -> unit lookup an LDS bisection) or, waypoint-major,
    // its problem; without it states go in flat order.
    const bool chunked = a.C.tab != nullptr;
    const long n_work = chunked ? (long)a.C.n_chunks : (n_states + kSelfStates - 1) / kSelfStates;
    // the lane's joint once per wave, the next chunk's table entry a round ahead
    JointRegs jt;
    jt.load(R, sub);
    int4 chn = make_int4(0, 0, 0, 0);
    if (chunked && (long)blockIdx.x < n_work) chn = a.C.tab[blockIdx.x];
    for (long w = blockIdx.x; w < n_work; w += gridDim.x) {
    long base, g;
    bool active;
    int u0 = -1, prob = 0;
    if (chunked) {
        const int4 ch = chn;
        if (w + gridDim.x < n_work) chn = a.C.tab[w + gridDim.x];
        base = ch.y;
        g = base + st;
        active = g < ch.z;
        u0 = ch.w;
        prob = ch.x;
        stage_unit_ends(a.X, u0, s_end);
        __syncthreads();
    } else {
        base = w * kSelfStates;
        g = base + st;
        active = g < n_states;
        if (a.C.unit_hint) {
            u0 = uniform(a.C.unit_hint[base >> 6]);
            stage_unit_ends(a.X, u0, s_end);
            __syncthreads();
        }
    }
    // units already decided need no configuration, FK or pairs (the unit
    // first-hit mode runs over densified trajectories and edge midpoints)
    const bool by_unit = a.unit_first_hit && (a.X.source == kSrcDense || a.X.source == kSrcBfs);
    if (by_unit) {
        int b0, b1;
        const int u = find_unit(a.X.dense_off, a.X.n_traj, active ? g : base, u0, s_end, &b0, &b1);
        if (active && a.unit_first_hit[u] >= 0) active = false;
        if (!wave_any(active)) continue;
    }
    // Every lane of a state group resolves the state; lane 0 stores its q.
    const StateRef ref = load_state(a.X, D, active ? g : base, true, s_q, u0, s_end, prob, st, kSelfStates, sub == 0);
    if (a.unit_first_hit && !by_unit) {
        if (active && unit_settled(a, ref)) active = false;
        if (!wave_any(active)) continue;
    }
    __syncthreads();
    float* Ts = L.T + st * fstride;
    group_frames(jt, J, s_q + st, kSelfStates, Ts, L.par + st * J, sub);
    self_place(R, L, st, sub);
    __syncthreads();
    bool live = active;   // states whose pairs are checked (gated: an approximate pair collides)
    if (GATED) {
        // Approximate pairs first (two_phase_cc.cuh:114-131): a state none of
        // whose approximate pairs collide has no self collision. Their frames
        // come from the approximate chain when the model has its own (the
        // exact positions above no longer need the full chain's).
        if (R.aft) {
            JointRegs ja;
            ja.load<true>(R, sub);
            group_frames(ja, J, s_q + st, kSelfStates, Ts, L.par + st * J, sub);
        }
        float4* apos = s_apos + st * R.n_apx;
        for (int k = sub; k < R.n_apx; k += kSelfGroup) {
            const float4 sp = R.apx_orig[k];
            const float4* Tq = reinterpret_cast<const float4*>(Ts + 12 * R.apx_jnt[k]);
            const float4 t0 = Tq[0], t1 = Tq[1], t2 = Tq[2];
            apos[k] = make_float4(fmaf(t0.x, sp.x, fmaf(t0.y, sp.y, fmaf(t0.z, sp.z, t0.w))),
                                  fmaf(t1.x, sp.x, fmaf(t1.y, sp.y, fmaf(t1.z, sp.z, t1.w))),
                                  fmaf(t2.x, sp.x, fmaf(t2.y, sp.y, fmaf(t2.z, sp.z, t2.w))), sp.w);
        }
        __syncthreads();
        bool ah = false;
        for (int p = sub; p < R.n_apx_pairs && live; p += kSelfGroup) {
            const int2 pr = R.apx_pairs[p];
            const float4 u = apos[pr.x], v = apos[pr.y];
            const float ux = u.x - v.x, uy = u.y - v.y, uz = u.z - v.z;
            const float r2 = u.w + v.w;
            ah = ah || fmaf(uz, uz, fmaf(uy, uy, ux * ux)) - r2 * r2 < 0.0f;
        }
        live = live && ((__ballot(ah) >> (st * kSelfGroup)) & 0xFFFFull) != 0ull;
    }
    self_pairs<MODE>(a, L, st, sub, active, live, ref.gs, ref.unit, ref.k);
    __syncthreads();   // positions of this round are dead before the next load
    }
}

// ===========================================================================
// Any-collision self pass in two steps, for models with rigid transforms
// (DRobot::far_blk): rough distances settle nearly every state, and the few
// they leave open go through the exact pass above, four at a time.
//
// kFar lanes share a state: they take its joints' sines in turn and walk the
// tree in step (frames kept in LDS for the pairs), place the clusters' centres,
// test every kFar-th block's two enclosing spheres each, and for the blocks
// near in some state take every kFar-th sphere b of the smaller cluster, place it
// in the larger cluster's link frame and measure it against that link's
// constant spheres a, |b - a|^2 = |b|^2 + (-2a . b + |a|^2): four multiply-adds a
// pair with a's constants in SGPRs. val = |b - a|^2 - (ra + rb + slack)^2 above
// its rounding err for all pairs proves the state free (slack bounds the frames'
// and the transforms' errors), val below -(4 rs slack + err) for one proves it
// hit (of a slack up to the radii). What is open is decided by the exact pass, so
// the verdicts are its own.
// Bound by VALU issue: frames once per state instead of in every group's rounds,
// and 210 pairs of near blocks a wave of states where the exact pass spends about
// 1,000 instructions on four states. Where it runs: see self_far.
// ===========================================================================
constexpr int kFar = 4;
constexpr int kFarStates = kWave / kFar;

struct FarLds {
    size_t T, cen, enc, sph, gate, q, end, list, ref, bytes;
    __host__ __device__ explicit FarLds(const DRobot& R) {
        constexpr int kn = kFarStates;
        size_t o = 0;
        auto take = [&](size_t n) {
            const size_t at = o;
            o += (n + 15) & ~(size_t)15;
            return at;
        };
        T = take((size_t)R.n_joints * kn * 48);
        cen = take((size_t)R.n_clu * kn * 12);
        const size_t exact = SelfLds::bytes(R.n_sph, R.n_clu, R.n_joints);   // takes T's and cen's place
        if (o < exact) o = (exact + 15) & ~(size_t)15;
        enc = take((size_t)R.n_clu * 16);
        sph = take((size_t)R.n_sph * 16);
        gate = take((size_t)R.n_cpb * 4);
        q = take((size_t)R.n_dof * kn * 4);
        end = take(2 * kWave * 4);
        list = take((size_t)kn * 4);
        ref = take((size_t)kn * 16);
        bytes = o;
    }
};

__global__ __launch_bounds__(64, 4) void k_self_far(SelfArgs a) {
    extern __shared__ float4 s_dyn4[];
    constexpr int G = kFar, kN = kFarStates;
    const DRobot& R = a.R;
    const int lane = lane_id(), sub = lane & (G - 1), slot = lane / G;
    const int S = R.n_sph, D = R.n_dof, J = R.n_joints, NC = R.n_clu;
    const FarLds lay(R);
    char* base_lds = reinterpret_cast<char*>(s_dyn4);
    float* s_T = reinterpret_cast<float*>(base_lds + lay.T);      // [J][kN][12]; a joint's sine and cosine first
    float* s_cen = reinterpret_cast<float*>(base_lds + lay.cen);  // [NC][3][kN]
    float4* s_enc = reinterpret_cast<float4*>(base_lds + lay.enc);
    float4* s_sph = reinterpret_cast<float4*>(base_lds + lay.sph);
    int* s_gate = reinterpret_cast<int*>(base_lds + lay.gate);
    float* s_q = reinterpret_cast<float*>(base_lds + lay.q);      // [D][kN]
    int* s_end = reinterpret_cast<int*>(base_lds + lay.end);
    int* s_list = reinterpret_cast<int*>(base_lds + lay.list);    // states left open
    int4* s_ref = reinterpret_cast<int4*>(base_lds + lay.ref);    // per state: plan index, unit, state of the unit
    for (int k = lane; k < NC; k += kWave) s_enc[k] = R.clu_enc[k];
    for (int k = lane; k < S; k += kWave) s_sph[k] = R.sph[k];
    for (int k = lane; k < R.n_cpb; k += kWave) s_gate[k] = R.far_gate[k];
    const float rsure = 8.0f * R.far_rmax;
    const long n_states = state_count(a.X);
    const bool chunked = a.C.tab != nullptr;
    const long n_work = chunked ? (long)a.C.n_chunks : (n_states + kN - 1) / kN;
    for (long w = blockIdx.x; w < n_work; w += gridDim.x) {
        __syncthreads();   // the last round's LDS is read
        long base, g;
        bool active;
        int u0 = -1, prob = 0;
        if (chunked) {
            const int4 ch = a.C.tab[w];
            base = ch.y;
            g = base + slot;
            active = g < ch.z;
            u0 = ch.w;
            prob = ch.x;
            stage_unit_ends(a.X, u0, s_end);
        } else {
            base = w * kN;
            g = base + slot;
            active = g < n_states;
            if (a.C.unit_hint) {
                u0 = uniform(a.C.unit_hint[base >> 6]);
                // a chunk inside one unit that has its hit
                if (a.unit_first_hit && a.X.source != kSrcEdge && a.X.dense_off[u0 + 1] >= base + kN &&
                    a.unit_first_hit[u0] >= 0)
                    continue;
                stage_unit_ends(a.X, u0, s_end);
            }
        }
        __syncthreads();
        const bool by_unit = a.unit_first_hit && (a.X.source == kSrcDense || a.X.source == kSrcBfs);
        if (by_unit) {
            int b0, b1;
            const int u = find_unit(a.X.dense_off, a.X.n_traj, active ? g : base, u0, s_end, &b0, &b1);
            if (active && a.unit_first_hit[u] >= 0) active = false;
            if (!wave_any(active)) continue;
        }
        const StateRef ref = load_state(a.X, D, active ? g : base, true, s_q, u0, s_end, prob, slot, kN, sub == 0);
        if (a.unit_first_hit && !by_unit) {
            if (active && unit_settled(a, ref)) active = false;
            if (!wave_any(active)) continue;
        }
        if (sub == 0) s_ref[slot] = make_int4((int)ref.gs, ref.unit, ref.k, 0);
        __syncthreads();
        // frames and cluster centres
        for (int jj = sub; jj < J; jj += G) {
            const int4 meta = R.jmeta[jj];
            float sn = 0.0f, cs = 1.0f;
            if (meta.x >= kXRot) sincosf(meta.y >= 0 ? s_q[meta.y * kN + slot] : 0.0f, &sn, &cs);
            *reinterpret_cast<float2*>(s_T + 12 * (jj * kN + slot)) = make_float2(sn, cs);
        }
        __syncthreads();
        float T[12];
        float far_at = 0.0f;   // the joint farthest from the origin
        for (int jj = 0; jj < J; ++jj) {
            const i4u meta = uload<i4u>(R.jmeta, jj);
            float* Tj = s_T + 12 * (jj * kN + slot);
            if (jj == 0) {
                aff_identity(T);
            } else {
                float P[12], A[12];
                const int par = uload<int>(R.parent, jj);
                if (par == 0) {
                    aff_identity(P);
                } else if (par == jj - 1) {
#pragma unroll
                    for (int k = 0; k < 12; ++k) P[k] = T[k];
                } else {
                    __syncthreads();   // another lane of the state stored it
                    const float* Tp = s_T + 12 * (par * kN + slot);
#pragma unroll
                    for (int k = 0; k < 12; ++k) P[k] = Tp[k];
                }
                const float2 sc = *reinterpret_cast<const float2*>(Tj);
                joint_step_u(R.ft, jj, meta.x, meta.y >= 0 ? s_q[meta.y * kN + slot] : 0.0f, sc.x, sc.y, A);
                aff_compose(P, A, T);
            }
            far_at = max_nan(far_at, fabsf(T[3]) + fabsf(T[7]) + fabsf(T[11]));
            if (sub == (jj & (G - 1))) {
                float4* d = reinterpret_cast<float4*>(Tj);
                d[0] = make_float4(T[0], T[1], T[2], T[3]);
                d[1] = make_float4(T[4], T[5], T[6], T[7]);
                d[2] = make_float4(T[8], T[9], T[10], T[11]);
            }
            const int c1 = uload<int>(R.clu_off, jj + 1);
            for (int c = uload<int>(R.clu_off, jj) + sub; c < c1; c += G) {
                const float4 ce = s_enc[c];
                float x, y, z;
                aff_point(T, ce.x, ce.y, ce.z, x, y, z);
                float* o = s_cen + 3 * c * kN + slot;
                o[0] = x; o[kN] = y; o[2 * kN] = z;
            }
        }
        __syncthreads();
        // A joint far off its limits adds its place's rounding. The proofs need a
        // slack below the radii: a place beyond that, or that is no number, is
        // left to the exact pass.
        const float slack = R.far_slack + 4e-6f * far_at;
        const bool lost = !(slack <= R.far_rmax);
        float open = 1.0f, sure = 1.0f;   // smallest margins: open < 0 not proven clear, sure < 0 proven hit
        for (int b0 = 0; b0 < R.n_cpb; b0 += G) {
            const int bb = b0 + sub;
            bool near = active && !lost && bb < R.n_cpb;
            if (near) {
                const int ids = s_gate[bb], cA = ids & 0xFFFF, cB = ids >> 16;
                const float* p = s_cen + 3 * cA * kN + slot;
                const float* q = s_cen + 3 * cB * kN + slot;
                const float dx = p[0] - q[0], dy = p[kN] - q[kN], dz = p[2 * kN] - q[2 * kN];
                const float rs = s_enc[cA].w + s_enc[cB].w + slack;
                near = fmaf(dz, dz, fmaf(dy, dy, dx * dx)) < rs * rs;
            }
            const unsigned long long bal = __ballot(near);
            if (bal == 0ull) continue;
            unsigned todo = 0u;   // bit p: block b0 + p is near in some state
#pragma unroll
            for (int p = 0; p < G; ++p) {
                unsigned long long col = 1ull << p;
#pragma unroll
                for (int k = G; k < kWave; k <<= 1) col |= col << k;
                todo |= (bal & col) ? 1u << p : 0u;
            }
            while (todo) {
                const int p = __builtin_ctz(todo);
                todo &= todo - 1u;
                const i4u blk = uload<i4u>(R.far_blk, b0 + p);
                const int a0 = blk.x & 0xFFFF, na = blk.x >> 16, s0 = blk.y & 0xFFFF, nb = blk.y >> 16;
                const float4* A = reinterpret_cast<const float4*>(s_T + 12 * ((blk.z & 0xFFFF) * kN + slot));
                const float4* B = reinterpret_cast<const float4*>(s_T + 12 * ((blk.z >> 16) * kN + slot));
                // M: B's link frame to A's, rotation transposed
                float M[12];
                {
                    const float4 a0r = A[0], a1r = A[1], a2r = A[2], b0r = B[0], b1r = B[1], b2r = B[2];
                    const float tx = b0r.w - a0r.w, ty = b1r.w - a1r.w, tz = b2r.w - a2r.w;
                    auto row = [&](float u, float v, float x, float* m) {
                        m[0] = fmaf(x, b2r.x, fmaf(v, b1r.x, u * b0r.x));
                        m[1] = fmaf(x, b2r.y, fmaf(v, b1r.y, u * b0r.y));
                        m[2] = fmaf(x, b2r.z, fmaf(v, b1r.z, u * b0r.z));
                        m[3] = fmaf(x, tz, fmaf(v, ty, u * tx));
                    };
                    row(a0r.x, a1r.x, a2r.x, M);
                    row(a0r.y, a1r.y, a2r.y, M + 4);
                    row(a0r.z, a1r.z, a2r.z, M + 8);
                }
                for (int k0 = 0; k0 < nb; k0 += G) {
                    const int k = min(k0 + sub, nb - 1);   // past the end: the last one again
                    const float4 sp = s_sph[s0 + k];
                    float x, y, z;
                    aff_point(M, sp.x, sp.y, sp.z, x, y, z);
                    const float bbq = fmaf(z, z, fmaf(y, y, x * x));
                    const float cb = sp.w + slack;
                    float mn = INFINITY;
                    if (blk.w < 0) {
                        for (int i = 0; i < na; i += 4) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int t = 2 * (a0 + min(i + e, na - 1));
                                const f4u c = uload<f4u>(R.far_sph, t);
                                const float r2 = uload<float>(R.far_sph, 4 * (t + 1));
                                mn = fminf(mn, fmaf(x, c.x, fmaf(y, c.y, fmaf(z, c.z, fmaf(cb, r2, c.w)))));
                            }
                        }
                    } else {
                        const int mask = R.far_mask[blk.w + k];
                        for (int i = 0; i < na; ++i) {
                            const int t = 2 * (a0 + i);
                            const f4u c = uload<f4u>(R.far_sph, t);
                            const float r2 = uload<float>(R.far_sph, 4 * (t + 1));
                            const float v = fmaf(x, c.x, fmaf(y, c.y, fmaf(z, c.z, fmaf(cb, r2, c.w))));
                            mn = fminf(mn, (mask >> i) & 1 ? v : INFINITY);
                        }
                    }
                    const float val = fmaf(-cb, cb, bbq) + mn, err = 1e-6f * (bbq + R.far_scale2 + cb * cb);
                    open = fminf(open, val - err);
                    sure = fminf(sure, val + err + rsure * slack);
                }
            }
        }
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            open = fminf(open, __shfl_xor(open, o));
            sure = fminf(sure, __shfl_xor(sure, o));
        }
        const bool is_hit = active && sure < 0.0f && !lost;
        const bool is_open = active && (open < 0.0f || lost) && !is_hit;
        if (active && sub == 0 && !is_open) {
            if (!a.unit_first_hit) a.hit_out[ref.gs] = is_hit ? 1 : 0;
            else if (is_hit) atomicMin((unsigned*)&a.unit_first_hit[ref.unit], (unsigned)ref.k);
        }
        // what is open, four states at a time
        const unsigned long long om = __ballot(is_open && sub == 0);
        if (om == 0ull) continue;
        if (is_open && sub == 0) s_list[rank_below(om)] = slot;
        const int n_open = __popcll(om);
        const int sub16 = lane & (kSelfGroup - 1), st = lane / kSelfGroup;
        const SelfLds L(base_lds, S, NC, J);
        for (int i0 = 0; i0 < n_open; i0 += kSelfStates) {
            __syncthreads();
            const bool on = i0 + st < n_open;
            const int col = s_list[on ? i0 + st : i0];
            const int4 rf = s_ref[col];
            JointRegs jt;
            jt.load(R, sub16);
            group_frames(jt, J, s_q + col, kN, L.T + st * (J * 12 + 4), L.par + st * J, sub16);
            self_place(R, L, st, sub16);
            __syncthreads();
            self_pairs<0>(a, L, st, sub16, on, on, rf.x, rf.y, rf.z);
        }
    }
}

// ===========================================================================
// FK outputs: every joint's world frame (fk_joint_transforms_runtime,
// planning/runtime_kinematics.cuh:97-171: column-major, out[c*4 + r] = T[r][c])
// and every sphere's world centre (fk_runtime), in original joint / sphere order.
//
// Bound by its writes (Fetch: 576 + 1,776 B a configuration against 32 B read).
// A wave takes four configurations at a time, 16 lanes each for the frames
// (group_frames), then the whole wave for one configuration's outputs after
// another: lane i stores float4 i of its frames in output order, and sphere i
// of the emission order, whose outputs lie within one link's few hundred
// bytes, so that every store instruction covers whole cache lines. One lane
// per configuration, which this replaced, stored 4 and 16 bytes at the
// configurations' strides (65,537 Fetch configurations: 67.3 us,
// against 35.0 us now; a fill of as many bytes takes 26).
// WIDE: both outputs are 16-byte aligned; else they go out float by float (a
// flag instead splits every store into floats).
// ===========================================================================
template <bool WIDE>
__global__ __launch_bounds__(64) void k_fk_out(DRobot R, DStates X, float* frames, float* spheres) {
    extern __shared__ float4 s_fk[];
    const int lane = lane_id(), sub = lane & (kGrp - 1), slot = lane / kGrp;
    const int J = R.n_joints, D = R.n_dof, S = R.n_sph;
    const int fstride = J * 12 + 4;
    float* s_T = reinterpret_cast<float*>(s_fk);                         // [slot][J][12]
    float* s_q = s_T + kGrpStates * fstride;                             // [slot][D]
    int* s_par = reinterpret_cast<int*>(s_q + kGrpStates * kMaxDof);     // [slot][J]
    const long n = X.n_states;
    const long step = (long)gridDim.x * kGrpStates;
    long base = (long)blockIdx.x * kGrpStates;
    // the next four configurations (4 D <= 60 floats) are loaded a round ahead
    auto fetch = [&](long b) {
        const long left = n - b;
        const int m = left > 0 ? D * (int)(left < kGrpStates ? left : kGrpStates) : 0;
        return lane < m ? X.cfg[(size_t)b * D + lane] : 0.0f;
    };
    auto put = [&](float* o, const float4& v) {
        if (WIDE) {
            *reinterpret_cast<float4*>(o) = v;
        } else {
            o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
        }
    };
    JointRegs jt;
    jt.load(R, sub);
    float qn = fetch(base);
    // 4 J <= 64: lane i's frame column, lane & 3, of joint position fj
    int fj = 0;
    for (int k = 0; k < J; ++k)
        if (R.jorig[k] == lane >> 2) fj = k;
    // table entries of the first two rounds of spheres (every sphere of a
    // model of up to 128) stay in registers
    float4 spa = make_float4(0.0f, 0.0f, 0.0f, 0.0f), spb = spa;
    int ja = 0, ida = 0, jb = 0, idb = 0;
    if (lane < S) { spa = R.sph[lane]; ja = R.sph_jnt[lane]; ida = R.sph_id[lane]; }
    if (lane + kWave < S) { spb = R.sph[lane + kWave]; jb = R.sph_jnt[lane + kWave]; idb = R.sph_id[lane + kWave]; }
    for (; base < n; base += step) {
        const int m = (int)(n - base < kGrpStates ? n - base : kGrpStates);
        if (lane < kGrpStates * D) s_q[lane] = qn;
        qn = fetch(base + step);
        __syncthreads();
        group_frames(jt, J, s_q + slot * D, 1, s_T + slot * fstride, s_par + slot * J, sub);
        for (int g = 0; g < m; ++g) {
            const float* Tg = s_T + g * fstride;
            if (frames && lane < 4 * J) {
                const float* T = Tg + 12 * fj + (lane & 3);
                put(frames + ((size_t)(base + g) * J * 4 + lane) * 4,
                    make_float4(T[0], T[4], T[8], (lane & 3) == 3 ? 1.0f : 0.0f));
            }
            auto place = [&](const float4& sp, int jj, int id) {
                const float4* Tq = reinterpret_cast<const float4*>(Tg + 12 * jj);
                const float4 t0 = Tq[0], t1 = Tq[1], t2 = Tq[2];
                put(spheres + ((size_t)(base + g) * S + id) * 4,
                    make_float4(fmaf(t0.x, sp.x, fmaf(t0.y, sp.y, fmaf(t0.z, sp.z, t0.w))),
                                fmaf(t1.x, sp.x, fmaf(t1.y, sp.y, fmaf(t1.z, sp.z, t1.w))),
                                fmaf(t2.x, sp.x, fmaf(t2.y, sp.y, fmaf(t2.z, sp.z, t2.w))), sp.w));
            };
            if (spheres) {
                if (lane < S) place(spa, ja, ida);
                if (lane + kWave < S) place(spb, jb, idb);
                for (int k = lane + 2 * kWave; k < S; k += kWave) place(R.sph[k], R.sph_jnt[k], R.sph_id[k]);
            }
        }
        __syncthreads();   // the frames are read before the next round's
    }
}

// ===========================================================================
// CHOMP optimiser (planning/chomp.cu:261-351, 459-557 semantics, batched)
// ===========================================================================
// Sub-states per segment of each trajectory: ceil(max segment length / step)
// when the longest segment exceeds the step, else 1 (chomp.cu:459-475, FP32 as
// the host code: squares summed in dof order, no contraction), capped at
// nsub_max (the joint-limit box diagonal over the step, which no clamped
// trajectory exceeds). One wave per trajectory.
__global__ __launch_bounds__(64) void k_chomp_nsub(ChompArgs a) {
    const int b = blockIdx.x;
    if (b >= a.X.n_traj) return;
    const int lane = lane_id();
    const int D = a.R.n_dof;
    const int t0 = a.X.traj_off[b], T = a.X.traj_off[b + 1] - t0;
    const float* th = a.theta + (size_t)t0 * D;
    float m = 0.0f;
    for (int t = lane; t < T - 1; t += kWave) {
        float d2 = 0.0f;
        for (int d = 0; d < D; ++d) {
            const float diff = __fsub_rn(th[(size_t)d * T + t + 1], th[(size_t)d * T + t]);
            d2 = __fadd_rn(d2, __fmul_rn(diff, diff));
        }
        m = fmaxf(m, __fsqrt_rn(d2));
    }
    m = wave_max(m);
    if (lane == 0) {
        int n = 1;
        if (a.check_step > 0.0f && m > a.check_step)
            n = (int)fminf(ceilf(__fdiv_rn(m, a.check_step)), (float)a.nsub_max);
        a.nsub[b] = n;
        a.first_hit[b] = -1;   // for the validity pass that follows
    }
}

// dense_off = exclusive scan of (T_b - 1) nsub[b] + 1 (dense_off[B] = total).
// One workgroup of 256 threads, each scanning a contiguous slice.
__global__ __launch_bounds__(256) void k_chomp_scan(ChompArgs a) {
    __shared__ int part[256];
    const int B = a.X.n_traj, tid = threadIdx.x;
    const int per = (B + 255) / 256, lo = tid * per, hi = min(B, lo + per);
    int acc = 0;
    for (int b = lo; b < hi; ++b) acc += (a.X.traj_off[b + 1] - a.X.traj_off[b] - 1) * a.nsub[b] + 1;
    part[tid] = acc;
    __syncthreads();
    if (tid == 0) {
        int run = 0;
        for (int k = 0; k < 256; ++k) {
            const int v = part[k];
            part[k] = run;
            run += v;
        }
        a.dense_off[B] = run;
    }
    __syncthreads();
    int run = part[tid];
    for (int b = lo; b < hi; ++b) {
        a.dense_off[b] = run;
        run += (a.X.traj_off[b + 1] - a.X.traj_off[b] - 1) * a.nsub[b] + 1;
    }
}

// Per-trajectory bookkeeping after an evaluation (chomp.cu:484-557): best
// valid snapshot, convergence streak on the best cost, polish count, done.
// One wave per trajectory (the snapshot copy uses every lane).
__global__ __launch_bounds__(64) void k_chomp_book(ChompArgs a, int initial) {
    const int b = blockIdx.x;
    if (b >= a.X.n_traj) return;
    const int lane = lane_id();
    const int D = a.R.n_dof;
    float* rec = a.record + 8 * (size_t)b;
    const float total = a.total[b];
    const bool valid = a.first_hit[b] < 0;
    bool copy = false;
    if (initial) {
        copy = valid;
    } else {
        copy = rec[PPL_CHOMP_DONE] == 0.0f && valid && total < rec[PPL_CHOMP_BEST_COST];
    }
    __syncthreads();
    if (lane == 0) {
        if (initial) {
            rec[PPL_CHOMP_BEST_COST] = valid ? total : INFINITY;
            rec[PPL_CHOMP_PREV_COST] = INFINITY;
            rec[PPL_CHOMP_SOLVED] = valid ? 1.0f : 0.0f;
            rec[PPL_CHOMP_STREAK] = 0.0f;
            rec[PPL_CHOMP_POLISH_LEFT] = (float)a.polish0;
            rec[PPL_CHOMP_DONE] = 0.0f;
            rec[PPL_CHOMP_ITERS] = 0.0f;
        } else if (rec[PPL_CHOMP_DONE] == 0.0f) {
            rec[PPL_CHOMP_ITERS] += 1.0f;
            if (copy) {
                rec[PPL_CHOMP_BEST_COST] = total;
                rec[PPL_CHOMP_SOLVED] = 1.0f;
            }
            if (rec[PPL_CHOMP_SOLVED] != 0.0f) {
                const float impr = rec[PPL_CHOMP_PREV_COST] - rec[PPL_CHOMP_BEST_COST];
                rec[PPL_CHOMP_STREAK] = (impr >= 0.0f && impr < a.convergence_eps) ? rec[PPL_CHOMP_STREAK] + 1.0f : 0.0f;
                rec[PPL_CHOMP_PREV_COST] = rec[PPL_CHOMP_BEST_COST];
                rec[PPL_CHOMP_POLISH_LEFT] -= 1.0f;
                if (rec[PPL_CHOMP_STREAK] >= 2.0f) rec[PPL_CHOMP_DONE] = 1.0f;
            }
        }
        // the next iteration starts only while no valid result is polished out
        if (rec[PPL_CHOMP_SOLVED] != 0.0f && rec[PPL_CHOMP_POLISH_LEFT] <= 0.0f) rec[PPL_CHOMP_DONE] = 1.0f;
        rec[PPL_CHOMP_LAST_COST] = total;
    }
    if (copy) {
        const size_t o = (size_t)a.X.traj_off[b] * D;
        const int n = (a.X.traj_off[b + 1] - a.X.traj_off[b]) * D;
        for (int i = lane; i < n; i += kWave) a.best[o + i] = a.theta[o + i];
    }
}

// Covariant step for one (dof, trajectory) (chomp.cu:261-290):
//   g = grad_d + lambda R theta_d with R theta = dt A^T (A theta) for the
//   5-point stencil A on the zero-padded grid, step = A^-1 g,
//   theta_d[t] -= step_size step[t] for 0 < t < T-1, clamped to the limits.
__global__ __launch_bounds__(256) void k_chomp_update(ChompArgs a) {
    extern __shared__ float s_u[];
    const int d = blockIdx.x, b = blockIdx.y;
    const float* rec = a.record + 8 * (size_t)b;
    if (rec[PPL_CHOMP_DONE] != 0.0f) return;
    const int D = a.R.n_dof;
    const int t0 = a.X.traj_off[b], T = a.X.traj_off[b + 1] - t0;
    float* x = s_u;             // [T + 8], theta with 4 zeros each side
    float* v = x + T + 8;       // [T + 4], A theta on [-2, T + 2)
    float* g = v + T + 4;       // [T]
    float* row = a.theta + (size_t)t0 * D + (size_t)d * T;
    const float* gr = a.grad + (size_t)t0 * D + (size_t)d * T;
    const float dt = a.dt;
    const float inv = 1.0f / (12.0f * dt * dt);
    for (int i = threadIdx.x; i < T + 8; i += blockDim.x) x[i] = (i >= 4 && i < T + 4) ? row[i - 4] : 0.0f;
    __syncthreads();
    for (int i = threadIdx.x; i < T + 4; i += blockDim.x) {
        const float* c = x + i + 2;   // centre at grid index i - 2
        v[i] = (-c[-2] + 16.0f * c[-1] - 30.0f * c[0] + 16.0f * c[1] - c[2]) * inv;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
        const float* c = v + t + 2;
        const float rt = dt * ((-c[-2] + 16.0f * c[-1] - 30.0f * c[0] + 16.0f * c[1] - c[2]) * inv);
        g[t] = gr[t] + a.smoothness_weight * rt;
    }
    __syncthreads();
    const float* ai = a.ainv[b];
    const float2 lim = a.R.lim[d];
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
        float step = 0.0f;
        for (int u = 0; u < T; ++u) step = fmaf(ai[(size_t)u * T + t], g[u], step);   // A^-1 symmetric
        if (t == 0 || t == T - 1) continue;
        const float nv = x[t + 4] - a.step_size * step;
        row[t] = fmaxf(lim.x, fminf(lim.y, nv));
    }
}

// ===========================================================================
// STOMP optimiser (planning/stomp.cu:565-930). Population rows are [D][T_b]
// blocks; every kernel finds a slot's row through stomp_row.
// ===========================================================================
__device__ __forceinline__ void stomp_row(const StompPop& p, int off_b, int T, int D, int r, int n_roll,
                                          const float** x, const float** cost) {
    size_t base;
    if (r < p.nf) {
        base = (size_t)p.nf * off_b + (size_t)r * T;
        *x = p.fresh + base * D;
        *cost = p.fresh_cost + base;
    } else if (r < n_roll - 1) {
        base = (size_t)p.nkeep * off_b + (size_t)(r - p.nf) * T;
        *x = p.keep + base * D;
        *cost = p.keep_cost + base;
    } else {
        *x = p.slot + (size_t)off_b * D;
        *cost = p.slot_cost + off_b;
    }
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): ten rounds of two
// 32 x 32 -> 64-bit products, the key advanced by the Weyl constants.
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, unsigned k0, unsigned k1) {
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        if (i) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        const unsigned hi0 = __umulhi(0xD2511F53u, c.x), lo0 = 0xD2511F53u * c.x;
        const unsigned hi1 = __umulhi(0xCD9E8D57u, c.z), lo1 = 0xCD9E8D57u * c.z;
        c = make_uint4(hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0);
    }
    return c;
}

// z ~ N(0, 1) for waypoint t of row (b, r, d): Box-Muller on the Philox words
// of counter (t >> 2, r | d << 16, b, iter); t % 4 picks the pair and cos / sin.
__device__ __forceinline__ float stomp_normal(const StompArgs& a, int b, int r, int d, int t) {
    const unsigned it = a.iter_dev ? *a.iter_dev + a.iter : a.iter;
    const uint4 w = philox4x32_10(make_uint4((unsigned)t >> 2, (unsigned)r | ((unsigned)d << 16), (unsigned)b, it),
                                  a.key0, a.key1);
    const int j = t & 3;
    const unsigned w1 = j < 2 ? w.x : w.z, w2 = j < 2 ? w.y : w.w;
    const float u1 = ((float)(w1 >> 9) + 0.5f) * 1.1920928955078125e-7f;   // (0, 1), exact
    const float u2 = ((float)(w2 >> 9) + 0.5f) * 1.1920928955078125e-7f;
    const float rad = sqrtf(-2.0f * logf(u1));
    float sn, cs;
    sincospif(2.0f * u2, &sn, &cs);
    return rad * ((j & 1) ? sn : cs);
}

// Kept rollouts (stomp.cu:131-170): the n_old cheapest slots of the previous
// population by total cost (state sum + control sum), ties to the lower slot,
// copied with their state costs into slots nf.. of the current one.
__global__ __launch_bounds__(64) void k_stomp_select(StompArgs a) {
    extern __shared__ float s_tot[];
    const int b = blockIdx.x;
    if (b >= a.B) return;
    const int lane = lane_id();
    const int D = a.R.n_dof, off = a.traj_off[b], T = a.traj_off[b + 1] - off;
    for (int r = lane; r < a.n_roll; r += kWave) {
        const float *x, *c;
        stomp_row(a.prev, off, T, D, r, a.n_roll, &x, &c);
        float s = 0.0f;
        for (int t = 0; t < T; ++t) s += c[t];
        const float* cs = a.ctrl_sum + ((size_t)b * a.n_roll + r) * D;
        for (int d = 0; d < D; ++d) s += cs[d];
        s_tot[r] = s == s ? s : INFINITY;
    }
    __syncthreads();
    for (int r = lane; r < a.n_roll; r += kWave) {
        const float v = s_tot[r];
        int rank = 0;
        for (int j = 0; j < a.n_roll; ++j) {
            const float u = s_tot[j];
            rank += (u < v || (u == v && j < r)) ? 1 : 0;
        }
        if (rank < a.n_old) a.sel[(size_t)b * a.n_old + rank] = r;
    }
}

__global__ __launch_bounds__(256) void k_stomp_gather(StompArgs a) {
    const int k = blockIdx.x, b = blockIdx.y;
    const int D = a.R.n_dof, off = a.traj_off[b], T = a.traj_off[b + 1] - off;
    const int src = a.sel[(size_t)b * a.n_old + k];
    const float *x, *c;
    stomp_row(a.prev, off, T, D, src, a.n_roll, &x, &c);
    const size_t base = (size_t)a.n_old * off + (size_t)k * T;
    float* dx = a.keep + base * D;
    float* dc = a.keep_cost + base;
    for (int i = threadIdx.x; i < D * T; i += blockDim.x) dx[i] = x[i];
    for (int i = threadIdx.x; i < T; i += blockDim.x) dc[i] = c[i];
}

// The optimum as the last slot (stomp.cu:172-189).
__global__ __launch_bounds__(256) void k_stomp_seed(StompArgs a) {
    const int b = blockIdx.x;
    const int D = a.R.n_dof, off = a.traj_off[b], T = a.traj_off[b + 1] - off;
    const size_t o = (size_t)off * D;
    for (int i = threadIdx.x; i < D * T; i += blockDim.x) a.slot[o + i] = a.theta[o + i];
    for (int i = threadIdx.x; i < T; i += blockDim.x) a.slot_cost[off + i] = a.theta_cost[off + i];
}

// Fresh sample rows (stomp.cu:100-127): x = clamp(theta + L z) with the
// endpoints pinned; one wave per (dof, slot, trajectory).
__global__ __launch_bounds__(64) void k_stomp_sample(StompArgs a) {
    extern __shared__ float s_z[];
    const int d = blockIdx.x, r = blockIdx.y, b = blockIdx.z;
    const int lane = lane_id();
    const int D = a.R.n_dof, off = a.traj_off[b], T = a.traj_off[b + 1] - off;
    for (int t = lane; t < T; t += kWave) s_z[t] = stomp_normal(a, b, r, d, t);
    __syncthreads();
    const float* Lt = a.Lt[b];
    const float* th = a.theta + (size_t)off * D + (size_t)d * T;
    float* out = a.fresh + ((size_t)a.cur.nf * off + (size_t)r * T) * D + (size_t)d * T;
    const float2 lim = a.R.lim[d];
    for (int t = lane; t < T; t += kWave) {
        float e = 0.0f;
        for (int k = 0; k <= t; ++k) e += Lt[(size_t)k * T + t] * s_z[k];
        if (t == 0 || t == T - 1) e = 0.0f;
        out[t] = fmaxf(lim.x, fminf(lim.y, th[t] + e));
    }
}

// Per (dof, trajectory): control cost of every population row, the
// exponentiated-cost probabilities per waypoint, the weighted noise average,
// its M projection and the unconditional step (stomp.cu:255-403, 406-460).
// Control: w x_t (R x)_t with R = dt A^T A, (A^T A x)_t the 9-point
// autocorrelation stencil of the 5-point acceleration rule, zero beyond the
// ends (the padded-grid block of stomp_precompute.cpp:24-44).
__global__ __launch_bounds__(256) void k_stomp_update(StompArgs a) {
    extern __shared__ float s_u[];
    const int d = blockIdx.x, b = blockIdx.y;
    const int D = a.R.n_dof, off = a.traj_off[b], T = a.traj_off[b + 1] - off;
    const int NR = a.n_roll;
    float* tot = s_u;             // [NR][T]: total cost, then the unnormalised weight
    float* delta = tot + NR * T;  // [T]
    const int lane = lane_id(), wave = threadIdx.x / kWave, n_waves = blockDim.x / kWave;
    const float scale = 1.0f / (144.0f * a.dt * a.dt * a.dt);
    for (int r = wave; r < NR; r += n_waves) {
        const float *x, *c;
        stomp_row(a.cur, off, T, D, r, NR, &x, &c);
        x += (size_t)d * T;
        auto X = [&](int k) { return (k >= 0 && k < T) ? x[k] : 0.0f; };
        float part = 0.0f;
        for (int t = lane; t < T; t += kWave) {
            const float xt = x[t];
            // the weights sum to zero, so the stencil is taken over x_{t+k} - x_t:
            // FP32 error then scales with the local variation, not with |x|
            auto P2 = [&](int k) { return (X(t - k) - xt) + (X(t + k) - xt); };
            const float st = P2(4) - 32.0f * P2(3) + 316.0f * P2(2) - 992.0f * P2(1);
            const float ctrl = a.w_u * xt * (st * scale);
            tot[r * T + t] = c[t] + ctrl;
            part += ctrl;
        }
        part = wave_sum(part);
        if (lane == 0) a.ctrl_sum[((size_t)b * NR + r) * D + d] = part;
    }
    __syncthreads();
    const float* th = a.theta + (size_t)off * D + (size_t)d * T;
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
        float mn = tot[t], mx = tot[t];
        for (int r = 1; r < NR; ++r) {
            mn = fminf(mn, tot[r * T + t]);
            mx = fmaxf(mx, tot[r * T + t]);
        }
        const float denom = fmaxf(mx - mn, 1.0e-8f);
        float sum = 0.0f;
        for (int r = 0; r < NR; ++r) {
            const float u = expf(-a.h * (tot[r * T + t] - mn) / denom);
            tot[r * T + t] = u;
            sum += u;
        }
        sum = fmaxf(sum, 1.0e-12f);
        const float tht = th[t];
        float acc = 0.0f;
        for (int r = 0; r < NR; ++r) {
            const float *x, *c;
            stomp_row(a.cur, off, T, D, r, NR, &x, &c);
            acc += (x[(size_t)d * T + t] - tht) * (tot[r * T + t] / sum);
        }
        delta[t] = (t == 0 || t == T - 1) ? 0.0f : acc;
    }
    __syncthreads();
    if (a.record[8 * (size_t)b + PPL_CHOMP_DONE] != 0.0f) return;
    const float* Mt = a.Mt[b];
    float* row = a.theta + (size_t)off * D + (size_t)d * T;
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
        float acc = 0.0f;
        for (int u = 0; u < T; ++u) acc += Mt[(size_t)u * T + t] * delta[u];
        if (t != 0 && t != T - 1) row[t] = th[t] + acc;
    }
}

// ===========================================================================
// MIT* substrate consumers (planning/MITStar.cu:212-329, 832-1375)
// ===========================================================================
// Per edge: FP32 length in the kernels' order, segment count
// max(1, ceil(len / seg)), and the breadth-first midpoints still to check:
// [done, min(sparse, total - 1)), or [done, total - 1) when sparse < 0.
__global__ void k_bfs_count(const float* nodes, int dim, const int* src, const int* dst, const int* done, int n_edges,
                            float seg_len, int sparse, int* k0, int* cnt) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_edges) return;
    const float* a = nodes + (size_t)src[e] * dim;
    const float* b = nodes + (size_t)dst[e] * dim;
    float len = 0.0f;
    for (int i = 0; i < dim; ++i) {
        const float diff = __fsub_rn(a[i], b[i]);
        len = fmaf(diff, diff, len);
    }
    const int total = max(1, (int)ceilf(__fdiv_rn(__fsqrt_rn(len), seg_len)));
    const int target = sparse >= 0 ? min(sparse, total - 1) : total - 1;
    const int start = done ? done[e] : 0;
    k0[e] = start;
    cnt[e] = max(0, target - start);
}

// off = exclusive scan of cnt (off[n] = total): one workgroup of 1024 threads
// takes passes of 16,384 counts, 16 consecutive counts per thread loaded
// together (one memory latency per pass), scanned in registers, then across
// the workgroup by wave scans of the thread totals. Offsets are only used when
// the 64-bit total (*total64, summed separately) is below 2^31, so every
// partial sum then fits 32 bits.
constexpr int kScanPer = 16;
__global__ __launch_bounds__(1024) void k_scan_i32(const int* cnt, int n, int* off, long long* total64) {
    __shared__ int wsum[16];
    __shared__ long long part[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int carry = 0;
    long long acc = 0;
    for (int base = 0; base < n; base += 1024 * kScanPer) {
        const int i0 = base + tid * kScanPer;
        int v[kScanPer];
        int local = 0;
#pragma unroll
        for (int k = 0; k < kScanPer; ++k) v[k] = i0 + k < n ? cnt[i0 + k] : 0;
#pragma unroll
        for (int k = 0; k < kScanPer; ++k) {
            local += v[k];
            acc += v[k];
        }
        int x = local;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int t = __shfl_up(x, o);
            if (lane >= o) x += t;
        }
        if (lane == kWave - 1) wsum[wave] = x;
        __syncthreads();
        int before = 0, tile = 0;
        for (int w = 0; w < 16; ++w) {
            const int y = wsum[w];
            before += w < wave ? y : 0;
            tile += y;
        }
        int run = carry + before + x - local;
#pragma unroll
        for (int k = 0; k < kScanPer; ++k) {
            if (i0 + k < n) off[i0 + k] = run;
            run += v[k];
        }
        carry += tile;
        __syncthreads();
    }
    // 64-bit total, reduced from 32-bit halves
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const int lo = __shfl_xor((int)(unsigned)(acc & 0xffffffffll), o);
        const int hi = __shfl_xor((int)(acc >> 32), o);
        acc += ((long long)hi << 32) | (unsigned)lo;
    }
    if (lane == 0) part[wave] = acc;
    __syncthreads();
    if (tid == 0) {
        long long t = 0;
        for (int w = 0; w < 16; ++w) t += part[w];
        *total64 = t;
        off[n] = (int)min(t, (long long)INT_MAX);
    }
}

// hint[c] = the unit holding state 64 c, for every 64-state block below the
// total (one thread per block; c < n_hint, the buffer's capacity)
__global__ void k_unit_hint(const int* off, int n, int* hint, int n_hint) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n_hint) return;
    const long g = (long)c << 6;
    if (g >= off[n]) return;
    hint[c] = upper_bound_idx(off, n, g);
}

__global__ void k_bfs_finish(const int* first_hit, const int* cnt, int n, uint8_t* cc, int* new_checks) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const bool hit = first_hit[e] >= 0;
    cc[e] = hit ? 1 : 0;
    if (new_checks) new_checks[e] = hit ? 0 : cnt[e];   // only verified-free midpoints count
}

// batch_cc: clearance of the free samples only (weight > 0: the min
// clearance, else 1000); colliding samples keep their entry.
__global__ void k_sample_clearance(const uint8_t* cc, const float* clr, int n, float weight, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || cc[i]) return;
    out[i] = weight > 0.0f ? clr[i] : 1000.0f;
}

__global__ void k_gather_rows(const float* src, int dim, const int* idx, int base, int n, float* out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)n * dim) return;
    const int r = (int)(i / dim), d = (int)(i % dim);
    const int node = idx ? idx[r] : base + r;
    out[i] = src[(size_t)node * dim + d];
}

__global__ void k_scatter(const float* v, const int* idx, int base, int n, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[idx ? idx[i] : base + i] = v[i];
}

// ===========================================================================
// Small helpers
// ===========================================================================
__global__ void k_add_u32(unsigned* p, unsigned v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p += v;
}

__global__ void k_fill_i32(int* p, int v, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// out[b] = sum of x over segment b (one wave per segment, fixed order).
__global__ __launch_bounds__(64) void k_segment_sum(const float* x, const int* off, int n_seg, float* out) {
    const int b = blockIdx.x;
    if (b >= n_seg) return;
    const int lane = lane_id();
    float acc = 0.0f;
    for (int i = off[b] + lane; i < off[b + 1]; i += kWave) acc += x[i];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) out[b] = acc;
}

// Control cost w * sum_d theta_d^T R theta_d for the 5-point acceleration
// metric R = dt * (A^T A)[pad..pad+T] (chomp_precompute.cpp:20-38), evaluated
// as dt * sum_i acc_i^2 over the stencil rows that touch the trajectory,
// acc_i = (-x[i-2] + 16x[i-1] - 30x[i] + 16x[i+1] - x[i+2]) / (12 dt^2) with
// x = 0 outside [0, T). One wave per trajectory; with `stage` the wave first
// copies its trajectory's D x T block into LDS rows padded by four zeros on
// each side (eight loads per lane in flight at a time), then evaluates the
// stencil from LDS. state (nullable): the trajectory's per-waypoint state
// costs, whose sum joins the total (the STOMP rollout total in one launch).
__global__ __launch_bounds__(64) void k_control(const float* theta, const int* traj_off, int n_traj, int D, float dt,
                                                float w, const float* state, float* out, int accumulate, int stage) {
    extern __shared__ float s_x[];
    const int b = blockIdx.x;
    if (b >= n_traj) return;
    const int lane = lane_id();
    const int t0 = traj_off[b], Tn = traj_off[b + 1] - t0;
    const float* th = theta + (size_t)t0 * D;
    const float inv = 1.0f / (12.0f * dt * dt);
    float ssum = 0.0f;
    if (state)
        for (int i = lane; i < Tn; i += kWave) ssum += state[t0 + i];
    float acc = 0.0f;
    if (stage) {
        const int rs = Tn + 8, n = D * rs;
        for (int k0 = 0; k0 < n; k0 += 8 * kWave) {
            float v[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int k = k0 + c * kWave + lane;
                const int d = k / rs, i = k - d * rs - 4;
                v[c] = (k < n && i >= 0 && i < Tn) ? th[(size_t)d * Tn + i] : 0.0f;
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int k = k0 + c * kWave + lane;
                if (k < n) s_x[k] = v[c];
            }
        }
        __syncthreads();
        for (int d = 0; d < D; ++d) {
            const float* x = s_x + d * rs + 4;
            for (int i = lane - 2; i < Tn + 2; i += kWave) {
                const float v = (-x[i - 2] + 16.0f * x[i - 1] - 30.0f * x[i] + 16.0f * x[i + 1] - x[i + 2]) * inv;
                acc = fmaf(v, v, acc);
            }
        }
    } else {
        for (int d = 0; d < D; ++d) {
            const float* x = th + (size_t)d * Tn;
            for (int i = lane - 2; i < Tn + 2; i += kWave) {
                auto X = [&](int k) { return (k >= 0 && k < Tn) ? x[k] : 0.0f; };
                const float v = (-X(i - 2) + 16.0f * X(i - 1) - 30.0f * X(i) + 16.0f * X(i + 1) - X(i + 2)) * inv;
                acc = fmaf(v, v, acc);
            }
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        acc += __shfl_xor(acc, o);
        ssum += __shfl_xor(ssum, o);
    }
    if (lane == 0) {
        const float c = w * dt * acc;
        const float base = accumulate ? out[b] : 0.0f;
        out[b] = state ? base + (ssum + c) : base + c;
    }
}

// ESDF node values = -min_o sdf_o(node), positive inside.
//
// Bound by VALU issue: a node tested against every box costs 24 instructions
// a box (128^3 nodes, 60 boxes: 71.9 us a call; its 8.4 MB of writes take 4). A
// wave takes a run of kEsdfRun 4 x 4 x 4 bricks along z, one node per lane and
// brick, and first finds the boxes that can be nearest anywhere in the brick:
// lane i measures box i at the brick's centre. A box's signed distance changes
// by at most L rho over the brick (rho its half diagonal, L the norm of the
// box's map, 1 for a unit quaternion), so a box whose distance at the centre
// exceeds the smallest (d + L rho) by more than L rho is nowhere the nearest;
// a few are left, and only they are walked: 17.4 us (20.5 a call). Rounding is covered
// by a slack of some 1e-6 of the coordinates. Boxes pass through LDS in tiles
// of 64; a tile's bound takes in the earlier tiles'. first: the launch's first run
// (a launch takes fewer than 2^32 threads, and a grid may have more).
constexpr int kEsdfRun = 4;
constexpr long kEsdfLaunch = 1L << 25;   // runs of a launch

__global__ __launch_bounds__(64) void k_esdf_build(const float* __restrict__ obb_dims, const float* __restrict__ obb_pose,
                                                   int n_obbs, float4 prm, float4 gp0, float4 gp1, int nx, int ny, int nz,
                                                   long first, float* __restrict__ out) {
    __shared__ float4 s_obb[4 * kWave];
    const float gpose[8] = {gp0.x, gp0.y, gp0.z, gp0.w, gp1.x, gp1.y, gp1.z, gp1.w};
    const int lane = lane_id();
    const int nbz = (nz + 4 * kEsdfRun - 1) / (4 * kEsdfRun), nby = (ny + 3) / 4;
    const long run = first + blockIdx.x;
    const long bxy = run / nbz;
    const int bz = (int)(run - bxy * nbz), bx = (int)(bxy / nby), by = (int)(bxy - (long)bx * nby);
    const int ix = 4 * bx + (lane >> 4), iy = 4 * by + ((lane >> 2) & 3);
    // node coordinates (may lie past the grid's end: such lanes store nothing)
    auto world = [&](float fx, float fy, float fz, float& px, float& py, float& pz) {
        const float lx = fx * prm.w - 0.5f * prm.x - gpose[0];
        const float ly = fy * prm.w - 0.5f * prm.y - gpose[1];
        const float lz = fz * prm.w - 0.5f * prm.z - gpose[2];
        // grid-local -> world with the conjugate of the stored rotation
        const float qw = gpose[3], qx = -gpose[4], qy = -gpose[5], qz = -gpose[6];
        const float tx = 2.0f * (qy * lz - qz * ly), ty = 2.0f * (qz * lx - qx * lz), tz = 2.0f * (qx * ly - qy * lx);
        px = lx + qw * tx + (qy * tz - qz * ty);
        py = ly + qw * ty + (qz * tx - qx * tz);
        pz = lz + qw * tz + (qx * ty - qy * tx);
    };
    // norm of v -> v + w t + u x t, t = 2 u x v: |q|^2 times a rotation plus (1 - |q|^2) times v
    auto map_norm = [](float w, float x, float y, float z) {
        const float n2 = w * w + x * x + y * y + z * z;
        return n2 + fabsf(1.0f - n2);
    };
    const float rho = 1.001f * 2.5980762f * fabsf(prm.w) * map_norm(gpose[3], gpose[4], gpose[5], gpose[6]);   // 1.5 sqrt(3) voxels
    float best[kEsdfRun], bound[kEsdfRun];
#pragma unroll
    for (int r = 0; r < kEsdfRun; ++r) {
        best[r] = FLT_MAX;
        bound[r] = INFINITY;
    }
    for (int t0 = 0; t0 < n_obbs; t0 += kWave) {
        const int m = min(kWave, n_obbs - t0);
        float4 rec[4] = {};
        float lip = 1.0f, mag = 0.0f;
        __syncthreads();   // the last tile's records are read
        if (lane < m) {
            const float* d = obb_dims + 4 * (size_t)(t0 + lane);
            const float* p = obb_pose + 8 * (size_t)(t0 + lane);
            const float w = p[3], x = p[4], y = p[5], z = p[6];
            rec[0] = make_float4(1.0f - 2.0f * (y * y + z * z), 2.0f * (x * y - w * z), 2.0f * (x * z + w * y), p[0]);
            rec[1] = make_float4(2.0f * (x * y + w * z), 1.0f - 2.0f * (x * x + z * z), 2.0f * (y * z - w * x), p[1]);
            rec[2] = make_float4(2.0f * (x * z - w * y), 2.0f * (y * z + w * x), 1.0f - 2.0f * (x * x + y * y), p[2]);
            rec[3] = make_float4(0.5f * d[0], 0.5f * d[1], 0.5f * d[2], 0.0f);
#pragma unroll
            for (int k = 0; k < 4; ++k) s_obb[4 * lane + k] = rec[k];
            lip = map_norm(w, x, y, z);
            mag = fabsf(p[0]) + fabsf(p[1]) + fabsf(p[2]) + fabsf(rec[3].x) + fabsf(rec[3].y) + fabsf(rec[3].z);
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kEsdfRun; ++r) {
            const int z0 = 4 * (bz * kEsdfRun + r);
            if (z0 >= nz) break;
            float px, py, pz, lx, ly, lz;
            world((float)(4 * bx) + 1.5f, (float)(4 * by) + 1.5f, (float)z0 + 1.5f, px, py, pz);
            to_box(rec[0], rec[1], rec[2], px, py, pz, lx, ly, lz);
            const float d = key_to_sdf(box_key(lx, ly, lz, rec[3]));
            const float slack = 1e-5f + 4e-6f * (mag + lip * (fabsf(px) + fabsf(py) + fabsf(pz)));
            // NaN distances bound nothing and exclude nothing
            float hi = lane < m && d == d ? d + lip * rho + slack : INFINITY;
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) hi = fminf(hi, __shfl_xor(hi, o));
            bound[r] = fminf(bound[r], hi);
            unsigned long long bits = __ballot(lane < m && !(d - lip * rho - slack > bound[r]));
            world((float)ix, (float)iy, (float)(z0 + (lane & 3)), px, py, pz);
            while (bits) {
                const int o = __ffsll(bits) - 1;
                bits &= bits - 1ull;
                to_box(s_obb[4 * o], s_obb[4 * o + 1], s_obb[4 * o + 2], px, py, pz, lx, ly, lz);
                best[r] = fminf(best[r], box_key(lx, ly, lz, s_obb[4 * o + 3]));
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kEsdfRun; ++r) {
        const int iz = 4 * (bz * kEsdfRun + r) + (lane & 3);
        if (ix < nx && iy < ny && iz < nz) out[((size_t)ix * ny + iy) * nz + iz] = -key_to_sdf(best[r]);
    }
}

int g_cus = 0;

}  // namespace

int device_cus() {
    if (g_cus == 0) {
        int dev = 0;
        (void)hipGetDevice(&dev);
        hipDeviceProp_t prop;
        (void)hipGetDeviceProperties(&prop, dev);
        g_cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    }
    return g_cus;
}

namespace {

int occupancy_grid(const void* fn, size_t dyn_smem) {
    (void)device_cus();
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 64, dyn_smem) != hipSuccess || per_cu <= 0) per_cu = 4;
    return per_cu * g_cus;
}

// The last occupancy grid asked for, by LDS bytes (calls may come from several threads).
struct GridCache {
    std::mutex mu;
    size_t lds = (size_t)-1;
    int grid = 0;
    int get(const void* fn, size_t bytes) {
        std::lock_guard<std::mutex> lk(mu);
        if (bytes != lds) {
            grid = occupancy_grid(fn, bytes);
            lds = bytes;
        }
        return grid;
    }
};

}  // namespace

size_t lds_bytes(int obb_cap, int n_dof) {
    return (size_t)obb_cap * 64 + (size_t)(n_dof + 2) * kWave * sizeof(float);
}

size_t lds_bytes_collide(int obb_cap, const DRobot& R) {
    const size_t b = lds_bytes(obb_cap, R.n_dof);
    // + record padding, sphere table, hit flags
    return R.scene_gate_fused ? b + (size_t)obb_cap * 16 * (kObbRec - 4) + (size_t)R.n_sph * 16 + kWave * sizeof(int) : b;
}

size_t lds_bytes_cost(int obb_cap, int n_dof, int n_joints, int G, bool grad) {
    size_t b = lds_bytes(obb_cap, n_dof);
    if (!grad) b += (size_t)obb_cap * 16 * (kObbRec - 4);   // record padding
    if (grad) b += (size_t)(kWave / G) * (rec_stride(n_joints) + dq_stride(n_dof)) * sizeof(float);
    return b;
}

template <int P>
static const void* collide_variant(const DRobot& R, const DScene& S) {
    if (S.n_voxel_layers > 0) return R.line ? (const void*)k_collide<true, true, P> : (const void*)k_collide<true, false, P>;
    return R.line ? (const void*)k_collide<false, true, P> : (const void*)k_collide<false, false, P>;
}

static const void* collide_kernel(const DRobot& R, const DScene& S, int chunk) {
    if (!R.scene_gate_fused) return (const void*)k_collide_gated;
    return chunk == kWave ? collide_variant<1>(R, S) : collide_variant<kCollideParts>(R, S);
}

// Workgroups that the chip holds at once (of the one-lane variant).
int grid_collide(const DRobot& R, const DScene& S, int obb_cap) {
    static GridCache cache[5];
    const int i = !R.scene_gate_fused ? 4 : (S.n_voxel_layers > 0 ? 2 : 0) + (R.line ? 1 : 0);
    return cache[i].get(collide_kernel(R, S, kWave), lds_bytes_collide(obb_cap, R));
}

int collide_lanes(const DRobot& R, long n_states) {
    return R.scene_gate_fused && n_states <= kCollideSplit ? kCollideParts : 1;
}

static const void* cost_kernel(const DRobot& R, bool esdf, bool grad) {
    if (grad) return (const void*)k_cost_grad;
    if (esdf) return R.line ? (const void*)k_state_cost<true, true> : (const void*)k_state_cost<true, false>;
    return R.line ? (const void*)k_state_cost<false, true> : (const void*)k_state_cost<false, false>;
}

int grid_cost(const DRobot& R, bool grad, size_t lds) {
    static GridCache cache[3];
    return cache[grad ? 2 : R.line ? 1 : 0].get(cost_kernel(R, false, grad), lds);
}

// A launch with its argument block; with t0/t1 the runtime records the two
// events at the kernel's own start and end (timing without event packets of
// their own around the launch).
static hipError_t launch_args(const void* k, int grid, size_t lds, hipStream_t s, void* arg, hipEvent_t t0,
                              hipEvent_t t1) {
    void* params[] = {arg};
    if (t0) return hipExtLaunchKernel(k, dim3(grid), dim3(64), params, lds, s, t0, t1, 0);
    return hipLaunchKernel(k, dim3(grid), dim3(64), params, lds, s);
}

hipError_t launch_collide(const CollideArgs& a, int grid, hipStream_t s, hipEvent_t t0, hipEvent_t t1) {
    CollideArgs arg = a;
    const void* k = collide_kernel(a.R, a.S, a.C.chunk);
    return launch_args(k, grid, lds_bytes_collide(a.C.obb_cap, a.R), s, &arg, t0, t1);
}

hipError_t launch_cost(const CostArgs& a, int grid, hipStream_t s, hipEvent_t t0, hipEvent_t t1) {
    if (a.C.tiled) return hipErrorInvalidValue;   // these kernels stage one OBB tile: tiled problems take k_cost_grp
    const size_t lds = lds_bytes_cost(a.C.obb_cap, a.R.n_dof, a.R.n_joints, a.group, a.grad != 0);
    CostArgs arg = a;
    const void* k = cost_kernel(a.R, a.P.use_esdf != 0 && a.S.n_voxel_layers > 0, a.grad != 0);
    return launch_args(k, grid, lds, s, &arg, t0, t1);
}

size_t lds_bytes_grp(int obb_cap, int n_dof, int n_joints, int n_sph, int n_clu, bool grad, bool tiled) {
    return lds_floats_grp(obb_cap, n_dof, n_joints, n_sph, n_clu, grad, tiled) * sizeof(float);
}

// Variant table: [grad][world - 1][tiled] (ESDF-only launches stage no OBBs;
// there the third index says whether the scene is a single layer, esdf_single).
const void* grp_kernel(bool grad, int world, bool tiled) {
    static const void* const tab[2][3][2] = {
        {{(const void*)k_cost_grp<false, 1, false>, (const void*)k_cost_grp<false, 1, true>},
         {(const void*)k_cost_grp_esdf<false, false>, (const void*)k_cost_grp_esdf<false, true>},
         {(const void*)k_cost_grp<false, 3, false>, (const void*)k_cost_grp<false, 3, true>}},
        {{(const void*)k_cost_grp<true, 1, false>, (const void*)k_cost_grp<true, 1, true>},
         {(const void*)k_cost_grp_esdf<true, false>, (const void*)k_cost_grp_esdf<true, true>},
         {(const void*)k_cost_grp<true, 3, false>, (const void*)k_cost_grp<true, 3, true>}}};
    return tab[grad ? 1 : 0][world - 1][tiled ? 1 : 0];
}

int grp_world(const CostArgs& a) {
    const bool obb = a.P.use_obb != 0 && a.S.n_obbs > 0;
    const bool esdf = a.P.use_esdf != 0 && a.S.n_voxel_layers > 0;
    return obb && esdf ? 3 : esdf ? 2 : 1;
}

int grid_cost_grp(bool grad, int world, bool tiled, size_t lds) {
    static std::mutex mu;
    static size_t last[2][3][2];
    static int g[2][3][2];
    static bool init = false;
    std::lock_guard<std::mutex> lk(mu);
    if (!init) {
        for (auto& x : last) for (auto& y : x) for (auto& z : y) z = (size_t)-1;
        init = true;
    }
    const int i = grad ? 1 : 0, w = world - 1, t = tiled ? 1 : 0;
    if (lds != last[i][w][t]) {
        g[i][w][t] = occupancy_grid(grp_kernel(grad, world, tiled), lds);
        last[i][w][t] = lds;
    }
    return g[i][w][t];
}

hipError_t launch_cost_grp(const CostArgs& a, int grid, hipStream_t s, hipEvent_t t0, hipEvent_t t1) {
    const size_t lds = lds_bytes_grp(a.C.obb_cap, a.R.n_dof, a.R.n_joints, a.R.n_sph, a.R.n_clu, a.grad != 0,
                                     a.C.tiled != 0);
    const int world = grp_world(a);
    const bool tiled = world == 2 ? esdf_single(a.S) : a.C.tiled != 0;   // the variant table's third index
    grid = std::max(1, std::min(grid, grid_cost_grp(a.grad != 0, world, tiled, lds)));   // persistent: occupancy x CUs
    CostArgs arg = a;
    return launch_args(grp_kernel(a.grad != 0, world, tiled), grid, lds, s, &arg, t0, t1);
}

// Lanes per state: 16 up to two waves a SIMD of them, else 8. Measured, us a call,
// Baxter (Panda): 256 configurations 13.7 against 15.3 (11 and 11), 8,192 19.6
// against 21.0 (14.3, 14.9), 20,000 35.8 against 26.6 (26.6, 21.9), 500,000 502
// against 329 (367, 288); 4 lanes lie within 15% of 8 from 50,000 on, and one
// lane needs 500,000 to be as fast (302, 318).
hipError_t launch_clear(const ClearArgs& a, hipStream_t s) {
    const long n = a.X.n_states;
    if (n <= 0) return hipSuccess;
    const int G = n * 16 <= (long)device_cus() * 4 * 2 * kWave ? 16 : 8;
    const int kn = kWave / G;
    const bool one = esdf_single(a.S);
    const void* k = G == 8 ? (one ? (const void*)k_clear<8, true> : (const void*)k_clear<8, false>)
                           : (one ? (const void*)k_clear<16, true> : (const void*)k_clear<16, false>);
    const size_t lds = sizeof(float) * kn * ((size_t)a.R.n_dof + 12 * (size_t)a.R.n_joints);
    const long blocks = std::min((n + kn - 1) / kn, (long)device_cus() * 32);
    ClearArgs arg = a;
    return launch_args(k, (int)blocks, lds, s, &arg, nullptr, nullptr);
}

// Whether a self pass takes the two steps of k_self_far: any-collision checks
// whose exact pairs decide alone, over at least 65,536 states in an order that
// keeps neighbours near (edges and trajectories; a wave's near blocks are then
// few), of models of up to 64 blocks. Measured, edges of 10 boxes with the
// self check, us a call with it and without: Panda (23 blocks) 51,132 states 67
// and 66, 180,857 106 and 124, 736,240 290 and 416; Fetch (153 blocks) 48,403 126
// and 104, 174,587 219 and 222, 699,268 664 and 787; Baxter (150), some 700,000,
// 877 and 714. Uncorrelated configurations: Panda 262,144 170 and 173, Fetch 605 and 371.
// The limit of blocks takes what wins on every size from 65,536 on; the number of
// blocks does not tell Fetch from Baxter, so large Fetch sets go without, too.
static bool self_far(const DRobot& R, int mode, int source, long n_states) {
    return mode == 0 && R.far_blk && R.self_gate_implied && R.n_cpb <= 64 && n_states >= 65536 && source != kSrcConfig &&
           source != kSrcBfs && FarLds(R).bytes <= 65536;
}

int self_chunk(const DRobot& R, int mode, int source, long n_states) {
    return self_far(R, mode, source, n_states) ? kFarStates : kSelfStates;
}

hipError_t launch_self(const SelfArgs& a, hipStream_t s) {
    const bool far = self_far(a.R, a.mode, a.X.source, a.X.n_states);
    const int kn = far ? kFarStates : kSelfStates;
    if (a.C.chunk != kn) return hipErrorInvalidValue;   // the caller's chunks are another size
    // X.n_states bounds the state count (a device-side count may be smaller,
    // then a bounded grid strides over it)
    long blocks = a.C.tab ? (long)a.C.n_chunks : (a.X.n_states + kn - 1) / kn;
    if (a.X.n_dyn && blocks > 16384) blocks = 16384;
    if (blocks <= 0) return hipSuccess;
    if (far) {
        SelfArgs arg = a;
        return launch_args((const void*)k_self_far, (int)blocks, FarLds(a.R).bytes, s, &arg, nullptr, nullptr);
    }
    const bool gate = a.mode == 0 && !a.R.self_gate_implied;   // approximate pair positions
    const size_t smem = SelfLds::bytes(a.R.n_sph, a.R.n_clu, a.R.n_joints) + sizeof(float) * (size_t)kMaxDof * kSelfStates +
                        sizeof(int) * 2 * kWave + (gate ? sizeof(float4) * (size_t)kSelfStates * a.R.n_apx : 0);
    // one chunk a wave: chunks differ in cost, and the dispatcher evens them out
    // (STOMP's rollouts: 718 us a call, 731 with four times the waves the chip
    // holds, 881 with as many)
    const void* k = a.mode != 0 ? (const void*)k_self<1, false> : gate ? (const void*)k_self<0, true> : (const void*)k_self<0, false>;
    SelfArgs arg = a;
    return launch_args(k, (int)blocks, smem, s, &arg, nullptr, nullptr);
}

hipError_t launch_fk_out(const DRobot& R, const DStates& X, float* frames, float* spheres, hipStream_t s) {
    const long groups = (X.n_states + kGrpStates - 1) / kGrpStates;
    if (groups <= 0) return hipSuccess;
    const size_t lds = sizeof(float) * (size_t)kGrpStates * (R.n_joints * 12 + 4 + kMaxDof) +
                       sizeof(int) * (size_t)kGrpStates * R.n_joints;
    const bool wide = (((uintptr_t)frames | (uintptr_t)spheres) & 15) == 0;
    static GridCache cache[2];
    const void* k = wide ? (const void*)k_fk_out<true> : (const void*)k_fk_out<false>;
    const long grid = std::min(groups, (long)cache[wide ? 1 : 0].get(k, lds));
    if (wide) hipLaunchKernelGGL(k_fk_out<true>, dim3((unsigned)grid), dim3(64), lds, s, R, X, frames, spheres);
    else hipLaunchKernelGGL(k_fk_out<false>, dim3((unsigned)grid), dim3(64), lds, s, R, X, frames, spheres);
    return hipGetLastError();
}

hipError_t launch_chomp_nsub(const ChompArgs& a, hipStream_t s) {
    if (a.X.n_traj <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_chomp_nsub, dim3(a.X.n_traj), dim3(64), 0, s, a);
    hipLaunchKernelGGL(k_chomp_scan, dim3(1), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_chomp_book(const ChompArgs& a, int initial, hipStream_t s) {
    if (a.X.n_traj <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_chomp_book, dim3(a.X.n_traj), dim3(64), 0, s, a, initial);
    return hipGetLastError();
}

hipError_t launch_chomp_update(const ChompArgs& a, int max_t, hipStream_t s) {
    if (a.X.n_traj <= 0) return hipSuccess;
    const size_t smem = sizeof(float) * (3 * (size_t)max_t + 12);
    hipLaunchKernelGGL(k_chomp_update, dim3(a.R.n_dof, a.X.n_traj), dim3(256), smem, s, a);
    return hipGetLastError();
}

hipError_t launch_stomp_reuse(const StompArgs& a, int, hipStream_t s) {
    if (a.B <= 0 || a.n_old <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stomp_select, dim3(a.B), dim3(64), sizeof(float) * (size_t)a.n_roll, s, a);
    hipLaunchKernelGGL(k_stomp_gather, dim3(a.n_old, a.B), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_stomp_sample(const StompArgs& a, int max_t, hipStream_t s) {
    if (a.B <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stomp_seed, dim3(a.B), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_stomp_sample, dim3(a.R.n_dof, a.cur.nf, a.B), dim3(64), sizeof(float) * (size_t)max_t, s, a);
    return hipGetLastError();
}

size_t stomp_update_lds(int n_roll, int max_t) { return sizeof(float) * ((size_t)n_roll + 1) * (size_t)max_t; }

hipError_t launch_stomp_update(const StompArgs& a, int max_t, hipStream_t s) {
    if (a.B <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stomp_update, dim3(a.R.n_dof, a.B), dim3(256), stomp_update_lds(a.n_roll, max_t), s, a);
    return hipGetLastError();
}

hipError_t launch_bfs_count(const float* nodes, int dim, const int* src, const int* dst, const int* done, int n,
                            float seg_len, int sparse, int* k0, int* cnt, int* off, long long* total, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bfs_count, dim3((n + 255) / 256), dim3(256), 0, s, nodes, dim, src, dst, done, n, seg_len,
                       sparse, k0, cnt);
    hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, s, cnt, n, off, total);
    return hipGetLastError();
}

hipError_t launch_unit_hint(const int* off, int n, int* hint, int n_hint, hipStream_t s) {
    if (n <= 0 || n_hint <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_unit_hint, dim3((n_hint + 255) / 256), dim3(256), 0, s, off, n, hint, n_hint);
    return hipGetLastError();
}

hipError_t launch_bfs_finish(const int* first_hit, const int* cnt, int n, uint8_t* cc, int* new_checks, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bfs_finish, dim3((n + 255) / 256), dim3(256), 0, s, first_hit, cnt, n, cc, new_checks);
    return hipGetLastError();
}

hipError_t launch_sample_clearance(const uint8_t* cc, const float* clr, int n, float weight, float* out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sample_clearance, dim3((n + 255) / 256), dim3(256), 0, s, cc, clr, n, weight, out);
    return hipGetLastError();
}

hipError_t launch_gather_rows(const float* src, int dim, const int* idx, int base, int n, float* out, hipStream_t s) {
    const long total = (long)n * dim;
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_rows, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, src, dim, idx, base, n, out);
    return hipGetLastError();
}

hipError_t launch_scatter(const float* v, const int* idx, int base, int n, float* out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_scatter, dim3((n + 255) / 256), dim3(256), 0, s, v, idx, base, n, out);
    return hipGetLastError();
}

hipError_t launch_add_u32(unsigned* p, unsigned v, hipStream_t s) {
    hipLaunchKernelGGL(k_add_u32, dim3(1), dim3(64), 0, s, p, v);
    return hipGetLastError();
}

hipError_t launch_fill_i32(int* p, int v, long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    long blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

hipError_t launch_segment_sum(const float* x, const int* off, int n_seg, float, float* out, hipStream_t s) {
    if (n_seg <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_segment_sum, dim3(n_seg), dim3(64), 0, s, x, off, n_seg, out);
    return hipGetLastError();
}

hipError_t launch_control_cost(const float* theta, const int* traj_off, int n_traj, int D, float dt, float w, float* out,
                               int accumulate, hipStream_t s, int t_max, const float* state) {
    if (n_traj <= 0) return hipSuccess;
    // LDS staging when the longest trajectory's padded block fits 32 KiB
    const size_t lds = t_max > 0 ? (size_t)D * (t_max + 8) * sizeof(float) : 0;
    const int stage = lds > 0 && lds <= 32768 ? 1 : 0;
    hipLaunchKernelGGL(k_control, dim3(n_traj), dim3(64), stage ? lds : 0, s, theta, traj_off, n_traj, D, dt, w, state,
                       out, accumulate, stage);
    return hipGetLastError();
}

hipError_t launch_esdf_build(const float* obb_dims, const float* obb_pose, int n_obbs, const float* voxel_params,
                             const float* voxel_pose, float* out, hipStream_t s) {
    // voxel_params / voxel_pose are host arrays here
    const float inv = 1.0f / voxel_params[3];
    auto rf = [](float x) {
        const float nearest = roundf(x);
        if (x - nearest >= 1e-4f) return (int)floorf(x);
        return (int)nearest;
    };
    const int nx = rf(voxel_params[0] * inv) + 1, ny = rf(voxel_params[1] * inv) + 1, nz = rf(voxel_params[2] * inv) + 1;
    if (nx <= 0 || ny <= 0 || nz <= 0) return hipErrorInvalidValue;   // no nodes
    const long runs = (((long)nx + 3) / 4) * (((long)ny + 3) / 4) * (((long)nz + 4 * kEsdfRun - 1) / (4 * kEsdfRun));
    for (long first = 0; first < runs; first += kEsdfLaunch)
        hipLaunchKernelGGL(k_esdf_build, dim3((unsigned)std::min(kEsdfLaunch, runs - first)), dim3(64), 0, s, obb_dims,
                           obb_pose, n_obbs, make_float4(voxel_params[0], voxel_params[1], voxel_params[2], voxel_params[3]),
                           make_float4(voxel_pose[0], voxel_pose[1], voxel_pose[2], voxel_pose[3]),
                           make_float4(voxel_pose[4], voxel_pose[5], voxel_pose[6], voxel_pose[7]), nx, ny, nz, first, out);
    return hipGetLastError();
}

}  // namespace ppl
