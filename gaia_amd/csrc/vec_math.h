// Small float3 helpers and the 3x3 block solve used by every per-vertex kernel.
#pragma once
#include <hip/hip_runtime.h>

namespace gvbd {

struct f3 {
    float x, y, z;
};

__device__ __forceinline__ f3 mk(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ f3 xyz(float4 a) { return {a.x, a.y, a.z}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator*(float s, f3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// Symmetric 3x3 block: (xx, xy, xz, yy, yz, zz).
struct Sym3 {
    float xx, xy, xz, yy, yz, zz;
};

__device__ __forceinline__ f3 sym_mul(const Sym3& h, f3 v) {
    return mk(h.xx * v.x + h.xy * v.y + h.xz * v.z, h.xy * v.x + h.yy * v.y + h.yz * v.z,
              h.xz * v.x + h.yz * v.y + h.zz * v.z);
}

// Solves H dx = b for a symmetric 3x3 block by adjugate / determinant.
// Stands in for CuMatrix::solve3x3_psd_stable (VBDPhysics.cpp:2449,
// VBDPhysicsCompute.cu:896), whose source is not available: failure iff the
// determinant is not finite or |det| <= 1e-12 |h_xx h_yy h_zz|. Returns false on
// failure, and then the caller takes a gradient step (VBDPhysics.cpp:2452-2459).
// XX_FIRST: the order in which the determinant's products fuse. Left to the compiler, which of two
// products it fuses with their sum differs between kernels and from build to build; each keeps the one it
// had: h_xx C00 rounded first in the cloth solve and in the tet solve of contact scenes, h_xy C01 in the
// plain tet solve.
template <bool XX_FIRST>
__device__ __forceinline__ bool solve_sym3(const Sym3& h, f3 b, f3& x) {
    const float C00 = h.yy * h.zz - h.yz * h.yz;
    const float C01 = h.yz * h.xz - h.xy * h.zz;
    const float C02 = h.xy * h.yz - h.yy * h.xz;
    const float C11 = h.xx * h.zz - h.xz * h.xz;
    const float C12 = h.xy * h.xz - h.xx * h.yz;
    const float C22 = h.xx * h.yy - h.xy * h.xy;
    const float det = fmaf(h.xz, C02, XX_FIRST ? fmaf(h.xy, C01, h.xx * C00) : fmaf(h.xx, C00, h.xy * C01));
    const float scale = fabsf(h.xx * h.yy * h.zz);
    if (!isfinite(det) || !(fabsf(det) > 1e-12f * scale)) return false;
    const float inv = 1.0f / det;
    x.x = (C00 * b.x + C01 * b.y + C02 * b.z) * inv;
    x.y = (C01 * b.x + C11 * b.y + C12 * b.z) * inv;
    x.z = (C02 * b.x + C12 * b.y + C22 * b.z) * inv;
    return isfinite(x.x) && isfinite(x.y) && isfinite(x.z);
}

// Force and Hessian parts of one incident tet (TetInc) on its vertex at x, the others at p0..p2:
// F m_v, g = cof(F) m_v, det F and |m_v|^2.
struct TetTerms {
    f3 Fm, g;
    float J, mm;
};
__device__ __forceinline__ TetTerms tet_terms(f3 x, f3 p0, f3 p1, f3 p2, float c, float w0, float w1, float w2) {
    const f3 d0 = p0 - x;
    TetTerms t;
    t.Fm = w0 * d0 + w1 * (p1 - x) + w2 * (p2 - x);
    t.g = c * cross(p1 - p0, p2 - p0);
    t.J = -dot(t.g, d0);
    t.mm = -(w0 + w1 + w2);
    return t;
}

// The same by the shape-matrix rows m0..m2 (TetRow).
__device__ __forceinline__ TetTerms tet_terms_rows(f3 x, f3 p0, f3 p1, f3 p2, f3 m0, f3 m1, f3 m2) {
    const f3 d0 = p0 - x, d1 = p1 - x, d2 = p2 - x;
    // F columns: F e_c = sum_k d_k m_k[c]
    const f3 c0 = m0.x * d0 + m1.x * d1 + m2.x * d2;
    const f3 c1 = m0.y * d0 + m1.y * d1 + m2.y * d2;
    const f3 c2 = m0.z * d0 + m1.z * d1 + m2.z * d2;
    const f3 mv = mk(-(m0.x + m1.x + m2.x), -(m0.y + m1.y + m2.y), -(m0.z + m1.z + m2.z));
    // cof(F) columns are c1 x c2, c2 x c0, c0 x c1
    const f3 k0 = cross(c1, c2);
    const f3 k1 = cross(c2, c0);
    const f3 k2 = cross(c0, c1);
    TetTerms t;
    t.J = dot(c0, k0);
    t.g = mv.x * k0 + mv.y * k1 + mv.z * k2;
    t.Fm = mv.x * c0 + mv.y * c1 + mv.z * c2;
    t.mm = dot(mv, mv);
    return t;
}

}  // namespace gvbd
