// spk_scene.hip -- leaf-ordered triangle records formed on the device.
//
// A scene's vertices, normals and ids go up as the caller holds them and one thread a triangle
// writes what the kernels read: 72 bytes (plus vertex normals where any triangle is smooth), in FP64
// as spica sets its triangles up (triangle.cc:17-52, 119-138), rounded to float at the end.  The
// arithmetic is the host's, operation by operation (no contraction; FP64 division and square root
// are correctly rounded on both), so the records are bit for bit those the host code formed; that
// code took 12 ms for 164,000 triangles, single-threaded, against 0.012 ms here.  Bound by the gather of
// vertices in leaf order and by FP64 divisions; the uploads around it cost more.
#include "spk_internal.h"

#pragma clang fp contract(off)

namespace spk {

namespace {

struct V3 {
    double x, y, z;
};
__device__ __forceinline__ V3 v3(double x, double y, double z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 vsub(V3 a, V3 b) { return v3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ double vdot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 vcross(V3 a, V3 b) {
    return v3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ V3 vnormalize(V3 a) {
    const double n = sqrt(vdot(a, a));
    return v3(a.x / n, a.y / n, a.z / n);
}
__device__ __forceinline__ float4 to_f4(V3 a, float w) { return make_float4((float)a.x, (float)a.y, (float)a.z, w); }

struct Frame {
    V3 p[3], n[3], ng;
    bool smooth;
};
__device__ __forceinline__ Frame frame_of(const float* __restrict__ v, const float* __restrict__ nrm) {
    Frame t;
    for (int i = 0; i < 3; i++) t.p[i] = v3(v[3 * i], v[3 * i + 1], v[3 * i + 2]);
    const V3 c = vcross(vsub(t.p[1], t.p[0]), vsub(t.p[2], t.p[0]));
    t.smooth = false;
    // a triangle whose three normals are all zero is flat (a flat mesh among smooth ones)
    bool zero = nrm != nullptr;
    for (int i = 0; nrm && i < 9; i++) zero = zero && nrm[i] == 0.0f;
    V3 fn;
    if (!nrm || zero) {
        fn = vnormalize(c);
        t.n[0] = t.n[1] = t.n[2] = fn;
    } else {
        for (int i = 0; i < 3; i++) t.n[i] = vnormalize(v3(nrm[3 * i], nrm[3 * i + 1], nrm[3 * i + 2]));
        fn = c;
        if (sqrt(vdot(fn, fn)) < 1e-12) {
            const double third = 1.0 / 3.0;
            fn = v3((t.n[0].x + t.n[1].x + t.n[2].x) * third, (t.n[0].y + t.n[1].y + t.n[2].y) * third,
                    (t.n[0].z + t.n[1].z + t.n[2].z) * third);
        }
        fn = vnormalize(fn);
        for (int i = 0; i < 3; i++)
            if (fabs(vdot(t.n[i], fn)) < 1.0 - 1e-12) t.smooth = true;
    }
    // the geometric normal through the tangent frame of vect_math.h:121-128
    const V3 du = fabs(fn.x) > fabs(fn.y) ? vnormalize(v3(-fn.z, 0.0, fn.x)) : vnormalize(v3(0.0, fn.z, -fn.y));
    const V3 dv = vnormalize(vcross(fn, du));
    t.ng = vnormalize(vcross(du, dv));
    return t;
}

__global__ __launch_bounds__(256) void k_tri_records(const float* __restrict__ verts, const float* __restrict__ normals,
                                                     const uint32_t* __restrict__ order, const int32_t* __restrict__ mat_ids,
                                                     const int32_t* __restrict__ light_ids, int64_t n,
                                                     float4* __restrict__ tris, float4* __restrict__ tri_ng,
                                                     int2* __restrict__ tri_ids, float4* __restrict__ tri_n) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const uint32_t prim = order[k];
    const float* v = verts + 9 * (size_t)prim;
    const Frame f = frame_of(v, normals ? normals + 9 * (size_t)prim : nullptr);
    tris[3 * k] = make_float4(v[0], v[1], v[2], __uint_as_float(prim));
    tris[3 * k + 1] = to_f4(vsub(f.p[1], f.p[0]), 0.0f);
    tris[3 * k + 2] = to_f4(vsub(f.p[2], f.p[0]), 0.0f);
    tri_ng[k] = to_f4(f.ng, __uint_as_float((uint32_t)mat_ids[prim] | (f.smooth ? 0x80000000u : 0u)));
    tri_ids[k] = make_int2((int)prim, light_ids ? light_ids[prim] : -1);
    if (tri_n)
        for (int j = 0; j < 3; j++) tri_n[3 * k + j] = to_f4(f.n[j], 0.0f);
}

}  // namespace

int launch_tri_records(const float* verts, const float* normals, const uint32_t* order, const int32_t* mat_ids,
                       const int32_t* light_ids, int64_t n, float4* tris, float4* tri_ng, int2* tri_ids, float4* tri_n) {
    if (n == 0) return SPK_OK;
    hipLaunchKernelGGL(k_tri_records, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, verts, normals, order, mat_ids,
                       light_ids, n, tris, tri_ng, tri_ids, tri_n);
    SPK_CHECK_HIP(hipGetLastError());
    return SPK_OK;
}

}  // namespace spk
