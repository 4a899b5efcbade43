// Exterior pressure p = D phi - S psi at points (solver.py:140-147) without
// forming the potential operators: the boundary data are contracted inside
// the evaluation.
//
// Both potentials share the point difference, r and e^{ikr}: per (point,
// quadrature point) G (-(1 - ikr) (y - x).n / r^2 phi(y) - psi(y)) w, about 23
// vector instructions and three transcendentals, nothing stored but the
// pressures.  Bound by vector issue.  Forming the two [np, n] operators first
// (P1: three corner values per pair to scratch, a gather, two products) moved
// 40 bytes per pair four times: 8192 points x 5120 triangles took 1976 us (now 197), of
// which 1500 us the gather.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bem_device.hpp"
#include "bem_internal.hpp"

namespace bem {

namespace {

constexpr int kFieldQ = 6;                          // the potentials' triangle rule
constexpr int kFieldRec = Rec<kFieldQ>::kFloats;
constexpr int kFieldWaves = 4;                      // wavefronts of a workgroup: same points, different triangles
constexpr int kFieldGroup = 16;                     // triangles summed in FP32 before an FP64 addition

// pre[z][6 t + b] = (w phi, w psi)(y_b) / 4 pi: the boundary data of system z
// at every quadrature point, the weight folded in, so the sweep reads them as
// wave-uniform values (interpolated inside the sweep they cost 72 vector
// instructions per triangle next to its ~210)
__global__ __launch_bounds__(256) void field_data_kernel(const float* __restrict__ rec6, int64_t gstride,
                                                         const int4* __restrict__ tris, int64_t nt, int p1, int64_t n,
                                                         const float2* __restrict__ phi, const float2* __restrict__ psi,
                                                         float4* __restrict__ pre)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= nt * kFieldQ) return;
    const int z = blockIdx.y;
    const int64_t t = e / kFieldQ;
    const int b = (int)(e - t * kFieldQ);
    phi += (int64_t)z * n;
    psi += (int64_t)z * n;
    const float w = rec6[(int64_t)z * gstride + t * kFieldRec + 3 * kFieldQ + b] * kInv4Pi;
    float2 f, g;
    if (p1) {
        const int4 v = tris[t];
        const float2 f0 = phi[v.x], f1 = phi[v.y], f2 = phi[v.z];
        const float2 g0 = psi[v.x], g1 = psi[v.y], g2 = psi[v.z];
        float b1 = TriRule<kFieldQ>::x1[0], b2 = TriRule<kFieldQ>::x2[0];
#pragma unroll
        for (int q = 1; q < kFieldQ; ++q)
            if (b == q) {
                b1 = TriRule<kFieldQ>::x1[q];
                b2 = TriRule<kFieldQ>::x2[q];
            }
        const float b0 = 1.0f - b1 - b2;
        f = make_float2(b0 * f0.x + b1 * f1.x + b2 * f2.x, b0 * f0.y + b1 * f1.y + b2 * f2.y);
        g = make_float2(b0 * g0.x + b1 * g1.x + b2 * g2.x, b0 * g0.y + b1 * g1.y + b2 * g2.y);
    } else {
        f = phi[t];
        g = psi[t];
    }
    pre[(int64_t)z * nt * kFieldQ + e] = make_float4(w * f.x, w * f.y, w * g.x, w * g.y);
}

// Lane = point, triangles wave-uniform (their records and boundary data are
// scalar operands).  A workgroup owns 64 points and 4 tper triangles; its
// wavefronts meet in LDS.  grid (point tiles, triangle splits, systems).
// Sums: FP32 over kFieldGroup triangles, FP64 beyond, in a fixed order.
template <bool CLAMP>
__global__ __launch_bounds__(64 * kFieldWaves) void field_kernel(const float* __restrict__ rec6, int64_t nt,
                                                                 const float* __restrict__ pts, int64_t np,
                                                                 const KBatch kb, const float4* __restrict__ pre,
                                                                 int64_t tper, double2* __restrict__ part,
                                                                 float2* __restrict__ out)
{
    __shared__ double2 red[kFieldWaves][64];
    const int z = blockIdx.z;
    const float k = kb.k[z], krev = k * kInv2Pi;
    rec6 += (int64_t)z * kb.gstride;
    pts += (int64_t)z * kb.pstride;
    pre += (int64_t)z * nt * kFieldQ;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t p = (int64_t)blockIdx.x * 64 + lane;
    const int64_t pc = p < np ? p : np - 1;
    const float x0 = pts[3 * pc], x1 = pts[3 * pc + 1], x2 = pts[3 * pc + 2];
    const int64_t t0 = min(nt, ((int64_t)blockIdx.y * kFieldWaves + wave) * tper), t1 = min(nt, t0 + tper);
    double accr = 0.0, acci = 0.0;
    for (int64_t g0 = t0; g0 < t1; g0 += kFieldGroup) {
        const int64_t g1 = min(t1, g0 + kFieldGroup);
        float sr = 0.f, si = 0.f;
        for (int64_t t = g0; t < g1; ++t) {
            const float* rr = rec6 + t * kFieldRec;
            const float4* f = pre + t * kFieldQ;
            // (x - y).n is the same at every point y of the triangle
            const float dn = (x0 - rr[0]) * rr[4 * kFieldQ] + (x1 - rr[1]) * rr[4 * kFieldQ + 1] +
                             (x2 - rr[2]) * rr[4 * kFieldQ + 2];
#pragma unroll
            for (int b = 0; b < kFieldQ; ++b) {
                const float dx = rr[3 * b] - x0, dy = rr[3 * b + 1] - x1, dz = rr[3 * b + 2] - x2;
                float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                if (CLAMP) r2 = fmaxf(r2, kEps2);
                const float rinv = __builtin_amdgcn_rsqf(r2);
                const float r = r2 * rinv;
                float sn, cs;
                sincos_rev(r * krev, sn, cs);
                const float th = r * k, q = dn * rinv * rinv;
                // q (1 - ikr) phi - psi
                const float er = fmaf(q, fmaf(th, f[b].y, f[b].x), -f[b].z);
                const float ei = fmaf(q, fmaf(-th, f[b].x, f[b].y), -f[b].w);
                const float gr = cs * rinv, gi = sn * rinv;
                sr = fmaf(gr, er, fmaf(-gi, ei, sr));
                si = fmaf(gr, ei, fmaf(gi, er, si));
            }
        }
        accr += (double)sr;
        acci += (double)si;
    }
    red[wave][lane] = make_double2(accr, acci);
    __syncthreads();
    if (wave != 0 || p >= np) return;
    for (int w = 1; w < kFieldWaves; ++w) {
        accr += red[w][lane].x;
        acci += red[w][lane].y;
    }
    if (part)
        part[((int64_t)z * gridDim.y + blockIdx.y) * np + p] = make_double2(accr, acci);
    else
        out[(int64_t)z * np + p] = make_float2((float)accr, (float)acci);
}

// out[z][p] = sum over the triangle splits: a workgroup takes 16 points, 16
// threads each every 16th split, combined in order
__global__ __launch_bounds__(256) void field_reduce_kernel(const double2* __restrict__ part, int ns, int64_t np,
                                                           float2* __restrict__ out)
{
    __shared__ double2 red[16][16];
    const int q = threadIdx.x & 15, sl = threadIdx.x >> 4;
    const int64_t p = (int64_t)blockIdx.x * 16 + q;
    part += (int64_t)blockIdx.y * ns * np;
    double sr = 0.0, si = 0.0;
    if (p < np)
        for (int s = sl; s < ns; s += 16) {
            const double2 v = part[(int64_t)s * np + p];
            sr += v.x;
            si += v.y;
        }
    red[sl][q] = make_double2(sr, si);
    __syncthreads();
    if (sl != 0 || p >= np) return;
    for (int s = 1; s < 16; ++s) {
        sr += red[s][q].x;
        si += red[s][q].y;
    }
    out[(int64_t)blockIdx.y * np + p] = make_float2((float)sr, (float)si);
}

// Triangles per wavefront and splits of a sweep: about kFieldFill workgroups
// (four wavefronts each, two per SIMD) however few points or triangles there
// are, at least kFieldMinTris triangles per wavefront
constexpr int64_t kFieldFill = 2048, kFieldMinTris = 4, kFieldMaxSplits = 4096;

struct FieldSplit {
    int64_t tper;
    int ns;
};
FieldSplit field_split(int64_t nt, int64_t np, int nz)
{
    const int64_t tiles = std::max<int64_t>(1, (np + 63) / 64 * nz);
    const int64_t want = std::clamp<int64_t>((kFieldFill + tiles - 1) / tiles, 1, kFieldMaxSplits);
    const int64_t tper = std::max(kFieldMinTris, (nt + want * kFieldWaves - 1) / (want * kFieldWaves));
    return {tper, (int)((nt + tper * kFieldWaves - 1) / (tper * kFieldWaves))};
}

size_t field_pre_bytes(int64_t nt, int nz) { return sizeof(float4) * (size_t)nt * kFieldQ * (size_t)nz; }

}  // namespace

int64_t field_work_bytes(int64_t nt, int64_t np, int nz)
{
    if (np <= 0) return 0;
    nz = std::min(nz, kMaxBatchK);
    // a last, smaller launch of a batch may split finer: sized for every count
    size_t part = 0;
    for (int z = 1; z <= nz; ++z) {
        const int ns = field_split(nt, np, z).ns;
        if (ns > 1) part = std::max(part, sizeof(double2) * (size_t)ns * (size_t)np * (size_t)z);
    }
    return (int64_t)(field_pre_bytes(nt, nz) + part);
}

hipError_t launch_field(const MeshDev& mg, int64_t gstride, const float* pts, int64_t np, int64_t pstride,
                        const float* ks, int nk, int basis, int clamp, const float2* psi, const float2* phi,
                        float2* out, void* work, hipStream_t s)
{
    if (np <= 0) return hipSuccess;
    const int64_t n = basis == DP0 ? mg.nt : mg.nv, nt = mg.nt;
    for (int z0 = 0; z0 < nk; z0 += kMaxBatchK) {
        const int nz = std::min(kMaxBatchK, nk - z0);
        KBatch kb{};
        for (int z = 0; z < nz; ++z) kb.k[z] = ks[z0 + z];
        kb.gstride = gstride;
        kb.pstride = pstride;
        const float* rec = mg.rec6 + (int64_t)z0 * gstride;
        const float* pz = pts + (int64_t)z0 * pstride;
        float4* pre = (float4*)work;
        const FieldSplit sp = field_split(nt, np, nz);
        double2* part = sp.ns > 1 ? (double2*)((char*)work + field_pre_bytes(nt, nz)) : nullptr;
        float2* oz = out + (int64_t)z0 * np;
        hipLaunchKernelGGL(field_data_kernel, dim3((unsigned)((nt * kFieldQ + 255) / 256), (unsigned)nz), dim3(256), 0,
                           s, rec, gstride, mg.tris, nt, basis == P1 ? 1 : 0, n, phi + (int64_t)z0 * n,
                           psi + (int64_t)z0 * n, pre);
        const dim3 grid((unsigned)((np + 63) / 64), (unsigned)sp.ns, (unsigned)nz);
        if (clamp)
            hipLaunchKernelGGL(field_kernel<true>, grid, dim3(64 * kFieldWaves), 0, s, rec, nt, pz, np, kb,
                               (const float4*)pre, sp.tper, part, oz);
        else
            hipLaunchKernelGGL(field_kernel<false>, grid, dim3(64 * kFieldWaves), 0, s, rec, nt, pz, np, kb,
                               (const float4*)pre, sp.tper, part, oz);
        if (part)
            hipLaunchKernelGGL(field_reduce_kernel, dim3((unsigned)((np + 15) / 16), (unsigned)nz), dim3(256), 0, s,
                               (const double2*)part, sp.ns, np, oz);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace bem
