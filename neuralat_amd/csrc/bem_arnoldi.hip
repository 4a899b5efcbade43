// The Arnoldi step of the GMRES solvers after the product w = A v_j: classical
// Gram-Schmidt (one or two passes, FP64 sums), |w|^2, v_{j+1} = w / |w|, the
// previous Givens rotations on column j, the new one, and the convergence flag.
//
// One step is microseconds of work, so what it costs is launches and the
// dependent trips to L2 inside them.  Two forms replace a kernel per operation
// (nine launches on one system, seven on a batch, 46 us of kernels at 20480
// unknowns and 35 basis vectors):
//  * arnoldi_lds_kernel: one workgroup per system, the whole basis of the step
//    in LDS, read from memory once (the four Gram-Schmidt sweeps over it ran
//    from L2 before, 17.8 us at 642 unknowns);
//  * four chunked kernels (dots; update + dots; update + norm + rotations;
//    normalise + new rotation): a workgroup owns kChunk elements of one system,
//    and every workgroup sums the partial dot products it needs by itself.
// Beyond both (long bases: the partial sums outgrow the vectors) the solvers'
// separate kernels remain, which split each basis vector over the chip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bem_device.hpp"
#include "bem_linalg.hpp"

namespace bem {

namespace {

constexpr int kChunk = 512;          // elements, and threads, of a chunked workgroup
constexpr int kChunkWaves = kChunk / 64;
constexpr int kChunkMaxQ = 1024;     // basis vectors (their coefficients sit in LDS)
constexpr int kChunkMaxPart = 4096;  // partial sums per system: 64 KB each workgroup reads
constexpr int kLdsThreads = 1024;
constexpr size_t kLdsBytes = 128 << 10;  // of a CU's 160 KB
// one workgroup takes 15 us a step at 3380 unknowns, 25 at 5120, 40 at 8000; the chunked form 24 to 28
constexpr int64_t kLdsMaxN = 5120;

// system s: its length and where its vectors start
struct SysView {
    int64_t n, off;
};
__device__ __forceinline__ SysView sys_view(const ArnoldiDesc& D, int s)
{
    if (D.sys) return {D.sys[s].n, D.sys[s].off};
    return {D.n, (int64_t)s * D.sstride};
}

// the new rotation (c, s) from column entries a = H[j][j] (rotated) and
// |w| = H[j+1][j], applied to g; res = |g_{j+1}|
__device__ __forceinline__ void finish_column(const ArnoldiDesc& D, int s, int j, double2 a, double nrm2)
{
    double2* col = D.H + (int64_t)s * (D.m + 1) * D.m + (int64_t)j * (D.m + 1);
    double2* gg = D.g + (int64_t)s * (D.m + 1);
    const double b = sqrt(nrm2);
    const double den = sqrt(a.x * a.x + a.y * a.y + b * b);
    double2 c = make_double2(1.0, 0.0);
    double sv = 0.0;
    if (den > 0.0) {
        c = make_double2(a.x / den, -a.y / den);
        sv = b / den;
    }
    D.cs[(int64_t)s * D.m + j] = c;
    D.sn[(int64_t)s * D.m + j] = make_double2(sv, 0.0);
    col[j] = make_double2(den, 0.0);
    col[j + 1] = make_double2(0.0, 0.0);
    const double2 gj = gg[j];
    const double2 gn = make_double2(-(sv * gj.x), -(sv * gj.y));
    gg[j + 1] = gn;
    gg[j] = make_double2(c.x * gj.x - c.y * gj.y, c.x * gj.y + c.y * gj.x);
    const double rj = sqrt(gn.x * gn.x + gn.y * gn.y);
    D.res[s] = rj;
    D.wn2[s] = nrm2;
    if (D.nk) D.nk[s] = j + 1;
    if (D.done && rj <= D.target[s]) D.done[s] = 1;
}

// rotations 0 .. j - 1 applied to the column (hh[0 .. j], cs, sn in LDS);
// returns the entry that enters the new rotation
__device__ __forceinline__ double2 rotate_column(double2* __restrict__ col, int j, const double2* hh,
                                                 const double2* cs, const double2* sn)
{
    double2 carry = hh[0];
    for (int q = 0; q < j; ++q) {
        const double2 c = cs[q], sv = sn[q], a = carry, b = hh[q + 1];
        col[q] = make_double2(c.x * a.x - c.y * a.y + sv.x * b.x - sv.y * b.y,
                              c.x * a.y + c.y * a.x + sv.x * b.y + sv.y * b.x);
        carry = make_double2(-(sv.x * a.x + sv.y * a.y) + (c.x * b.x + c.y * b.y),
                             -(sv.x * a.y - sv.y * a.x) + (c.x * b.y - c.y * b.x));
    }
    return carry;
}

// ---- one workgroup per system, the basis in LDS ------------------------------
size_t lds_bytes(int64_t n, int j) { return (size_t)(j + 2) * (size_t)n * sizeof(float2) + (size_t)(j + 1) * 64 + 256; }

__global__ __launch_bounds__(kLdsThreads) void arnoldi_lds_kernel(const ArnoldiDesc D, int j, int passes)
{
    extern __shared__ double2 lds[];
    constexpr int nw = kLdsThreads / 64;
    const int s = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (D.done && D.done[s]) return;  // uniform over the workgroup
    const SysView S = sys_view(D, s);
    const int n = (int)S.n, nq = j + 1;
    double2* hh = lds;             // both passes' coefficients, summed
    double2* hp = hh + nq;         // this pass's
    double2* scs = hp + nq;        // previous rotations
    double2* ssn = scs + nq;
    double* red = (double*)(ssn + nq);  // nw + 1 used (256 bytes)
    float2* wl = (float2*)(red + 32);
    float2* Vl = wl + n;
    const float2* Vs = D.V + S.off;
    float2* ws = D.w + S.off;
    for (int q = t; q < j; q += kLdsThreads) {
        scs[q] = D.cs[(int64_t)s * D.m + q];
        ssn[q] = D.sn[(int64_t)s * D.m + q];
    }
    for (int e = t; e < n; e += kLdsThreads) wl[e] = ws[e];
    // wavefront q, q + 16, ... copies basis vector q: eight loads in flight
    for (int q = wave; q < nq; q += nw) {
        const float2* vq = Vs + (int64_t)q * D.qstride;
        for (int e0 = lane; e0 < n; e0 += 64 * 8) {
            float2 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = vq[min(e0 + 64 * u, n - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (e0 + 64 * u < n) Vl[q * n + e0 + 64 * u] = v[u];
        }
    }
    __syncthreads();
    for (int pass = 0; pass < passes; ++pass) {
        for (int q = wave; q < nq; q += nw) {
            double sr = 0.0, si = 0.0;
            for (int e = lane; e < n; e += 64) {
                const float2 a = Vl[q * n + e], b = wl[e];
                sr += (double)a.x * b.x + (double)a.y * b.y;
                si += (double)a.x * b.y - (double)a.y * b.x;
            }
            sr = wave_sum64(sr);
            si = wave_sum64(si);
            if (lane == 0) {
                hp[q] = make_double2(sr, si);
                hh[q] = pass ? make_double2(hh[q].x + sr, hh[q].y + si) : make_double2(sr, si);
            }
        }
        __syncthreads();
        for (int e = t; e < n; e += kLdsThreads) {
            double ar = 0.0, ai = 0.0;
#pragma unroll 4
            for (int q = 0; q < nq; ++q) {
                const double2 c = hp[q];
                const float2 v = Vl[q * n + e];
                ar += c.x * v.x - c.y * v.y;
                ai += c.x * v.y + c.y * v.x;
            }
            const float2 wo = wl[e];
            wl[e] = make_float2((float)((double)wo.x - ar), (float)((double)wo.y - ai));
        }
        __syncthreads();
    }
    // the last wavefront rotates the column while the others form the norm
    double2 carry = make_double2(0.0, 0.0);
    if (wave == nw - 1) {
        if (lane == 0) {
            carry = rotate_column(D.H + (int64_t)s * (D.m + 1) * D.m + (int64_t)j * (D.m + 1), j, hh, scs, ssn);
            hp[0] = carry;
        }
    } else {
        double a2 = 0.0;
        for (int e = t; e < n; e += kLdsThreads - 64) {
            const float2 v = wl[e];
            a2 += (double)v.x * v.x + (double)v.y * v.y;
        }
        a2 = wave_sum64(a2);
        if (lane == 0) red[wave] = a2;
    }
    __syncthreads();
    double nrm2 = 0.0;
    for (int q = 0; q < nw - 1; ++q) nrm2 += red[q];
    const float inv = nrm2 > 0.0 ? (float)(1.0 / sqrt(nrm2)) : 0.f;
    float2* vn = D.V + S.off + (int64_t)(j + 1) * D.qstride;
    for (int e = t; e < n; e += kLdsThreads) {
        const float2 v = wl[e];
        vn[e] = make_float2(v.x * inv, v.y * inv);
    }
    if (t == kLdsThreads - 64) finish_column(D, s, j, hp[0], nrm2);
}

// ---- chunked form -----------------------------------------------------------
// partial sums of system s, basis vector q, chunk c
__device__ __forceinline__ double2* part_of(double2* part, const ArnoldiDesc& D, int s, int q)
{
    return part + ((int64_t)s * D.qcap + q) * D.nch;
}

// <V_q, w> over this chunk for every q, w as eight values per lane
__device__ __forceinline__ void chunk_dots(const ArnoldiDesc& D, const SysView& S, int s, int c, int nq,
                                           const float2 (&w8)[8], double2* __restrict__ part)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t e0 = (int64_t)c * kChunk + lane;
    for (int q = wave; q < nq; q += kChunkWaves) {
        const float2* vq = D.V + S.off + (int64_t)q * D.qstride;
        float2 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = vq[min(e0 + 64 * u, S.n - 1)];
        double sr = 0.0, si = 0.0;
#pragma unroll
        for (int u = 0; u < 8; ++u) {  // w8 is zero past the end
            sr += (double)v[u].x * w8[u].x + (double)v[u].y * w8[u].y;
            si += (double)v[u].x * w8[u].y - (double)v[u].y * w8[u].x;
        }
        sr = wave_sum64(sr);
        si = wave_sum64(si);
        if (lane == 0) part_of(part, D, s, q)[c] = make_double2(sr, si);
    }
}

// hh[q] = sum of the chunks' partials, in a fixed order
__device__ __forceinline__ void chunk_sum(const ArnoldiDesc& D, int s, int nch, int nq, double2* part, double2* hh)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int q = wave; q < nq; q += kChunkWaves) {
        const double2* p = part_of(part, D, s, q);
        double sr = 0.0, si = 0.0;
        for (int c = lane; c < nch; c += 64) {
            sr += p[c].x;
            si += p[c].y;
        }
        sr = wave_sum64(sr);
        si = wave_sum64(si);
        if (lane == 0) hh[q] = make_double2(sr, si);
    }
    __syncthreads();
}

// w_e - sum_q hh[q] V_q[e] for this thread's element
__device__ __forceinline__ float2 chunk_update(const ArnoldiDesc& D, const SysView& S, int64_t e, int nq,
                                               const double2* hh, float2 wo)
{
    const float2* Ve = D.V + S.off + min(e, S.n - 1);
    double ar = 0.0, ai = 0.0;
    for (int q0 = 0; q0 < nq; q0 += 8) {
        float2 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = Ve[(int64_t)min(q0 + u, nq - 1) * D.qstride];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (q0 + u < nq) {
                const double2 c = hh[q0 + u];
                ar += c.x * v[u].x - c.y * v[u].y;
                ai += c.x * v[u].y + c.y * v[u].x;
            }
    }
    return make_float2((float)((double)wo.x - ar), (float)((double)wo.y - ai));
}

__global__ __launch_bounds__(kChunk) void arnoldi_dots_kernel(const ArnoldiDesc D, int j)
{
    const int s = blockIdx.y, c = blockIdx.x;
    if (D.done && D.done[s]) return;
    const SysView S = sys_view(D, s);
    const int64_t e0 = (int64_t)c * kChunk + (threadIdx.x & 63);
    if ((int64_t)c * kChunk >= S.n) return;  // uniform: this system is shorter
    float2 w8[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w8[u] = e0 + 64 * u < S.n ? D.w[S.off + e0 + 64 * u] : make_float2(0.f, 0.f);
    chunk_dots(D, S, s, c, j + 1, w8, D.part);
}

// first update, then the second pass's dots
__global__ __launch_bounds__(kChunk) void arnoldi_update_dots_kernel(const ArnoldiDesc D, int j)
{
    __shared__ double2 hh[kChunkMaxQ];
    __shared__ float2 wl[kChunk];
    const int s = blockIdx.y, c = blockIdx.x, nq = j + 1;
    if (D.done && D.done[s]) return;
    const SysView S = sys_view(D, s);
    if ((int64_t)c * kChunk >= S.n) return;  // uniform
    const int64_t e = (int64_t)c * kChunk + threadIdx.x;
    const float2 wo = e < S.n ? D.w[S.off + e] : make_float2(0.f, 0.f);
    chunk_sum(D, s, (int)((S.n + kChunk - 1) / kChunk), nq, D.part, hh);
    if (c == 0)
        for (int q = threadIdx.x; q < nq; q += kChunk) D.h[(int64_t)s * D.hs + q] = hh[q];
    const float2 wn = chunk_update(D, S, e, nq, hh, wo);
    wl[threadIdx.x] = e < S.n ? wn : make_float2(0.f, 0.f);
    if (e < S.n) D.w[S.off + e] = wn;
    __syncthreads();
    float2 w8[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w8[u] = wl[(threadIdx.x & 63) + 64 * u];
    chunk_dots(D, S, s, c, nq, w8, D.part2);
}

// last update and the chunk's |w|^2; the workgroup past the chunks applies the
// previous rotations to the column (it needs no norm) and leaves the entry that
// enters the new rotation in h[0]
__global__ __launch_bounds__(kChunk) void arnoldi_update_norm_kernel(const ArnoldiDesc D, int j, int passes)
{
    __shared__ double2 hh[kChunkMaxQ];
    __shared__ double red[kChunkWaves];
    __shared__ double2 scs[kChunk], ssn[kChunk];
    const int s = blockIdx.y, c = blockIdx.x, nq = j + 1, t = threadIdx.x;
    if (D.done && D.done[s]) return;
    const SysView S = sys_view(D, s);
    const bool rotate = c == (int)gridDim.x - 1;
    if (!rotate && (int64_t)c * kChunk >= S.n) return;  // uniform
    const int64_t e = (int64_t)c * kChunk + t;
    const float2 wo = !rotate && e < S.n ? D.w[S.off + e] : make_float2(0.f, 0.f);
    chunk_sum(D, s, (int)((S.n + kChunk - 1) / kChunk), nq, passes == 2 ? D.part2 : D.part, hh);
    if (rotate) {
        double2* hs = D.h + (int64_t)s * D.hs;
        if (passes == 2) {
            for (int q = t; q < nq; q += kChunk) hh[q] = make_double2(hh[q].x + hs[q].x, hh[q].y + hs[q].y);
            __syncthreads();
        }
        double2* col = D.H + (int64_t)s * (D.m + 1) * D.m + (int64_t)j * (D.m + 1);
        double2 carry = hh[0];
        for (int q0 = 0; q0 < j; q0 += kChunk) {
            const int cnt = min(kChunk, j - q0);
            if (t < cnt) {
                scs[t] = D.cs[(int64_t)s * D.m + q0 + t];
                ssn[t] = D.sn[(int64_t)s * D.m + q0 + t];
            }
            __syncthreads();
            if (t == 0) {
                hh[q0] = carry;
                carry = rotate_column(col + q0, cnt, hh + q0, scs, ssn);
            }
            __syncthreads();
        }
        if (t == 0) hs[0] = carry;
        return;
    }
    const float2 wn = chunk_update(D, S, e, nq, hh, wo);
    double a2 = 0.0;
    if (e < S.n) {
        D.w[S.off + e] = wn;
        a2 = (double)wn.x * wn.x + (double)wn.y * wn.y;
    }
    a2 = wave_sum64(a2);
    if ((t & 63) == 0) red[t >> 6] = a2;
    __syncthreads();
    if (t == 0) {
        double sum = 0.0;
        for (int q = 0; q < kChunkWaves; ++q) sum += red[q];
        D.partn[(int64_t)s * D.nch + c] = sum;
    }
}

__global__ __launch_bounds__(kChunk) void arnoldi_finish_kernel(const ArnoldiDesc D, int j)
{
    const int s = blockIdx.y, c = blockIdx.x, lane = threadIdx.x & 63;
    // the first workgroup may raise done[s] while others start: a finished
    // system's v_{j+1} is not used, so their skipping it is harmless
    if (D.done && D.done[s]) return;
    const SysView S = sys_view(D, s);
    if ((int64_t)c * kChunk >= S.n) return;  // uniform
    const int nch = (int)((S.n + kChunk - 1) / kChunk);
    double nrm2 = 0.0;
    for (int q = lane; q < nch; q += 64) nrm2 += D.partn[(int64_t)s * D.nch + q];
    nrm2 = wave_sum64(nrm2);
    const int64_t e = (int64_t)c * kChunk + threadIdx.x;
    if (e < S.n) {
        const float inv = nrm2 > 0.0 ? (float)(1.0 / sqrt(nrm2)) : 0.f;
        const float2 v = D.w[S.off + e];
        D.V[S.off + (int64_t)(j + 1) * D.qstride + e] = make_float2(v.x * inv, v.y * inv);
    }
    if (c == 0 && threadIdx.x == 0) finish_column(D, s, j, D.h[(int64_t)s * D.hs], nrm2);
}

}  // namespace

int arnoldi_chunks(int64_t n) { return (int)std::max<int64_t>(1, (n + kChunk - 1) / kChunk); }

int arnoldi_qcap(int64_t n, int m)
{
    return (int)std::min<int64_t>({(int64_t)m + 1, (int64_t)kChunkMaxQ, (int64_t)kChunkMaxPart / arnoldi_chunks(n)});
}

int64_t arnoldi_part_elems(int64_t n, int m, int ns)
{
    return 2 * (int64_t)ns * arnoldi_chunks(n) * arnoldi_qcap(n, m);
}

void arnoldi_set_part(ArnoldiDesc& D, double2* part, double* partn)
{
    D.nch = arnoldi_chunks(D.n);
    D.qcap = arnoldi_qcap(D.n, D.m);
    D.part = part;
    D.part2 = part + (int64_t)D.ns * D.qcap * D.nch;
    D.partn = partn;
}

bool arnoldi_fused(const ArnoldiDesc& D, int j)
{
    return (D.n <= kLdsMaxN && lds_bytes(D.n, j) <= kLdsBytes) || j < D.qcap;
}

hipError_t launch_arnoldi_step(const ArnoldiDesc& D, int j, int passes, hipStream_t s)
{
    const size_t lb = lds_bytes(D.n, j);
    if (D.n <= kLdsMaxN && lb <= kLdsBytes) {
        if (lb > (64 << 10)) {  // more than the default limit of dynamic LDS
            const hipError_t e = hipFuncSetAttribute((const void*)arnoldi_lds_kernel,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(arnoldi_lds_kernel, dim3((unsigned)D.ns), dim3(kLdsThreads), lb, s, D, j, passes);
        return hipGetLastError();
    }
    const dim3 g((unsigned)D.nch, (unsigned)D.ns);
    hipLaunchKernelGGL(arnoldi_dots_kernel, g, dim3(kChunk), 0, s, D, j);
    if (passes == 2) hipLaunchKernelGGL(arnoldi_update_dots_kernel, g, dim3(kChunk), 0, s, D, j);
    hipLaunchKernelGGL(arnoldi_update_norm_kernel, dim3(g.x + 1, g.y), dim3(kChunk), 0, s, D, j, passes);
    hipLaunchKernelGGL(arnoldi_finish_kernel, g, dim3(kChunk), 0, s, D, j);
    return hipGetLastError();
}

}  // namespace bem
