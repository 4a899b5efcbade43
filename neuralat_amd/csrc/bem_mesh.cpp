// Mesh set-up: validation, neighbour pairs, vertex->triangle lists and the P1
// tiling on the host; the position-dependent arrays (quadrature records,
// surface curls, singular-pair geometry) by a kernel from the vertex positions.
//
// The reference recomputes normals and curls in torch (solver.py:40-58) and
// finds neighbour pairs with an O(N) scan per triangle inside the singular
// kernel (bind.cu:90-97); here they are built once per mesh in O(N log N).
// The lists are made by counting and stamping (sorting the pairs by kind and
// searching the tiles' vertex lists took most of 4.4 ms at 5120 triangles),
// and what is uploaded goes through one pinned buffer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "bem_device.hpp"
#include "bem_internal.hpp"

namespace bem {

namespace {

struct V3 {
    double x, y, z;
};
// no fused multiply-adds: host and device round alike
#pragma clang fp contract(off)
__host__ __device__ inline V3 sub(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__host__ __device__ inline V3 add(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__host__ __device__ inline V3 mul(double s, V3 a) { return {s * a.x, s * a.y, s * a.z}; }
__host__ __device__ inline double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__host__ __device__ inline V3 cross(V3 a, V3 b)
{
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

uint32_t spread10(uint32_t v)
{
    v &= 0x3ff;
    v = (v | (v << 16)) & 0x030000FF;
    v = (v | (v << 8)) & 0x0300F00F;
    v = (v | (v << 4)) & 0x030C30C3;
    v = (v | (v << 2)) & 0x09249249;
    return v;
}

struct Tiling {
    std::vector<int32_t> ptr, vptr, verts;
    std::vector<int32_t> slot;  // 4 per position
};

// Greedy tiling of the ordered triangle list: a tile closes when it holds
// max_tris triangles, one more would exceed max_verts distinct vertices, or
// the next position is in stops (sorted; tiles never cross one).
Tiling make_tiling(const std::vector<int32_t>& perm, const int32_t* tris, int64_t nv, int max_tris, int max_verts,
                   const std::vector<int32_t>& stops = {})
{
    Tiling T;
    const int64_t nt = (int64_t)perm.size();
    T.slot.assign((size_t)nt * 4, 0);
    T.ptr.push_back(0);
    T.vptr.push_back(0);
    T.verts.reserve((size_t)nt * 2);
    int64_t pos = 0;
    std::vector<int32_t> local;
    // tile (plus 1) a vertex was last seen in, and its slot there
    std::vector<int32_t> seen((size_t)nv, 0), slot((size_t)nv, 0);
    int32_t tile = 0;
    size_t next_stop = 0;
    while (pos < nt) {
        ++tile;
        local.clear();
        int64_t start = pos;
        while (next_stop < stops.size() && stops[next_stop] <= start) ++next_stop;
        const int64_t limit = next_stop < stops.size() ? std::min<int64_t>(nt, stops[next_stop]) : nt;
        while (pos < limit && pos - start < max_tris) {
            const int32_t* t = tris + 3 * (int64_t)perm[pos];
            const int fresh = (seen[t[0]] != tile) + (seen[t[1]] != tile) + (seen[t[2]] != tile);
            if ((int)local.size() + fresh > max_verts) break;
            for (int a = 0; a < 3; ++a)
                if (seen[t[a]] != tile) {
                    seen[t[a]] = tile;
                    local.push_back(t[a]);
                }
            ++pos;
        }
        std::sort(local.begin(), local.end());
        for (size_t q = 0; q < local.size(); ++q) slot[local[q]] = (int32_t)q;
        for (int64_t p = start; p < pos; ++p) {
            const int32_t* t = tris + 3 * (int64_t)perm[p];
            for (int a = 0; a < 3; ++a) T.slot[4 * p + a] = slot[t[a]];
        }
        T.verts.insert(T.verts.end(), local.begin(), local.end());
        T.ptr.push_back((int32_t)pos);
        T.vptr.push_back((int32_t)T.verts.size());
    }
    return T;
}

// Pinned host staging for uploads (a DMA copy instead of a staged pageable
// one: 1 MB takes 27 us against 140 to 315).  One process-wide buffer, grown
// on demand up to kPinnedStageMax and kept until the process ends.  Its user
// holds it until the copy is done, which may be behind other work on its
// stream, so nobody waits for it: while it is taken, and for larger uploads,
// pageable memory is the stage.
constexpr size_t kPinnedStageMax = (size_t)64 << 20;
std::mutex g_stage_mu;
char* g_stage = nullptr;
size_t g_stage_cap = 0;

class Stage {
public:
    char* get(size_t bytes)
    {
        if (bytes <= kPinnedStageMax) {
            lk_ = std::unique_lock<std::mutex>(g_stage_mu, std::try_to_lock);
            if (lk_.owns_lock() && g_stage_cap < bytes) {
                if (g_stage) (void)hipHostFree(g_stage);
                g_stage = nullptr;
                g_stage_cap = 0;
                const size_t want = std::min(kPinnedStageMax, (bytes + ((size_t)1 << 20) - 1) >> 20 << 20);
                if (hipHostMalloc((void**)&g_stage, want, hipHostMallocDefault) == hipSuccess) {
                    g_stage_cap = want;
                } else {
                    (void)hipGetLastError();
                    g_stage = nullptr;
                }
            }
            if (lk_.owns_lock()) {
                if (g_stage) return g_stage;
                lk_.unlock();
            }
        }
        pageable_.resize(bytes);
        return pageable_.data();
    }

private:
    std::unique_lock<std::mutex> lk_;
    std::vector<char> pageable_;
};

}  // namespace

// A fault of one sample's positions: kind 0 = a non-finite coordinate, 1 = a
// triangle of zero area; the first (kind, triangle) is kept as the smallest key.
constexpr unsigned long long kGeomOk = ~0ull;
static __host__ __device__ inline unsigned long long geom_key(int kind, int64_t t)
{
    return ((unsigned long long)kind << 32) | (unsigned long long)t;
}
static std::string geom_fault(unsigned long long key)
{
    return (key >> 32) == 0 ? "non-finite vertex coordinate"
                            : "triangle " + std::to_string((int64_t)(key & 0xffffffffu)) + " has zero area";
}

__device__ __forceinline__ void load_triangle(const float* __restrict__ verts, int4 tr, V3 (&v)[3])
{
    const int id[3] = {tr.x, tr.y, tr.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float* p = verts + 3 * (int64_t)id[a];
        v[a] = {p[0], p[1], p[2]};
    }
}

// keys[z] = the first fault of sample z (verts + z vstride), kGeomOk without one
// (every vertex belongs to a triangle, so the triangles see every coordinate)
__global__ __launch_bounds__(256) void geometry_check_kernel(const float* __restrict__ verts, int64_t vstride,
                                                             const int4* __restrict__ tris, int64_t nt,
                                                             unsigned long long* __restrict__ keys)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    V3 v[3];
    load_triangle(verts + (int64_t)blockIdx.y * vstride, tris[t], v);
    bool finite = true;
    for (int a = 0; a < 3; ++a) finite = finite && isfinite(v[a].x) && isfinite(v[a].y) && isfinite(v[a].z);
    const V3 c = cross(sub(v[1], v[0]), sub(v[2], v[0]));
    const double J = sqrt(dot(c, c));
    if (!finite) atomicMin(&keys[blockIdx.y], geom_key(0, t));
    else if (!(J > 0.0) || !isfinite(J)) atomicMin(&keys[blockIdx.y], geom_key(1, t));
}

template <int Q>
__device__ __forceinline__ void write_record(float* __restrict__ r, V3 v0, V3 e1, V3 e2, V3 n, double J)
{
    // the device rules' points in double
    constexpr double a = 0.445948490915965, b = 0.091576213509771;
    constexpr double wa = 0.223381589678011, wb = 0.109951743655322;
    constexpr double x6[6] = {a, b, 1 - 2 * a, a, 1 - 2 * b, b}, y6[6] = {a, b, a, 1 - 2 * a, b, 1 - 2 * b};
    constexpr double w6[6] = {wa, wb, wa, wa, wb, wb};
    constexpr double x3[3] = {1.0 / 6, 2.0 / 3, 1.0 / 6}, y3[3] = {1.0 / 6, 1.0 / 6, 2.0 / 3};
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const double x1 = Q == 6 ? x6[q] : (Q == 3 ? x3[q % 3] : 1.0 / 3);
        const double x2 = Q == 6 ? y6[q] : (Q == 3 ? y3[q % 3] : 1.0 / 3);
        const double w = Q == 6 ? w6[q] : (Q == 3 ? 1.0 / 3 : 1.0);
        const V3 p = add(v0, add(mul(x1, e1), mul(x2, e2)));
        r[3 * q] = (float)p.x;
        r[3 * q + 1] = (float)p.y;
        r[3 * q + 2] = (float)p.z;
        r[3 * Q + q] = (float)(w * 0.5 * J);
    }
    r[4 * Q] = (float)n.x;
    r[4 * Q + 1] = (float)n.y;
    r[4 * Q + 2] = (float)n.z;
#pragma unroll
    for (int e = 4 * Q + 3; e < Rec<Q>::kFloats; ++e) r[e] = 0.f;
}

// The position-dependent arrays of every sample from its vertices (FP64,
// rounded once); sample z's arrays lie gstride floats further on.  One thread
// per triangle: a few hundred bytes written each, microseconds per mesh (the
// host loop and the upload of its 368 bytes per triangle took 0.7 ms for 48
// samples of 640 triangles on 16 threads).
__global__ __launch_bounds__(256) void geometry_kernel(const int4* __restrict__ tris, int64_t nt, int64_t gstride,
                                                       const float* __restrict__ verts, float* __restrict__ rec6,
                                                       float* __restrict__ rec3, float* __restrict__ rec1,
                                                       float* __restrict__ curls, float* __restrict__ geo)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    const int64_t off = (int64_t)blockIdx.y * gstride;
    V3 v[3];
    load_triangle(verts + off, tris[t], v);
    const V3 e1 = sub(v[1], v[0]), e2 = sub(v[2], v[0]);
    const V3 c = cross(e1, e2);
    const double J = sqrt(dot(c, c));
    const V3 n = mul(1.0 / J, c);
    write_record<6>(rec6 + off + t * Rec<6>::kFloats, v[0], e1, e2, n, J);
    write_record<3>(rec3 + off + t * Rec<3>::kFloats, v[0], e1, e2, n, J);
    write_record<1>(rec1 + off + t * Rec<1>::kFloats, v[0], e1, e2, n, J);
    // P1 surface curls: row a = n x grad(phi_a), grad from the dual basis
    const double g11 = dot(e1, e1), g12 = dot(e1, e2), g22 = dot(e2, e2);
    const double det = g11 * g22 - g12 * g12;
    const V3 b1 = add(mul(g22 / det, e1), mul(-g12 / det, e2));
    const V3 b2 = add(mul(-g12 / det, e1), mul(g11 / det, e2));
    const V3 grad[3] = {mul(-1.0, add(b1, b2)), b1, b2};
    float* cu = curls + off + t * 12;
    float* gr = geo + off + t * 16;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const V3 w = cross(n, grad[a]);
        cu[3 * a] = (float)w.x;
        cu[3 * a + 1] = (float)w.y;
        cu[3 * a + 2] = (float)w.z;
        gr[3 * a] = (float)v[a].x;
        gr[3 * a + 1] = (float)v[a].y;
        gr[3 * a + 2] = (float)v[a].z;
    }
    cu[9] = cu[10] = cu[11] = 0.f;
    gr[9] = (float)n.x;
    gr[10] = (float)n.y;
    gr[11] = (float)n.z;
    gr[12] = (float)J;
    gr[13] = gr[14] = gr[15] = 0.f;
}

static hipError_t launch_geometry(const MeshDev& g, int64_t gstride, int ns, hipStream_t s)
{
    for (int z0 = 0; z0 < ns; z0 += 65535) {  // grid y limit
        const int64_t off = (int64_t)z0 * gstride;
        hipLaunchKernelGGL(geometry_kernel, dim3((unsigned)((g.nt + 255) / 256), (unsigned)std::min(65535, ns - z0)),
                           dim3(256), 0, s, g.tris, g.nt, gstride, g.verts + off, g.rec6 + off, g.rec3 + off,
                           g.rec1 + off, g.curls + off, g.geo + off);
    }
    return hipGetLastError();
}

static hipError_t launch_geometry_check(const float* verts, int64_t vstride, int ns, const int4* tris, int64_t nt,
                                        unsigned long long* keys, hipStream_t s)
{
    hipError_t e = hipMemsetAsync(keys, 0xff, sizeof(*keys) * (size_t)ns, s);
    if (e != hipSuccess) return e;
    for (int z0 = 0; z0 < ns; z0 += 65535)
        hipLaunchKernelGGL(geometry_check_kernel, dim3((unsigned)((nt + 255) / 256), (unsigned)std::min(65535, ns - z0)),
                           dim3(256), 0, s, verts + (int64_t)z0 * vstride, vstride, tris, nt, keys + z0);
    return hipGetLastError();
}

// host check of a mesh's positions (the same faults)
static unsigned long long check_positions(const float* v, int64_t nv, const int32_t* tris, int64_t nt)
{
    for (int64_t e = 0; e < 3 * nv; ++e)
        if (!std::isfinite(v[e])) return geom_key(0, 0);
    for (int64_t t = 0; t < nt; ++t) {
        const float *a = v + 3 * (int64_t)tris[3 * t], *b = v + 3 * (int64_t)tris[3 * t + 1],
                    *c = v + 3 * (int64_t)tris[3 * t + 2];
        const V3 n = cross({(double)b[0] - a[0], (double)b[1] - a[1], (double)b[2] - a[2]},
                           {(double)c[0] - a[0], (double)c[1] - a[1], (double)c[2] - a[2]});
        const double J = std::sqrt(dot(n, n));
        if (!(J > 0.0) || !std::isfinite(J)) return geom_key(1, t);
    }
    return kGeomOk;
}

int mesh_build(const float* h_verts, int64_t nv, const int32_t* h_tris, int64_t nt, hipStream_t stream, MeshDev& m,
               std::string& err)
{
    if (nv < 3 || nt < 1) {
        err = "mesh needs at least 3 vertices and 1 triangle";
        return 1;
    }
    if (nt > (int64_t)1 << 30 || nv > (int64_t)1 << 30) {
        err = "mesh too large (more than 2^30 vertices or triangles)";
        return 1;
    }
    for (int64_t t = 0; t < nt; ++t) {
        const int32_t* tr = h_tris + 3 * t;
        for (int a = 0; a < 3; ++a)
            if (tr[a] < 0 || tr[a] >= nv) {
                err = "triangle " + std::to_string(t) + " has a vertex index out of range";
                return 2;
            }
        if (tr[0] == tr[1] || tr[1] == tr[2] || tr[0] == tr[2]) {
            err = "triangle " + std::to_string(t) + " repeats a vertex";
            return 2;
        }
    }
    m.nv = nv;
    m.nt = nt;

    if (const unsigned long long key = check_positions(h_verts, nv, h_tris, nt); key != kGeomOk) {
        err = geom_fault(key);
        return 2;
    }
    std::vector<int32_t> tris4((size_t)nt * 4, 0);
    for (int64_t t = 0; t < nt; ++t)
        for (int a = 0; a < 3; ++a) tris4[4 * t + a] = h_tris[3 * t + a];

    // ---- vertex -> triangle CSR ----
    std::vector<int32_t> vt_ptr((size_t)nv + 1, 0), vt_idx((size_t)nt * 3), vt_corner((size_t)nt * 3);
    for (int64_t t = 0; t < 3 * nt; ++t) vt_ptr[h_tris[t] + 1]++;
    for (int64_t v = 0; v < nv; ++v) vt_ptr[v + 1] += vt_ptr[v];
    {
        std::vector<int32_t> fillp(vt_ptr.begin(), vt_ptr.end() - 1);
        for (int64_t t = 0; t < nt; ++t)
            for (int a = 0; a < 3; ++a) {
                const int32_t q = fillp[h_tris[3 * t + a]]++;
                vt_idx[q] = (int32_t)t;
                vt_corner[q] = (int32_t)(3 * t + a);
            }
    }
    for (int64_t v = 0; v < nv; ++v)
        if (vt_ptr[v + 1] == vt_ptr[v]) {
            err = "vertex " + std::to_string(v) + " belongs to no triangle";
            return 2;
        }

    // ---- neighbour pairs (share >= 1 vertex, self included) ----
    struct Pair {
        int32_t i, j, shared, pad;
    };
    std::vector<Pair> pairs;
    pairs.reserve((size_t)nt * 14);
    m.h_pair_ptr.assign((size_t)nt + 1, 0);
    int32_t maxnb = 0;
    int64_t kinds[4] = {0, 0, 0, 0};
    {
        // triangles around t's corners, counted: a triangle met s times shares s vertices
        std::vector<int32_t> seen((size_t)nt, -1), at((size_t)nt, 0);
        std::vector<std::pair<int32_t, int32_t>> cand;  // (triangle, vertices shared)
        for (int64_t t = 0; t < nt; ++t) {
            cand.clear();
            for (int a = 0; a < 3; ++a) {
                const int32_t v = h_tris[3 * t + a];
                for (int32_t q = vt_ptr[v]; q < vt_ptr[v + 1]; ++q) {
                    const int32_t u = vt_idx[q];
                    if (seen[u] != (int32_t)t) {
                        seen[u] = (int32_t)t;
                        at[u] = (int32_t)cand.size();
                        cand.push_back({u, 1});
                    } else {
                        ++cand[at[u]].second;
                    }
                }
            }
            std::sort(cand.begin(), cand.end());
            maxnb = std::max(maxnb, (int32_t)cand.size());
            for (const auto& [u, s] : cand) {
                if (s == 3 && u != t) {
                    err = "triangles " + std::to_string(t) + " and " + std::to_string(u) + " share all three vertices";
                    return 2;
                }
                pairs.push_back({(int32_t)t, u, s, 0});
                ++kinds[s];
            }
            m.h_pair_ptr[t + 1] = (int64_t)pairs.size();
        }
    }
    m.npairs = (int64_t)pairs.size();
    // the P1 neighbour-pair launches take every pair in any order: grouped by
    // kind, the pairs that share a wavefront take the same quadrature branch
    // (the last entry: the pair's place in its row of the (i, j) order, which
    // fits 32 bits however many pairs there are)
    std::vector<Pair> pairs_kind(pairs.size());
    {
        int64_t next[4] = {0, kinds[3] + kinds[2], kinds[3], 0};
        for (size_t q = 0; q < pairs.size(); ++q) {
            Pair& p = pairs_kind[(size_t)next[pairs[q].shared]++];
            p = pairs[q];
            p.pad = (int32_t)((int64_t)q - m.h_pair_ptr[p.i]);
        }
    }
    m.max_neighbors = maxnb;

    // ---- P1 tiling on a Morton order of the centroids ----
    std::vector<int32_t> perm((size_t)nt);
    {
        V3 lo{1e300, 1e300, 1e300}, hi{-1e300, -1e300, -1e300};
        for (int64_t v = 0; v < nv; ++v) {
            const V3 p{h_verts[3 * v], h_verts[3 * v + 1], h_verts[3 * v + 2]};
            lo = {std::min(lo.x, p.x), std::min(lo.y, p.y), std::min(lo.z, p.z)};
            hi = {std::max(hi.x, p.x), std::max(hi.y, p.y), std::max(hi.z, p.z)};
        }
        const double sx = hi.x - lo.x > 0 ? 1023.0 / (hi.x - lo.x) : 0.0;
        const double sy = hi.y - lo.y > 0 ? 1023.0 / (hi.y - lo.y) : 0.0;
        const double sz = hi.z - lo.z > 0 ? 1023.0 / (hi.z - lo.z) : 0.0;
        // (code, triangle) keys sorted by three passes of ten bits (stable)
        struct Key {
            uint32_t code;
            int32_t t;
        };
        std::vector<Key> key((size_t)nt), tmp((size_t)nt);
        for (int64_t t = 0; t < nt; ++t) {
            V3 v[3];
            for (int a = 0; a < 3; ++a) {
                const float* p = h_verts + 3 * (int64_t)h_tris[3 * t + a];
                v[a] = {p[0], p[1], p[2]};
            }
            const V3 c = mul(1.0 / 3.0, add(add(v[0], v[1]), v[2]));
            const uint32_t ix = (uint32_t)((c.x - lo.x) * sx);
            const uint32_t iy = (uint32_t)((c.y - lo.y) * sy);
            const uint32_t iz = (uint32_t)((c.z - lo.z) * sz);
            key[t] = {spread10(ix) | (spread10(iy) << 1) | (spread10(iz) << 2), (int32_t)t};
        }
        for (int shift = 0; shift < 30; shift += 10) {
            std::vector<int32_t> first(1025, 0);
            for (const Key& k : key) ++first[((k.code >> shift) & 1023) + 1];
            for (int q = 0; q < 1024; ++q) first[q + 1] += first[q];
            for (const Key& k : key) tmp[(size_t)first[(k.code >> shift) & 1023]++] = k;
            key.swap(tmp);
        }
        for (int64_t t = 0; t < nt; ++t) perm[t] = key[t].t;
    }
    std::vector<int32_t> pos((size_t)nt);
    for (int64_t q = 0; q < nt; ++q) pos[perm[q]] = (int32_t)q;
    // P1 numbering: vertices in the order they first appear along the Morton
    // order of the triangles, so the vertices of a tile are (nearly)
    // consecutive and its accumulator flush lands in few cache lines; the
    // P1 kernels accumulate in this numbering (see p1_vnew / p1_vold)
    std::vector<int32_t> vnew((size_t)nv, -1), vold;
    vold.reserve((size_t)nv);
    for (int64_t q = 0; q < nt; ++q)
        for (int a = 0; a < 3; ++a) {
            const int32_t v = h_tris[3 * (int64_t)perm[q] + a];
            if (vnew[v] < 0) {
                vnew[v] = (int32_t)vold.size();
                vold.push_back(v);
            }
        }
    for (int64_t v = 0; v < nv; ++v)  // vertices in no triangle
        if (vnew[v] < 0) {
            vnew[v] = (int32_t)vold.size();
            vold.push_back((int32_t)v);
        }
    std::vector<int32_t> tris_p1((size_t)nt * 3);
    for (int64_t e = 0; e < 3 * nt; ++e) tris_p1[e] = vnew[h_tris[e]];
    // row tiles nest in column tiles, so the symmetric sweep can pair a row
    // tile with the column tiles from its own on
    const Tiling colT = make_tiling(perm, tris_p1.data(), nv, kP1ColTris, kP1ColVerts);
    const Tiling rowT = make_tiling(perm, tris_p1.data(), nv, kP1RowTris, kP1RowVerts, colT.ptr);
    const int nrowt = (int)rowT.ptr.size() - 1, ncolt = (int)colT.ptr.size() - 1;
    std::vector<int32_t> row_ctile((size_t)nrowt);
    std::vector<int64_t> sym_ptr((size_t)nrowt + 1, 0);
    for (int r = 0, c = 0; r < nrowt; ++r) {
        while (colT.ptr[c + 1] <= rowT.ptr[r]) ++c;
        row_ctile[r] = c;
        sym_ptr[r + 1] = sym_ptr[r] + (ncolt - c);
    }
    // incidences of each column-tile vertex slot (CSR over the global slot index)
    std::vector<int32_t> inc_ptr(colT.verts.size() + 1, 0), inc;
    {
        const int ntile = (int)colT.ptr.size() - 1;
        for (int tl = 0; tl < ntile; ++tl)
            for (int32_t p = colT.ptr[tl]; p < colT.ptr[tl + 1]; ++p)
                for (int b = 0; b < 3; ++b) ++inc_ptr[colT.vptr[tl] + colT.slot[4 * (size_t)p + b] + 1];
        for (size_t g = 0; g + 1 < inc_ptr.size(); ++g) inc_ptr[g + 1] += inc_ptr[g];
        inc.assign((size_t)inc_ptr.back(), 0);
        std::vector<int32_t> fill(inc_ptr.begin(), inc_ptr.end() - 1);
        for (int tl = 0; tl < ntile; ++tl)
            for (int32_t p = colT.ptr[tl]; p < colT.ptr[tl + 1]; ++p)
                for (int b = 0; b < 3; ++b) {
                    const int32_t g = colT.vptr[tl] + colT.slot[4 * (size_t)p + b];
                    inc[(size_t)fill[g]++] = 4 * (p - colT.ptr[tl]) + b;
                }
    }

    // ---- one device allocation ----
    struct Part {
        const void* src;
        size_t bytes;
        void** dst;
    };
    std::vector<Part> parts;
    // the position-dependent arrays first, one contiguous region that
    // geometry_kernel fills from the vertices at its start
    float* d_verts = nullptr;
    parts.push_back({h_verts, (size_t)nv * 12, (void**)&d_verts});
    parts.push_back({nullptr, (size_t)nt * Rec<6>::kFloats * 4, (void**)&m.rec6});
    parts.push_back({nullptr, (size_t)nt * Rec<3>::kFloats * 4, (void**)&m.rec3});
    parts.push_back({nullptr, (size_t)nt * Rec<1>::kFloats * 4, (void**)&m.rec1});
    parts.push_back({nullptr, (size_t)nt * 12 * 4, (void**)&m.curls});
    parts.push_back({nullptr, (size_t)nt * 16 * 4, (void**)&m.geo});
    constexpr size_t kGeomParts = 6;
    parts.push_back({tris4.data(), tris4.size() * 4, (void**)&m.tris});
    parts.push_back({pairs.data(), pairs.size() * sizeof(Pair), (void**)&m.pairs});
    parts.push_back({pairs_kind.data(), pairs_kind.size() * sizeof(Pair), (void**)&m.pairs_by_kind});
    parts.push_back({m.h_pair_ptr.data(), m.h_pair_ptr.size() * 8, (void**)&m.pair_ptr});
    parts.push_back({vt_ptr.data(), vt_ptr.size() * 4, (void**)&m.vt_ptr});
    parts.push_back({vt_idx.data(), vt_idx.size() * 4, (void**)&m.vt_idx});
    parts.push_back({vt_corner.data(), vt_corner.size() * 4, (void**)&m.vt_corner});
    int32_t *d_perm, *d_pos, *d_rp, *d_rvp, *d_rv, *d_cp, *d_cvp, *d_cv, *d_cip, *d_ci, *d_rct;
    int64_t* d_sym;
    int4 *d_rs, *d_cs;
    parts.push_back({perm.data(), perm.size() * 4, (void**)&d_perm});
    parts.push_back({pos.data(), pos.size() * 4, (void**)&d_pos});
    parts.push_back({rowT.ptr.data(), rowT.ptr.size() * 4, (void**)&d_rp});
    parts.push_back({rowT.vptr.data(), rowT.vptr.size() * 4, (void**)&d_rvp});
    parts.push_back({rowT.verts.data(), rowT.verts.size() * 4, (void**)&d_rv});
    parts.push_back({rowT.slot.data(), rowT.slot.size() * 4, (void**)&d_rs});
    parts.push_back({colT.ptr.data(), colT.ptr.size() * 4, (void**)&d_cp});
    parts.push_back({colT.vptr.data(), colT.vptr.size() * 4, (void**)&d_cvp});
    parts.push_back({colT.verts.data(), colT.verts.size() * 4, (void**)&d_cv});
    parts.push_back({colT.slot.data(), colT.slot.size() * 4, (void**)&d_cs});
    parts.push_back({inc_ptr.data(), inc_ptr.size() * 4, (void**)&d_cip});
    parts.push_back({inc.data(), inc.size() * 4, (void**)&d_ci});
    parts.push_back({row_ctile.data(), row_ctile.size() * 4, (void**)&d_rct});
    parts.push_back({sym_ptr.data(), sym_ptr.size() * 8, (void**)&d_sym});
    parts.push_back({vnew.data(), vnew.size() * 4, (void**)&m.p1_vnew});
    parts.push_back({vold.data(), vold.size() * 4, (void**)&m.p1_vold});
    parts.push_back({nullptr, sizeof(unsigned long long), (void**)&m.geom_flag});
    size_t total = 0;
    std::vector<size_t> off;
    for (auto& p : parts) {
        off.push_back(total);
        total += (p.bytes + 255) / 256 * 256;
    }
    m.geom_bytes = off[kGeomParts];
    if (hipGetDevice(&m.device) != hipSuccess) {
        err = "no HIP device";
        return 5;
    }
    if (hipMalloc(&m.block, total) != hipSuccess) {
        err = "device allocation of " + std::to_string(total) + " bytes failed";
        (void)hipGetLastError();
        return 6;
    }
    // the vertices, then every connectivity array, through one host staging
    // buffer and two copies (a copy per array cost more than the rest of the
    // set-up for small meshes)
    for (size_t q = 0; q < parts.size(); ++q) *parts[q].dst = (char*)m.block + off[q];
    m.verts = d_verts;
    {
        Stage st;
        const size_t head = ((size_t)nv * 12 + 255) / 256 * 256, conn = off[kGeomParts];
        char* host = st.get(head + (total - conn));
        std::memcpy(host, h_verts, (size_t)nv * 12);
        for (size_t q = kGeomParts; q < parts.size(); ++q)
            if (parts[q].src && parts[q].bytes) std::memcpy(host + head + (off[q] - conn), parts[q].src, parts[q].bytes);
        hipError_t e = hipMemcpyAsync(m.block, host, (size_t)nv * 12, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync((char*)m.block + conn, host + head, total - conn, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = launch_geometry(m, 0, 1, stream);
        // the handle may be used on any stream from here on
        const hipError_t es = hipStreamSynchronize(stream);
        if (e == hipSuccess) e = es;
        if (e != hipSuccess) {
            err = std::string("mesh upload: ") + hipGetErrorString(e);
            (void)hipFree(m.block);
            m.block = nullptr;
            return 3;
        }
    }
    m.tiles.perm = d_perm;
    m.tiles.pos = d_pos;
    m.tiles.row_ptr = d_rp;
    m.tiles.row_vptr = d_rvp;
    m.tiles.row_verts = d_rv;
    m.tiles.row_slot = d_rs;
    m.tiles.col_ptr = d_cp;
    m.tiles.col_vptr = d_cvp;
    m.tiles.col_verts = d_cv;
    m.tiles.col_slot = d_cs;
    m.tiles.col_inc_ptr = d_cip;
    m.tiles.col_inc = d_ci;
    m.tiles.row_ctile = d_rct;
    m.tiles.sym_ptr = d_sym;
    m.tiles.nsym = sym_ptr.back();
    m.tiles.nrow_tiles = nrowt;
    m.tiles.ncol_tiles = ncolt;
    m.h_row_slots = rowT.vptr.empty() ? 0 : rowT.vptr.back();
    return 0;
}

// the position-dependent pointers of m moved from its own block to region
static void rebase_geometry(MeshDev& g, const MeshDev& m, void* region)
{
    auto at = [&](float* p) { return (float*)((char*)region + ((char*)p - (char*)m.block)); };
    g.verts = at(m.verts);
    g.rec6 = at(m.rec6);
    g.rec3 = at(m.rec3);
    g.rec1 = at(m.rec1);
    g.curls = at(m.curls);
    g.geo = at(m.geo);
}

int geomset_build(const MeshDev& m, const float* h_verts, int ns, hipStream_t s, MeshDev& view, void** block,
                  std::string& err)
{
    const size_t vb = (size_t)m.nv * 12, bytes = m.geom_bytes * (size_t)ns;
    const size_t key_at = (bytes + 255) / 256 * 256;
    *block = nullptr;
    if (hipMalloc(block, key_at + sizeof(unsigned long long) * (size_t)ns) != hipSuccess) {
        (void)hipGetLastError();
        err = "device allocation of " + std::to_string(bytes) + " bytes failed";
        return 6;
    }
    view = m;
    rebase_geometry(view, m, *block);
    unsigned long long* keys = (unsigned long long*)((char*)*block + key_at);
    std::vector<unsigned long long> hk((size_t)ns, kGeomOk);
    hipError_t e;
    {
        Stage st;
        char* host = st.get(vb * (size_t)ns);
        std::memcpy(host, h_verts, vb * (size_t)ns);
        // the vertices lead each sample's region
        e = hipMemcpy2DAsync(*block, m.geom_bytes, host, vb, vb, (size_t)ns, hipMemcpyHostToDevice, s);
        const int64_t gstride = (int64_t)(m.geom_bytes / sizeof(float));
        if (e == hipSuccess) e = launch_geometry_check(view.verts, gstride, ns, m.tris, m.nt, keys, s);
        if (e == hipSuccess) e = launch_geometry(view, gstride, ns, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(hk.data(), keys, sizeof(hk[0]) * hk.size(), hipMemcpyDeviceToHost, s);
        const hipError_t es = hipStreamSynchronize(s);
        if (e == hipSuccess) e = es;
    }
    int rc = 0;
    if (e != hipSuccess) {
        err = std::string("geometry set: ") + hipGetErrorString(e);
        rc = 3;
    }
    for (int z = 0; z < ns && rc == 0; ++z)
        if (hk[z] != kGeomOk) {
            err = "sample " + std::to_string(z) + ": " + geom_fault(hk[z]);
            rc = 2;
        }
    if (rc) {
        (void)hipFree(*block);
        *block = nullptr;
    }
    return rc;
}

// memory the kernels of this device may read: its own allocation (another GPU's
// need not be mapped here)
static bool owned_by(const void* p, int device)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeDevice && a.device == device;
}

int mesh_set_vertices(MeshDev& m, const float* verts, bool on_device, hipStream_t s, std::string& err)
{
    if (!m.block) {
        err = "mesh has no device data";
        return 1;
    }
    const size_t vb = (size_t)m.nv * 12;
    Stage st;
    void* tmp = nullptr;
    const float* src = verts;
    hipError_t e = hipSuccess;
    if (!on_device || !owned_by(verts, m.device)) {  // checked on this device as well: through a temporary
        e = hipMallocAsync(&tmp, vb, s);
        if (e == hipSuccess) {
            const void* from = verts;
            if (!on_device) from = std::memcpy(st.get(vb), verts, vb);
            e = hipMemcpyAsync(tmp, from, vb, on_device ? hipMemcpyDefault : hipMemcpyHostToDevice, s);
            src = (const float*)tmp;
        }
    }
    unsigned long long key = kGeomOk;
    if (e == hipSuccess) e = launch_geometry_check(src, 0, 1, m.tris, m.nt, m.geom_flag, s);
    if (e == hipSuccess) e = hipMemcpyAsync(&key, m.geom_flag, sizeof(key), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e == hipSuccess && key == kGeomOk) {
        e = hipMemcpyAsync(m.verts, src, vb, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess) e = launch_geometry(m, 0, 1, s);
    }
    if (tmp) (void)hipFreeAsync(tmp, s);
    // other streams may use the new positions from here on
    const hipError_t es = hipStreamSynchronize(s);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) {
        err = std::string("set_vertices: ") + hipGetErrorString(e);
        return 3;
    }
    if (key != kGeomOk) {
        err = geom_fault(key);
        return 2;
    }
    return 0;
}

void mesh_free(MeshDev& m)
{
    if (m.block) (void)hipFree(m.block);
    m.block = nullptr;
}

}  // namespace bem
