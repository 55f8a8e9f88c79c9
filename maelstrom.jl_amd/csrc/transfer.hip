// APIC transfers on the dense grid: particles to grid (flip.jl:501-606) and grid to
// particles (flip.jl:1208-1252).
//
// The deposit is deterministic: each contribution is rounded once to 64-bit fixed point
// (2^-32) and added with an integer atomic. Integer addition is associative, so the
// accumulated momentum and weight are the same whatever order the particles arrive in,
// unlike the reference's float atomics (flip.jl:532-533). The level-set splat keeps the
// reference's integer atomic minimum over order keys, which is order-independent too.
#include "dense.hpp"
#include "scan.hpp"
#include "p2g_tiled.hpp"
#include <cmath>
#include <cstring>

namespace mael {

// flip.jl:513-537 p2g_kernel!: the tiled deposit over the dense grid's face arrays.
struct DenseNodes {
    // The adjoint's gather reads the faces directly: particles2grid_adjoint takes 265 us for
    // 1.6 M particles on 256 x 256 x 128, in cell order and in two interleaved runs, and took
    // 295 and 355 through boxes.
    static constexpr bool ADJ_BOXED = false;
    __device__ static int boxes() { return 0; }
    int n[3];
    __device__ int64_t index(int a, int I, int J, int K) const {
        int n1 = n[0] + (a == 0), n2 = n[1] + (a == 1), n3 = n[2] + (a == 2);
        if (I < 0 || I >= n1 || J < 0 || J >= n2 || K < 0 || K >= n3) return -1;
        return (int64_t)I + (int64_t)n1 * ((int64_t)J + (int64_t)n2 * K);
    }
    static constexpr int TAB = 1;   // no table
    struct Near {};
    __device__ Near near(const int*, const int*) const { return {}; }
    __device__ void stage(const Near&, int32_t*) const {}
    __device__ int64_t at(const Near&, const int32_t*, int a, int I, int J, int K) const { return index(a, I, J, K); }
};

struct DenseCells {
    int n[3];
    __device__ int64_t index(int I, int J, int K) const {
        if (I < 0 || I >= n[0] || J < 0 || J >= n[1] || K < 0 || K >= n[2]) return -1;
        return (int64_t)I + (int64_t)n[0] * ((int64_t)J + (int64_t)n[1] * K);
    }
    static constexpr int TAB = 1;   // no table
    struct Near {};
    __device__ Near near(const int*, const int*) const { return {}; }
    __device__ void stage(const Near&, int32_t*) const {}
    __device__ int64_t at(const Near&, const int32_t*, int I, int J, int K) const { return index(I, J, K); }
};

// flip.jl:562-565 union_kernel!.
__global__ void k_union(size_t C, float* __restrict__ phi, const float* __restrict__ phi0, const int32_t* __restrict__ phip,
                        float dx) {
    size_t l = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l < C) phi[l] = jmin(phi0[l] + dx, orderfloat(phip[l]));
}

// flip.jl:567-585 combine_kernel! for axis A, from the fixed-point accumulators.
template <int A>
__global__ __launch_bounds__(256) void k_dense_combine(float* __restrict__ u, const float* __restrict__ u0,
                                                       const unsigned long long* __restrict__ mom,
                                                       const unsigned long long* __restrict__ wt,
                                                       const float* __restrict__ phi, int3 n, float r, float full) {
    int n1 = n.x + (A == 0), n2 = n.y + (A == 1), n3 = n.z + (A == 2);
    int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
    if (i >= n1 || j >= n2 || k >= n3) return;
    int bi = i - (A == 0), bj = j - (A == 1), bk = k - (A == 2);
    auto at = [&](int a, int b, int c) { return phi[(size_t)a + (size_t)n.x * ((size_t)b + (size_t)n.y * c)]; };
    bool inb = bi >= 0 && bj >= 0 && bk >= 0;
    bool ina = i < n.x && j < n.y && k < n.z;
    float fa = inb ? at(bi, bj, bk) : at(min(i, n.x - 1), min(j, n.y - 1), min(k, n.z - 1));
    float fb = ina ? at(i, j, k) : fa;
    float phif = 0.5f * (fa + fb);
    size_t idx = (size_t)i + (size_t)n1 * ((size_t)j + (size_t)n2 * k);
    float wgt = fromfix(wt[idx]);
    float m = fromfix(mom[idx]);
    float v0 = u0[idx];
    u[idx] = phif >= -r ? __fdiv_rn(m + jmax(full - wgt, 0.0f) * v0, jmax(full, wgt)) : v0;
}

void DenseBasin::p2g(float dt) {
    hipStream_t s = st.s;
    for (int a = 0; a < 3; ++a) {
        fill_async(mom[a].p, faces(a), 0ull, s);
        fill_async(wt[a].p, faces(a), 0ull, s);
    }
    size_t C = cells();
    int32_t big;
    {
        float f = 1e30f;
        int32_t bits;
        std::memcpy(&bits, &f, 4);
        big = bits;   // orderkey of a positive float is its bit pattern
    }
    fill_async(phip.p, C, big, s);
    if (n > 0) {
        PView ps = view(cur);
        kt.begin(K_P2G, s);
        DenseNodes map{{g.n[0], g.n[1], g.n[2]}};
        P2GArgs A{{g.lo[0], g.lo[1], g.lo[2]}, g.dx, {mom[0].p, mom[1].p, mom[2].p}, {wt[0].p, wt[1].p, wt[2].p}, 1.0f};
        hipLaunchKernelGGL((k_p2g_tiled<DenseNodes, P2GSource>), p2g_grid(n), dim3(P2G_THREADS), 0, s, ps, n,
                           map, P2GSource{ps, dt}, A);
        kt.end(K_P2G, s);
        kt.begin(K_SPLAT, s);
        hipLaunchKernelGGL((k_splat_tiled<DenseCells>), dim3(cdiv(n, P2G_THREADS)), dim3(P2G_THREADS), 0, s, ps, n,
                           DenseCells{{g.n[0], g.n[1], g.n[2]}}, g.lo[0], g.lo[1], g.lo[2], g.dx, dt, phip.p);
        kt.end(K_SPLAT, s);
        MAEL_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_union, dim3(cdiv(C, 256)), dim3(256), 0, s, C, phi.p, phi0.p, phip.p, g.dx);
    float r = (float)(band - 1) * g.dx, full = (float)nmin;
    int3 nn = make_int3(g.n[0], g.n[1], g.n[2]);
    dim3 blk(64, 4, 1);
    kt.begin(K_COMBINE, s);
    hipLaunchKernelGGL(k_dense_combine<0>, dim3(cdiv(g.n[0] + 1, 64), cdiv(g.n[1], 4), g.n[2]), blk, 0, s, u[0].p, u0[0].p,
                       mom[0].p, wt[0].p, phi.p, nn, r, full);
    hipLaunchKernelGGL(k_dense_combine<1>, dim3(cdiv(g.n[0], 64), cdiv(g.n[1] + 1, 4), g.n[2]), blk, 0, s, u[1].p, u0[1].p,
                       mom[1].p, wt[1].p, phi.p, nn, r, full);
    hipLaunchKernelGGL(k_dense_combine<2>, dim3(cdiv(g.n[0], 64), cdiv(g.n[1], 4), g.n[2] + 1), blk, 0, s, u[2].p, u0[2].p,
                       mom[2].p, wt[2].p, phi.p, nn, r, full);
    kt.end(K_COMBINE, s);
    MAEL_LAUNCH_CHECK();
}

// The gather's face nodes: indices clamped to the array (flip.jl:1210-1224).
struct DenseClampNodes {
    // Two boxes (a row of cells that crosses the funnel's ring), one while the launch's
    // workgroups are all on the chip at once and its time is one's chain of boxes: 98,000
    // particles in two interleaved runs 21 us with one box, 57 with up to four (18.9 and 18.4
    // in cell order); 1.6 M 176 us with two, 211 with one and 186 with four (123, 163 and 125
    // in cell order).
    __device__ static int boxes() { return gridDim.x <= 512 ? 1 : 2; }
    static constexpr bool HOLES = false;
    int n[3];
    __device__ int64_t index(int a, int I, int J, int K) const {
        int n1 = n[0] + (a == 0), n2 = n[1] + (a == 1), n3 = n[2] + (a == 2);
        I = min(max(I, 0), n1 - 1); J = min(max(J, 0), n2 - 1); K = min(max(K, 0), n3 - 1);
        return (int64_t)I + (int64_t)n1 * ((int64_t)J + (int64_t)n2 * K);
    }
    static constexpr int TAB = 1;   // no table
    struct Near {};
    __device__ Near near(const int*, const int*) const { return {}; }
    __device__ void stage(const Near&, int32_t*) const {}
    __device__ int64_t at(const Near&, const int32_t*, int a, int I, int J, int K) const { return index(a, I, J, K); }
};

void DenseBasin::g2p(float dt, float grav) {
    if (n == 0) return;
    kt.begin(K_G2P, st.s);
    const G2PFaces F{{u[0].p, u[1].p, u[2].p}, {flag[0].p, flag[1].p, flag[2].p}};
    hipLaunchKernelGGL(k_g2p_tiled<DenseClampNodes>, dim3(cdiv(n, P2G_THREADS)), dim3(P2G_THREADS), 0, st.s, view(cur), n,
                       DenseClampNodes{{g.n[0], g.n[1], g.n[2]}}, g.lo[0], g.lo[1], g.lo[2], g.dx, F, dt, grav);
    kt.end(K_G2P, st.s);
    MAEL_LAUNCH_CHECK();
}

}  // namespace mael

namespace mael {

// ─── adjoints of the transfers (no counterpart in the reference) ─────────────
// With the particles' positions and time lags and the level set fixed, P2G is linear in
// the particles' velocities and APIC rows (and in u0), and G2P is linear in the face
// velocities; these are their transposes, for reverse-mode gradients. The G2P adjoint is
// a deposit (the tiled fixed-point scatter, so it is deterministic), the P2G adjoint a
// gather.

// u-bar = the accumulated deposit / scale.
__global__ void k_adj_fromfix(float* __restrict__ ub, const unsigned long long* __restrict__ acc, size_t n, double inv) {
    size_t l = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l < n) ub[l] = (float)((double)(long long)acc[l] * FIX_INV * inv);
}
// The particles' input cotangents: v passes through G2P where the grid was not reached
// (flip.jl:1239-1242), the rows never do.
__global__ void k_g2p_adj_post(PB12 pb, const uint8_t* __restrict__ reached, int64_t n) {
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    bool k = reached[p] != 0;
    for (int f = 0; f < 12; ++f)
        if (k || f >= 3) pb.f[f][p] = 0.0f;
}

void DenseBasin::adj_alloc() {
    if (ub[0].p) return;
    hipStream_t s = st.s;
    for (int a = 0; a < 3; ++a) {
        ub[a].alloc(faces(a)); ub0[a].alloc(faces(a)); adjacc[a].alloc(faces(a));
        fill_async(ub[a].p, faces(a), 0.0f, s);
        fill_async(ub0[a].p, faces(a), 0.0f, s);
    }
    for (int f = 0; f < 12; ++f) {
        pb[f].alloc(capacity);
        fill_async(pb[f].p, (size_t)capacity, 0.0f, s);
    }
    reached.alloc(capacity);
    MAEL_LAUNCH_CHECK();
}

// The transpose of grid2particles! (flip.jl:1226-1252) in u: ub = G2P^T (pb); pb becomes
// the cotangent of the input particle velocities.
void DenseBasin::g2p_adjoint(float dt) {
    (void)dt;
    adj_alloc();
    hipStream_t s = st.s;
    for (int a = 0; a < 3; ++a) fill_async(adjacc[a].p, faces(a), 0ull, s);
    if (n == 0) {
        for (int a = 0; a < 3; ++a) fill_async(ub[a].p, faces(a), 0.0f, s);
        return;
    }
    PB12 P;
    for (int f = 0; f < 12; ++f) P.f[f] = pb[f].p;
    int* bound = (int*)partials.p;
    fill_async(bound, (size_t)1, 0, s);
    const G2PFaces F{{nullptr, nullptr, nullptr}, {flag[0].p, flag[1].p, flag[2].p}};
    hipLaunchKernelGGL(k_g2p_adj_reached<DenseClampNodes>, dim3(cdiv(n, P2G_THREADS)), dim3(P2G_THREADS), 0, s, view(cur), n,
                       DenseClampNodes{{g.n[0], g.n[1], g.n[2]}}, g.lo[0], g.lo[1], g.lo[2], g.dx, F, reached.p, P, bound);
    int bits = 0;
    MAEL_HIP(hipMemcpyAsync(st.pinned, bound, sizeof(int), hipMemcpyDeviceToHost, s));
    st.sync();
    std::memcpy(&bits, st.pinned, sizeof(int));
    float m;
    std::memcpy(&m, &bits, sizeof(float));
    // a node takes at most 27 cells' particles (2 nmin each): keep the sum within 2^30
    double lim = std::ldexp(1.0, 30) / (27.0 * 2.0 * std::max(nmin, 1)), scale = 1.0;
    if (m > 0.0f) scale = std::ldexp(1.0, std::min(60, std::max(-60, (int)std::floor(std::log2(lim / (double)m)))));
    G2PAdjSource src{{P.f[0], P.f[1], P.f[2], P.f[3], P.f[4], P.f[5], P.f[6], P.f[7], P.f[8], P.f[9], P.f[10], P.f[11]},
                     reached.p, 4.0f / (g.dx * g.dx)};
    P2GArgs A{{g.lo[0], g.lo[1], g.lo[2]}, g.dx, {adjacc[0].p, adjacc[1].p, adjacc[2].p}, {nullptr, nullptr, nullptr},
              (float)scale};
    hipLaunchKernelGGL((k_p2g_tiled<DenseClampNodes, G2PAdjSource>), p2g_grid(n), dim3(P2G_THREADS), 0, s,
                       view(cur), n, DenseClampNodes{{g.n[0], g.n[1], g.n[2]}}, src, A);
    for (int a = 0; a < 3; ++a)
        hipLaunchKernelGGL(k_adj_fromfix, dim3(cdiv(faces(a), 256)), dim3(256), 0, s, ub[a].p, adjacc[a].p, faces(a),
                           1.0 / scale);
    hipLaunchKernelGGL(k_g2p_adj_post, dim3(cdiv(n, 256)), dim3(256), 0, s, P, reached.p, n);
    MAEL_LAUNCH_CHECK();
}

// The P2G adjoint's face part: the cotangent of a face's momentum sum (s = ub / max(nmin,
// W) in the band, else 0) and of u0 (flip.jl:567-585 combine, differentiated).
template <int A>
__global__ __launch_bounds__(256) void k_p2g_adj_faces(float* __restrict__ sface, float* __restrict__ ub0,
                                                       const float* __restrict__ ub, const unsigned long long* __restrict__ wt,
                                                       const float* __restrict__ phi, int3 n, float r, float full) {
    int n1 = n.x + (A == 0), n2 = n.y + (A == 1), n3 = n.z + (A == 2);
    int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
    if (i >= n1 || j >= n2 || k >= n3) return;
    int bi = i - (A == 0), bj = j - (A == 1), bk = k - (A == 2);
    auto at = [&](int a, int b, int c) { return phi[(size_t)a + (size_t)n.x * ((size_t)b + (size_t)n.y * c)]; };
    bool inb = bi >= 0 && bj >= 0 && bk >= 0;
    bool ina = i < n.x && j < n.y && k < n.z;
    float fa = inb ? at(bi, bj, bk) : at(min(i, n.x - 1), min(j, n.y - 1), min(k, n.z - 1));
    float fb = ina ? at(i, j, k) : fa;
    float phif = 0.5f * (fa + fb);
    size_t idx = (size_t)i + (size_t)n1 * ((size_t)j + (size_t)n2 * k);
    float u = ub[idx];
    if (phif >= -r) {
        float W = fromfix(wt[idx]), den = jmax(full, W);
        sface[idx] = u / den;
        ub0[idx] = u * (jmax(full - W, 0.0f) / den);
    } else {
        sface[idx] = 0.0f;
        ub0[idx] = u;
    }
}
// The transpose of particles2grid! (flip.jl:587-606) in the particles' v and APIC rows and
// in u0, at the positions, lags, level set and weights of the last deposit: pb += P2G^T
// (ub) for the particles (added to what G2P's adjoint passed through), ub0 = its part for
// u0.
void DenseBasin::p2g_adjoint(float dt) {
    adj_alloc();
    hipStream_t s = st.s;
    float r = (float)(band - 1) * g.dx, full = (float)nmin;
    int3 nn = make_int3(g.n[0], g.n[1], g.n[2]);
    dim3 blk(64, 4, 1);
    float* sf[3];
    for (int a = 0; a < 3; ++a) sf[a] = reinterpret_cast<float*>(adjacc[a].p);   // scratch, faces(a) floats
    hipLaunchKernelGGL(k_p2g_adj_faces<0>, dim3(cdiv(g.n[0] + 1, 64), cdiv(g.n[1], 4), g.n[2]), blk, 0, s, sf[0], ub0[0].p,
                       ub[0].p, wt[0].p, phi.p, nn, r, full);
    hipLaunchKernelGGL(k_p2g_adj_faces<1>, dim3(cdiv(g.n[0], 64), cdiv(g.n[1] + 1, 4), g.n[2]), blk, 0, s, sf[1], ub0[1].p,
                       ub[1].p, wt[1].p, phi.p, nn, r, full);
    hipLaunchKernelGGL(k_p2g_adj_faces<2>, dim3(cdiv(g.n[0], 64), cdiv(g.n[1], 4), g.n[2] + 1), blk, 0, s, sf[2], ub0[2].p,
                       ub[2].p, wt[2].p, phi.p, nn, r, full);
    if (n > 0) {
        PB12 P;
        for (int f = 0; f < 12; ++f) P.f[f] = pb[f].p;
        hipLaunchKernelGGL(k_p2g_adj_gather<DenseNodes>, dim3(cdiv(n, P2G_THREADS)), dim3(P2G_THREADS), 0, s, view(cur), n,
                           DenseNodes{{g.n[0], g.n[1], g.n[2]}}, g.lo[0], g.lo[1], g.lo[2], g.dx, dt,
                           AdjFaces{{sf[0], sf[1], sf[2]}}, P);
    }
    MAEL_LAUNCH_CHECK();
}

}  // namespace mael
