// The transfers between particles and faces, tiled: the APIC deposit (flip.jl:513-537) as a
// reduction, the gather (flip.jl:1226-1244), and the level-set splat.
//
// In the deposit a workgroup takes 256 consecutive particles (resampling leaves them in
// cell order, so they are close in space) and, one velocity component at a time,
// accumulates their 27-node contributions into a box of nodes in LDS with 64-bit integer
// adds, then adds each touched node of the box to HBM once. Contributions are rounded to
// 2^-32 fixed point exactly as a per-particle deposit does and integer addition is
// associative, so the result is bit-identical to depositing every contribution with its
// own global atomic, in any order.
#pragma once
#include "common.hpp"
#include <type_traits>

namespace mael {

constexpr int P2G_THREADS = 256;
// Nodes per component in LDS (mom + wt: 16 B a node): 32 KB, four workgroups a CU.
constexpr int P2G_BOX = 2048;

// The wavefront's minimum in every lane: six DPP steps (a row's 16 lanes, then the rows),
// no LDS. Every lane must be active.
__device__ inline int wave_min(int v) {
#define MAEL_DPP_MIN(ctrl, rows) v = min(v, __builtin_amdgcn_update_dpp(v, v, ctrl, rows, 0xf, false))
    MAEL_DPP_MIN(0xB1, 0xf);    // quad_perm [1,0,3,2]
    MAEL_DPP_MIN(0x4E, 0xf);    // quad_perm [2,3,0,1]
    MAEL_DPP_MIN(0x141, 0xf);   // row_half_mirror
    MAEL_DPP_MIN(0x140, 0xf);   // row_mirror
    MAEL_DPP_MIN(0x142, 0xa);   // row_bcast15 into rows 1 and 3
    MAEL_DPP_MIN(0x143, 0xc);   // row_bcast31 into rows 2 and 3
#undef MAEL_DPP_MIN
    return __builtin_amdgcn_readlane(v, 63);
}
// K workgroup minima at once (one pair of barriers); red, 16-byte aligned, holds K x (P2G_THREADS / 64).
template <int K> __device__ inline void wg_mins(int (&v)[K], int* red) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_min(v[k]);
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) red[k * (P2G_THREADS / 64) + (threadIdx.x >> 6)] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int4 r = *reinterpret_cast<const int4*>(red + 4 * k);
        v[k] = min(min(r.x, r.y), min(r.z, r.w));
    }
}
// (i, j, k) of entry l of a box of ex x ey columns: the quotients from float reciprocals,
// exact for l < 2^21 (a quotient's distance from an integer, 1 / (2 ex), exceeds its
// rounding error).
struct BoxIndex {
    int ex, ey;
    float rx, ry;
    __device__ BoxIndex(int ex_, int ey_) : ex(ex_), ey(ey_), rx(1.0f / (float)ex_), ry(1.0f / (float)ey_) {}
    __device__ void at(int l, int& i, int& j, int& k) const {
        const int r = (int)(((float)l + 0.5f) * rx);
        i = l - r * ex;
        k = (int)(((float)r + 0.5f) * ry);
        j = r - k * ey;
    }
};

struct P2GArgs {
    float lo[3];
    float dx;
    unsigned long long* mom[3];
    unsigned long long* wt[3];   // null: no weights accumulated
    float scale;                 // every momentum contribution is multiplied by it before rounding
};

// The particle side of the deposit: the temporal weight of particle p, and the value and
// affine row it deposits for component a.
struct P2GSource {   // flip.jl:513-537: v_a and the APIC row c_a, weighted by temporal(lag, dt)
    static constexpr bool WEIGHTS = true, SCALED = false;   // weights are summed; P2GArgs::scale is 1
    PView ps;
    float dt;
    __device__ float weight(int64_t p) const { return temporal(ps.f[15][p], dt); }
    __device__ void comp(int64_t p, int a, float& v, float& c0, float& c1, float& c2) const {
        v = ps.f[3 + a][p];
        c0 = ps.f[6 + 3 * a][p]; c1 = ps.f[7 + 3 * a][p]; c2 = ps.f[8 + 3 * a][p];
    }
};

// b + m where b may be the saturated coordinate of a particle far off the grid or not finite:
// a defined wrap, so that the bounds test of the sum and its use see one value. (In signed
// arithmetic the compiler tested b < -m on one side and b + m + 1 > n on the other, which
// together pass INT_MAX, and the add went out of bounds.)
__device__ inline int node_at(int b, int m) { return (int)((unsigned)b + (unsigned)m); }

// The contributions of a particle to the 27 nodes from (bx.b, by.b, bz.b), in the order of
// operations of flip.jl:524-533 with the factors shared along rows hoisted:
// wgt = ((wT w_x) w_y) w_z and v = vp + ((c0 d0 + c1 d1) + c2 d2) are the same operations on
// the same values, so the same bits. add(mx, my, mz, momentum, weight) takes them.
template <bool SCALED, class Add>
__device__ inline void p2g_nodes(const BSpline& bx, const BSpline& by, const BSpline& bz, float q0, float q1, float q2,
                                 float vp, float c0, float c1, float c2, float wT, float dx, float scale, Add add) {
    const float wx[3] = {bx.w0, bx.w1, bx.w2}, wy[3] = {by.w0, by.w1, by.w2}, wz[3] = {bz.w0, bz.w1, bz.w2};
    float cd0[3], cd1[3], cd2[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        cd0[m] = c0 * (((float)(bx.b + m) - q0) * dx);
        cd1[m] = c1 * (((float)(by.b + m) - q1) * dx);
        cd2[m] = c2 * (((float)(bz.b + m) - q2) * dx);
    }
#pragma unroll
    for (int my = 0; my < 3; ++my)
#pragma unroll
        for (int mx = 0; mx < 3; ++mx) {
            const float wxy = (wT * wx[mx]) * wy[my], cxy = cd0[mx] + cd1[my];
#pragma unroll
            for (int mz = 0; mz < 3; ++mz) {
                const float wgt = wxy * wz[mz];
                const float m = wgt * (vp + (cxy + cd2[mz]));
                add(mx, my, mz, SCALED ? m * scale : m, wgt);
            }
        }
}
// The same contributions one by one (the rare paths, kept rolled), rounded by tofix.
template <bool SCALED, class Add>
__device__ __forceinline__ void p2g_one_by_one(int a, float qx, float qy, float qz, float vp, float c0, float c1, float c2,
                                               float wT, float dx, float scale, Add add) {
    const float q0 = a == 0 ? qx : qx - 0.5f, q1 = a == 1 ? qy : qy - 0.5f, q2 = a == 2 ? qz : qz - 0.5f;
    const BSpline bx = bspline(q0), by = bspline(q1), bz = bspline(q2);
    const float x0 = bx.w0, x1 = bx.w1, x2 = bx.w2, y0 = by.w0, y1 = by.w1, y2 = by.w2, z0 = bz.w0, z1 = bz.w1, z2 = bz.w2;
#pragma unroll 1
    for (int m = 0; m < 27; ++m) {
        const int mx = m % 3, my = (m / 3) % 3, mz = m / 9;
        const int I = node_at(bx.b, mx), J = node_at(by.b, my), K = node_at(bz.b, mz);
        const float wx = mx == 0 ? x0 : (mx == 1 ? x1 : x2), wy = my == 0 ? y0 : (my == 1 ? y1 : y2),
                    wz = mz == 0 ? z0 : (mz == 1 ? z1 : z2);
        const float wgt = wT * wx * wy * wz;
        const float d0 = ((float)I - q0) * dx, d1 = ((float)J - q1) * dx, d2 = ((float)K - q2) * dx;
        const float mo = wgt * (vp + (c0 * d0 + c1 * d1 + c2 * d2));
        add(I, J, K, tofix(SCALED ? mo * scale : mo), tofix(wgt));
    }
}

// The boxes a workgroup's particles take: over its `act` lanes, the bounds of the first
// nodes of the three components. A component sits at offset 0 along its own axis and 1/2
// along the others; a particle's first nodes at the two, o and h, are o = h or o = h + 1,
// and both follow from o + h without a decrease, so one pair of reductions an axis bounds
// them exactly.
struct NodeBoxes {
    int lo[3], hi[3];   // least and greatest o + h
    bool any;
    __device__ static int first_o(float qo) { return (int)floorf(qo - 0.5f); }              // bspline(qo).b
    __device__ static int first_h(float qo) { return (int)floorf((qo - 0.5f) - 0.5f); }     // bspline(qo - 0.5f).b
    // finite positions near enough for integer arithmetic on their nodes
    __device__ static bool fits(float qo) {
        return fabsf(qo) < 8388608.0f && (unsigned)first_o(qo) - (unsigned)first_h(qo) <= 1u;
    }
    __device__ static int sum(bool act, float qo) { return act ? first_o(qo) + first_h(qo) : 0; }
    __device__ NodeBoxes(bool act, const float (&qo)[3], int* red) {
        const int BIG = 1 << 30;
        int v[6];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int s = sum(act, qo[k]);
            v[k] = act ? s : BIG; v[3 + k] = act ? -s : BIG;
        }
        wg_mins(v, red);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = __builtin_amdgcn_readfirstlane(v[k]);
            hi[k] = -__builtin_amdgcn_readfirstlane(v[3 + k]);
        }
        any = lo[0] != BIG;
    }
    // component a's first nodes along axis k, from their sum: o = ceil(s / 2), h = floor(s / 2)
    __device__ int first(int a, int k) const { return (lo[k] + (a == k)) >> 1; }
    // extents are cut to 1024 so that their product does not overflow (it exceeds any box)
    __device__ int extent(int a, int k) const { return min(((hi[k] + (a == k)) >> 1) - first(a, k) + 3, 1 << 10); }
    __device__ int size(int a) const { return extent(a, 0) * extent(a, 1) * extent(a, 2); }
    __device__ int largest() const { return max(size(0), max(size(1), size(2))); }
    // the nodes of the three components' boxes together
    __device__ void nodes(int first[3], int last[3]) const {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            first[k] = lo[k] >> 1;
            last[k] = ((hi[k] + 1) >> 1) + 2;
        }
    }
};

// The words of LDS for a workgroup's reductions: wg_mins' six, and a wavefront's counts.
constexpr int BOX_RED = 7 * (P2G_THREADS / 64);
// The boxes for the workgroup's `act` lanes: theirs if it has at most `cap`
// nodes, else that of the lanes on one side of the middle of the widest extent, halved
// again until it fits (its least lane is below the middle and its greatest is not: both
// sides hold particles, so this ends). act becomes the lanes of the box. With `left` 0 the low
// side (the deposit, where a particle that no box takes costs global adds); else the side with
// more lanes, and no box (`any` false) where `left` boxes of as many lanes would not take them
// all: a gather's workgroup that leaves any particle to its own reads waits for those once,
// whether they are few or all 256.
__device__ inline NodeBoxes fitting_boxes(bool& act, const float (&qo)[3], int cap, int left, int* red) {
    NodeBoxes B(act, qo, red);
    const int s0 = NodeBoxes::sum(act, qo[0]), s1 = NodeBoxes::sum(act, qo[1]), s2 = NodeBoxes::sum(act, qo[2]);
    int whole = 0;
    while (B.any && B.largest() > cap) {
        const int e0 = B.hi[0] - B.lo[0], e1 = B.hi[1] - B.lo[1], e2 = B.hi[2] - B.lo[2];
        const int k = e0 >= e1 && e0 >= e2 ? 0 : (e1 >= e2 ? 1 : 2);
        const int lo = k == 0 ? B.lo[0] : (k == 1 ? B.lo[1] : B.lo[2]), hi = k == 0 ? B.hi[0] : (k == 1 ? B.hi[1] : B.hi[2]);
        const bool below = (k == 0 ? s0 : (k == 1 ? s1 : s2)) < (lo + hi + 1) >> 1;
        bool low = true;
        if (left > 0) {
            // (NodeBoxes' barriers lie between two uses of these words)
            const int n = (int)(__popcll(__ballot(act)) << 16 | __popcll(__ballot(act && below)));
            if ((threadIdx.x & 63) == 0) red[24 + (threadIdx.x >> 6)] = n;
            __syncthreads();
            const int4 r = *reinterpret_cast<const int4*>(red + 24);
            const int both = __builtin_amdgcn_readfirstlane(r.x + r.y + r.z + r.w), all = both >> 16, under = both & 0xffff;
            if (whole == 0) whole = all;
            low = 2 * under >= all;
            if ((low ? under : all - under) * left < whole) {
                B.any = false;
                break;
            }
        }
        act = act && below == low;
        B = NodeBoxes(act, qo, red);
    }
    return B;
}
// Boxes a workgroup of the deposit takes before what is left goes to global memory node by node.
constexpr int BOX_ROUNDS = 4;

// NodeMap: `index(a, I, J, K)` of a face node, < 0 off the grid (the dense grid's array
// bounds, or no fine block holding the face); `near` / `stage` / `at` the same through a
// table in LDS of TAB entries set up for a box (index itself where the map needs none).
// `ps` gives the positions (fields 0-2).
//
// Bound by its 64-bit LDS adds (54 a particle and component) and by the arithmetic beside
// them. The positions and their index-space coordinates are taken once for the three
// components, and all their boxes from one round of reductions; the rounding to fixed
// point is three instructions. Particles that do not fit one box (a workgroup that
// straddles blocks, or a row that crosses the funnel's ring: 8 % of the workgroups at 5 cm,
// 44 % on the dense grid) take up to BOX_ROUNDS boxes in turn; the global adds of those that
// fitted neither the workgroup's box nor one per wavefront were half the kernel's time. 14.2 M
// particles at 5 cm 3,200 -> 1,850 us (of which the arithmetic issues for 0.8 ms and the LDS
// is busy for 0.7 ms), 1.6 M on 256 x 256 x 128 626 -> 199 us. Boxes of 1,024 and 1,536
// nodes were 3-8 % slower at 5 cm (more rounds), 3,072 and 4,096 2-4 % slower on the dense grid
// (fewer workgroups a CU), as were five workgroups a CU with 1,984.
template <class NodeMap, class Source, int BOX = P2G_BOX>
__global__ __launch_bounds__(P2G_THREADS, 4) void k_p2g_tiled(PView ps, int64_t n, NodeMap map, Source src,
                                                                              P2GArgs A) {
    __shared__ unsigned long long smom[BOX], swt[Source::WEIGHTS ? BOX : 1];
    __shared__ alignas(16) int red[BOX_RED];
    __shared__ int32_t stab[NodeMap::TAB];
    const int64_t p0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * P2G_THREADS;   // neighbouring tiles on one XCD
    // A wavefront takes every eighth particle: particles of one cell (consecutive in cell
    // order) would otherwise add to the same LDS nodes in the same instruction, which
    // serialises the atomics. Integer sums do not depend on the order.
    const int64_t p = p0 + (int64_t)((threadIdx.x & 31) * 8 + (threadIdx.x >> 5));
    const bool live = p < n;
    float qo[3] = {0.0f, 0.0f, 0.0f}, wT = 0.0f;   // index space at offset 0; at 1/2 it is qo - 0.5f
    bool ok = live;
    if (live) {
#pragma unroll
        for (int k = 0; k < 3; ++k) qo[k] = ispace(ps.f[k][p], A.lo[k], A.dx, 0.0f);
        wT = src.weight(p);
    }
    // finite, in-range positions only shape the boxes; others take the direct path
#pragma unroll
    for (int k = 0; k < 3; ++k) ok = ok && NodeBoxes::fits(qo[k]);

    // the workgroup's components: all three, or the launch's y-th (p2g_grid)
    auto takes = [&](int a) { return gridDim.y == 1 || (int)blockIdx.y == a; };
    int large = 0;   // the components left to the direct path
    bool todo = ok;
#pragma unroll 1
    for (int round = 0; round < BOX_ROUNDS; ++round) {
        // (opaque, so that the compiler does not move a particle's 81 contributions, the
        // same in every round, out of the loop and into registers that it does not have)
        asm volatile("" : "+v"(qo[0]), "+v"(qo[1]), "+v"(qo[2]));
        bool act = todo;
        const NodeBoxes B = fitting_boxes(act, qo, BOX, 0, red);
        if (!B.any) break;   // none left (the bounds are the workgroup's)
        todo = todo && !act;
        int lo[3], hi[3];
        B.nodes(lo, hi);
        const typename NodeMap::Near near = map.near(lo, hi);
        map.stage(near, stab);
        auto component = [&](auto axis) __attribute__((always_inline)) {
            constexpr int a = decltype(axis)::value;
            if (!takes(a)) return;   // the whole workgroup
            const int x0 = B.first(a, 0), y0 = B.first(a, 1), z0 = B.first(a, 2);
            const int ex = B.extent(a, 0), ey = B.extent(a, 1), size = B.size(a);
            float vp = 0, c0 = 0, c1 = 0, c2 = 0;
            if (act) src.comp(p, a, vp, c0, c1, c2);
            // a thread clears the entries that it flushed before
            for (int k = threadIdx.x; k < size; k += P2G_THREADS) {
                smom[k] = 0ull;
                if (Source::WEIGHTS) swt[k] = 0ull;
            }
            __syncthreads();
            // A particle whose contributions all lie within 2^18 in magnitude takes the short
            // fixed-point rounding (tofix_near), and others go direct at the end; the
            // adjoint's deposit, whose scale brings most of them past that, takes tofix.
            const float bound = wT * (fabsf(vp) + (fabsf(c0) + fabsf(c1) + fabsf(c2)) * (2.0f * A.dx)) * fabsf(A.scale);
            if (act) {
                const float q0 = a == 0 ? qo[0] : qo[0] - 0.5f, q1 = a == 1 ? qo[1] : qo[1] - 0.5f,
                            q2 = a == 2 ? qo[2] : qo[2] - 0.5f;
                const BSpline bx = bspline(q0), by = bspline(q1), bz = bspline(q2);
                const int sz = ex * ey, l0 = (bx.b - x0) + ex * (by.b - y0) + sz * (bz.b - z0);
                if (Source::SCALED || bound < 262144.0f) {
                    p2g_nodes<Source::SCALED>(bx, by, bz, q0, q1, q2, vp, c0, c1, c2, wT, A.dx, A.scale,
                                              [&](int mx, int my, int mz, float m, float w) {
                                                  const int l = l0 + mx + ex * my + sz * mz;
                                                  atomicAdd(&smom[l], Source::SCALED ? tofix(m) : tofix_near(m));
                                                  if (Source::WEIGHTS) atomicAdd(&swt[l], tofix_near(w));
                                              });
                } else {
                    large |= 1 << a;
                }
            }
            __syncthreads();
            const BoxIndex at(ex, ey);
            for (int k = threadIdx.x; k < size; k += P2G_THREADS) {
                const unsigned long long m = smom[k], w = Source::WEIGHTS ? swt[k] : 0ull;
                if (m == 0ull && w == 0ull) continue;
                int i, j, kk;
                at.at(k, i, j, kk);
                auto idx = map.at(near, stab, a, x0 + i, y0 + j, z0 + kk);
                if (idx >= 0) {
                    if (m) atomicAdd(&A.mom[a][idx], m);
                    if (w) atomicAdd(&A.wt[a][idx], w);
                }
            }
        };
        component(std::integral_constant<int, 0>{});
        component(std::integral_constant<int, 1>{});
        component(std::integral_constant<int, 2>{});
    }
    if (todo || (live && !ok)) large = 7;   // far apart, not finite or far off the grid
    if (large) {
#pragma unroll 1
        for (int a = 0; a < 3; ++a) {
            if (!takes(a) || !(large >> a & 1)) continue;
            float vp, c0, c1, c2;
            src.comp(p, a, vp, c0, c1, c2);
            p2g_one_by_one<Source::SCALED>(a, qo[0], qo[1], qo[2], vp, c0, c1, c2, wT, A.dx, A.scale,
                                           [&](int I, int J, int K, unsigned long long m, unsigned long long w) {
                                               auto idx = map.index(a, I, J, K);
                                               if (idx >= 0) {
                                                   atomicAdd(&A.mom[a][idx], m);
                                                   if (Source::WEIGHTS) atomicAdd(&A.wt[a][idx], w);
                                               }
                                           });
        }
    }
}

// A workgroup per 256 particles; while those leave half of the chip's 1,024 places (four
// workgroups on each of 256 CUs) idle, one per component: the deposit of 42,000 particles
// (166 workgroups) is one workgroup's chain of clear, add and flush, three times over.
inline dim3 p2g_grid(int64_t n) {
    const unsigned g = cdiv(n, P2G_THREADS);
    return dim3(g, g <= 512 ? 3 : 1);
}

// flip.jl:1226-1244 g2p_kernel!: a workgroup's 256 particles gather each component from a
// box of faces staged in LDS, loaded once per box node instead of once per particle and
// node; several boxes in turn as in the deposit, and what is left reads the faces directly.
// Every path takes the flags' sum and the value and affine row over the 27 nodes in the
// reference's order (gather, sflip.jl:193-215 finegather), so the same bits.
//
// NodeMap::boxes() is how many a workgroup takes. Particles come in cell order from a step,
// where several boxes pay, but a caller may set them in any: 98,000 (27 in cell order) and 1.6 M
// (112) in random order on the sparse basin take 59 and 1,100 us, as many as without boxes,
// and took 115 and 1,350 with up to four boxes whatever those held.
//
// NodeMap as k_p2g_tiled's; HOLES: a node may be missing (index < 0) and is skipped. In a
// box, a missing node's flag is -1 and its value 0 and it adds zero products instead: the
// sums start at +0 and are never -0, so adding a zero leaves them bit for bit as skipping.
// Where every face of the box is there and valid (most boxes: the flow is extrapolated past
// the band), the flags' sum is that of the weights, 1 to a few ulp, and is not taken. (A bit
// mask per row of the other boxes, so that a particle off their invalid faces skips it too,
// cost more than it saved: 892 -> 943 us for 14.2 M particles.) Bound by its arithmetic (about
// 2,300 vector instructions a wavefront): 14.2 M particles at 5 cm 1,207 -> 892 us, 1.6 M on
// 256 x 256 x 128 161 -> 135 us against the kernels that staged (value, flag) pairs and sent
// what did not fit one box to global memory.
struct G2PFaces {
    const float* u[3];
    const uint8_t* f[3];
};
constexpr int G2P_BOX = 2048;   // 16 KB
template <class NodeMap>
__global__ __launch_bounds__(P2G_THREADS, 4) void k_g2p_tiled(PView ps, int64_t n, NodeMap map, float lo0, float lo1, float lo2,
                                                              float dx, G2PFaces F, float dt, float gravity) {
    __shared__ float sval[G2P_BOX], sflag[G2P_BOX];
    __shared__ alignas(16) int red[BOX_RED];
    __shared__ int32_t stab[NodeMap::TAB];
    const int64_t p = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * P2G_THREADS + threadIdx.x;   // neighbouring tiles on one XCD
    const bool live = p < n;
    float qo[3] = {0.0f, 0.0f, 0.0f};   // index space at offset 0; at 1/2 it is qo - 0.5f
    if (live) {
        qo[0] = ispace(ps.f[0][p], lo0, dx, 0.0f);
        qo[1] = ispace(ps.f[1][p], lo1, dx, 0.0f);
        qo[2] = ispace(ps.f[2][p], lo2, dx, 0.0f);
    }
    const float c4 = __fdiv_rn(4.0f, dx * dx);
    // v and the rows (fields 3..14) from the three components' sums, stored unconditionally,
    // so no store's target depends on a divergent branch (see k_dense_spawn)
    auto finish = [&](bool reached, float (&rec)[12]) {
        if (!reached) {
            rec[0] = ps.f[3][p];
            rec[1] = ps.f[4][p];
            rec[2] = ps.f[5][p] - gravity * dt;
#pragma unroll
            for (int f = 3; f < 12; ++f) rec[f] = 0.0f;
        }
#pragma unroll
        for (int f = 0; f < 12; ++f) ps.f[3 + f][p] = rec[f];
    };

    bool todo = live && NodeBoxes::fits(qo[0]) && NodeBoxes::fits(qo[1]) && NodeBoxes::fits(qo[2]);
    const bool far = live && !todo;
#pragma unroll 1
    for (int left = NodeMap::boxes(); left > 0; --left) {
        asm volatile("" : "+v"(qo[0]), "+v"(qo[1]), "+v"(qo[2]));   // as in k_p2g_tiled: nothing moved out of the loop
        bool act = todo;
        const NodeBoxes B = fitting_boxes(act, qo, G2P_BOX, left, red);
        if (!B.any) break;
        todo = todo && !act;
        int lo[3], hi[3];
        B.nodes(lo, hi);
        const typename NodeMap::Near near = map.near(lo, hi);
        map.stage(near, stab);
        __syncthreads();
        float rec[12];
        bool reached = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int x0 = B.first(a, 0), y0 = B.first(a, 1), z0 = B.first(a, 2);
            const int ex = B.extent(a, 0), ey = B.extent(a, 1), size = B.size(a);
            const BoxIndex at(ex, ey);
            bool good = true;
            for (int k = threadIdx.x; k < size; k += P2G_THREADS) {
                int i, j, kk;
                at.at(k, i, j, kk);
                const auto idx = map.at(near, stab, a, x0 + i, y0 + j, z0 + kk);
                const float val = idx >= 0 ? F.u[a][idx] : 0.0f, flag = idx >= 0 ? (float)F.f[a][idx] : -1.0f;
                sval[k] = val;
                sflag[k] = flag;
                good = good && flag == 1.0f;
            }
            const bool whole = __syncthreads_and(good);
            if (act) {
                const float q0 = a == 0 ? qo[0] : qo[0] - 0.5f, q1 = a == 1 ? qo[1] : qo[1] - 0.5f,
                            q2 = a == 2 ? qo[2] : qo[2] - 0.5f;
                const BSpline bx = bspline(q0), by = bspline(q1), bz = bspline(q2);
                const float wx[3] = {bx.w0, bx.w1, bx.w2}, wy[3] = {by.w0, by.w1, by.w2}, wz[3] = {bz.w0, bz.w1, bz.w2};
                float d0[3], d1[3], d2[3];
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                    d0[m] = (float)(bx.b + m) - q0;
                    d1[m] = (float)(by.b + m) - q1;
                    d2[m] = (float)(bz.b + m) - q2;
                }
                const int l0 = (bx.b - x0) + ex * ((by.b - y0) + ey * (bz.b - z0));
                float f_ = 0.0f, v_ = 0.0f, s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
                auto sum = [&](auto flags) {
#pragma unroll
                    for (int mz = 0; mz < 3; ++mz)
#pragma unroll
                        for (int my = 0; my < 3; ++my) {
                            const int l = l0 + ex * (my + ey * mz);
#pragma unroll
                            for (int mx = 0; mx < 3; ++mx) {
                                float wgt = (wx[mx] * wy[my]) * wz[mz];
                                if (flags) {
                                    const float fl = sflag[l + mx];
                                    if (NodeMap::HOLES) wgt = fl >= 0.0f ? wgt : 0.0f;
                                    f_ += wgt * fl;
                                }
                                const float t = wgt * sval[l + mx];
                                v_ += t;
                                s0 += (t * d0[mx]) * dx;
                                s1 += (t * d1[my]) * dx;
                                s2 += (t * d2[mz]) * dx;
                            }
                        }
                };
                if (whole) {
                    sum(std::false_type{});
                } else {
                    sum(std::true_type{});
                    reached = reached && f_ > 0.999f;
                }
                rec[a] = v_; rec[3 + 3 * a] = s0 * c4; rec[4 + 3 * a] = s1 * c4; rec[5 + 3 * a] = s2 * c4;
            }
            __syncthreads();   // the box is reused
        }
        if (act) finish(reached, rec);
    }
    if (todo || far) {   // far apart, not finite or far off the grid
        // (a component at a time in a loop, its sums kept in the box, which is free now: the
        // nodes' reads of all three together would not fit the registers)
        static_assert(6 * P2G_THREADS <= G2P_BOX, "the sums of a thread fit the box");
        auto sums = [&](int f) -> float& {
            return f < 6 ? sval[f * P2G_THREADS + threadIdx.x] : sflag[(f - 6) * P2G_THREADS + threadIdx.x];
        };
        bool reached = true;
#pragma unroll 1
        for (int a = 0; a < 3; ++a) {
            const float* __restrict__ u = a == 0 ? F.u[0] : (a == 1 ? F.u[1] : F.u[2]);
            const uint8_t* __restrict__ fl = a == 0 ? F.f[0] : (a == 1 ? F.f[1] : F.f[2]);
            const float q0 = a == 0 ? qo[0] : qo[0] - 0.5f, q1 = a == 1 ? qo[1] : qo[1] - 0.5f, q2 = a == 2 ? qo[2] : qo[2] - 0.5f;
            const BSpline bx = bspline(q0), by = bspline(q1), bz = bspline(q2);
            float f_ = 0.0f, v_ = 0.0f, s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
            auto nodes = [&](auto each) {
#pragma unroll
                for (int mz = 0; mz < 3; ++mz)
#pragma unroll
                    for (int my = 0; my < 3; ++my)
#pragma unroll
                        for (int mx = 0; mx < 3; ++mx) {
                            const int I = node_at(bx.b, mx), J = node_at(by.b, my), K = node_at(bz.b, mz);
                            const auto idx = map.index(a, I, J, K);
                            if (!NodeMap::HOLES || idx >= 0) each(idx, pick(bx, mx) * pick(by, my) * pick(bz, mz), I, J, K);
                        }
            };
            auto flagsum = [&](auto idx, float wgt, int, int, int) { f_ += wgt * (float)fl[idx]; };
            auto sum = [&](auto idx, float wgt, int I, int J, int K) {
                const float t = wgt * u[idx];
                v_ += t;
                s0 += (t * ((float)I - q0)) * dx;
                s1 += (t * ((float)J - q1)) * dx;
                s2 += (t * ((float)K - q2)) * dx;
            };
            if (NodeMap::HOLES) {   // (looking a node's block up costs more than a read)
                nodes([&](auto idx, float wgt, int I, int J, int K) { flagsum(idx, wgt, I, J, K); sum(idx, wgt, I, J, K); });
            } else {
                nodes(flagsum);
                nodes(sum);
            }
            reached = reached && f_ > 0.999f;
            sums(a) = v_;
            sums(3 + 3 * a) = s0 * c4; sums(4 + 3 * a) = s1 * c4; sums(5 + 3 * a) = s2 * c4;
        }
        float rec[12];
#pragma unroll
        for (int f = 0; f < 12; ++f) rec[f] = sums(f);
        finish(reached, rec);
    }
}

// The particles' level-set splat (flip.jl:539-560) tiled the same way: a workgroup's 256
// particles take their minimum over a box of cells in LDS (several boxes in turn as in the
// deposit), then each touched cell of the box takes one global atomic min. The box holds the
// squared distances' bits: the root, the particle's radius taken off it and the order key
// are non-decreasing, so the minimum goes through them once a cell instead of 27 times a
// particle. Minimum is order-independent, so the result is the direct splat's bit for bit.
// CellMap: `index(I, J, K)` of a cell (< 0 off the grid or outside the fine blocks), `near`
// / `stage` / `at` as k_p2g_tiled's. 14.2 M particles at 5 cm 629 -> 314 us, 1.6 M on 256 x
// 256 x 128 85 -> 45 us.
constexpr int SPLAT_BOX = 4096;   // 16 KB

template <class CellMap>
__global__ __launch_bounds__(P2G_THREADS) void k_splat_tiled(PView ps, int64_t n, CellMap map, float lo0, float lo1, float lo2,
                                                            float dx, float dt, int32_t* __restrict__ phip) {
    __shared__ int32_t box[SPLAT_BOX];
    __shared__ alignas(16) int red[BOX_RED];
    __shared__ int32_t stab[CellMap::TAB];
    const int64_t p0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * P2G_THREADS;   // neighbouring tiles on one XCD
    // every eighth particle per lane group, as in k_p2g_tiled
    const int64_t p = p0 + (int64_t)((threadIdx.x & 31) * 8 + (threadIdx.x >> 5));
    const bool live = p < n;
    float xp = 0, yp = 0, zp = 0;
    // the cells ci - 1 .. ci + 1 are the nodes ci .. ci + 2 of a box one lower: the boxes of
    // an index-space coordinate ci + 1 (first_o = first_h = ci)
    float qo[3] = {0.0f, 0.0f, 0.0f};
    if (live) {   // the particle's advanced position and cell
        const float vx = ps.f[3][p], vy = ps.f[4][p], vz = ps.f[5][p];
        const float sp = sqrtf(vx * vx + vy * vy + vz * vz);
        const float s = ps.f[15][p] + ahead(strength(sp, dt, dx)) * dt;
        xp = ps.f[0][p] + s * vx; yp = ps.f[1][p] + s * vy; zp = ps.f[2][p] + s * vz;
        qo[0] = floorf(__fdiv_rn(xp - lo0, dx)) + 1.0f;
        qo[1] = floorf(__fdiv_rn(yp - lo1, dx)) + 1.0f;
        qo[2] = floorf(__fdiv_rn(zp - lo2, dx)) + 1.0f;
    }
    const int ci = (int)(qo[0] - 1.0f), cj = (int)(qo[1] - 1.0f), ck = (int)(qo[2] - 1.0f);
    const float radius = 0.5f * dx;
    float sx[3], sy[3], sz[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const float ex_ = lo0 + ((float)node_at(ci, m - 1) + 0.5f) * dx - xp;
        const float ey_ = lo1 + ((float)node_at(cj, m - 1) + 0.5f) * dx - yp;
        const float ez_ = lo2 + ((float)node_at(ck, m - 1) + 0.5f) * dx - zp;
        sx[m] = ex_ * ex_; sy[m] = ey_ * ey_; sz[m] = ez_ * ez_;
    }
    bool todo = live && NodeBoxes::fits(qo[0]) && NodeBoxes::fits(qo[1]) && NodeBoxes::fits(qo[2]);
    const bool far = live && !todo;
#pragma unroll 1
    for (int round = 0; round < BOX_ROUNDS; ++round) {
        bool act = todo;
        const NodeBoxes B = fitting_boxes(act, qo, SPLAT_BOX, 0, red);
        if (!B.any) break;
        todo = todo && !act;
        const int x0 = (B.lo[0] >> 1) - 1, y0 = (B.lo[1] >> 1) - 1, z0 = (B.lo[2] >> 1) - 1;
        const int ex = ((B.hi[0] - B.lo[0]) >> 1) + 3, ey = ((B.hi[1] - B.lo[1]) >> 1) + 3, ez = ((B.hi[2] - B.lo[2]) >> 1) + 3;
        const int lo[3] = {x0, y0, z0}, hi[3] = {x0 + ex - 1, y0 + ey - 1, z0 + ez - 1};
        const typename CellMap::Near near = map.near(lo, hi);
        map.stage(near, stab);
        const int V = ex * ey * ez;
        // a thread clears the entries that it flushed before
        for (int k = threadIdx.x; k < V; k += P2G_THREADS) box[k] = 0x7fffffff;
        __syncthreads();
        if (act) {
            const int l0 = (ci - 1 - x0) + ex * ((cj - 1 - y0) + ey * (ck - 1 - z0));
#pragma unroll
            for (int mj = 0; mj < 3; ++mj)
#pragma unroll
                for (int mi = 0; mi < 3; ++mi) {
                    const float sxy = sx[mi] + sy[mj];
#pragma unroll
                    for (int mk = 0; mk < 3; ++mk)
                        atomicMin(&box[l0 + mi + ex * (mj + ey * mk)], __float_as_int(sxy + sz[mk]));
                }
        }
        __syncthreads();
        const BoxIndex at(ex, ey);
        for (int k = threadIdx.x; k < V; k += P2G_THREADS) {
            const int32_t v = box[k];
            if (v == 0x7fffffff) continue;
            int i, j, kk;
            at.at(k, i, j, kk);
            auto idx = map.at(near, stab, x0 + i, y0 + j, z0 + kk);
            if (idx >= 0) atomicMin(&phip[idx], orderkey(sqrtf(__int_as_float(v)) - radius));
        }
    }
    if (todo || far) {   // left over: far apart, not finite or far off the grid
#pragma unroll
        for (int mk = 0; mk < 3; ++mk)
#pragma unroll
            for (int mj = 0; mj < 3; ++mj)
#pragma unroll
                for (int mi = 0; mi < 3; ++mi) {
                    auto idx = map.index(node_at(ci, mi - 1), node_at(cj, mj - 1), node_at(ck, mk - 1));
                    if (idx >= 0) atomicMin(&phip[idx], orderkey(sqrtf(sx[mi] + sy[mj] + sz[mk]) - radius));
                }
    }
}

// ─── adjoints of the transfers (no counterpart in the reference) ─────────────
// With positions, lags, level set and weights fixed, P2G is linear in the particles' v
// and APIC rows and G2P in the face velocities. The G2P adjoint deposits through
// k_p2g_tiled with this source; the P2G adjoint gathers with k_p2g_adj_gather.

// The G2P adjoint's particle side: the output cotangents, the rows times the gather's
// 4 / dx^2, for the particles that took the grid's velocity (the others deposit 0).
struct G2PAdjSource {
    static constexpr bool WEIGHTS = false, SCALED = true;
    const float* pb[12];
    const uint8_t* reached;
    float cs;
    __device__ float weight(int64_t p) const { return reached[p] ? 1.0f : 0.0f; }
    __device__ void comp(int64_t p, int a, float& v, float& c0, float& c1, float& c2) const {
        if (!reached[p]) { v = c0 = c1 = c2 = 0.0f; return; }
        v = pb[a][p];
        c0 = pb[3 + 3 * a][p] * cs; c1 = pb[4 + 3 * a][p] * cs; c2 = pb[5 + 3 * a][p] * cs;
    }
};
struct PB12 { float* f[12]; };

// The workgroup's largest v (floats >= 0 by their bits) into *bound: an atomic only from a
// workgroup that raises it.
__device__ inline void wg_raise(float m, int* bound, int* red) {
    const int v = -wave_min(-__float_as_int(m));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int w = max(max(red[0], red[1]), max(red[2], red[3]));
        if (w > __hip_atomic_load(bound, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(bound, w);
    }
}

// A workgroup's 256 particles over boxes of faces in LDS, component by component, as
// k_g2p_tiled: stage(k, idx) puts face idx (< 0: none there) of component a at k in the box;
// take(a, k0, ex, exy, bx, by, bz, q0, q1, q2) reads the box for a particle whose first node
// is at k0; done() follows a particle's three components. left(a, ...) is a component of a
// particle that no box took (or that is not to be boxed).
template <int CAP, bool BOXED, class NodeMap, class Stage, class Take, class Left, class Done>
__device__ __forceinline__ void over_boxes(bool live, bool boxed, float (&qo)[3], const NodeMap& map, int* red, int32_t* stab,
                                           Stage stage, Take take, Left left, Done done) {
    bool todo = live && boxed && NodeBoxes::fits(qo[0]) && NodeBoxes::fits(qo[1]) && NodeBoxes::fits(qo[2]);
    const bool far = live && !todo;
#pragma unroll 1
    for (int left = BOXED ? NodeMap::boxes() : 0; left > 0; --left) {
        asm volatile("" : "+v"(qo[0]), "+v"(qo[1]), "+v"(qo[2]));   // as in k_p2g_tiled: nothing moved out of the loop
        bool act = todo;
        const NodeBoxes B = fitting_boxes(act, qo, CAP, left, red);
        if (!B.any) break;
        todo = todo && !act;
        int lo[3], hi[3];
        B.nodes(lo, hi);
        const typename NodeMap::Near near = map.near(lo, hi);
        map.stage(near, stab);
        __syncthreads();
        auto component = [&](auto axis) __attribute__((always_inline)) {
            constexpr int a = decltype(axis)::value;
            const int x0 = B.first(a, 0), y0 = B.first(a, 1), z0 = B.first(a, 2);
            const int ex = B.extent(a, 0), ey = B.extent(a, 1), size = B.size(a);
            const BoxIndex at(ex, ey);
            for (int k = threadIdx.x; k < size; k += P2G_THREADS) {
                int i, j, kk;
                at.at(k, i, j, kk);
                stage(axis, k, map.at(near, stab, a, x0 + i, y0 + j, z0 + kk));
            }
            __syncthreads();
            if (act) {
                const float q0 = a == 0 ? qo[0] : qo[0] - 0.5f, q1 = a == 1 ? qo[1] : qo[1] - 0.5f,
                            q2 = a == 2 ? qo[2] : qo[2] - 0.5f;
                const BSpline bx = bspline(q0), by = bspline(q1), bz = bspline(q2);
                take(axis, (bx.b - x0) + ex * ((by.b - y0) + ey * (bz.b - z0)), ex, ex * ey, bx, by, bz, q0, q1, q2);
            }
            __syncthreads();   // the box is reused
        };
        component(std::integral_constant<int, 0>{});
        component(std::integral_constant<int, 1>{});
        component(std::integral_constant<int, 2>{});
        if (act) done();
    }
    if (todo || far) {   // far apart, not finite or far off the grid
        auto component = [&](auto axis) __attribute__((always_inline)) {
            constexpr int a = decltype(axis)::value;
            const float q0 = a == 0 ? qo[0] : qo[0] - 0.5f, q1 = a == 1 ? qo[1] : qo[1] - 0.5f, q2 = a == 2 ? qo[2] : qo[2] - 0.5f;
            left(axis, bspline(q0), bspline(q1), bspline(q2), q0, q1, q2);
        };
        component(std::integral_constant<int, 0>{});
        component(std::integral_constant<int, 1>{});
        component(std::integral_constant<int, 2>{});
        done();
    }
}

// Which particles took the grid's velocity in G2P (the three flag sums > 0.999, in the
// gather's order of operations), and the largest contribution one of them makes to a node,
// as float bits (for the deposit's scale). 1.6 M particles at 15 cm 176 -> 78 us against
// reading the flags from global memory node by node.
template <class NodeMap>
__global__ __launch_bounds__(P2G_THREADS, 6) void k_g2p_adj_reached(PView ps, int64_t n, NodeMap map, float lo0, float lo1, float lo2,
                                                                 float dx, G2PFaces F, uint8_t* __restrict__ reached, PB12 pb,
                                                                 int* __restrict__ bound) {
    __shared__ float sflag[G2P_BOX];
    __shared__ alignas(16) int red[BOX_RED];
    __shared__ int32_t stab[NodeMap::TAB];
    const int64_t p = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * P2G_THREADS + threadIdx.x;
    const bool live = p < n;
    float qo[3] = {0.0f, 0.0f, 0.0f}, m = 0.0f;
    if (live) {
        qo[0] = ispace(ps.f[0][p], lo0, dx, 0.0f);
        qo[1] = ispace(ps.f[1][p], lo1, dx, 0.0f);
        qo[2] = ispace(ps.f[2][p], lo2, dx, 0.0f);
    }
    bool ok = true;
    over_boxes<G2P_BOX, true>(
        live, true, qo, map, red, stab,
        [&](auto axis, int k, auto idx) {
            constexpr int a = decltype(axis)::value;
            sflag[k] = idx >= 0 ? (float)F.f[a][idx] : -1.0f;
        },
        [&](auto, int k0, int ex, int exy, const BSpline& bx, const BSpline& by, const BSpline& bz, float, float, float) {
            const float wx[3] = {bx.w0, bx.w1, bx.w2}, wy[3] = {by.w0, by.w1, by.w2}, wz[3] = {bz.w0, bz.w1, bz.w2};
            float f = 0.0f;
#pragma unroll
            for (int mz = 0; mz < 3; ++mz)
#pragma unroll
                for (int my = 0; my < 3; ++my)
#pragma unroll
                    for (int mx = 0; mx < 3; ++mx) {
                        const float fl = sflag[k0 + mx + ex * my + exy * mz];
                        const float wgt = (wx[mx] * wy[my]) * wz[mz];
                        f += (NodeMap::HOLES && fl < 0.0f ? 0.0f : wgt) * fl;
                    }
            ok = ok && f > 0.999f;
        },
        [&](auto axis, const BSpline& bx, const BSpline& by, const BSpline& bz, float, float, float) {
            constexpr int a = decltype(axis)::value;
            float f = 0.0f;
#pragma unroll 1
            for (int r = 0; r < 9; ++r) {   // a row's three nodes are read together
                const int my = r % 3, mz = r / 3;
                float flag[3];
#pragma unroll
                for (int mx = 0; mx < 3; ++mx) {
                    const auto idx = map.index(a, node_at(bx.b, mx), node_at(by.b, my), node_at(bz.b, mz));
                    flag[mx] = !NodeMap::HOLES || idx >= 0 ? (float)F.f[a][idx] : -1.0f;
                }
#pragma unroll
                for (int mx = 0; mx < 3; ++mx)
                    if (!NodeMap::HOLES || flag[mx] >= 0.0f) f += pick(bx, mx) * pick(by, my) * pick(bz, mz) * flag[mx];
            }
            ok = ok && f > 0.999f;
        },
        [&] {
            reached[p] = ok ? 1 : 0;
            if (!ok) return;
            const float cd = 6.0f / dx;   // |row . d| <= (4 / dx^2)(1.5 dx) sum |row|
#pragma unroll
            for (int a = 0; a < 3; ++a)
                m = fmaxf(m, fabsf(pb.f[a][p]) +
                                 cd * (fabsf(pb.f[3 + 3 * a][p]) + fabsf(pb.f[4 + 3 * a][p]) + fabsf(pb.f[5 + 3 * a][p])));
            if (!(m <= 3.0e38f)) m = 3.0e38f;
        });
    wg_raise(m, bound, red);
}

// The P2G adjoint's particle part: each particle gathers the momentum cotangents s of the
// nodes it deposited to (NodeMap as k_p2g_tiled's), with the deposit's weights and
// offsets, and adds them to its v and row cotangents. 1.6 M particles at 15 cm 310 -> 132 us
// against reading the faces from global memory node by node.
struct AdjFaces { const float* s[3]; };
template <class NodeMap>
__global__ __launch_bounds__(P2G_THREADS) void k_p2g_adj_gather(PView ps, int64_t n, NodeMap map, float lo0, float lo1, float lo2,
                                                                float dx, float dt, AdjFaces S, PB12 pb) {
    __shared__ float sval[G2P_BOX];
    __shared__ alignas(16) int red[BOX_RED];
    __shared__ int32_t stab[NodeMap::TAB];
    const uint32_t tile = NodeMap::ADJ_BOXED ? xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t p = (int64_t)tile * P2G_THREADS + threadIdx.x;
    const bool live = p < n;
    float qo[3] = {0.0f, 0.0f, 0.0f}, wT = 0.0f;
    if (live) {
        qo[0] = ispace(ps.f[0][p], lo0, dx, 0.0f);
        qo[1] = ispace(ps.f[1][p], lo1, dx, 0.0f);
        qo[2] = ispace(ps.f[2][p], lo2, dx, 0.0f);
        wT = temporal(ps.f[15][p], dt);
    }
    over_boxes<G2P_BOX, NodeMap::ADJ_BOXED>(
        live, wT == wT, qo, map, red, stab,
        [&](auto axis, int k, auto idx) {   // (0 where there is no node: its terms vanish, unless wT is NaN)
            constexpr int a = decltype(axis)::value;
            sval[k] = idx >= 0 ? S.s[a][idx] : 0.0f;
        },
        [&](auto axis, int k0, int ex, int exy, const BSpline& bx, const BSpline& by, const BSpline& bz, float q0, float q1,
            float q2) {
            constexpr int a = decltype(axis)::value;
            const float wx[3] = {bx.w0, bx.w1, bx.w2}, wy[3] = {by.w0, by.w1, by.w2}, wz[3] = {bz.w0, bz.w1, bz.w2};
            float d0[3], d1[3], d2[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                d0[m] = ((float)(bx.b + m) - q0) * dx;
                d1[m] = ((float)(by.b + m) - q1) * dx;
                d2[m] = ((float)(bz.b + m) - q2) * dx;
            }
            float v = 0.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
#pragma unroll
            for (int mz = 0; mz < 3; ++mz)
#pragma unroll
                for (int my = 0; my < 3; ++my)
#pragma unroll
                    for (int mx = 0; mx < 3; ++mx) {
                        const float t = (((wT * wx[mx]) * wy[my]) * wz[mz]) * sval[k0 + mx + ex * my + exy * mz];
                        v += t;
                        c0 += t * d0[mx];
                        c1 += t * d1[my];
                        c2 += t * d2[mz];
                    }
            pb.f[a][p] += v;
            pb.f[3 + 3 * a][p] += c0; pb.f[4 + 3 * a][p] += c1; pb.f[5 + 3 * a][p] += c2;
        },
        [&](auto axis, const BSpline& bx, const BSpline& by, const BSpline& bz, float q0, float q1, float q2) {
            constexpr int a = decltype(axis)::value;
            float v = 0.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
            constexpr int PLANES = NodeMap::ADJ_BOXED ? 1 : 3;   // whose nodes are read together
#pragma unroll PLANES
            for (int mz = 0; mz < 3; ++mz) {
                const int K = node_at(bz.b, mz);
                float val[9];
                int in = 0;
#pragma unroll
                for (int m = 0; m < 9; ++m) {
                    const auto idx = map.index(a, node_at(bx.b, m % 3), node_at(by.b, m / 3), K);
                    in |= (int)(idx >= 0) << m;
                    val[m] = idx >= 0 ? S.s[a][idx] : 0.0f;
                }
#pragma unroll
                for (int m = 0; m < 9; ++m) {
                    if (!(in >> m & 1)) continue;
                    const int mx = m % 3, my = m / 3;
                    const float t = wT * pick(bx, mx) * pick(by, my) * pick(bz, mz) * val[m];
                    v += t;
                    c0 += t * (((float)node_at(bx.b, mx) - q0) * dx);
                    c1 += t * (((float)node_at(by.b, my) - q1) * dx);
                    c2 += t * (((float)K - q2) * dx);
                }
            }
            pb.f[a][p] += v;
            pb.f[3 + 3 * a][p] += c0; pb.f[4 + 3 * a][p] += c1; pb.f[5 + 3 * a][p] += c2;
        },
        [] {});
}

}  // namespace mael
