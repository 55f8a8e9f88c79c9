// The small levels of the dense basin's V-cycle (flip.jl:838-1014) in few launches: a
// level's way down (red-black Gauss-Seidel from zero, two sweeps, the residual and its
// restriction) in one, its way up (prolongation and two sweeps) in one, and the last two
// levels with the coarsest solve in one workgroup.
//
// A colour pass of a small level is a launch and a memory round trip around little work
// (2.6 us at 2,048 cells as at 131,072). Here a workgroup holds a tile with a halo as deep
// as its chain of passes in LDS and computes its neighbours' cells in the halo again, with the
// operations of the kernels that take a launch a pass (pressure.hip) in their order, so the
// values do not change. A row is its diagonal alone (-1 here off the LIQUID cells): the
// pressure is 0 off them and off the grid, so the neighbours' sum takes all six, adding
// zeros where those kernels skip a neighbour.
//
// Bound by launch and LDS latency, and past the chip's 256 CUs by the halo's repeated cells
// (18^3 rows for a tile of 8^3 down, 16^3 up). Levels of 131,072 and 16,384 cells take 9.0 us
// down and 8.1 us up, against 21 and 14 us in six and five launches; the last two (2,048 and
// 256 cells) 21.8 us, against 58 us in twelve. A 64x64x32 solve 1,430 -> 707 us.
#pragma once
#include "dense.hpp"
#include "quotient.hpp"
#include <type_traits>

namespace mael {

constexpr int RB = 8, RB_THREADS = 1024;   // tiles of RB^3 cells

// A cell's diagonal as the rows here take it.
__device__ inline float rb_diag(const float* __restrict__ dg, const uint8_t* __restrict__ types, size_t l) {
    const float d = dg[l];
    return types[l] == LIQUID ? d : -1.0f;
}

// A tile and H cells round it in LDS. The cells of one colour are numbered in rows of
// pairs, and thread t has those numbered t, t + RB_THREADS, ...
template <int H> struct RBTile {
    static constexpr int R = RB + 2 * H, N = R * R * R, HALF = N / 2, M = (HALF + RB_THREADS - 1) / RB_THREADS;
    __device__ static int place(int colour, int m, int& i, int& j, int& k) {
        const int e = (int)threadIdx.x + m * RB_THREADS, r = e / (R / 2);
        j = r % R; k = r / R;
        // tiles start at even cells: the colour (i' + j' + k' + 1) & 1 of the grid's cell
        // i' = first + i - H, ... is that of i + j + k + H + 1
        i = 2 * (e % (R / 2)) + ((colour + j + k + H + 1) & 1);
        return i + R * (j + R * k);
    }
    __device__ static int ring(int i, int j, int k) { return min(min(min(i, R - 1 - i), min(j, R - 1 - j)), min(k, R - 1 - k)); }
    // the six neighbours of an inner cell in the order of nb6
    __device__ static float sum(const float* v, int e) {
        float s = 0.0f;
        s += v[e + 1]; s += v[e - 1]; s += v[e + R]; s += v[e - R]; s += v[e + R * R]; s += v[e - R * R];
        return s;
    }
};
// The tile's first cell.
__device__ inline int3 rb_tile(uint32_t g, int3 n) {
    const uint32_t nx = (uint32_t)(n.x + RB - 1) / RB, ny = (uint32_t)(n.y + RB - 1) / RB;
    return make_int3((int)(g % nx) * RB, (int)((g / nx) % ny) * RB, (int)(g / (nx * ny)) * RB);
}
__device__ inline bool rb_in(int I, int J, int K, int3 n) { return I >= 0 && J >= 0 && K >= 0 && I < n.x && J < n.y && K < n.z; }
__device__ inline size_t rb_lin(int I, int J, int K, int3 n) { return (size_t)I + (size_t)n.x * ((size_t)J + (size_t)n.y * K); }

// Down, two sweeps: x from b, and the coarser level's right-hand side bc (tc: its types). The restriction reads the residual one cell past the tile, the residual x one
// further, and each pass one further again.
constexpr int RB_DOWN = 5, RB_UP = 4;
__global__ __launch_bounds__(RB_THREADS) void k_rbdown(float* __restrict__ x, float* __restrict__ bc, const float* __restrict__ b,
                                                       const float* __restrict__ dg, const uint8_t* __restrict__ tf,
                                                       const uint8_t* __restrict__ tc, int3 n, int3 nc) {
    using T = RBTile<RB_DOWN>;
    __shared__ float v[T::N], rs[T::N];
    const int3 o = rb_tile(blockIdx.x, n);
    float bv[2][T::M], dv[2][T::M];
    int i, j, k;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            T::place(c, m, i, j, k);
            const int I = o.x + i - RB_DOWN, J = o.y + j - RB_DOWN, K = o.z + k - RB_DOWN;
            const bool in = k < T::R && rb_in(I, J, K, n);
            const size_t l = in ? rb_lin(I, J, K, n) : 0;
            bv[c][m] = in ? b[l] : 0.0f;
            dv[c][m] = in ? rb_diag(dg, tf, l) : -1.0f;
        }
    // colour 0 from zero (flip.jl:964-973), the others 0
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            const int e = T::place(c, m, i, j, k);
            if (k < T::R) v[e] = c == 0 && dv[c][m] > 0.0f ? __fdiv_rn(bv[c][m], dv[c][m]) : 0.0f;
        }
    __syncthreads();
    auto pass = [&](auto colour, int inside) {
        constexpr int c = decltype(colour)::value;
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            const int e = T::place(c, m, i, j, k);
            if (k < T::R && T::ring(i, j, k) >= inside && dv[c][m] > 0.0f) v[e] = __fdiv_rn(bv[c][m] + T::sum(v, e), dv[c][m]);
        }
        __syncthreads();
    };
    pass(std::integral_constant<int, 1>{}, 1);
    pass(std::integral_constant<int, 0>{}, 2);
    pass(std::integral_constant<int, 1>{}, 3);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            const int e = T::place(c, m, i, j, k);
            if (k >= T::R || T::ring(i, j, k) < 4) continue;
            const float xl = v[e], d = dv[c][m];
            rs[e] = d >= 0.0f ? bv[c][m] - (d * xl - T::sum(v, e)) : 0.0f;
            const int I = o.x + i - RB_DOWN, J = o.y + j - RB_DOWN, K = o.z + k - RB_DOWN;
            if (T::ring(i, j, k) >= RB_DOWN && I < n.x && J < n.y && K < n.z) x[rb_lin(I, J, K, n)] = xl;
        }
    __syncthreads();
    constexpr int HC = RB / 2;
    if (threadIdx.x < HC * HC * HC) {   // flip.jl:891-906 restrict_kernel!
        const int t = (int)threadIdx.x, ci = t % HC, cj = (t / HC) % HC, ck = t / (HC * HC);
        const int I = (o.x >> 1) + ci, J = (o.y >> 1) + cj, K = (o.z >> 1) + ck;
        if (I < nc.x && J < nc.y && K < nc.z) {
            const size_t C = rb_lin(I, J, K, nc);
            const bool liquid = tc[C] == LIQUID;
            const float w[4] = {0.125f, 0.375f, 0.375f, 0.125f};
            const int e0 = (RB_DOWN + 2 * ci - 1) + T::R * ((RB_DOWN + 2 * cj - 1) + T::R * (RB_DOWN + 2 * ck - 1));
            float s = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int bb = 0; bb < 4; ++bb)
#pragma unroll
                    for (int a = 0; a < 4; ++a) s += w[a] * w[bb] * w[c] * rs[e0 + a + T::R * (bb + T::R * c)];
            bc[C] = liquid ? 4.0f * s : 0.0f;
        }
    }
}

// flip.jl:908-929 prolong_kernel!'s correction at cell (I, J, K) of the finer level, from the
// coarser level's values `at(a, b, c)`, 0 off its LIQUID cells and off its grid.
template <class At> __device__ inline float rb_prolong(int I, int J, int K, At at) {
    const int A = (I + 1) / 2 - 1, B = (J + 1) / 2 - 1, Cc = (K + 1) / 2 - 1;   // the lower of each pair
    const float wa[2] = {I & 1 ? 0.75f : 0.25f, I & 1 ? 0.25f : 0.75f}, wb[2] = {J & 1 ? 0.75f : 0.25f, J & 1 ? 0.25f : 0.75f},
                wc[2] = {K & 1 ? 0.75f : 0.25f, K & 1 ? 0.25f : 0.75f};
    float s = 0.0f;
#pragma unroll
    for (int m = 0; m < 8; ++m)
        s += wa[m & 1] * wb[(m >> 1) & 1] * wc[m >> 2] * at(A + (m & 1), B + ((m >> 1) & 1), Cc + (m >> 2));
    return s;
}

// Up, two sweeps: out from x plus the correction of the coarser level's xc.
__global__ __launch_bounds__(RB_THREADS) void k_rbup(float* __restrict__ out, const float* __restrict__ x,
                                                     const float* __restrict__ xc, const float* __restrict__ b,
                                                     const float* __restrict__ dg, const uint8_t* __restrict__ tf, int3 n,
                                                     int3 nc) {
    using T = RBTile<RB_UP>;
    constexpr int RC = RB / 2 + RB_UP + 2;   // the coarser cells under the region and one round them
    __shared__ float v[T::N], vc[RC * RC * RC];
    const int3 o = rb_tile(blockIdx.x, n);
    const int a0 = (o.x - RB_UP) / 2 - 1, b0 = (o.y - RB_UP) / 2 - 1, c0 = (o.z - RB_UP) / 2 - 1;   // exact: even
    float xv[2][T::M], bv[2][T::M], dv[2][T::M];
    int i, j, k;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            T::place(c, m, i, j, k);
            const int I = o.x + i - RB_UP, J = o.y + j - RB_UP, K = o.z + k - RB_UP;
            const bool in = k < T::R && rb_in(I, J, K, n);
            const size_t l = in ? rb_lin(I, J, K, n) : 0;
            xv[c][m] = in ? x[l] : 0.0f;
            bv[c][m] = in ? b[l] : 0.0f;
            dv[c][m] = in ? rb_diag(dg, tf, l) : -1.0f;
        }
    for (int t = threadIdx.x; t < RC * RC * RC; t += RB_THREADS) {
        const int I = a0 + t % RC, J = b0 + (t / RC) % RC, K = c0 + t / (RC * RC);
        vc[t] = rb_in(I, J, K, nc) ? xc[rb_lin(I, J, K, nc)] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            const int e = T::place(c, m, i, j, k);
            if (k >= T::R) continue;
            const int I = o.x + i - RB_UP, J = o.y + j - RB_UP, K = o.z + k - RB_UP;
            float val = 0.0f;
            if (dv[c][m] > 0.0f)   // in the grid
                val = xv[c][m] + rb_prolong(I, J, K, [&](int A, int B, int Cc) {
                          return vc[(A - a0) + RC * ((B - b0) + RC * (Cc - c0))];
                      });
            v[e] = val;
        }
    __syncthreads();
    auto pass = [&](auto colour, int inside) {
        constexpr int c = decltype(colour)::value;
#pragma unroll
        for (int m = 0; m < T::M; ++m) {
            const int e = T::place(c, m, i, j, k);
            if (k < T::R && T::ring(i, j, k) >= inside && dv[c][m] > 0.0f) v[e] = __fdiv_rn(bv[c][m] + T::sum(v, e), dv[c][m]);
        }
        __syncthreads();
    };
    pass(std::integral_constant<int, 1>{}, 1);
    pass(std::integral_constant<int, 0>{}, 2);
    pass(std::integral_constant<int, 1>{}, 3);
    pass(std::integral_constant<int, 0>{}, 4);
    for (int t = threadIdx.x; t < RB * RB * RB; t += RB_THREADS) {
        const int I = o.x + t % RB, J = o.y + (t / RB) % RB, K = o.z + t / (RB * RB);
        if (I < n.x && J < n.y && K < n.z)
            out[rb_lin(I, J, K, n)] = v[(RB_UP + t % RB) + T::R * ((RB_UP + (t / RB) % RB) + T::R * (RB_UP + t / (RB * RB)))];
    }
}

// ─── the last two levels in one workgroup ────────────────────────────────────

// The level before the coarsest (even sides, at most 2 M RB_THREADS cells and CELLS with the
// layer round it; none where M is 0) and the coarsest (at most 1,024 cells), in LDS with a
// layer of zeros round each.
struct RBLevel {
    float *x;
    const float *b, *dg;
    const uint8_t* types;
    int3 n;
};
// flip.jl:931-962 coarse_kernel!: `sweeps` sweeps from zero and as many in reverse colour
// order, from the right-hand side in v (which becomes the result). A thread has a cell of
// each colour of a row, so half the threads do a pass and the fewer wavefronts meet sooner,
// and the division by the same diagonal (a count of neighbours) each pass is a product.
__device__ inline void rb_coarsest(float* v, const float* dg, int3 n, int sweeps) {
    const int sx = n.x + 2, sxy = sx * (n.y + 2), hx = (n.x + 1) >> 1, t = (int)threadIdx.x;
    const int h = t % hx, j = (t / hx) % n.y, k = t / (hx * n.y);
    int at[2];
    bool act[2];
    float bv[2];
    double rc[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int i = 2 * h + ((c + j + k + 1) & 1);
        const bool in = i < n.x && k < n.z;
        const float d = in ? dg[rb_lin(i, j, k, n)] : 0.0f;
        act[c] = d > 0.0f;
        at[c] = in ? (i + 1) + sx * (j + 1) + sxy * (k + 1) : 0;
        bv[c] = act[c] ? v[at[c]] : 0.0f;
        rc[c] = act[c] ? 1.0 / (double)d : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c)
        if (at[c]) v[at[c]] = 0.0f;
    __syncthreads();
    auto pass = [&](auto colour) {
        constexpr int c = decltype(colour)::value;
        if (act[c]) {
            const float* p = v + at[c];
            const float w[6] = {p[1], p[-1], p[sx], p[-sx], p[sxy], p[-sxy]};
            float acc = bv[c];
#pragma unroll
            for (int m = 0; m < 6; ++m) acc += w[m];
            v[at[c]] = quotient(acc, 0.0f, rc[c]);
        }
        __syncthreads();
    };
    const std::integral_constant<int, 0> c0;
    const std::integral_constant<int, 1> c1;
    for (int s = 0; s < sweeps; ++s) { pass(c0); pass(c1); }
    for (int s = 0; s < sweeps; ++s) { pass(c1); pass(c0); }
}
__host__ __device__ inline int rb_padded(int3 n) { return (n.x + 2) * (n.y + 2) * (n.z + 2); }

constexpr int RB_TAIL_COARSE = 9248;   // 1 x 1 x 1,024 cells with their layer of zeros
template <int M, int CELLS>
__global__ __launch_bounds__(RB_THREADS) void k_rbtail(RBLevel F, RBLevel K, int sweeps, int coarse) {
    __shared__ float v[M ? CELLS : 1], rs[M ? CELLS : 1], vc[RB_TAIL_COARSE];
    for (int t = threadIdx.x; t < rb_padded(K.n); t += RB_THREADS) vc[t] = 0.0f;
    const int cx = K.n.x + 2, cxy = cx * (K.n.y + 2), NC = K.n.x * K.n.y * K.n.z, t = (int)threadIdx.x;
    int ci, cj, ck;
    unlin((size_t)min(t, NC - 1), K.n.x, K.n.y, ci, cj, ck);
    const int ce = (ci + 1) + cx * (cj + 1) + cxy * (ck + 1);
    if constexpr (M == 0) {
        __syncthreads();
        if (t < NC) vc[ce] = K.b[t];
        __syncthreads();
        rb_coarsest(vc, K.dg, K.n, coarse);
    } else {
        const int sx = F.n.x + 2, sxy = sx * (F.n.y + 2), hx = F.n.x >> 1;
        for (int q = t; q < rb_padded(F.n); q += RB_THREADS) v[q] = rs[q] = 0.0f;
        int at[2][M], own[2][M];
        float bv[2][M], dv[2][M];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int e = t + m * RB_THREADS, r = e / hx, j = r % F.n.y, k = r / F.n.y;
                const int i = 2 * (e % hx) + ((c + j + k + 1) & 1);
                const bool in = k < F.n.z;
                own[c][m] = in ? i + F.n.x * (j + F.n.y * k) : 0;
                at[c][m] = in ? (i + 1) + sx * (j + 1) + sxy * (k + 1) : 0;
                bv[c][m] = in ? F.b[own[c][m]] : 0.0f;
                dv[c][m] = in ? rb_diag(F.dg, F.types, own[c][m]) : -1.0f;
            }
        auto sum = [&](int e) {
            const float* p = v + e;
            float s = 0.0f;
            s += p[1]; s += p[-1]; s += p[sx]; s += p[-sx]; s += p[sxy]; s += p[-sxy];
            return s;
        };
        auto pass = [&](auto colour) {
            constexpr int c = decltype(colour)::value;
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (dv[c][m] > 0.0f) v[at[c][m]] = __fdiv_rn(bv[c][m] + sum(at[c][m]), dv[c][m]);
            __syncthreads();
        };
        const std::integral_constant<int, 0> c0;
        const std::integral_constant<int, 1> c1;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (dv[0][m] > 0.0f) v[at[0][m]] = __fdiv_rn(bv[0][m], dv[0][m]);
        __syncthreads();
        pass(c1);
        for (int s = 1; s < sweeps; ++s) { pass(c0); pass(c1); }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (at[c][m]) {
                    const float d = dv[c][m];
                    rs[at[c][m]] = d >= 0.0f ? bv[c][m] - (d * v[at[c][m]] - sum(at[c][m])) : 0.0f;
                }
        __syncthreads();
        if (t < NC) {
            const float w[4] = {0.125f, 0.375f, 0.375f, 0.125f};
            const int e0 = 2 * ci + sx * 2 * cj + sxy * 2 * ck;   // cell 2 c - 1 in the padded numbering
            float s = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int a = 0; a < 4; ++a) s += w[a] * w[b] * w[c] * rs[e0 + a + sx * b + sxy * c];
            vc[ce] = K.types[t] == LIQUID ? 4.0f * s : 0.0f;
        }
        __syncthreads();
        rb_coarsest(vc, K.dg, K.n, coarse);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (dv[c][m] > 0.0f) {
                    int i, j, k;
                    unlin((size_t)own[c][m], F.n.x, F.n.y, i, j, k);
                    v[at[c][m]] += rb_prolong(i, j, k, [&](int A, int B, int C) { return vc[(A + 1) + cx * (B + 1) + cxy * (C + 1)]; });
                }
        __syncthreads();
        for (int s = 0; s < sweeps; ++s) { pass(c1); pass(c0); }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (at[c][m]) F.x[own[c][m]] = v[at[c][m]];
    }
    if constexpr (M == 0)
        if (t < NC) K.x[t] = vc[ce];
}

}  // namespace mael
