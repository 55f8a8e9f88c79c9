// The small dense levels of the sparse basin's V-cycle (sflip.jl:1572-1762) in few
// launches: a level's way down (two damped-Jacobi sweeps from zero, the residual and its
// restriction) in one, its way up (prolongation and two sweeps) in one, and the last levels
// with the coarsest solve in one workgroup.
//
// A sweep of a small level is a launch and a memory round trip around little work. Here a
// workgroup takes a tile with a halo of two cells, a thread keeps the rows of its cells in
// registers through the sweeps and the values go through LDS; a neighbour's cells are
// computed again in the halo. Every value goes through the same operations and roundings to
// the storage type as in a launch of its own (k_rowdense, k_residrestrict;
// a face without a coupling adds a zero product instead of being skipped), so the V-cycle's
// values do not change.
//
// Bound by launch and LDS latency. A level of 9,216 or 73,728 FP32 cells takes 5.1 us down and
// 5.1 us up, against 13 and 9 us in six launches; one of 368,640 FP16 cells 10.5 and 10.5 us.
// (With the couplings staged in LDS and read again each sweep the tiles took 10 us.)
#pragma once
#include "sparse.hpp"
#include "precision.hpp"
#include "quotient.hpp"
#include <type_traits>

namespace mael {

template <class C> struct DViewT {
    int3 n;
    const C* c[3];
    const C* dD;
    const uint8_t* act;
};

// A cell's row: its six couplings (0 where there is none), the full diagonal (-1 where the
// cell is not active) and the right-hand side.
struct MGRow {
    float c[6], d, b;
    // cell (i, j, k) of the level, `in` it
    template <class T, class C> __device__ void load(const DViewT<C>& L, const T* __restrict__ bg, int i, int j, int k, bool in) {
        const int n0 = L.n.x, n1 = L.n.y, n2 = L.n.z;
        if (!in) i = j = k = 0;
        const size_t l = cl(i, j, k, n0, n1);
        const float own = lf(L.dD[l]), bv = bg ? lf(bg[l]) : 0.0f;
        const bool on = L.act[l] != 0;
        const float f[6] = {lf(L.c[0][cl(i, j, k, n0 + 1, n1)]), lf(L.c[0][cl(i + 1, j, k, n0 + 1, n1)]),
                            lf(L.c[1][cl(i, j, k, n0, n1 + 1)]), lf(L.c[1][cl(i, j + 1, k, n0, n1 + 1)]),
                            lf(L.c[2][cl(i, j, k, n0, n1)]),     lf(L.c[2][cl(i, j, k + 1, n0, n1)])};
        const bool there[6] = {i > 0, i < n0 - 1, j > 0, j < n1 - 1, k > 0, k < n2 - 1};
        d = own;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            c[q] = in && there[q] && f[q] > 0.0f ? f[q] : 0.0f;
            d += c[q];
        }
        if (!(in && on)) d = -1.0f;
        b = in ? bv : 0.0f;
    }
    __device__ float off(const float (&x)[6]) const {
        float s = 0.0f;
#pragma unroll
        for (int q = 0; q < 6; ++q) s += c[q] * x[q];
        return s;
    }
    // a sweep from x (`from_zero`: x and its neighbours are 0), the residual
    template <class T> __device__ float jacobi(float x, const float (&nb)[6]) const {
        return d > 0.0f ? lf(sf<T>(x + __fdiv_rn(OMEGA * (b - (d * x - off(nb))), d))) : 0.0f;
    }
    template <class T> __device__ float from_zero() const {
        return d > 0.0f ? lf(sf<T>(0.0f + __fdiv_rn(OMEGA * (b - 0.0f), d))) : 0.0f;
    }
    template <class T> __device__ float residual(float x, const float (&nb)[6]) const {
        return d >= 0.0f ? lf(sf<T>(b - (d * x - off(nb)))) : 0.0f;   // an active row may have an empty diagonal
    }
};

constexpr int MG_H = 2, MG_THREADS = 1024;

// A tile of X x Y x Z cells and MG_H around it. Thread t has the region's cells t, t +
// MG_THREADS, ...; `ring` is how many cells a cell lies inside the region (MG_H or more: in
// the tile).
template <int X, int Y, int Z> struct MGTile {
    static constexpr int RX = X + 2 * MG_H, RY = Y + 2 * MG_H, RZ = Z + 2 * MG_H, RN = RX * RY * RZ;
    static constexpr int M = (RN + MG_THREADS - 1) / MG_THREADS;
    float v[2][RN];

    __device__ static int place(int m, int& i, int& j, int& k) {
        const int e = (int)threadIdx.x + m * MG_THREADS;
        i = e % RX; j = (e / RX) % RY; k = e / (RX * RY);
        return e;
    }
    __device__ static int ring(int i, int j, int k) {
        return min(min(min(i, RX - 1 - i), min(j, RY - 1 - j)), min(k, RZ - 1 - k));
    }
    __device__ void around(int w, int e, float (&x)[6]) const {
        x[0] = v[w][e - 1]; x[1] = v[w][e + 1]; x[2] = v[w][e - RX]; x[3] = v[w][e + RX];
        x[4] = v[w][e - RX * RY]; x[5] = v[w][e + RX * RY];
    }
};
// Workgroup g's tile over a level of n cells: its first cell.
template <int X, int Y, int Z> __device__ inline int3 mg_tile(uint32_t g, int3 n) {
    const uint32_t nx = (uint32_t)(n.x + X - 1) / X, ny = (uint32_t)(n.y + Y - 1) / Y;
    return make_int3((int)(g % nx) * X, (int)((g / nx) % ny) * Y, (int)(g / (nx * ny)) * Z);
}

// Down: x = two sweeps from zero on b, and the coarser level's right-hand side bc.
template <class T, class C, int X, int Y, int Z>
__global__ __launch_bounds__(MG_THREADS) void k_mgdown(T* __restrict__ x, T* __restrict__ bc, const T* __restrict__ b,
                                                       DViewT<C> L, int3 nc, float scale) {
    using R = MGTile<X, Y, Z>;
    __shared__ R S;
    const int3 o = mg_tile<X, Y, Z>(xcd_tile(blockIdx.x, gridDim.x), L.n);
    MGRow row[R::M];
    int i, j, k;
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k), I = o.x + i - MG_H, J = o.y + j - MG_H, K = o.z + k - MG_H;
        row[m].load(L, b, I, J, K, e < R::RN && I >= 0 && I < L.n.x && J >= 0 && J < L.n.y && K >= 0 && K < L.n.z);
    }
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k);
        if (e < R::RN) S.v[0][e] = row[m].template from_zero<T>();
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k);
        if (e >= R::RN || R::ring(i, j, k) < 1) continue;
        float w[6];
        S.around(0, e, w);
        S.v[1][e] = row[m].template jacobi<T>(S.v[0][e], w);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k), I = o.x + i - MG_H, J = o.y + j - MG_H, K = o.z + k - MG_H;
        if (e >= R::RN || R::ring(i, j, k) < MG_H) continue;
        float w[6];
        S.around(1, e, w);
        const float xl = S.v[1][e];
        S.v[0][e] = row[m].template residual<T>(xl, w);
        if (I < L.n.x && J < L.n.y && K < L.n.z) x[cl(I, J, K, L.n.x, L.n.y)] = sf<T>(xl);
    }
    __syncthreads();
    const int t = (int)threadIdx.x;
    if (t < X * Y * Z / 8) {
        const int ci = t % (X / 2), cj = (t / (X / 2)) % (Y / 2), ck = t / (X / 2 * (Y / 2));
        const int I = (o.x >> 1) + ci, J = (o.y >> 1) + cj, K = (o.z >> 1) + ck;
        const int e = (MG_H + 2 * ci) + R::RX * ((MG_H + 2 * cj) + R::RY * (MG_H + 2 * ck));
        float acc = 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) acc += S.v[0][e + (m & 1) + R::RX * ((m >> 1) & 1) + R::RX * R::RY * (m >> 2)];
        if (I < nc.x && J < nc.y && K < nc.z) bc[cl(I, J, K, nc.x, nc.y)] = sf<T>(acc * scale);
    }
}
// Up: out = two sweeps on b from x plus `boost` times the coarser level's xc.
template <class T, class C, int X, int Y, int Z>
__global__ __launch_bounds__(MG_THREADS) void k_mgup(T* __restrict__ out, const T* __restrict__ x, const T* __restrict__ xc,
                                                     const T* __restrict__ b, DViewT<C> L, int3 nc, float boost) {
    using R = MGTile<X, Y, Z>;
    __shared__ R S;
    const int3 o = mg_tile<X, Y, Z>(xcd_tile(blockIdx.x, gridDim.x), L.n);
    MGRow row[R::M];
    float x0[R::M], up[R::M];
    int i, j, k;
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k), I = o.x + i - MG_H, J = o.y + j - MG_H, K = o.z + k - MG_H;
        const bool in = e < R::RN && I >= 0 && I < L.n.x && J >= 0 && J < L.n.y && K >= 0 && K < L.n.z;
        x0[m] = in ? lf(x[cl(I, J, K, L.n.x, L.n.y)]) : 0.0f;
        up[m] = in ? lf(xc[cl(I >> 1, J >> 1, K >> 1, nc.x, nc.y)]) : 0.0f;
        row[m].load(L, b, I, J, K, in);
    }
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k);
        if (e < R::RN) S.v[0][e] = row[m].d >= 0.0f ? lf(sf<T>(x0[m] + boost * up[m])) : x0[m];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k);
        if (e >= R::RN || R::ring(i, j, k) < 1) continue;
        float w[6];
        S.around(0, e, w);
        S.v[1][e] = row[m].template jacobi<T>(S.v[0][e], w);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < R::M; ++m) {
        const int e = R::place(m, i, j, k), I = o.x + i - MG_H, J = o.y + j - MG_H, K = o.z + k - MG_H;
        if (e >= R::RN || R::ring(i, j, k) < MG_H) continue;
        float w[6];
        S.around(1, e, w);
        if (I < L.n.x && J < L.n.y && K < L.n.z) out[cl(I, J, K, L.n.x, L.n.y)] = sf<T>(row[m].template jacobi<T>(S.v[1][e], w));
    }
}

// ─── the last levels in one workgroup ────────────────────────────────────────

// The tail: up to three levels, the first of at most 2 THREADS cells, each next an eighth.
// Bound by the 160 passes of the coarsest solve, one LDS round trip and barrier each: 1,152
// and 144 FP32 cells 26 us, 512 cells 23 us (28 us with a thread per cell and a division a
// pass, without the level above), 720 cells in FP64 36 us (54 us). With the 1,152 cells'
// rows in LDS instead of registers the first took 50 us.
constexpr int MG_TAIL_LEVELS = 3;
template <class T, class C> struct MGTailArgs {
    DViewT<C> L[MG_TAIL_LEVELS];
    int nl;          // levels, the coarsest last
    const T* b;      // the first level's right-hand side
    T* x;            // and its result
};

// A level's cells in a workgroup: M a thread, their rows and neighbours in registers, the
// values in LDS (x fastest; a missing neighbour reads the cell itself).
template <class T, int M, int THREADS> struct MGLocal {
    MGRow row[M];
    int nb[M][6];
    int n;
    float *x, *y;
    template <class C> __device__ void load(const DViewT<C>& L, const T* __restrict__ b, float* x_, float* y_) {
        n = L.n.x * L.n.y * L.n.z;
        x = x_; y = y_;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int e = (int)threadIdx.x + m * THREADS;
            int i, j, k;
            unlin((size_t)min(e, n - 1), L.n.x, L.n.y, i, j, k);
            row[m].load(L, b, i, j, k, e < n);
            const int s[6] = {-1, 1, -L.n.x, L.n.x, -L.n.x * L.n.y, L.n.x * L.n.y};
#pragma unroll
            for (int q = 0; q < 6; ++q) nb[m][q] = row[m].c[q] > 0.0f ? e + s[q] : min(e, n - 1);
        }
    }
    template <class F> __device__ void each(F f) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int e = (int)threadIdx.x + m * THREADS;
            if (e < n) f(m, e);
        }
        __syncthreads();
    }
    __device__ void around(const float* v, int m, float (&w)[6]) const {
#pragma unroll
        for (int q = 0; q < 6; ++q) w[q] = v[nb[m][q]];
    }
    __device__ void sweep(float* to, const float* from) {
        each([&](int m, int e) {
            float w[6];
            around(from, m, w);
            to[e] = row[m].template jacobi<T>(from[e], w);
        });
    }
    __device__ void down() {   // x from zero, its residual in y
        each([&](int m, int e) { y[e] = row[m].template from_zero<T>(); });
        sweep(x, y);
        each([&](int m, int e) {
            float w[6];
            around(x, m, w);
            y[e] = row[m].template residual<T>(x[e], w);
        });
    }
};
// The coarser level's right-hand side, into its rows.
template <class T, class Fine, class Coarse>
__device__ inline void mg_restrict(const Fine& F, int3 nf, Coarse& K, int3 nc, float scale) {
    K.each([&](int m, int e) {
        int i, j, k;
        unlin((size_t)e, nc.x, nc.y, i, j, k);
        const int f = 2 * i + nf.x * (2 * j + nf.y * 2 * k);
        float acc = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q) acc += F.y[f + (q & 1) + nf.x * ((q >> 1) & 1) + nf.x * nf.y * (q >> 2)];
        K.row[m].b = lf(sf<T>(acc * scale));
    });
}
template <class T, class Fine, class Coarse>
__device__ inline void mg_rise(Fine& F, int3 nf, const Coarse& K, int3 nc, float boost) {
    F.each([&](int m, int e) {
        int i, j, k;
        unlin((size_t)e, nf.x, nf.y, i, j, k);
        if (F.row[m].d >= 0.0f) F.x[e] = lf(sf<T>(F.x[e] + boost * K.x[(i >> 1) + nc.x * ((j >> 1) + nc.y * (k >> 1))]));
    });
    F.sweep(F.y, F.x);
    F.sweep(F.x, F.y);
}
// sflip.jl:1623-1657 coarsest_kernel!: red-black Gauss-Seidel from zero in arithmetic A
// (FP64 in the mixed-precision solve), `sweeps` passes and as many in reverse colour order.
// A thread has a cell of each colour of a row, so half the threads do a pass and the fewer
// wavefronts meet sooner; the division by the same diagonal each pass is a product (quotient.hpp).
// An FP32 solve that came upon a subnormal quotient, where the product may round the wrong
// way, is made again with divisions: to look at each quotient at once and divide took 36 us
// instead of 29 for 1,152 and 144 cells.
template <class T, class A, int THREADS, class C, class Local>
__device__ inline void mg_coarsest(Local& K, const DViewT<C>& L, A* X, const float* bs, int sweeps) {
    const int n0 = L.n.x, n1 = L.n.y, n2 = L.n.z, hx = (n0 + 1) >> 1, t = (int)threadIdx.x;
    const int h = t % hx, j = (t / hx) % n1, k = t / (hx * n1);
    bool act[2];
    int at[2], nb[2][6];
    A bi[2], dg[2], cw[2][6];
    double rc[2];
#pragma unroll
    for (int colour = 0; colour < 2; ++colour) {
        const int i = 2 * h + ((colour + j + k + 1) & 1);
        const bool in = i < n0 && k < n2;
        MGRow row;
        row.load(L, (const T*)nullptr, i, j, k, in);
        act[colour] = in && row.d >= 0.0f;
        at[colour] = in ? i + n0 * (j + n1 * k) : 0;
        bi[colour] = (A)bs[at[colour]];
        A d = (A)lf(L.dD[at[colour]]);
        const int s[6] = {-1, 1, -n0, n0, -n0 * n1, n0 * n1};
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            cw[colour][q] = (A)row.c[q];
            d += cw[colour][q];
            nb[colour][q] = row.c[q] > 0.0f ? at[colour] + s[q] : at[colour];
        }
        dg[colour] = d;
        rc[colour] = d > A(0) ? 1.0 / (double)d : 0.0;
        act[colour] = act[colour] && d > A(0);   // (an empty row keeps its 0)
        if (in) X[at[colour]] = A(0);
    }
    __syncthreads();
    auto solve = [&](auto divide) {
        auto pass = [&](int c) {
            if (act[c]) {
                A v[6];
#pragma unroll
                for (int q = 0; q < 6; ++q) v[q] = X[nb[c][q]];
                A acc = bi[c];
#pragma unroll
                for (int q = 0; q < 6; ++q) acc += cw[c][q] * v[q];
                X[at[c]] = divide(acc, c);
            }
            __syncthreads();
        };
        for (int s = 0; s < sweeps; ++s) { pass(0); pass(1); }
        for (int s = 0; s < sweeps; ++s) { pass(1); pass(0); }
    };
    if constexpr (std::is_same<A, float>::value) {
        uint32_t least = ~0u;
        solve([&](float acc, int c) {
            const float q = quotient(acc, dg[c], rc[c]);
            least = min(least, subnormal_rank(q));
            return q;
        });
        if (__syncthreads_or(least < SUBNORMALS)) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (act[c]) X[at[c]] = 0.0f;
            __syncthreads();
            solve([&](float acc, int c) { return acc / dg[c]; });
        }
    } else {
        solve([&](A acc, int c) { return quotient(acc, dg[c], rc[c]); });
    }
    K.each([&](int m, int e) { K.x[e] = lf(sf<T>((float)X[e])); });
}

template <class T, class C, class A, int THREADS>
__global__ __launch_bounds__(THREADS) void k_mgtail(MGTailArgs<T, C> G, int sweeps, float scale, float boost) {
    __shared__ float v0[2][2 * THREADS], v1[2][THREADS], v2[2][THREADS], bs[1024];
    __shared__ A X[1024];
    MGLocal<T, 2, THREADS> L0;
    MGLocal<T, 1, THREADS> L1, L2;
    L0.load(G.L[0], G.b, v0[0], v0[1]);
    if (G.nl > 1) L1.load(G.L[1], (const T*)nullptr, v1[0], v1[1]);
    if (G.nl > 2) L2.load(G.L[2], (const T*)nullptr, v2[0], v2[1]);
    auto solve = [&](auto& K, const DViewT<C>& L) {
        K.each([&](int m, int e) { bs[e] = K.row[m].b; });
        mg_coarsest<T, A, THREADS>(K, L, X, bs, sweeps);
    };
    if (G.nl == 1) {
        solve(L0, G.L[0]);
    } else {
        L0.down();
        mg_restrict<T>(L0, G.L[0].n, L1, G.L[1].n, scale);
        if (G.nl == 2) {
            solve(L1, G.L[1]);
        } else {
            L1.down();
            mg_restrict<T>(L1, G.L[1].n, L2, G.L[2].n, scale);
            solve(L2, G.L[2]);
            mg_rise<T>(L1, G.L[1].n, L2, G.L[2].n, boost);
        }
        mg_rise<T>(L0, G.L[0].n, L1, G.L[1].n, boost);
    }
    L0.each([&](int m, int e) { G.x[e] = sf<T>(L0.x[e]); });
}

}  // namespace mael
