// p4g_tail_kernels.hpp -- the coarse end of a V-cycle in one launch.
//
// A coarse level has too few points to fill the chip: its residual,
// restriction and prolongation passes take 3-5 us each, almost all of it
// launch and memory latency, and five levels of them were most of a small
// solve (129^2: 17 of the 24 launches of a CG iteration).  k_vtail runs the
// levels from 0 up to the largest whose three vectors fit the LDS of one
// compute unit (65^2 or 17^3 points in FP64) as one workgroup: every
// neighbour read is an LDS access and every phase ends in a workgroup barrier
// instead of a launch.  Bound by the instructions that one workgroup issues:
// indices, masks and addresses of every point in every phase (129^2: 23 us,
// of which the LDS bytes would take about 3).
// Constant-coefficient levels with a Jacobi-preconditioned Chebyshev or
// Richardson smoother; the formulas are those of the passes it stands for
// (OpConst, OutCheb, OutResid, the Q1 transfers).
#pragma once

namespace p4g {

constexpr int kTailLevels = 8, kTailSteps = 4, kTailThreads = 1024;
constexpr size_t kTailLds = 156 * 1024;   // of the compute unit's 160 KiB
// coarsest points: their inverse is read by this one workgroup, n^2 words at
// one compute unit's rate (a tail over 13x11x9 and 210 coarsest points took
// 29 us, the 7 launches that it stood for 20)
constexpr int kTailCoarse = 128;

template <typename T>
struct TailLevel {
    int mx, my, mz, n, off;               // off: the level's b, u, v in LDS
    T d, sx, sy, sz, idg;
    T c0[kTailSteps], c1[kTailSteps], c2[kTailSteps];   // smoothing step m: c0 x_{m-2} + c1 x_{m-1} + c2 D^-1 (b - A x_{m-1})
    int diff;
};

template <typename T>
struct TailArgs {
    int nl, nu, n0;                       // levels (the top is nl - 1), smoothing steps, coarsest points
    const double* Ainv;
    const T* b;
    T* x;
    TailLevel<T> lv[kTailLevels];
};

// (i, j, k) of point q by float reciprocals: exact for the few thousand points here
__device__ __forceinline__ void tail_ijk(int q, int mx, int my, float rx, float ry, int& i, int& j, int& k) {
    const int row = (int)((q + 0.5f) * rx);
    i = q - row * mx;
    k = (int)((row + 0.5f) * ry);
    j = row - k * my;
}

// A u at point q (boundary neighbours are eliminated: they enter as 0)
template <typename T, int DIM>
__device__ __forceinline__ T tail_apply(const TailLevel<T>& L, const T* u, T scale, int q, int i, int j, int k) {
    const T uc = scale * u[q];
    const bool bnd = i == 0 || i == L.mx - 1 || j == 0 || j == L.my - 1 || (DIM == 3 && (k == 0 || k == L.mz - 1));
    if (bnd) return L.d * uc;
    const int sy = L.mx, sz = L.mx * L.my;
    const T w = i > 1 ? scale * u[q - 1] : T(0), e = i < L.mx - 2 ? scale * u[q + 1] : T(0);
    const T s = j > 1 ? scale * u[q - sy] : T(0), n = j < L.my - 2 ? scale * u[q + sy] : T(0);
    T dn = T(0), up = T(0);
    if (DIM == 3) {
        dn = k > 1 ? scale * u[q - sz] : T(0);
        up = k < L.mz - 2 ? scale * u[q + sz] : T(0);
    }
    if (L.diff) return L.sx * ((uc - w) + (uc - e)) + L.sy * ((uc - s) + (uc - n)) + L.sz * ((uc - dn) + (uc - up));
    return L.d * uc - L.sx * (w + e) - L.sy * (s + n) - L.sz * (dn + up);
}

template <typename T, int DIM>
__global__ void __launch_bounds__(kTailThreads) k_vtail(TailArgs<T> A) {
    extern __shared__ __align__(16) unsigned char tail_lds[];
    T* const lds = (T*)tail_lds;
    const int tid = threadIdx.x, top = A.nl - 1, nu = A.nu;
    {
        const TailLevel<T>& L = A.lv[top];
        T* const b = lds + L.off;
        for (int q = tid; q < L.n; q += kTailThreads) b[q] = A.b[q];
    }
    __syncthreads();
    // down: pre-smoothing from zero, residual, restriction
    for (int l = top; l > 0; --l) {
        const TailLevel<T>& L = A.lv[l];
        const TailLevel<T>& C = A.lv[l - 1];
        T* const b = lds + L.off;
        T* u = b + L.n;
        T* v = u + L.n;
        const float rx = 1.0f / L.mx, ry = 1.0f / L.my;
        const T c = L.c2[0] * L.idg;
        if (nu > 1) {
            for (int q = tid; q < L.n; q += kTailThreads) u[q] = c * b[q];
            __syncthreads();
            for (int m = 1; m < nu; ++m) {
                for (int q = tid; q < L.n; q += kTailThreads) {
                    int i, j, k;
                    tail_ijk(q, L.mx, L.my, rx, ry, i, j, k);
                    const T Au = tail_apply<T, DIM>(L, u, T(1), q, i, j, k);
                    T y = L.c1[m] * u[q] + L.c2[m] * (L.idg * (b[q] - Au));
                    if (m > 1) y += L.c0[m] * v[q];
                    v[q] = y;
                }
                __syncthreads();
                T* const t = u;
                u = v;
                v = t;
            }
        }
        for (int q = tid; q < L.n; q += kTailThreads) {
            int i, j, k;
            tail_ijk(q, L.mx, L.my, rx, ry, i, j, k);
            v[q] = b[q] - (nu > 1 ? tail_apply<T, DIM>(L, u, T(1), q, i, j, k) : tail_apply<T, DIM>(L, b, c, q, i, j, k));
        }
        __syncthreads();
        T* const bc = lds + C.off;
        const float cx = 1.0f / C.mx, cy = 1.0f / C.my;
        const int sy = L.mx, sz = L.mx * L.my;
        for (int q = tid; q < C.n; q += kTailThreads) {
            int I, J, K;
            tail_ijk(q, C.mx, C.my, cx, cy, I, J, K);
            const int f = (2 * K * L.my + 2 * J) * L.mx + 2 * I;
            const T h = T(0.5);
            auto row = [&](int p) {
                return v[p] + h * ((I > 0 ? v[p - 1] : T(0)) + (I < C.mx - 1 ? v[p + 1] : T(0)));
            };
            auto plane = [&](int p) {
                return row(p) + h * ((J > 0 ? row(p - sy) : T(0)) + (J < C.my - 1 ? row(p + sy) : T(0)));
            };
            T s = plane(f);
            if (DIM == 3) s += h * ((K > 0 ? plane(f - sz) : T(0)) + (K < C.mz - 1 ? plane(f + sz) : T(0)));
            bc[q] = s;
        }
        __syncthreads();
    }
    {   // the coarsest level: x = A^-1 b in FP64, a wave per row, four rows in flight
        const TailLevel<T>& L = A.lv[0];
        const T* const b = lds + L.off;
        T* const x = top == 0 ? A.x : lds + L.off + L.n;
        const int lane = tid & 63;
        constexpr int WV = kTailThreads / 64, RW = 4;
        for (int row = tid >> 6; row < A.n0; row += RW * WV) {
            double s[RW] = {};
            for (int c = lane; c < A.n0; c += 64) {
                const double bc = double(b[c]);
#pragma unroll
                for (int h = 0; h < RW; ++h) s[h] += A.Ainv[(long)min(row + h * WV, A.n0 - 1) * A.n0 + c] * bc;
            }
#pragma unroll
            for (int h = 0; h < RW; ++h) {
                const double t = wave_sum(s[h]);
                if (lane == 0 && row + h * WV < A.n0) x[row + h * WV] = T(t);
            }
        }
    }
    __syncthreads();
    // up: prolongation and post-smoothing; a level's result is in u of its arrays
    for (int l = 1; l <= top; ++l) {
        const TailLevel<T>& L = A.lv[l];
        const TailLevel<T>& C = A.lv[l - 1];
        T* const b = lds + L.off;
        // the pre-smoothed iterate is in u or v (nu - 1 swaps); the level below left its own in xc
        T* u = b + L.n;
        T* v = u + L.n;
        if ((nu - 1) & 1) {
            T* const t = u;
            u = v;
            v = t;
        }
        const T* const xc = lds + C.off + C.n;
        const float rx = 1.0f / L.mx, ry = 1.0f / L.my;
        const T c = L.c2[0] * L.idg;
        const int cy = C.mx, cz = C.mx * C.my;
        for (int q = tid; q < L.n; q += kTailThreads) {   // t = pre + P x_c
            int i, j, k;
            tail_ijk(q, L.mx, L.my, rx, ry, i, j, k);
            const int p = ((k >> 1) * C.my + (j >> 1)) * C.mx + (i >> 1);
            const T h = T(0.5);
            auto row = [&](int a) { return i & 1 ? h * (xc[a] + xc[a + 1]) : xc[a]; };
            auto plane = [&](int a) { return j & 1 ? h * (row(a) + row(a + cy)) : row(a); };
            const T e = DIM == 3 && (k & 1) ? h * (plane(p) + plane(p + cz)) : plane(p);
            v[q] = (nu > 1 ? u[q] : c * b[q]) + e;
        }
        __syncthreads();
        // step m: from v (and u, two steps before) into u; the result has to
        // end in the first array, or in x on the top level
        for (int m = 0; m < nu; ++m) {
            const bool last = m == nu - 1;
            T* const out = last && l == top ? A.x : u;
            for (int q = tid; q < L.n; q += kTailThreads) {
                int i, j, k;
                tail_ijk(q, L.mx, L.my, rx, ry, i, j, k);
                const T Av = tail_apply<T, DIM>(L, v, T(1), q, i, j, k);
                T y = L.c1[m] * v[q] + L.c2[m] * (L.idg * (b[q] - Av));
                if (m > 0) y += L.c0[m] * u[q];
                out[q] = y;
            }
            __syncthreads();
            T* const t = u;
            u = v;
            v = t;
        }
        if (l < top && v != b + L.n) {     // (v: the result after the last swap)
            T* const first = b + L.n;
            for (int q = tid; q < L.n; q += kTailThreads) first[q] = v[q];
            __syncthreads();
        }
    }
}

}  // namespace p4g
