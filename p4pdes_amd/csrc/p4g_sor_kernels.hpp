// p4g_sor_kernels.hpp -- pipelined SOR sweeps (PETSc's MatSOR with omega 1
// and a zero initial guess, lexicographic order) of 2D and 3D levels.
//
// What bounds a directional sweep is its chain of dependent points, not
// memory: mx + my (+ mz) points one after the other.  The kernels below keep
// that chain in registers.  A wave owns a strip of 64 rows (in 3D of K
// planes); lane r marches along row r one point per step, `lag` steps behind
// lane r - 1, so the neighbour row toward the sweep's origin is lane r - 1's
// recent results (a DPP shift) and the neighbours in the row and in the
// planes of the wave are the lane's own.  Everything else is off the chain:
//
//  * Forward: S = b - (couplings to earlier points), x = S / a_qq, and S is
//    kept.  Backward: x = (S - (couplings to later points)) / a_qq.  S is
//    exactly what the sequential backward sweep forms first (its sum runs
//    over the earlier neighbours' forward values, in the same order), so the
//    forward x is never stored and the results are those of k_sor_plane, bit
//    for bit.
//  * S is stored by step (all 64 lanes of a step side by side), and the
//    backward sweep visits the steps in reverse, so its accesses are full
//    lines with addresses known at compile time; operands are loaded
//    kSorAhead batches of steps early.
//  * A strip (plane group) hands its last row (plane) to the next one
//    through global memory as pairs of 8-byte words, each half of the value
//    with the sweep's 32-bit tag: a word is either the awaited one or not,
//    so there is no flag, no fence and no cache write-back, and nothing to
//    clear between sweeps.  A tag is read from ctl[1], which the backward
//    sweep's last workgroup advances, so a recorded launch can be replayed.
//
// Workgroups depend on workgroups of lower index only (the dispatch order).
// A wait longer than spin_limit polls sets ctl[0] and gives up, and a launch
// that finds ctl[0] set waits for nothing: every kernel ends, and the host
// checks ctl[0] after the solve.  `extra` is added to every awaited tag (0;
// the host's stall test awaits a tag that no workgroup writes).
#pragma once

namespace p4g {

typedef unsigned long long u64;

__device__ __forceinline__ double dbl_of(int lo, int hi) {
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// lane i takes lane i-1's value, lane 0 `first`'s own
__device__ __forceinline__ double wave_shr1(double v, double first) {
    const long long b = __double_as_longlong(v), f = __double_as_longlong(first);
    const int rlo = __builtin_amdgcn_update_dpp((int)f, (int)b, 0x138, 0xf, 0xf, false);
    const int rhi = __builtin_amdgcn_update_dpp((int)(f >> 32), (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return dbl_of(rlo, rhi);
}

// a value and its tag as two self-validating words
struct Tagged {
    u64 lo, hi;
    __device__ __forceinline__ bool is(unsigned tag) const {
        return (unsigned)(lo >> 32) == tag && (unsigned)(hi >> 32) == tag;
    }
    __device__ __forceinline__ double value() const { return dbl_of((int)(unsigned)lo, (int)(unsigned)hi); }
};
__device__ __forceinline__ u64 ld_word(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_tagged(u64* lo, u64* hi, double v, unsigned tag) {
    const u64 b = (u64)__double_as_longlong(v), t = (u64)tag << 32;
    __hip_atomic_store(lo, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(hi, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// accesses through a buffer descriptor: past its bytes a load gives zero and
// a store is dropped; voff per lane, soff uniform
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ double buffer_ld(__amdgpu_buffer_rsrc_t b, unsigned voff) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(b, (int)voff, 0, 0);
    return dbl_of((int)v.x, (int)v.y);
}
__device__ __forceinline__ void buffer_st(__amdgpu_buffer_rsrc_t b, unsigned voff, double v) {
    const long long q = __double_as_longlong(v);
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{(unsigned)q, (unsigned)(q >> 32)}, b, (int)voff, 0, 0);
}
__device__ __forceinline__ T2<double> buffer_ld2(__amdgpu_buffer_rsrc_t b, unsigned voff, unsigned soff) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, (int)voff, (int)soff, 0);
    return T2<double>{dbl_of((int)v.x, (int)v.y), dbl_of((int)v.z, (int)v.w)};
}
__device__ __forceinline__ void buffer_st2(__amdgpu_buffer_rsrc_t b, unsigned voff, unsigned soff, double v0, double v1) {
    const long long p = __double_as_longlong(v0), q = __double_as_longlong(v1);
    __builtin_amdgcn_raw_buffer_store_b128(
        u32x4{(unsigned)p, (unsigned)(p >> 32), (unsigned)q, (unsigned)(q >> 32)}, b, (int)voff, (int)soff, 0);
}
// the sweep's control words and the state of its waits (uniform)
struct SorCtl {
    unsigned* ctl;        // [0] stalled, [1] sweeps done
    long spin_limit;
    unsigned extra;
};

__device__ __forceinline__ bool sor_dead(const SorCtl& c) {
    return __hip_atomic_load(c.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}
__device__ __forceinline__ unsigned sor_tag(const SorCtl& c, bool backward) {
    const unsigned e = __hip_atomic_load(c.ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_amdgcn_readfirstlane(2u * e + (backward ? 2u : 1u));
}
// one more failed poll: true when the waiting has to end
__device__ __forceinline__ bool sor_give_up(const SorCtl& c, long& spins) {
    if (++spins > c.spin_limit) {
        if (threadIdx.x == 0) atomicExch(c.ctl, 1u);
        return true;
    }
    __builtin_amdgcn_s_sleep(1);
    return (spins & 63) == 0 && __builtin_amdgcn_readfirstlane((int)sor_dead(c)) != 0;
}

// ------------------------------------------------------------------- 2D
//
// NINE = false: constant 5-point levels.  The strips cover the interior
// points (boundary rows are b / db and couple to nothing: blocks past the
// strips of the forward launch write them); lag 1.
// NINE = true: 9-point levels with stored coefficients (the Galerkin and
// finite-difference operators, planes 9..17 of the 27), all points; lag 2,
// because the neighbour row is needed one point ahead.
// Steps: at step t lane r takes point c = t - r - sh (5-point) or
// t - 1 - 2 r - sh (9-point) of its row in sweep order; tf = t forward and
// Tp - 1 - t backward indexes S and the packed coefficients, and sh makes
// the two agree.
constexpr int kXcds = 8;

template <bool NINE>
struct Sor2 {
    static constexpr int SB = NINE ? 8 : 16;          // steps per batch
    static constexpr int AH = 2;                      // batches of steps whose operands are in flight
    static constexpr int YD = 2;                      // batches whose neighbour-row words are in flight
    static constexpr int P0 = NINE ? 127 : 63;        // steps from a column at lane 0 to lane 63
    static constexpr int PAD = 192;                   // slots before column 0
    // slots of a strip's handed-over row: every batch's, in range or not
    __host__ __device__ static long slots(int Tp) { return Tp + PAD + 64; }
    // steps of a strip, padded to whole rounds of the operand ring
    __host__ __device__ static int steps(int mx) {
        const int need = NINE ? mx + 128 : mx - 2 + 63;
        static_assert(32 % (SB * AH) == 0 && AH % YD == 0, "whole rounds of the operand rings, whole tiles of k_sor9_pack");
        return (need + 31) / 32 * 32;
    }
    __host__ __device__ static int cols(int mx) { return NINE ? mx : mx - 2; }
    __host__ __device__ static int rows(int my) { return NINE ? my : my - 2; }
    __host__ __device__ static int strips(int my) { return (rows(my) + 63) / 64; }
};

struct Sor2Args {
    int mx, my, Tp, ns;
    double d, db, sx, sy;            // 5-point
    const T2<double>* pk;            // 9-point: per step 4 x 64 coefficient pairs (k_sor9_pack)
    const T2<double>* inv;           // 9-point: reciprocal diagonals, two steps per pair
    const double* b;
    T2<double>* S;                   // two steps per pair
    double* x;
    u64* yh;                         // per strip G::slots(Tp) tagged values: the strip's last row
    SorCtl c;
};

template <bool NINE, bool BWD>
__global__ void __launch_bounds__(64) k_sor2(Sor2Args A) {
    typedef Sor2<NINE> G;
    constexpr int SB = G::SB, AH = G::AH, YD = G::YD;
    const int r = threadIdx.x, mx = A.mx, my = A.my, ns = A.ns;
    if ((int)blockIdx.x < ns * kXcds && blockIdx.x % kXcds) return;      // every strip on one XCD
    const int o = (int)blockIdx.x < ns * kXcds ? blockIdx.x / kXcds : blockIdx.x - ns * (kXcds - 1);
    if (!NINE && !BWD && o >= ns) {          // the boundary rows
        const double idb = 1.0 / A.db;
        const int per = 2 * mx + 2 * (my - 2);
        for (int p = (o - ns) * 64 + r; p < per; p += (gridDim.x - ns * kXcds) * 64) {
            long q;
            if (p < mx) q = p;
            else if (p < 2 * mx) q = (long)(my - 1) * mx + (p - mx);
            else q = (long)(1 + ((p - 2 * mx) >> 1)) * mx + (((p - 2 * mx) & 1) ? mx - 1 : 0);
            A.x[q] = A.b[q] * idb;
        }
        return;
    }
    const int Tp = A.Tp, ncol = G::cols(mx), nrow = G::rows(my);
    const int s = BWD ? ns - 1 - o : o, rho = BWD ? 63 - r : r;
    const int row = 64 * s + rho;
    const bool rl = row < nrow;
    const int sh = BWD ? (NINE ? Tp - 2 - (mx + 126) : Tp - (ncol + 63)) : 0;
    const int off = sh + (NINE ? 1 + 2 * r : r);                 // c = t - off
    // b and x: the rows of the strip, relative to the first.  Off the strip a
    // load gives zero and a store is dropped, so no address is clamped; what
    // a lane reads past its row's ends is masked by `live`.
    const long strip0 = ((long)64 * s + (NINE ? 0 : 1)) * mx;
    const unsigned nrows = min(64, nrow - 64 * s);
    const __amdgpu_buffer_rsrc_t br = buffer_of((BWD ? (const double*)A.x : A.b) + strip0, nrows * mx * 8u);
    const unsigned rowq = (unsigned)rho * mx + (NINE ? 0 : 1);
    const unsigned vb = BWD ? (rowq + ncol - SB + off) * 8u : (rowq - off) * 8u;   // at t0: - or + 8 t0
    const __amdgpu_buffer_rsrc_t Sr = buffer_of(A.S + (long)s * (Tp / 2) * 64, Tp * 512u);
    const __amdgpu_buffer_rsrc_t Ir = buffer_of(NINE ? A.inv + (long)s * (Tp / 2) * 64 : A.S, Tp * 512u);
    const __amdgpu_buffer_rsrc_t Kr = buffer_of(NINE ? A.pk + (long)s * Tp * 256 : A.S, Tp * 4096u);
    const unsigned v16 = rho * 16u, vk = v16 + (BWD ? 2048u : 0u);
    const double invd = NINE ? 0.0 : 1.0 / A.d;
    // handed-over rows, by slot (the column in sweep order); lanes past the
    // batch repeat its slots, so that nothing has to be masked inside
    char* const yout = (char*)(A.yh + ((long)o * G::slots(Tp) + G::PAD - G::P0 - sh) * 2);
    const char* const yin = (const char*)(A.yh + ((long)(o > 0 ? o - 1 : 0) * G::slots(Tp) + G::PAD - sh) * 2);
    const int l = r & (SB - 1);
    const unsigned l16 = l * 16u;
    const unsigned tag = sor_tag(A.c, BWD), want = tag + A.c.extra;
    bool dead = __builtin_amdgcn_readfirstlane((int)sor_dead(A.c)) != 0;
    const bool full = 64 * s + 64 <= nrow;
    __shared__ double ybuf[64];             // the neighbour row of the next batch's steps (0..SB - 1)
    __shared__ double obuf[2][SB][64];      // the batch's results and those of the batch before

    struct Ops {
        double v[SB];                       // b (forward) or S (backward)
        T2<double> a[NINE ? 2 * SB : 1];    // the earlier (later) four couplings
        double inv[NINE ? SB : 1];
    } ops[AH];
    Tagged yw[YD];                          // lane e < SB: the neighbour row at step e of the next batches

    auto yload = [&](int t0, Tagged& w) {
        const char* const p = yin + (long)t0 * 16;
        w.lo = ld_word((const u64*)(p + l16));
        w.hi = ld_word((const u64*)(p + l16 + 8));
    };
    // every path issues the same loads, so that the compiler can count them
    auto load = [&](int t0, Ops& P) {
        unsigned vo = vb + t0 * 8u;
        asm volatile("" : "+v"(vo));        // one address per batch, the steps by immediate offsets
        // two addresses where a pair of steps may straddle the strip's bytes
        // (one access of both would then be out of range as a whole)
        unsigned vo1 = vo;
        if (NINE) asm volatile("" : "+v"(vo1));
#pragma unroll
        for (int e = 0; e < SB; e += 2) {
            const int m = BWD ? (Tp - 2 - (t0 + e)) >> 1 : (t0 + e) >> 1;    // pair of steps
            if (BWD) {
                const T2<double> v = buffer_ld2(Sr, v16, m * 1024u);
                P.v[e] = v.b;
                P.v[e + 1] = v.a;
            } else {
                P.v[e] = buffer_ld(br, vo + e * 8u);
                P.v[e + 1] = buffer_ld(br, vo1 + e * 8u + 8u);
            }
            if (NINE) {
                const T2<double> i2 = buffer_ld2(Ir, v16, m * 1024u);
                P.inv[e] = BWD ? i2.b : i2.a;
                P.inv[e + 1] = BWD ? i2.a : i2.b;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const unsigned tf = BWD ? Tp - 1 - (t0 + e + h) : t0 + e + h;
                    P.a[2 * (e + h)] = buffer_ld2(Kr, vk, tf * 4096u);
                    P.a[2 * (e + h) + 1] = buffer_ld2(Kr, vk + 1024u, tf * 4096u);
                }
            }
        }
    };
    double h1 = 0.0, u1 = 0.0, u2 = 0.0;    // own last result; the neighbour row's last two
    double y[SB], keep = 0.0;
    // steps E .. E + SB / 2 - 1 of a batch; edge: some lane is off the grid
    auto half = [&](int t0, const Ops& P, bool edge, int E) {
        unsigned vo = vb - t0 * 8u;
        asm volatile("" : "+v"(vo));
#pragma unroll
        for (int e = E; e < E + SB / 2; ++e) {
            const int c = t0 + e - off;
            const bool live = !edge || (rl && (unsigned)c < (unsigned)ncol);
            const double u3 = u2;
            u2 = u1;
            u1 = wave_shr1(h1, y[e]);
            double sum = live || NINE ? P.v[e] : 0.0, res;
            if (!NINE) {
                if (!BWD) {
                    sum += A.sy * u1;
                    sum += A.sx * h1;
                } else {
                    sum += A.sx * h1;
                    sum += A.sy * u1;
                }
                res = sum * invd;
            } else {             // off the grid every coefficient is zero, and so is the result
                const T2<double> p0 = P.a[2 * e], p1 = P.a[2 * e + 1];
                if (!BWD) {      // (j-1, i-1), (j-1, i), (j-1, i+1), (j, i-1)
                    sum -= p0.a * u3;
                    sum -= p0.b * u2;
                    sum -= p1.a * u1;
                    sum -= p1.b * h1;
                } else {         // (j, i+1), (j+1, i-1), (j+1, i), (j+1, i+1)
                    sum -= p0.a * h1;
                    sum -= p0.b * u1;
                    sum -= p1.a * u2;
                    sum -= p1.b * u3;
                }
                res = sum * P.inv[e];
            }
            if (!BWD) {
                if (e & 1) buffer_st2(Sr, v16, (t0 + e - 1) * 512u, keep, sum);
                else keep = sum;
            } else {
                buffer_st(br, (live ? vo : 0x80000000u) + (SB - 1 - e) * 8u, res);
            }
            h1 = res;
            obuf[(t0 / SB) & 1][e][r] = res;
        }
    };
    // the neighbour row of the batch at t0, loaded in yw[q], into LDS
    auto ywait = [&](int t0, int q, bool edge) __attribute__((always_inline)) {
        if (o == 0) return;
        const int slot = t0 + l - sh;
        const bool need = !edge || (slot >= 0 && slot < ncol);
        if (__builtin_expect(!__all(!need || yw[q].is(want)), 0)) {
            long spins = 0;
            while (!dead && !__all(!need || yw[q].is(want))) {
                dead = sor_give_up(A.c, spins);
                yload(t0, yw[q]);
            }
            // the words of the batches after were loaded too early as well
#pragma unroll
            for (int h = 1; h < YD; ++h) yload(t0 + h * SB, yw[(q + h) % YD]);
            __builtin_amdgcn_s_waitcnt(0);   // so that the other path's waits stay as they are
        }
        ybuf[r] = need ? yw[q].value() : 0.0;
        wave_lds_order();
    };
    // the last lane's results of the batch at t0, at the slots their columns give
    auto publish = [&](int t0, double v, bool edge) __attribute__((always_inline)) {
        const int slot = t0 + l - G::P0 - sh;
        char* const p = yout + (long)t0 * 16;
        if (!edge || (slot >= 0 && slot < ncol)) st_tagged((u64*)(p + l16), (u64*)(p + l16 + 8), v, tag);
    };
    ybuf[r] = 0.0;
    wave_lds_order();
#pragma unroll
    for (int h = 0; h < YD; ++h) yload(h * SB, yw[h]);
    ywait(0, 0, true);
#pragma unroll
    for (int e = 0; e < SB; ++e) y[e] = ybuf[e];
    wave_lds_order();
    yload(YD * SB, yw[0]);
#pragma unroll
    for (int q = 0; q < AH; ++q) load(q * SB, ops[q]);
    // a round of the operand ring; off the grid or not is settled per round,
    // because a taken branch costs a lone wave as much as a step
    auto round = [&](int t0, bool edge) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < AH; ++q) {
            const int t = t0 + q * SB;
            // the words awaited below and the results published below were
            // asked for half a batch before
            const double v = obuf[((t / SB) & 1) ^ 1][l][63];
            half(t, ops[q], edge, 0);
            publish(t - SB, v, edge);
            ywait(t + SB, (q + 1) % YD, edge);
            double yn[SB];
#pragma unroll
            for (int e = 0; e < SB; ++e) yn[e] = ybuf[e];
            half(t, ops[q], edge, SB / 2);
            wave_lds_order();
#pragma unroll
            for (int e = 0; e < SB; ++e) y[e] = yn[e];
            yload(t + (YD + 1) * SB, yw[(q + 1) % YD]);
            load(min(t + SB * AH, Tp - SB), ops[q]);
        }
    };
    round(0, true);      // apart from the loop, whose waits it would shorten (fewer accesses precede it)
    for (int t0 = SB * AH; t0 < Tp; t0 += SB * AH) {
        if (!full || t0 < 63 * (NINE ? 2 : 1) + sh + 1 || t0 + SB * AH + SB - sh > ncol) round(t0, true);
        else round(t0, false);
    }
    publish(Tp - SB, obuf[((Tp / SB) & 1) ^ 1][l][63], true);
    if (BWD && o == ns - 1 && r == 0) A.c.ctl[1] += 1;
}

// the packed operator of a 9-point level: pk[(s Tp + tf) 4 + p][rho] the
// couplings (c = 9,10), (11,12), (14,15), (16,17) and inv two steps of the
// reciprocal diagonal (0 for a null row) of point (column tf - 1 - 2 rho, row
// 64 s + rho); zeros where there is no point, and for a neighbour outside the
// grid.  Rows are read along x and written by step through LDS.  Grid
// (Tp / 32, strips), 256 threads.
__global__ void __launch_bounds__(256)
k_sor9_pack(int mx, int my, int Tp, const double* __restrict__ g, T2<double>* __restrict__ pk,
            T2<double>* __restrict__ inv) {
    __shared__ double tile[2][64][33];
    const int t0 = blockIdx.x * 32, s = blockIdx.y, w = threadIdx.x >> 5, l = threadIdx.x & 31;
    const long n = (long)mx * my;
    const int grp[5][2] = {{0, 1}, {2, 3}, {5, 6}, {7, 8}, {4, 4}};
#pragma unroll
    for (int p = 0; p < 5; ++p) {
        for (int rho = w; rho < 64; rho += 8) {
            const int c = t0 + l - 1 - 2 * rho, j = 64 * s + rho;
            const bool in = c >= 0 && c < mx && j < my;
#pragma unroll
            for (int h = 0; h < (p < 4 ? 2 : 1); ++h) {
                const int k = grp[p][h], ii = c + k % 3 - 1, jj = j + k / 3 - 1;
                double v = 0.0;
                if (in && ii >= 0 && ii < mx && jj >= 0 && jj < my) v = g[(long)(9 + k) * n + (long)j * mx + c];
                if (p == 4) v = v != 0.0 ? 1.0 / v : 0.0;
                tile[h][rho][l] = v;
            }
        }
        __syncthreads();
        if (p < 4) {
            for (int q = threadIdx.x; q < 32 * 64; q += 256) {
                const int tt = q >> 6, rho = q & 63;
                pk[(((long)s * Tp + t0 + tt) * 4 + p) * 64 + rho] = T2<double>{tile[0][rho][tt], tile[1][rho][tt]};
            }
        } else {
            for (int q = threadIdx.x; q < 16 * 64; q += 256) {
                const int m = q >> 6, rho = q & 63;
                inv[((long)s * (Tp / 2) + t0 / 2 + m) * 64 + rho] =
                    T2<double>{tile[0][rho][2 * m], tile[0][rho][2 * m + 1]};
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------- 3D
//
// Constant 7-point levels, interior points.  A wave owns 64 rows of
// kSor7Planes planes: at step t lane r takes column t - r - kk - sh of plane
// kk, so plane kk - 1's value at that point is the lane's result of the step
// before, and the planes of a step are independent chains that hide each
// other's latency.  The wave's last plane goes to the next plane group by
// step, tagged; its last row to the next strip as in 2D.
constexpr int kSor7Planes = 4;

struct Sor7 {
    static constexpr int K = kSor7Planes, SB = 4, D = 4;
    __host__ __device__ static int steps(int mx) {
        const int need = mx - 2 + 63 + K - 1;
        static_assert(64 % (SB * D) == 0, "whole tiles of the pack kernels, whole rounds of the ring");
        return (need + 63) / 64 * 64;
    }
    __host__ __device__ static int strips(int my) { return (my - 2 + 63) / 64; }
    __host__ __device__ static int groups(int mz) { return (mz - 2 + K - 1) / K; }
};

struct Sor7Args {
    int mx, my, mz, Tp, ns, ng;
    double d, sx, sy, sz;
    T2<double>* S;                   // per step K / 2 x 64 plane pairs: b in, x out
    u64* yh;                         // per workgroup, column and plane: the last row, tagged
    u64* zh;                         // per workgroup and step 2 x 64: the last plane, tagged
    SorCtl c;
};

template <bool BWD>
__global__ void __launch_bounds__(64) k_sor7(Sor7Args A) {
    constexpr int K = Sor7::K, SB = Sor7::SB, D = Sor7::D;
    const int r = threadIdx.x, o = blockIdx.x, ns = A.ns, ng = A.ng;
    const int os = o % ns, og = o / ns;
    const int s = BWD ? ns - 1 - os : os, g = BWD ? ng - 1 - og : og, rho = BWD ? 63 - r : r;
    const int Tp = A.Tp, ncol = A.mx - 2;
    const bool rl = 64 * s + rho < A.my - 2;
    const int sh = BWD ? Tp - (ncol + 63 + K - 1) : 0;
    const int off = sh + r;                               // plane 0's column is t - off
    const __amdgpu_buffer_rsrc_t Sr = buffer_of(A.S + ((long)(g * ns + s) * Tp) * (K / 2) * 64, Tp * (K / 2) * 1024u);
    const unsigned v16 = rho * 16u, v8 = r * 8u;
    const double inv = 1.0 / A.d;
    const long ysz = (long)ncol * K * 2, zsz = (long)(Tp + K - 1) * 128;
    const bool hy = os > 0, hz = og > 0;
    u64* const yout = A.yh + o * ysz;
    const u64* const yin = A.yh + (hy ? o - 1 : 0) * ysz;
    char* const zout = (char*)(A.zh + o * zsz);
    const char* const zin = (const char*)(A.zh + (hz ? o - ns : 0) * zsz + (K - 1) * 128);
    int planes[K];                                        // live planes, in sweep order
#pragma unroll
    for (int kk = 0; kk < K; ++kk) planes[kk] = g * K + (BWD ? K - 1 - kk : kk) < A.mz - 2;
    const bool full = 64 * s + 64 <= A.my - 2 && g * K + K <= A.mz - 2;
    const unsigned tag = sor_tag(A.c, BWD), want = tag + A.c.extra;
    bool dead = __builtin_amdgcn_readfirstlane((int)sor_dead(A.c)) != 0;
    __shared__ double ybuf[2][SB * K];     // the previous strip's last row, of a batch's steps
    __shared__ double obuf[SB * K][64];    // the batch's results
    const int ye = r / K, yk = r % K;      // lane r < SB * K carries step ye, plane yk

    struct Ops {
        T2<double> v[SB][K / 2];
        Tagged z[SB];            // the previous group's last plane at the lane's column
        Tagged y;                // lane r < SB * K: the previous strip's last row, of the batch after
    } ops[D];

    auto yload = [&](int t0, Ops& P) {
        const int c = min(max(t0 + min(ye, SB - 1) - yk - sh, 0), ncol - 1);
        P.y.lo = ld_word(yin + 2 * (c * K + yk));
        P.y.hi = ld_word(yin + 2 * (c * K + yk) + 1);
    };
    auto zload = [&](int t0, Ops& P) {
#pragma unroll
        for (int e = 0; e < SB; ++e) {
            const char* const p = zin + (long)(t0 + e) * 1024;
            P.z[e].lo = ld_word((const u64*)(p + v8));
            P.z[e].hi = ld_word((const u64*)(p + 512 + v8));
        }
    };
    // every path issues the same loads, so that the compiler can count them
    auto load = [&](int t0, Ops& P) {
        yload(t0 + SB, P);
        zload(t0, P);
#pragma unroll
        for (int e = 0; e < SB; ++e) {
            const unsigned tf = BWD ? Tp - 1 - (t0 + e) : t0 + e;
#pragma unroll
            for (int p = 0; p < K / 2; ++p) P.v[e][p] = buffer_ld2(Sr, v16, (tf * (K / 2) + p) * 1024u);
        }
    };
    auto yneed = [&](int t0) {
        const int c = t0 + ye - yk - sh;
        return hy && r < SB * K && c >= 0 && c < ncol;
    };
    auto zready = [&](int t0, const Ops& P) {
        bool ok = true;
#pragma unroll
        for (int e = 0; e < SB; ++e) {
            const int c = t0 + e - off;
            ok = ok && (!(rl && (unsigned)c < (unsigned)ncol) || P.z[e].is(want));
        }
        return (bool)__all(ok);
    };
    double xs[K];
#pragma unroll
    for (int kk = 0; kk < K; ++kk) xs[kk] = 0.0;
    // the steps of a batch; edge: some point is off the grid
    auto steps = [&](int t0, const Ops& P, bool edge) {
        const double* const yb = ybuf[(t0 / SB) & 1];
#pragma unroll
        for (int e = 0; e < SB; ++e) {
            const int t = t0 + e, c0 = t - off;
            const unsigned tf = BWD ? Tp - 1 - t : t;
            const double z0 = hz && (!edge || (rl && (unsigned)c0 < (unsigned)ncol)) ? P.z[e].value() : 0.0;
            double keep[K];
#pragma unroll
            for (int kk = K - 1; kk >= 0; --kk) {      // plane kk - 1 still holds the step before
                const int kf = BWD ? K - 1 - kk : kk;
                const double nb = wave_shr1(xs[kk], yb[e * K + kk]);
                const double below = kk ? xs[kk > 0 ? kk - 1 : 0] : z0;
                const double own = xs[kk];
                double sum = (kf & 1) ? P.v[e][kf / 2].b : P.v[e][kf / 2].a;
                if (!BWD) {
                    sum += A.sz * below;
                    sum += A.sy * nb;
                    sum += A.sx * own;
                } else {
                    sum += A.sx * own;
                    sum += A.sy * nb;
                    sum += A.sz * below;
                }
                xs[kk] = sum * inv;
                // S is zero off the grid: the backward sweep starts from those points
                keep[kf] = BWD ? xs[kk]
                               : (!edge || (rl && planes[kk] && (unsigned)(c0 - kk) < (unsigned)ncol) ? sum : 0.0);
                obuf[e * K + kk][r] = xs[kk];
            }
#pragma unroll
            for (int p = 0; p < K / 2; ++p)
                buffer_st2(Sr, v16, (tf * (K / 2) + p) * 1024u, keep[2 * p], keep[2 * p + 1]);
            if (og < ng - 1) {
                char* const p = zout + (long)t * 1024;
                st_tagged((u64*)(p + v8), (u64*)(p + 512 + v8), xs[K - 1], tag);
            }
        }
    };
    // waits for the words of batch t0's planes and of the next batch's rows
    auto wait = [&](int t0, Ops& P, int q) {
        const bool need = yneed(t0 + SB);
        if (!dead && !((!hz || zready(t0, P)) && (!hy || __all(!need || P.y.is(want))))) {
            long spins = 0;
            do {
                dead = sor_give_up(A.c, spins);
                zload(t0, P);
                yload(t0 + SB, P);
            } while (!dead && !((!hz || zready(t0, P)) && (!hy || __all(!need || P.y.is(want)))));
            // the words of the batches after were loaded too early as well
#pragma unroll
            for (int h = 1; h < D; ++h) {
                zload(min(t0 + h * SB, Tp - SB), ops[(q + h) % D]);
                yload(t0 + h * SB + SB, ops[(q + h) % D]);
            }
            __builtin_amdgcn_s_waitcnt(0);   // so that the other path's waits stay as they are
        }
        if (r < SB * K) ybuf[((t0 / SB) & 1) ^ 1][r] = need ? P.y.value() : 0.0;
        wave_lds_order();
    };
    {   // the first batch's rows
        Ops first;
        yload(0, first);
        const bool need = yneed(0);
        long spins = 0;
        while (!dead && !__all(!need || first.y.is(want))) {
            dead = sor_give_up(A.c, spins);
            yload(0, first);
        }
        if (r < SB * K) ybuf[0][r] = need ? first.y.value() : 0.0;
        __builtin_amdgcn_s_waitcnt(0);
    }
#pragma unroll
    for (int q = 0; q < D; ++q) load(q * SB, ops[q]);
    for (int t0 = 0; t0 < Tp; t0 += SB * D) {
#pragma unroll
        for (int q = 0; q < D; ++q) {
            const int t = t0 + q * SB;
            wait(t, ops[q], q);
            if (full && t - sh >= 63 + K - 1 && t + SB - sh <= ncol) steps(t, ops[q], false);
            else steps(t, ops[q], true);
            wave_lds_order();
            if (os < ns - 1) {             // the last lane's results, at their columns
                const int c = t + ye - 63 - yk - sh;
                const double v = obuf[r & (SB * K - 1)][63];
                if (r < SB * K && c >= 0 && c < ncol)
                    st_tagged(yout + 2 * (c * K + yk), yout + 2 * (c * K + yk) + 1, v, tag);
            }
            wave_lds_order();
            load(min(t + SB * D, Tp - SB), ops[q]);
        }
    }
    if (BWD && o == ns * ng - 1 && r == 0) A.c.ctl[1] += 1;
}

// r in natural order into the sweep's order (zeros off the grid), and the
// sweep's result back with the smoother's recurrence y = a p + c q + e z (p
// or q may be null): rows are moved along x on the natural side and by step
// on the other, through LDS.  Tiles of 64 steps; grid (Tp / 64, strips x
// groups), 256 threads; the result's blocks past Tp / 64 take the boundary,
// where z = r / db.
__global__ void __launch_bounds__(256)
k_sor7_pack(int mx, int my, int mz, int Tp, int ns, const double* __restrict__ r, T2<double>* __restrict__ S) {
    constexpr int K = Sor7::K;
    __shared__ double tile[2][64][65];
    const int t0 = blockIdx.x * 64, blk = blockIdx.y, s = blk % ns, g = blk / ns;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    for (int p = 0; p < K / 2; ++p) {
        for (int h = 0; h < 2; ++h) {
            const int kk = 2 * p + h, k = g * K + kk;
            for (int rho = w; rho < 64; rho += 4) {
                const int c = t0 + l - rho - kk, row = 64 * s + rho;
                double v = 0.0;
                if (c >= 0 && c < mx - 2 && row < my - 2 && k < mz - 2)
                    v = r[((long)(k + 1) * my + row + 1) * mx + c + 1];
                tile[h][rho][l] = v;
            }
        }
        __syncthreads();
        for (int tt = w; tt < 64; tt += 4)
            S[(((long)blk * Tp + t0 + tt) * (K / 2) + p) * 64 + l] = T2<double>{tile[0][l][tt], tile[1][l][tt]};
        __syncthreads();
    }
}

__device__ __forceinline__ double sor_comb(double z, long m, double a, const double* __restrict__ p, double c,
                                           const double* __restrict__ q, double e) {
    double v = e * z;
    if (p) v += a * p[m];
    if (q) v += c * q[m];
    return v;
}

__global__ void __launch_bounds__(256)
k_sor7_unpack(int mx, int my, int mz, int Tp, int ns, const T2<double>* __restrict__ S, const double* __restrict__ r,
              double db, double a, const double* __restrict__ p, double c, const double* __restrict__ q, double e,
              double* __restrict__ y) {
    constexpr int K = Sor7::K;
    const int nt = Tp / 64;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if ((int)blockIdx.x >= nt) {          // the boundary, row by row of each plane
        const double idb = 1.0 / db;
        const long rows = (long)my * mz, nblk = (long)(gridDim.x - nt) * gridDim.y;
        for (long R = ((long)(blockIdx.x - nt) * gridDim.y + blockIdx.y) * 4 + w; R < rows; R += nblk * 4) {
            const int j = (int)(R % my), k = (int)(R / my);
            const bool all = j == 0 || j == my - 1 || k == 0 || k == mz - 1;
            const long m0 = R * mx;
            if (all)
                for (int i = l; i < mx; i += 64) y[m0 + i] = sor_comb(r[m0 + i] * idb, m0 + i, a, p, c, q, e);
            else if (l < 2)
                y[m0 + l * (mx - 1)] = sor_comb(r[m0 + l * (mx - 1)] * idb, m0 + l * (mx - 1), a, p, c, q, e);
        }
        return;
    }
    __shared__ double tile[2][64][65];
    const int t0 = blockIdx.x * 64, blk = blockIdx.y, s = blk % ns, g = blk / ns;
    for (int pp = 0; pp < K / 2; ++pp) {
        for (int tt = w; tt < 64; tt += 4) {
            const T2<double> v = S[(((long)blk * Tp + t0 + tt) * (K / 2) + pp) * 64 + l];
            tile[0][l][tt] = v.a;
            tile[1][l][tt] = v.b;
        }
        __syncthreads();
        for (int h = 0; h < 2; ++h) {
            const int kk = 2 * pp + h, k = g * K + kk;
            for (int rho = w; rho < 64; rho += 4) {
                const int cc = t0 + l - rho - kk, row = 64 * s + rho;
                if (cc >= 0 && cc < mx - 2 && row < my - 2 && k < mz - 2) {
                    const long m = ((long)(k + 1) * my + row + 1) * mx + cc + 1;
                    y[m] = sor_comb(tile[h][rho][l], m, a, p, c, q, e);
                }
            }
        }
        __syncthreads();
    }
}

}  // namespace p4g
