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
//    lines with addresses known at compile time; operands are loaded batches
//    of steps early.
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
// checks ctl[0] after the call (sor_pipes_check).  `extra` is added to every awaited tag (0;
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
// a store is dropped; voff per lane, soff uniform.  16-byte stores take no
// uniform register offset: a store of more than 8 bytes reads its data late,
// and an instruction right behind it that writes one of its registers needs a
// wait state between, which the compiler leaves out where the offset is in a
// register.  With other kernels on the GPU such stores then stored the next
// instruction's result (the low half of a sum, an error of 1e-9 in one of ten
// applications with five solvers at once).
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
__device__ __forceinline__ void buffer_st2(__amdgpu_buffer_rsrc_t b, unsigned voff, double v0, double v1) {
    const long long p = __double_as_longlong(v0), q = __double_as_longlong(v1);
    __builtin_amdgcn_raw_buffer_store_b128(
        u32x4{(unsigned)p, (unsigned)(p >> 32), (unsigned)q, (unsigned)(q >> 32)}, b, (int)voff, 0, 0);
}
// the sweep's control words and the state of its waits (uniform)
struct SorCtl {
    unsigned* ctl;        // [0] stalled, [1] sweeps done
    long spin_limit;
    unsigned extra;
};

// the levels' control words after a call that stalled or was cut short: no
// stall, and tags that such a call has not used (a workgroup that started late
// in a stalled backward sweep may have tagged its words for the next one)
__global__ void k_sor_reset(int nlev, unsigned* ctl) {
    for (int l = threadIdx.x; l < nlev; l += 64) {
        ctl[2 * l] = 0;
        ctl[2 * l + 1] += 1;
    }
}

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
        if ((threadIdx.x & 63) == 0) atomicExch(c.ctl, 1u);
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
//
// A strip is one workgroup on a compute unit of its own, and its waves have
// one task each, so that the chain's wave (a lone wave issues an instruction
// in four cycles, and a step's chain is 14 ns) does nothing but the steps:
//   wave 0  the chain: operands from LDS, results to LDS, S to memory;
//   wave 1  the previous strip's row: polls 64 columns at once;
//   wave 2  the strip's own last row to the next strip;
//   wave 3 (and 4)  step-ordered operands, NR batches ahead;
//   the last wave  rows read along x and turned into steps (forward, b), or
//           steps turned into rows and written (backward, x).
// They meet in LDS words that count batches: a batch of SB steps is computed
// when every word exceeds its index.  Measured, forward + backward: 1025^2
// 5-point 336 -> 189 us, 513^2 9-point 342 -> 221 us against one wave a strip
// that did all of it (a step 37-47 -> 25 ns in 5-point, 75 -> 55 in 9-point,
// which moves 3 KB a step through one compute unit).  What is left: about
// 2.7 us from strip to strip (0.3 to be seen and sent, 0.6 through L2, a
// batch at either end) and 3 us to start.
constexpr int kXcds = 8;

template <bool NINE>
struct Sor2 {
    static constexpr int SB = NINE ? 8 : 16;          // steps per batch
    static constexpr int P0 = NINE ? 127 : 63;        // steps from a column at lane 0 to lane 63
    static constexpr int PAD = 192;                   // slots before column 0
    static constexpr int ND = NINE ? 2 : 1;           // operand waves
    static constexpr int NT = 64 * (4 + ND);
    static constexpr int NR = NINE ? 5 : 8, NO = 4;   // batches of operands and of results in LDS
    static constexpr int VS = 1024 + (NINE ? 128 : 64);         // bytes of a pair of steps (turned without bank conflicts)
    static constexpr int AB = NINE ? SB * 2048 : 0;             // a batch's couplings,
    static constexpr int IB = NINE ? SB / 2 * 1024 : 0;         //   reciprocal diagonals
    static constexpr int OB = SB / 2 * VS;                      //   and values (or results)
    static constexpr int OPB = AB + IB + OB;
    static constexpr int YN = 256;                              // neighbour-row steps in LDS
    static constexpr int LO = NR * OPB, LY = LO + NO * OB, LW = LY + YN * 8, LD = LW + 64;
    static constexpr size_t LDS = LD + 256;
    // slots of a strip's handed-over row: every window's, in range or not
    __host__ __device__ static long slots(int Tp) { return Tp + PAD + 64; }
    // steps of a strip, padded to whole batches and tiles of k_sor9_pack
    __host__ __device__ static int steps(int mx) {
        const int need = NINE ? mx + 128 : mx - 2 + 63;
        return (need + 31) / 32 * 32;
    }
    __host__ __device__ static int cols(int mx) { return NINE ? mx : mx - 2; }
    __host__ __device__ static int rows(int my) { return NINE ? my : my - 2; }
    __host__ __device__ static int strips(int my) { return (rows(my) + 63) / 64; }
    // strip o's block: runs of 32 strips on one XCD, whose L2 hands rows over
    // soonest (264-271 ns one way against 330-494), in dispatch order.  A
    // launch takes 256 strips at most, a compute unit each, so that an XCD's
    // strips wait for lower ones on it or on a lower XCD only, also where
    // several sweeps share the GPU.  (Sweeps of up to 32 strips of several
    // solvers meet on XCD 0; measured, an application at 1025^2, 16 strips, with
    // 1 / 2 / 4 / 8 solvers at once: 1.98 / 2.05 / 4.08 / 6.3 ms, and at 257^2,
    // where eight solvers' strips together have a compute unit each, 0.74 / 0.76 /
    // 1.49 / 2.26: the queues set this, not the compute units.)
    static constexpr int NSTRIP = 32 * kXcds;
    __host__ __device__ static int block_of(int o) { return o * kXcds + (o >> 5); }
    __host__ __device__ static int blocks(int ns) { return block_of(ns - 1) + 1; }
};

struct Sor2Args {
    int mx, my, Tp, ns, o0;          // strips, and the launch's first (in sweep order)
    double d, db, sx, sy;            // 5-point
    const T2<double>* pk;            // 9-point: per step 4 x 64 coefficient pairs (k_sor9_pack)
    const T2<double>* inv;           // 9-point: reciprocal diagonals, two steps per pair
    const double* b;
    T2<double>* S;                   // two steps per pair
    double* x;
    u64* yh;                         // per strip G::slots(Tp) tagged values: the strip's last row
    SorCtl c;
};

typedef volatile __attribute__((address_space(3))) int* lds_words;
typedef double f64x2 __attribute__((ext_vector_type(2)));

template <bool NINE, bool BWD>
__global__ void __launch_bounds__(Sor2<NINE>::NT) k_sor2(Sor2Args A) {
    typedef Sor2<NINE> G;
    constexpr int SB = G::SB, H = SB / 2, R = 64 / SB, lag = NINE ? 2 : 1;
    constexpr int kNever = 0x7fffffff;
    extern __shared__ __attribute__((aligned(16))) char sor_lds[];
    // the chain is the fourth wave: the one that shares its SIMD with no other
    // (waves go to the four SIMDs in turn; as the first of five the 5-point
    // chain took 31 ns a step, alone 24)
    const int r = threadIdx.x & 63, place = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = place == 3 ? 0 : (place == 0 ? 3 : place);
    const int mx = A.mx, my = A.my, ns = A.ns;
    const int nl = min(ns - A.o0, (int)G::NSTRIP), ol = (int)blockIdx.x >> 3, o = A.o0 + ol;
    if (!NINE && !BWD && (int)blockIdx.x >= G::blocks(nl)) {          // the boundary rows
        const double idb = 1.0 / A.db;
        const int per = 2 * mx + 2 * (my - 2), b0 = G::blocks(nl);
        for (int p = ((int)blockIdx.x - b0) * G::NT + threadIdx.x; p < per; p += (gridDim.x - b0) * G::NT) {
            long q;
            if (p < mx) q = p;
            else if (p < 2 * mx) q = (long)(my - 1) * mx + (p - mx);
            else q = (long)(1 + ((p - 2 * mx) >> 1)) * mx + (((p - 2 * mx) & 1) ? mx - 1 : 0);
            A.x[q] = A.b[q] * idb;
        }
        return;
    }
    if (ol >= nl || (int)blockIdx.x != G::block_of(ol)) return;
    const int Tp = A.Tp, NB = Tp / SB, ncol = G::cols(mx), nrow = G::rows(my);
    const int s = BWD ? ns - 1 - o : o;
    const int sh = BWD ? (NINE ? Tp - 2 - (mx + 126) : Tp - (ncol + 63)) : 0;
    // b and x: the rows of the strip, relative to the first; off the strip a
    // load gives zero and a store is dropped
    const long strip0 = ((long)64 * s + (NINE ? 0 : 1)) * mx;
    const unsigned nrows = min(64, nrow - 64 * s);
    const __amdgpu_buffer_rsrc_t br = buffer_of((BWD ? (const double*)A.x : A.b) + strip0, nrows * mx * 8u);
    const __amdgpu_buffer_rsrc_t Sr = buffer_of(A.S + (long)s * (Tp / 2) * 64, Tp * 512u);
    const unsigned v16 = (BWD ? 63 - r : r) * 16u;
    const unsigned tag = sor_tag(A.c, BWD), want = tag + A.c.extra;
    bool dead = __builtin_amdgcn_readfirstlane((int)sor_dead(A.c)) != 0;
    // the words: batches ready of each operand wave (the next of its own), of
    // the values and of the neighbour row, and the first batch without room
    // for its results
    enum { W_OP = 0, W_VAL = G::ND, W_Y, W_OUT, W_X };
    lds_words const words = (lds_words)(sor_lds + G::LW);
    lds_words const done = (lds_words)(sor_lds + G::LD);     // [lane]: batches computed
    if (threadIdx.x < 8) {
        int w = kNever;
        if ((int)threadIdx.x < G::ND) w = NINE || BWD ? (int)threadIdx.x : kNever;
        else if (threadIdx.x == W_VAL) w = BWD ? kNever : 0;
        else if (threadIdx.x == W_Y) w = 0;
        else if (threadIdx.x == W_OUT) w = o + 1 < ns ? G::NO : kNever;
        else if (threadIdx.x == W_X) w = BWD ? G::NO : kNever;
        words[threadIdx.x] = w;
    }
    if (threadIdx.x < 64) done[threadIdx.x] = 0;
    __syncthreads();
    // Waits inside the workgroup end with it.  Only wave 1 polls another
    // workgroup, and its limit is the one that counts: when it gives up it
    // releases the chain (W_Y), and the chain the rest.  These waits, the
    // chain's for W_Y among them, have a limit only so that no mistake can
    // make them endless: 64 polls of LDS (63 ns each) for each of wave
    // 1's polls through L2 (0.35 us), so wave 1 always comes first.
    const long inner_limit = (A.c.spin_limit << 6) + (1L << 16);
    auto inner_wait = [&](auto ready) __attribute__((always_inline)) {
        long spins = 0;
        while (!dead && !ready()) {
            if (++spins > inner_limit) {
                if (r == 0) atomicExch(A.c.ctl, 1u);
                dead = true;
                __builtin_amdgcn_s_waitcnt(0);      // so that the other path's waits stay as they are
            }
            if (wave) __builtin_amdgcn_s_sleep(1);
        }
        wave_lds_order();
    };

    if (wave == 0) {                        // ------------------------------- the chain
        __builtin_amdgcn_s_setprio(3);
        const double invd = NINE ? 0.0 : 1.0 / A.d;
        struct Ops {
            f64x2 v[H / 2], y[H / 2];       // b (forward) or S (backward), the neighbour row
            f64x2 a[NINE ? 2 * H : 1];      // the earlier (later) four couplings
            f64x2 inv[NINE ? H / 2 : 1];
        } P0, P1;
        const char* const mine = sor_lds + r * 16;
        auto read = [&](int slot, int k, int part, Ops& P) __attribute__((always_inline)) {
            const char* const p = mine + slot * G::OPB;
            const f64x2* const yp = (const f64x2*)(sor_lds + G::LY) + ((k * SB + part * H) & (G::YN - 1)) / 2;
#pragma unroll
            for (int e = 0; e < H / 2; ++e) {
                const int f = part * (H / 2) + e;
                P.y[e] = yp[e];
                P.v[e] = *(const f64x2*)(p + G::AB + G::IB + f * G::VS);
                if (NINE) {
                    P.inv[e] = *(const f64x2*)(p + G::AB + f * 1024);
#pragma unroll
                    for (int h = 0; h < 4; ++h) P.a[4 * e + h] = *(const f64x2*)(p + f * 4096 + h * 1024);
                }
            }
        };
        double h1 = 0.0, u1 = 0.0, u2 = 0.0;    // own last result; the neighbour row's last two
        auto steps = [&](int k, int oslot, int part, const Ops& P) __attribute__((always_inline)) {
            char* const op = sor_lds + G::LO + oslot * G::OB + r * 16;
            const unsigned vs = v16 + (k * SB + part * H) * 512u;
            f64x2 keep, kres;
#pragma unroll
            for (int e = 0; e < H; ++e) {
                // backward, a pair's later step is stored first
                const int g = BWD ? (e ^ 1) : e;
                const double u3 = u2;
                u2 = u1;
                u1 = wave_shr1(h1, P.y[e / 2][e & 1]);
                double sum = P.v[e / 2][(BWD ? g : e) & 1], res;
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
                    const f64x2 p0 = P.a[2 * e], p1 = P.a[2 * e + 1];
                    if (!BWD) {      // (j-1, i-1), (j-1, i), (j-1, i+1), (j, i-1)
                        sum -= p0[0] * u3;
                        sum -= p0[1] * u2;
                        sum -= p1[0] * u1;
                        sum -= p1[1] * h1;
                    } else {         // (j, i+1), (j+1, i-1), (j+1, i), (j+1, i+1)
                        sum -= p0[0] * h1;
                        sum -= p0[1] * u1;
                        sum -= p1[0] * u2;
                        sum -= p1[1] * u3;
                    }
                    res = sum * P.inv[e / 2][g & 1];
                }
                keep[e & 1] = sum;
                kres[e & 1] = res;
                h1 = res;
                if (e & 1) {
                    if (!BWD) buffer_st2(Sr, vs + (e / 2) * 1024u, keep[0], keep[1]);
                    *(f64x2*)(op + (part * H + e) / 2 * G::VS) = kres;
                }
            }
        };
        lds_words const my_word = words + (r & 7);
        inner_wait([&] { return __all(*my_word > 0); });
        read(0, 0, 0, P0);
        int slot = 0;
        for (int k = 0; k < NB; ++k) {
            const int w = *my_word;
            wave_lds_order();
            read(slot, k, 1, P1);
            steps(k, k & (G::NO - 1), 0, P0);
            slot = slot + 1 == G::NR ? 0 : slot + 1;
            if (__all(w > k + 1)) {
                read(slot, k + 1, 0, P0);
                steps(k, k & (G::NO - 1), 1, P1);
                wave_lds_order();
                done[r] = k + 1;
            } else {                 // what there is goes on to the next strip first
                steps(k, k & (G::NO - 1), 1, P1);
                wave_lds_order();
                done[r] = k + 1;
                inner_wait([&] { return __all(*my_word > k + 1); });
                read(slot, k + 1, 0, P0);
            }
        }
        return;
    }
    if (wave == 1) {                        // ------------------------------- the neighbour row
        double* const yl = (double*)(sor_lds + G::LY);
        if (o == 0) {
            for (int q = r; q < G::YN; q += 64) yl[q] = 0.0;
        } else {
            const char* const yin = (const char*)(A.yh + ((long)(o - 1) * G::slots(Tp) + G::PAD - sh + r) * 2);
            long spins = 0;
            for (int t = 0; t < Tp;) {
                inner_wait([&] { return __builtin_amdgcn_readfirstlane(done[0]) * SB + G::YN >= t + 64; });
                if (dead) break;
                const int slot = t + r - sh;
                const bool need = slot >= 0 && slot < ncol;
                const char* const p = yin + (long)t * 16;
                Tagged w;
                w.lo = ld_word((const u64*)p);
                w.hi = ld_word((const u64*)(p + 8));
                const unsigned long long bad = __ballot(need && !w.is(want));
                const int n = bad ? (int)__builtin_ctzll(bad) / SB * SB : 64;
                if (n > 0) {
                    if (r < n) yl[(t + r) & (G::YN - 1)] = need ? w.value() : 0.0;
                    t += n;
                    wave_lds_order();
                    words[W_Y] = t / SB;
                    spins = 0;
                } else if (sor_give_up(A.c, spins)) {
                    break;
                }
            }
        }
        wave_lds_order();
        words[W_Y] = kNever;
        return;
    }

    // tasks of the waves 2.., in batches: a lane of those that turn rows into
    // steps (or back) has step te of a batch and rows r0, r0 + R, ..
    const int te = r & (SB - 1), r0 = r / SB;
    const int c0 = te - sh - (NINE ? 1 : 0) - lag * r0;          // its column at batch 0, row r0
    const int rho0 = BWD ? 63 - r0 : r0, x0 = NINE ? 0 : 1;
    const unsigned va = (unsigned)(rho0 * mx + x0 + (BWD ? ncol - 1 - c0 : c0)) * 8u;
    const int dva = (BWD ? -1 : 1) * R * (mx - lag) * 8;         // from row to row
    // batches t of the whole strip's rows and no column off the grid
    const bool full = nrows == 64;
    auto inside = [&](int t) { return full && t >= sh + G::P0 && t + SB - sh <= ncol; };
    const unsigned turned = (te >> 1) * G::VS + r0 * 16u + (te & 1) * 8u;
    // b by rows into steps; GD batches of loads in flight, in whole rounds (a
    // batch past the last one reads nothing and is not computed), so that the
    // compiler can count them
    constexpr int GD = 4;
    auto turn = [&](int word) __attribute__((always_inline)) {
        double g[GD][SB];
        auto ask = [&](int k, double (&v)[SB]) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < SB; ++q) {
                const bool live = (unsigned)(k * SB + c0 - q * R * lag) < (unsigned)ncol;
                v[q] = buffer_ld(br, live ? va + k * SB * 8u + q * dva : 0x80000000u);
            }
        };
#pragma unroll
        for (int h = 0; h < GD; ++h) {
            ask(h, g[h]);
            __builtin_amdgcn_sched_barrier(0);      // in this order, as the loop does
        }
        for (int k = 0; k < NB; k += GD) {
#pragma unroll
            for (int h = 0; h < GD; ++h) {
                inner_wait([&] { return __builtin_amdgcn_readfirstlane(done[0]) + G::NR > k + h; });
                char* const p = sor_lds + (k + h) % G::NR * G::OPB + G::AB + G::IB + turned;
#pragma unroll
                for (int q = 0; q < SB; ++q) *(double*)(p + q * R * 16) = g[h][q];
                wave_lds_order();
                words[word] = k + h + 1;
                ask(k + h + GD, g[h]);
            }
        }
        words[word] = kNever;
    };
    // batches of results as the chain leaves them in LDS
    auto results = [&](int word, auto take) __attribute__((always_inline)) {
        for (int k = 0; k < NB; ++k) {
            inner_wait([&] { return __builtin_amdgcn_readfirstlane(done[0]) > k; });
            take(sor_lds + G::LO + (k & (G::NO - 1)) * G::OB, k * SB);
            wave_lds_order();
            words[word] = k + 1 + G::NO;
        }
    };
    if (wave == 2) {                        // ------------------------------- the last row, to the next strip
        char* const yout = (char*)(A.yh + ((long)o * G::slots(Tp) + G::PAD - G::P0 - sh + te) * 2);
        if (o + 1 < ns) {
            results(W_OUT, [&](const char* ob, int t) __attribute__((always_inline)) {
                const int slot = t + te - G::P0 - sh;
                const double v = *(const double*)(ob + (te >> 1) * G::VS + 63 * 16 + (te & 1) * 8);
                char* const p = yout + (long)t * 16;
                if (r < SB && slot >= 0 && slot < ncol) st_tagged((u64*)p, (u64*)(p + 8), v, tag);
            });
        }
        return;
    }
    if (wave == 3 + G::ND) {                // ------------------------------- rows
        if (!BWD) {
            turn(W_VAL);
        } else {
            results(W_X, [&](const char* ob, int t) __attribute__((always_inline)) {
                double xv[SB];
#pragma unroll
                for (int q = 0; q < SB; ++q) xv[q] = *(const double*)(ob + turned + q * R * 16);
                if (inside(t)) {
#pragma unroll
                    for (int q = 0; q < SB; ++q) buffer_st(br, va - t * 8u + q * dva, xv[q]);
                } else {
#pragma unroll
                    for (int q = 0; q < SB; ++q) {
                        const int c = t + c0 - q * R * lag;
                        const bool live = (unsigned)c < (unsigned)ncol && (unsigned)(rho0 - q * R) < nrows;
                        buffer_st(br, live ? va - t * 8u + q * dva : 0x80000000u, xv[q]);
                    }
                }
            });
            if (o == ns - 1 && r == 0) A.c.ctl[1] += 1;
        }
        return;
    }
    if constexpr (!NINE) {                  // ------------------------------- 5-point sums
        if (BWD) {                          // S; off the grid it is left as the forward sweep's chain ran on
            f64x2 g[GD][H];
            const bool rl = 64 * s + 63 - r < nrow;
            auto ask = [&](int k, f64x2 (&v)[H]) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < H; ++e) {
                    const T2<double> t = buffer_ld2(Sr, v16, (unsigned)((Tp - 2 - (k * SB + 2 * e)) >> 1) * 1024u);
                    v[e] = f64x2{t.a, t.b};
                }
            };
#pragma unroll
            for (int h = 0; h < GD; ++h) {
                ask(min(h, NB - 1), g[h]);
                __builtin_amdgcn_sched_barrier(0);      // in this order, as the loop does
            }
            for (int k = 0; k < NB; k += GD) {
#pragma unroll
                for (int h = 0; h < GD; ++h) {
                    inner_wait([&] { return __builtin_amdgcn_readfirstlane(done[0]) + G::NR > k + h; });
                    char* const p = sor_lds + (k + h) % G::NR * G::OPB + r * 16;
                    const int c = (k + h) * SB - sh - r;
                    if (!inside((k + h) * SB)) {
#pragma unroll
                        for (int e = 0; e < H; ++e) {     // (a pair's later step comes first)
                            if (!rl || (unsigned)(c + 2 * e) >= (unsigned)ncol) g[h][e][1] = 0.0;
                            if (!rl || (unsigned)(c + 2 * e + 1) >= (unsigned)ncol) g[h][e][0] = 0.0;
                        }
                    }
#pragma unroll
                    for (int e = 0; e < H; ++e) *(f64x2*)(p + e * G::VS) = g[h][e];
                    wave_lds_order();
                    words[W_OP] = k + h + 1;
                    ask(min(k + h + GD, NB - 1), g[h]);
                }
            }
            words[W_OP] = kNever;
        }
    } else {                                // ------------------------------- 9-point operands
        const int i = wave - 3;
        const __amdgpu_buffer_rsrc_t Ir = buffer_of(A.inv + (long)s * (Tp / 2) * 64, Tp * 512u);
        const __amdgpu_buffer_rsrc_t Kr = buffer_of(A.pk + (long)s * Tp * 256, Tp * 4096u);
        const unsigned vk = v16 + (BWD ? 2048u : 0u);
        constexpr int NL = 2 * SB + H * (BWD ? 2 : 1), GW = 2;   // loads of a batch, batches in flight
        f64x2 g[GW][NL];
        auto ld = [&](__amdgpu_buffer_rsrc_t b, unsigned vo, unsigned so) __attribute__((always_inline)) {
            const T2<double> t = buffer_ld2(b, vo, so);
            return f64x2{t.a, t.b};
        };
        auto ask = [&](int k, f64x2 (&v)[NL]) __attribute__((always_inline)) {
            const int t = min(k, NB - 1) * SB;
#pragma unroll
            for (int e = 0; e < H; ++e) {
                const int m = BWD ? (Tp - 2 - (t + 2 * e)) >> 1 : (t + 2 * e) >> 1;    // pair of steps
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const unsigned tf = BWD ? Tp - 1 - (t + 2 * e + h) : t + 2 * e + h;
                    v[2 * (2 * e + h)] = ld(Kr, vk, tf * 4096u);
                    v[2 * (2 * e + h) + 1] = ld(Kr, vk + 1024u, tf * 4096u);
                }
                v[2 * SB + e] = ld(Ir, v16, m * 1024u);
                if (BWD) v[2 * SB + H + e] = ld(Sr, v16, m * 1024u);
            }
        };
#pragma unroll
        for (int h = 0; h < GW; ++h) {
            ask(i + h * G::ND, g[h]);
            __builtin_amdgcn_sched_barrier(0);      // in this order, as the loop does
        }
        int sl = i;
        for (int k = i; k < NB; k += GW * G::ND) {
#pragma unroll
            for (int h = 0; h < GW; ++h) {
                const int kk = k + h * G::ND;
                inner_wait([&] { return __builtin_amdgcn_readfirstlane(done[0]) + G::NR > kk; });
                char* const p = sor_lds + sl * G::OPB + r * 16;
                sl = sl + G::ND >= G::NR ? sl + G::ND - G::NR : sl + G::ND;
#pragma unroll
                for (int e = 0; e < 2 * SB; ++e) *(f64x2*)(p + e * 1024) = g[h][e];
#pragma unroll
                for (int e = 0; e < H; ++e) {
                    *(f64x2*)(p + G::AB + e * 1024) = g[h][2 * SB + e];
                    if (BWD) *(f64x2*)(p + G::AB + G::IB + e * G::VS) = g[h][2 * SB + H + e];
                }
                wave_lds_order();
                words[W_OP + i] = kk + G::ND;
                ask(kk + GW * G::ND, g[h]);
            }
        }
        words[W_OP + i] = kNever;
    }
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
// step, tagged; its last row to the next strip as in 2D.  Bound by the
// hand-over from group to group (257^3: 63 of them at 5-6 us each, in sweeps
// of 467 us forward and 402 us backward; a step is 0.22 us), so the words are
// asked for half a batch before they are needed: four batches ahead, they were
// asked for too early and a group settled four batches behind the one before
// (sweeps run on their own over and over: 393 us, four batches ahead 553 us,
// batches of 2 steps 415 us).  A level holds S, padded to whole strips and
// steps, and every group's last plane besides the solver's vectors (257^3: 1.5
// and 0.75 vectors).
constexpr int kSor7Planes = 4;

struct Sor7 {
    static constexpr int K = kSor7Planes, SB = 4, D = 4;
    // steps of a strip, in whole tiles of the pack kernels: its columns, and
    // the lag of the last row and plane.  A single strip's last row may come
    // before lane 63 (a 5^3 level took 128 steps for 8, now 64: an application
    // 349 -> 242 us, 306 with the flagged strips that these sweeps replaced)
    __host__ __device__ static int steps(int mx, int my) {
        const int need = mx - 2 + (strips(my) > 1 ? 63 : my - 3) + K - 1;
        static_assert(64 % (SB * D) == 0, "whole tiles of the pack kernels, whole rounds of the ring");
        return (need + 63) / 64 * 64;
    }
    __host__ __device__ static int strips(int my) { return (my - 2 + 63) / 64; }
    // workgroup o's block, in dispatch order: an eighth of the workgroups, but
    // no fewer than 32, on one XCD
    __host__ __device__ static int block_of(int o, int nwg) {
        return o * kXcds + o / (nwg > 32 * kXcds ? (nwg + kXcds - 1) / kXcds : 32);
    }
    __host__ __device__ static int blocks(int nwg) { return block_of(nwg - 1, nwg) + 1; }
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
    const int r = threadIdx.x, o = blockIdx.x >> 3, ns = A.ns, ng = A.ng;
    if ((int)blockIdx.x != Sor7::block_of(o, ns * ng)) return;
    const int os = o % ns, og = o / ns;
    const int s = BWD ? ns - 1 - os : os, g = BWD ? ng - 1 - og : og, rho = BWD ? 63 - r : r;
    const int Tp = A.Tp, ncol = A.mx - 2;
    const bool rl = 64 * s + rho < A.my - 2;
    const int sh = BWD ? Tp - (ncol + 63 + K - 1) : 0;    // (below zero where a single strip's lanes start late)
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

    T2<double> ops[D][SB][K / 2];
    struct Words {               // loaded half a batch ahead: any earlier, and they are not there yet
        Tagged z[SB];            // the previous group's last plane at the lane's column
        Tagged y;                // lane r < SB * K: the previous strip's last row, of the batch after
    } zw[2];

    auto yload = [&](int t0, Words& P) {
        const int c = min(max(t0 + min(ye, SB - 1) - yk - sh, 0), ncol - 1);
        P.y.lo = ld_word(yin + 2 * (c * K + yk));
        P.y.hi = ld_word(yin + 2 * (c * K + yk) + 1);
    };
    auto zload = [&](int t0, Words& P) {
#pragma unroll
        for (int e = 0; e < SB; ++e) {
            const char* const p = zin + (long)(t0 + e) * 1024;
            P.z[e].lo = ld_word((const u64*)(p + v8));
            P.z[e].hi = ld_word((const u64*)(p + 512 + v8));
        }
    };
    // every path issues the same loads, so that the compiler can count them
    auto load = [&](int t0, T2<double> (&P)[SB][K / 2]) {
#pragma unroll
        for (int e = 0; e < SB; ++e) {
            const unsigned tf = BWD ? Tp - 1 - (t0 + e) : t0 + e;
#pragma unroll
            for (int p = 0; p < K / 2; ++p) P[e][p] = buffer_ld2(Sr, v16, (tf * (K / 2) + p) * 1024u);
        }
    };
    auto yneed = [&](int t0) {
        const int c = t0 + ye - yk - sh;
        return hy && r < SB * K && c >= 0 && c < ncol;
    };
    auto zready = [&](int t0, const Words& P) {
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
    // half the steps of a batch; edge: some point is off the grid
    auto steps = [&](int t0, const T2<double> (&P)[SB][K / 2], const Words& W, bool edge, int E) __attribute__((always_inline)) {
        const double* const yb = ybuf[(t0 / SB) & 1];
#pragma unroll
        for (int e = E; e < E + SB / 2; ++e) {
            const int t = t0 + e, c0 = t - off;
            const unsigned tf = BWD ? Tp - 1 - t : t;
            const double z0 = hz && (!edge || (rl && (unsigned)c0 < (unsigned)ncol)) ? W.z[e].value() : 0.0;
            double keep[K];
#pragma unroll
            for (int kk = K - 1; kk >= 0; --kk) {      // plane kk - 1 still holds the step before
                const int kf = BWD ? K - 1 - kk : kk;
                const double nb = wave_shr1(xs[kk], yb[e * K + kk]);
                const double below = kk ? xs[kk > 0 ? kk - 1 : 0] : z0;
                const double own = xs[kk];
                double sum = (kf & 1) ? P[e][kf / 2].b : P[e][kf / 2].a;
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
                buffer_st2(Sr, v16 + tf * (K / 2) * 1024u + p * 1024u, keep[2 * p], keep[2 * p + 1]);
            if (og < ng - 1) {
                char* const p = zout + (long)t * 1024;
                st_tagged((u64*)(p + v8), (u64*)(p + 512 + v8), xs[K - 1], tag);
            }
        }
    };
    // waits for the words of batch t0's planes and of the next batch's rows
    auto wait = [&](int t0, Words& P) __attribute__((always_inline)) {
        const bool need = yneed(t0 + SB);
        if (!dead && !((!hz || zready(t0, P)) && (!hy || __all(!need || P.y.is(want))))) {
            long spins = 0;
            do {
                dead = sor_give_up(A.c, spins);
                zload(t0, P);
                yload(t0 + SB, P);
            } while (!dead && !((!hz || zready(t0, P)) && (!hy || __all(!need || P.y.is(want)))));
            __builtin_amdgcn_s_waitcnt(0);   // so that the other path's waits stay as they are
        }
        if (r < SB * K) ybuf[((t0 / SB) & 1) ^ 1][r] = need ? P.y.value() : 0.0;
        wave_lds_order();
    };
    {   // the first batch's rows
        Words first;
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
    for (int q = 0; q < D; ++q) {
        load(q * SB, ops[q]);
        __builtin_amdgcn_sched_barrier(0);
    }
    zload(0, zw[0]);
    yload(SB, zw[0]);
    auto round = [&](int t0, bool edge) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < D; ++q) {
            const int t = t0 + q * SB;
            wait(t, zw[q & 1]);
            steps(t, ops[q], zw[q & 1], edge, 0);
            const int tn = min(t + SB, Tp - SB);
            zload(tn, zw[(q & 1) ^ 1]);
            yload(tn + SB, zw[(q & 1) ^ 1]);
            steps(t, ops[q], zw[q & 1], edge, SB / 2);
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
    };
    // three loops, because a ring that two paths of one loop load ends in
    // moves between registers
    int t0 = 0;
    const int lo = full ? sh + 63 + K - 1 : Tp, hi = ncol + sh - SB * D;
    for (; t0 < min(lo, Tp); t0 += SB * D) round(t0, true);
    for (; t0 <= hi; t0 += SB * D) round(t0, false);
    for (; t0 < Tp; t0 += SB * D) round(t0, true);
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
