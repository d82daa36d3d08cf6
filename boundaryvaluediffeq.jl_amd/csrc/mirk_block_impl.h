// mirk_block_impl.h -- MIRK collocation on gfx950 for larger state dimensions
// (M = 8, 16, 32; family LINEAR_TANH f = A y + c tanh(y)), one workgroup of NW
// wavefronts per BVP instance.
//
// The intervals of an instance are split over the waves of its workgroup:
//   * FP64 stage work (residual, defect, J d products) has no order: a wave takes
//     64 / M intervals at a time, one component per lane, its row of A in registers,
//     the stage arguments exchanged through a 512-byte LDS vector of the wave's own;
//   * the block elimination runs as one contiguous chunk of intervals per wave.  One
//     row of the stacked 2M x (3M+1) system [relation; new block row] lives in each
//     lane's registers for the whole chunk: the pivot row of a step is broadcast with
//     v_readlane, every other row is reduced (Gauss-Jordan, so the record needs no
//     triangular solve), the M lanes whose rows became pivots store their record and
//     take the rows of the next interval, and the other lanes keep the relation;
//   * the chunk relations are merged pairwise through LDS by the same elimination, and
//     the 2M x 2M end-node system is solved in FP64 by the first wave;
//   * corrections run back down the merges and then through every chunk in parallel.
// Jacobian blocks [S_k | R_k] come from the stage recursion in the factorisation
// precision LT.  With f's Jacobian A + c diag(sech^2) every product of two stage
// Jacobians is elementwise in A, A^2 and the diagonals; only MIRK6's last stage needs
// one A dY product, on the matrix cores (v_mfma_f32_16x16x4_f32) for LT = float, M >= 16.
// LT = float is the FP32 factorisation; FP64 iterative refinement then solves
// J d = -F with residuals r = -F - J d in FP64 (an exact one-direction derivative),
// each pushed through the stored multipliers.
//
// What bounds it: the elimination, per interval a chain of M pivot steps with a readlane
// and an FMA per column of the row (M = 32: 17.5 us per interval and wave at two waves
// per SIMD, about four fifths of a Newton iteration); the refinement steps cost 7% each.
// One wave per instance walking all intervals in order, its LDS object passed by reference
// (flat accesses) and the rows staged through LDS per interval, measured at
// M = 32, MIRK6, FP32 factors + 2 refinement steps: 1 instance of 301 intervals 120 ms,
// 64 instances of 272..720 intervals 300 ms; M = 16, MIRK4, FP64, 200 instances of
// 200..600 intervals 65 ms.  This split: 7.3 ms, 17.1 ms, 5.2 ms (5.1 ms with pivots compared in FP32).
// Reference counterparts as in mirk_wave_impl.h (MIRK/collocation.jl:44-102,
// MIRK/mirk.jl:697-862 and 927-1002, MIRK/adaptivity.jl:23-75, 250-304, 370-461).
#pragma once

#include <type_traits>

#include "mirk_wave_impl.h"

namespace bvpdev {

// Waves per instance: 8 (512 threads) leave 256 registers per lane, which the row of the
// M = 32 system (97 values), the tangent tiles and their addresses need.
// (M = 32 with FP64 blocks, component operations only: 4, by its LDS.)
// Short meshes in large batches, where most of the waves hold no chunk, pay too: 4,096 instances of
// 4 / 16 intervals, one wave per instance before and now, M = 8 FP64 1.30 / 4.85 -> 1.00 / 1.69 ms,
// M = 16 FP64 2.19 / 7.15 -> 2.16 / 4.21 ms, M = 32 FP32 17.9 / 43.8 -> 7.9 / 13.5 ms.
template <int M, typename LT> constexpr int kBlockWaves = (M == 32 && sizeof(LT) == 8) ? 4 : 8;
// Steps of the elimination per unrolled group.
template <int M, typename LT> constexpr int kBlockGroup = M < 16 ? M : 16;
// The factorisation is switched off for M = 32 with FP64 factors (an earlier kernel for it
// hung on the GPU; cause not identified): the entry points refuse it.
template <int M, typename LT> constexpr bool kBlockFactors = !(M == 32 && sizeof(LT) == 8);

template <int M, int METHOD, typename LT> struct BShared {
    static constexpr int NW = kBlockWaves<M, LT>;
    static constexpr int S = Tab<METHOD>::s;
    static constexpr int SW = 2 * M + 1;  // block row [S | R | rhs]; odd stride spreads rows over the banks
    double At[M][M];                      // A transposed (At[q][i] = A[i][q]): conflict-free lane reads
    // A and A^2 in the factorisation precision; the row stride puts the rows 4 (l / 16)
    // that the lanes of a matrix-core tile read together into different banks
    LT Al[M][M + 4], A2[M][M + 4];
    double c;
    struct Wave {
        alignas(16) double vec[WAVE];     // stage arguments of the wave's intervals, one component per lane
        alignas(16) double vv[2 * M];     // [d_a | d_{k+1}] of the back-substitution
        LT blk[M * SW];                   // block row handed to the pivot lanes; relations of the merges
        LT dd[S][M];                      // c sech^2(Y_r), the diagonal part of the stage Jacobians
    } wv[NW];
    double lo[NW][M], hi[NW][M];          // corrections at the chunk ends
    double xr[2 * M];
    double bcres[M];
    double red[3][NW];
    int bc_end[M], bcc[M];
    double bcv[M];
    int flag, item;
};

// The workgroup's LDS object.  Functions that are not inlined name it through this accessor
// instead of taking a reference: a reference is a generic pointer there, and every access
// through it a flat_* instruction.
template <int M, int METHOD, typename LT> __device__ __forceinline__ BShared<M, METHOD, LT> &bshared() {
    __shared__ BShared<M, METHOD, LT> sh;
    return sh;
}

// order LDS (and register) traffic between the lanes of one wave
__device__ __forceinline__ void wsync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// as wsync(), for memory other than LDS as well
struct WaveSync {
    __device__ void operator()() const {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
};

// wave w's contiguous chunk of N intervals over P = min(N, NW) waves (len = 0 past P)
template <int NW>
__device__ __forceinline__ void bchunk(int N, int w, int &P, int &start, int &len) {
    P = N < NW ? N : NW;
    if (w >= P) { start = N; len = 0; return; }
    const int q = N / P, r = N % P;
    len = q + (w < r ? 1 : 0);
    start = w * q + (w < r ? w : r);
}

template <typename T> __device__ inline T rdlane(T v, int l);
template <> __device__ inline float rdlane<float>(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
template <> __device__ inline double rdlane<double>(double v, int l) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Lane of the first maximum of v over the wave: an inclusive max-scan inside
// each row of 16 lanes and across rows with DPP moves (no LDS round trips), the
// maximum read from lane 63, the first lane holding it found by a ballot.
__device__ inline int wave_argmax_first(float v) {
    float m = v;
#define BVP_DPP_MAX(ctrl, rmask) \
    m = fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(m), __float_as_int(m), ctrl, rmask, 0xf, false)))
    BVP_DPP_MAX(0x111, 0xf);  // row_shr:1
    BVP_DPP_MAX(0x112, 0xf);  // row_shr:2
    BVP_DPP_MAX(0x114, 0xf);  // row_shr:4
    BVP_DPP_MAX(0x118, 0xf);  // row_shr:8
    BVP_DPP_MAX(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
    BVP_DPP_MAX(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef BVP_DPP_MAX
    const float mx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), 63));
    const unsigned long long b = __ballot(v == mx);
    return __builtin_amdgcn_readfirstlane(b ? __ffsll((long long)b) - 1 : 0);
}
// maximum of v over the wave, by the same moves
__device__ inline int wave_max_int(int v) {
#define BVP_DPP_MAX(ctrl, rmask) v = max(v, __builtin_amdgcn_update_dpp(v, v, ctrl, rmask, 0xf, false))
    BVP_DPP_MAX(0x111, 0xf);
    BVP_DPP_MAX(0x112, 0xf);
    BVP_DPP_MAX(0x114, 0xf);
    BVP_DPP_MAX(0x118, 0xf);
    BVP_DPP_MAX(0x142, 0xa);
    BVP_DPP_MAX(0x143, 0xc);
#undef BVP_DPP_MAX
    return __builtin_amdgcn_readlane(v, 63);
}

// Lane of the first maximum of |v| over the lanes that are not done, compared in the
// precision of v.  FP64: by the high words (whose order as integers is that of the values),
// and only where several lanes share the largest one by the low words too.
__device__ inline int pivot_lane(float v, bool done) { return wave_argmax_first(done ? -1.f : fabsf(v)); }
__device__ inline int pivot_lane(double v, bool done) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(v));
    const int hi = done ? -1 : (int)(b >> 32);
    const bool in = hi == wave_max_int(hi);
    unsigned long long c = __ballot(in);
    if (__builtin_expect((c & (c - 1)) != 0, 0)) {
        const int lo = in ? (int)((unsigned)b ^ 0x80000000u) : (int)0x80000000;
        const int ml = wave_max_int(lo);
        c = __ballot(in && lo == ml);
    }
    return __builtin_amdgcn_readfirstlane(__ffsll((long long)c) - 1);
}

// ------------------------------------------------------------------ records
// Per eliminated node k (and in the same slots the nodes between the chunks):
//   d_k = H - X d_a - Z d_c,   XZ[c][j] (c < M: X, else Z; row j = component), H[j].
// The FP32 factorisation also keeps the multipliers [j][lane] of its steps (the pivot
// lane's own entry: the inverse pivot) and per lane its pivot step and, in lanes < M,
// the pivot lane of that step, so that new right-hand sides run through the same
// elimination.
template <int M, typename LT> struct BRec {
    static constexpr size_t XZ = 0, H = 2 * (size_t)M * M;
    static constexpr size_t MULT = H + M;                     // [M][64]
    static constexpr size_t PS = MULT + (size_t)M * WAVE;     // [64] int words
    static constexpr size_t SIZE = sizeof(LT) == 4 ? PS + WAVE : H + M;
};
// multipliers and pivot words of the end-node system (behind the node records)
template <int M> struct BRoot {
    static constexpr size_t BYTES = (2 * (size_t)M * WAVE) * sizeof(double) + WAVE * sizeof(int);
};

// ------------------------------------------------------------------ elimination
// Gauss-Jordan elimination with partial pivoting on the first NC columns of a system
// whose row l is lane l's row[NW_] (rows >= NR take no part); the remaining columns are
// left in row[0 .. NW_-NC).  Steps run in groups of G with compile-time column indexes
// (the row stays in registers); between groups the row is shifted by G columns, which
// keeps the code of one group for all.  The pivot of a step is the first maximum of
// |row[j]| over rows not used yet.  Pivot rows stay in their lanes,
// unscaled; dinv receives 1 / pivot in those lanes, pstep the step (else -1).
// put(j, m) stores lane's multiplier of step j; pivs: lane j's value is the pivot lane
// of step j (j < 64).  The columns are updated 16 (FP64: 8) at a time: left to itself the
// scheduler broadcasts the whole pivot row first and spills scalar registers (one wave,
// 32 steps of 97 columns: 25.6 us; in groups of 16: 18.8 us).
template <int NC, int NR, int NW_, int G, typename T, typename Put>
__device__ __forceinline__ void gauss_jordan(T (&row)[NW_], int lane, int &pstep, T &dinv, int &pivs, Put &&put) {
    static_assert(NC % G == 0, "whole groups");
    bool done = lane >= NR;
    pstep = -1;
    dinv = (T)0;
    pivs = 0;
#pragma unroll 1
    for (int jb = 0; jb < NC; jb += G) {
#pragma unroll
        for (int jj = 0; jj < G; ++jj) {
            const T rj = row[jj];
            const int p = pivot_lane(rj, done);
            const T inv = (T)1 / rdlane(rj, p);
            const bool mine = lane == p;
            const T m = mine ? (T)0 : rj * inv;
            put(jb + jj, mine ? inv : m);
            if (mine) { done = true; pstep = jb + jj; dinv = inv; }
            if (lane == jb + jj) pivs = p;
            constexpr int CB = sizeof(T) == 4 ? 16 : 8;
#pragma unroll
            for (int c0 = jj + 1; c0 < NW_; c0 += CB) {
                T s[CB];
#pragma unroll
                for (int k = 0; k < CB; ++k)
                    if (c0 + k < NW_) s[k] = rdlane(row[c0 + k], p);
#pragma unroll
                for (int k = 0; k < CB; ++k)
                    if (c0 + k < NW_) row[c0 + k] -= m * s[k];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int c = 0; c + G < NW_; ++c) row[c] = row[c + G];
    }
}

// ------------------------------------------------------------------ instance
template <int M, int METHOD, typename LT>
__device__ inline void bload_inst(const BatchDev &B, int b, int tid) {
    auto &sh = bshared<M, METHOD, LT>();
    constexpr int NT = kBlockWaves<M, LT> * WAVE;
    const int po = B.param_off[b];
    const double *A = B.params + po + 1;
    for (int e = tid; e < M * M; e += NT) {
        const int i = e / M, q = e % M;
        sh.At[q][i] = A[e];
        sh.Al[i][q] = (LT)A[e];
    }
    if (tid == 0) sh.c = B.params[po];
    const double t0 = B.t0[b];
    if (tid < M) {
        sh.bc_end[tid] = (B.bc_t[(size_t)b * M + tid] == t0) ? 0 : 1;
        sh.bcc[tid] = B.bc_comp[(size_t)b * M + tid];
        sh.bcv[tid] = B.bc_val[(size_t)b * M + tid];
    }
    __syncthreads();
    for (int e = tid; e < M * M; e += NT) {  // A^2, summed in FP64
        const int i = e / M, q = e % M;
        double a = 0.0;
#pragma unroll 8
        for (int k = 0; k < M; ++k) a += sh.At[k][i] * sh.At[q][k];
        sh.A2[i][q] = (LT)a;
    }
    __syncthreads();
}

// maximum, any and sum over the workgroup, in every thread
template <class SH>
__device__ inline void block_reduce(SH &sh, int w, int lane, double &mx, bool &bad, double &sum) {
    const double m = wave_max(mx), s = wave_sum(sum);
    const bool any = wave_any(bad);
    if (lane == 0) { sh.red[0][w] = m; sh.red[1][w] = s; sh.red[2][w] = any ? 1.0 : 0.0; }
    __syncthreads();
    double a = sh.red[0][0], t = sh.red[1][0], f = sh.red[2][0];
#pragma unroll
    for (int k = 1; k < SH::NW; ++k) { a = fmax(a, sh.red[0][k]); t += sh.red[1][k]; f += sh.red[2][k]; }
    mx = uniform(a);
    sum = uniform(t);
    bad = uni(f != 0.0 ? 1 : 0) != 0;
    __syncthreads();
}

// ------------------------------------------------------------------ FP64 stage work
// A lane's component of the intervals its wave holds: its row of A, and the exchange
// vector of its group of M lanes.
template <int M> struct BRowA {
    double a[M];
    const double *v;  // the group's M stage arguments in LDS
    double *own;      // this lane's slot of them
};
template <int M, int METHOD, typename LT>
__device__ __forceinline__ void brow_load(BShared<M, METHOD, LT> &sh, int w, int lane, BRowA<M> &R) {
    const int i = lane % M;
#pragma unroll
    for (int q = 0; q < M; ++q) R.a[q] = sh.At[q][i];
    R.own = &sh.wv[w].vec[lane];
    R.v = &sh.wv[w].vec[lane - i];
}
// (A y)_i with y the group's vector, y this lane's component of it
template <int M>
__device__ __forceinline__ double brow_mul(const BRowA<M> &R, double y) {
    wsync();  // the vector's earlier readers are done
    *R.own = y;
    wsync();
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int q = 0; q < M; q += 2) {
        s0 += R.a[q] * R.v[q];
        s1 += R.a[q + 1] * R.v[q + 1];
    }
    return s0 + s1;
}

// K_r = f(Y_r), Y_r = (1-v_r) a + v_r b + h sum_{j<r} x_rj K_j; dd_r = c sech^2(Y_r)
template <int M, int METHOD>
__device__ __forceinline__ void bstages(const BRowA<M> &R, double c, double h, double a, double b,
                                        double (&K)[Tab<METHOD>::s], double (&dd)[Tab<METHOD>::s]) {
    using TB = Tab<METHOD>;
#pragma unroll
    for (int r = 0; r < TB::s; ++r) {
        double y = (1.0 - TB::v(r)) * a + TB::v(r) * b;
        double acc = 0.0;
        bool any = false;
#pragma unroll
        for (int j = 0; j < r; ++j)
            if (TB::x(r, j) != 0.0) { acc += TB::x(r, j) * K[j]; any = true; }
        if (any) y += h * acc;
        const double Ay = brow_mul<M>(R, y);
        const double th = tanh(y);
        K[r] = Ay + c * th;
        dd[r] = c * (1.0 - th * th);
    }
}

// Phi_k component of this lane: (b - a) - h sum b_r K_r
template <int METHOD>
__device__ __forceinline__ double bphi(const double (&K)[Tab<METHOD>::s], double h, double a, double b) {
    using TB = Tab<METHOD>;
    double acc = 0.0;
#pragma unroll
    for (int r = 0; r < TB::s; ++r) acc += TB::b(r) * K[r];
    return (b - a) - h * acc;
}

// Component of S_k da + R_k db, exactly in FP64 (the stage recursion's derivative along
// (da, db)) with the diagonals dd of the stage Jacobians.
template <int M, int METHOD>
__device__ __forceinline__ double bphi_tangent(const BRowA<M> &R, const double (&dd)[Tab<METHOD>::s], double h,
                                               double da, double db) {
    using TB = Tab<METHOD>;
    double Kd[TB::s], g = 0.0;
#pragma unroll
    for (int r = 0; r < TB::s; ++r) {
        double y = (1.0 - TB::v(r)) * da + TB::v(r) * db;
        double acc = 0.0;
        bool any = false;
#pragma unroll
        for (int j = 0; j < r; ++j)
            if (TB::x(r, j) != 0.0) { acc += TB::x(r, j) * Kd[j]; any = true; }
        if (any) y += h * acc;
        Kd[r] = brow_mul<M>(R, y) + dd[r] * y;
        g += TB::b(r) * Kd[r];
    }
    return (db - da) - h * g;
}

// Extra interpolation stages (MIRK/interpolation.jl:337-372)
template <int M, int METHOD>
__device__ __forceinline__ void binterp_stages(const BRowA<M> &R, double c, double h, double a, double b,
                                               const double (&K)[Tab<METHOD>::s],
                                               double (&KI)[Tab<METHOD>::sstar - Tab<METHOD>::s]) {
    using TB = Tab<METHOD>;
#pragma unroll
    for (int r = 0; r < TB::sstar - TB::s; ++r) {
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < TB::s; ++j)
            if (TB::xs(r, j) != 0.0) s += K[j] * TB::xs(r, j);
#pragma unroll
        for (int j = 0; j < r; ++j)
            if (TB::xs(r, TB::s + j) != 0.0) s += KI[j] * TB::xs(r, TB::s + j);
        const double y = s * h + (1.0 - TB::vs(r)) * a + TB::vs(r) * b;
        KI[r] = brow_mul<M>(R, y) + c * tanh(y);
    }
}

// What the factorisation and the refinement read of an interval's stages at the current
// state, written by the residual pass: Phi, then the S diagonals, [S + 1][M] doubles.
template <int M, int METHOD> constexpr int kBStage = (Tab<METHOD>::s + 1) * M;

// The phases below (residual, factorisation, refinement, defect, transfer) are kept out
// of line: each gets its own register allocation instead of one for their union.
//
struct BNorm {
    double mx, ss;
};
// FP64 residual of all intervals at y (+ alpha*delta if delta): max|F| and the sum of
// squares (NaN if not finite).  BC residuals are left in sh.bcres, Phi in phi_out and the stage records in st where those are set.
template <int M, int METHOD, typename LT>
__device__ __noinline__ BNorm bresidual(const double *mesh, const double *y,
                                         const double *delta, double alpha, int N, int tid, double *st,
                                         double *phi_out = nullptr) {
    auto &sh = bshared<M, METHOD, LT>();
    N = uni(N);
    mesh = uni(mesh);
    y = uni(y);
    delta = uni(delta);
    st = uni(st);
    phi_out = uni(phi_out);
    constexpr int NW = kBlockWaves<M, LT>, GP = WAVE / M, S = Tab<METHOD>::s;
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int i = lane % M, g = lane / M;
    BRowA<M> R;
    brow_load<M, METHOD, LT>(sh, w, lane, R);
    const double c = sh.c;
    double mx = 0.0, acc = 0.0;
    bool bad = false;
    for (int k0 = w * GP; k0 < N; k0 += NW * GP) {
        const bool on = k0 + g < N;
        const int k = on ? k0 + g : N - 1;
        const double h = mesh[k + 1] - mesh[k];
        const size_t e = (size_t)k * M + i;
        double a = y[e], b = y[e + M];
        if (delta) { a += alpha * delta[e]; b += alpha * delta[e + M]; }
        double K[S], dd[S];
        bstages<M, METHOD>(R, c, h, a, b, K, dd);
        const double ph = bphi<METHOD>(K, h, a, b);
        if (on) {
            if (phi_out) phi_out[e] = ph;
            if (st) {
                double *s = st + (size_t)k * kBStage<M, METHOD> + i;
                s[0] = ph;
#pragma unroll
                for (int r = 0; r < S; ++r) s[(r + 1) * M] = dd[r];
            }
            bad |= !(fabs(ph) <= 1.7976931348623157e308);
            mx = fmax(mx, fabs(ph));
            acc += ph * ph;
        }
    }
    if (tid < M) {
        const size_t e = (size_t)(sh.bc_end[tid] ? N : 0) * M + sh.bcc[tid];
        double v = y[e];
        if (delta) v += alpha * delta[e];
        const double r = v - sh.bcv[tid];
        sh.bcres[tid] = r;
        bad |= !(fabs(r) <= 1.7976931348623157e308);
        mx = fmax(mx, fabs(r));
        acc += r * r;
    }
    block_reduce(sh, w, lane, mx, bad, acc);
    return {bad ? NAN : mx, bad ? NAN : acc};
}

// r = -F(y) - J(y) d  (FP64) from the stage records of y: Phi rows at k*M, BC rows at N*M
template <int M, int METHOD, typename LT>
__device__ __noinline__ void brefine_residual(const double *mesh, const double *st,
                                              const double *d, int N, int tid, double *rout) {
    auto &sh = bshared<M, METHOD, LT>();
    N = uni(N);
    mesh = uni(mesh);
    st = uni(st);
    d = uni(d);
    rout = uni(rout);
    constexpr int NW = kBlockWaves<M, LT>, GP = WAVE / M, S = Tab<METHOD>::s;
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int i = lane % M, g = lane / M;
    BRowA<M> R;
    brow_load<M, METHOD, LT>(sh, w, lane, R);
    for (int k0 = w * GP; k0 < N; k0 += NW * GP) {
        const bool on = k0 + g < N;
        const int k = on ? k0 + g : N - 1;
        const double h = mesh[k + 1] - mesh[k];
        const size_t e = (size_t)k * M + i;
        const double *s = st + (size_t)k * kBStage<M, METHOD> + i;
        double dd[S];
#pragma unroll
        for (int r = 0; r < S; ++r) dd[r] = s[(r + 1) * M];
        const double jd = bphi_tangent<M, METHOD>(R, dd, h, d[e], d[e + M]);
        if (on) rout[e] = -s[0] - jd;
    }
    if (tid < M) rout[(size_t)N * M + tid] = -sh.bcres[tid] - d[(size_t)(sh.bc_end[tid] ? N : 0) * M + sh.bcc[tid]];
    __syncthreads();
}

// ------------------------------------------------------------------ Jacobian blocks
// The stage Jacobians are J_r = A + D_r, D_r = diag(dd_r).  Wrt y_k (side 0) and y_{k+1}
// (side 1) the first two stages give dK = J_side, and every middle stage r (2; 2 and 3
// for MIRK6) has dY_r = al_r I + h x_r J_side, so that a weighted sum of the middle
// stages' dK_r = J_r dY_r is elementwise in A and A^2:
//   U_ij = A_ij [c1 + h c2 d0_j + h sum w_r x_r dd_r,i] + h c2 (A^2)_ij
//        + delta_ij [sum w_r al_r dd_r,i + h sum w_r x_r dd_r,i d0_j],
// c1 = sum w_r al_r, c2 = sum w_r x_r, d0 the diagonal of J_side.  MIRK6's last stage has
// dY = al I + h (x J_side + U) and dK = A dY + D dY: the one matrix product.
template <int METHOD, typename LT> struct BSide {
    using TB = Tab<METHOD>;
    static constexpr int MID = TB::s > 3 ? 4 : 3;  // middle stages are 2 .. MID-1
    static constexpr double al(int r, int side) { return side ? TB::v(r) : 1.0 - TB::v(r); }
    static constexpr double x(int r, int side) { return TB::x(r, side); }
    // weights: target 0 the quadrature (b_r), target 1 the last stage's argument (x_{s-1,r})
    static constexpr double wt(int r, int target) { return target ? TB::x(TB::s - 1, r) : TB::b(r); }
    static constexpr double c1(int side, int target) {
        double s = 0.0;
        for (int r = 2; r < MID; ++r) s += wt(r, target) * al(r, side);
        return s;
    }
    static constexpr double c2(int side, int target) {
        double s = 0.0;
        for (int r = 2; r < MID; ++r) s += wt(r, target) * x(r, side);
        return s;
    }
};
// U_ij (see above); a = A_ij, a2 = (A^2)_ij, d0 = d0_j, di(r) = dd_r,i, diag: i == j
template <int METHOD, typename LT, int SIDE, int TARGET, typename DI>
__device__ __forceinline__ LT bmiddle(LT h, LT a, LT a2, LT d0, DI &&di, bool diag) {
    using BS = BSide<METHOD, LT>;
    LT e = (LT)0, f = (LT)0;
#pragma unroll
    for (int r = 2; r < BS::MID; ++r) {
        e += (LT)(BS::wt(r, TARGET) * BS::x(r, SIDE)) * di(r);
        f += (LT)(BS::wt(r, TARGET) * BS::al(r, SIDE)) * di(r);
    }
    const LT hc2 = h * (LT)BS::c2(SIDE, TARGET);
    LT u = a * ((LT)BS::c1(SIDE, TARGET) + hc2 * d0 + h * e) + hc2 * a2;
    if (diag) u += f + h * e * d0;
    return u;
}

// Block row of one interval into the wave's blk: [S | R] (the right-hand side column is
// the caller's).  dd: the diagonals in LDS.
template <int M, int METHOD, typename LT>
__device__ __forceinline__ void btangent(BShared<M, METHOD, LT> &sh, int w, int lane, LT h) {
    using TB = Tab<METHOD>;
    using SHT = BShared<M, METHOD, LT>;
    constexpr int SW = SHT::SW;
    constexpr int LS = TB::s - 1;  // the last stage
    LT *blk = sh.wv[w].blk;
    const LT(*dd)[M] = sh.wv[w].dd;
    if constexpr (sizeof(LT) == 4 && M >= 16) {
        // Lane l holds, for each 16 x 16 tile, rows 4 (l / 16) .. +3 of column l % 16: the
        // layout of the v_mfma_f32_16x16x4_f32 result (operands: A[i][k] in lane i + 16 k,
        // B[k][j] in lane j + 16 k).
        typedef float f4 __attribute__((ext_vector_type(4)));
        constexpr int RT = M / 16, CT = 2 * M / 16, KS = M / 4;
        const int l16 = lane & 15, l4 = lane >> 4;
        float G[RT][CT][4], Y[RT][CT][4];
        auto entry = [&](auto side, int rt, int ct, int v) {
            constexpr int SIDE = decltype(side)::value;
            const int i = 16 * rt + 4 * l4 + v, j = (16 * ct + l16) % M;
            const bool diag = (rt == (ct * 16 % M) / 16) && i == j;
            const float a = sh.Al[i][j], a2 = sh.A2[i][j], d0 = dd[SIDE][j];
            auto di = [&](int r) { return dd[r][i]; };
            float js = a;
            if (diag) js += d0;
            G[rt][ct][v] = (float)TB::b(SIDE) * js + bmiddle<METHOD, float, SIDE, 0>(h, a, a2, d0, di, diag);
            if constexpr (TB::s > 3) {
                float dy = h * ((float)TB::x(LS, SIDE) * js + bmiddle<METHOD, float, SIDE, 1>(h, a, a2, d0, di, diag));
                if (diag) dy += (float)BSide<METHOD, float>::al(LS, SIDE);
                Y[rt][ct][v] = dy;
            }
        };
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (ct < CT / 2) entry(std::integral_constant<int, 0>{}, rt, ct, v);
                    else entry(std::integral_constant<int, 1>{}, rt, ct, v);
                }
        if constexpr (TB::s > 3) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int v = 0; v < 4; ++v) blk[(16 * rt + 4 * l4 + v) * SW + 16 * ct + l16] = Y[rt][ct][v];
            wsync();
            f4 acc[RT][CT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float aop[RT], bop[CT];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) aop[rt] = sh.Al[16 * rt + l16][4 * ks + l4];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) bop[ct] = blk[(4 * ks + l4) * SW + 16 * ct + l16];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
                        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(aop[rt], bop[ct], acc[rt][ct], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int i = 16 * rt + 4 * l4 + v;
                        G[rt][ct][v] += (float)TB::b(LS) * (acc[rt][ct][v] + dd[LS][i] * Y[rt][ct][v]);
                    }
            wsync();  // dY is read by every lane before the block row overwrites it
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const bool left = ct < CT / 2;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * rt + 4 * l4 + v, j = (16 * ct + l16) % M;
                    blk[i * SW + 16 * ct + l16] = ((i == j) ? (left ? -1.f : 1.f) : 0.f) - h * G[rt][ct][v];
                }
            }
    } else {
        // one column per lane, the rows split over the 64 / 2M lane groups
        constexpr int NG = WAVE / (2 * M), RP = M / NG;
        const int col = lane % (2 * M), r0 = (lane / (2 * M)) * RP;
        auto column = [&](auto side) {
            constexpr int SIDE = decltype(side)::value;
            const int j = col % M;
            const LT d0 = dd[SIDE][j];
            LT dy[TB::s > 3 ? M : 1];
            if constexpr (TB::s > 3) {
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    const LT a = sh.Al[q][j], a2 = sh.A2[q][j];
                    auto di = [&](int r) { return dd[r][q]; };
                    const LT js = a + (q == j ? d0 : (LT)0);
                    dy[q] = h * ((LT)TB::x(LS, SIDE) * js + bmiddle<METHOD, LT, SIDE, 1>(h, a, a2, d0, di, q == j)) +
                            (q == j ? (LT)BSide<METHOD, LT>::al(LS, SIDE) : (LT)0);
                }
            }
#pragma unroll
            for (int ii = 0; ii < RP; ++ii) {
                const int i = r0 + ii;
                const LT a = sh.Al[i][j], a2 = sh.A2[i][j];
                auto di = [&](int r) { return dd[r][i]; };
                const LT js = a + (i == j ? d0 : (LT)0);
                LT G = (LT)TB::b(SIDE) * js + bmiddle<METHOD, LT, SIDE, 0>(h, a, a2, d0, di, i == j);
                if constexpr (TB::s > 3) {
                    LT t = (LT)0, dyi = (LT)0;
#pragma unroll
                    for (int q = 0; q < M; ++q) {
                        t += sh.Al[i][q] * dy[q];
                        dyi = (q == i) ? dy[q] : dyi;
                    }
                    G += (LT)TB::b(LS) * (t + dd[LS][i] * dyi);
                }
                blk[i * SW + col] = (i == j ? (SIDE ? (LT)1 : (LT)-1) : (LT)0) - h * G;
            }
        };
        if (col < M) column(std::integral_constant<int, 0>{});
        else column(std::integral_constant<int, 1>{});
    }
}

// ------------------------------------------------------------------ factorisation
// Eliminates J(y) d = -F(y) down to its end nodes (stage records st and BC residuals of
// y in place), keeping what back-substitution and further right-hand sides need, and
// leaves (d_0, d_N) in sh.xr.  rec: node records, index = node; root: BRoot bytes;
// keep: store the multipliers.
template <int M, int METHOD, typename LT>
__device__ __noinline__ void bfactor(const double *mesh, const double *st, int N, int tid,
                                     LT *rec, double *root, bool keep) {
    auto &sh = bshared<M, METHOD, LT>();
    N = uni(N);
    mesh = uni(mesh);
    st = uni(st);
    rec = uni(rec);
    root = uni(root);
    keep = uni(keep ? 1 : 0) != 0;
    using SHT = BShared<M, METHOD, LT>;
    constexpr int NW = kBlockWaves<M, LT>, SW = SHT::SW, S = Tab<METHOD>::s;
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    int P, start, len;
    bchunk<NW>(N, w, P, start, len);
    const int L = (N + P - 1) / P;
    int D = 0;
    while ((1 << D) < P) ++D;
    LT row[3 * M + 1];  // after a step: [E | F | g] of the relation in row[0 .. 2M]
#pragma unroll
    for (int c = 0; c < 3 * M + 1; ++c) row[c] = (LT)0;
    int src = -1;       // block row this lane takes next (-1: the lane holds a relation row)
    for (int t = 0; t < L + D; ++t) {
        bool act;
        int node;
        const LT *nb = sh.wv[w].blk;
        if (t < L) {
            act = t < len;
            node = start + t;
            if (act) {
                // block row of interval start + t
                const double *s = st + (size_t)node * kBStage<M, METHOD>;
                const LT h = (LT)(mesh[node + 1] - mesh[node]);
                wsync();
                for (int e = lane; e < S * M; e += WAVE) sh.wv[w].dd[e / M][e % M] = (LT)s[M + e];
                if (lane < M) sh.wv[w].blk[lane * SW + 2 * M] = (LT)(-s[lane]);
                wsync();
                btangent<M, METHOD, LT>(sh, w, lane, h);
                wsync();
                if (t == 0) {
                    // the chunk's first interval is its first relation
                    if (lane < M) {
#pragma unroll
                        for (int c = 0; c < 2 * M + 1; ++c) row[c] = nb[lane * SW + c];
                    } else if (lane < 2 * M) {
                        src = lane - M;
                    }
                    act = false;
                }
            }
        } else {
            // merge with the relation of the chunks to the right
            const int span = 1 << (t - L);
            __syncthreads();
            if (w < P && (w & (2 * span - 1)) == span) {
                const bool kp = src < 0 && lane < 2 * M;
                const int rank = __popcll(__ballot(kp) & ((1ull << lane) - 1ull));
                if (kp && rank < M) {
#pragma unroll
                    for (int c = 0; c < 2 * M + 1; ++c) sh.wv[w].blk[rank * SW + c] = row[c];
                }
            }
            __syncthreads();
            act = (w & (2 * span - 1)) == 0 && w + span < P;
            int pp, pl;
            bchunk<NW>(N, w + span, pp, node, pl);
            nb = sh.wv[act ? w + span : w].blk;
        }
        if (!act) continue;
        // stacked rows: relation [F | E | 0 | g], new block row [S | 0 | R | rhs]
        if (src >= 0) {
            const LT *r = nb + src * SW;
#pragma unroll
            for (int c = 0; c < M; ++c) { row[c] = r[c]; row[M + c] = (LT)0; row[2 * M + c] = r[M + c]; }
            row[3 * M] = r[2 * M];
        } else {
            row[3 * M] = row[2 * M];
#pragma unroll
            for (int c = 0; c < M; ++c) {
                const LT e = row[c];
                row[c] = row[M + c];
                row[M + c] = e;
                row[2 * M + c] = (LT)0;
            }
        }
        LT *R = rec + (size_t)node * BRec<M, LT>::SIZE;
        int pstep, pivs;
        LT dinv;
        auto put = [&](int j, LT m) {
            if constexpr (sizeof(LT) == 4) {
                if (keep) R[BRec<M, LT>::MULT + (size_t)j * WAVE + lane] = m;
            }
        };
        gauss_jordan<M, 2 * M, 3 * M + 1, kBlockGroup<M, LT>>(row, lane, pstep, dinv, pivs, put);
        if (pstep >= 0) {
#pragma unroll
            for (int c = 0; c < 2 * M; ++c) R[BRec<M, LT>::XZ + (size_t)c * M + pstep] = row[c] * dinv;
            R[BRec<M, LT>::H + pstep] = row[2 * M] * dinv;
        }
        if constexpr (sizeof(LT) == 4) {
            if (keep) reinterpret_cast<int *>(R + BRec<M, LT>::PS)[lane] = (pstep & 0xff) | (pivs << 8);
        }
        src = pstep;
    }
    // ---- end nodes: BC rows and the relation E d_0 + F d_N = g (FP64)
    if (w == 0) {
        wsync();
        const bool kp = src < 0 && lane < 2 * M;
        const int rank = __popcll(__ballot(kp) & ((1ull << lane) - 1ull));
        LT *blk = sh.wv[0].blk;
        if (kp && rank < M) {
#pragma unroll
            for (int c = 0; c < 2 * M + 1; ++c) blk[rank * SW + c] = row[c];
        }
        wsync();
        double rr[2 * M + 1];
        if (lane < M) {
            const bool end = sh.bc_end[lane] != 0;
            const int comp = sh.bcc[lane];
#pragma unroll
            for (int c = 0; c < M; ++c) {
                rr[c] = (!end && c == comp) ? 1.0 : 0.0;
                rr[M + c] = (end && c == comp) ? 1.0 : 0.0;
            }
            rr[2 * M] = -sh.bcres[lane];
        } else {
            const int i = lane < 2 * M ? lane - M : 0;
#pragma unroll
            for (int c = 0; c < 2 * M + 1; ++c) rr[c] = (double)blk[i * SW + c];
        }
        int pstep, pivs;
        double dinv;
        auto put = [&](int j, double m) {
            if constexpr (sizeof(LT) == 4) {
                if (keep) root[(size_t)j * WAVE + lane] = m;
            }
        };
        gauss_jordan<2 * M, 2 * M, 2 * M + 1, 8>(rr, lane, pstep, dinv, pivs, put);
        if (pstep >= 0) sh.xr[pstep] = rr[0] * dinv;
        if constexpr (sizeof(LT) == 4) {
            if (keep)
                reinterpret_cast<int *>(root + 2 * (size_t)M * WAVE)[lane] = (pstep & 0xff) | (pivs << 8);
        }
    }
    __syncthreads();
}

// The elimination of bfactor on another right-hand side r (Phi rows at k*M, BC rows at
// N*M), through the stored multipliers: writes the records' H and leaves (d_0, d_N) in sh.xr.
template <int M, int METHOD>
__device__ __noinline__ void bpush(int N, int tid, float *rec, const double *root,
                                   const double *rin) {
    auto &sh = bshared<M, METHOD, float>();
    N = uni(N);
    rec = uni(rec);
    root = uni(root);
    rin = uni(rin);
    using BR = BRec<M, float>;
    constexpr int NW = kBlockWaves<M, float>;
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    int P, start, len;
    bchunk<NW>(N, w, P, start, len);
    const int L = (N + P - 1) / P;
    int D = 0;
    while ((1 << D) < P) ++D;
    float q = 0.f;
    int src = -1;
    if (len > 0) {
        if (lane < M) q = (float)rin[(size_t)start * M + lane];
        else if (lane < 2 * M) src = lane - M;
    }
    for (int t = 1; t < L + D; ++t) {
        bool act;
        int node = start + t;
        if (t < L) {
            act = t < len;
            if (act && src >= 0) q = (float)rin[(size_t)node * M + src];
        } else {
            const int span = 1 << (t - L);
            __syncthreads();
            if (w < P && (w & (2 * span - 1)) == span) {
                const bool kp = src < 0 && lane < 2 * M;
                const int rank = __popcll(__ballot(kp) & ((1ull << lane) - 1ull));
                if (kp && rank < M) sh.wv[w].blk[rank] = q;
            }
            __syncthreads();
            act = (w & (2 * span - 1)) == 0 && w + span < P;
            int pp, pl;
            bchunk<NW>(N, w + span, pp, node, pl);
            if (act && src >= 0) q = sh.wv[w + span].blk[src];
        }
        if (!act) continue;
        float *R = rec + (size_t)node * BR::SIZE;
        float m[M];
#pragma unroll
        for (int j = 0; j < M; ++j) m[j] = R[BR::MULT + (size_t)j * WAVE + lane];
        const int ps = reinterpret_cast<const int *>(R + BR::PS)[lane];
        const int pstep = (int)(signed char)(ps & 0xff), pv = (ps >> 8) & 0xff;
        float dinv = 0.f;
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const float qp = rdlane(q, __builtin_amdgcn_readlane(pv, j));
            const bool mine = pstep == j;
            dinv = mine ? m[j] : dinv;
            q -= mine ? 0.f : m[j] * qp;
        }
        if (pstep >= 0) R[BR::H + pstep] = q * dinv;
        src = pstep;
    }
    if (w == 0) {
        wsync();
        const bool kp = src < 0 && lane < 2 * M;
        const int rank = __popcll(__ballot(kp) & ((1ull << lane) - 1ull));
        if (kp && rank < M) sh.wv[0].blk[rank] = q;
        wsync();
        double x = 0.0, dinv = 0.0;
        if (lane < M) x = rin[(size_t)N * M + lane];
        else if (lane < 2 * M) x = (double)sh.wv[0].blk[lane - M];
        const int ps = reinterpret_cast<const int *>(root + 2 * (size_t)M * WAVE)[lane];
        const int pstep = (int)(signed char)(ps & 0xff), pv = (ps >> 8) & 0xff;
#pragma unroll 8
        for (int j = 0; j < 2 * M; ++j) {
            const double m = root[(size_t)j * WAVE + lane];
            const double xp = rdlane(x, __builtin_amdgcn_readlane(pv, j));
            const bool mine = pstep == j;
            dinv = mine ? m : dinv;
            x -= mine ? 0.0 : m * xp;
        }
        if (pstep >= 0) sh.xr[pstep] = x * dinv;
    }
    __syncthreads();
}

// Back-substitution from (d_0, d_N) in sh.xr through the merges and the chunks:
// dout = d, or dout += d with add (point-major, M (N+1)).  False when d is not finite.
template <int M, int METHOD, typename LT>
__device__ __noinline__ bool bback(int N, int tid, const LT *rec, double *dout, bool add) {
    auto &sh = bshared<M, METHOD, LT>();
    N = uni(N);
    rec = uni(rec);
    dout = uni(dout);
    add = uni(add ? 1 : 0) != 0;
    using BR = BRec<M, LT>;
    constexpr int NW = kBlockWaves<M, LT>;
    constexpr int G = WAVE / M, CP = 2 * M / G;  // column groups; columns per lane
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int j = lane % M, g = lane / M;
    int P, start, len;
    bchunk<NW>(N, w, P, start, len);
    int D = 0;
    while ((1 << D) < P) ++D;
    double *vv = sh.wv[w].vv;
    // column c = i G + g of [X | Z] in lane group g: record element i * 64 + lane
    auto load = [&](int node, LT (&x)[CP], LT &hh) {
        const LT *R = rec + (size_t)node * BR::SIZE;
#pragma unroll
        for (int i = 0; i < CP; ++i) x[i] = R[i * WAVE + lane];
        hh = R[BR::H + j];
    };
    auto apply = [&](const LT (&x)[CP], LT hh) {  // component j of H - [X | Z] vv, in every group
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int i = 0; i < CP; i += 2) {
            s0 += (double)x[i] * vv[i * G + g];
            s1 += (double)x[i + 1] * vv[(i + 1) * G + g];
        }
        double s = s0 + s1;
#pragma unroll
        for (int o = M; o < WAVE; o <<= 1) s += __shfl_xor(s, o);
        return (double)hh - s;
    };
    if (tid < M) { sh.lo[0][tid] = sh.xr[tid]; sh.hi[0][tid] = sh.xr[M + tid]; }
    __syncthreads();
    for (int d = D - 1; d >= 0; --d) {
        const int span = 1 << d;
        if ((w & (2 * span - 1)) == 0 && w + span < P) {
            int pp, node, pl;
            bchunk<NW>(N, w + span, pp, node, pl);
            LT x[CP], hh;
            load(node, x, hh);
            if (lane < M) { vv[lane] = sh.lo[w][lane]; vv[M + lane] = sh.hi[w][lane]; }
            wsync();
            const double mid = apply(x, hh);
            if (lane < M) {
                sh.hi[w + span][lane] = sh.hi[w][lane];
                sh.lo[w + span][lane] = mid;
                sh.hi[w][lane] = mid;
            }
            wsync();
        }
        __syncthreads();
    }
    bool bad = false;
    auto out = [&](int node, double v) {
        if (lane < M) {
            const size_t e = (size_t)node * M + j;
            dout[e] = add ? dout[e] + v : v;
            bad |= !(fabs(v) <= 1.7976931348623157e308);
        }
    };
    if (len > 0) {
        LT x[CP], hh;
        if (len > 1) load(start + len - 1, x, hh);
        double d = sh.hi[w][j];
        if (w == P - 1) out(N, d);
        if (lane < M) vv[lane] = sh.lo[w][lane];
        for (int k = start + len - 1; k > start; --k) {
            if (lane < M) vv[M + lane] = d;
            wsync();
            LT xn[CP], hn = hh;
            if (k - 1 > start) load(k - 1, xn, hn);
            d = apply(x, hh);
            wsync();
            out(k, d);
#pragma unroll
            for (int i = 0; i < CP; ++i) x[i] = xn[i];
            hh = hn;
        }
        out(start, sh.lo[w][j]);
    }
    double mx = 0.0, sum = 0.0;
    block_reduce(sh, w, lane, mx, bad, sum);
    return !bad;
}

// d = -J(y)^-1 F(y): factorisation, and with FP32 factors `refine` steps of FP64 iterative
// refinement (r = -F - J d, J e = r through the factors, d += e).
template <int M, int METHOD, typename LT>
__device__ inline bool bcorrection(const double *mesh, const double *st, int N, int tid,
                                   LT *rec, double *root, int refine, double *rbuf, double *delta) {
    bfactor<M, METHOD, LT>(mesh, st, N, tid, rec, root, refine > 0);
    bool ok = uni(bback<M, METHOD, LT>(N, tid, rec, delta, false) ? 1 : 0) != 0;
    if constexpr (sizeof(LT) == 4) {
        for (int r = 0; ok && r < refine; ++r) {
            brefine_residual<M, METHOD, LT>(mesh, st, delta, N, tid, rbuf);
            bpush<M, METHOD>(N, tid, rec, root, rbuf);
            ok = uni(bback<M, METHOD, LT>(N, tid, rec, delta, true) ? 1 : 0) != 0;
        }
    }
    return ok;
}

// ------------------------------------------------------------------ Newton (block)
// Work areas of a slot behind its records: correction, refinement residual, stage records.
template <int M, int METHOD, typename LT> struct BWork {
    LT *rec;
    double *root, *delta, *rbuf, *st;
    int *idx;
};

// NewtonRaphson, then NewtonRaphson + BackTracking from the same start (bits 0
// and 1 of B.stages; Core/default_internal_solve.jl:37-43).  The TrustRegion
// stage (bit 2) is run by the wave kernels only.
template <int M, int METHOD, typename LT>
__device__ NewtonOut bnewton(const BatchDev &B, const double *mesh, double *y,
                             double *ybak, const BWork<M, METHOD, LT> &W, int N, int tid) {
    constexpr int NT = kBlockWaves<M, LT> * WAVE;
    NewtonOut out{BVP_RET_MAXITERS, 0, -1, 0, NAN};
    const int refine = (sizeof(LT) == 4 && B.refine_iters > 0) ? B.refine_iters : 0;
    const int stages = B.stages & 3;
    const bool restart = stages == 3;
    if (restart) {
        for (int e = tid; e < (N + 1) * M; e += NT) ybak[e] = y[e];
        __syncthreads();
    }
    bool first = true;
    for (int stage = 0; stage < 2; ++stage) {
        if (!((stages >> stage) & 1)) continue;
        if (!first) {
            for (int e = tid; e < (N + 1) * M; e += NT) y[e] = ybak[e];
            __syncthreads();
        }
        first = false;
        out.stage = stage;
        int ret = BVP_RET_MAXITERS;
        for (int it = 0;; ++it) {
            const BNorm F = bresidual<M, METHOD, LT>(mesh, y, nullptr, 0.0, N, tid, W.st);
            const double fn = uniform(F.mx), ss = uniform(F.ss);
            out.fn = fn;
            if (!(fn <= 1.7976931348623157e308)) { ret = BVP_RET_UNSTABLE; break; }
            if (fn <= B.newton_tol) { ret = BVP_RET_SUCCESS; break; }
            if (it >= B.max_newton) { ret = BVP_RET_MAXITERS; break; }
            if (!bcorrection<M, METHOD, LT>(mesh, W.st, N, tid, W.rec, W.root, refine, W.rbuf, W.delta)) {
                ret = BVP_RET_FAILURE;
                break;
            }
            out.iters++;
            double alpha = 1.0;
            if (stage == 1) {
                // BackTracking on |F(y + a d)|^2 / 2 with phi'(0) = -|F|^2 (Newton direction)
                auto phi = [&](double a) {
                    return 0.5 * uniform(bresidual<M, METHOD, LT>(mesh, y, W.delta, a, N, tid, nullptr).ss);
                };
                if (!backtracking(phi, 0.5 * ss, -ss, alpha)) { ret = BVP_RET_FAILURE; break; }
            }
            for (int e = tid; e < (N + 1) * M; e += NT) y[e] += alpha * W.delta[e];
            __syncthreads();
        }
        out.ret = ret;
        if (ret == BVP_RET_SUCCESS) break;
    }
    return out;
}

// maximum over the M lanes of a group
template <int M> __device__ __forceinline__ double group_max(double v) {
#pragma unroll
    for (int o = M / 2; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

// ------------------------------------------------------------------ defect (block)
// the defect norm (NaN if not finite), and the maximum and sum of shat
struct BDefect {
    double norm, r1, r2;
};
template <int M, int METHOD, typename LT>
__device__ __noinline__ BDefect bdefect(const double *mesh, const double *y, int N, int tid,
                                        double abstol, double *shat, double *errors) {
    auto &sh = bshared<M, METHOD, LT>();
    N = uni(N);
    mesh = uni(mesh);
    y = uni(y);
    shat = uni(shat);
    errors = uni(errors);
    using TB = Tab<METHOD>;
    constexpr int NW = kBlockWaves<M, LT>, GP = WAVE / M, S = TB::s, NS = TB::sstar - TB::s;
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int i = lane % M, g = lane / M;
    BRowA<M> R;
    brow_load<M, METHOD, LT>(sh, w, lane, R);
    const double c = sh.c;
    double w1[TB::sstar], w1p[TB::sstar], w2[TB::sstar], w2p[TB::sstar];
    interp_weights<METHOD>(TB::tau(), w1, w1p);
    interp_weights<METHOD>(1.0 - TB::tau(), w2, w2p);
    const double ex = 1.0 / (TB::order + 1);
    double dmax = 0.0, smax = 0.0, ssum = 0.0;
    bool bad = false;
    for (int k0 = w * GP; k0 < N; k0 += NW * GP) {
        const bool on = k0 + g < N;
        const int k = on ? k0 + g : N - 1;
        const double h = mesh[k + 1] - mesh[k];
        const size_t e = (size_t)k * M + i;
        const double a = y[e], b = y[e + M];
        double K[S], dd[S], KI[NS];
        bstages<M, METHOD>(R, c, h, a, b, K, dd);
        binterp_stages<M, METHOD>(R, c, h, a, b, K, KI);
        double d[2], er[2];
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const double *wt = side ? w2 : w1, *wp = side ? w2p : w1p;
            double z = 0.0, zp = 0.0;
#pragma unroll
            for (int r = 0; r < S; ++r) { z += K[r] * wt[r]; zp += K[r] * wp[r]; }
#pragma unroll
            for (int r = 0; r < NS; ++r) { z += KI[r] * wt[S + r]; zp += KI[r] * wp[S + r]; }
            z = z * h + a;
            const double f = brow_mul<M>(R, z) + c * tanh(z);
            d[side] = (zp - f) / (fabs(f) + 1.0);
            er[side] = group_max<M>(fabs(d[side]));
        }
        const bool first = er[0] > er[1];
        const double dv = first ? d[0] : d[1], ei = first ? er[0] : er[1];
        if (on) {
            if (errors) errors[e] = dv;
            bad |= !(fabs(dv) <= 1.7976931348623157e308);
            dmax = fmax(dmax, ei);
            const double shv = pow(ei / abstol, ex);
            if (i == 0) {
                if (shat) shat[k] = shv;
                ssum += shv;
            }
            smax = fmax(smax, shv);
        }
    }
    bool none = false;
    double zero = 0.0;
    block_reduce(sh, w, lane, dmax, bad, ssum);
    block_reduce(sh, w, lane, smax, none, zero);
    return {bad ? NAN : dmax, smax, ssum};
}

// Transfer of the old continuous extension to the new nodes (MIRK/mirk.jl:366-370).  The
// increments z - y_ii of all new nodes are formed in parallel (into inc, with their
// intervals in idx); REFERENCE mode then reads the base value y0.u[ii] from the array
// being written where ii < j, as the reference's in-place update does, one component per
// lane of the first wave in order.
template <int M, int METHOD, typename LT>
__device__ __noinline__ void btransfer(const double *mesh, const double *y, int N,
                                       const double *nm, double *ny, int Nn, int mode, int tid, double *inc,
                                       int *idx) {
    auto &sh = bshared<M, METHOD, LT>();
    N = uni(N);
    Nn = uni(Nn);
    mode = uni(mode);
    mesh = uni(mesh);
    y = uni(y);
    nm = uni(nm);
    ny = uni(ny);
    inc = uni(inc);
    idx = uni(idx);
    using TB = Tab<METHOD>;
    constexpr int NW = kBlockWaves<M, LT>, GP = WAVE / M, S = TB::s, NS = TB::sstar - TB::s;
    const int lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int i = lane % M, g = lane / M;
    BRowA<M> R;
    brow_load<M, METHOD, LT>(sh, w, lane, R);
    const double c = sh.c;
    for (int j0 = w * GP; j0 <= Nn; j0 += NW * GP) {
        const bool on = j0 + g <= Nn;
        const int j = on ? j0 + g : Nn;
        const double m = nm[j];
        const int ii = interval_of(mesh, N, m);
        const double ti = mesh[ii], dt = mesh[ii + 1] - ti, tau = (m - ti) / dt;
        const double a = y[(size_t)ii * M + i], b = y[(size_t)(ii + 1) * M + i];
        double K[S], dd[S], KI[NS], wt[TB::sstar];
        bstages<M, METHOD>(R, c, dt, a, b, K, dd);
        binterp_stages<M, METHOD>(R, c, dt, a, b, K, KI);
        interp_weights<METHOD>(tau, wt, nullptr);
        double z = 0.0;
#pragma unroll
        for (int r = 0; r < S; ++r) z += K[r] * wt[r];
#pragma unroll
        for (int r = 0; r < NS; ++r) z += KI[r] * wt[S + r];
        if (on) {
            const bool chained = mode == BVP_TRANSFER_REFERENCE && ii < j;
            if (chained) inc[(size_t)j * M + i] = z * dt;
            else ny[(size_t)j * M + i] = z * dt + a;
            if (i == 0) idx[j] = chained ? ii : -1;
        }
    }
    __syncthreads();
    if (mode == BVP_TRANSFER_REFERENCE && tid < M)
        for (int j = 0; j <= Nn; ++j) {
            const int ii = idx[j];
            if (ii >= 0) ny[(size_t)j * M + tid] = inc[(size_t)j * M + tid] + ny[(size_t)ii * M + tid];
        }
    __syncthreads();
}

// Work areas of the workgroup's slot (BatchDev::scratch, BatchDev::aux).
template <int M, int METHOD, typename LT>
__device__ inline BWork<M, METHOD, LT> bwork_of(const BatchDev &B) {
    BWork<M, METHOD, LT> W;
    char *slot = (char *)B.scratch + (size_t)blockIdx.x * B.scratch_per_slot;
    W.root = as_global((double *)slot);
    W.rec = as_global((LT *)(slot + ((BRoot<M>::BYTES + 255) & ~(size_t)255)));
    double *aux = as_global(B.aux + (size_t)blockIdx.x * B.aux_per_slot);
    const size_t v = (size_t)B.cap * M;
    W.delta = aux;
    W.rbuf = aux + v;
    W.st = aux + 2 * v;
    W.idx = (int *)(W.st + (size_t)B.cap * kBStage<M, METHOD>);
    return W;
}

// ------------------------------------------------------------------ full solve (block)
template <int M, int METHOD, typename LT>
__device__ void bsolve_instance(const BatchDev &B, int b, int tid,
                                const BWork<M, METHOD, LT> &W) {
    constexpr int NT = kBlockWaves<M, LT> * WAVE;
    auto &sh = bshared<M, METHOD, LT>();
    bload_inst<M, METHOD, LT>(B, b, tid);
    double *mesh_b[2], *y_b[2];
    {
        const size_t cap = (size_t)B.cap;
        mesh_b[0] = B.mesh + (size_t)b * 2 * cap;
        mesh_b[1] = mesh_b[0] + cap;
        y_b[0] = B.y + (size_t)b * 2 * cap * M;
        y_b[1] = y_b[0] + cap * M;
    }
    int cur = 0;
    int N = uni(B.N0[b]);
    {
        const long long off = B.init_off[b];
        for (int k = tid; k <= N; k += NT) mesh_b[0][k] = B.init_mesh[off + k];
        for (long long e = tid; e < (long long)(N + 1) * M; e += NT) y_b[0][e] = B.init_y[off * M + e];
        __syncthreads();
    }
    double *shat = B.shat + (size_t)b * B.cap;
    int info = BVP_RET_SUCCESS, nl_ret = BVP_RET_SUCCESS;
    int outer = 0, iters = 0, fb = 0;
    double last_defect = NAN;
    long long cnt_it = 0, cnt_def = 0, cnt_tr = 0, cnt_chk = 0;
    for (;;) {
        ++outer;
        double *mesh = mesh_b[cur], *y = y_b[cur];
        double *mesh_o = mesh_b[1 - cur], *y_o = y_b[1 - cur];
        NewtonOut nl;
        if (N > B.rec_cap) {
            nl.ret = BVP_RET_FAILURE;
            nl.iters = 0;
            nl.stage = -1;
            fb |= 8;  // records of this instance do not fit the slot's factor storage
        } else {
            nl = bnewton<M, METHOD, LT>(B, mesh, y, y_o, W, N, tid);
        }
        iters += nl.iters;
        cnt_it += (long long)N * nl.iters;
        cnt_chk += N;
        if (nl.stage == 1) fb |= 1;
        nl_ret = nl.ret;
        double error_norm = 2.0 * B.abstol;
        if (!B.adaptive || (fb & 8)) { info = nl.ret; break; }
        info = nl.ret;
        double r1 = 0.0, r2 = 0.0;
        if (info == BVP_RET_SUCCESS) {
            const BDefect df = bdefect<M, METHOD, LT>(mesh, y, N, tid, B.abstol, shat, nullptr);
            error_norm = uniform(df.norm);
            r1 = uniform(df.r1);
            r2 = uniform(df.r2);
            cnt_def += N;
            last_defect = error_norm;
            info = (error_norm > B.defect_threshold || isnan(error_norm)) ? BVP_RET_FAILURE : BVP_RET_SUCCESS;
        }
        __syncthreads();
        if (info == BVP_RET_SUCCESS) {
            if (error_norm > B.abstol) {
                if (tid < WAVE) {
                    const int n = mesh_select<WaveSync>(mesh, N, shat, r1, r2, B.max_sub, mesh_o, tid);
                    if (tid == 0) sh.flag = n;
                }
                __syncthreads();
                const int Nn = uni(sh.flag);
                __syncthreads();
                if (Nn < 0) {
                    info = BVP_RET_FAILURE;
                } else {
                    btransfer<M, METHOD, LT>(mesh, y, N, mesh_o, y_o, Nn, B.transfer_mode, tid, W.rbuf, W.idx);
                    cnt_tr += N + Nn;
                    N = Nn;
                    cur = 1 - cur;
                }
            }
        } else {
            if (2 * N > B.max_sub) {
                info = BVP_RET_FAILURE;
            } else {
                if (tid < WAVE) half_mesh_into(mesh, N, mesh_o, tid);
                for (long long e = tid; e < (long long)(2 * N + 1) * M; e += NT) y_o[e] = 0.0;
                __syncthreads();
                N = 2 * N;
                cur = 1 - cur;
                info = BVP_RET_SUCCESS;
            }
        }
        if (!(info == BVP_RET_SUCCESS && error_norm > B.abstol)) break;
        if (outer >= MAX_OUTER) { info = BVP_RET_FAILURE; break; }
    }
    const double rn = bresidual<M, METHOD, LT>(mesh_b[cur], y_b[cur], nullptr, 0.0, N, tid, W.st).mx;
    // distance of the returned state from the discrete solution on its mesh: one more
    // Newton correction (factors in the plan's precision, refined as in the solve)
    double err = NAN;
    if (B.report_err && N <= B.rec_cap) {
        const int refine = (sizeof(LT) == 4 && B.refine_iters > 0) ? B.refine_iters : 0;
        if (bcorrection<M, METHOD, LT>(mesh_b[cur], W.st, N, tid, W.rec, W.root, refine, W.rbuf, W.delta)) {
            const double *y = y_b[cur];
            double e_ = 0.0, none = 0.0;
            bool no = false;
            for (int e = tid; e < (N + 1) * M; e += NT) e_ = fmax(e_, fabs(W.delta[e]) / fmax(1.0, fabs(y[e])));
            block_reduce(sh, tid / WAVE, tid % WAVE, e_, no, none);
            err = e_;
        }
        __syncthreads();
    }
    if (tid == 0) {
        B.err[b] = err;
        B.retcode[b] = (nl_ret == BVP_RET_SUCCESS) ? info : nl_ret;
        B.N_final[b] = N;
        B.newton_iters[b] = iters;
        B.outer_iters[b] = outer;
        B.fallback[b] = fb;
        B.cur_buf[b] = cur;
        B.defect_norm[b] = last_defect;
        B.resid_norm[b] = rn;
        B.cnt[(size_t)b * 4 + 0] = cnt_it;
        B.cnt[(size_t)b * 4 + 1] = cnt_def;
        B.cnt[(size_t)b * 4 + 2] = cnt_tr;
        B.cnt[(size_t)b * 4 + 3] = cnt_chk;
    }
    __syncthreads();
}

template <class SH> __device__ inline int bnext_item(unsigned *counter, SH &sh, int tid) {
    if (tid == 0) sh.item = (int)atomicAdd(counter, 1u);
    __syncthreads();
    const int item = uni(sh.item);
    __syncthreads();
    return item;
}

template <int M, int METHOD, typename LT>
__global__ __launch_bounds__((kBlockWaves<M, LT> * WAVE)) void k_bsolve(BatchDev B) {
    auto &sh = bshared<M, METHOD, LT>();
    const int tid = threadIdx.x;
    const BWork<M, METHOD, LT> W = bwork_of<M, METHOD, LT>(B);
    for (;;) {
        const int item = bnext_item(B.counter, sh, tid);
        if (item >= B.n) break;
        bsolve_instance<M, METHOD, LT>(B, uni(B.order[item]), tid, W);
    }
}

// Component operations on a given state (parity entry points).
template <int M, int METHOD, typename LT>
__global__ __launch_bounds__((kBlockWaves<M, LT> * WAVE)) void k_bcomponent(BatchDev B, int op) {
    auto &sh = bshared<M, METHOD, LT>();
    constexpr int NT = kBlockWaves<M, LT> * WAVE;
    const int tid = threadIdx.x, lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const BWork<M, METHOD, LT> W = bwork_of<M, METHOD, LT>(B);
    for (;;) {
        const int b = bnext_item(B.counter, sh, tid);
        if (b >= B.n) break;
        bload_inst<M, METHOD, LT>(B, b, tid);
        const int N = uni(B.N0[b]);
        const long long off = B.init_off[b];
        double *mesh = B.mesh + (size_t)b * 2 * B.cap;
        double *y = B.y + (size_t)b * 2 * B.cap * M;
        for (int k = tid; k <= N; k += NT) mesh[k] = B.init_mesh[off + k];
        for (long long e = tid; e < (long long)(N + 1) * M; e += NT) y[e] = B.init_y[off * M + e];
        __syncthreads();
        if (op == OP_RESIDUAL) {
            // two-point layout [bca; Phi; bcb] (rows at t0 first, rows at t1 last)
            double *out = B.out0 + off * M;
            int La = 0;
            for (int k = 0; k < M; ++k) La += sh.bc_end[k] ? 0 : 1;
            bresidual<M, METHOD, LT>(mesh, y, nullptr, 0.0, N, tid, nullptr, out + La);
            if (tid == 0) {
                int ia = 0, ib = 0;
                for (int k = 0; k < M; ++k) {
                    if (sh.bc_end[k]) out[La + (size_t)N * M + (ib++)] = sh.bcres[k];
                    else out[ia++] = sh.bcres[k];
                }
            }
        } else if (op == OP_JACOBIAN) {
            const long long ioff = off - b;
            bresidual<M, METHOD, LT>(mesh, y, nullptr, 0.0, N, tid, W.st);
            for (int k = w; k < N; k += kBlockWaves<M, LT>) {
                const double *s = W.st + (size_t)k * kBStage<M, METHOD>;
                for (int e = lane; e < Tab<METHOD>::s * M; e += WAVE) sh.wv[w].dd[e / M][e % M] = (LT)s[M + e];
                wsync();
                btangent<M, METHOD, LT>(sh, w, lane, (LT)(mesh[k + 1] - mesh[k]));
                wsync();
                double *So = B.out0 + (ioff + k) * M * M, *Ro = B.out1 + (ioff + k) * M * M;
                for (int e = lane; e < M * M; e += WAVE) {
                    const int i = e / M, c = e % M;
                    So[e] = (double)sh.wv[w].blk[i * (2 * M + 1) + c];
                    Ro[e] = (double)sh.wv[w].blk[i * (2 * M + 1) + M + c];
                }
                wsync();
            }
            if (tid < M) B.iout[(size_t)b * M + tid] = sh.bc_end[tid] ? N : 0;
        } else if (op == OP_NEWTON_STEP) {
            if constexpr (kBlockFactors<M, LT>) {
                bresidual<M, METHOD, LT>(mesh, y, nullptr, 0.0, N, tid, W.st);
                const int refine = (sizeof(LT) == 4 && B.refine_iters > 0) ? B.refine_iters : 0;
                const bool ok = (N <= B.rec_cap) &&
                                bcorrection<M, METHOD, LT>(mesh, W.st, N, tid, W.rec, W.root, refine, W.rbuf, W.delta);
                double *d = B.out0 + off * M;
                for (long long e = tid; e < (long long)(N + 1) * M; e += NT) d[e] = W.delta[e];
                if (tid == 0) B.iout[b] = ok ? 0 : 1;
            }
        } else if (op == OP_DEFECT) {
            const long long ioff = off - b;
            const BDefect df = bdefect<M, METHOD, LT>(mesh, y, N, tid, B.abstol, nullptr, B.out0 + ioff * M);
            if (tid == 0) B.out1[b] = df.norm;
        } else if (op == OP_MESH_SELECT) {
            double *shat = B.shat + (size_t)b * B.cap;
            const BDefect df = bdefect<M, METHOD, LT>(mesh, y, N, tid, B.abstol, shat, nullptr);
            __syncthreads();
            double *nm = mesh + B.cap, *ny = y + (size_t)B.cap * M;
            if (tid < WAVE) {
                const int n = mesh_select<WaveSync>(mesh, N, shat, df.r1, df.r2, B.max_sub, nm, tid);
                if (tid == 0) sh.flag = n;
            }
            __syncthreads();
            const int Nn = uni(sh.flag);
            __syncthreads();
            if (Nn < 0) {
                if (tid == 0) { B.iout[(size_t)b * 2] = N; B.iout[(size_t)b * 2 + 1] = BVP_RET_FAILURE; }
            } else {
                btransfer<M, METHOD, LT>(mesh, y, N, nm, ny, Nn, B.transfer_mode, tid, W.rbuf, W.idx);
                double *om = B.out0 + (size_t)b * B.cap, *oy = B.out1 + (size_t)b * B.cap * M;
                for (int k = tid; k <= Nn; k += NT) om[k] = nm[k];
                for (long long e = tid; e < (long long)(Nn + 1) * M; e += NT) oy[e] = ny[e];
                if (tid == 0) { B.iout[(size_t)b * 2] = Nn; B.iout[(size_t)b * 2 + 1] = BVP_RET_SUCCESS; }
            }
        }
        __syncthreads();
    }
}

template <int M, int METHOD, typename LT>
hipError_t launch_bsolve_t(const BatchDev &B, int blocks, hipStream_t s) {
    if constexpr (!kBlockFactors<M, LT>) return hipErrorInvalidValue;
    else k_bsolve<M, METHOD, LT><<<blocks, kBlockWaves<M, LT> * WAVE, 0, s>>>(B);
    return hipGetLastError();
}
template <int M, int METHOD, typename LT>
hipError_t launch_bcomponent_t(const BatchDev &B, int op, int blocks, hipStream_t s) {
    k_bcomponent<M, METHOD, LT><<<blocks, kBlockWaves<M, LT> * WAVE, 0, s>>>(B, op);
    return hipGetLastError();
}
template <int M, int METHOD, typename LT>
int boccupancy_t() {
    if constexpr (kBlockFactors<M, LT>) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_bsolve<M, METHOD, LT>, kBlockWaves<M, LT> * WAVE, 0) ==
            hipSuccess)
            return nb;
    }
    return 1;
}

}  // namespace bvpdev
