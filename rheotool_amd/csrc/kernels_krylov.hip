// kernels_krylov.hip -- lockstep multi-component PBiCGStab for the theta solve (gfx950).
//
// The reference solves each valid symmTensor component separately with
// OpenFOAM's PBiCGStab (the segregated loop restated in
// sparseMatrixSolvers/segregated/eigenSolver/eigenSolver.C:422-562, residual
// normalisation sparseSolver.C:129-180).  The components share the matrix, so
// here one pass over the matrix serves every component still iterating:
// each kernel walks the sliced-ELL rows once and updates all active
// components (stored interleaved, [N][6]) with per-component convergence
// masks.  Every scalar of the recurrence (rho, alpha, omega, beta, residuals,
// flags) stays on the device: each row kernel writes per-workgroup partial
// sums and a one-workgroup finalize kernel on the same stream reduces them in
// a fixed order and updates the component records, so no host round trip is
// needed inside an iteration.
//
// Preconditioning is right-Jacobi with the column-scaled matrix
// Ahat = A D^-1 stored explicitly: A M^-1 p = p + offdiag(Ahat) p.
//
// Precision: the vector type T is double (FP64 drop-in) or float (inner
// solve of the FP64-refined "mixed" solve).  x (theta), b, the matrix used
// for the true residual and the grid-level reductions are FP64; per-thread
// partial sums use T.
#include <unistd.h>

#include <cstring>

#include "rt_device.h"

namespace rt {

template <class T>
struct KryArgs {
    int32_t N;
    const int64_t* ellOff;
    const int32_t* ellWidth;
    const int32_t* ellCol;
    const double* aval;  // FP64 matrix (true residual)
    const uint32_t* slotMask;  // [nSlices] live column-order slots, NULL: all live
    const double* diag;
    const T* ahat;       // A D^-1 off-diagonal values
    const double* rD;    // 1 / diag
    const double* b;     // [N][6]
    double* x;           // [N][6]
    T *r, *r0, *p, *v, *t;  // [N][6]
    T* e;                // [N][6] mixed: the inner solve's correction to x (NULL in FP64)
    // preconditioner M (right preconditioning of PBiCGStab, M^-1 of PBiCG):
    // rM = M^-1 as a diagonal (1/diag for Jacobi, NULL for none: 1), and
    // dg = diag(A M^-1) (NULL: 1, Jacobi) -- D itself for none
    const double* rM;
    const double* dg;
    // PBiCG: wT = s, the off-diagonals of A and A^T in T, FP64 A^T for rT
    T* s;
    const T* aA;
    const T* aT;
    const double* atval;
    double* partials;
    CompState* cs;
    CompState* host;     // page-locked copy of the records the host reads, or NULL
    int32_t valid[6];
    KryCtl ctl;
    int32_t G;           // workgroups of the row kernels (partials rows)
    int32_t nRed;        // colour-blocked rows: the first colour's count (0: not coloured)
    int32_t rowBegin;    // k_residual: rows [rowBegin, N) (the red-black sweep's second colour)
};

// ---- true residual r = b - A x (FP64): MODE 0 initial, MODE 1 refinement ----
// A refinement sweep (MODE 1) waits until no inner solve is running; the
// gate is read on the device so a sweep may be queued ahead of knowing.
// Matrix streams of the FP32 solve's passes are read once per pass: load
// them non-temporal, which leaves more of L2 to the gathered neighbour rows
// (measured 1.5% faster on those passes at 256^3; the FP64 passes keep
// ordinary loads).
template <class T, class U>
__device__ __forceinline__ U ld_stream(const U* p) {
    if constexpr (std::is_same<T, float>::value) return __builtin_nontemporal_load(p);
    else return *p;
}

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v) {
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v));
    const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
    return __hiloint2double(hi, lo);
}

// The live entries of row r in column order, W at a time: f(col, av) gets W
// columns and values (value 0: none).  A wavefront's rows are one slice, so
// which slots are live is the same for its lanes.  The W loads of an entry's
// column and value, and f's W gathers, are in flight together: taken one entry
// after another, each waits for two memory round trips.
template <int W, class T, class V, class F>
__device__ __forceinline__ void for_entries(const KryArgs<T>& a, int32_t r, const V* vals, F&& f) {
    const int s = uni(r >> 6);
    const int64_t base = a.ellOff[s] + (r & 63);
    const int width = a.ellWidth[s];
    uint32_t m = a.slotMask ? a.slotMask[s] : 0xffffffffu;
    if (width < 32) m &= (1u << width) - 1u;
    m = (uint32_t)uni((int)m);
    while (m) {
        int32_t col[W];
        V av[W];
#pragma unroll
        for (int j = 0; j < W; ++j) {
            col[j] = r;
            av[j] = (V)0;
            if (m) {
                const int64_t e = base + (int64_t)SLICE * __builtin_ctz(m);
                m &= m - 1;
                col[j] = ld_stream<T>(a.ellCol + e);
                av[j] = ld_stream<T>(vals + e);
            }
        }
        f(col, av);
    }
    for (int k = 32; k < width; k += W) {
        int32_t col[W];
        V av[W];
#pragma unroll
        for (int j = 0; j < W; ++j) {
            col[j] = r;
            av[j] = (V)0;
            if (k + j < width) {
                const int64_t e = base + (int64_t)SLICE * (k + j);
                col[j] = ld_stream<T>(a.ellCol + e);
                av[j] = ld_stream<T>(vals + e);
            }
        }
        f(col, av);
    }
}

// acc += av * src[col] (NEG: acc -= ...) over W entries; entries with no
// coefficient (the downwind side of a face) are not gathered
template <bool NEG, int W, class U, class V>
__device__ __forceinline__ void gather(const U* src, const int32_t (&col)[W], const V (&av)[W], U (&acc)[6]) {
    U g[W][6];
#pragma unroll
    for (int j = 0; j < W; ++j)
        if (av[j] != (V)0) ld6(src + (int64_t)NCMP * col[j], g[j]);
#pragma unroll
    for (int j = 0; j < W; ++j)
        if (av[j] != (V)0) {
#pragma unroll
            for (int c = 0; c < 6; ++c) acc[c] = NEG ? acc[c] - av[j] * g[j][c] : acc[c] + av[j] * g[j][c];
        }
}
// the same of s = r - alpha v
template <int W, class T>
__device__ __forceinline__ void gather_s(const T* rv, const T* vv, const T (&alpha)[6], const int32_t (&col)[W],
                                         const T (&av)[W], T (&acc)[6]) {
    T g[W][6], h[W][6];
#pragma unroll
    for (int j = 0; j < W; ++j)
        if (av[j] != (T)0) {
            ld6(rv + (int64_t)NCMP * col[j], g[j]);
            ld6(vv + (int64_t)NCMP * col[j], h[j]);
        }
#pragma unroll
    for (int j = 0; j < W; ++j)
        if (av[j] != (T)0) {
#pragma unroll
            for (int c = 0; c < 6; ++c) acc[c] += av[j] * (g[j][c] - alpha[c] * h[j][c]);
        }
}
// entries in flight: four rows of six words (two vectors of FP64: two)
template <class T, int NV = 1>
constexpr int ENT = sizeof(T) * NV <= 8 ? 4 : 2;

template <class T>
__device__ __forceinline__ bool inner_running(const KryArgs<T>& a) {
    bool run = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) run |= a.valid[c] > 0 && a.cs[c].active;
    return run;
}

// The active components of a PBiCGStab round.  They are always in the same
// inner iteration: a solve's components start together (the initial residual,
// or a sweep that waits until no inner solve is running) and only leave.
// In the first iteration p = r = r0, and r0 keeps that residual, so the passes
// read r0 for all three: the sweep writes one vector instead of two, the copy
// p = r is not made, and the second iteration takes its old p from r0.
struct Round {
    bool on[6];
    bool any = false;
    int inner = 0;  // the inner iteration of the active components
};
template <class T>
__device__ __forceinline__ Round round_of(const KryArgs<T>& a) {
    Round q;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        q.on[c] = uni(a.cs[c].active);
        const int i = uni(a.cs[c].innerIter);
        if (q.on[c]) q.inner = i;
        q.any |= q.on[c];
    }
    return q;
}

template <class T, int MODE>
__device__ __forceinline__ void k_residual_body(const KryArgs<T>& a, const Blk& k_) {
    constexpr int NQ = 18;
    bool on[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.valid[c] > 0 && (MODE == 0 || a.cs[c].needRefine);
        any |= on[c];
    }
    if (!any || (MODE == 1 && inner_running(a))) return;
    double q[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) q[i] = 0;
    double xbar[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) xbar[c] = MODE == 0 ? a.cs[c].xbar : 0.0;
    // rows [rowBegin, N): all rows, or the second colour of a red-black sweep
    // (the first colour's residual is zero once it has been eliminated)
    const int32_t rowB = a.rowBegin & ~(SLICE - 1);  // wavefronts on whole slices
    const int64_t nRows = (int64_t)a.N - rowB;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = a.rowBegin > 0 ? tile_of_g(it, nRows, 0, k_.G, k_.b) : tile_of_g(it, a.N, a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int64_t t0 = tl * BLK;
        const int32_t r = (int32_t)(rowB + t0 + k_.tid);
        if (r < a.rowBegin || r >= a.N) continue;
        const double d = a.diag[r];
        double y[6], xv[6];
        ld6(a.x + (int64_t)NCMP * r, xv);
#pragma unroll
        for (int c = 0; c < 6; ++c) y[c] = d * xv[c];
        double sumA = d;
        for_entries<ENT<double>>(a, r, a.aval, [&](const auto& col, const auto& av) {
            if (MODE == 0) {
#pragma unroll
                for (int j = 0; j < ENT<double>; ++j) sumA += av[j];
            }
            gather<false>(a.x, col, av, y);
        });
        double bb[6];
        ld6(a.b + (int64_t)NCMP * r, bb);
        // rows are written whole (three 2-wide stores): the entries of
        // components that are off belong to finished or frozen solves, which
        // no later kernel reads
        T rt[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const double res = bb[c] - y[c];
            rt[c] = (T)res;
            if (!on[c]) continue;
            q[c] += fabs(res);
            q[6 + c] += (double)rt[c] * (double)rt[c];
            if (MODE == 0) {
                const double pA = sumA * xbar[c];
                q[12 + c] += fabs(y[c] - pA) + fabs(bb[c] - pA);
            } else {
                // (M^-1 r, r): the rho of a PBiCG restart with rT = r
                const double rm = a.rM ? a.rM[r] : 1.0;
                q[12 + c] += (rm * (double)rt[c]) * (double)rt[c];
            }
        }
        if (MODE == 1 || !a.ctl.bicg) st6(a.r0 + (int64_t)NCMP * r, rt);
        if (a.ctl.bicg) st6(a.r + (int64_t)NCMP * r, rt);
    }
    write_partials<NQ>(q, a.partials, k_);
}

template <class T, int MODE>
__global__ void __launch_bounds__(BLK) k_residual(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_residual_body<T, MODE>(a, blk_of_launch(red));
}

// The finalize bodies: every thread of the workgroup sums the partials, then
// lane c of the first wavefront updates component c's record.  (Thread 0
// updating the six records one after another, with a memory round trip for
// each, was most of these kernels' time.)
template <class T, int MODE, int NT = FBLK>
__device__ __forceinline__ void k_fin_residual_body(const KryArgs<T>& a, double* lds) {
    constexpr int NQ = 18;
    bool on = false, any = false;
    const int c = threadIdx.x;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const bool o = a.valid[i] > 0 && (MODE == 0 || a.cs[i].needRefine);
        any |= o;
        if (i == c) on = o;
    }
    if (!any || (MODE == 1 && inner_running(a))) return;
    Comp cs;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<NQ, NT>(a.partials, a.G, lds, sums);
    if (!on) return;
    if (MODE == 0) {
        finish_initial(cs, a.ctl, sums[c], sums[6 + c], sums[12 + c]);
    } else {
        cs.needRefine = 0;
        cs.foldE = 0;
        cs.nRefine += 1;
        cs.finalRes = sums[c] / cs.normFactor;
        if (conv_outer(cs, a.ctl, cs.finalRes) && cs.iter >= a.ctl.minIter) {
            cs.converged = 1;
            cs.active = 0;
        } else if (cs.nRefine >= a.ctl.maxRefine || cs.iter >= a.ctl.maxIter) {
            cs.active = 0;
        } else {
            start_inner(cs, a.ctl, a.ctl.bicg ? sums[12 + c] : sums[6 + c]);
        }
    }
    cs.store(a.cs[c]);
    if (a.host) cs.store(a.host[c]);
}

template <class T, int MODE>
__global__ void __launch_bounds__(FBLK) k_fin_residual(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_residual_body<T, MODE>(a, lds);
}

// ---- p = r + beta (p - omega v), from the second inner iteration on ---------
template <class T>
__device__ __forceinline__ void k_kry_p_body(const KryArgs<T>& a, const Blk& k_) {
    const Round q = round_of(a);
    if (!q.any || q.inner == 0) return;
    T beta[6], omega[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        beta[c] = (T)uni(a.cs[c].beta);
        omega[c] = (T)uni(a.cs[c].omega);
    }
    const T* pOld = q.inner == 1 ? a.r0 : a.p;
    const int64_t N = a.N;
    for (int64_t i = (int64_t)k_.b * BLK + k_.tid; k_.b < k_.G && i < N; i += (int64_t)k_.G * BLK) {
        T rr[6], pp[6], vv[6];
        ld6(a.r + NCMP * i, rr);
        ld6(pOld + NCMP * i, pp);
        ld6(a.v + NCMP * i, vv);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (q.on[c]) pp[c] = rr[c] + beta[c] * (pp[c] - omega[c] * vv[c]);
        st6(a.p + NCMP * i, pp);
    }
}

template <class T>
__global__ void __launch_bounds__(BLK) k_kry_p(KryArgs<T> a) {
    k_kry_p_body<T>(a, blk_of_launch(nullptr));
}

// ---- v = A M^-1 p = p + Ahat p ;  sigma = (r0, v) -------------------------
template <class T>
__device__ __forceinline__ void k_kry_v_body(const KryArgs<T>& a, const Blk& k_) {
    const Round rd = round_of(a);
    if (!rd.any) return;
    const T* pv = rd.inner == 0 ? a.r0 : a.p;
    T q[6] = {0, 0, 0, 0, 0, 0};
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, a.N, a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int64_t t0 = tl * BLK;
        const int32_t r = (int32_t)(t0 + k_.tid);
        if (r >= a.N) continue;
        T acc[6], rr0[6];
        ld6(pv + (int64_t)NCMP * r, acc);
        ld6(a.r0 + (int64_t)NCMP * r, rr0);
        if (a.dg) {
            const T dgr = (T)a.dg[r];
#pragma unroll
            for (int c = 0; c < 6; ++c) acc[c] = dgr * acc[c];
        }
        for_entries<ENT<T>>(a, r, a.ahat, [&](const auto& col, const auto& av) { gather<false>(pv, col, av, acc); });
        st6(a.v + (int64_t)NCMP * r, acc);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (rd.on[c]) q[c] += rr0[c] * acc[c];
    }
    double qd[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) qd[c] = q[c];
    write_partials<6>(qd, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_kry_v(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_kry_v_body<T>(a, blk_of_launch(red));
}

template <class T, int NT = FBLK>
__device__ __forceinline__ void k_fin_v_body(const KryArgs<T>& a, double* lds) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; ++i) any |= a.cs[i].active != 0;
    if (!any) return;
    const int c = threadIdx.x;
    Comp cs;
    cs.active = 0;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<6, NT>(a.partials, a.G, lds, sums);
    if (!cs.active) return;
    cs.alpha = cs.rho / sums[c];
    cs.store(a.cs[c]);
}

template <class T>
__global__ void __launch_bounds__(FBLK) k_fin_v(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_v_body<T>(a, lds);
}

// ---- s = r - alpha v ; t = A M^-1 s ; |s|, (t,s), (t,t) --------------------
template <class T>
__device__ __forceinline__ void k_kry_t_body(const KryArgs<T>& a, const Blk& k_) {
    const Round rd = round_of(a);
    if (!rd.any) return;
    const T* rv = rd.inner == 0 ? a.r0 : a.r;
    T alpha[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) alpha[c] = (T)uni(a.cs[c].alpha);
    T q[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) q[i] = 0;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, a.N, a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int64_t t0 = tl * BLK;
        const int32_t r = (int32_t)(t0 + k_.tid);
        if (r >= a.N) continue;
        T sv[6], acc[6], rr[6], vv[6];
        ld6(rv + (int64_t)NCMP * r, rr);
        ld6(a.v + (int64_t)NCMP * r, vv);
        const T dgr = a.dg ? (T)a.dg[r] : (T)1;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            sv[c] = rr[c] - alpha[c] * vv[c];
            acc[c] = a.dg ? dgr * sv[c] : sv[c];
        }
        for_entries<ENT<T, 2>>(a, r, a.ahat,
                               [&](const auto& col, const auto& av) { gather_s(rv, a.v, alpha, col, av, acc); });
        st6(a.t + (int64_t)NCMP * r, acc);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (!rd.on[c]) continue;
            q[c] += fabs(sv[c]);
            q[6 + c] += acc[c] * sv[c];
            q[12 + c] += acc[c] * acc[c];
        }
    }
    double qd[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) qd[i] = q[i];
    write_partials<18>(qd, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_kry_t(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_kry_t_body<T>(a, blk_of_launch(red));
}

template <class T, int NT = FBLK>
__device__ __forceinline__ void k_fin_t_body(const KryArgs<T>& a, double* lds) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; ++i) any |= a.cs[i].active != 0;
    if (!any) return;
    const int c = threadIdx.x;
    Comp cs;
    cs.active = 0;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<18, NT>(a.partials, a.G, lds, sums);
    if (!cs.active) return;
    const double res = sums[c] / cs.normFactor;
    if (!a.ctl.mixed) cs.finalRes = res;
    if (conv_inner(cs, a.ctl, res)) {
        cs.exitAtS = 1;
    } else {
        cs.omega = sums[6 + c] / sums[12 + c];
    }
    cs.store(a.cs[c]);
}

template <class T>
__global__ void __launch_bounds__(FBLK) k_fin_t(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_t_body<T>(a, lds);
}

// ---- x += alpha M^-1 p + omega M^-1 s ; r = s - omega t ; |r|, (r0, r) ------
template <class T>
__device__ __forceinline__ void k_kry_xr_body(const KryArgs<T>& a, const Blk& k_) {
    // FP64: x += alpha M^-1 p + omega M^-1 s in place.  Mixed: the inner
    // solve accumulates the same update into its FP32 correction e (from 0 at
    // the solve's first iteration) and k_fold adds e to x in FP64 before the
    // refinement sweep, so the pass moves 4-byte instead of 8-byte x words.
    constexpr bool MIX = std::is_same<T, float>::value;
    const Round rd_ = round_of(a);
    if (!rd_.any) return;
    const bool start = rd_.inner == 0;
    const T* pv = start ? a.r0 : a.p;
    const T* rv = start ? a.r0 : a.r;
    bool ex[6];
    double alpha[6], omega[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        ex[c] = uni(a.cs[c].exitAtS);
        alpha[c] = uni(a.cs[c].alpha);
        omega[c] = uni(a.cs[c].omega);
    }
    T q[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) q[i] = 0;
    // red-black: the second colour's rows, as the v and t passes take them
    const int32_t first = a.ctl.rb ? a.nRed : 0, row0 = first & ~(SLICE - 1);
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, (int64_t)a.N - row0, a.ctl.rb ? 0 : a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int64_t t0 = tl * BLK;
        const int32_t r = (int32_t)(row0 + t0 + k_.tid);
        if (r < first || r >= a.N) continue;
        const double rd = a.rM ? a.rM[r] : 1.0;
        const int64_t j = (int64_t)NCMP * r;
        double xv[6];
        T ev[6];
        T pp[6], rr[6], vv[6], tt[6], rr0[6];
        if constexpr (MIX) {
            if (start) {
#pragma unroll
                for (int c = 0; c < 6; ++c) xv[c] = 0.0;
            } else {
                ld6(a.e + j, ev);
#pragma unroll
                for (int c = 0; c < 6; ++c) xv[c] = (double)ev[c];
            }
        } else {
            ld6(a.x + j, xv);
        }
        ld6(pv + j, pp);
        ld6(rv + j, rr);
        ld6(a.v + j, vv);
        ld6(a.t + j, tt);
        ld6(a.r0 + j, rr0);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (!rd_.on[c]) continue;
            const double y = rd * (double)pp[c];
            if (ex[c]) {
                xv[c] += alpha[c] * y;
                continue;
            }
            const T sv = rr[c] - (T)alpha[c] * vv[c];
            const double z = rd * (double)sv;
            xv[c] += alpha[c] * y + omega[c] * z;
            const T rn = sv - (T)omega[c] * tt[c];
            rr[c] = rn;
            q[c] += fabs(rn);
            q[6 + c] += rr0[c] * rn;
        }
        if constexpr (MIX) {
#pragma unroll
            for (int c = 0; c < 6; ++c) ev[c] = (T)xv[c];
            st6(a.e + j, ev);
        } else {
            st6(a.x + j, xv);
        }
        st6(a.r + j, rr);
    }
    double qd[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) qd[i] = q[i];
    write_partials<12>(qd, a.partials, k_);
}

// (FP32: held to the 102 VGPRs of five workgroups a CU, the grid of the solve's
// passes is the least over them)
template <class T>
__global__ void __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 5 : 4, 8)))
k_kry_xr(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_kry_xr_body<T>(a, blk_of_launch(red));
}

// ---- mixed: x += e (FP64) for the components about to be refined ----------
// Gated like the refinement sweep it precedes (no inner solve running, the
// component waiting for refinement); the sweep's finalize then clears the
// wait, so a correction is added once.
template <class T>
__device__ __forceinline__ void k_fold_body(const KryArgs<T>& a, const Blk& k_) {
    bool on[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.valid[c] > 0 && a.cs[c].needRefine && a.cs[c].foldE;
        any |= on[c];
    }
    if (!any || inner_running(a)) return;
    for (int64_t i = (int64_t)k_.b * BLK + k_.tid; k_.b < k_.G && i < a.N; i += (int64_t)k_.G * BLK) {
        double xv[6];
        T ev[6];
        ld6(a.x + NCMP * i, xv);
        ld6(a.e + NCMP * i, ev);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (on[c]) xv[c] += (double)ev[c];
        st6(a.x + NCMP * i, xv);
    }
}

template <class T>
__global__ void __launch_bounds__(BLK) k_fold(KryArgs<T> a) {
    k_fold_body<T>(a, blk_of_launch(nullptr));
}

template <class T, int NT = FBLK>
__device__ __forceinline__ void k_fin_xr_body(const KryArgs<T>& a, double* lds) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; ++i) any |= a.cs[i].active != 0;
    if (!any) return;
    const int c = threadIdx.x;
    Comp cs;
    cs.active = 0;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<12, NT>(a.partials, a.G, lds, sums);
    if (!cs.active) return;
    cs.iter += 1;
    cs.innerIter += 1;
    bool stop, breakdown = false;
    if (cs.exitAtS) {
        cs.exitAtS = 0;
        stop = true;
    } else {
        const double res = sums[c] / cs.normFactor;
        if (!a.ctl.mixed) cs.finalRes = res;
        const bool conv = conv_inner(cs, a.ctl, res);
        bool cont = (!conv && cs.iter < a.ctl.maxIter) ||
                    (!a.ctl.mixed && cs.iter < a.ctl.minIter);
        if (a.ctl.mixed && cs.innerIter >= a.ctl.maxInner) cont = false;
        stop = !cont;
        if (cont) {
            cs.rhoOld = cs.rho;
            cs.rho = sums[6 + c];
            if (fabs(cs.rho) < 1e-300 || fabs(cs.omega) < 1e-300) {
                stop = true;
                breakdown = true;
            } else {
                cs.beta = (cs.rho / cs.rhoOld) * (cs.alpha / cs.omega);
            }
        }
    }
    if (stop) {
        cs.active = 0;
        // A breakdown ((r0, r) or omega vanishing before convergence)
        // restarts from the true residual with r0 = r, through the same
        // pass as a refinement sweep (at most maxRefine times); [OF9]
        // PBiCGStab stops unconverged there instead (checkSingularity), but its
        // DILU preconditioner meets breakdowns in other places than
        // right Jacobi does, so stopping would leave results that differ
        // from it by more than the tolerance.
        if (a.ctl.mixed || breakdown || a.ctl.rb) {
            // mixed: fold the inner solve's correction, then refine;
            // red-black: the closing sweep eliminates the first colour
            cs.needRefine = 1;
            cs.foldE = a.ctl.mixed && cs.innerIter > 0 ? 1 : 0;
        } else {
            cs.converged = conv_outer(cs, a.ctl, cs.finalRes);
        }
    }
    cs.store(a.cs[c]);
    if (a.host) cs.store(a.host[c]);
}

template <class T>
__global__ void __launch_bounds__(FBLK) k_fin_xr(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_xr_body<T>(a, lds);
}

// ================================== red-black ILU0 (multicolour ILU0, two colours)
// On a two-colourable cell graph stored colour by colour (rows [0, nRed) =: R,
// [nRed, N) =: B; A_RR = D_R and A_BB = D_B are diagonal), ILU(0) in this
// ordering factors A exactly except for the pivots of B, which become
// Ds = diag(S) of the Schur complement S = D_B - A_BR D_R^-1 A_RB (D_B itself
// when every product A_ij A_ji vanishes, as for the upwind theta matrix).
// ILU(0)-preconditioned Krylov is the same method as Krylov on S with the
// Jacobi preconditioner Ds and R eliminated exactly,
// x_R = D_R^-1 (b_R - A_RB x_B): the residual of the whole system is then zero
// on R and S's residual on B.  So the lockstep PBiCGStab runs on B's rows with
// right preconditioning M = Ds, each product S M^-1 y in two passes:
//   R rows gather  w   = D_R^-1 A_RB Ds^-1 y   (ahat = A_jk / (D_j Ds_k) there)
//   B rows gather  S M^-1 y = (D_B Ds^-1) y - A_BR w   (ahat = A_ij there).
// r, r0, p, v, t live on B's rows; w uses R's rows of v, w' R's rows of t.
// Every solve opens with a sweep (x_R from x_B, then the true residual on B)
// and closes with one, so x_R is always the exact elimination of x_B.

// R rows: w = D_R^-1 A_RB Ds^-1 y, y = p (SRC 0) or s = r - alpha v (SRC 1)
template <class T, int SRC>
__device__ __forceinline__ void k_rb_w_body(const KryArgs<T>& a, const Blk& k_) {
    T* w = SRC == 0 ? a.v : a.t;
    const Round rd = round_of(a);
    if (!rd.any) return;
    const T* pv = rd.inner == 0 ? a.r0 : a.p;
    const T* rv = rd.inner == 0 ? a.r0 : a.r;
    T alpha[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) alpha[c] = (T)uni(a.cs[c].alpha);
    const int64_t n = a.nRed;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, n, 0, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(tl * BLK + k_.tid);
        if (r >= n) continue;
        T acc[6] = {0, 0, 0, 0, 0, 0};
        if constexpr (SRC == 0)
            for_entries<ENT<T>>(a, r, a.ahat, [&](const auto& col, const auto& av) { gather<false>(pv, col, av, acc); });
        else
            for_entries<ENT<T, 2>>(a, r, a.ahat,
                                   [&](const auto& col, const auto& av) { gather_s(rv, a.v, alpha, col, av, acc); });
        st6(w + (int64_t)NCMP * r, acc);
    }
}

template <class T, int SRC>
__global__ void __launch_bounds__(BLK) k_rb_w(KryArgs<T> a) {
    k_rb_w_body<T, SRC>(a, blk_of_launch(nullptr));
}

// B rows: v = S M^-1 p = (D_B Ds^-1) p - A_BR w ;  sigma = (r0, v)
template <class T>
__device__ __forceinline__ void k_rb_v_body(const KryArgs<T>& a, const Blk& k_) {
    const T* w = a.v;
    const Round rd = round_of(a);
    if (!rd.any) return;
    const T* pv = rd.inner == 0 ? a.r0 : a.p;
    T q[6] = {0, 0, 0, 0, 0, 0};
    const int32_t r0b = a.nRed & ~(SLICE - 1);  // wavefronts on whole slices
    const int64_t n = (int64_t)a.N - r0b;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, n, 0, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(r0b + tl * BLK + k_.tid);
        if (r < a.nRed || r >= a.N) continue;
        T acc[6], rr0[6];
        ld6(pv + (int64_t)NCMP * r, acc);
        ld6(a.r0 + (int64_t)NCMP * r, rr0);
        if (a.dg) {
            const T dgr = (T)a.dg[r];
#pragma unroll
            for (int c = 0; c < 6; ++c) acc[c] = dgr * acc[c];
        }
        for_entries<ENT<T>>(a, r, a.ahat, [&](const auto& col, const auto& av) { gather<true>(w, col, av, acc); });
        st6(a.v + (int64_t)NCMP * r, acc);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (rd.on[c]) q[c] += rr0[c] * acc[c];
    }
    double qd[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) qd[c] = q[c];
    write_partials<6>(qd, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_rb_v(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_rb_v_body<T>(a, blk_of_launch(red));
}

// B rows: s = r - alpha v ; t = S M^-1 s = (D_B Ds^-1) s - A_BR w' ;
// |s|, (t, s), (t, t)
template <class T>
__device__ __forceinline__ void k_rb_t_body(const KryArgs<T>& a, const Blk& k_) {
    const T* w = a.t;
    const Round rd = round_of(a);
    if (!rd.any) return;
    const T* rv = rd.inner == 0 ? a.r0 : a.r;
    T alpha[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) alpha[c] = (T)uni(a.cs[c].alpha);
    T q[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) q[i] = 0;
    const int32_t r0b = a.nRed & ~(SLICE - 1);  // wavefronts on whole slices
    const int64_t n = (int64_t)a.N - r0b;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, n, 0, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(r0b + tl * BLK + k_.tid);
        if (r < a.nRed || r >= a.N) continue;
        T sv[6], acc[6], rr[6], vv[6];
        ld6(rv + (int64_t)NCMP * r, rr);
        ld6(a.v + (int64_t)NCMP * r, vv);
        const T dgr = a.dg ? (T)a.dg[r] : (T)1;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            sv[c] = rr[c] - alpha[c] * vv[c];
            acc[c] = a.dg ? dgr * sv[c] : sv[c];
        }
        for_entries<ENT<T>>(a, r, a.ahat, [&](const auto& col, const auto& av) { gather<true>(w, col, av, acc); });
        st6(a.t + (int64_t)NCMP * r, acc);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (!rd.on[c]) continue;
            q[c] += fabs(sv[c]);
            q[6 + c] += acc[c] * sv[c];
            q[12 + c] += acc[c] * acc[c];
        }
    }
    double qd[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) qd[i] = q[i];
    write_partials<18>(qd, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_rb_t(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_rb_t_body<T>(a, blk_of_launch(red));
}

// The sweep's elimination of R (FP64): x_R = D_R^-1 (b_R - A_RB x_B) for the
// components about to be refined; gated like the refinement sweep it opens.
template <class T>
__device__ __forceinline__ void k_rb_backsub_body(const KryArgs<T>& a, const Blk& k_) {
    bool on[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.valid[c] > 0 && a.cs[c].needRefine;
        any |= on[c];
    }
    if (!any || inner_running(a)) return;
    const int64_t n = a.nRed;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, n, 0, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(tl * BLK + k_.tid);
        if (r >= n) continue;
        double acc[6];
        ld6(a.b + (int64_t)NCMP * r, acc);
        for_entries<ENT<double>>(a, r, a.aval, [&](const auto& col, const auto& av) { gather<true>(a.x, col, av, acc); });
        double xv[6];
        ld6(a.x + (int64_t)NCMP * r, xv);
        const double rd = a.rD[r];
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (on[c]) xv[c] = rd * acc[c];
        st6(a.x + (int64_t)NCMP * r, xv);
    }
}

template <class T>
__global__ void __launch_bounds__(BLK) k_rb_backsub(KryArgs<T> a) {
    k_rb_backsub_body<T>(a, blk_of_launch(nullptr));
}

// Pivots of B for a general LDU matrix (the sparseSolver surface):
// Ds_i = D_i - sum over i's faces of lower_f upper_f / D_other, in face order;
// out[0, N) = 1/Ds (1/D on R), out[N, 2N) = D Ds^-1 (1 on R)
__global__ void k_rb_schur_diag(int32_t N, int32_t nRed, const int64_t* __restrict__ off,
                                const int32_t* __restrict__ width, const int32_t* __restrict__ fid,
                                const uint8_t* __restrict__ slot, const int32_t* __restrict__ col,
                                const double* __restrict__ lower, const double* __restrict__ upper,
                                const double* __restrict__ diag, double* __restrict__ out) {
    const int64_t r = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (r >= N) return;
    const double D = diag[r];
    double ds = D;
    if (r >= nRed) {
        const int s = (int)(r >> 6), lane = (int)(r & 63);
        const int64_t base = off[s] + lane;
        const int w = width[s];
        for (int k = 0; k < w; ++k) {
            const int64_t e = base + (int64_t)SLICE * k;
            const int32_t f = fid[e];
            if (f == RT_FID_PAD) continue;
            const int32_t face = f >= 0 ? f : -f - 1;
            const int32_t other = col[base + (int64_t)SLICE * slot[e]];
            ds = ds - (lower[face] * upper[face]) / diag[other];
        }
    }
    out[r] = 1.0 / ds;
    out[N + r] = D / ds;
}

// ================================================= PBiCG ([OF9] PBiCG::solve)
// The reference's tutorials solve theta with PBiCG (bi-conjugate gradients,
// e.g. tutorials/rheoFoam/Channel/Oldroyd-BLog/system/fvSolution:32): per
// iteration wA = M^-1 rA, wT = M^-T rT, wArT = (wA, rT), pA = wA + beta pA,
// pT = wT + beta pT, wA = A pA, wT = A^T pT, alpha = wArT / (wA, pT),
// psi += alpha pA, rA -= alpha wA, rT -= alpha wT.  Lockstep over the
// components like the PBiCGStab above, with M diagonal (rM).  Vectors:
// rA = r, rT = r0, pA = p, pT = v, wA = t, wT = s.

// rT = b - A^T x (FP64) and the first wArT = (M^-1 rA, rT), after the
// initial residual has written rA
template <class T>
__device__ __forceinline__ void k_bicg_init_body(const KryArgs<T>& a, const Blk& k_) {
    bool on[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.cs[c].active;
        any |= on[c];
    }
    if (!any) return;
    double q[6] = {0, 0, 0, 0, 0, 0};
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, a.N, a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(tl * BLK + k_.tid);
        if (r >= a.N) continue;
        const double d = a.diag[r];
        double xv[6], y[6];
        ld6(a.x + (int64_t)NCMP * r, xv);
#pragma unroll
        for (int c = 0; c < 6; ++c) y[c] = d * xv[c];
        KryArgs<T> at = a;
        at.slotMask = nullptr;
        for_entries<ENT<double>>(at, r, a.atval, [&](const auto& col, const auto& av) { gather<false>(a.x, col, av, y); });
        double bb[6];
        ld6(a.b + (int64_t)NCMP * r, bb);
        T rA[6], rT[6];
        ld6(a.r + (int64_t)NCMP * r, rA);
        const double rm = a.rM ? a.rM[r] : 1.0;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            rT[c] = (T)(bb[c] - y[c]);
            if (on[c]) q[c] += (rm * (double)rA[c]) * (double)rT[c];
        }
        st6(a.r0 + (int64_t)NCMP * r, rT);
    }
    write_partials<6>(q, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_bicg_init(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_bicg_init_body<T>(a, blk_of_launch(red));
}

template <class T, int NT = FBLK>
__device__ __forceinline__ void k_fin_bicg_init_body(const KryArgs<T>& a, double* lds) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; ++i) any |= a.cs[i].active != 0;
    if (!any) return;
    const int c = threadIdx.x;
    Comp cs;
    cs.active = 0;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<6, NT>(a.partials, a.G, lds, sums);
    if (!cs.active) return;
    cs.rho = sums[c];
    cs.store(a.cs[c]);
}

template <class T>
__global__ void __launch_bounds__(FBLK) k_fin_bicg_init(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_bicg_init_body<T>(a, lds);
}

// pA = M^-1 rA (+ beta pA), pT = M^-1 rT (+ beta pT)
template <class T>
__device__ __forceinline__ void k_bicg_p_body(const KryArgs<T>& a, const Blk& k_) {
    bool on[6], first[6];
    T beta[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.cs[c].active;
        first[c] = a.cs[c].innerIter == 0;
        beta[c] = (T)a.cs[c].beta;
        any |= on[c];
    }
    if (!any) return;
    for (int64_t i = (int64_t)k_.b * BLK + k_.tid; k_.b < k_.G && i < a.N; i += (int64_t)k_.G * BLK) {
        const T rm = a.rM ? (T)a.rM[i] : (T)1;
        T rA[6], rT[6], pA[6], pT[6];
        ld6(a.r + NCMP * i, rA);
        ld6(a.r0 + NCMP * i, rT);
        ld6(a.p + NCMP * i, pA);
        ld6(a.v + NCMP * i, pT);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (!on[c]) continue;
            const T wA = rm * rA[c], wT = rm * rT[c];
            pA[c] = first[c] ? wA : wA + beta[c] * pA[c];
            pT[c] = first[c] ? wT : wT + beta[c] * pT[c];
        }
        st6(a.p + NCMP * i, pA);
        st6(a.v + NCMP * i, pT);
    }
}

template <class T>
__global__ void __launch_bounds__(BLK) k_bicg_p(KryArgs<T> a) {
    k_bicg_p_body<T>(a, blk_of_launch(nullptr));
}

// wA = A pA, wT = A^T pT; (wA, pT)
template <class T>
__device__ __forceinline__ void k_bicg_w_body(const KryArgs<T>& a, const Blk& k_) {
    bool on[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.cs[c].active;
        any |= on[c];
    }
    if (!any) return;
    T q[6] = {0, 0, 0, 0, 0, 0};
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, a.N, a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(tl * BLK + k_.tid);
        if (r >= a.N) continue;
        const T d = (T)a.diag[r];
        T wA[6], wT[6], pT[6];
        ld6(a.p + (int64_t)NCMP * r, wA);
        ld6(a.v + (int64_t)NCMP * r, pT);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            wA[c] = d * wA[c];
            wT[c] = d * pT[c];
        }
        for_entries<ENT<T>>(a, r, a.aA, [&](const auto& col, const auto& av) { gather<false>(a.p, col, av, wA); });
        KryArgs<T> at = a;
        at.slotMask = nullptr;
        for_entries<ENT<T>>(at, r, a.aT, [&](const auto& col, const auto& av) { gather<false>(a.v, col, av, wT); });
        st6(a.t + (int64_t)NCMP * r, wA);
        st6(a.s + (int64_t)NCMP * r, wT);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (on[c]) q[c] += wA[c] * pT[c];
    }
    double qd[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) qd[c] = q[c];
    write_partials<6>(qd, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_bicg_w(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_bicg_w_body<T>(a, blk_of_launch(red));
}

template <class T, int NT = FBLK>
__device__ __forceinline__ void k_fin_bicg_w_body(const KryArgs<T>& a, double* lds) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; ++i) any |= a.cs[i].active != 0;
    if (!any) return;
    const int c = threadIdx.x;
    Comp cs;
    cs.active = 0;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<6, NT>(a.partials, a.G, lds, sums);
    if (!cs.active) return;
    // checkSingularity(mag(wApT)/normFactor): stop; restarted from the
    // true residual as after a PBiCGStab breakdown
    if (fabs(sums[c]) / cs.normFactor < 1e-300) {
        cs.active = 0;
        cs.needRefine = 1;
        // a correction to fold exists once this inner solve has updated e
        cs.foldE = a.ctl.mixed && cs.innerIter > 0 ? 1 : 0;
    } else {
        cs.alpha = cs.rho / sums[c];
    }
    cs.store(a.cs[c]);
    if (a.host) cs.store(a.host[c]);
}

template <class T>
__global__ void __launch_bounds__(FBLK) k_fin_bicg_w(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_bicg_w_body<T>(a, lds);
}

// psi += alpha pA, rA -= alpha wA, rT -= alpha wT; |rA|, (M^-1 rA, rT)
template <class T>
__device__ __forceinline__ void k_bicg_xr_body(const KryArgs<T>& a, const Blk& k_) {
    constexpr bool MIX = std::is_same<T, float>::value;
    bool on[6], first[6];
    double alpha[6];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        on[c] = a.cs[c].active;
        first[c] = a.cs[c].innerIter == 0;
        alpha[c] = a.cs[c].alpha;
        any |= on[c];
    }
    if (!any) return;
    T q[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) q[i] = 0;
    for (int64_t it = 0; k_.b < k_.G; ++it) {
        const int64_t tl = tile_of_g(it, a.N, a.nRed, k_.G, k_.b);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int32_t r = (int32_t)(tl * BLK + k_.tid);
        if (r >= a.N) continue;
        const int64_t j = (int64_t)NCMP * r;
        const T rm = a.rM ? (T)a.rM[r] : (T)1;
        double xv[6];
        T ev[6], pA[6], wA[6], wT[6], rA[6], rT[6];
        if constexpr (MIX) {
            ld6(a.e + j, ev);
#pragma unroll
            for (int c = 0; c < 6; ++c) xv[c] = first[c] ? 0.0 : (double)ev[c];
        } else {
            ld6(a.x + j, xv);
        }
        ld6(a.p + j, pA);
        ld6(a.t + j, wA);
        ld6(a.s + j, wT);
        ld6(a.r + j, rA);
        ld6(a.r0 + j, rT);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (!on[c]) continue;
            xv[c] += alpha[c] * (double)pA[c];
            rA[c] = rA[c] - (T)alpha[c] * wA[c];
            rT[c] = rT[c] - (T)alpha[c] * wT[c];
            q[c] += fabs(rA[c]);
            q[6 + c] += (rm * rA[c]) * rT[c];
        }
        if constexpr (MIX) {
#pragma unroll
            for (int c = 0; c < 6; ++c) ev[c] = (T)xv[c];
            st6(a.e + j, ev);
        } else {
            st6(a.x + j, xv);
        }
        st6(a.r + j, rA);
        st6(a.r0 + j, rT);
    }
    double qd[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) qd[i] = q[i];
    write_partials<12>(qd, a.partials, k_);
}

template <class T>
__global__ void __launch_bounds__(BLK) k_bicg_xr(KryArgs<T> a) {
    __shared__ double red[RED_MAX * (BLK / 64)];
    k_bicg_xr_body<T>(a, blk_of_launch(red));
}

template <class T, int NT = FBLK>
__device__ __forceinline__ void k_fin_bicg_xr_body(const KryArgs<T>& a, double* lds) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; ++i) any |= a.cs[i].active != 0;
    if (!any) return;
    const int c = threadIdx.x;
    Comp cs;
    cs.active = 0;
    if (c < 6) cs.load(a.cs[c]);
    double* sums;
    sum_partials<12, NT>(a.partials, a.G, lds, sums);
    if (!cs.active) return;
    cs.iter += 1;
    cs.innerIter += 1;
    const double res = sums[c] / cs.normFactor;
    if (!a.ctl.mixed) cs.finalRes = res;
    const bool conv = conv_inner(cs, a.ctl, res);
    bool cont = (!conv && cs.iter < a.ctl.maxIter) || (!a.ctl.mixed && cs.iter < a.ctl.minIter);
    if (a.ctl.mixed && cs.innerIter >= a.ctl.maxInner) cont = false;
    bool breakdown = false;
    if (cont) {
        cs.rhoOld = cs.rho;
        cs.rho = sums[6 + c];
        if (fabs(cs.rho) < 1e-300) {
            cont = false;
            breakdown = true;
        } else {
            cs.beta = cs.rho / cs.rhoOld;
        }
    }
    if (!cont) {
        cs.active = 0;
        if (a.ctl.mixed || breakdown) {
            cs.needRefine = 1;
            cs.foldE = a.ctl.mixed && cs.innerIter > 0 ? 1 : 0;
        } else {
            cs.converged = conv_outer(cs, a.ctl, cs.finalRes);
        }
    }
    cs.store(a.cs[c]);
    if (a.host) cs.store(a.host[c]);
}

template <class T>
__global__ void __launch_bounds__(FBLK) k_fin_bicg_xr(KryArgs<T> a) {
    __shared__ double lds[FIN_LDS];
    k_fin_bicg_xr_body<T>(a, lds);
}

// float copies of the off-diagonals of A and A^T (mixed PBiCG)
__global__ void k_to_f32(int64_t n, const double* __restrict__ a, const double* __restrict__ b,
                         float* __restrict__ fa, float* __restrict__ fb) {
    const int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (i >= n) return;
    fa[i] = (float)a[i];
    fb[i] = (float)b[i];
}

// ---- Ahat = offdiag(A) D^-1 (column scaled), rD = 1/diag ---------------------
__global__ void k_rdiag(int32_t N, const double* __restrict__ diag, double* __restrict__ rD) {
    const int64_t r = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (r < N) rD[r] = 1.0 / diag[r];
}
template <class T>
__device__ __forceinline__ void k_scale_body(const KryArgs<T>& a, const Blk& k_) {
    T* ahat = const_cast<T*>(a.ahat);
    for (int64_t r = (int64_t)k_.b * BLK + k_.tid; k_.b < k_.G && r < a.N; r += (int64_t)k_.G * BLK) {
        const int s = (int)(r >> 6), lane = (int)(r & 63);
        const int64_t base = a.ellOff[s] + lane;
        const int w = a.ellWidth[s];
        const uint32_t live = a.slotMask ? a.slotMask[s] : 0xffffffffu;
        // red-black: A_jk / (D_j Ds_k) on the first colour's rows, A_ij on the second's
        const bool red = r < a.nRed;
        const double rdr = a.ctl.rb && red ? a.rD[r] : 1.0;
        for (int k = 0; k < w; ++k) {
            if (k < 32 && !((live >> k) & 1u)) continue;
            const int64_t e = base + (int64_t)SLICE * k;
            const double av = a.aval[e];
            if (a.ctl.rb) ahat[e] = red ? (T)((av * rdr) * a.rM[a.ellCol[e]]) : (T)av;
            else ahat[e] = a.rM ? (T)(av * a.rM[a.ellCol[e]]) : (T)av;
        }
    }
}
template <class T>
__global__ void __launch_bounds__(BLK) k_scale(KryArgs<T> a) {
    k_scale_body<T>(a, blk_of_launch(nullptr));
}

// ---- mean of x per component (normalisation factor's gAverage(psi)) ---------
__global__ void __launch_bounds__(BLK) k_mean6(int32_t N, const double* __restrict__ x, double* partials) {
    double q[6] = {0, 0, 0, 0, 0, 0};
    for (int64_t it = 0;; ++it) {
        const int64_t tl = tile_of(it, N);
        if (tl < 0) {
            if (tl == -1) break;
            continue;
        }
        const int64_t t0 = tl * BLK;
        const int64_t r = t0 + threadIdx.x;
        if (r >= N) continue;
        double v[6];
        ld6(x + NCMP * r, v);
#pragma unroll
        for (int c = 0; c < 6; ++c) q[c] += v[c];
    }
    __shared__ double red[RED_MAX * (BLK / 64)];
    write_partials<6>(q, partials, blk_of_launch(red));
}

__global__ void __launch_bounds__(FBLK) k_fin_mean6(int32_t N, int G, const double* partials, CompState* cs) {
    __shared__ double lds[FIN_LDS];
    double* sums;
    sum_partials<6>(partials, G, lds, sums);
    if (threadIdx.x < 6) cs[threadIdx.x].xbar = sums[threadIdx.x] / N;
}

// ============================================ resident solve (small meshes)
// The whole solve in one launch.  On a mesh of some ten thousand cells a pass
// is a few microseconds of dependent loads and a launch costs as much again; a
// 128 x 128 channel's step spent two thirds of its time in the solve's 38
// launches and five host round trips.  Here P workgroups of RBLK threads stay
// for the solve, one for each of the row kernels' workgroups that has a tile: it
// runs their bodies (the same tile, the same partial sums), a barrier between the
// passes replaces the launch, and every workgroup finalizes each reduction by
// itself on its own copy of the component records, so all take the same
// branches without asking the host.  The fields are the bits the launches give.
//
// The barrier is one of the XCDs' own (an atomic in the L2 its workgroups share)
// and, where the workgroups are on several XCDs, one of their last arrivals:
// those alone write their L2 back (release) and drop what it holds of the others'
// (acquire).  As one counter for all, with every workgroup fencing, a barrier of
// 98 workgroups took 4.7 us.  A solve that fits one XCD (workgroups are dealt
// round-robin over the eight, so every eighth one of the grid takes part) needs
// no L2 traffic at all.  Where each workgroup runs is read from the hardware.
//
// A workgroup is one tile of BLK rows, so that few waves share a SIMD: a pass of
// one row a thread is bound by instruction issue and latency (512 threads took
// 2.6 us for the x/r pass, 256 take 1.2 us).
//
// The barrier needs the workgroups resident together: the launches take their CUs
// from a budget (ResBudget), but other processes may hold them, so the wait is
// bounded: a workgroup that polls maxPolls times marks the counter and leaves,
// which the others see in their own waits.  The records on the device
// and the saved vectors then still hold the solve's start, and the host runs it
// by launches.
constexpr int RBLK = BLK;
constexpr int XCDS = RES_XCDS;
// workgroups a CU holds: FP32 solves are held to 256 registers a lane for two,
// FP64 ones take up to 350 (held to 256 they spill, and a 128 x 128 channel's
// step took 200 us instead of 179)
template <class T>
constexpr int RES_PER_CU = sizeof(T) == 4 ? 2 : 1;

template <class T>
struct ResArgs {
    KryArgs<T> a, b, s;   // all rows; red-black: the second colour's rows, its sweep residual
    // workgroups: the first P of the row kernels' a.G, those that have a tile;
    // row-kernel workgroups of the pointwise and first-colour passes
    int32_t P, pg, Gw;
    int32_t doScale;
    uint32_t maxPolls, epoch;  // epoch: this launch, what resDone or resFail is set to
    SolveState* st;
    SolveState* host;     // the page-locked copy, or NULL
    // NULL when P = 1: x [N][6], and where the assembly's residual starts the
    // solve (not red-black, whose first sweep makes it) r0 and PBiCG's r
    double* xSave;
};

// the operations of the barrier's words (rt_resident.h)
struct ResAt {
    template <ResScope S>
    static constexpr int scope = S == RES_XCD ? __HIP_MEMORY_SCOPE_WORKGROUP : __HIP_MEMORY_SCOPE_AGENT;
    template <ResScope S>
    static __device__ __forceinline__ uint32_t add(uint32_t* p, uint32_t v) {
        return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, scope<S>);
    }
    template <ResScope S>
    static __device__ __forceinline__ uint32_t or_(uint32_t* p, uint32_t v) {
        return __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, scope<S>);
    }
    template <ResScope S>
    static __device__ __forceinline__ uint32_t swap(uint32_t* p, uint32_t v) {
        return __hip_atomic_exchange(p, v, __ATOMIC_RELAXED, scope<S>);
    }
    static __device__ __forceinline__ uint32_t get(const uint32_t* p) {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ void set(uint32_t* p, uint32_t v) {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ void sleep() { __builtin_amdgcn_s_sleep(1); }
    static __device__ __forceinline__ void release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent"); }
    static __device__ __forceinline__ void acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }
};
__device__ __forceinline__ bool res_enter(ResBar& B, int* bad) {
    if (B.P == 1) {
        __syncthreads();
        return true;
    }
    const uint32_t x = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & 7u;  // hwreg XCC_ID, bits 0..3
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        *bad = res_enter_wait<ResAt>(B, x);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    res_enter_place<ResAt>(B, x);
    return *bad == 0;
}
// Every wave's stores have reached its L2 before the first wave arrives; no wave
// goes on before that one has dropped the CU's L1 (the load after the fence
// returns behind it).
__device__ __forceinline__ bool res_barrier(ResBar& B, int* bad) {
    if (B.P == 1) {
        __syncthreads();
        return true;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    ++B.ph;
    if (threadIdx.x == 0) {
        *bad = res_wait<ResAt>(B);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    return *bad == 0;
}

// RF_RB_ROW, RF_BICG_ROW: every thread keeps one row (red-black: one of each
// colour) for the whole solve, its matrix entries and its words of the vectors
// in registers, and only the vectors that other rows gather go to memory.
enum ResForm { RF_JACOBI = 0, RF_REDBLACK = 1, RF_BICG = 2, RF_RB_ROW = 3, RF_BICG_ROW = 4 };
constexpr int ROW_W = 6;  // entries of a kept row

// A row of a [N][6] vector by its byte offset: 32 bits (a resident mesh has at
// most RES_MAX_ROWS rows), so that an address is a scalar base and one register.
template <class T>
__device__ __forceinline__ uint32_t row_off(int32_t r) {
    return (uint32_t)r * (uint32_t)(NCMP * sizeof(T));
}
template <class T>
__device__ __forceinline__ const T* at_off(const T* p, uint32_t off) {
    return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + off);
}
template <class T>
__device__ __forceinline__ T* at_off(T* p, uint32_t off) {
    return reinterpret_cast<T*>(reinterpret_cast<char*>(p) + off);
}

// the entries of a kept row in column order; 0 where there is none
template <class T>
struct RowEnts {
    uint32_t off[ROW_W];  // of the column's row
    T val[ROW_W];
    // SCALE 0: vals as they are; 1, 2: the FP64 matrix scaled for the red-black
    // solve's first, second colour (k_scale_body's arithmetic)
    template <int SCALE, class V>
    __device__ __forceinline__ void load(const KryArgs<T>& a, int32_t r, const V* vals, bool masked) {
        const int s = r >= 0 ? r >> 6 : 0;
        const int64_t base = a.ellOff[s] + (r & 63);
        const int width = r >= 0 ? a.ellWidth[s] : 0;
        const uint32_t live = masked && a.slotMask ? a.slotMask[s] : 0xffffffffu;
        V v[ROW_W];
        int32_t col[ROW_W];
#pragma unroll
        for (int k = 0; k < ROW_W; ++k) {
            col[k] = 0;
            v[k] = (V)0;
            if (k < width && ((live >> k) & 1u)) {
                const int64_t e = base + (int64_t)SLICE * k;
                col[k] = a.ellCol[e];
                v[k] = vals[e];
            }
        }
        if constexpr (SCALE == 1) {
            const double rdr = r >= 0 ? a.rD[r] : 1.0;
            double m[ROW_W];
#pragma unroll
            for (int k = 0; k < ROW_W; ++k) m[k] = v[k] != (V)0 ? a.rM[col[k]] : 0.0;
#pragma unroll
            for (int k = 0; k < ROW_W; ++k) val[k] = (T)((v[k] * rdr) * m[k]);
        } else {
#pragma unroll
            for (int k = 0; k < ROW_W; ++k) val[k] = (T)v[k];
        }
#pragma unroll
        for (int k = 0; k < ROW_W; ++k) off[k] = row_off<T>(col[k]);
    }
    // acc += val src[col] (NEG: -=), three rows in flight
    template <bool NEG>
    __device__ __forceinline__ void gather(const T* src, T (&acc)[6]) const {
#pragma unroll
        for (int k0 = 0; k0 < ROW_W; k0 += 3) {
            T g[3][6];
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (val[k0 + j] != (T)0) ld6(at_off(src, off[k0 + j]), g[j]);
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (val[k0 + j] != (T)0) {
                    const T v = val[k0 + j];
#pragma unroll
                    for (int c = 0; c < 6; ++c) acc[c] = NEG ? acc[c] - v * g[j][c] : acc[c] + v * g[j][c];
                }
        }
    }
    // the same of s = r - alpha v
    __device__ __forceinline__ void gather_s(const T* rv, const T* vv, const T (&alpha)[6], T (&acc)[6]) const {
#pragma unroll
        for (int k0 = 0; k0 < ROW_W; k0 += 3) {
            T g[3][6], h[3][6];
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (val[k0 + j] != (T)0) {
                    ld6(at_off(rv, off[k0 + j]), g[j]);
                    ld6(at_off(vv, off[k0 + j]), h[j]);
                }
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (val[k0 + j] != (T)0) {
                    const T v = val[k0 + j];
#pragma unroll
                    for (int c = 0; c < 6; ++c) acc[c] += v * (g[j][c] - alpha[c] * h[j][c]);
                }
        }
    }
};

template <class T, int FORM>
__device__ __forceinline__ void solve_resident(const ResArgs<T>& m, int p) {
    constexpr bool RB = FORM == RF_REDBLACK || FORM == RF_RB_ROW, BICG = FORM == RF_BICG || FORM == RF_BICG_ROW;
    constexpr bool MIX = std::is_same<T, float>::value;
    __shared__ CompState cs[6];
    __shared__ double lds[FIN_LDS];
    __shared__ double red[RED_MAX * (BLK / 64)];
    __shared__ int bad;
    const int P = m.P, tid = threadIdx.x;
    for (int i = threadIdx.x; i < (int)(sizeof(cs) / 8); i += RBLK)
        reinterpret_cast<double*>(cs)[i] = reinterpret_cast<const double*>(m.a.cs)[i];
    __syncthreads();
    KryArgs<T> a = m.a, b = m.b, sw = m.s;
    a.cs = b.cs = sw.cs = cs;
    a.host = b.host = sw.host = nullptr;
    // Each pass with a reduction writes its plan's slot of the partial sums.  No
    // barrier stands between a workgroup's reads of a reduction and the passes
    // after it: Jacobi's t pass follows the v pass's finalizer at once, and its v
    // pass (no p pass in an inner solve's first round) the sweep's.
    constexpr ResPlan plan = BICG ? RES_PLAN_BICG : RES_PLAN_STAB;
    auto slot = [&](ResSlot s) { return m.a.partials + (int64_t)RES_SLOT_BEGIN[s] * m.a.G; };
    KryArgs<T> av = a, at = a, ax = a;  // the v (PBiCG: w), t and x/r passes
    av.partials = slot(plan.slot[0]);
    at.partials = slot(plan.slot[1]);
    ax.partials = slot(plan.slot[plan.n - 1]);
    sw.partials = a.partials = slot(RES_SWEEP_SLOT);
    // the finalizers sum the workgroups that have a tile: the others add zeros
    KryArgs<T> fv = av, ft = at, fx = ax, fs = a;
    fv.G = ft.G = fx.G = fs.G = P;
    ResBar bar{m.st->bar, m.st->barL2, P, 1, P, nullptr, m.maxPolls, 0, (uint32_t)(m.P > 0)};
    auto wait = [&] { return res_barrier(bar, &bad); };
    // workgroup p of a pass of G row-kernel workgroups
    auto pass = [&](int G, auto&& body) {
        if (p < G) body(Blk{G, p, tid, red});
    };
    if (m.xSave) {
        const int64_t n6 = (int64_t)NCMP * a.N;
        for (int64_t i = (int64_t)p * RBLK + threadIdx.x; i < n6; i += (int64_t)P * RBLK) {
            m.xSave[i] = a.x[i];
            if constexpr (!RB) reinterpret_cast<T*>(m.xSave + n6)[i] = a.r0[i];
            if constexpr (BICG) reinterpret_cast<T*>(m.xSave + 2 * n6)[i] = a.r[i];
        }
    }
    if (m.doScale && FORM < RF_RB_ROW) {
        if constexpr (BICG) {
            // the float copies of A and A^T, by rows
            if constexpr (MIX)
                for (int64_t r = (int64_t)p * RBLK + threadIdx.x; r < a.N; r += (int64_t)P * RBLK) {
                    const int64_t base = a.ellOff[r >> 6] + (r & 63);
                    for (int k = 0; k < a.ellWidth[r >> 6]; ++k) {
                        const int64_t e = base + (int64_t)SLICE * k;
                        const_cast<T*>(a.aA)[e] = (T)a.aval[e];
                        const_cast<T*>(a.aT)[e] = (T)a.atval[e];
                    }
                }
        } else {
            pass(P, [&](const Blk& k) { k_scale_body<T>(a, k); });
        }
    }
    bool ok = res_enter(bar, &bad);
    // the kept rows: tile p of the rows (red-black: of each colour)
    constexpr bool ROW = FORM == RF_RB_ROW || FORM == RF_BICG_ROW;
    const Blk kRow{a.G, p, tid, red};
    int32_t rR = -1, rB = -1;
    RowEnts<T> eR, eB;  // red-black: the first and the second colour's row; PBiCG: A^T's and A's
    T w0[6], wr[6], wp[6], wv[6], dgB = (T)1;
    using XT = std::conditional_t<MIX, float, double>;
    XT X[6];
    double rdB = 1.0;
    uint32_t oR = 0, oB = 0;
    if constexpr (ROW) {
        const int64_t i = (int64_t)p * BLK + tid;
        if constexpr (RB) {
            const int64_t rb = (a.nRed & ~(SLICE - 1)) + i;
            if (i < a.nRed) rR = (int32_t)i;
            if (rb >= a.nRed && rb < a.N) rB = (int32_t)rb;
            eR.template load<1>(a, rR, a.aval, true);
            eB.template load<2>(a, rB, a.aval, true);
            if (rB >= 0 && a.dg) dgB = (T)a.dg[rB];
        } else {
            if (i < a.N) rB = (int32_t)i;
            // the FP32 solve's float copies of A and A^T are made here
            eB.template load<0>(a, rB, a.aval, true);
            eR.template load<0>(a, rB, a.atval, false);
            if (rB >= 0) dgB = (T)a.diag[rB];
        }
        if (rB >= 0 && a.rM) rdB = a.rM[rB];
        if (rR >= 0) oR = row_off<T>(rR);
        if (rB >= 0) oB = row_off<T>(rB);
#pragma unroll
        for (int c = 0; c < 6; ++c) w0[c] = wr[c] = wp[c] = wv[c] = (T)0, X[c] = 0;
    }
    for (int round = 0; ok && round < 100000; ++round) {
        bool act = false, ref = false, fold = false;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (a.valid[c] <= 0) continue;
            act |= cs[c].active != 0;
            ref |= cs[c].needRefine != 0;
            fold |= cs[c].needRefine && cs[c].foldE;
        }
        if (!act && !ref) break;
        if (!act) {
            if (fold) {
                pass(m.pg, [&](const Blk& k) { k_fold_body<T>(RB ? b : a, k); });
                ok = wait();
            }
            if constexpr (RB) {
                if (ok) {
                    pass(m.Gw, [&](const Blk& k) { k_rb_backsub_body<T>(a, k); });
                    ok = wait();
                }
            }
            if (!ok) break;
            pass(a.G, [&](const Blk& k) { k_residual_body<T, 1>(RB ? sw : a, k); });
            ok = wait();
            if (!ok) break;
            k_fin_residual_body<T, 1, RBLK>(fs, lds);
            __syncthreads();
            continue;
        }
        if constexpr (FORM == RF_RB_ROW) {
            const Round rd = round_of(a);
            const bool start = rd.inner == 0;
            const T* pv = start ? a.r0 : a.p;
            const T* rv = start ? a.r0 : a.r;
            if (start) {
                if (rB >= 0) ld6(at_off(a.r0, oB), w0);
                if constexpr (!MIX)
                    if (rB >= 0) ld6(at_off(a.x, oB), X);
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    wr[c] = wp[c] = w0[c];
                    if constexpr (MIX) X[c] = 0.0f;
                }
            } else {
                T be[6], om[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    be[c] = (T)uni(cs[c].beta);
                    om[c] = (T)uni(cs[c].omega);
                }
#pragma unroll
                for (int c = 0; c < 6; ++c)
                    if (rd.on[c]) wp[c] = wr[c] + be[c] * (wp[c] - om[c] * wv[c]);
                if (rB >= 0) st6(at_off(a.p, oB), wp);
                ok = wait();
                if (!ok) break;
            }
            {
                T acc[6] = {0, 0, 0, 0, 0, 0};
                eR.template gather<false>(pv, acc);
                if (rR >= 0) st6(at_off(a.v, oR), acc);
            }
            ok = wait();
            if (!ok) break;
            {
#pragma unroll
                for (int c = 0; c < 6; ++c) wv[c] = a.dg ? dgB * wp[c] : wp[c];
                eB.template gather<true>(a.v, wv);
                double q[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) q[c] = rd.on[c] && rB >= 0 ? (T)0 + w0[c] * wv[c] : (T)0;
                if (rB >= 0) st6(at_off(a.v, oB), wv);
                write_partials<6>(q, av.partials, kRow);
            }
            ok = wait();
            if (!ok) break;
            k_fin_v_body<T, RBLK>(fv, lds);
            __syncthreads();
            T al[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) al[c] = (T)uni(cs[c].alpha);
            {
                T acc[6] = {0, 0, 0, 0, 0, 0};
                eR.gather_s(rv, a.v, al, acc);
                if (rR >= 0) st6(at_off(a.t, oR), acc);
            }
            ok = wait();
            if (!ok) break;
            T wt[6];
            {
                T sv[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    sv[c] = wr[c] - al[c] * wv[c];
                    wt[c] = a.dg ? dgB * sv[c] : sv[c];
                }
                eB.template gather<true>(a.t, wt);
                double q[18];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    const bool o = rd.on[c] && rB >= 0;
                    q[c] = o ? (T)fabs(sv[c]) : (T)0;
                    q[6 + c] = o ? (T)0 + wt[c] * sv[c] : (T)0;
                    q[12 + c] = o ? (T)0 + wt[c] * wt[c] : (T)0;
                }
                write_partials<18>(q, at.partials, kRow);
            }
            ok = wait();
            if (!ok) break;
            k_fin_t_body<T, RBLK>(ft, lds);
            __syncthreads();
            {
                double q[12], alphas[6], omegas[6];
                bool ex[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    alphas[c] = uni(cs[c].alpha);
                    omegas[c] = uni(cs[c].omega);
                    ex[c] = uni(cs[c].exitAtS);
                }
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    q[c] = q[6 + c] = (T)0;
                    if (!rd.on[c]) continue;
                    const double alpha = alphas[c], omega = omegas[c];
                    double xv = X[c];
                    const double y = rdB * (double)wp[c];
                    if (ex[c]) {
                        xv += alpha * y;
                    } else {
                        const T sv = wr[c] - (T)alpha * wv[c];
                        const double z = rdB * (double)sv;
                        xv += alpha * y + omega * z;
                        const T rn = sv - (T)omega * wt[c];
                        wr[c] = rn;
                        if (rB >= 0) {
                            q[c] = (T)fabs(rn);
                            q[6 + c] = (T)0 + w0[c] * rn;
                        }
                    }
                    X[c] = (XT)xv;
                }
                if (rB >= 0) {
                    st6(at_off(a.r, oB), wr);
                    if constexpr (MIX) st6(at_off(a.e, oB), X);
                    else st6(at_off(a.x, oB), X);
                }
                write_partials<12>(q, ax.partials, kRow);
            }
            ok = wait();
            if (!ok) break;
            k_fin_xr_body<T, RBLK>(fx, lds);
            __syncthreads();
        } else if constexpr (FORM == RF_BICG_ROW) {
            const Round rd = round_of(a);
            const bool start = rd.inner == 0;
            if (start) {
                if (rB >= 0) ld6(at_off(a.r, oB), wr);
                if (rB >= 0) ld6(at_off(a.r0, oB), w0);
                if constexpr (!MIX)
                    if (rB >= 0) ld6(at_off(a.x, oB), X);
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    wp[c] = wv[c] = (T)0;
                    if constexpr (MIX) X[c] = 0.0f;
                }
            }
            const T rm = a.rM ? (T)rdB : (T)1;
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                if (!rd.on[c]) continue;
                const T be = (T)uni(cs[c].beta);
                const T wA = rm * wr[c], wT = rm * w0[c];
                wp[c] = start ? wA : wA + be * wp[c];
                wv[c] = start ? wT : wT + be * wv[c];
            }
            if (rB >= 0) {
                st6(at_off(a.p, oB), wp);
                st6(at_off(a.v, oB), wv);
            }
            ok = wait();
            if (!ok) break;
            T wA[6], wT[6];
            {
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    wA[c] = dgB * wp[c];
                    wT[c] = dgB * wv[c];
                }
                eB.template gather<false>(a.p, wA);
                eR.template gather<false>(a.v, wT);
                double q[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) q[c] = rd.on[c] && rB >= 0 ? (T)0 + wA[c] * wv[c] : (T)0;
                write_partials<6>(q, av.partials, kRow);
            }
            ok = wait();
            if (!ok) break;
            k_fin_bicg_w_body<T, RBLK>(fv, lds);
            __syncthreads();
            {
                double q[12];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    q[c] = q[6 + c] = (T)0;
                    if (!uni(cs[c].active)) continue;
                    const double alpha = uni(cs[c].alpha);
                    X[c] = (XT)((double)X[c] + alpha * (double)wp[c]);
                    wr[c] = wr[c] - (T)alpha * wA[c];
                    w0[c] = w0[c] - (T)alpha * wT[c];
                    if (rB >= 0) {
                        q[c] = (T)fabs(wr[c]);
                        q[6 + c] = (T)0 + (rm * wr[c]) * w0[c];
                    }
                }
                if (rB >= 0) {
                    if constexpr (MIX) st6(at_off(a.e, oB), X);
                    else st6(at_off(a.x, oB), X);
                }
                write_partials<12>(q, ax.partials, kRow);
            }
            ok = wait();
            if (!ok) break;
            k_fin_bicg_xr_body<T, RBLK>(fx, lds);
            __syncthreads();
        } else if constexpr (BICG) {
            pass(m.pg, [&](const Blk& k) { k_bicg_p_body<T>(a, k); });
            ok = wait();
            if (!ok) break;
            pass(a.G, [&](const Blk& k) { k_bicg_w_body<T>(av, k); });
            ok = wait();
            if (!ok) break;
            k_fin_bicg_w_body<T, RBLK>(fv, lds);
            __syncthreads();
            pass(a.G, [&](const Blk& k) { k_bicg_xr_body<T>(ax, k); });
            ok = wait();
            if (!ok) break;
            k_fin_bicg_xr_body<T, RBLK>(fx, lds);
            __syncthreads();
        } else {
            if (round_of(a).inner > 0) {
                pass(m.pg, [&](const Blk& k) { k_kry_p_body<T>(RB ? b : a, k); });
                ok = wait();
                if (!ok) break;
            }
            if constexpr (RB) {
                pass(m.Gw, [&](const Blk& k) { k_rb_w_body<T, 0>(a, k); });
                ok = wait();
                if (!ok) break;
                pass(a.G, [&](const Blk& k) { k_rb_v_body<T>(av, k); });
            } else {
                pass(a.G, [&](const Blk& k) { k_kry_v_body<T>(av, k); });
            }
            ok = wait();
            if (!ok) break;
            k_fin_v_body<T, RBLK>(fv, lds);
            __syncthreads();
            if constexpr (RB) {
                pass(m.Gw, [&](const Blk& k) { k_rb_w_body<T, 1>(a, k); });
                ok = wait();
                if (!ok) break;
                pass(a.G, [&](const Blk& k) { k_rb_t_body<T>(at, k); });
            } else {
                pass(a.G, [&](const Blk& k) { k_kry_t_body<T>(at, k); });
            }
            ok = wait();
            if (!ok) break;
            k_fin_t_body<T, RBLK>(ft, lds);
            __syncthreads();
            pass(a.G, [&](const Blk& k) { k_kry_xr_body<T>(ax, k); });
            ok = wait();
            if (!ok) break;
            k_fin_xr_body<T, RBLK>(fx, lds);
            __syncthreads();
        }
    }
    if (ok && p == 0)
        for (int i = threadIdx.x; i < (int)(sizeof(cs) / 8); i += RBLK) {
            const double w = reinterpret_cast<const double*>(cs)[i];
            reinterpret_cast<double*>(m.a.cs)[i] = w;
            if (m.host) reinterpret_cast<double*>(m.host->c)[i] = w;
        }
    if (threadIdx.x == 0 && (!ok || p == 0)) {
        (ok ? m.st->resDone : m.st->resFail) = m.epoch;
        if (m.host) (ok ? m.host->resDone : m.host->resFail) = m.epoch;
    }
    if (ok && P > 1 && threadIdx.x == 0) res_depart<ResAt>(bar);
}

// map: per workgroup of the grid its member and index in it, -1 for none
template <class T, int FORM>
__global__ void __launch_bounds__(RBLK, RES_PER_CU<T>) k_solve_group(const ResArgs<T>* __restrict__ tab, const int2* __restrict__ map) {
    const int2 w = map[blockIdx.x];
    if (w.x < 0) return;
    solve_resident<T, FORM>(tab[w.x], w.y);
}

// workgroup b of the grid: b % XCDS is the XCD it is dealt to; xcd < 0: on all
template <class T, int FORM>
__global__ void __launch_bounds__(RBLK, RES_PER_CU<T>) k_solve_one(ResArgs<T> m, int xcd) {
    if (xcd >= 0 && (int)(blockIdx.x % XCDS) != xcd) return;
    solve_resident<T, FORM>(m, xcd >= 0 ? blockIdx.x / XCDS : blockIdx.x);
}

// ----------------------------------------------------------------- driver
static inline unsigned kblk(int64_t n) { return (unsigned)((n + BLK - 1) / BLK); }

void launch_rb_schur_diag(Ctx* ctx, const Mesh& m, const double* lower, const double* upper, const double* diag,
                          double* out) {
    if (m.N <= 0) return;
    ProfScope ps(ctx, "k_rb_schur_diag", (double)m.N * 32 + (double)m.nEll * 9 + (double)m.F * 16);
    hipLaunchKernelGGL(k_rb_schur_diag, dim3(kblk(m.N)), dim3(BLK), 0, ctx->stream, m.N, m.nRed,
                       m.ellOff.as<int64_t>(), m.ellWidth.as<int32_t>(), m.ellFid.as<int32_t>(),
                       m.ellSlot.as<uint8_t>(), m.ellCol.as<int32_t>(), lower, upper, diag, out);
    RT_HIP(hipGetLastError());
}

void launch_mean6(Ctx* ctx, int32_t N, const double* x, double* partials, CompState* cs,
                  int grid) {
    {
        ProfScope ps(ctx, "k_mean6", (double)N * 48);
        hipLaunchKernelGGL(k_mean6, dim3(grid), dim3(BLK), 0, ctx->stream, N, x, partials);
    }
    hipLaunchKernelGGL(k_fin_mean6, dim3(1), dim3(FBLK), 0, ctx->stream, N, grid, partials, cs);
    RT_HIP(hipGetLastError());
}

KryCtl kryCtl(const Controls& C, bool mixed, const Mesh& m) {
    KryCtl k{};
    k.tol = C.tolerance;
    k.relTol = C.relTol;
    k.innerRelTol = C.innerRelTol;
    k.maxIter = C.maxIter;
    k.minIter = C.minIter;
    k.maxInner = 200;
    k.maxRefine = C.maxRefine;
    k.mixed = mixed ? 1 : 0;
    k.bicg = C.solver == SV_PBICG ? 1 : 0;
    k.precond = C.precond;
    // multicolour ILU0 runs as the red-black solve on a colour-blocked mesh
    // with PBiCGStab; the DILU keyword takes it where it is available and the
    // diagonal preconditioner elsewhere, multicolourILU0 demands it
    k.rb = C.precond == PC_MCILU0 && m.nRed > 0 && C.solver == SV_PBICGSTAB ? 1 : 0;
    if (C.precond == PC_MCILU0 && !k.rb) {
        if (C.precondStrict)
            throw Error{RT_E_UNSUPPORTED,
                        std::string("preconditioner multicolourILU0 needs solver PBiCGStab and a mesh whose cell "
                                    "graph is two-colourable (this one is ") +
                            (m.nRed > 0 ? "two-coloured; the solver is " + C.solverName : std::string("not")) + ")"};
        k.precond = PC_JACOBI;
    }
    return k;
}

void Krylov::ensure(Ctx* run, Mesh& m, bool mixed, bool bicg) {
    if (!ctx) ctx = m.ctx;
    const size_t vec = (size_t)6 * m.N;
    if (noAlloc) {
        const bool ok = N == m.N && partials.p && state.p && rD.p && (mixed ? rs.p && r0s.p && ps.p && vs.p &&
                                                                          ts.p && es.p && ahat32.p
                                                                    : r.p && r0.p && p.p && v.p && t.p && ahat64.p) &&
                        (!bicg || (atval.p && (mixed ? s32.p && a32.p && at32.p : s64.p != nullptr)));
        if (!ok) throw Error{RT_E_BAD_ARG, "Krylov workspace bound to scratch memory does not fit the solve"};
        return;
    }
    if (N != m.N) {
        N = m.N;
        grid = grid_for(ctx, N);
        r = DBuf(); r0 = DBuf(); p = DBuf(); v = DBuf(); t = DBuf();
        rs = DBuf(); r0s = DBuf(); ps = DBuf(); vs = DBuf(); ts = DBuf(); es = DBuf();
        ahat32 = DBuf(); ahat64 = DBuf();
        // a resident solve's reductions have slots of their own
        partials = ctx->alloc((size_t)grid * (N <= RES_MAX_ROWS ? RES_SUMS : 24) * sizeof(double));
        state = ctx->alloc(sizeof(SolveState));
        // on the solve's stream: on the mesh's, behind other work, the zeros could
        // land on records the assembly had written
        static_assert(sizeof(SolveState) % 8 == 0, "filled by 8-byte words");
        launch_fill(run, state.as<double>(), sizeof(SolveState) / 8, 0.0);
        rD = ctx->alloc(std::max<size_t>(1, (size_t)m.N) * sizeof(double));
    }
    if (!mixed && !r.p) {
        r = ctx->alloc(vec * 8); r0 = ctx->alloc(vec * 8); p = ctx->alloc(vec * 8);
        v = ctx->alloc(vec * 8); t = ctx->alloc(vec * 8);
        ahat64 = ctx->alloc(std::max<int64_t>(1, m.nEll) * 8);
    }
    if (mixed && !rs.p) {
        rs = ctx->alloc(vec * 4); r0s = ctx->alloc(vec * 4); ps = ctx->alloc(vec * 4);
        vs = ctx->alloc(vec * 4); ts = ctx->alloc(vec * 4); es = ctx->alloc(vec * 4);
        ahat32 = ctx->alloc(std::max<int64_t>(1, m.nEll) * 4);
    }
    if (bicg) {
        if (!atval.p) atval = ctx->alloc(std::max<int64_t>(1, m.nEll) * 8);
        if (!mixed && !s64.p) s64 = ctx->alloc(vec * 8);
        if (mixed && !s32.p) {
            s32 = ctx->alloc(vec * 4);
            a32 = ctx->alloc(std::max<int64_t>(1, m.nEll) * 4);
            at32 = ctx->alloc(std::max<int64_t>(1, m.nEll) * 4);
        }
    }
}

// Resumable solve: begin() launches the initial residual (unless the assembly
// already produced it), every advance() reads the device state of the
// previous round (non-blocking when asked) and launches the next round, so
// several solves can progress on their own streams at once (the serving loop)
// or one can run to completion (rt_model_correct / rt_symm_solve).
struct SolveRun {
    bool mixed = false;
    KryArgs<float> af{};
    KryArgs<double> ad{};
    int G = 1, pgrid = 1;
    int Gw = 1;                       // red-black: the first colour's gather passes (no partial sums)
    double N = 0, ne = 0, nValid = 0;
    int32_t valid[6];
    Ctx* ctx = nullptr;
    SolveState* hostState = nullptr;  // pinned block of ctx
    CompState* host = nullptr;        // = hostState->c
    bool neFromDevice = false;        // matrix entry count comes with the first status pull
    bool needScale = false;           // Ahat (or the float copies of A, A^T) not built yet
    bool bicg = false;                // PBiCG instead of PBiCGStab
    bool rb = false;                  // red-black ILU0: Krylov on the second colour's Schur complement
    double nRed = 0;                  // first colour's rows
    KryArgs<float> bf{};              // red-black: af/ad shifted to the second colour's rows
    KryArgs<double> bd{};             // (the pointwise passes p and the fold)
    KryArgs<float> sf{};              // red-black: the residual restricted to the second colour
    KryArgs<double> sd{};
    int64_t nEll = 0;                 // all ELL entries (the float copies of A, A^T)
    hipEvent_t ev = nullptr;
    bool ownsHost = false;            // hostState is a pinned block of ctx
    bool pending = false, done = false;
    int rounds = 0;
    // the whole solve in one launch of P workgroups (k_solve_one / k_solve_group)
    bool resident = false, resLaunched = false;
    int P = 1, form = 0;
    uint32_t maxPolls = 0, epoch = 0;
    DBuf xSave;  // the start of a resident solve of several workgroups (ResArgs::xSave)
    SolveState* st = nullptr;
    ResHold hold;  // the resident launch's CUs
    ~SolveRun() {
        if (hostState && ownsHost) ctx->givePinnedBlock(hostState);
        if (ev) (void)hipEventDestroy(ev);
    }
};

void SolveRunDeleter::operator()(SolveRun* r) const { delete r; }

namespace {

template <class T>
KryArgs<T>& argsOf(SolveRun& R);
template <>
KryArgs<float>& argsOf<float>(SolveRun& R) { return R.af; }
template <>
KryArgs<double>& argsOf<double>(SolveRun& R) { return R.ad; }
template <class T>
KryArgs<T>& blackOf(SolveRun& R);
template <>
KryArgs<float>& blackOf<float>(SolveRun& R) { return R.bf; }
template <>
KryArgs<double>& blackOf<double>(SolveRun& R) { return R.bd; }
template <class T>
KryArgs<T>& sweepOf(SolveRun& R);
template <>
KryArgs<float>& sweepOf<float>(SolveRun& R) { return R.sf; }
template <>
KryArgs<double>& sweepOf<double>(SolveRun& R) { return R.sd; }

// Workgroups of the solve's row kernels (the passes that launch with the
// solve grid and write partial sums) that fit on the chip at once: the least
// over those kernels of the workgroups per CU their VGPRs allow, times the CUs.
// Each workgroup walks its share of the tiles in a loop, so a grid larger than
// that runs in rounds, and the workgroups of a later round find the
// neighbours they gather gone from L2.
template <class T>
int solve_grid(const Ctx* ctx, int cap, bool rb, bool bicg) {
    static int perCU[2][2] = {{0, 0}, {0, 0}};  // [rb][bicg], the same on every gfx950 device
    int& pc = perCU[rb ? 1 : 0][bicg ? 1 : 0];
    if (pc == 0) {
        int least = 8;
        auto take = [&](auto fn) {
            int nb = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, BLK, 0) == hipSuccess && nb > 0)
                least = std::min(least, nb);
        };
        take(k_residual<T, 0>);
        take(k_residual<T, 1>);
        if (bicg) {
            take(k_bicg_init<T>);
            take(k_bicg_w<T>);
            take(k_bicg_xr<T>);
        } else if (rb) {
            take(k_rb_backsub<T>);
            take(k_rb_w<T, 0>);
            take(k_rb_w<T, 1>);
            take(k_rb_v<T>);
            take(k_rb_t<T>);
            take(k_kry_xr<T>);
        } else {
            take(k_kry_v<T>);
            take(k_kry_t<T>);
            take(k_kry_xr<T>);
        }
        pc = least;
    }
    int64_t g = std::min<int64_t>(cap, (int64_t)ctx->numCUs * pc);
    if (g >= 64 && g < cap) g = g / 8 * 8;
    return (int)std::max<int64_t>(1, g);
}

// The red-black passes over the first colour's rows (w, w', the elimination)
// reduce nothing, so they take a grid of their own: every workgroup their
// VGPRs allow at once.
template <class T>
int rb_wide_grid(const Ctx* ctx, int cap) {
    static int perCU = 0;
    if (perCU == 0) {
        int least = 8;
        auto take = [&](auto fn) {
            int nb = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, BLK, 0) == hipSuccess && nb > 0)
                least = std::min(least, nb);
        };
        take(k_rb_w<T, 0>);
        take(k_rb_w<T, 1>);
        take(k_rb_backsub<T>);
        perCU = least;
    }
    int64_t g = std::min<int64_t>(cap, (int64_t)ctx->numCUs * perCU);
    if (g >= 64 && g < cap) g = g / 8 * 8;
    return (int)std::max<int64_t>(1, g);
}

template <class T>
void fill_args(Ctx* ctx, const SolveArgs& sa, SolveRun& R) {
    Mesh& m = *sa.mesh;
    Krylov& K = *sa.kry;
    const bool mixed = std::is_same<T, float>::value;
    const int32_t N = m.N;
    SolveState* st = K.state.as<SolveState>();
    double* rD = K.rD.as<double>();
    if (!sa.initDone) {
        ProfScope ps(ctx, "k_rdiag", (double)N * 16);
        hipLaunchKernelGGL(k_rdiag, dim3(kblk(N)), dim3(BLK), 0, ctx->stream, N, sa.diag, rD);
    }
    T* ahat = mixed ? (T*)K.ahat32.p : (T*)K.ahat64.p;
    R.needScale = m.nEll > 0;  // launched with the first round, once the entry count is known
    RT_HIP(hipGetLastError());
    KryArgs<T>& a = argsOf<T>(R);
    a = KryArgs<T>{};
    a.N = N;
    a.ellOff = m.ellOff.as<int64_t>();
    a.ellWidth = m.ellWidth.as<int32_t>();
    a.ellCol = m.ellCol.as<int32_t>();
    a.aval = sa.aval;
    a.slotMask = sa.slotMask;
    a.diag = sa.diag;
    a.ahat = ahat;
    a.rD = rD;
    a.b = sa.b;
    a.x = sa.x;
    if (mixed) {
        a.r = (T*)K.rs.p; a.r0 = (T*)K.r0s.p; a.p = (T*)K.ps.p; a.v = (T*)K.vs.p; a.t = (T*)K.ts.p;
        a.e = (T*)K.es.p;
    } else {
        a.r = (T*)K.r.p; a.r0 = (T*)K.r0.p; a.p = (T*)K.p.p; a.v = (T*)K.v.p; a.t = (T*)K.t.p;
        a.e = nullptr;
    }
    a.partials = K.partials.as<double>();
    a.cs = st->c;
    a.host = R.ownsHost ? R.hostState->c : nullptr;
    for (int c = 0; c < 6; ++c) a.valid[c] = sa.valid[c];
    a.ctl = kryCtl(*sa.ctl, mixed, m);
    R.G = solve_grid<T>(ctx, K.grid, a.ctl.rb != 0, sa.ctl->solver == SV_PBICG);
    R.Gw = a.ctl.rb ? rb_wide_grid<T>(ctx, K.grid) : R.G;
    a.G = R.G;
    a.nRed = m.nRed;
    a.rowBegin = 0;
    // the preconditioner: Jacobi M = D (M^-1 = rD, A M^-1 has a unit diagonal)
    // or none (M^-1 = 1, diag(A M^-1) = D); red-black: M = Ds on the second
    // colour (M^-1 = 1/Ds, diag(S M^-1) = D Ds^-1, 1 when Ds = D)
    const bool jac = a.ctl.precond == PC_JACOBI;
    a.rM = jac ? rD : nullptr;
    a.dg = jac ? nullptr : sa.diag;
    R.rb = a.ctl.rb != 0;
    R.nRed = m.nRed;
    if (R.rb) {
        a.rM = sa.rDs ? sa.rDs : rD;
        a.dg = sa.rDs ? sa.rDs + N : nullptr;
        // pointwise passes on the second colour's rows: the same kernels on
        // pointers shifted by nRed rows
        const int64_t o = (int64_t)NCMP * m.nRed;
        KryArgs<T>& b = blackOf<T>(R);
        b = a;
        b.N = N - m.nRed;
        b.nRed = 0;
        b.x = a.x + o;
        b.b = a.b + o;
        b.r += o; b.r0 += o; b.p += o; b.v += o; b.t += o;
        if (b.e) b.e += o;
        b.rM = a.rM + m.nRed;
        b.dg = a.dg ? a.dg + m.nRed : nullptr;
        b.rD = a.rD + m.nRed;
        b.diag = a.diag + m.nRed;
        KryArgs<T>& sw = sweepOf<T>(R);
        sw = a;
        sw.rowBegin = m.nRed;
    }
    R.bicg = sa.ctl->solver == SV_PBICG;
    if (R.bicg) {
        a.atval = sa.atval;
        a.s = mixed ? (T*)K.s32.p : (T*)K.s64.p;
        a.aA = mixed ? (const T*)K.a32.p : (const T*)sa.aval;
        a.aT = mixed ? (const T*)K.at32.p : (const T*)sa.atval;
    }
}

// algorithmic bytes per launch for nc participating components: ELL entries
// (col + value) once per SpMV, each vector once per pass (interleaved rows
// move all 6 components; gathered vectors counted once)
struct Bytes {
    double N, ne, w;
    double res(double nc) const { return N * 8.0 + ne * 12 + nc * N * (8 + 8 + w); }
    double p(double nc) const { return nc * N * 4 * w; }
    double v(double nc, bool start) const { return ne * (4 + w) + nc * N * (start ? 2 : 3) * w; }
    double t(double nc) const { return ne * (4 + w) + nc * N * 3 * w; }
    // FP64: x read and written in place; mixed: the FP32 correction instead
    double xr(double nc, bool start) const {
        return N * 8.0 + nc * N * (w == 4 ? (start ? 5 : 8) * w : 16 + (start ? 4 : 6) * w);
    }
    double fold(double nc) const { return nc * N * (8 + 8 + w); }
    // PBiCG: rT = b - A^T x; the p pass; A pA and A^T pT; the x/r pass
    double binit(double nc) const { return N * 16.0 + ne * 12 + nc * N * (8 + 8 + 2 * w); }
    double bp(double nc) const { return N * 8.0 + nc * N * 6 * w; }
    double bw(double nc) const { return N * 8.0 + 2 * ne * (4 + w) + nc * N * 4 * w; }
    double bxr(double nc) const { return N * 8.0 + nc * N * (w == 4 ? 9 * w : 16 + 7 * w); }
    // red-black (N = rows of the colour the pass runs on, ne its ELL entries):
    // w gathers one or two vectors of the other colour and writes one; the
    // second colour's v and t passes gather w and stream their own vectors;
    // the elimination of the first colour and the sweep's residual in FP64
    double rbw(double nc, int src) const { return ne * (4 + w) + nc * N * (src ? 3 : 2) * w; }
    double rbv(double nc, bool start) const { return ne * (4 + w) + nc * N * (start ? 3 : 4) * w; }
    double rbt(double nc) const { return ne * (4 + w) + nc * N * 5 * w; }
    double rbx(double nc) const { return N * 8.0 + ne * 12 + nc * N * (8 + 8 + 8); }
};

// the scaled off-diagonals of the solve (Jacobi: A D^-1; red-black: its two
// colours' forms), built before the first iteration
template <class T>
void launch_scale_of(Ctx* ctx, SolveRun& R) {
    const bool mixed = std::is_same<T, float>::value;
    KryArgs<T>& a = argsOf<T>(R);
    ProfScope ps(ctx, R.rb ? (mixed ? "k_rb_scale<f32>" : "k_rb_scale<f64>") : (mixed ? "k_scale<f32>" : "k_scale<f64>"),
                 R.ne * (4 + 8 + sizeof(T)) + R.N * 8);
    hipLaunchKernelGGL(k_scale<T>, dim3(kblk((int64_t)R.N)), dim3(BLK), 0, ctx->stream, a);
    RT_HIP(hipGetLastError());
    R.needScale = false;
}

template <class T>
void launch_init(Ctx* ctx, SolveRun& R) {
    const bool mixed = std::is_same<T, float>::value;
    Bytes B{R.N, R.ne, (double)sizeof(T)};
    {
        ProfScope ps(ctx, mixed ? "k_residual<f32>" : "k_residual<f64>", B.res(R.nValid));
        hipLaunchKernelGGL((k_residual<T, 0>), dim3(R.G), dim3(BLK), 0, ctx->stream, argsOf<T>(R));
    }
    hipLaunchKernelGGL((k_fin_residual<T, 0>), dim3(1), dim3(FBLK), 0, ctx->stream, argsOf<T>(R));
}

// PBiCG: rT = b - A^T x and the first wArT, once the initial residual is in
template <class T>
void launch_bicg_init(Ctx* ctx, SolveRun& R) {
    const bool mixed = std::is_same<T, float>::value;
    Bytes B{R.N, R.ne, (double)sizeof(T)};
    {
        ProfScope ps(ctx, mixed ? "k_bicg_init<f32>" : "k_bicg_init<f64>", B.binit(R.nValid));
        hipLaunchKernelGGL(k_bicg_init<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, argsOf<T>(R));
    }
    hipLaunchKernelGGL(k_fin_bicg_init<T>, dim3(1), dim3(FBLK), 0, ctx->stream, argsOf<T>(R));
}

// The refinement sweep: mixed-precision fold, then the FP64 true residual and
// its finalize (which converges, restarts or stops each waiting component).
// fold: a component about to be refined holds an inner correction (the
// blocking path knows; queued rounds launch it gated on the device).
// Red-black: the fold and the residual run on the second colour's rows and
// the elimination of the first colour runs between them.
template <class T>
void launch_refine(Ctx* ctx, SolveRun& R, double nRef, bool fold = true) {
    const bool mixed = std::is_same<T, float>::value;
    Bytes B{R.N, R.ne, (double)sizeof(T)};
    KryArgs<T>& a = argsOf<T>(R);
    if (R.rb) {
        const double w = (double)sizeof(T);
        Bytes Bb{R.N - R.nRed, 0.5 * R.ne, w}, Br{R.nRed, 0.5 * R.ne, w};
        const int pg = std::max(1, std::min<int>(R.pgrid, (int)((R.N - R.nRed + BLK - 1) / BLK)));
        if (mixed && fold) {
            ProfScope ps(ctx, "k_fold<f32>", Bb.fold(nRef));
            hipLaunchKernelGGL(k_fold<T>, dim3(pg), dim3(BLK), 0, ctx->stream, blackOf<T>(R));
        }
        {
            ProfScope ps(ctx, mixed ? "k_rb_backsub<f32>" : "k_rb_backsub<f64>", Br.rbx(nRef));
            hipLaunchKernelGGL(k_rb_backsub<T>, dim3(R.Gw), dim3(BLK), 0, ctx->stream, a);
        }
        {
            ProfScope ps(ctx, mixed ? "k_residual<f32>" : "k_residual<f64>", Bb.res(nRef));
            hipLaunchKernelGGL((k_residual<T, 1>), dim3(R.G), dim3(BLK), 0, ctx->stream, sweepOf<T>(R));
        }
        hipLaunchKernelGGL((k_fin_residual<T, 1>), dim3(1), dim3(FBLK), 0, ctx->stream, a);
        return;
    }
    if (mixed && fold) {
        ProfScope ps(ctx, "k_fold<f32>", B.fold(nRef));
        hipLaunchKernelGGL(k_fold<T>, dim3(R.pgrid), dim3(BLK), 0, ctx->stream, a);
    }
    {
        ProfScope ps(ctx, mixed ? "k_residual<f32>" : "k_residual<f64>", B.res(nRef));
        hipLaunchKernelGGL((k_residual<T, 1>), dim3(R.G), dim3(BLK), 0, ctx->stream, a);
    }
    hipLaunchKernelGGL((k_fin_residual<T, 1>), dim3(1), dim3(FBLK), 0, ctx->stream, a);
}

// One lockstep PBiCGStab iteration of the nAct active components.  start: the
// host knows it to be their inner solve's first (no p pass).
template <class T>
void launch_iter(Ctx* ctx, SolveRun& R, double nAct, bool start) {
    const bool mixed = std::is_same<T, float>::value;
    Bytes B{R.N, R.ne, (double)sizeof(T)};
    KryArgs<T>& a = argsOf<T>(R);
    if (R.bicg) {
        if (R.needScale && mixed) {
            const int64_t n = std::max<int64_t>(1, R.nEll);
            ProfScope ps(ctx, "k_to_f32", (double)n * 24);
            hipLaunchKernelGGL(k_to_f32, dim3(kblk(n)), dim3(BLK), 0, ctx->stream, n, a.aval, a.atval,
                               (float*)const_cast<T*>(a.aA), (float*)const_cast<T*>(a.aT));
        }
        R.needScale = false;
        {
            ProfScope ps(ctx, mixed ? "k_bicg_p<f32>" : "k_bicg_p<f64>", B.bp(nAct));
            hipLaunchKernelGGL(k_bicg_p<T>, dim3(R.pgrid), dim3(BLK), 0, ctx->stream, a);
        }
        {
            ProfScope ps(ctx, mixed ? "k_bicg_w<f32>" : "k_bicg_w<f64>", B.bw(nAct));
            hipLaunchKernelGGL(k_bicg_w<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
        }
        hipLaunchKernelGGL(k_fin_bicg_w<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
        {
            ProfScope ps(ctx, mixed ? "k_bicg_xr<f32>" : "k_bicg_xr<f64>", B.bxr(nAct));
            hipLaunchKernelGGL(k_bicg_xr<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
        }
        hipLaunchKernelGGL(k_fin_bicg_xr<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
        return;
    }
    if (R.rb) {
        if (R.needScale) launch_scale_of<T>(ctx, R);
        const double w = (double)sizeof(T);
        Bytes Bb{R.N - R.nRed, 0.5 * R.ne, w}, Br{R.nRed, 0.5 * R.ne, w};
        KryArgs<T>& b = blackOf<T>(R);
        const int pg = std::max(1, std::min<int>(R.pgrid, (int)((R.N - R.nRed + BLK - 1) / BLK)));
        // w lives on the first colour's rows of v, w' on those of t
        if (!start) {
            ProfScope ps(ctx, mixed ? "k_kry_p<f32>" : "k_kry_p<f64>", Bb.p(nAct));
            hipLaunchKernelGGL(k_kry_p<T>, dim3(pg), dim3(BLK), 0, ctx->stream, b);
        }
        {
            ProfScope ps(ctx, mixed ? "k_rb_w<f32>" : "k_rb_w<f64>", Br.rbw(nAct, 0));
            hipLaunchKernelGGL((k_rb_w<T, 0>), dim3(R.Gw), dim3(BLK), 0, ctx->stream, a);
        }
        {
            ProfScope ps(ctx, mixed ? "k_rb_v<f32>" : "k_rb_v<f64>", Bb.rbv(nAct, start));
            hipLaunchKernelGGL(k_rb_v<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
        }
        hipLaunchKernelGGL(k_fin_v<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
        {
            ProfScope ps(ctx, mixed ? "k_rb_ws<f32>" : "k_rb_ws<f64>", Br.rbw(nAct, 1));
            hipLaunchKernelGGL((k_rb_w<T, 1>), dim3(R.Gw), dim3(BLK), 0, ctx->stream, a);
        }
        {
            ProfScope ps(ctx, mixed ? "k_rb_t<f32>" : "k_rb_t<f64>", Bb.rbt(nAct));
            hipLaunchKernelGGL(k_rb_t<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
        }
        hipLaunchKernelGGL(k_fin_t<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
        {
            ProfScope ps(ctx, mixed ? "k_kry_xr<f32>" : "k_kry_xr<f64>", Bb.xr(nAct, start));
            hipLaunchKernelGGL(k_kry_xr<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
        }
        hipLaunchKernelGGL(k_fin_xr<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
        return;
    }
    if (R.needScale) launch_scale_of<T>(ctx, R);
    if (!start) {
        ProfScope ps(ctx, mixed ? "k_kry_p<f32>" : "k_kry_p<f64>", B.p(nAct));
        hipLaunchKernelGGL(k_kry_p<T>, dim3(R.pgrid), dim3(BLK), 0, ctx->stream, a);
    }
    {
        ProfScope ps(ctx, mixed ? "k_kry_v<f32>" : "k_kry_v<f64>", B.v(nAct, start));
        hipLaunchKernelGGL(k_kry_v<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
    }
    hipLaunchKernelGGL(k_fin_v<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
    {
        ProfScope ps(ctx, mixed ? "k_kry_t<f32>" : "k_kry_t<f64>", B.t(nAct));
        hipLaunchKernelGGL(k_kry_t<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
    }
    hipLaunchKernelGGL(k_fin_t<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
    {
        ProfScope ps(ctx, mixed ? "k_kry_xr<f32>" : "k_kry_xr<f64>", B.xr(nAct, start));
        hipLaunchKernelGGL(k_kry_xr<T>, dim3(R.G), dim3(BLK), 0, ctx->stream, a);
    }
    hipLaunchKernelGGL(k_fin_xr<T>, dim3(1), dim3(FBLK), 0, ctx->stream, a);
}

// the workgroups of a member's pointwise passes (p, fold)
int point_grid(const SolveRun& R) {
    if (!R.rb) return R.pgrid;
    return std::max(1, std::min<int>(R.pgrid, (int)((R.N - R.nRed + BLK - 1) / BLK)));
}

// Whether the solve runs as one resident launch, and its workgroups (a row a
// thread): a mesh of at most RES_MAX_ROWS rows, with the workspace it needs and
// no kernel timing (which charges every pass its bytes).
// f(kernel instantiation of the form)
template <class T, class F>
auto with_form(int form, F&& f) {
    switch (form) {
    case RF_REDBLACK: return f(std::integral_constant<int, RF_REDBLACK>{});
    case RF_BICG: return f(std::integral_constant<int, RF_BICG>{});
    case RF_RB_ROW: return f(std::integral_constant<int, RF_RB_ROW>{});
    case RF_BICG_ROW: return f(std::integral_constant<int, RF_BICG_ROW>{});
    default: return f(std::integral_constant<int, RF_JACOBI>{});
    }
}

// whether a CU holds the workgroups its share of the budget stands for
template <class T>
bool resident_fits(int form) {
    return with_form<T>(form, [](auto F) {
        static const bool fits = [] {  // the same on every gfx950 device
            int one = 0, grp = 0;
            return hipOccupancyMaxActiveBlocksPerMultiprocessor(&one, k_solve_one<T, decltype(F)::value>, RBLK, 0) == hipSuccess &&
                   hipOccupancyMaxActiveBlocksPerMultiprocessor(&grp, k_solve_group<T, decltype(F)::value>, RBLK, 0) == hipSuccess &&
                   std::min(one, grp) >= RES_PER_CU<T>;
        }();
        return fits;
    });
}

constexpr int RES_DEVICES = 64;
ResBudget resBudgets[RES_DEVICES];
constexpr int HALF_CUS = 2;  // the budget's units on a CU
int half_cus(const Ctx* ctx) { return HALF_CUS * ctx->numCUs / XCDS; }

template <class T>
void choose_resident(Ctx* ctx, const SolveArgs& sa, SolveRun& R) {
    Krylov& K = *sa.kry;
    R.resident = R.resLaunched = false;
    if (sa.ctl->residentPolls == 0 || ctx->profiling || K.N > RES_MAX_ROWS || ctx->device >= RES_DEVICES) return;
    if (R.G % 8 == 0 || R.Gw % 8 == 0 || K.partials.bytes < (size_t)RES_SUMS * K.grid * sizeof(double)) return;
    const Mesh& m = *sa.mesh;
    // row-kernel workgroups with a tile: the first ones (tile t is workgroup t's where
    // the grid is no multiple of 8)
    const int32_t row0 = R.rb ? m.nRed & ~(SLICE - 1) : 0;
    R.P = std::max((int)kblk(m.N - row0), R.rb ? (int)kblk(m.nRed) : 1);
    if (R.P > R.G) return;
    const bool row = m.maxWidth <= ROW_W;
    R.form = R.bicg ? (row ? RF_BICG_ROW : RF_BICG) : R.rb ? (row ? RF_RB_ROW : RF_REDBLACK) : RF_JACOBI;
    if (R.P > ctx->numCUs / 2) return;
    // Half the CUs at a row a thread (red-black: one of each colour): 65536 rows
    // red-black, 32768 in the other forms.  Measured (us a step, by launches /
    // resident): rows kept, red-black FP64 233 / 146 at 4096 cells, 285 / 207 at
    // 16384, 356 / 299 at 65536, PBiCG 511 / 326 at 16384; the passes over memory of
    // Jacobi 338 / 266 at 16384 and, before the limit on the CUs, 385 / 349 at 36864 and
    // 466 / 475 at 65536.  (Red-black rows wider than six take the passes over memory
    // too.)
    if (R.form < RF_RB_ROW && m.N > RES_MAX_ROWS / 2) return;
    if (R.P > 1 && K.noAlloc && !K.xSave.p) return;
    if (!resident_fits<T>(R.form) || (R.P > 1 && ctx->backoff->skip())) return;
    R.maxPolls = sa.ctl->residentPolls;
    R.st = K.state.as<SolveState>();
    R.resident = true;
}

template <class T>
ResArgs<T> resident_args(SolveRun& R) {
    ResArgs<T> m{};
    m.a = argsOf<T>(R);
    m.b = R.rb ? blackOf<T>(R) : m.a;
    m.s = R.rb ? sweepOf<T>(R) : m.a;
    m.P = R.P;
    m.pg = point_grid(R);
    m.Gw = R.Gw;
    m.doScale = R.needScale ? 1 : 0;
    m.maxPolls = R.maxPolls;
    m.epoch = R.epoch = ++R.ctx->resEpoch;
    m.st = R.st;
    m.host = R.ownsHost ? R.hostState : nullptr;
    m.xSave = R.xSave.as<double>();
    return m;
}

// Memory for the solve's start, taken at the launch, behind everything the step
// allocates, and given back when the solve has finished: a budget that holds the
// step holds it without this, and then the solve runs by launches (false).
bool take_save(Krylov& K, SolveRun& R) {
    if (R.P == 1) return true;
    const size_t bytes = sizeof(double) * NCMP * K.N * (1 + !R.rb + R.bicg);
    if (K.noAlloc) {
        R.xSave = DBuf::viewOf(K.xSave.p, K.xSave.bytes);
        return true;
    }
    try {
        // the mesh's context, where the solve's vectors are from; if that has a
        // budget, a server's other requests may still need it
        R.xSave = (K.ctx->budget ? R.ctx : K.ctx)->alloc(bytes);
    } catch (const Error& e) {
        if (e.code != RT_E_OOM) throw;
        return false;
    }
    return true;
}

// false: no memory for its start, or the device has no room for its workgroups
// beside the resident launches under way (a single workgroup waits for none)
template <class T>
bool launch_resident(Ctx* ctx, Krylov& K, SolveRun& R) {
    int xcd = ctx->xcd;
    if (!take_save(K, R)) return false;
    if (R.P > 1) {
        xcd = resBudgets[ctx->device].take(R.P, HALF_CUS / RES_PER_CU<T>, half_cus(ctx), ctx->xcd, ctx->lane, R.hold);
        if (xcd == RES_FULL) return false;
    }
    const ResArgs<T> m = resident_args<T>(R);
    const int grid = xcd < 0 ? R.P : R.P == 1 ? xcd + 1 : XCDS * R.P;
    with_form<T>(R.form, [&](auto F) {
        hipLaunchKernelGGL((k_solve_one<T, decltype(F)::value>), dim3(grid), dim3(RBLK), 0, ctx->stream, m, xcd);
    });
    RT_HIP(hipGetLastError());
    R.resLaunched = true;
    return true;
}

// rounds a non-blocking advance queues per host round trip
constexpr int kRoundsAhead = 3;

// The records' way to the host: the kernels write the page-locked copy
// themselves, so only the event is left (a copy was a kernel of 2 to 5 us and a
// launch in every round trip); a caller's pageable block is copied to.
void queue_pull(Ctx* ctx, Krylov& K, SolveRun& R) {
    if (!R.ownsHost)
        RT_HIP(hipMemcpyAsync(R.hostState, K.state.as<SolveState>(), sizeof(SolveState), hipMemcpyDeviceToHost,
                              ctx->stream));
    if (R.ev) RT_HIP(hipEventRecord(R.ev, ctx->stream));
    R.pending = true;
}

}  // namespace

SolveState* solve_prepare(Ctx* ctx, Krylov& K, SolveState* hostStatus) {
    if (K.run && hostStatus && K.run->hostState != hostStatus) K.run.reset();
    if (!K.run) {
        static_assert(sizeof(SolveState) <= Ctx::kPinnedBlock, "status block too small");
        K.run.reset(new SolveRun);
        K.run->ctx = ctx;
        if (hostStatus) {
            // the caller's pageable block, no event: a blocking solve waits on
            // the stream (the no-allocation path)
            K.run->hostState = hostStatus;
        } else {
            K.run->hostState = static_cast<SolveState*>(ctx->takePinnedBlock());
            memset(static_cast<void*>(K.run->hostState), 0, sizeof(SolveState));
            K.run->ownsHost = true;
            RT_HIP(hipEventCreateWithFlags(&K.run->ev, hipEventDisableTiming));
        }
        K.run->host = K.run->hostState->c;
    }
    return K.run->ownsHost ? K.run->hostState : nullptr;
}

void solve_begin(Ctx* ctx, const SolveArgs& sa) {
    Mesh& m = *sa.mesh;
    Krylov& K = *sa.kry;
    const bool mixed = sa.ctl->mixed;
    const bool bicg = sa.ctl->solver == SV_PBICG;
    K.ensure(ctx, m, mixed, bicg);
    if (bicg && !sa.atval) throw Error{RT_E_BAD_ARG, "PBiCG needs the transposed matrix"};
    (void)solve_prepare(ctx, K, sa.hostStatus);
    SolveRun& R = *K.run;
    R.ctx = ctx;
    R.mixed = mixed;
    R.G = K.grid;
    R.pgrid = std::min<int>(K.grid, (int)kblk(m.N));
    R.N = m.N;
    R.ne = (double)m.nEll;
    R.nEll = m.nEll;
    R.neFromDevice = sa.slotMask != nullptr;
    R.nValid = 0;
    for (int c = 0; c < 6; ++c) {
        R.valid[c] = sa.valid[c];
        R.nValid += sa.valid[c] > 0;
    }
    R.done = false;
    R.rounds = 0;
    R.hold.release();
    R.xSave.release();
    if (mixed) {
        fill_args<float>(ctx, sa, R);
        choose_resident<float>(ctx, sa, R);
        if (!sa.initDone) launch_init<float>(ctx, R);
        if (bicg) launch_bicg_init<float>(ctx, R);
    } else {
        fill_args<double>(ctx, sa, R);
        choose_resident<double>(ctx, sa, R);
        if (!sa.initDone) launch_init<double>(ctx, R);
        if (bicg) launch_bicg_init<double>(ctx, R);
    }
    RT_HIP(hipGetLastError());
    if (R.resident) {
        // nothing to decide on the host before the resident launch; the event
        // is what a group's stream waits for
        R.pending = false;
        if (R.ev) RT_HIP(hipEventRecord(R.ev, ctx->stream));
        return;
    }
    queue_pull(ctx, K, R);
}

namespace {

void back_off(Ctx* ctx) {
    ctx->backoff->gaveUp();
    // the contexts of processes that share a device all start on the same XCDs:
    // each leaves in steps of its own
    ctx->xcd = (ctx->xcd + 1 + (int)(getpid() % (XCDS - 1))) % XCDS;
}

// components of the state last pulled that are still iterating or waiting for a sweep
void open_components(const SolveRun& R, double& nAct, double& nRef) {
    nAct = nRef = 0;
    for (int c = 0; c < 6; ++c) {
        if (R.valid[c] <= 0) continue;
        nAct += R.host[c].active != 0;
        nRef += R.host[c].needRefine != 0;
    }
}

// A resident launch whose state is back.  True: the solve is finished.  A
// workgroup's wait that gave up leaves the counters set; the records then
// either are final (it gave up behind the last barrier, which every workgroup
// had reached) or still the start's, and the solve is run by launches from the
// saved vectors.
bool resident_done(Ctx* ctx, SolveRun& R) {
    if (R.hostState->resFail == R.epoch) {
        launch_fill(ctx, reinterpret_cast<double*>(R.st->bar), sizeof(R.st->bar) / 8, 0.0);
        launch_fill(ctx, reinterpret_cast<double*>(R.st->barL2), sizeof(R.st->barL2) / 8, 0.0);
    }
    if (R.hostState->resDone == R.epoch) return true;
    ++R.ctx->solveCounts[1];
    const size_t n6 = (size_t)6 * (size_t)R.N;
    const size_t w = R.mixed ? sizeof(float) : sizeof(double);
    const size_t nv = (n6 * w + 15) / 16 * 16;  // whole 16-byte words; the buffers are padded to 256
    const double* save = R.xSave.as<double>();
    launch_copy(ctx, save, R.mixed ? R.af.x : R.ad.x, n6 * sizeof(double));
    if (!R.rb) launch_copy(ctx, save + n6, R.mixed ? (void*)R.af.r0 : (void*)R.ad.r0, nv);
    if (R.bicg) launch_copy(ctx, save + 2 * n6, R.mixed ? (void*)R.af.r : (void*)R.ad.r, nv);
    R.resident = R.resLaunched = false;
    R.needScale = R.nEll > 0;
    return false;
}

}  // namespace

bool solve_queue_resident(Ctx* ctx, Krylov& K, SolveGate& gate) {
    SolveRun& R = *K.run;
    if (!R.resident || R.resLaunched || R.done) return false;
    R.resident = R.mixed ? launch_resident<float>(ctx, K, R) : launch_resident<double>(ctx, K, R);
    queue_pull(ctx, K, R);
    if (!R.resident) return false;
    gate = SolveGate{&R.st->resDone, R.epoch};
    return true;
}

bool solve_resident(const Krylov& K) { return K.run->resident; }
SolveGate solve_gate(const Krylov& K) { return SolveGate{&K.run->st->resDone, K.run->epoch}; }

bool solve_advance(Ctx* ctx, Krylov& K, bool block) {
    SolveRun& R = *K.run;
    if (R.done) return true;
    if (R.resident && !R.resLaunched && !block && R.P > 1) {
        // many solves advanced without batching would launch their barriers on
        // many streams at once, more workgroups than fit together
        R.resident = false;
        queue_pull(ctx, K, R);
        return false;
    }
    SolveGate gate;
    if (solve_queue_resident(ctx, K, gate)) return false;
    if (R.pending) {
        if (block) {
            if (R.ev) RT_HIP(hipEventSynchronize(R.ev));
            else RT_HIP(hipStreamSynchronize(ctx->stream));
        } else if (!R.ev) {
            throw Error{RT_E_BAD_ARG, "a solve without a status event can only be advanced blocking"};
        } else {
            hipError_t e = hipEventQuery(R.ev);
            if (e == hipErrorNotReady) return false;
            RT_HIP(e);
        }
        R.pending = false;
        R.hold.release();
        if (R.neFromDevice) {
            R.ne = R.hostState->misc[0];
            R.neFromDevice = false;
        }
    }
    if (R.resident) {
        if (resident_done(ctx, R)) {
            ctx->backoff->finished();
            R.done = true;
            return true;
        }
        back_off(ctx);
    }
    double nAct = 0, nRef = 0;
    bool start = true;  // every component of the round begins an inner solve (p = r = r0)
    for (int c = 0; c < 6; ++c) {
        if (R.valid[c] <= 0) continue;
        nAct += R.host[c].active != 0;
        nRef += R.host[c].needRefine != 0;
        if (R.host[c].active && R.host[c].innerIter != 0) start = false;
    }
    if ((nAct == 0 && nRef == 0) || R.rounds >= 100000) {
        R.done = true;
        return true;
    }
    // A refinement sweep costs a full FP64 pass whatever the number of
    // components in it: components whose inner solve stopped wait (idle, no
    // state change) until every inner solve has stopped, then refine together.
    if (nAct > 0) nRef = 0;
    if (block) {
        // Blocking callers (rt_model_correct, rt_symm_solve, every profiled
        // run) launch exactly what the host's view of the state asks for: a
        // round is either one refinement sweep or one Krylov iteration of the
        // components active now.  A sweep may converge every component, so the
        // iteration after it is only launched once its state is back; no
        // kernel is launched (or charged bytes) for a finished solve.
        if (nAct > 0) {
            if (R.mixed) launch_iter<float>(ctx, R, nAct, start);
            else launch_iter<double>(ctx, R, nAct, start);
        } else {
            bool fold = false;
            for (int c = 0; c < 6; ++c) fold |= R.valid[c] > 0 && R.host[c].needRefine && R.host[c].foldE;
            if (R.mixed) launch_refine<float>(ctx, R, nRef, fold);
            else launch_refine<double>(ctx, R, nRef, fold);
        }
        ++R.rounds;
    } else {
        // Non-blocking callers (the serving loop) queue kRoundsAhead rounds of
        // sweep + iteration before the state comes back: every kernel reads
        // the component records on the device and does nothing for finished
        // components, and the sweep is gated there on no inner solve running,
        // so a round launched ahead does what the host would have launched.
        // This hides the host round trip, which dominates small solves.
        for (int k = 0; k < kRoundsAhead; ++k) {
            const double nR = k == 0 ? nRef : 1, nA = k == 0 ? nAct + nRef : nAct;
            if (R.mixed) {
                if (nR > 0) launch_refine<float>(ctx, R, nR);
                launch_iter<float>(ctx, R, nA, k == 0 && start && nRef == 0);
            } else {
                if (nR > 0) launch_refine<double>(ctx, R, nR);
                launch_iter<double>(ctx, R, nA, k == 0 && start && nRef == 0);
            }
            ++R.rounds;
        }
    }
    RT_HIP(hipGetLastError());
    queue_pull(ctx, K, R);
    return false;
}

// ---------------------------------------------------------- grouped rounds
namespace {

// the member of workgroup blk: starts[i] <= blk < starts[i + 1]
__device__ __forceinline__ int group_of(const int32_t* __restrict__ starts, int n, int blk) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (starts[mid] <= blk) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template <class T, void (*Body)(const KryArgs<T>&, const Blk&)>
__global__ void __launch_bounds__(BLK) k_group(const KryArgs<T>* __restrict__ tab, const int32_t* __restrict__ starts,
                                               int n) {
    const int i = group_of(starts, n, blockIdx.x);
    const KryArgs<T> a = tab[i];
    __shared__ double red[RED_MAX * (BLK / 64)];
    Body(a, Blk{starts[i + 1] - starts[i], (int)blockIdx.x - starts[i], (int)threadIdx.x, red});
}

template <class T, void (*Body)(const KryArgs<T>&, double*)>
__global__ void __launch_bounds__(FBLK) k_group_fin(const KryArgs<T>* __restrict__ tab) {
    __shared__ double lds[FIN_LDS];
    const KryArgs<T> a = tab[blockIdx.x];
    Body(a, lds);
}

// device tables of a group: the members' arguments (whole rows; the red-black
// second colour's rows; its sweep residual) and the workgroup offsets of each
// launch shape (row kernels, pointwise passes, finalizers)
template <class T>
struct GroupDev {
    const KryArgs<T>* A;
    const KryArgs<T>* B;
    const KryArgs<T>* S;
    const int32_t *G, *P, *W;
    int n, totG, totP, totW;
};

template <class T, void (*Body)(const KryArgs<T>&, const Blk&)>
void glaunch(hipStream_t st, const KryArgs<T>* tab, const int32_t* starts, int total, int n) {
    if (total > 0) hipLaunchKernelGGL((k_group<T, Body>), dim3(total), dim3(BLK), 0, st, tab, starts, n);
}

template <class T, void (*Body)(const KryArgs<T>&, double*)>
void glaunch_fin(hipStream_t st, const KryArgs<T>* tab, int n) {
    hipLaunchKernelGGL((k_group_fin<T, Body>), dim3(n), dim3(FBLK), 0, st, tab);
}

// One round as solve_advance queues it ahead for one solve: the refinement
// sweep (every kernel gated on the device) and one iteration.
template <class T>
void group_round(bool rb, hipStream_t st, const GroupDev<T>& d) {
    const int n = d.n;
    if (rb) {
        glaunch<T, &k_fold_body<T>>(st, d.B, d.P, d.totP, n);
        glaunch<T, &k_rb_backsub_body<T>>(st, d.A, d.W, d.totW, n);
        glaunch<T, &k_residual_body<T, 1>>(st, d.S, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_residual_body<T, 1>>(st, d.A, n);
        glaunch<T, &k_kry_p_body<T>>(st, d.B, d.P, d.totP, n);
        glaunch<T, &k_rb_w_body<T, 0>>(st, d.A, d.W, d.totW, n);
        glaunch<T, &k_rb_v_body<T>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_v_body<T>>(st, d.A, n);
        glaunch<T, &k_rb_w_body<T, 1>>(st, d.A, d.W, d.totW, n);
        glaunch<T, &k_rb_t_body<T>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_t_body<T>>(st, d.A, n);
        glaunch<T, &k_kry_xr_body<T>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_xr_body<T>>(st, d.A, n);
    } else {
        glaunch<T, &k_fold_body<T>>(st, d.A, d.P, d.totP, n);
        glaunch<T, &k_residual_body<T, 1>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_residual_body<T, 1>>(st, d.A, n);
        glaunch<T, &k_kry_p_body<T>>(st, d.A, d.P, d.totP, n);
        glaunch<T, &k_kry_v_body<T>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_v_body<T>>(st, d.A, n);
        glaunch<T, &k_kry_t_body<T>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_t_body<T>>(st, d.A, n);
        glaunch<T, &k_kry_xr_body<T>>(st, d.A, d.G, d.totG, n);
        glaunch_fin<T, &k_fin_xr_body<T>>(st, d.A, n);
    }
    RT_HIP(hipGetLastError());
}

// page-locked staging and device memory for a group's tables
void group_tables(SolveGroup& g, size_t bytes) {
    if (g.hostBytes < bytes) {
        if (g.hostTables) (void)hipHostFree(g.hostTables);
        g.hostTables = nullptr;
        RT_HIP(hipHostMalloc(&g.hostTables, bytes, hipHostMallocDefault));
        g.hostBytes = bytes;
    }
    if (g.tables.bytes < bytes) g.tables = g.ctx->alloc(bytes);
}

// the member leaves the group and goes on by launches, behind the group's queued work
void group_evict(SolveGroup& g, size_t i, std::vector<SolveGroup::Member>& evicted) {
    SolveRun& R = *g.members[i].K->run;
    R.resident = false;
    queue_pull(g.ctx, *g.members[i].K, R);
    evicted.push_back(g.members[i]);
    g.members.erase(g.members.begin() + i);
    g.dirty = true;
}

// A group of resident solves: every member's whole solve, in launches that the
// budget has the CUs for.
template <class T>
void group_launch_resident(SolveGroup& g, std::vector<SolveGroup::Member>& evicted) {
    std::vector<ResMember> ms;
    std::vector<int> left;
    for (size_t i = g.members.size(); i-- > 0;)
        if (!take_save(*g.members[i].K, *g.members[i].K->run)) group_evict(g, i, evicted);
    for (const auto& mb : g.members) ms.push_back({mb.K->run->P, mb.K->run->form});
    const std::vector<ResLaunch> launches =
        resBudgets[g.ctx->device].group(ms, HALF_CUS / RES_PER_CU<T>, half_cus(g.ctx), g.ctx->lane, g.hold, left);
    std::vector<SolveGroup::Member> all = g.members;  // the launches' maps index these
    for (size_t k = left.size(); k-- > 0;) group_evict(g, left[k], evicted);
    if (g.members.empty()) return;
    const int n = (int)all.size();
    size_t blocks = 0;
    for (auto& L : launches) blocks += L.map.size();
    const size_t szA = sizeof(ResArgs<T>) * n, bytes = szA + sizeof(int2) * blocks;
    group_tables(g, bytes);
    auto* tab = static_cast<ResArgs<T>*>(g.hostTables);
    auto* map = reinterpret_cast<int2*>(static_cast<unsigned char*>(g.hostTables) + szA);
    for (int i = 0; i < n; ++i)
        if (all[i].K->run->resident) tab[i] = resident_args<T>(*all[i].K->run);
    for (auto& L : launches)
        for (const auto& w : L.map) *map++ = int2{w[0], w[1]};
    RT_HIP(hipMemcpyAsync(g.tables.p, g.hostTables, bytes, hipMemcpyHostToDevice, g.ctx->stream));
    const auto* dt = static_cast<const ResArgs<T>*>(g.tables.p);
    const auto* dm = reinterpret_cast<const int2*>(static_cast<const unsigned char*>(g.tables.p) + szA);
    for (auto& L : launches) {
        const dim3 grid((unsigned)L.map.size());
        with_form<T>(L.form, [&](auto F) {
            hipLaunchKernelGGL((k_solve_group<T, decltype(F)::value>), grid, dim3(RBLK), 0, g.ctx->stream, dt, dm);
        });
        dm += L.map.size();
    }
    RT_HIP(hipGetLastError());
    for (auto& mb : g.members) {
        mb.K->run->resLaunched = true;
        queue_pull(g.ctx, *mb.K, *mb.K->run);
    }
    g.launched = true;
    ++g.launches;
}

template <class T>
void group_launch(SolveGroup& g) {
    const int n = (int)g.members.size();
    const size_t szA = sizeof(KryArgs<T>) * n, szI = sizeof(int32_t) * (n + 1);
    const size_t offB = szA, offS = 2 * szA, offG = 3 * szA, offP = offG + szI, offW = offP + szI;
    const size_t bytes = offW + szI;
    int totG = 0, totP = 0, totW = 0;
    if (g.dirty) {
        group_tables(g, bytes);
        unsigned char* h = static_cast<unsigned char*>(g.hostTables);
        auto* tA = reinterpret_cast<KryArgs<T>*>(h);
        auto* tB = reinterpret_cast<KryArgs<T>*>(h + offB);
        auto* tS = reinterpret_cast<KryArgs<T>*>(h + offS);
        auto* sG = reinterpret_cast<int32_t*>(h + offG);
        auto* sP = reinterpret_cast<int32_t*>(h + offP);
        auto* sW = reinterpret_cast<int32_t*>(h + offW);
        sG[0] = sP[0] = sW[0] = 0;
        for (int i = 0; i < n; ++i) {
            SolveRun& R = *g.members[i].K->run;
            tA[i] = argsOf<T>(R);
            tB[i] = g.rb ? blackOf<T>(R) : argsOf<T>(R);
            tS[i] = g.rb ? sweepOf<T>(R) : argsOf<T>(R);
            sG[i + 1] = sG[i] + R.G;
            sP[i + 1] = sP[i] + point_grid(R);
            sW[i + 1] = sW[i] + R.Gw;
        }
        // the previous launch's kernels have all finished (their pulls are back)
        RT_HIP(hipMemcpyAsync(g.tables.p, h, bytes, hipMemcpyHostToDevice, g.ctx->stream));
        g.dirty = false;
    }
    for (auto& mb : g.members) {
        SolveRun& R = *mb.K->run;
        totG += R.G;
        totP += point_grid(R);
        totW += R.Gw;
    }
    const unsigned char* d = static_cast<const unsigned char*>(g.tables.p);
    GroupDev<T> dv{reinterpret_cast<const KryArgs<T>*>(d), reinterpret_cast<const KryArgs<T>*>(d + offB),
                   reinterpret_cast<const KryArgs<T>*>(d + offS), reinterpret_cast<const int32_t*>(d + offG),
                   reinterpret_cast<const int32_t*>(d + offP), reinterpret_cast<const int32_t*>(d + offW),
                   n, totG, totP, totW};
    for (int k = 0; k < kRoundsAhead; ++k) group_round<T>(g.rb, g.ctx->stream, dv);
    for (auto& mb : g.members) {
        SolveRun& R = *mb.K->run;
        R.rounds += kRoundsAhead;
        queue_pull(g.ctx, *mb.K, R);
    }
    g.launched = true;
    ++g.launches;
}

}  // namespace

SolveGroup::~SolveGroup() {
    if (hostTables) (void)hipHostFree(hostTables);
}

bool solve_groupable(const Krylov& K, bool* mixed, bool* rb, bool* resident) {
    if (!K.run || K.run->bicg || !K.run->ev) return false;
    if (resident) *resident = K.run->resident;
    if (mixed) *mixed = K.run->mixed;
    if (rb) *rb = K.run->rb;
    return true;
}

void group_join(SolveGroup& g, Krylov& K, hipStream_t home) {
    SolveRun& R = *K.run;
    if (R.bicg || R.mixed != g.mixed || R.rb != g.rb || R.resident != g.resident || !R.ev)
        throw Error{RT_E_BAD_ARG, "group_join: the solve does not belong to this group"};
    // the group's stream waits for the solve's own queued work (the assembly,
    // the initial residual and the first state pull)
    RT_HIP(hipStreamWaitEvent(g.ctx->stream, R.ev, 0));
    if (R.needScale && !R.resident) {  // the scaled matrix its first iteration would build
        if (R.mixed) launch_scale_of<float>(g.ctx, R);
        else launch_scale_of<double>(g.ctx, R);
    }
    g.members.push_back({&K, home});
    g.dirty = true;
}

void group_remove(SolveGroup& g, Krylov& K) {
    for (size_t i = 0; i < g.members.size(); ++i)
        if (g.members[i].K == &K) {
            RT_HIP(hipStreamSynchronize(g.ctx->stream));
            g.hold.release();
            if (K.run) K.run->pending = false;
            g.members.erase(g.members.begin() + i);
            g.dirty = true;
            return;
        }
}

void group_advance(SolveGroup& g, std::vector<Krylov*>& finished, std::vector<SolveGroup::Member>& evicted) {
    bool allBack = true;
    for (auto& mb : g.members) {
        SolveRun& R = *mb.K->run;
        if (!R.pending) continue;
        hipError_t e = hipEventQuery(R.ev);
        if (e == hipErrorNotReady) {
            allBack = false;
            continue;
        }
        RT_HIP(e);
        R.pending = false;
        if (R.neFromDevice) {
            R.ne = R.hostState->misc[0];
            R.neFromDevice = false;
        }
    }
    if (!allBack) return;
    g.launched = false;
    g.hold.release();
    // members whose solve has finished leave; their streams go on after the
    // group's queued work (which reads them) has drained
    hipEvent_t drained = nullptr;
    bool gaveUp = false;
    for (size_t i = 0; i < g.members.size();) {
        SolveRun& R = *g.members[i].K->run;
        double nAct = 0, nRef = 0;
        open_components(R, nAct, nRef);
        bool fin;
        if (R.resident) {
            fin = R.resLaunched;
            if (fin && !resident_done(g.ctx, R)) {
                gaveUp = true;
                group_evict(g, i, evicted);
                continue;
            }
            if (fin) g.ctx->backoff->finished();
        } else {
            fin = (nAct == 0 && nRef == 0) || R.rounds >= 100000;
        }
        if (fin) {
            if (!drained) {
                RT_HIP(hipEventCreateWithFlags(&drained, hipEventDisableTiming));
                RT_HIP(hipEventRecord(drained, g.ctx->stream));
            }
            RT_HIP(hipStreamWaitEvent(g.members[i].home, drained, 0));
            R.done = true;
            finished.push_back(g.members[i].K);
            g.members.erase(g.members.begin() + i);
            g.dirty = true;
        } else {
            ++i;
        }
    }
    if (gaveUp) back_off(g.ctx);
    if (drained) RT_HIP(hipEventDestroy(drained));  // released once the waits are satisfied
    if (g.members.empty()) return;
    if (g.resident) {
        if (g.mixed) group_launch_resident<float>(g, evicted);
        else group_launch_resident<double>(g, evicted);
    } else if (g.mixed) {
        group_launch<float>(g);
    } else {
        group_launch<double>(g);
    }
}

void solve_finish(Krylov& K, rt_solver_perf perf[6]) {
    SolveRun& R = *K.run;
    ++R.ctx->solveCounts[R.resident ? 0 : 2];
    R.xSave.release();  // the launches that use it have ended
    for (int c = 0; c < 6; ++c) {
        rt_solver_perf& pf = perf[c];
        pf = rt_solver_perf{0, 0, 0, 0, 0, 0};
        if (R.valid[c] <= 0) continue;
        pf.initialResidual = R.host[c].initRes;
        pf.finalResidual = R.host[c].finalRes;
        pf.nIterations = R.host[c].iter;
        pf.nRefinements = R.host[c].nRefine;
        pf.converged = R.host[c].converged;
        pf.solved = 1;
    }
}

void solve_lockstep(Ctx* ctx, const SolveArgs& a, rt_solver_perf perf[6]) {
    solve_begin(ctx, a);
    while (!solve_advance(ctx, *a.kry, true)) {
    }
    solve_finish(*a.kry, perf);
}

// Workgroups of the row kernels: one per tile up to eight per CU.  A multiple of
// 8 gives each XCD a slab of the tiles; it has to be large enough that every
// tile of the two colours' slabs has a workgroup: with the next smaller multiple
// a few workgroups walked two tiles and the pass took twice as long (397 tiles
// on 392 workgroups).  Meshes that may be solved resident take no slabs: tile t
// is workgroup t's.
int grid_for(const Ctx* ctx, int32_t N) {
    const int64_t need = ((int64_t)N + BLK - 1) / BLK;
    const int64_t cap = (int64_t)ctx->numCUs * 8;
    if (N <= RES_MAX_ROWS) return (int)std::max<int64_t>(1, need % 8 == 0 ? need + 1 : need);
    return (int)std::min(((need + 7) / 8 + 1) * 8, cap);
}

}  // namespace rt
