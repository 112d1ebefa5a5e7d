// rt_device.h -- device helpers shared by the cell and Krylov kernels (gfx950).
#pragma once

#include "rt_internal.h"

namespace rt {

constexpr int BLK = 256;

// Row tiles of BLK rows.  Workgroups are dealt round-robin to the 8 XCDs
// (XCD = blockIdx.x % 8), each with its own L2.  XCD x owns the contiguous
// slab of tiles [x*S, (x+1)*S), S = ceil(T/8), and its G/8 workgroups walk
// the slab together: tile i*(G/8) + blockIdx.x/8 of the slab at step i.  The
// rows a tile gathers (bandwidth-reduced numbering keeps them within a level
// of the row) were touched moments before by the same XCD, so they are still
// in its L2.
// nRed > 0: the rows are colour-blocked (rows [0, nRed) have neighbours only
// in [nRed, N) and the other way round).  The tiles of each block are cut
// into 8 slabs and XCD x walks slab x of both blocks, alternating, so the
// other colour's rows a tile gathers are the ones the same XCD walks at the
// same time.
// Returns the tile, -2 for a step with no tile (a slab shorter than the
// others), -1 once the workgroup's share is done.
// tile_of_g: the same for workgroup b of G (a request's share of a grouped launch)
__device__ __forceinline__ int64_t tile_of_g(int64_t i, int64_t N, int64_t nRed, int G, int b) {
    const int64_t T = (N + BLK - 1) / BLK;
    if (G % 8 != 0) {
        const int64_t t = i * G + b;
        return t < T ? t : -1;
    }
    const int64_t local = i * (G / 8) + b / 8;
    const int64_t x = b % 8;
    const int64_t Ts = nRed / BLK;  // tiles [0, Ts) hold first-colour rows only
    if (nRed <= 0 || Ts == 0 || Ts >= T) {
        const int64_t S = (T + 7) / 8;
        if (local >= S) return -1;
        const int64_t t = x * S + local;
        return t < T ? t : -1;
    }
    const int64_t S1 = (Ts + 7) / 8, S2 = (T - Ts + 7) / 8;
    if (local >= S1 + S2) return -1;
    const int64_t m = S1 < S2 ? S1 : S2;
    bool first;
    int64_t k;
    if (local < 2 * m) {
        first = (local & 1) == 0;
        k = local >> 1;
    } else {
        first = S1 > S2;
        k = local - m;
    }
    if (first) {
        const int64_t t = x * S1 + k;
        return t < Ts ? t : -2;
    }
    const int64_t t = Ts + x * S2 + k;
    return t < T ? t : -2;
}
__device__ __forceinline__ int64_t tile_of(int64_t i, int64_t N, int64_t nRed = 0) {
    return tile_of_g(i, N, nRed, gridDim.x, blockIdx.x);
}

// A row kernel's workgroup: index b of G workgroups of BLK threads, this
// thread's index in it, and its LDS slots for partial sums ([RED_MAX][BLK/64]).
// Bodies take it as an argument so that a launch of several solves, and a
// resident solve, run them with the same arithmetic.
// b < G always; the row loops test it all the same, because the compiler then
// needs fewer registers for their bodies: k_rb_t<float> 74 instead of 88, and the
// x/r pass of 500000 rows takes 17.4 us instead of 18.1.
constexpr int RED_MAX = 19;
struct Blk {
    int G, b, tid;
    double* red;
};

__device__ __forceinline__ Blk blk_of_launch(double* red) {
    return Blk{(int)gridDim.x, (int)blockIdx.x, (int)threadIdx.x, red};
}

// Lane exchanges inside a wavefront, on the VALU (a shuffle through LDS has ten
// times their latency).  Level O pairs lanes l and l ^ O (l ^ 7 at O = 4, the
// mirror of a half row).
template <int O>
__device__ __forceinline__ uint32_t lane_pair(uint32_t v) {
    constexpr int ctrl = O == 8 ? 0x128 : O == 4 ? 0x141 : O == 2 ? 0x4e : 0xb1;
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, 0xf, 0xf, false);
}
// a + its pair's a on the lanes without bit O, b + its pair's b on the others
template <int O>
__device__ __forceinline__ double pair_sum(double a, double b, bool up) {
    const uint32_t al = (uint32_t)__double2loint(a), ah = (uint32_t)__double2hiint(a);
    const uint32_t bl = (uint32_t)__double2loint(b), bh = (uint32_t)__double2hiint(b);
    if constexpr (O == 32 || O == 16) {
        // swaps the lanes with bit O of a for those without of b
        auto sw = [](uint32_t x, uint32_t y) {
            if constexpr (O == 32) return __builtin_amdgcn_permlane32_swap(x, y, false, false);
            else return __builtin_amdgcn_permlane16_swap(x, y, false, false);
        };
        const auto l = sw(al, bl), h = sw(ah, bh);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    } else {
        const double keep = up ? b : a;
        const uint32_t sl = up ? al : bl, sh = up ? ah : bh;
        return keep + __hiloint2double((int)lane_pair<O>(sh), (int)lane_pair<O>(sl));
    }
}

// Sums of N per-lane values over the 64 lanes of a wavefront, halving the values
// a lane carries at each exchange: 21 exchanges for 18 values where a butterfly
// per value takes 108.  Lane l ends with the sum of value lo (valid if n > 0).
template <int N, int O>
__device__ __forceinline__ double wave_scatter(const double (&v)[N], int lane, int& lo, int& n) {
    if constexpr (O == 0) {
        return v[0];
    } else if constexpr (N == 1) {
        const double w[1] = {pair_sum<O>(v[0], v[0], lane & O)};
        return wave_scatter<1, O / 2>(w, lane, lo, n);
    } else {
        constexpr int H = (N + 1) / 2;
        const bool up = lane & O;
        double w[H];
#pragma unroll
        for (int i = 0; i < H; ++i) w[i] = pair_sum<O>(v[i], H + i < N ? v[H + i] : 0.0, up);
        lo += up ? H : 0;
        n = up ? n - H : (n < H ? n : H);
        return wave_scatter<H, O / 2>(w, lane, lo, n);
    }
}

// Grid reductions in two launches: every workgroup of the row kernel writes
// its NQ partial sums to partials[block][NQ] (plain stores, no fence), then a
// one-workgroup finalize kernel on the same stream reduces all partials in a
// fixed order (deterministic) and updates the solver state.  The kernel
// boundary makes the partials visible across the XCDs' L2s without per-block
// agent-scope release fences.
template <int NQ>
__device__ __forceinline__ void write_partials(const double (&v)[NQ], double* partials, const Blk& k) {
    static_assert(NQ <= RED_MAX, "partial-sum slots");
    constexpr int W = BLK / 64;
    int lo = 0, n = NQ;
    const double s = wave_scatter<NQ, 32>(v, k.tid & 63, lo, n);
    if (n > 0) k.red[lo * W + (k.tid >> 6)] = s;
    __syncthreads();
    if (k.tid < NQ) {
        double t = 0;
        for (int w = 0; w < W; ++w) t += k.red[k.tid * W + w];
        partials[(int64_t)k.b * NQ + k.tid] = t;
    }
}

// The finalize kernels' workgroup.  sum_partials: sums over the G blocks'
// partials into sums[NQ] (LDS), by every thread of the workgroup.  The
// partials are read as one flat array, thread t < J NQ the words t, t + J NQ,
// ... (always quantity t % NQ), so a wavefront's loads are contiguous and
// independent.  Latency bounds these kernels: against 256 threads with a row
// each (144 B apart for NQ = 18) and thread 0 updating the records, the t
// pass's finalize went from 7.0 to 3.8 us at 64 blocks (a 128 x 128 channel)
// and from 11.8 to 8.3 us at 1280 (a 160^3 box).  The order of the sums
// depends on G alone.
constexpr int FBLK = 1024;
constexpr int FIN_LDS = FBLK + 9 * RED_MAX;
// NT: threads of the workgroup that runs it (each takes FBLK / NT of the sums)
template <int NQ, int NT = FBLK>
__device__ __forceinline__ void sum_partials(const double* partials, int G, double* lds, double*& sums) {
    constexpr int J = FBLK / NQ, J2 = 8, S = J * NQ;
    double* s2 = lds + FBLK;
    sums = s2 + J2 * NQ;
    const int total = G * NQ;
#pragma unroll
    for (int t = threadIdx.x; t < FBLK; t += NT) {
        if (t >= S) break;
        double acc = 0;
        int i = t;
        for (; i + 7 * S < total; i += 8 * S) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = partials[i + u * S];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += v[u];
        }
        for (; i < total; i += S) acc += partials[i];
        lds[t] = acc;
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (t < J2 * NQ) {
        const int q = t % NQ;
        double acc = 0;
#pragma unroll
        for (int j = t / NQ; j < J; j += J2) acc += lds[j * NQ + q];
        s2[t] = acc;
    }
    __syncthreads();
    if (t < NQ) {
        double acc = 0;
#pragma unroll
        for (int j = 0; j < J2; ++j) acc += s2[j * NQ + t];
        sums[t] = acc;
    }
    __syncthreads();
}

// A component record in registers, field by field (copied as a whole the
// compiler keeps it in memory).
struct Comp {
    double rho, rhoOld, alpha, omega, beta, normFactor, initRes, finalRes, innerTarget;
    int32_t iter, active, converged, solved, exitAtS, needRefine, nRefine, innerIter, foldE;
    __device__ __forceinline__ void load(const CompState& c) {
        rho = c.rho, rhoOld = c.rhoOld, alpha = c.alpha, omega = c.omega, beta = c.beta;
        normFactor = c.normFactor, initRes = c.initRes, finalRes = c.finalRes, innerTarget = c.innerTarget;
        iter = c.iter, active = c.active, converged = c.converged, solved = c.solved, exitAtS = c.exitAtS;
        needRefine = c.needRefine, nRefine = c.nRefine, innerIter = c.innerIter, foldE = c.foldE;
    }
    __device__ __forceinline__ void store(CompState& c) const {
        c.rho = rho, c.rhoOld = rhoOld, c.alpha = alpha, c.omega = omega, c.beta = beta;
        c.normFactor = normFactor, c.initRes = initRes, c.finalRes = finalRes, c.innerTarget = innerTarget;
        c.iter = iter, c.active = active, c.converged = converged, c.solved = solved, c.exitAtS = exitAtS;
        c.needRefine = needRefine, c.nRefine = nRefine, c.innerIter = innerIter, c.foldE = foldE;
    }
};

// interleaved [N][6] rows: three 2-wide vector loads/stores per row
template <class T> struct Vec2;
template <> struct Vec2<float> { typedef float2 type; };
template <> struct Vec2<double> { typedef double2 type; };

template <class T>
__device__ __forceinline__ void ld6(const T* p, T* v) {
    typedef typename Vec2<T>::type V2;
    const V2* q = reinterpret_cast<const V2*>(p);
    const V2 a = q[0], b = q[1], c = q[2];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y; v[4] = c.x; v[5] = c.y;
}
template <class T>
__device__ __forceinline__ void st6(T* p, const T* v) {
    typedef typename Vec2<T>::type V2;
    V2* q = reinterpret_cast<V2*>(p);
    V2 a, b, c;
    a.x = v[0]; a.y = v[1]; b.x = v[2]; b.y = v[3]; c.x = v[4]; c.y = v[5];
    q[0] = a; q[1] = b; q[2] = c;
}

// wedge patch value of a symmTensor ([OF9] wedgeFvPatchField::evaluate,
// transform(faceT, theta_P)): T theta_P T^T, T (row-major) the patch's faceT;
// the same operations as the oracle's
__device__ __forceinline__ void wedge_value(const double* __restrict__ T, const double th[6], double out[6]) {
    double A[3][3], M[3][3];
    A[0][0] = th[0]; A[0][1] = A[1][0] = th[1]; A[0][2] = A[2][0] = th[2];
    A[1][1] = th[3]; A[1][2] = A[2][1] = th[4]; A[2][2] = th[5];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) M[i][k] = T[3 * i] * A[0][k] + T[3 * i + 1] * A[1][k] + T[3 * i + 2] * A[2][k];
    constexpr int I6[6] = {0, 0, 0, 1, 1, 2}, J6[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const int i = I6[q], l = J6[q];
        out[q] = M[i][0] * T[3 * l] + M[i][1] * T[3 * l + 1] + M[i][2] * T[3 * l + 2];
    }
}

// symmetryPlane / symmetry patch value of a symmTensor ([OF9]
// basicSymmetryFvPatchField::evaluate): (theta_P + T theta_P T^T)/2 with
// T = I - 2 n n, n = Sf/|Sf|; the same operations as the oracle's
__device__ __forceinline__ void symmetry_value(const double sf[3], const double th[6], double out[6]) {
    const double mag = sqrt(sf[0] * sf[0] + sf[1] * sf[1] + sf[2] * sf[2]);
    const double n[3] = {sf[0] / mag, sf[1] / mag, sf[2] / mag};
    double T[3][3], A[3][3], M[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) T[i][j] = (i == j ? 1.0 : 0.0) - 2.0 * n[i] * n[j];
    A[0][0] = th[0]; A[0][1] = A[1][0] = th[1]; A[0][2] = A[2][0] = th[2];
    A[1][1] = th[3]; A[1][2] = A[2][1] = th[4]; A[2][2] = th[5];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) M[i][k] = T[i][0] * A[0][k] + T[i][1] * A[1][k] + T[i][2] * A[2][k];
    constexpr int I6[6] = {0, 0, 0, 1, 1, 2}, J6[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const int i = I6[q], l = J6[q];
        const double r = M[i][0] * T[l][0] + M[i][1] * T[l][1] + M[i][2] * T[l][2];
        out[q] = (th[q] + r) / 2.0;
    }
}

// ------------------------------------------------- Krylov control (OpenFOAM)
// SolverPerformance::checkConvergence: final < tolerance, or relTol > 0 and
// final < relTol * initial
__device__ __forceinline__ bool conv_outer(const Comp& c, const KryCtl& k, double res) {
    return res < k.tol || (k.relTol > 0 && res < k.relTol * c.initRes);
}
__device__ __forceinline__ bool conv_inner(const Comp& c, const KryCtl& k, double res) {
    return k.mixed ? res < c.innerTarget : conv_outer(c, k, res);
}

// begin an inner Krylov solve on a component whose r, r0 were just set
__device__ __forceinline__ void start_inner(Comp& c, const KryCtl& k, double rr) {
    c.innerIter = 0;
    c.rho = rr;
    c.exitAtS = 0;
    if (k.mixed) c.innerTarget = fmax(k.innerRelTol * c.finalRes, 0.3 * k.tol);
    if (fabs(rr) < 1e-300) {  // singular: nothing to iterate on
        c.active = 0;
        c.converged = conv_outer(c, k, c.finalRes);
        return;
    }
    c.active = 1;
}

// after the initial residual: normalisation factor, initial residual, start
__device__ __forceinline__ void finish_initial(Comp& cs, const KryCtl& k, double absR, double rr,
                                               double nrm) {
    cs.normFactor = nrm + 1e-20;
    cs.initRes = absR / cs.normFactor;
    cs.finalRes = cs.initRes;
    cs.iter = 0;
    cs.nRefine = 0;
    cs.solved = 1;
    cs.converged = 0;
    cs.needRefine = 0;
    cs.foldE = 0;
    if (k.minIter > 0 || !conv_outer(cs, k, cs.initRes)) {
        if (k.rb) {
            // red-black: a first sweep eliminates the first colour (x there
            // from the second colour's x) and leaves the Schur residual
            cs.active = 0;
            cs.needRefine = 1;
        } else {
            start_inner(cs, k, rr);
        }
    } else {
        cs.active = 0;
        cs.converged = 1;
    }
}

}  // namespace rt
