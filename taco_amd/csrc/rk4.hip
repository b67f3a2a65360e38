// rk4.hip — RK4 on vec(rho) with prebuilt generators, and its reverse.
#include <type_traits>

#include "rk4.hpp"

#pragma clang fp contract(off)

namespace taco_engine {

// ---------------------------------------------------------------------------
// RK4 on vec(rho) with prebuilt generators (rk4_dense.cpp:133-160, 246-320),
// one workgroup, D <= 1024.  Matvecs sum over j in order per row.
// ---------------------------------------------------------------------------
// Matrices are read as L[r + c * ld]: ld = D in global memory, D + 1 when
// staged in LDS (the padded column stride spreads the column reads of L^H
// products over the banks).  Everything down to the kernels is inlined and
// each code path sees either LDS or global matrices, so the compiler knows
// the address space of every access (LDS reads, not flat ones).  Every product sums over c in order per row, so
// staged and unstaged runs, and every instantiation below, give identical
// values.  DT > 0 fixes D at compile time (the row loop is unrolled, so its
// loads issue together); DT = 0 is the general case.
// In the general case (DT = 0, D a runtime value) the columns are taken in
// blocks of kMvBlk whose loads are issued before the block's products, so a
// thread keeps kMvBlk generator loads in flight (the sum order is unchanged).
constexpr int kMvBlk = 16;

template <int DT>
__device__ __forceinline__ void matvec_rows(const double2* __restrict__ L, int ld, const double2* x, double2* y,
                                            int D) {
    const int n = DT ? DT : D;
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
        double2 s = make_double2(0.0, 0.0);
        if constexpr (DT == 0) {
            int c = 0;
            for (; c + kMvBlk <= n; c += kMvBlk) {
                double2 v[kMvBlk];
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) v[j] = L[r + static_cast<long>(c + j) * ld];
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) s = cadd(s, cmul(v[j], x[c + j]));
            }
            for (; c < n; ++c) s = cadd(s, cmul(L[r + static_cast<long>(c) * ld], x[c]));
        } else {
#pragma unroll
            for (int c = 0; c < DT; ++c) s = cadd(s, cmul(L[r + static_cast<long>(c) * ld], x[c]));
        }
        y[r] = s;
    }
}

// y = 0.5 (L0 + L1) x, the midpoint generator formed per element.
template <int DT>
__device__ __forceinline__ void matvec_half(const double2* __restrict__ L0, const double2* __restrict__ L1, int ld,
                                            const double2* x, double2* y, int D) {
    const int n = DT ? DT : D;
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
        double2 s = make_double2(0.0, 0.0);
        if constexpr (DT == 0) {
            int c = 0;
            for (; c + kMvBlk <= n; c += kMvBlk) {
                double2 v0[kMvBlk], v1[kMvBlk];
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) {
                    const long e = r + static_cast<long>(c + j) * ld;
                    v0[j] = L0[e];
                    v1[j] = L1[e];
                }
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) s = cadd(s, cmul(cscale(cadd(v0[j], v1[j]), 0.5), x[c + j]));
            }
            for (; c < n; ++c) {
                const long e = r + static_cast<long>(c) * ld;
                s = cadd(s, cmul(cscale(cadd(L0[e], L1[e]), 0.5), x[c]));
            }
        } else {
#pragma unroll
            for (int c = 0; c < DT; ++c) {
                const long e = r + static_cast<long>(c) * ld;
                const double2 h = cscale(cadd(L0[e], L1[e]), 0.5);
                s = cadd(s, cmul(h, x[c]));
            }
        }
        y[r] = s;
    }
}

// One RK4 step x <- x + dt/6 (k1 + 2 k2 + 2 k3 + k4) by the whole workgroup
// (rk4_dense.cpp:133-160); Lh null: midpoint 0.5 (L0 + L1) per element.
// L0 and L1 have column stride ld; Lh (global) has D.
template <int DT>
__device__ __forceinline__ void rk4_step(const double2* L0, const double2* L1, int ld, const double2* Lh, double2* x,
                                         double2* k1, double2* k2, double2* k3, double2* k4, double2* tmp, int D,
                                         double dt, double2* stash = nullptr) {
    // stash (optional): receives the stage points u1, u2, u3 (3 x D)
    const double hdt = 0.5 * dt;
    const double s6 = dt / 6.0;
    matvec_rows<DT>(L0, ld, x, k1, D);
    __syncthreads();
    for (int e = threadIdx.x; e < D; e += blockDim.x) {
        tmp[e] = cadd(x[e], cscale(k1[e], hdt));
        if (stash) stash[e] = tmp[e];
    }
    __syncthreads();
    if (Lh) matvec_rows<DT>(Lh, D, tmp, k2, D); else matvec_half<DT>(L0, L1, ld, tmp, k2, D);
    __syncthreads();
    for (int e = threadIdx.x; e < D; e += blockDim.x) {
        tmp[e] = cadd(x[e], cscale(k2[e], hdt));
        if (stash) stash[D + e] = tmp[e];
    }
    __syncthreads();
    if (Lh) matvec_rows<DT>(Lh, D, tmp, k3, D); else matvec_half<DT>(L0, L1, ld, tmp, k3, D);
    __syncthreads();
    for (int e = threadIdx.x; e < D; e += blockDim.x) {
        tmp[e] = cadd(x[e], cscale(k3[e], dt));
        if (stash) stash[2 * D + e] = tmp[e];
    }
    __syncthreads();
    matvec_rows<DT>(L1, ld, tmp, k4, D);
    __syncthreads();
    for (int e = threadIdx.x; e < D; e += blockDim.x) {
        const double2 acc = cadd(cadd(cadd(k1[e], cscale(k2[e], 2.0)), cscale(k3[e], 2.0)), k4[e]);
        x[e] = cadd(x[e], cscale(acc, s6));
    }
    __syncthreads();
}

// Copies generators L_first .. L_first+count-1 into LDS with column stride D + 1.
__device__ __forceinline__ void stage_mats(double2* dst, const double2* Ls, long first, int count, int D) {
    const long D2 = static_cast<long>(D) * D;
    const int ld = D + 1;
    const double2* src = Ls + first * D2;
    for (long e = threadIdx.x; e < count * D2; e += blockDim.x) {
        const long m = e / D2, w = e % D2;
        const int r = static_cast<int>(w % D), c = static_cast<int>(w / D);
        dst[m * D * ld + r + static_cast<long>(c) * ld] = src[e];
    }
}

// One system's RK4 run by the whole workgroup; x, k1..k4, tmp in LDS, then
// (nstage >= 2, no Lh) the generators staged nstage at a time.  Reads the
// initial vector from r_in and writes the final one to r_out.
template <int DT>
__device__ __forceinline__ void rk4_body(double2* sh, int nstage, const double2* Ls, const double2* Lh, long steps, int D,
                         const double2* r_in, double2* r_out, double dt, long every, double2* samples,
                         long* nsamples) {
    double2* x = sh;
    double2* k1 = x + D;
    double2* k2 = k1 + D;
    double2* k3 = k2 + D;
    double2* k4 = k3 + D;
    double2* tmp = k4 + D;
    double2* M = tmp + D;
    for (int e = threadIdx.x; e < D; e += blockDim.x) x[e] = r_in[e];
    __syncthreads();
    const long D2 = static_cast<long>(D) * D;
    const int ld = D + 1;
    long ns = 0;
    if (nstage >= 2 && !Lh) {
        for (long s = 0; s < steps; s += nstage - 1) {
            const int cnt = static_cast<int>(min(static_cast<long>(nstage), steps - s + 1));
            stage_mats(M, Ls, s, cnt, D);
            __syncthreads();
            for (int q = 0; q + 1 < cnt; ++q) {
                const long st = s + q;
                if (samples && st % every == 0) {
                    for (int e = threadIdx.x; e < D; e += blockDim.x) samples[ns * D + e] = x[e];
                    ++ns;
                }
                rk4_step<DT>(M + static_cast<long>(q) * D * ld, M + static_cast<long>(q + 1) * D * ld, ld, nullptr,
                             x, k1, k2, k3, k4, tmp, D, dt);
            }
        }
    } else {
        for (long st = 0; st < steps; ++st) {
            if (samples && st % every == 0) {
                for (int e = threadIdx.x; e < D; e += blockDim.x) samples[ns * D + e] = x[e];
                ++ns;
            }
            rk4_step<DT>(Ls + st * D2, Ls + (st + 1) * D2, D, Lh ? Lh + st * D2 : nullptr, x, k1, k2, k3, k4, tmp,
                         D, dt);
        }
    }
    if (samples) {
        for (int e = threadIdx.x; e < D; e += blockDim.x) samples[ns * D + e] = x[e];
        ++ns;
    }
    for (int e = threadIdx.x; e < D; e += blockDim.x) r_out[e] = x[e];
    if (threadIdx.x == 0 && nsamples) *nsamples = ns;
}

// Dispatch on D = N^2 for the sizes of N = 2..8 (unrolled rows), else general.
#define TACO_RK4_DISPATCH(D, CALL)      \
    switch (D) {                        \
        case 4: CALL(4); break;         \
        case 9: CALL(9); break;         \
        case 16: CALL(16); break;       \
        case 25: CALL(25); break;       \
        case 36: CALL(36); break;       \
        case 49: CALL(49); break;       \
        case 64: CALL(64); break;       \
        default: CALL(0); break;        \
    }

#include "rk4_rows.hpp"

// One system on the row-group path (D = N^2, N = 2..8), 64 W threads.
template <int DT>
__global__ __launch_bounds__(64 * RowGroup<DT>::W) void k_rk4_rows(const double2* Ls, long steps, double2* r,
                                                                   double dt, long every, double2* samples,
                                                                   long* nsamples) {
    extern __shared__ double2 sh[];
    rk4_rows<DT, false>(sh, Ls, 0, steps, r, r, dt, every, samples, nsamples, nullptr);
}

// Calls f(std::integral_constant<int, D>) for a D with a row-group path.
template <class F>
__host__ __device__ inline bool rows_dispatch(int D, F&& f) {
    switch (D) {
        case 4: f(std::integral_constant<int, 4>{}); return true;
        case 9: f(std::integral_constant<int, 9>{}); return true;
        case 16: f(std::integral_constant<int, 16>{}); return true;
        case 25: f(std::integral_constant<int, 25>{}); return true;
        case 36: f(std::integral_constant<int, 36>{}); return true;
        case 49: f(std::integral_constant<int, 49>{}); return true;
        case 64: f(std::integral_constant<int, 64>{}); return true;
        default: return false;
    }
}

__global__ __launch_bounds__(kRkBlock) void k_rk4(const double2* Ls, const double2* Lh, long steps, int D, double2* r,
                                                double dt, long every, double2* samples, long* nsamples, int nstage) {
    extern __shared__ double2 sh[];
#define TACO_RK4_CALL(DT) rk4_body<DT>(sh, nstage, Ls, Lh, steps, D, r, r, dt, every, samples, nsamples)
    TACO_RK4_DISPATCH(D, TACO_RK4_CALL)
#undef TACO_RK4_CALL
}

__global__ __launch_bounds__(kRkBlockMax) void k_rk4_batch(const Rk4Sys* sys) {
    extern __shared__ double2 sh[];
    const Rk4Sys S = sys[blockIdx.x];
    if (S.q) return;  // chunked
    // sizes with a row-group path have no separate midpoint series here
    if (!rows_dispatch(S.D, [&](auto dc) {
            constexpr int DT = decltype(dc)::value;
            rk4_rows<DT, false>(sh, S.Ls, 0, S.steps, S.r0, S.r, S.dt, 1, S.samples, nullptr, nullptr);
        }))
        rk4_body<0>(sh, S.nstage, S.Ls, S.Lh, S.steps, S.D, S.r0, S.r, S.dt, 1, S.samples, nullptr);
}

// y = L^H x (column r of L conjugated, column stride ld), summed over c in order.
// (General D: column blocks of kMvBlk loads issued ahead, as in matvec_rows.)
template <int DT>
__device__ __forceinline__ void matvec_h(const double2* __restrict__ L, int ld, const double2* x, double2* y, int D) {
    const int n = DT ? DT : D;
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
        double2 s = make_double2(0.0, 0.0);
        const double2* col = L + static_cast<long>(r) * ld;
        if constexpr (DT == 0) {
            int c = 0;
            for (; c + kMvBlk <= n; c += kMvBlk) {
                double2 v[kMvBlk];
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) v[j] = col[c + j];
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) s = cadd(s, cmul(cconj(v[j]), x[c + j]));
            }
            for (; c < n; ++c) s = cadd(s, cmul(cconj(col[c]), x[c]));
        } else {
#pragma unroll
            for (int c = 0; c < DT; ++c) s = cadd(s, cmul(cconj(col[c]), x[c]));
        }
        y[r] = s;
    }
}

// y = (0.5 (L0 + L1))^H x.
template <int DT>
__device__ __forceinline__ void matvec_h_half(const double2* __restrict__ L0, const double2* __restrict__ L1, int ld,
                                              const double2* x, double2* y, int D) {
    const int n = DT ? DT : D;
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
        double2 s = make_double2(0.0, 0.0);
        const long o = static_cast<long>(r) * ld;
        if constexpr (DT == 0) {
            int c = 0;
            for (; c + kMvBlk <= n; c += kMvBlk) {
                double2 v0[kMvBlk], v1[kMvBlk];
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) {
                    v0[j] = L0[o + c + j];
                    v1[j] = L1[o + c + j];
                }
#pragma unroll
                for (int j = 0; j < kMvBlk; ++j) s = cadd(s, cmul(cconj(cscale(cadd(v0[j], v1[j]), 0.5)), x[c + j]));
            }
            for (; c < n; ++c) s = cadd(s, cmul(cconj(cscale(cadd(L0[o + c], L1[o + c]), 0.5)), x[c]));
        } else {
#pragma unroll
            for (int c = 0; c < DT; ++c)
                s = cadd(s, cmul(cconj(cscale(cadd(L0[o + c], L1[o + c]), 0.5)), x[c]));
        }
        y[r] = s;
    }
}

// ---------------------------------------------------------------------------
// RK4 adjoint.  Forward step n (rk4_step): k1 = L0 r, u1 = r + h k1,
// k2 = Lh u1, u2 = r + h k2, k3 = Lh u2, u3 = r + dt k3, k4 = L1 u3,
// r' = r + s (k1 + 2 k2 + 2 k3 + k4), h = dt/2, s = dt/6, Lh = (L0 + L1)/2.
// Two launches.  k_rk4_recompute: one workgroup per checkpoint segment (K
// steps) recomputes, from the checkpoint ck[q] = r_{qK} and with the forward
// step's arithmetic, the states r_n and stage points u1..u3 of its
// segment; segments are independent, so all run at once.  k_rk4_adjoint:
// one workgroup walks n = steps-1 .. 0, mapping lam_{n+1} to
// lam_n = M_n^H lam_{n+1} + gbar_n and forming the cotangents of L_n and
// L_{n+1}.  LDS: vectors of D, then (nstage >= 2) a window of generators
// staged with column stride D + 1.  Lbar(t) collects the L1 part of step t-1
// and the L0 part of step t: the latter is carried in registers
// (D^2 <= 16 x 256) and each Lbar(t) stored once.  Larger D take the wide
// runs below.
// ---------------------------------------------------------------------------

// Makes generators L_a..L_b resident in the LDS window M (column stride
// D + 1), restaging the window [first, last] when they are not.
struct GenWindow {
    long lo = 0, hi = -1;
    __device__ __forceinline__ void need(double2* M, const double2* Ls, long a, long b, long first, long last, int D) {
        if (a >= lo && b <= hi) return;
        __syncthreads();
        lo = first;
        hi = last;
        stage_mats(M, Ls, lo, static_cast<int>(hi - lo + 1), D);
        __syncthreads();
    }
};

__device__ __forceinline__ void rk4_recompute_body(double2* sh, const Rk4AdjArgs& A, long sg) {
    const int D = A.D;
    double2* x = sh;
    double2* k1 = x + D;
    double2* k2 = k1 + D;
    double2* k3 = k2 + D;
    double2* k4 = k3 + D;
    double2* tmp = k4 + D;
    double2* M = tmp + D;
    const int ld = D + 1;
    GenWindow w;
    const long s0 = sg * A.K, s1 = min(s0 + A.K, A.steps);
    for (int e = threadIdx.x; e < D; e += blockDim.x) x[e] = A.ck[sg * D + e];
    __syncthreads();
    for (long n = s0; n < s1; ++n) {
        double2* row = A.seg + n * 4 * D;
        for (int e = threadIdx.x; e < D; e += blockDim.x) row[e] = x[e];
        w.need(M, A.Ls, n, n + 1, n, min(n + A.nstage - 1, s1), D);
        rk4_step<0>(M + (n - w.lo) * D * ld, M + (n + 1 - w.lo) * D * ld, ld, nullptr, x, k1, k2, k3, k4, tmp, D, A.dt,
                    row + D);
    }
}

// Row-group recompute (rk4_rows with the stage points stashed) for the sizes
// that have one: the plain forward step (a chunked forward's states differ from
// it by rounding).  One workgroup per checkpoint segment.
template <int DT>
__global__ __launch_bounds__(64 * RowGroup<DT>::W) void k_rk4_recompute_rows(Rk4AdjArgs A) {
    extern __shared__ double2 sh[];
    const long sg = blockIdx.x;
    const long s0 = sg * A.K, s1 = min(s0 + A.K, A.steps);
    rk4_rows<DT, true>(sh, A.Ls, s0, s1, A.ck + sg * DT, nullptr, A.dt, 1, nullptr, nullptr, A.seg);
}

__global__ __launch_bounds__(kRkBlock) void k_rk4_recompute(Rk4AdjArgs A) {
    extern __shared__ double2 sh[];
    rk4_recompute_body(sh, A, blockIdx.x);
}

template <int DT>
__device__ __forceinline__ void rk4_adjoint_body(double2* sh, const Rk4AdjArgs& A) {
    const int D = A.D;
    double2* x = sh;          // r_n
    double2* k3 = x + D;      // cotangent of k3
    double2* k4 = k3 + D;     // cotangent of k4
    double2* tmp = k4 + D;
    double2* lam = tmp + D;   // cotangent of r_{n+1}, then of r_n
    double2* u1 = lam + D;
    double2* u2 = u1 + D;
    double2* u3 = u2 + D;
    double2* kb1 = u3 + D;    // cotangents of k1, k2
    double2* kb2 = kb1 + D;
    double2* rb = kb2 + D;    // cotangent of r_n being accumulated
    double2* M = rb + D;      // staged generators
    const long D2 = static_cast<long>(D) * D;
    const int ld = D + 1;
    double2 Lc[kRkCarry];     // L0 part of the step after the current one
#pragma unroll
    for (int q = 0; q < kRkCarry; ++q) Lc[q] = make_double2(0.0, 0.0);
    GenWindow w;
    const double h = 0.5 * A.dt, s6 = A.dt / 6.0;
    for (int e = threadIdx.x; e < D; e += blockDim.x) lam[e] = A.gbar[A.steps * D + e];
    __syncthreads();
    for (long n = A.steps - 1; n >= 0; --n) {
        w.need(M, A.Ls, n, n + 1, max(0L, n + 2 - A.nstage), n + 1, D);
        const double2* L0 = M + (n - w.lo) * D * ld;
        const double2* L1 = L0 + D * ld;
        const double2* row = A.seg + n * 4 * D;
        for (int e = threadIdx.x; e < D; e += blockDim.x) {
            x[e] = row[e];
            u1[e] = row[D + e];
            u2[e] = row[2 * D + e];
            u3[e] = row[3 * D + e];
            k4[e] = cscale(lam[e], s6);                                                    // kb4
        }
        __syncthreads();
        // reverse: r' = r + s (k1 + 2 k2 + 2 k3 + k4)
        matvec_h<DT>(L1, ld, k4, tmp, D);  // ub3
        __syncthreads();
        for (int e = threadIdx.x; e < D; e += blockDim.x) {
            k3[e] = cadd(cscale(lam[e], 2.0 * s6), cscale(tmp[e], A.dt));                  // kb3
            rb[e] = cadd(lam[e], tmp[e]);
        }
        __syncthreads();
        matvec_h_half<DT>(L0, L1, ld, k3, tmp, D);  // ub2
        __syncthreads();
        for (int e = threadIdx.x; e < D; e += blockDim.x) {
            kb2[e] = cadd(cscale(lam[e], 2.0 * s6), cscale(tmp[e], h));
            rb[e] = cadd(rb[e], tmp[e]);
        }
        __syncthreads();
        matvec_h_half<DT>(L0, L1, ld, kb2, tmp, D);  // ub1
        __syncthreads();
        for (int e = threadIdx.x; e < D; e += blockDim.x) {
            kb1[e] = cadd(cscale(lam[e], s6), cscale(tmp[e], h));
            rb[e] = cadd(rb[e], tmp[e]);
        }
        __syncthreads();
        matvec_h<DT>(L0, ld, kb1, tmp, D);
        __syncthreads();
        // generator cotangents: Lbar_h = kb3 u2^H + kb2 u1^H, split half/half
        double2* Lb1 = A.Lbar + (n + 1) * D2;
#pragma unroll
        for (int q = 0; q < kRkCarry; ++q) {
            const long e = threadIdx.x + static_cast<long>(q) * blockDim.x;
            if (e < D2) {
                const int r = static_cast<int>(e % D), c = static_cast<int>(e / D);
                const double2 lh = cadd(cmul(k3[r], cconj(u2[c])), cmul(kb2[r], cconj(u1[c])));
                Lb1[e] = cadd(Lc[q], cadd(cmul(k4[r], cconj(u3[c])), cscale(lh, 0.5)));
                Lc[q] = cadd(cmul(kb1[r], cconj(x[c])), cscale(lh, 0.5));
            }
        }
        for (int e = threadIdx.x; e < D; e += blockDim.x) lam[e] = cadd(cadd(rb[e], tmp[e]), A.gbar[n * D + e]);
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kRkCarry; ++q) {
        const long e = threadIdx.x + static_cast<long>(q) * blockDim.x;
        if (e < D2) A.Lbar[e] = Lc[q];
    }
    for (int e = threadIdx.x; e < D; e += blockDim.x) A.r0bar[e] = lam[e];
}

// Row-group reverse walk for D <= 16 (one wave of 64 threads).
template <int DT>
__global__ __launch_bounds__(64) void k_rk4_adjoint_rows(Rk4AdjArgs A) {
    extern __shared__ double2 sh[];
    const double2* lam = A.gbar + A.steps * DT;
    if (A.vec)
        rk4_rows_adjoint<DT, WALK_VEC>(sh, A, 0, A.steps, lam, A.r0bar);
    else
        rk4_rows_adjoint<DT, WALK_LBAR>(sh, A, 0, A.steps, lam, A.r0bar);
}

__global__ __launch_bounds__(kRkBlock) void k_rk4_adjoint(Rk4AdjArgs A) {
    extern __shared__ double2 sh[];
    switch (A.D) {  // 4, 9 and 16 have the row-group walk
        case 25: rk4_adjoint_body<25>(sh, A); break;
        case 36: rk4_adjoint_body<36>(sh, A); break;
        case 49: rk4_adjoint_body<49>(sh, A); break;
        case 64: rk4_adjoint_body<64>(sh, A); break;
        default: rk4_adjoint_body<0>(sh, A); break;
    }
}

// Lbar(t), t = 0..steps, from a walk's vectors: the L0 part of step t
// (kb1 x^H + (kb3 u2^H + kb2 u1^H)/2) added to zero, then the L1 part of
// step t-1 (kb4 u3^H + (kb3 u2^H + kb2 u1^H)/2): the sums a walk that forms
// them in place takes, in its order.  Grid: (element blocks of D^2, steps + 1[, tapes]).
__device__ __forceinline__ void rk4_lbar_body(const Rk4AdjArgs& A) {
    const int D = A.D;
    const long D2 = static_cast<long>(D) * D;
    const long e = static_cast<long>(blockIdx.x) * kRkBlock + threadIdx.x;
    const long t = blockIdx.y;
    if (e >= D2 || t > A.steps) return;
    const int r = static_cast<int>(e % D), c = static_cast<int>(e / D);
    double2 acc = make_double2(0.0, 0.0);
    if (t < A.steps) {
        const double2* v = A.vec + t * 4 * D;
        const double2* sg = A.seg + t * 4 * D;
        const double2 lh = cadd(cmul(v[2 * D + r], cconj(sg[2 * D + c])), cmul(v[D + r], cconj(sg[D + c])));
        acc = cadd(acc, cadd(cmul(v[r], cconj(sg[c])), cscale(lh, 0.5)));
    }
    if (t >= 1) {
        const double2* v = A.vec + (t - 1) * 4 * D;
        const double2* sg = A.seg + (t - 1) * 4 * D;
        const double2 lh = cadd(cmul(v[2 * D + r], cconj(sg[2 * D + c])), cmul(v[D + r], cconj(sg[D + c])));
        acc = cadd(acc, cadd(cmul(v[3 * D + r], cconj(sg[3 * D + c])), cscale(lh, 0.5)));
    }
    A.Lbar[t * D2 + e] = acc;
}

__global__ __launch_bounds__(kRkBlock) void k_rk4_lbar(Rk4AdjArgs A) { rk4_lbar_body(A); }

__global__ __launch_bounds__(kRkBlock) void k_rk4_lbar_multi(const Rk4AdjArgs* As) {
    const Rk4AdjArgs A = As[blockIdx.z];
    rk4_lbar_body(A);
}

// Many tapes of one D, steps and K in one launch: the recompute with
// blockIdx.y choosing the tape, the walk with one workgroup per tape; each
// workgroup runs the single-tape body on its own arguments.
template <int DT>
__global__ __launch_bounds__(64 * RowGroup<DT>::W) void k_rk4_recompute_rows_multi(const Rk4AdjArgs* As) {
    extern __shared__ double2 sh[];
    const Rk4AdjArgs A = As[blockIdx.y];
    const long sg = blockIdx.x;
    const long s0 = sg * A.K, s1 = min(s0 + A.K, A.steps);
    rk4_rows<DT, true>(sh, A.Ls, s0, s1, A.ck + sg * DT, nullptr, A.dt, 1, nullptr, nullptr, A.seg);
}

__global__ __launch_bounds__(kRkBlock) void k_rk4_recompute_multi(const Rk4AdjArgs* As) {
    extern __shared__ double2 sh[];
    const Rk4AdjArgs A = As[blockIdx.y];
    rk4_recompute_body(sh, A, blockIdx.x);
}

template <int DT>
__global__ __launch_bounds__(64) void k_rk4_adjoint_rows_multi(const Rk4AdjArgs* As) {
    extern __shared__ double2 sh[];
    const Rk4AdjArgs A = As[blockIdx.x];
    const double2* lam = A.gbar + A.steps * DT;
    if (A.vec)
        rk4_rows_adjoint<DT, WALK_VEC>(sh, A, 0, A.steps, lam, A.r0bar);
    else
        rk4_rows_adjoint<DT, WALK_LBAR>(sh, A, 0, A.steps, lam, A.r0bar);
}

__global__ __launch_bounds__(kRkBlock) void k_rk4_adjoint_multi(const Rk4AdjArgs* As) {
    extern __shared__ double2 sh[];
    const Rk4AdjArgs A = As[blockIdx.x];
    switch (A.D) {  // 4, 9 and 16 have the row-group walk
        case 25: rk4_adjoint_body<25>(sh, A); break;
        case 36: rk4_adjoint_body<36>(sh, A); break;
        case 49: rk4_adjoint_body<49>(sh, A); break;
        case 64: rk4_adjoint_body<64>(sh, A); break;
        default: rk4_adjoint_body<0>(sh, A); break;
    }
}

// ---------------------------------------------------------------------------
// Chunked runs.  One RK4 step is linear, r_{n+1} = (I + E_n) r_n, so the
// recursion over many steps splits in time:
//   1. every chunk of kRkChunk steps forms Q_c = prod (I + E_n) - I, all
//      chunks at once (four D x D products a step);
//   2. one workgroup carries r over the chunks, r <- r + Q_c r, one product
//      per chunk where the plain run has four per step; chunks in which r may
//      decay (chunk_mild) take the plain steps here instead;
//   3. every chunk runs its steps from its first state with the plain step
//      (rk4_rows), all chunks at once.
// The dependent chain shrinks from 4 steps products to 4 kRkChunk (twice) and
// steps / kRkChunk.  E_n and Q_c are kept without the identity, so a chunk
// rounds r once where kRkChunk plain steps round it kRkChunk times.
// The reverse walk, affine in lam, splits alike: each chunk's walk from lam = 0
// gives its constant part, the carry is lam <- lam + Q_c^H lam + b_c, and every
// chunk's walk then runs from its true lam.
// Measured, forward: D = 16, 4000 steps 2.7 -> 0.12 ms (products 43 us, 250
// carries 59 us, states 15 us); D = 4, 2000 steps 1.02 -> 0.05 ms; D = 36,
// 800 steps 0.45 ms.  All three are latency: chunks of 16 keep the products
// at one workgroup per CU for 4000 steps and the carry at 0.25 us a chunk.
// ---------------------------------------------------------------------------
template <int DT>
struct Chunk {
    static constexpr int NT = DT < 16 ? 64 : 256;        // threads of step 1
    static constexpr int CPB = DT == 4 ? 4 : 1;          // chunks of a workgroup
    static constexpr int LPC = NT / CPB;                 // threads of a chunk
    static constexpr int EPT = (DT * DT + LPC - 1) / LPC;  // entries of a thread
    static constexpr int D2 = DT * DT;
};

// The kernels' arguments: arr[i], one block per system or tape, or the single
// `one` (arr null), by scalar loads.  A pointer that comes from memory is taken to
// be of any address space, and its loads wait with the LDS's (a step 25 % longer
// at D = 16): in_global says that it is global.
template <class T>
__device__ __forceinline__ void in_global(T*& p) {
    auto g = (__attribute__((address_space(1))) T*)p;
    asm("" : "+s"(g));  // the plain cast there and back is folded away
    p = (T*)g;
}
template <class S>
__device__ __forceinline__ S scalar_args(const S* arr, const S& one, unsigned i) {
    constexpr int W = sizeof(S) / 8;
    static_assert(sizeof(S) % 8 == 0, "whole words");
    S s = one;
    if (arr) {
        unsigned long w[W];
#pragma unroll
        for (int q = 0; q < W; ++q) w[q] = uload(reinterpret_cast<const unsigned long*>(arr + i) + q);
        __builtin_memcpy(&s, w, sizeof(S));
    }
    return s;
}
__device__ __forceinline__ Rk4Sys chunk_args(const Rk4Sys* arr, const Rk4Sys& one, unsigned i) {
    Rk4Sys s = scalar_args(arr, one, i);
    in_global(s.Ls), in_global(s.r0), in_global(s.r), in_global(s.samples), in_global(s.q), in_global(s.xs);
    in_global(s.plain), in_global(s.nsamples);
    return s;
}
__device__ __forceinline__ Rk4AdjArgs chunk_args(const Rk4AdjArgs* arr, const Rk4AdjArgs& one, unsigned i) {
    Rk4AdjArgs a = scalar_args(arr, one, i);
    in_global(a.Ls), in_global(a.gbar), in_global(a.seg), in_global(a.r0bar), in_global(a.vec), in_global(a.q);
    in_global(a.lam), in_global(a.bv), in_global(a.plain);
    return a;
}

// acc[i] = sum_k A(r_i, k) B(k, c_i) for the thread's entries.
template <int DT>
__device__ __forceinline__ void chunk_product(double2 (&acc)[Chunk<DT>::EPT], const double2* A, const double2* B, int lane) {
    using C = Chunk<DT>;
#pragma unroll
    for (int i = 0; i < C::EPT; ++i) acc[i] = make_double2(0.0, 0.0);
#pragma unroll(DT <= 16 ? DT : 4)
    for (int k = 0; k < DT; ++k) {
        double2 a = make_double2(0.0, 0.0);
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) {
            const int e = lane + i * C::LPC, r = e % DT, c = e / DT;
            if (i == 0 || C::LPC % DT != 0) a = A[r + k * DT];  // LPC a multiple of DT: one row per thread
            if (e < C::D2) acc[i] = cfma(a, B[k + c * DT], acc[i]);
        }
    }
}

// Whether the product may carry a chunk's state (chunk_mild): dt kRkChunk times the
// Frobenius norms of the entries' largest values over the chunk, of the generator
// (kMildNorm) and of its Hermitian part (kMildDamp), the rate at which the state
// or a decoupled part of it can shrink.  x + Q x then cancels at most to
// exp(-kMildDamp) of x, and RK4's own damping of a rotation is below 1e-4 a chunk.
// A chunk past either line is stepped: there the product loses what the state
// decays by (scalar generators of dt times rate 0.2, 0.5 and 1, 384 steps: 1e-14,
// 1e-12 and 5e-9 relative against 8e-15, 2e-14 and 4e-14 stepped).  Below the
// lines both are alike: 400 complex scalars each, 512 steps, error of the product
// over that of the steps 0.3 at norm 0.1, 0.8 at 0.5, 1.0 at 1 and 2; over 4096
// steps of a nearly constant generator 0.4, 1.3, 1.2 and 0.9.  TCL generators of
// d = 2..5 at dt = 0.01 have norms up to 1.3 and Hermitian parts of 0.2, up to 0.55
// at coupling 0.2, cutoff 12 and beta 0.4 together.  NaN and infinities are past
// the lines.
constexpr double kMildNorm = 2.0;
constexpr double kMildDamp = 0.5;

// Squared norms summed over a chunk's threads (LPC of them, consecutive).
template <int DT, int M>
__device__ __forceinline__ void chunk_sums(double (&sum)[M]) {
    using C = Chunk<DT>;
    constexpr int LW = C::LPC < 64 ? C::LPC : 64;
#pragma unroll
    for (int m = 1; m < LW; m *= 2)
#pragma unroll
        for (int q = 0; q < M; ++q) sum[q] += __shfl_xor(sum[q], m, 64);
    if constexpr (C::LPC > 64) {
        __shared__ double part[C::LPC / 64][M];
        if (threadIdx.x % 64 == 0)
#pragma unroll
            for (int q = 0; q < M; ++q) part[threadIdx.x / 64][q] = sum[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < M; ++q) {
            sum[q] = 0.0;
#pragma unroll
            for (int w = 0; w < C::LPC / 64; ++w) sum[q] += part[w][q];
        }
    }
}

__device__ __forceinline__ double norm2(double2 z) { return z.x * z.x + z.y * z.y; }

// gen: squared norm of a generator; herm: of L + L^H.  False for NaN.
__device__ __forceinline__ bool chunk_mild(double gen, double herm, double dt) {
    const double s = dt * kRkChunk;
    return s * s * gen <= kMildNorm * kMildNorm && s * s * (0.25 * herm) <= kMildDamp * kMildDamp;
}

// Of kProbes generators spread over the run, the same for every chunk, two past the
// lines by themselves make it one to step whole (below): no product is formed.
constexpr int kProbes = 4;

template <int DT>
__device__ __forceinline__ bool probes_mild(const double2* __restrict__ Ls, long steps, double dt, int lane) {
    using C = Chunk<DT>;
    constexpr int NP = DT * (DT + 1) / 2, PPT = (NP + C::LPC - 1) / C::LPC;  // pairs (r, c), r >= c
    double sum[2 * kProbes];
#pragma unroll
    for (int q = 0; q < 2 * kProbes; ++q) sum[q] = 0.0;
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
        const int p = lane + i * C::LPC;
        int c = 0, r = min(p, NP - 1);
        while (r >= DT - c) r -= DT - c++;
        r += c;
#pragma unroll
        for (int q = 0; q < kProbes; ++q) {
            const double2* L = Ls + (2 * q + 1) * steps / (2 * kProbes) * C::D2;
            const double2 v = L[r + c * DT], w = L[c + r * DT];
            if (p >= NP) continue;
            sum[2 * q] += r == c ? norm2(v) : norm2(v) + norm2(w);
            sum[2 * q + 1] += (r == c ? 1.0 : 2.0) * norm2(cadd(v, cconj(w)));
        }
    }
    chunk_sums<DT>(sum);
    int past = 0;
#pragma unroll
    for (int q = 0; q < kProbes; ++q) past += chunk_mild(sum[2 * q], sum[2 * q + 1], dt) ? 0 : 1;
    return past < 2;
}

// A run with more than a quarter of its chunks past the lines is stepped whole by
// step 3's first workgroup: the plain run and launches that only end (600 steps,
// D = 4..36: 1 to 2 % longer than the plain run).  Products formed for nothing,
// where fewer than two probes are past the lines, take 39 us at D = 16, 0.39 ms at
// D = 36.  The norms cost a carried run nothing that shows: they are taken from the
// generators as step 1 passes them through LDS (read beforehand: 3 to 20 us).
__device__ __forceinline__ bool step_whole(long stepped, long nch) { return 4 * stepped > nch; }

// How many chunks are past the lines (every wave counts them).
__device__ __forceinline__ long stepped_chunks(const int* plain, long nch) {
    long n = 0;
#pragma unroll 4
    for (long j0 = 0; j0 < nch; j0 += 64) {
        const long j = j0 + (threadIdx.x & 63);
        n += __popcll(__ballot(plain[min(j, nch - 1)] != 0 && j < nch));
    }
    return n;
}
constexpr int kWhole = 2;  // plain[0] of a run that step 3 steps whole

// Step 1.
template <int DT, class S>
__global__ __launch_bounds__(Chunk<DT>::NT) void k_chunk_products(const S* arr, S one) {
    using C = Chunk<DT>;
    __shared__ double2 sA[C::CPB][C::D2], sB[C::CPB][C::D2], sQ[C::CPB][C::D2];
    const S s = chunk_args(arr, one, blockIdx.y);
    if (s.D != DT || !s.q) return;
    const int sub = threadIdx.x / C::LPC, lane = threadIdx.x % C::LPC;
    const long c = static_cast<long>(blockIdx.x) * C::CPB + sub;
    if (static_cast<long>(blockIdx.x) * C::CPB * kRkChunk >= s.steps) return;
    const long n0 = c * kRkChunk;
    const double h2 = 0.5 * s.dt, s6 = s.dt / 6.0;
    double2 *A = sA[sub], *B = sB[sub], *Q = sQ[sub];
    double2 l0[C::EPT], l1[C::EPT], ln[C::EPT], q[C::EPT], acc[C::EPT];
    auto load = [&](double2 (&v)[C::EPT], long n) {
        const double2* L = s.Ls + min(n, s.steps) * C::D2;
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) v[i] = L[min(lane + i * C::LPC, C::D2 - 1)];
    };
    auto put = [&](double2* M, const double2 (&v)[C::EPT]) {
#pragma unroll
        for (int i = 0; i < C::EPT; ++i)
            if (lane + i * C::LPC < C::D2) M[lane + i * C::LPC] = v[i];
    };
    load(l0, n0);
    load(l1, n0 + 1);
    if (!probes_mild<DT>(s.Ls, s.steps, s.dt, lane)) {
        if (lane == 0 && n0 < s.steps) s.plain[c] = 1;
        return;
    }
    // the largest |L(r, c)|^2 and |L(r, c) + conj(L(c, r))|^2 of the thread's entries
    // over the chunk, from the generators as they pass through LDS
    double mx[C::EPT], hx[C::EPT];
    auto raise = [](double& m, double a) { m = a > m || a != a ? a : m; };  // a NaN stays
    auto norms = [&](const double2* M, const double2 (&v)[C::EPT]) {
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) {
            const int e = min(lane + i * C::LPC, C::D2 - 1);
            raise(mx[i], norm2(v[i]));
            raise(hx[i], norm2(cadd(v[i], cconj(M[e / DT + e % DT * DT]))));
        }
    };
#pragma unroll
    for (int i = 0; i < C::EPT; ++i) {
        q[i] = make_double2(0.0, 0.0);
        mx[i] = hx[i] = 0.0;
    }
    for (int m = 0; m < kRkChunk; ++m) {
        load(ln, n0 + m + 2);
        double2 lh[C::EPT], k2[C::EPT], k3[C::EPT];
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) lh[i] = cscale(cadd(l0[i], l1[i]), 0.5);
        put(A, lh);
        put(B, l0);
        put(Q, q);
        __syncthreads();
        if (m == 0) norms(B, l0);
        chunk_product<DT>(acc, A, B, lane);  // K2 = Lh (I + h/2 K1), K1 = L0
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) k2[i] = cadd(lh[i], cscale(acc[i], h2));
        __syncthreads();
        put(B, k2);
        __syncthreads();
        chunk_product<DT>(acc, A, B, lane);  // K3 = Lh (I + h/2 K2)
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) k3[i] = cadd(lh[i], cscale(acc[i], h2));
        __syncthreads();
        put(A, l1);
        put(B, k3);
        __syncthreads();
        norms(A, l1);
        chunk_product<DT>(acc, A, B, lane);  // K4 = L1 (I + h K3)
        double2 e[C::EPT];
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) {
            const double2 k4 = cadd(l1[i], cscale(acc[i], s.dt));
            e[i] = cscale(cadd(cadd(l0[i], cscale(cadd(k2[i], k3[i]), 2.0)), k4), s6);
        }
        __syncthreads();
        put(A, e);
        __syncthreads();
        chunk_product<DT>(acc, A, Q, lane);  // Q <- Q + E + E Q
        const bool live = n0 + m < s.steps;
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) {
            if (live) q[i] = cadd(q[i], cadd(e[i], acc[i]));
            l0[i] = l1[i];
            l1[i] = ln[i];
        }
        __syncthreads();
    }
    double sum[2] = {0.0, 0.0};
#pragma unroll
    for (int i = 0; i < C::EPT; ++i)
        if (lane + i * C::LPC < C::D2) {
            sum[0] += mx[i];
            sum[1] += hx[i];
        }
    chunk_sums<DT>(sum);
    if (n0 >= s.steps) return;
    if (lane == 0) s.plain[c] = chunk_mild(sum[0], sum[1], s.dt) ? 0 : 1;
    double2* out = s.q + c * C::D2;
#pragma unroll
    for (int i = 0; i < C::EPT; ++i)
        if (lane + i * C::LPC < C::D2) out[lane + i * C::LPC] = q[i];
}

// Step 2 on the row groups of rk4_rows: x over the i0-th to the i1-th chunk
// visited (REV: lam, visited from the last chunk down), the products' loads a
// ring of R chunks ahead.
template <int DT, bool REV>
__device__ __forceinline__ void chunk_carry(double2* sh, const double2* Q, const double2* b, long nch, long i0, long i1,
                                            const double2* x_in, double2* xs, double2* x_out) {
    using RG = RowGroup<DT>;
    constexpr int R = DT <= 16 ? 8 : 4;
    constexpr long D2 = static_cast<long>(DT) * DT;
    const int lane = static_cast<int>(threadIdx.x & 63), g = lane % RG::G;
    const int r = static_cast<int>(threadIdx.x >> 6) * RG::R + lane / RG::G;
    const bool own = r < DT && g == 0;
    auto at = [&](long i) { return REV ? nch - 1 - i : i; };  // i-th chunk visited
    double2 x = make_double2(0.0, 0.0);
    if (r < DT) x = x_in[r];
    double2 ring[R][RG::CK], rb[R];
    auto load = [&](int j, long i) {
        const long k = at(min(i, i1 - 1));
        load_gen<DT, !REV>(ring[j], Q + k * D2, r, g);
        rb[j] = REV ? b[k * DT + (r < DT ? r : 0)] : make_double2(0.0, 0.0);
    };
#pragma unroll
    for (int j = 0; j < R; ++j) load(j, i0 + j);
    int p = 0;
    if (own) sh[r] = x;
    __syncthreads();
    auto step = [&](int j, long i) {
        if (own) xs[at(i) * DT + r] = x;
        const double2 y = group_dot<DT, REV>(ring[j], sh + p * DT, g);
        x = cadd(x, y);
        if (REV) x = cadd(x, rb[j]);
        p ^= 1;
        if (own) sh[p * DT + r] = x;
        __builtin_amdgcn_sched_barrier(0);
        load(j, i + R);
        __syncthreads();
    };
    long i = i0;
    for (; i + R <= i1; i += R) {
#pragma unroll
        for (int j = 0; j < R; ++j) step(j, i + j);
    }
#pragma unroll
    for (int j = 0; j + 1 < R; ++j)
        if (i + j < i1) step(j, i + j);
    if (own && x_out) x_out[r] = x;
}

// End of the run of chunks, in visiting order, whose flag is that of the i-th.
template <bool REV>
__device__ __forceinline__ long carry_run(const int* plain, long i, long nch) {
    const long lane = threadIdx.x & 63;
    auto flag = [&](long j) { return plain[REV ? nch - 1 - j : j] != 0; };
    const bool first = flag(i);
    for (long b = i; b < nch; b += 64) {
        const unsigned long long other = __ballot(b + lane < nch && flag(b + lane) != first);
        if (other) return b + __ffsll(other) - 1;
    }
    return nch;
}

__device__ __forceinline__ long chunk_count(long steps) { return (steps + kRkChunk - 1) / kRkChunk; }

template <int DT>
__global__ __launch_bounds__(64 * RowGroup<DT>::W) void k_chunk_carry(const Rk4Sys* arr, Rk4Sys one) {
    __shared__ double2 sh[3 * DT];
    const Rk4Sys s = chunk_args(arr, one, blockIdx.x);
    if (s.D != DT || !s.q) return;
    const long nch = chunk_count(s.steps), stepped = stepped_chunks(s.plain, nch);
    if (step_whole(stepped, nch)) {
        if (threadIdx.x == 0) s.plain[0] = kWhole;
        return;
    }
    const double2* x = s.r0;
    for (long i = 0; i < nch;) {
        const long e = stepped ? carry_run<false>(s.plain, i, nch) : nch, last = min(e, nch - 1);
        double2* out = s.xs + last * DT;
        if (stepped && s.plain[i])  // first states as the run's samples
            rk4_rows<DT, false>(sh, s.Ls, i * kRkChunk, last * kRkChunk, x, out, s.dt, kRkChunk, s.xs, nullptr, nullptr,
                                false);
        else
            chunk_carry<DT, false>(sh, s.q, nullptr, nch, i, e, x, s.xs, e < nch ? out : nullptr);
        __syncthreads();
        x = out;
        i = e;
    }
}

template <int DT>
__global__ __launch_bounds__(64 * RowGroup<DT>::W) void k_chunk_states(const Rk4Sys* arr, Rk4Sys one) {
    __shared__ double2 sh[3 * DT];
    const Rk4Sys s = chunk_args(arr, one, blockIdx.y);
    const long c = blockIdx.x, n0 = c * kRkChunk;
    if (s.D != DT || !s.q || n0 >= s.steps) return;
    const bool whole = s.plain[0] == kWhole;
    if (whole && c) return;
    const long n1 = whole ? s.steps : min(n0 + kRkChunk, s.steps);
    const bool last = n1 == s.steps;
    rk4_rows<DT, false>(sh, s.Ls, n0, n1, whole ? s.r0 : s.xs + c * DT, last ? s.r : nullptr, s.dt, s.every, s.samples,
                        last ? s.nsamples : nullptr, nullptr, last);
}

// The reverse's chunk walks: CONST from lam = 0 (constant part to bv), else
// from the chunk's true lam, storing kb1..kb4.  One wave per workgroup and few
// workgroups: scheduled for at most two waves per SIMD (D = 16: a run that is
// stepped whole, 1000 steps, 786 -> 728 us; the plain walk 746).
template <int DT, bool CONST>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_chunk_walk(const Rk4AdjArgs* arr, Rk4AdjArgs one) {
    __shared__ double2 sh[5 * DT];
    const Rk4AdjArgs A = chunk_args(arr, one, blockIdx.y);
    const long c = blockIdx.x, n0 = c * kRkChunk;
    if (n0 >= A.steps) return;
    if constexpr (CONST) {
        if (!A.plain[c]) rk4_rows_adjoint<DT, WALK_NONE>(sh, A, n0, min(n0 + kRkChunk, A.steps), nullptr, A.bv + c * DT);
    } else {
        const bool whole = A.plain[0] == kWhole;
        if (whole && c) return;
        // lam at a chunk's first step is known from the carry: bv takes the repeated value
        rk4_rows_adjoint<DT, WALK_VEC>(sh, A, n0, whole ? A.steps : min(n0 + kRkChunk, A.steps),
                                       whole ? A.gbar + A.steps * DT : A.lam + c * DT, whole ? A.r0bar : A.bv + c * DT);
    }
}

template <int DT>
__global__ __launch_bounds__(64) void k_chunk_carry_rev(const Rk4AdjArgs* arr, Rk4AdjArgs one) {
    __shared__ double2 sh[5 * DT];
    const Rk4AdjArgs A = chunk_args(arr, one, blockIdx.x);
    const long nch = chunk_count(A.steps), stepped = stepped_chunks(A.plain, nch);
    const double2* x = A.gbar + A.steps * DT;
    if (step_whole(stepped, nch)) {
        if (threadIdx.x == 0) A.plain[0] = kWhole;
        return;
    }
    for (long i = 0; i < nch;) {
        const long e = stepped ? carry_run<true>(A.plain, i, nch) : nch, top = nch - 1 - i;  // chunks top .. nch - e
        double2* out = e < nch ? A.lam + (nch - 1 - e) * DT : A.r0bar;
        if (stepped && A.plain[top]) {
            if (threadIdx.x < DT) A.lam[top * DT + threadIdx.x] = x[threadIdx.x];
            rk4_rows_adjoint<DT, WALK_LAM>(sh, A, (nch - e) * kRkChunk, min((top + 1) * kRkChunk, A.steps), x, out);
        } else {
            chunk_carry<DT, true>(sh, A.q, A.bv, nch, i, e, x, A.lam, out);
        }
        __syncthreads();
        x = out;
        i = e;
    }
}

// ---------------------------------------------------------------------------
// Wide runs: D > 64 whose generators do not fit the LDS (rk4_wide).  One
// workgroup reads them at the rate of one CU (D = 256: 1 MB a product, 18 us);
// here a product is a launch whose workgroups share the rows, so a step is four
// dependent launches.  Every workgroup first forms the whole stage vector from
// the earlier products, with the first generator loads already in flight, and
// workgroup 0 keeps what later launches or the caller read.  Vectors that the
// next step's first launch both reads and writes alternate by the step's parity.
// The midpoint generators are formed on the fly: a step then touches one new
// matrix, the rest is in the L2 slices (row blocks keep their XCD).
// Sums: 32 (reverse: 64) partial sums a row, then a fixed tree.
// ---------------------------------------------------------------------------
constexpr int kWideRows = 8;    // rows of a workgroup: 128 B runs of a column
constexpr int kWideGroups = kRkBlock / kWideRows;
constexpr int kWideBlk = 8;     // generator loads in flight
constexpr int kWideOut = kRkBlock / 64;  // outputs of a reverse workgroup, a wave each

// y[r] = sum_c M(r, c) u[c] for the kWideRows rows of block rb, M = L0 (L1 null)
// or (L0 + L1) / 2; form() fills u (LDS) in between the first loads and their use.
template <class Form>
__device__ __forceinline__ void wide_rows(const double2* __restrict__ L0, const double2* __restrict__ L1, int D, long rb,
                                          const double2* u, double2* y, Form&& form) {
    __shared__ double2 part[kRkBlock / 64][kWideRows];
    const int lr = threadIdx.x % kWideRows, cg = threadIdx.x / kWideRows;
    const int r = static_cast<int>(rb) * kWideRows + lr;
    const double2* p0 = L0 + min(r, D - 1);
    const double2* p1 = L1 ? L1 + min(r, D - 1) : nullptr;
    double2 v0[kWideBlk], v1[kWideBlk];
    auto load = [&](int c0) {
#pragma unroll
        for (int j = 0; j < kWideBlk; ++j) v0[j] = p0[static_cast<long>(min(c0 + cg + j * kWideGroups, D - 1)) * D];
        if (p1) {
#pragma unroll
            for (int j = 0; j < kWideBlk; ++j) v1[j] = p1[static_cast<long>(min(c0 + cg + j * kWideGroups, D - 1)) * D];
#pragma unroll
            for (int j = 0; j < kWideBlk; ++j) v0[j] = cscale(cadd(v0[j], v1[j]), 0.5);
        }
    };
    load(0);
    form();
    __syncthreads();
    double2 s = make_double2(0.0, 0.0);
    for (int c0 = 0;;) {
#pragma unroll
        for (int j = 0; j < kWideBlk; ++j) {
            const int c = c0 + cg + j * kWideGroups;
            if (c < D) s = cfma(v0[j], u[c], s);
        }
        c0 += kWideBlk * kWideGroups;
        if (c0 >= D) break;
        load(c0);
    }
#pragma unroll
    for (int m = kWideRows; m < 64; m *= 2) {
        s.x += __shfl_xor(s.x, m);
        s.y += __shfl_xor(s.y, m);
    }
    if (threadIdx.x % 64 < kWideRows) part[threadIdx.x / 64][lr] = s;
    __syncthreads();
    if (threadIdx.x < kWideRows && r < D) {
        double2 t = part[0][lr];
#pragma unroll
        for (int w = 1; w < kRkBlock / 64; ++w) t = cadd(t, part[w][lr]);
        y[r] = t;
    }
}

// y[r] = sum_c conj(M(c, r)) u[c], one wave per r (columns are contiguous).
template <class Form>
__device__ __forceinline__ void wide_columns(const double2* __restrict__ L0, const double2* __restrict__ L1, int D,
                                             const double2* u, double2* y, Form&& form) {
    const int lane = threadIdx.x % 64, r = static_cast<int>(blockIdx.x) * kWideOut + threadIdx.x / 64;
    const long col = static_cast<long>(min(r, D - 1)) * D;
    constexpr int kBlk = 4;
    double2 v0[kBlk], v1[kBlk];
    auto load = [&](int c0) {
#pragma unroll
        for (int j = 0; j < kBlk; ++j) v0[j] = L0[col + min(c0 + lane + 64 * j, D - 1)];
        if (L1) {
#pragma unroll
            for (int j = 0; j < kBlk; ++j) v1[j] = L1[col + min(c0 + lane + 64 * j, D - 1)];
#pragma unroll
            for (int j = 0; j < kBlk; ++j) v0[j] = cscale(cadd(v0[j], v1[j]), 0.5);
        }
    };
    load(0);
    form();
    __syncthreads();
    double2 s = make_double2(0.0, 0.0);
    for (int c0 = 0;;) {
#pragma unroll
        for (int j = 0; j < kBlk; ++j) {
            const int c = c0 + lane + 64 * j;
            if (c < D) s = cfma_conj(v0[j], u[c], s);
        }
        c0 += 64 * kBlk;
        if (c0 >= D) break;
        load(c0);
    }
#pragma unroll
    for (int m = 1; m < 64; m *= 2) {
        s.x += __shfl_xor(s.x, m);
        s.y += __shfl_xor(s.y, m);
    }
    if (lane == 0 && r < D) y[r] = s;
}

__device__ __forceinline__ double2 wide_sum(double2 x, double2 k1, double2 k2, double2 k3, double2 k4, double s6) {
    return cadd(x, cscale(cadd(cadd(cadd(k1, cscale(k2, 2.0)), cscale(k3, 2.0)), k4), s6));
}

// Stage STAGE (0..3) of step n of every system; stage 0 at n = steps closes the
// run.  xs: r_n and k1 of both parities, k2, k3, k4.
template <int STAGE>
__global__ __launch_bounds__(kRkBlock) void k_wide_stage(const Rk4Sys* arr, Rk4Sys one, long n) {
    extern __shared__ double2 u[];
    const Rk4Sys S = arr ? arr[blockIdx.y] : one;
    if (n > S.steps || (STAGE && n == S.steps)) return;
    const int D = S.D;
    const long D2 = static_cast<long>(D) * D, cur = n & 1;
    double2 *x = S.xs + cur * D, *k1 = S.xs + (2 + cur) * D;
    double2 *k2 = S.xs + 4 * D, *k3 = S.xs + 5 * D, *k4 = S.xs + 6 * D;
    if constexpr (STAGE == 0) {
        const double2 *xo = S.xs + (1 - cur) * D, *ko = S.xs + (3 - cur) * D;
        auto form = [&] {
            const bool keep = S.samples && (n == S.steps || n % S.every == 0);
            double2* row = keep ? S.samples + (n + S.every - 1) / S.every * D : nullptr;
            for (int e = threadIdx.x; e < D; e += kRkBlock) {
                const double2 v = n ? wide_sum(xo[e], ko[e], k2[e], k3[e], k4[e], S.dt / 6.0) : S.r0[e];
                u[e] = v;
                if (blockIdx.x) continue;
                x[e] = v;
                if (keep) row[e] = v;
                if (n == S.steps) S.r[e] = v;
            }
        };
        if (n == S.steps) {
            if (blockIdx.x) return;
            form();
            if (threadIdx.x == 0 && S.nsamples) *S.nsamples = S.samples ? (n + S.every - 1) / S.every + 1 : 0;
            return;
        }
        wide_rows(S.Ls + n * D2, nullptr, D, blockIdx.x, u, k1, form);
    } else {
        const double2* k = STAGE == 1 ? k1 : STAGE == 2 ? k2 : k3;
        const double f = STAGE == 3 ? S.dt : 0.5 * S.dt;
        const double2* L0 = STAGE == 3 ? S.Ls + (n + 1) * D2 : S.Lh ? S.Lh + n * D2 : S.Ls + n * D2;
        const double2* L1 = STAGE == 3 || S.Lh ? nullptr : S.Ls + (n + 1) * D2;
        wide_rows(L0, L1, D, blockIdx.x, u, STAGE == 1 ? k2 : STAGE == 2 ? k3 : k4, [&] {
            for (int e = threadIdx.x; e < D; e += kRkBlock) u[e] = cadd(x[e], cscale(k[e], f));
        });
    }
}

// Stage STAGE of step j of every checkpoint segment: the states and stage
// points into seg.  The products of step n use vec's rows of n, which the walk
// fills afterwards.  Grid: (segments x row blocks, tapes).
template <int STAGE>
__global__ __launch_bounds__(kRkBlock) void k_wide_segment(const Rk4AdjArgs* arr, Rk4AdjArgs one, int j) {
    extern __shared__ double2 u[];
    const Rk4AdjArgs A = arr ? arr[blockIdx.y] : one;
    const int D = A.D, nrb = (D + kWideRows - 1) / kWideRows;
    const long sg = blockIdx.x / nrb, rb = blockIdx.x % nrb;
    const long n = sg * A.K + j, s1 = min((sg + 1) * A.K, A.steps);
    if (n >= s1) return;
    const long D2 = static_cast<long>(D) * D;
    double2 *row = A.seg + n * 4 * D, *k = A.vec + n * 4 * D;
    const double f = STAGE == 3 ? A.dt : 0.5 * A.dt;
    const double2* L0 = A.Ls + (STAGE == 3 ? n + 1 : n) * D2;
    const double2* L1 = STAGE == 1 || STAGE == 2 ? A.Ls + (n + 1) * D2 : nullptr;
    wide_rows(L0, L1, D, rb, u, k + STAGE * D, [&] {
        for (int e = threadIdx.x; e < D; e += kRkBlock) {
            double2 v;
            if (STAGE)
                v = cadd(row[e], cscale(k[(STAGE - 1) * D + e], f));
            else if (j == 0)
                v = A.ck[sg * D + e];
            else
                v = wide_sum(row[e - 4 * D], k[e - 4 * D], k[e - 3 * D], k[e - 2 * D], k[e - D], A.dt / 6.0);
            u[e] = v;
            if (rb == 0) row[STAGE * D + e] = v;
        }
    });
}

// Stage STAGE of the reverse of step n: ub3 = L1^H kb4, ub2 = Lh^H kb3,
// ub1 = Lh^H kb2, ub0 = L0^H kb1 (rk4_adjoint_body); stage 0 first forms
// lam_{n+1} of the step before, at n = -1 the result.  lam: lam and ub3 of both
// parities, ub2, ub1, ub0.
template <int STAGE>
__global__ __launch_bounds__(kRkBlock) void k_wide_walk(const Rk4AdjArgs* arr, Rk4AdjArgs one, long n) {
    extern __shared__ double2 u[];
    const Rk4AdjArgs A = arr ? arr[blockIdx.y] : one;
    const int D = A.D;
    const long D2 = static_cast<long>(D) * D, cur = n & 1;
    double2 *lam = A.lam + cur * D, *ub3 = A.lam + (2 + cur) * D;
    double2 *ub2 = A.lam + 4 * D, *ub1 = A.lam + 5 * D, *ub0 = A.lam + 6 * D;
    const double s6 = A.dt / 6.0, h = 0.5 * A.dt;
    double2* v = A.vec + n * 4 * D;  // kb1..kb4
    if constexpr (STAGE == 0) {
        const double2 *lo = A.lam + (1 - cur) * D, *uo = A.lam + (3 - cur) * D;
        auto form = [&] {
            for (int e = threadIdx.x; e < D; e += kRkBlock) {
                double2 l = A.gbar[(n + 1) * D + e];
                if (n + 1 < A.steps) l = cadd(cadd(cadd(cadd(cadd(lo[e], uo[e]), ub2[e]), ub1[e]), ub0[e]), l);
                const double2 kb4 = cscale(l, s6);
                u[e] = kb4;
                if (blockIdx.x) continue;
                if (n < 0) {
                    A.r0bar[e] = l;
                } else {
                    lam[e] = l;
                    v[3 * D + e] = kb4;
                }
            }
        };
        if (n < 0) {
            if (blockIdx.x == 0) form();
            return;
        }
        wide_columns(A.Ls + (n + 1) * D2, nullptr, D, u, ub3, form);
    } else {
        const double2* ub = STAGE == 1 ? ub3 : STAGE == 2 ? ub2 : ub1;
        const double2 *L0 = A.Ls + n * D2, *L1 = STAGE == 3 ? nullptr : L0 + D2;
        wide_columns(L0, L1, D, u, STAGE == 1 ? ub2 : STAGE == 2 ? ub1 : ub0, [&] {
            for (int e = threadIdx.x; e < D; e += kRkBlock) {
                const double2 kb = cadd(cscale(lam[e], STAGE == 3 ? s6 : 2.0 * s6), cscale(ub[e], STAGE == 1 ? A.dt : h));
                u[e] = kb;
                if (blockIdx.x == 0) v[(3 - STAGE) * D + e] = kb;
            }
        });
    }
}

// ---------------------------------------------------------------------------
// Launches
// ---------------------------------------------------------------------------
hipError_t rk4_set_lds_limits() {
    for (const void* fn : {reinterpret_cast<const void*>(k_rk4), reinterpret_cast<const void*>(k_rk4_batch),
                           reinterpret_cast<const void*>(k_rk4_adjoint), reinterpret_cast<const void*>(k_rk4_recompute),
                           reinterpret_cast<const void*>(k_rk4_adjoint_multi),
                           reinterpret_cast<const void*>(k_rk4_recompute_multi)}) {
        const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 static_cast<int>(kRkLds));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <class F>
static void chunk_dispatch(int D, F&& f) {
    switch (D) {
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        case 16: f(std::integral_constant<int, 16>{}); break;
        case 25: f(std::integral_constant<int, 25>{}); break;
        case 36: f(std::integral_constant<int, 36>{}); break;
        default: break;
    }
}

void launch_rk4_chunked(int D, const Rk4Sys* arr, const Rk4Sys& one, unsigned nsys, long max_steps, hipStream_t st) {
    const unsigned nch = static_cast<unsigned>((max_steps + kRkChunk - 1) / kRkChunk);
    chunk_dispatch(D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        const dim3 grid((nch + Chunk<DT>::CPB - 1) / Chunk<DT>::CPB, nsys), block(Chunk<DT>::NT);
        hipLaunchKernelGGL((k_chunk_products<DT, Rk4Sys>), grid, block, 0, st, arr, one);
        hipLaunchKernelGGL(k_chunk_carry<DT>, dim3(nsys), dim3(rk4_rows_threads(DT)), 0, st, arr, one);
        hipLaunchKernelGGL(k_chunk_states<DT>, dim3(nch, nsys), dim3(rk4_rows_threads(DT)), 0, st, arr, one);
    });
}

void launch_rk4_chunked_walk(int D, const Rk4AdjArgs* arr, const Rk4AdjArgs& one, unsigned ntapes, long steps,
                             hipStream_t st) {
    const unsigned nch = static_cast<unsigned>((steps + kRkChunk - 1) / kRkChunk);
    chunk_dispatch(D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        if constexpr (DT <= 16) {
            const dim3 grid((nch + Chunk<DT>::CPB - 1) / Chunk<DT>::CPB, ntapes), block(Chunk<DT>::NT);
                hipLaunchKernelGGL((k_chunk_products<DT, Rk4AdjArgs>), grid, block, 0, st, arr, one);
            hipLaunchKernelGGL((k_chunk_walk<DT, true>), dim3(nch, ntapes), dim3(64), 0, st, arr, one);
            hipLaunchKernelGGL(k_chunk_carry_rev<DT>, dim3(ntapes), dim3(64), 0, st, arr, one);
            hipLaunchKernelGGL((k_chunk_walk<DT, false>), dim3(nch, ntapes), dim3(64), 0, st, arr, one);
        }
    });
}

void launch_rk4_rows(int D, const double2* Ls, long steps, double2* r, double dt, long every, double2* samples,
                     long* nsamples, hipStream_t st) {
    rows_dispatch(D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        hipLaunchKernelGGL(k_rk4_rows<DT>, dim3(1), dim3(rk4_rows_threads(DT)), 3 * DT * 16, st, Ls, steps, r, dt, every,
                           samples, nsamples);
    });
}

void launch_rk4(int D, const double2* Ls, const double2* Lh, long steps, double2* r, double dt, long every,
                double2* samples, long* nsamples, int nstage, int block, std::size_t lds, hipStream_t st) {
    hipLaunchKernelGGL(k_rk4, dim3(1), dim3(block), lds, st, Ls, Lh, steps, D, r, dt, every, samples, nsamples, nstage);
}

void launch_rk4_batch(unsigned nsys, const Rk4Sys* sys, int block, std::size_t lds, hipStream_t st) {
    hipLaunchKernelGGL(k_rk4_batch, dim3(nsys), dim3(block), lds, st, sys);
}

static dim3 wide_grid(int D, unsigned y, int per = kWideRows) { return dim3(static_cast<unsigned>((D + per - 1) / per), y); }

void launch_rk4_wide(int D, const Rk4Sys* arr, const Rk4Sys& one, unsigned nsys, long max_steps, hipStream_t st) {
    const dim3 grid = wide_grid(D, nsys), block(kRkBlock);
    const std::size_t lds = static_cast<std::size_t>(D) * 16;
    for (long n = 0; n < max_steps; ++n) {
        hipLaunchKernelGGL(k_wide_stage<0>, grid, block, lds, st, arr, one, n);
        hipLaunchKernelGGL(k_wide_stage<1>, grid, block, lds, st, arr, one, n);
        hipLaunchKernelGGL(k_wide_stage<2>, grid, block, lds, st, arr, one, n);
        hipLaunchKernelGGL(k_wide_stage<3>, grid, block, lds, st, arr, one, n);
    }
    hipLaunchKernelGGL(k_wide_stage<0>, dim3(1, nsys), block, lds, st, arr, one, max_steps);
}

void launch_rk4_wide_reverse(int D, const Rk4AdjArgs* arr, const Rk4AdjArgs& one, unsigned ntapes, long steps, int K,
                             hipStream_t st) {
    const dim3 block(kRkBlock);
    const std::size_t lds = static_cast<std::size_t>(D) * 16;
    const dim3 gs(wide_grid(D, 1).x * static_cast<unsigned>((steps + K - 1) / K), ntapes);
    for (int j = 0; j < K && j < steps; ++j) {
        hipLaunchKernelGGL(k_wide_segment<0>, gs, block, lds, st, arr, one, j);
        hipLaunchKernelGGL(k_wide_segment<1>, gs, block, lds, st, arr, one, j);
        hipLaunchKernelGGL(k_wide_segment<2>, gs, block, lds, st, arr, one, j);
        hipLaunchKernelGGL(k_wide_segment<3>, gs, block, lds, st, arr, one, j);
    }
    const dim3 gw = wide_grid(D, ntapes, kWideOut);
    for (long n = steps - 1; n >= 0; --n) {
        hipLaunchKernelGGL(k_wide_walk<0>, gw, block, lds, st, arr, one, n);
        hipLaunchKernelGGL(k_wide_walk<1>, gw, block, lds, st, arr, one, n);
        hipLaunchKernelGGL(k_wide_walk<2>, gw, block, lds, st, arr, one, n);
        hipLaunchKernelGGL(k_wide_walk<3>, gw, block, lds, st, arr, one, n);
    }
    hipLaunchKernelGGL(k_wide_walk<0>, dim3(1, ntapes), block, lds, st, arr, one, -1L);
}

void launch_rk4_recompute(const Rk4AdjArgs& A, bool rows, unsigned nseg, std::size_t lds, hipStream_t st) {
    if (!rows) {
        hipLaunchKernelGGL(k_rk4_recompute, dim3(nseg), dim3(kRkBlock), lds, st, A);
        return;
    }
    rows_dispatch(A.D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        hipLaunchKernelGGL(k_rk4_recompute_rows<DT>, dim3(nseg), dim3(rk4_rows_threads(DT)), 3 * DT * 16, st, A);
    });
}

void launch_rk4_walk(const Rk4AdjArgs& A, bool rows, std::size_t lds, hipStream_t st) {
    if (!rows) {
        hipLaunchKernelGGL(k_rk4_adjoint, dim3(1), dim3(kRkBlock), lds, st, A);
        return;
    }
    rows_dispatch(A.D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        if constexpr (DT <= 16) hipLaunchKernelGGL(k_rk4_adjoint_rows<DT>, dim3(1), dim3(64), 5 * DT * 16, st, A);
    });
}

static dim3 lbar_grid(int D, long steps, unsigned ntapes) {
    return dim3(static_cast<unsigned>((D * D + kRkBlock - 1) / kRkBlock), static_cast<unsigned>(steps + 1), ntapes);
}

void launch_rk4_lbar(const Rk4AdjArgs& A, hipStream_t st) {
    hipLaunchKernelGGL(k_rk4_lbar, lbar_grid(A.D, A.steps, 1), dim3(kRkBlock), 0, st, A);
}

void launch_rk4_recompute_multi(const Rk4AdjArgs* As, unsigned ntapes, int D, bool rows, unsigned nseg,
                                std::size_t lds, hipStream_t st) {
    if (!rows) {
        hipLaunchKernelGGL(k_rk4_recompute_multi, dim3(nseg, ntapes), dim3(kRkBlock), lds, st, As);
        return;
    }
    rows_dispatch(D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        hipLaunchKernelGGL(k_rk4_recompute_rows_multi<DT>, dim3(nseg, ntapes), dim3(rk4_rows_threads(DT)), 3 * DT * 16, st,
                           As);
    });
}

void launch_rk4_walk_multi(const Rk4AdjArgs* As, unsigned ntapes, int D, bool rows, std::size_t lds, hipStream_t st) {
    if (!rows) {
        hipLaunchKernelGGL(k_rk4_adjoint_multi, dim3(ntapes), dim3(kRkBlock), lds, st, As);
        return;
    }
    rows_dispatch(D, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        if constexpr (DT <= 16)
            hipLaunchKernelGGL(k_rk4_adjoint_rows_multi<DT>, dim3(ntapes), dim3(64), 5 * DT * 16, st, As);
    });
}

void launch_rk4_lbar_multi(const Rk4AdjArgs* As, unsigned ntapes, int D, long steps, hipStream_t st) {
    hipLaunchKernelGGL(k_rk4_lbar_multi, lbar_grid(D, steps, ntapes), dim3(kRkBlock), 0, st, As);
}

}  // namespace taco_engine
