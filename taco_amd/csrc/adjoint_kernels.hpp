// Reverse-mode kernels of the TCL4 pipeline: RK4 -> fused L4 -> F/C/R.
//
// Included once by engine.hip after the forward kernels (it uses their device
// helpers).  The reference has no derivative code; these are the hand-written
// adjoints of the forward passes above.  Convention for every complex
// cotangent z_bar: dLoss = Re sum conj(z_bar) dz, i.e. z_bar = dLoss/dRe z +
// i dLoss/dIm z (torch's convention for real losses).
#pragma once

// ---------------------------------------------------------------------------
// Fused L4 adjoint, one workgroup per time t.  From Lbar(t) (the RK4 layout of
// L4(n,m;i,j) = GW(n,i;m,j)) it forms Tbar = GWbar + GWbar^H (GW = T + T^H)
// and, for every NAKZWAN term sigma * e1 e2 e3 e4 * S of T(n,i;m,j), adds
// sigma Tbar conj(e1 e2 e3 e4) to the slice entries S gathers from and
// sigma Tbar conj(S * prod of the other three) to each operator entry.  Slice
// cotangents accumulate in LDS (or global when they do not fit) with atomic
// adds; operator cotangents in LDS, written per time.
// ---------------------------------------------------------------------------
struct L4AdjArgs {
    const double2* Lbar;  // [T][N^4]
    const double2* Fs;    // [T][nf3] forward slices
    const double2* Cs;
    const double2* Rs;
    const int* p2f;
    const double2* ops;
    int N, nf, num_ops;
    long nf3;
    double2* sbar;        // [T][3][nf3]; zero on entry unless lds_slices
    double2* Abar;        // [T][num_ops][N^2]
    int lds_slices;
};

__device__ __forceinline__ void atomic_cadd(double2* p, double2 v) {
    atomicAdd(&p->x, v.x);
    atomicAdd(&p->y, v.y);
}

__global__ __launch_bounds__(kBlock) void k_l4_adjoint(L4AdjArgs A) {
    extern __shared__ double2 sm[];
    const int N = A.N, N2 = N * N, N4 = N2 * N2;
    const long t = blockIdx.x;
    double2* Tb = sm;                                   // N^4
    double2* opsS = Tb + N4;                            // num_ops N^2
    double2* Ab = opsS + A.num_ops * N2;                // num_ops N^2
    double2* sb = Ab + A.num_ops * N2;                  // 3 nf3 (lds_slices)
    int* f = reinterpret_cast<int*>(sb + (A.lds_slices ? 3 * A.nf3 : 0));
    const double2* Lb = A.Lbar + t * N4;
    for (int idx = threadIdx.x; idx < N4; idx += kBlock) {
        const int ru = idx % N2, cu = idx / N2;
        const int n = ru % N, i = ru / N, m = cu % N, j = cu / N;
        const double2 g1 = Lb[(n + m * N) + (i + j * N) * N2];
        const double2 g2 = Lb[(m + n * N) + (j + i * N) * N2];
        Tb[idx] = cadd(g1, cconj(g2));
    }
    for (int e = threadIdx.x; e < A.num_ops * N2; e += kBlock) {
        opsS[e] = A.ops[e];
        Ab[e] = make_double2(0.0, 0.0);
    }
    if (A.lds_slices)
        for (long e = threadIdx.x; e < 3 * A.nf3; e += kBlock) sb[e] = make_double2(0.0, 0.0);
    for (int e = threadIdx.x; e < N2; e += kBlock) f[e] = A.p2f[e];
    __syncthreads();
    const double2* Fp = A.Fs + t * A.nf3;
    const double2* Cp = A.Cs + t * A.nf3;
    const double2* Rp = A.Rs + t * A.nf3;
    double2* sF = A.lds_slices ? sb : A.sbar + t * 3 * A.nf3;
    double2* sC = sF + A.nf3;
    double2* sR = sC + A.nf3;
    const long nf = A.nf;
    auto id3 = [nf](int x, int y, int z) { return (static_cast<long>(x) * nf + y) * nf + z; };
    auto F2 = [f, N](int r, int c) { return f[r + c * N]; };
    // One term sigma * e1 e2 e3 e4 * S with S = sum of up to two slice
    // entries (w1 * slice1[x1] + w2 * slice2[x2]); d1..d4 are the operator
    // cotangent slots of e1..e4.
    auto term = [&](double sg, double2 Tv, double2 e1, double2 e2, double2 e3, double2 e4, double2* d1, double2* d2,
                    double2* d3, double2* d4, double2 S, double2* s1, long x1, double w1, double2* s2, long x2,
                    double w2) {
        const double2 p12 = cmul(e1, e2), p34 = cmul(e3, e4);
        const double2 Sb = cscale(cmul(Tv, cconj(cmul(p12, p34))), sg);
        atomic_cadd(s1 + x1, cscale(Sb, w1));
        if (s2) atomic_cadd(s2 + x2, cscale(Sb, w2));
        const double2 TS = cscale(cmul(Tv, cconj(S)), sg);
        atomic_cadd(d1, cmul(TS, cconj(cmul(e2, p34))));
        atomic_cadd(d2, cmul(TS, cconj(cmul(e1, p34))));
        atomic_cadd(d3, cmul(TS, cconj(cmul(p12, e4))));
        atomic_cadd(d4, cmul(TS, cconj(cmul(p12, e3))));
    };
    for (int idx = threadIdx.x; idx < N4; idx += kBlock) {
        const int row_u = idx % N2, col_u = idx / N2;
        const int n = row_u % N, i = row_u / N, m = col_u % N, j = col_u / N;
        const double2 Tv = Tb[idx];
        if (Tv.x == 0.0 && Tv.y == 0.0) continue;
        for (int iA = 0; iA < A.num_ops; ++iA) {
            const double2* Ap = opsS + iA * N2;
            double2* AbA = Ab + iA * N2;
            for (int iB = 0; iB < A.num_ops; ++iB) {
                const double2* Bp = opsS + iB * N2;
                double2* AbB = Ab + iB * N2;
#define AA(r, c) Ap[(r) + (c) * N]
#define BB(r, c) Bp[(r) + (c) * N]
#define DA(r, c) (AbA + (r) + (c) * N)
#define DB(r, c) (AbB + (r) + (c) * N)
                for (int a = 0; a < N; ++a) {
                    for (int b = 0; b < N; ++b) {
                        const long xM1 = id3(F2(b, a), F2(b, i), F2(n, b)), xM2 = id3(F2(b, a), F2(n, a), F2(a, i));
                        const long xI = id3(F2(a, n), F2(b, i), F2(n, b));
                        const long xK = id3(F2(i, b), F2(n, a), F2(a, i));
                        const long x1 = id3(F2(a, n), F2(j, b), F2(n, i));
                        const long x2 = id3(F2(i, a), F2(j, b), F2(n, i));
                        const long x3 = id3(F2(b, a), F2(j, m), F2(a, i));
                        const long x4 = id3(F2(i, b), F2(j, m), F2(a, i));
                        const double2 Mv = csub(Fp[xM1], Rp[xM2]);
                        const double2 Iv = Fp[xI], Kv = Rp[xK];
                        const double2 X1 = cadd(Cp[x1], Rp[x1]), X2 = cadd(Cp[x2], Rp[x2]);
                        const double2 X3 = cadd(Cp[x3], Rp[x3]), X4 = cadd(Cp[x4], Rp[x4]);
                        // T = -(t1 - t2 + t3 + t4 - t5 - t6 + t7)
                        term(-1.0, Tv, BB(n, a), AA(a, b), BB(b, i), AA(j, m), DB(n, a), DA(a, b), DB(b, i), DA(j, m),
                             Mv, sF, xM1, 1.0, sR, xM2, -1.0);
                        term(+1.0, Tv, AA(n, a), BB(a, b), BB(b, i), AA(j, m), DA(n, a), DB(a, b), DB(b, i), DA(j, m),
                             Iv, sF, xI, 1.0, nullptr, 0, 0.0);
                        term(-1.0, Tv, BB(n, a), BB(a, b), AA(b, i), AA(j, m), DB(n, a), DB(a, b), DA(b, i), DA(j, m),
                             Kv, sR, xK, 1.0, nullptr, 0, 0.0);
                        term(-1.0, Tv, AA(n, a), BB(a, i), BB(j, b), AA(b, m), DA(n, a), DB(a, i), DB(j, b), DA(b, m),
                             X1, sC, x1, 1.0, sR, x1, 1.0);
                        term(+1.0, Tv, BB(n, a), AA(a, i), BB(j, b), AA(b, m), DB(n, a), DA(a, i), DB(j, b), DA(b, m),
                             X2, sC, x2, 1.0, sR, x2, 1.0);
                        term(+1.0, Tv, AA(n, a), AA(a, b), BB(b, i), BB(j, m), DA(n, a), DA(a, b), DB(b, i), DB(j, m),
                             X3, sC, x3, 1.0, sR, x3, 1.0);
                        term(-1.0, Tv, AA(n, a), BB(a, b), AA(b, i), BB(j, m), DA(n, a), DB(a, b), DA(b, i), DB(j, m),
                             X4, sC, x4, 1.0, sR, x4, 1.0);
                    }
                }
                if (j == m) {
                    for (int a = 0; a < N; ++a)
                        for (int b = 0; b < N; ++b)
                            for (int c = 0; c < N; ++c) {
                                const long yM1 = id3(F2(c, b), F2(c, i), F2(a, c));
                                const long yM2 = id3(F2(c, b), F2(a, b), F2(b, i));
                                const long yK = id3(F2(i, c), F2(a, b), F2(b, i));
                                const long yI = id3(F2(b, a), F2(c, i), F2(a, c));
                                const double2 Mv = csub(Fp[yM1], Rp[yM2]);
                                const double2 Kv = Rp[yK], Iv = Fp[yI];
                                term(+1.0, Tv, AA(n, a), BB(a, b), AA(b, c), BB(c, i), DA(n, a), DB(a, b), DA(b, c),
                                     DB(c, i), Mv, sF, yM1, 1.0, sR, yM2, -1.0);
                                term(+1.0, Tv, AA(n, a), BB(a, b), BB(b, c), AA(c, i), DA(n, a), DB(a, b), DB(b, c),
                                     DA(c, i), Kv, sR, yK, 1.0, nullptr, 0, 0.0);
                                term(-1.0, Tv, AA(n, a), AA(a, b), BB(b, c), BB(c, i), DA(n, a), DA(a, b), DB(b, c),
                                     DB(c, i), Iv, sF, yI, 1.0, nullptr, 0, 0.0);
                            }
                }
#undef AA
#undef BB
#undef DA
#undef DB
            }
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < A.num_ops * N2; e += kBlock) A.Abar[t * A.num_ops * N2 + e] = Ab[e];
    if (A.lds_slices)
        for (long e = threadIdx.x; e < 3 * A.nf3; e += kBlock) A.sbar[t * 3 * A.nf3 + e] = sb[e];
}

// ---------------------------------------------------------------------------
// Factorised L4 adjoint: the reverse of k_l4f, O(N^5 + N^3 nf) per time
// instead of the O(N^6) term walk above.  Per operator pair (A, B) the
// forward builds
//   Q(a,i,g)  = sum_b A(a,b) B(b,i) X(f(b,a),g,f(a,i)) - B(a,b) A(b,i) X(f(i,b),g,f(a,i)),
//   S123(n,i) = sum_{a,b} -B(n,a)A(a,b)B(b,i) M + A(n,a)B(a,b)B(b,i) I - B(n,a)B(a,b)A(b,i) K,
//   S67(n,i,g) = sum_a A(n,a) Q(a,i,g),  D(n,i) = -sum_a A(n,a) S123(a,i),
//   T(n,i;m,j) = A(j,m) S123(n,i) + B(j,m) S67(n,i,f(j,m))
//                - sum_b B(j,b) A(b,m) Q(n,i,f(j,b)) + d_jm D(n,i),
// with X = C + R, M = F(f(b,a),f(b,i),f(n,b)) - R(f(b,a),f(n,a),f(a,i)),
// I = F(f(a,n),f(b,i),f(n,b)), K = R(f(i,b),f(n,a),f(a,i)) (the E
// intermediate of k_l4f equals -S123, and its Wd equals Q).  The reverse
// walks these back: Tbar -> (S123bar, S67bar, Dbar, U = A^H-contracted
// Tbar) -> Qbar, S123bar -> slice and operator cotangents.  Every cotangent
// entry has one owner thread per stage that sums its terms in a fixed order
// (gathers over host-built term lists for the slices), so gradients are
// reproducible bit for bit.  Slice cotangents sit in LDS when 3 nf^3 fits,
// else in global memory.  Each block walks times blockIdx.x, blockIdx.x +
// gridDim.x, ... with its own scratch.
// ---------------------------------------------------------------------------
struct L4fAdjArgs {
    const double2* Lbar;  // [T][N^4]
    const double2* Fs;    // [T][nf3] forward slices
    const double2* Cs;
    const double2* Rs;
    const int* p2f;
    const double2* ops;
    int N, nf, num_ops;
    long nf3;
    long T;
    double2* sbar;        // [T][3][nf3], the entries of the lists below written
    double2* Abar;        // [T][num_ops][N^2]
    int lds_slices;
    int lds_tb;           // Tbar in LDS (else after U in the scratch)
    double2* scr;         // [gridDim.x][scr_per]
    long scr_per;         // 4 N^2 nf + 3 N^2 + N^4, + N^4 when !lds_tb, + nxp nf with xtab
    // Gather lists (host-built from the pair map) that give every cotangent
    // entry one owner thread summing its terms in a fixed order:
    // X-form pairs (x, z) with their (a, i, b, form) terms; F and R slice
    // targets with their (n, i, a, b, kind) terms.  Packed: 8 bits per index.
    const int* xp_xz;     // [nxp] x + z * 65536
    const int* xp_start;  // [nxp + 1]
    const int* xp_ent;    // a | i << 8 | b << 16 | form << 24
    int nxp;
    const int* f_tgt;     // [nft] slice index of F targets
    const int* f_start;   // [nft + 1]
    const int* f_ent;     // n | i << 8 | a << 16 | b << 24 (kind in bit 31)
    int nft;
    const int* r_tgt;     // [nrt] bit 31: no X-form pair writes this entry
    const int* r_start;
    const int* r_ent;
    int nrt;
    int parts;            // room for entry_parts in LDS
    const int* xtab;      // [nf * nf] x nf + z -> pair index (null: X read from the slices)
};

// LDS_SLICES: slice cotangents accumulate in LDS (else in global memory);
// LDS_TB: the N^4 Tbar tile sits in LDS (else in the workgroup's scratch,
// for N above 8 where it exceeds the 160 KiB of a CU).  Both are fixed per
// instantiation so every access has a known address space.
template <bool LDS_SLICES, bool LDS_TB, int BS>
__device__ __forceinline__ void l4f_adjoint_body(double2* sm, const L4fAdjArgs& A) {
    const int N = A.N, N2 = N * N, N4 = N2 * N2, nf = A.nf;
    const long N2nf = static_cast<long>(N2) * nf;
    double2* const scr0 = A.scr + static_cast<long>(blockIdx.x) * A.scr_per;
    double2* Tb = LDS_TB ? sm : scr0 + 4 * N2nf + 3 * N2 + N4;  // N^4
    double2* opsS = LDS_TB ? Tb + N4 : sm;              // num_ops N^2
    double2* Ab = opsS + A.num_ops * N2;                // num_ops N^2
    double2* part = A.parts ? Ab + A.num_ops * N2 : nullptr;                 // 2 BS
    double2* sb = Ab + A.num_ops * N2 + (A.parts ? 2 * BS : 0);              // 3 nf3 (LDS_SLICES)
    int* f = reinterpret_cast<int*>(sb + (LDS_SLICES ? 3 * A.nf3 : 0));
    for (int e = threadIdx.x; e < A.num_ops * N2; e += BS) opsS[e] = A.ops[e];
    for (int e = threadIdx.x; e < N2; e += BS) f[e] = A.p2f[e];
    double2* Q = scr0;                                  // Q(a,i,g) at a + i N + g N^2
    double2* S67 = Q + N2nf;
    double2* S67b = S67 + N2nf;
    double2* Qb = S67b + N2nf;
    double2* S123 = Qb + N2nf;                          // N^2
    double2* S123b = S123 + N2;
    double2* Db = S123b + N2;
    double2* U = Db + N2;                               // U(n,i,b,j) at (n + i N) + (b + j N) N^2
    double2* Xc = U + N4 + (LDS_TB ? 0 : N4);           // X at [g][pair] (xtab)
    const long nfl = nf;
    auto id3 = [nfl](int x, int y, int z) { return (static_cast<long>(x) * nfl + y) * nfl + z; };
    auto F2 = [f, N](int r, int c) { return f[r + c * N]; };
    for (long t = blockIdx.x; t < A.T; t += gridDim.x) {
        __syncthreads();
        const double2* Lb = A.Lbar + t * N4;
        for (int idx = threadIdx.x; idx < N4; idx += BS) {
            const int ru = idx % N2, cu = idx / N2;
            const int n = ru % N, i = ru / N, m = cu % N, j = cu / N;
            Tb[idx] = cadd(Lb[(n + m * N) + (i + j * N) * N2], cconj(Lb[(m + n * N) + (j + i * N) * N2]));
        }
        for (int e = threadIdx.x; e < A.num_ops * N2; e += BS) Ab[e] = make_double2(0.0, 0.0);
        if constexpr (LDS_SLICES)  // entries that no list writes
            for (long e = threadIdx.x; e < 3 * A.nf3; e += BS) sb[e] = make_double2(0.0, 0.0);
        __syncthreads();
        const double2* Fp = A.Fs + t * A.nf3;
        const double2* Cp = A.Cs + t * A.nf3;
        const double2* Rp = A.Rs + t * A.nf3;
        // X = C + R at (x, g, z): its row over g starts at xrow(x, z) with stride
        // xstep.  The sums below read every X several times in orders that
        // touch a line for each 16 bytes; with xtab they read the pairs
        // gathered once per time, in the order of the slices.
        const bool packed = A.xtab != nullptr;
        const long xstep = packed ? A.nxp : nfl;
        auto xrow = [&](int x, int z) { return packed ? static_cast<long>(A.xtab[x * nf + z]) : x * nfl * nfl + z; };
        auto xval = [&](long e) { return packed ? Xc[e] : cadd(Cp[e], Rp[e]); };
        if (packed) {
            for (int e = threadIdx.x; e < A.nxp * nf; e += BS) {
                const int xz = A.xp_xz[e % A.nxp];
                const long x = id3(xz & 65535, e / A.nxp, xz >> 16);
                Xc[e] = cadd(Cp[x], Rp[x]);
            }
            __syncthreads();
        }
        double2* sF = LDS_SLICES ? sb : A.sbar + t * 3 * A.nf3;
        double2* sC = sF + A.nf3;
        double2* sR = sC + A.nf3;
        for (int iA = 0; iA < A.num_ops; ++iA)
            for (int iB = 0; iB < A.num_ops; ++iB) {
                const double2* Ap = opsS + iA * N2;
                const double2* Bp = opsS + iB * N2;
                double2* AbA = Ab + iA * N2;
                double2* AbB = Ab + iB * N2;
                const bool first = iA == 0 && iB == 0;  // stores the slice cotangents that later pairs add to
#define AA(r, c) Ap[(r) + (c) * N]
#define BB(r, c) Bp[(r) + (c) * N]
#define TB(n, i, m, j) Tb[((n) + (i) * N) + ((m) + (j) * N) * N2]
                // 1: forward Q and S123
                for (long e = threadIdx.x; e < N2nf; e += BS) {
                    const int a = static_cast<int>(e % N), i = static_cast<int>((e / N) % N);
                    const int g = static_cast<int>(e / N2);
                    double2 y = make_double2(0.0, 0.0);
                    for (int b = 0; b < N; ++b) {
                        const long x1 = xrow(F2(b, a), F2(a, i)) + g * xstep, x2 = xrow(F2(i, b), F2(a, i)) + g * xstep;
                        y = cadd(y, cmul(cmul(AA(a, b), BB(b, i)), xval(x1)));
                        y = csub(y, cmul(cmul(BB(a, b), AA(b, i)), xval(x2)));
                    }
                    Q[e] = y;
                }
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& s, double2&) {
                        const int n = e % N, i = e / N;
                        for (int q = p; q < N2; q += np) {
                            const int a = q / N, b = q % N;
                            const double2 Mv = csub(Fp[id3(F2(b, a), F2(b, i), F2(n, b))],
                                                    Rp[id3(F2(b, a), F2(n, a), F2(a, i))]);
                            const double2 Iv = Fp[id3(F2(a, n), F2(b, i), F2(n, b))];
                            const double2 Kv = Rp[id3(F2(i, b), F2(n, a), F2(a, i))];
                            s = csub(s, cmul(cmul(cmul(BB(n, a), AA(a, b)), BB(b, i)), Mv));
                            s = cadd(s, cmul(cmul(cmul(AA(n, a), BB(a, b)), BB(b, i)), Iv));
                            s = csub(s, cmul(cmul(cmul(BB(n, a), BB(a, b)), AA(b, i)), Kv));
                        }
                    },
                    [&](int e, double2 s, double2) { S123[e] = s; });
                __syncthreads();
                // 2: S67; S123bar, Dbar, S67bar, U from Tbar; A-bar of the A(j,m) S123 term
                for (long e = threadIdx.x; e < N2nf; e += BS) {
                    const int n = static_cast<int>(e % N);
                    const long rest = e - n;
                    double2 s = make_double2(0.0, 0.0);
                    for (int a = 0; a < N; ++a) s = cadd(s, cmul(AA(n, a), Q[rest + a]));
                    S67[e] = s;
                    const int ni = static_cast<int>(e % N2), g = static_cast<int>(e / N2);
                    double2 sb7 = make_double2(0.0, 0.0);
                    for (int j = 0; j < N; ++j)
                        for (int m = 0; m < N; ++m)
                            if (F2(j, m) == g) sb7 = cadd(sb7, cmul(cconj(BB(j, m)), Tb[ni + (m + j * N) * N2]));
                    S67b[e] = sb7;
                }
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& s, double2& d) {
                        for (int q = p; q < N2; q += np) {  // q = m + j N
                            const int j = q / N, m = q % N;
                            const double2 tb = Tb[e + q * N2];
                            s = cadd(s, cmul(cconj(AA(j, m)), tb));
                            if (j == m) d = cadd(d, tb);
                        }
                    },
                    [&](int e, double2 s, double2 d) {
                        S123b[e] = s;
                        Db[e] = d;
                    });
                for (int e = threadIdx.x; e < N4; e += BS) {
                    const int r = e % N2, c = e / N2, b = c % N, j = c / N;
                    double2 s = make_double2(0.0, 0.0);
                    for (int m = 0; m < N; ++m) s = cadd(s, cmul(cconj(AA(b, m)), Tb[r + (m + j * N) * N2]));
                    U[e] = s;
                }
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& s, double2&) {
                        const int j = e % N, m = e / N;
                        for (int r = p; r < N2; r += np) s = cadd(s, cmul(cconj(S123[r]), Tb[r + (m + j * N) * N2]));
                    },
                    [&](int e, double2 s, double2) { AbA[e] = cadd(AbA[e], s); });
                __syncthreads();
                // 3: Qbar; S123bar gets the D term; operator cotangents of the S67,
                // Q and D terms of T and of S67 = A Q and D = -A S123
                for (long e = threadIdx.x; e < N2nf; e += BS) {
                    const int a = static_cast<int>(e % N), i = static_cast<int>((e / N) % N);
                    const int g = static_cast<int>(e / N2);
                    double2 s = make_double2(0.0, 0.0);
                    for (int n = 0; n < N; ++n) s = cadd(s, cmul(cconj(AA(n, a)), S67b[n + i * N + g * N2]));
                    for (int j = 0; j < N; ++j)
                        for (int b = 0; b < N; ++b)
                            if (F2(j, b) == g) s = csub(s, cmul(cconj(BB(j, b)), U[(a + i * N) + (b + j * N) * N2]));
                    Qb[e] = s;
                }
                for (int e = threadIdx.x; e < N2; e += BS) {
                    const int a = e % N, i = e / N;
                    double2 s = S123b[e];
                    for (int n = 0; n < N; ++n) s = csub(s, cmul(cconj(AA(n, a)), Db[n + i * N]));
                    S123b[e] = s;
                }
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& s, double2&) {
                        const int j = e % N, m = e / N;
                        const long go = static_cast<long>(F2(j, m)) * N2;
                        for (int r = p; r < N2; r += np) s = cadd(s, cmul(cconj(S67[go + r]), Tb[r + (m + j * N) * N2]));
                    },
                    [&](int e, double2 s, double2) { AbB[e] = cadd(AbB[e], s); });
                __syncthreads();
                // v(j,b,m) = sum_r conj(Q(r, f(j,b))) Tbar(r; m,j), in U's space (U is done)
                double2* V = U;
                for (int e = threadIdx.x; e < N2 * N; e += BS) {
                    const int j = e % N, m = e / N2;
                    const long go = static_cast<long>(F2(j, (e / N) % N)) * N2;
                    double2 v = make_double2(0.0, 0.0);
                    for (int r = 0; r < N2; ++r) v = cadd(v, cmul(cconj(Q[go + r]), Tb[r + (m + j * N) * N2]));
                    V[e] = v;
                }
                __syncthreads();
                // the B(j,b) A(b,m) Q term: each cotangent entry sums its v's in j (or m) order
                for (int e = threadIdx.x; e < N2; e += BS) {
                    const int b = e % N, m = e / N;
                    double2 s = make_double2(0.0, 0.0);
                    for (int j = 0; j < N; ++j) s = cadd(s, cmul(cconj(BB(j, b)), V[j + b * N + m * N2]));
                    AbA[b + m * N] = csub(AbA[b + m * N], s);
                }
                __syncthreads();
                for (int e = threadIdx.x; e < N2; e += BS) {
                    const int j = e % N, b = e / N;
                    double2 s = make_double2(0.0, 0.0);
                    for (int m = 0; m < N; ++m) s = cadd(s, cmul(cconj(AA(b, m)), V[j + b * N + m * N2]));
                    AbB[j + b * N] = csub(AbB[j + b * N], s);
                }
                __syncthreads();
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& s, double2&) {
                        const int n = e % N, a = e / N;
                        for (int q = p; q < N * nf; q += np)  // q = i + g N
                            s = cadd(s, cmul(cconj(Q[a + q * N]), S67b[n + q * N]));
                        for (int i = p; i < N; i += np) s = csub(s, cmul(cconj(S123[a + i * N]), Db[n + i * N]));
                    },
                    [&](int e, double2 s, double2) { AbA[e] = cadd(AbA[e], s); });
                __syncthreads();
                // 4: slice and operator cotangents of Q and of S123, each entry owned by
                // one thread that sums its terms in a fixed order (no atomics)
                // X = C + R slices: pair (x, z) and bucket g gather the Q-bar terms
                for (long e = threadIdx.x; e < static_cast<long>(A.nxp) * nf; e += BS) {
                    const int pp = static_cast<int>(e % A.nxp), g = static_cast<int>(e / A.nxp);
                    double2 acc = make_double2(0.0, 0.0);
                    for (int q = A.xp_start[pp]; q < A.xp_start[pp + 1]; ++q) {
                        const int w = A.xp_ent[q];
                        const int a = w & 255, i = (w >> 8) & 255, b = (w >> 16) & 255;
                        const double2 qb = Qb[a + i * N + g * N2];
                        if (w >> 24)
                            acc = csub(acc, cmul(cconj(cmul(BB(a, b), AA(b, i))), qb));
                        else
                            acc = cadd(acc, cmul(cconj(cmul(AA(a, b), BB(b, i))), qb));
                    }
                    const int xz = A.xp_xz[pp];
                    const long x = id3(xz & 65535, g, xz >> 16);
                    sC[x] = first ? acc : cadd(sC[x], acc);
                    sR[x] = first ? acc : cadd(sR[x], acc);
                }
                __syncthreads();
                // F and R slices of the M, I, K terms of S123
                for (int e = threadIdx.x; e < A.nft; e += BS) {
                    double2 acc = make_double2(0.0, 0.0);
                    for (int q = A.f_start[e]; q < A.f_start[e + 1]; ++q) {
                        const unsigned w = static_cast<unsigned>(A.f_ent[q]);
                        const int n = w & 255, i = (w >> 8) & 255, a = (w >> 16) & 255, b = (w >> 24) & 127;
                        const double2 sv = S123b[n + i * N];
                        if (w >> 31)  // +A(n,a) B(a,b) B(b,i) I
                            acc = cadd(acc, cmul(cconj(cmul(cmul(AA(n, a), BB(a, b)), BB(b, i))), sv));
                        else          // -B(n,a) A(a,b) B(b,i) M, M = F - R
                            acc = csub(acc, cmul(cconj(cmul(cmul(BB(n, a), AA(a, b)), BB(b, i))), sv));
                    }
                    sF[A.f_tgt[e]] = first ? acc : cadd(sF[A.f_tgt[e]], acc);
                }
                for (int e = threadIdx.x; e < A.nrt; e += BS) {
                    double2 acc = make_double2(0.0, 0.0);
                    for (int q = A.r_start[e]; q < A.r_start[e + 1]; ++q) {
                        const unsigned w = static_cast<unsigned>(A.r_ent[q]);
                        const int n = w & 255, i = (w >> 8) & 255, a = (w >> 16) & 255, b = (w >> 24) & 127;
                        const double2 sv = S123b[n + i * N];
                        if (w >> 31)  // -B(n,a) B(a,b) A(b,i) K
                            acc = csub(acc, cmul(cconj(cmul(cmul(BB(n, a), BB(a, b)), AA(b, i))), sv));
                        else          // the -R part of M
                            acc = cadd(acc, cmul(cconj(cmul(cmul(BB(n, a), AA(a, b)), BB(b, i))), sv));
                    }
                    const int x = A.r_tgt[e] & 0x7fffffff;
                    sR[x] = first && A.r_tgt[e] < 0 ? acc : cadd(sR[x], acc);
                }
                __syncthreads();
                auto Mv = [&](int n, int i, int a, int b) {
                    return csub(Fp[id3(F2(b, a), F2(b, i), F2(n, b))], Rp[id3(F2(b, a), F2(n, a), F2(a, i))]);
                };
                auto Iv = [&](int n, int i, int a, int b) { return Fp[id3(F2(a, n), F2(b, i), F2(n, b))]; };
                auto Kv = [&](int n, int i, int a, int b) { return Rp[id3(F2(i, b), F2(n, a), F2(a, i))]; };
                // operator entries at (a,b) of the Q and S123 terms
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& sa, double2& sbb) {
                        const int a = e % N, b = e / N;
                        for (int g = p; g < nf; g += np)  // a bucket's row of X serves every i
                            for (int i = 0; i < N; ++i) {
                                const int z = F2(a, i);
                                const double2 qb = Qb[a + i * N + g * N2];
                                sa = cadd(sa, cmul(cconj(cmul(BB(b, i), xval(xrow(F2(b, a), z) + g * xstep))), qb));
                                sbb = csub(sbb, cmul(cconj(cmul(AA(b, i), xval(xrow(F2(i, b), z) + g * xstep))), qb));
                            }
                        for (int q = p; q < N2; q += np) {  // q = i + n N
                            const int n = q / N, i = q % N;
                            const double2 sv = S123b[n + i * N];
                            sa = csub(sa, cmul(cconj(cmul(cmul(BB(n, a), BB(b, i)), Mv(n, i, a, b))), sv));
                            sbb = cadd(sbb, cmul(cconj(cmul(cmul(AA(n, a), BB(b, i)), Iv(n, i, a, b))), sv));
                            sbb = csub(sbb, cmul(cconj(cmul(cmul(BB(n, a), AA(b, i)), Kv(n, i, a, b))), sv));
                        }
                    },
                    [&](int e, double2 sa, double2 sbb) {
                        AbA[e] = cadd(AbA[e], sa);
                        AbB[e] = cadd(AbB[e], sbb);
                    });
                __syncthreads();
                // operator entries at (b,i)
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& sa, double2& sbb) {
                        const int b = e % N, i = e / N;
                        for (int g = p; g < nf; g += np)
                            for (int a = 0; a < N; ++a) {
                                const int z = F2(a, i);
                                const double2 qb = Qb[a + i * N + g * N2];
                                sbb = cadd(sbb, cmul(cconj(cmul(AA(a, b), xval(xrow(F2(b, a), z) + g * xstep))), qb));
                                sa = csub(sa, cmul(cconj(cmul(BB(a, b), xval(xrow(F2(i, b), z) + g * xstep))), qb));
                            }
                        for (int q = p; q < N2; q += np) {  // q = a + n N
                            const int n = q / N, a = q % N;
                            const double2 sv = S123b[n + i * N];
                            sbb = csub(sbb, cmul(cconj(cmul(cmul(BB(n, a), AA(a, b)), Mv(n, i, a, b))), sv));
                            sbb = cadd(sbb, cmul(cconj(cmul(cmul(AA(n, a), BB(a, b)), Iv(n, i, a, b))), sv));
                            sa = csub(sa, cmul(cconj(cmul(cmul(BB(n, a), BB(a, b)), Kv(n, i, a, b))), sv));
                        }
                    },
                    [&](int e, double2 sa, double2 sbb) {
                        AbA[e] = cadd(AbA[e], sa);
                        AbB[e] = cadd(AbB[e], sbb);
                    });
                __syncthreads();
                // operator entries at (n,a)
                entry_parts<BS>(
                    N2, part,
                    [&](int e, int p, int np, double2& sa, double2& sbb) {
                        const int n = e % N, a = e / N;
                        for (int q = p; q < N2; q += np) {  // q = b + i N
                            const int i = q / N, b = q % N;
                            const double2 sv = S123b[n + i * N];
                            sbb = csub(sbb, cmul(cconj(cmul(cmul(AA(a, b), BB(b, i)), Mv(n, i, a, b))), sv));
                            sa = cadd(sa, cmul(cconj(cmul(cmul(BB(a, b), BB(b, i)), Iv(n, i, a, b))), sv));
                            sbb = csub(sbb, cmul(cconj(cmul(cmul(BB(a, b), AA(b, i)), Kv(n, i, a, b))), sv));
                        }
                    },
                    [&](int e, double2 sa, double2 sbb) {
                        AbA[e] = cadd(AbA[e], sa);
                        AbB[e] = cadd(AbB[e], sbb);
                    });
                __syncthreads();
#undef AA
#undef BB
#undef TB
            }
        for (int e = threadIdx.x; e < A.num_ops * N2; e += BS) A.Abar[t * A.num_ops * N2 + e] = Ab[e];
        if constexpr (LDS_SLICES)
            for (long e = threadIdx.x; e < 3 * A.nf3; e += BS) A.sbar[t * 3 * A.nf3 + e] = sb[e];
    }
}

// Every entry is summed by one thread in a fixed order, so the block size
// only changes which thread owns it and the results are identical at any
// size.  Large N (d >= 12: tens of thousands of entries per time, scattered
// slice gathers) runs 1024 threads per time, whose sixteen waves per CU hide
// the gathers' latency (d = 16, 201 times: 11.5 ms); small N keeps 256 threads
// (d = 4, 4001 times: 0.28 ms; twice the time at 1024).
constexpr int kL4AdjBlockLarge = 1024;
constexpr int kL4AdjLargeN = 12;
// Slices of nf^3 values and more (nf >= 26: 0.28 MB and more each) exceed what
// the caches hold of a time: the reverse then gathers X once per time (d = 16,
// nf = 81: 13.5 -> 11.5 ms; nf = 19 to 27 the same either way).
constexpr std::size_t kL4AdjPackedNf3 = std::size_t{1} << 14;
template <int BS>
__global__ __launch_bounds__(BS) void k_l4f_adjoint(L4fAdjArgs A) {
    extern __shared__ double2 sm[];
    if (A.lds_tb) {
        if (A.lds_slices)
            l4f_adjoint_body<true, true, BS>(sm, A);
        else
            l4f_adjoint_body<false, true, BS>(sm, A);
    } else {
        if (A.lds_slices)
            l4f_adjoint_body<true, false, BS>(sm, A);
        else
            l4f_adjoint_body<false, false, BS>(sm, A);
    }
}

// ---------------------------------------------------------------------------
// F/C/R adjoint per triple (t < T), the reverse of k_combine and the
// convolutions of phases A-C.  With g1 = Gamma_i, g2 = Gamma_j,
// gm = Gamma_mirror(j), pp = exp(+i Omega t dt), pm = conj(pp), w = g1 pm:
//   F = w PF - convF,  PF = dt cumsum(gm pp),       convF = dt (w * gm)
//   C = w PC - convC,  PC = dt cumsum(conj(g2) pp), convC = dt (w * conj g2)
//   R = g1 P3 - P4,    P3 = dt cumsum(g2 pm),       P4 = dt cumsum(g1 g2 pm)
// (tcl4_kernels.cpp:105-175).  Only t < T enters, so the convolution
// adjoints are direct correlations over [0, T).  Per position p of the
// combine list the scratch holds 11 series of length T:
//   0 w, 1 Fbar, 2 Cbar, 3 wbar, 4 g1bar, 5 g2bar, 6 gmbar, 7..10 P-bars.
// ---------------------------------------------------------------------------
struct FcrAdjArgs {
    const double2* gamma;   // [nf][Nt]
    const double* omegas;
    const int* mirror;
    int nf;
    long Nt;
    double dt;
    long T;
    const int* job_tri;     // combine-list position -> triple
    const unsigned char* job_mask;
    long ncomb;
    const double2* sbar;    // [T][3][nf3]
    long nf3;
    double2* scr;           // [ncomb][11][T] (k_fcr_adj_short: [ncomb][3][T])
    double* om;             // [ncomb] Omega cotangent
    const double2* ph_tab;  // phase table of the forward pass (TACO_PHASE_LIBM) or null
    const int* job_row;
    long ph_len;
};

__device__ __forceinline__ double block_sum(double v, double* ws) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    double tot = 0.0;
    if (threadIdx.x == 0) tot = (ws[0] + ws[1]) + (ws[2] + ws[3]);
    return tot;  // valid in thread 0
}

// Forward prefix scans and reverse suffix scans of one triple.  The suffix
// pass takes the phases from the GM series, where the prefix pass leaves them.
// Latency bounds it (a workgroup's chain of loads, phases and block scans), so
// the registers are held to four waves per SIMD (d = 16, 201 times, 1.5e5
// triples: 6.6 -> 6.0 ms).
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_fcr_adj_scan(FcrAdjArgs P) {
    __shared__ double wsum[8][4];
    __shared__ double wred[4];
    const long p = blockIdx.x;
    const long tri = P.job_tri[p];
    const int mask = P.job_mask[p];
    int i, j, k;
    decode_triple(tri, P.nf, i, j, k);
    const double omega = (P.omegas[i] + P.omegas[j]) + P.omegas[k];
    const double2* prow = P.ph_tab ? P.ph_tab + static_cast<long>(P.job_row[p]) * P.ph_len : nullptr;
    const double2* g1 = P.gamma + static_cast<long>(i) * P.Nt;
    const double2* g2 = P.gamma + static_cast<long>(j) * P.Nt;
    const double2* gm = P.gamma + static_cast<long>(P.mirror[j]) * P.Nt;
    const long T = P.T;
    double2* S = P.scr + p * 11 * T;
    double2 *W = S, *FB = S + T, *CB = S + 2 * T, *WB = S + 3 * T, *G1 = S + 4 * T, *G2 = S + 5 * T,
            *GM = S + 6 * T, *PbF = S + 7 * T, *PbC = S + 8 * T, *Pb3 = S + 9 * T, *Pb4 = S + 10 * T;
    const double dt = P.dt;
    double carry[6] = {0, 0, 0, 0, 0, 0};
    for (long t0 = 0; t0 < T; t0 += kBlock) {
        const long t = t0 + threadIdx.x;
        const bool valid = t < T;
        double2 a1 = make_double2(0, 0), a2 = a1, a3 = a1;
        double2 pp = a1, pm = a1, x1 = a1, x2 = a1;
        if (valid) {
            pp = phase_plus(prow, t, omega, dt);
            pm = cconj(pp);
            x1 = g1[t];
            x2 = g2[t];
            a1 = cmul(gm[t], pp);
            a2 = cmul(cconj(x2), pp);
            a3 = cmul(x2, pm);
        }
        double v[6] = {a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
        double tot[6];
        block_scan_n<6>(v, wsum, tot);
        for (int q = 0; q < 6; ++q) {
            v[q] = v[q] + carry[q];
            carry[q] += tot[q];
        }
        if (!valid) continue;
        const double2 PF = make_double2(v[0] * dt, v[1] * dt);
        const double2 PC = make_double2(v[2] * dt, v[3] * dt);
        const double2 P3 = make_double2(v[4] * dt, v[5] * dt);
        const double2* sb = P.sbar + t * 3 * P.nf3;
        const double2 z = make_double2(0.0, 0.0);
        const double2 Fb = (mask & 1) ? sb[tri] : z;
        const double2 Cb = (mask & 2) ? sb[P.nf3 + tri] : z;
        const double2 Rb = (mask & 4) ? sb[2 * P.nf3 + tri] : z;
        const double2 w = cmul(x1, pm);
        GM[t] = pp;
        W[t] = w;
        FB[t] = Fb;
        CB[t] = Cb;
        WB[t] = cadd(cmul(Fb, cconj(PF)), cmul(Cb, cconj(PC)));
        G1[t] = cmul(Rb, cconj(P3));
        PbF[t] = cmul(Fb, cconj(w));
        PbC[t] = cmul(Cb, cconj(w));
        Pb3[t] = cmul(Rb, cconj(x1));
        Pb4[t] = make_double2(-Rb.x, -Rb.y);
    }
    __syncthreads();
    // suffix sums ybar_m = dt sum_{t >= m} Pbar_t, last chunk first
    double sc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double om_part = 0.0;
    const long nch = (T + kBlock - 1) / kBlock;
    for (long ch = nch - 1; ch >= 0; --ch) {
        const long t = ch * kBlock + (kBlock - 1 - threadIdx.x);
        const bool valid = t < T;
        double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (valid) {
            v[0] = PbF[t].x; v[1] = PbF[t].y; v[2] = PbC[t].x; v[3] = PbC[t].y;
            v[4] = Pb3[t].x; v[5] = Pb3[t].y; v[6] = Pb4[t].x; v[7] = Pb4[t].y;
        }
        double tot[8];
        block_scan_n<8>(v, wsum, tot);
        for (int q = 0; q < 8; ++q) {
            v[q] = v[q] + sc[q];
            sc[q] += tot[q];
        }
        if (!valid) continue;
        const double2 yF = make_double2(v[0] * dt, v[1] * dt), yC = make_double2(v[2] * dt, v[3] * dt);
        const double2 y3 = make_double2(v[4] * dt, v[5] * dt), y4 = make_double2(v[6] * dt, v[7] * dt);
        const double tdt = static_cast<double>(t) * dt;
        const double2 pp = GM[t], pm = cconj(pp);
        const double2 x1 = g1[t], x2 = g2[t], xm = gm[t];
        GM[t] = cmul(yF, cconj(pp));
        G2[t] = cadd(cadd(cmul(cconj(yC), pp), cmul(y3, pp)), cmul(y4, cconj(cmul(x1, pm))));
        G1[t] = cadd(G1[t], cmul(y4, cconj(cmul(x2, pm))));
        const double2 ppb = cadd(cmul(yF, cconj(xm)), cmul(yC, x2));
        const double2 pmb = cadd(cmul(y3, cconj(x2)), cmul(y4, cconj(cmul(x1, x2))));
        // d pp / d Omega = i t dt pp, d pm / d Omega = -i t dt pm
        const double2 dpp = make_double2(-tdt * pp.y, tdt * pp.x);
        const double2 dpm = make_double2(tdt * pm.y, -tdt * pm.x);
        om_part += (ppb.x * dpp.x + ppb.y * dpp.y) + (pmb.x * dpm.x + pmb.y * dpm.y);
    }
    const double tot = block_sum(om_part, wred);
    if (threadIdx.x == 0) P.om[p] = tot;
}

// Correlation adjoints of the two convolutions for one block of 256 lags u:
//   wbar_u  += dt sum_{t>=u} (-Fbar_t conj(gm_{t-u}) - Cbar_t g2_{t-u})
//   gmbar_u += dt sum_{t>=u} -Fbar_t conj(w_{t-u})
//   g2bar_u += conj(dt sum_{t>=u} -Cbar_t conj(w_{t-u}))
// Bound by FP64 operations: 16 fused multiply-adds per (t, u) pair (unfused
// products and sums took 32 and twice the time).
__global__ __launch_bounds__(kBlock) void k_fcr_adj_corr(FcrAdjArgs P) {
    __shared__ double2 fb[kBlock], cb[kBlock];
    __shared__ double2 wgm[2 * kBlock], wg2[2 * kBlock], ww[2 * kBlock];
    const long p = blockIdx.x;
    const int mask = P.job_mask[p];
    if (!(mask & 3)) return;
    const long tri = P.job_tri[p];
    int i, j, k;
    decode_triple(tri, P.nf, i, j, k);
    const double2* g2 = P.gamma + static_cast<long>(j) * P.Nt;
    const double2* gm = P.gamma + static_cast<long>(P.mirror[j]) * P.Nt;
    const long T = P.T;
    double2* S = P.scr + p * 11 * T;
    const double2 *W = S, *FB = S + T, *CB = S + 2 * T;
    double2 *WB = S + 3 * T, *G2 = S + 5 * T, *GM = S + 6 * T;
    const long ub0 = static_cast<long>(blockIdx.y) * kBlock;
    const long u = ub0 + threadIdx.x;
    double2 xw = make_double2(0, 0), xm = xw, xc = xw;
    for (long t0 = ub0; t0 < T; t0 += kBlock) {
        // window of lags d = t - u for t in [t0, t0 + 256), u in [ub0, ub0 + 256):
        // d in [t0 - ub0 - 255, t0 - ub0 + 255], stored at d - (t0 - ub0 - 255)
        const long dlo = t0 - ub0 - (kBlock - 1);
        for (int e = threadIdx.x; e < 2 * kBlock; e += kBlock) {
            const long d = dlo + e;
            const bool ok = d >= 0 && d < T;
            wgm[e] = ok ? gm[d] : make_double2(0, 0);
            wg2[e] = ok ? g2[d] : make_double2(0, 0);
            ww[e] = ok ? W[d] : make_double2(0, 0);
        }
        {
            const long t = t0 + threadIdx.x;
            fb[threadIdx.x] = t < T ? FB[t] : make_double2(0, 0);
            cb[threadIdx.x] = t < T ? CB[t] : make_double2(0, 0);
        }
        __syncthreads();
        if (u < T) {
            const int qlo = static_cast<int>(max(0L, u - t0));
            const int qhi = static_cast<int>(min(static_cast<long>(kBlock), T - t0));
            for (int q = qlo; q < qhi; ++q) {
                const int e = static_cast<int>(t0 + q - u - dlo);
                const double2 f = fb[q], c = cb[q];
                xw = cfma_conj(wgm[e], f, cfma(wg2[e], c, xw));
                xm = cfma_conj(ww[e], f, xm);
                xc = cfma_conj(ww[e], c, xc);
            }
        }
        __syncthreads();
    }
    if (u < T) {
        const double dt = P.dt;
        WB[u] = csub(WB[u], cscale(xw, dt));
        GM[u] = csub(GM[u], cscale(xm, dt));
        G2[u] = csub(G2[u], cconj(cscale(xc, dt)));
    }
}

// g1bar += wbar pp; Omega cotangent of w = g1 pm.
__global__ __launch_bounds__(kBlock) void k_fcr_adj_fin(FcrAdjArgs P) {
    __shared__ double wred[4];
    const long p = blockIdx.x;
    const long tri = P.job_tri[p];
    int i, j, k;
    decode_triple(tri, P.nf, i, j, k);
    const double omega = (P.omegas[i] + P.omegas[j]) + P.omegas[k];
    const double2* prow = P.ph_tab ? P.ph_tab + static_cast<long>(P.job_row[p]) * P.ph_len : nullptr;
    const double2* g1 = P.gamma + static_cast<long>(i) * P.Nt;
    const long T = P.T;
    double2* S = P.scr + p * 11 * T;
    const double2* WB = S + 3 * T;
    double2* G1 = S + 4 * T;
    double om_part = 0.0;
    for (long t = threadIdx.x; t < T; t += kBlock) {
        const double tdt = static_cast<double>(t) * P.dt;
        const double2 pp = phase_plus(prow, t, omega, P.dt), pm = cconj(pp);
        const double2 wb = WB[t];
        G1[t] = cadd(G1[t], cmul(wb, pp));
        const double2 pmb = cmul(wb, cconj(g1[t]));
        const double2 dpm = make_double2(tdt * pm.y, -tdt * pm.x);
        om_part += pmb.x * dpm.x + pmb.y * dpm.y;
    }
    const double tot = block_sum(om_part, wred);
    if (threadIdx.x == 0) P.om[p] += tot;
}

// Scan, correlations and final sums of one triple of at most kAdjShort times by
// one wave: lane l holds the times l + 64 r, the series that the correlations
// shift stay in LDS, and only the three Gamma cotangents go to memory (the
// three kernels above store and reload eleven series, and their correlations
// read five LDS values for 16 fused multiply-adds; here up to four times of a
// lane share the unshifted values, two of which are scalar loads).
// d = 16, 201 times, 1.5e5 triples: 11.5 -> 5.9 ms.  Longer runs, whose series
// would need more registers and LDS than a wave can have beside others, take
// the three kernels.
constexpr int kAdjShort = 256;

// Sum over the lanes up to (UP) or from this one, plus carry; carry takes the total.
template <bool UP, int Q>
__device__ __forceinline__ void wave_scan_n(double (&v)[Q], double (&carry)[Q]) {
    const int lane = threadIdx.x;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double nb = UP ? __shfl_up(v[q], off, 64) : __shfl_down(v[q], off, 64);
            if (UP ? lane >= off : lane + off < 64) v[q] += nb;
        }
        const double tot = __shfl(v[q], UP ? 63 : 0, 64);
        v[q] += carry[q];
        carry[q] += tot;
    }
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_fcr_adj_short(FcrAdjArgs P) {
    constexpr int R = kAdjShort / 64;
    __shared__ double2 fb[kAdjShort], cb[kAdjShort], ww[kAdjShort];
    const long p = blockIdx.x;
    const int lane = threadIdx.x, T = static_cast<int>(P.T), mask = P.job_mask[p];
    const long tri = P.job_tri[p];
    int i, j, k;
    decode_triple(tri, P.nf, i, j, k);
    const int mj = P.mirror[j];
    const double omega = (P.omegas[i] + P.omegas[j]) + P.omegas[k];
    const double2* prow = P.ph_tab ? P.ph_tab + static_cast<long>(P.job_row[p]) * P.ph_len : nullptr;
    const double2* g1 = P.gamma + static_cast<long>(i) * P.Nt;
    const double2* g2 = P.gamma + static_cast<long>(j) * P.Nt;
    const double2* gm = P.gamma + static_cast<long>(mj) * P.Nt;
    double2 *G1 = P.scr + p * 3 * T, *G2 = G1 + T, *GM = G2 + T;
    const double dt = P.dt;
    const double2 z = make_double2(0.0, 0.0);
    double2 pp[R], Rb[R], wb[R], g1b[R];
    double carry[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        pp[r] = Rb[r] = wb[r] = g1b[r] = z;
        if (64 * r >= T) continue;
        const int t = lane + 64 * r;
        const bool valid = t < T;
        double2 a1 = z, a2 = z, a3 = z, w = z, Fb = z, Cb = z;
        if (valid) {
            const double2* sb = P.sbar + static_cast<long>(t) * 3 * P.nf3;
            if (mask & 1) Fb = sb[tri];
            if (mask & 2) Cb = sb[P.nf3 + tri];
            if (mask & 4) Rb[r] = sb[2 * P.nf3 + tri];
            pp[r] = phase_plus(prow, t, omega, dt);
            const double2 pm = cconj(pp[r]), x2 = g2[t];
            a1 = cmul(gm[t], pp[r]);
            a2 = cmul(cconj(x2), pp[r]);
            a3 = cmul(x2, pm);
            w = cmul(g1[t], pm);
        }
        double v[6] = {a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
        wave_scan_n<true>(v, carry);
        const double2 PF = make_double2(v[0] * dt, v[1] * dt);
        const double2 PC = make_double2(v[2] * dt, v[3] * dt);
        const double2 P3 = make_double2(v[4] * dt, v[5] * dt);
        fb[t] = Fb;
        cb[t] = Cb;
        ww[t] = w;
        if (!valid) continue;
        wb[r] = cadd(cmul(Fb, cconj(PF)), cmul(Cb, cconj(PC)));
        g1b[r] = cmul(Rb[r], cconj(P3));
    }
    __syncthreads();
    // correlations over the lags e: time t = u + e for u = lane + 64 r
    double2 xw[R], xm[R], xc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) xw[r] = xm[r] = xc[r] = z;
    auto lags = [&](auto nr, int e0, int e1) {
        constexpr int NR = decltype(nr)::value;
        for (int e = e0; e < e1; ++e) {
            const double2 m = uload2(gm + e), q = uload2(g2 + e), w = ww[e];
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int t = lane + 64 * r + e;
                if (r + 1 < NR || t < T) {  // the blocks before the last one end below T
                    const double2 f = fb[t], c = cb[t];
                    xw[r] = cfma_conj(m, f, cfma(q, c, xw[r]));
                    xm[r] = cfma_conj(w, f, xm[r]);
                    xc[r] = cfma_conj(w, c, xc[r]);
                }
            }
        }
    };
    if (mask & 3) {
        lags(std::integral_constant<int, 4>{}, 0, T - 192);
        lags(std::integral_constant<int, 3>{}, max(0, T - 192), T - 128);
        lags(std::integral_constant<int, 2>{}, max(0, T - 128), T - 64);
        lags(std::integral_constant<int, 1>{}, max(0, T - 64), T);
    }
    // suffix sums ybar_m = dt sum_{t >= m} Pbar_t, and the results
    double sc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double om_part = 0.0, om_fin = 0.0;
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
        if (64 * r >= T) continue;
        const int t = lane + 64 * r;
        const bool valid = t < T;
        double2 x1 = z, x2 = z, xmir = z;
        if (valid) {
            x1 = g1[t];
            x2 = g2[t];
            xmir = gm[t];
        }
        const double2 Fb = fb[t], Cb = cb[t], w = ww[t], pm = cconj(pp[r]);
        const double2 pF = cmul(Fb, cconj(w)), pC = cmul(Cb, cconj(w)), p3 = cmul(Rb[r], cconj(x1));
        double v[8] = {pF.x, pF.y, pC.x, pC.y, p3.x, p3.y, -Rb[r].x, -Rb[r].y};
        wave_scan_n<false>(v, sc);
        if (!valid) continue;
        const double2 yF = make_double2(v[0] * dt, v[1] * dt), yC = make_double2(v[2] * dt, v[3] * dt);
        const double2 y3 = make_double2(v[4] * dt, v[5] * dt), y4 = make_double2(v[6] * dt, v[7] * dt);
        const double tdt = static_cast<double>(t) * dt;
        const double2 wbar = csub(wb[r], cscale(xw[r], dt));
        GM[t] = csub(cmul(yF, pm), cscale(xm[r], dt));
        G2[t] = csub(cadd(cadd(cmul(cconj(yC), pp[r]), cmul(y3, pp[r])), cmul(y4, cconj(cmul(x1, pm)))),
                     cconj(cscale(xc[r], dt)));
        G1[t] = cadd(cadd(g1b[r], cmul(y4, cconj(cmul(x2, pm)))), cmul(wbar, pp[r]));
        const double2 ppb = cadd(cmul(yF, cconj(xmir)), cmul(yC, x2));
        const double2 pmb = cadd(cmul(y3, cconj(x2)), cmul(y4, cconj(cmul(x1, x2)))), pmf = cmul(wbar, cconj(x1));
        // d pp / d Omega = i t dt pp, d pm / d Omega = -i t dt pm
        const double2 dpp = make_double2(-tdt * pp[r].y, tdt * pp[r].x);
        const double2 dpm = make_double2(tdt * pm.y, -tdt * pm.x);
        om_part += (ppb.x * dpp.x + ppb.y * dpp.y) + (pmb.x * dpm.x + pmb.y * dpm.y);
        om_fin += pmf.x * dpm.x + pmf.y * dpm.y;
    }
    for (int off = 32; off > 0; off >>= 1) {
        om_part += __shfl_down(om_part, off, 64);
        om_fin += __shfl_down(om_fin, off, 64);
    }
    if (lane == 0) P.om[p] = om_part + om_fin;
}

// Gamma cotangent per bucket: gbar[b][t] = sum over the bucket's entries
// (position, role) of the series g1bar, g2bar, gmbar (from series `first` of a
// position's `rows`), in list order.
// Per bucket b (blockIdx.y), its list of (position, role) entries in
// gridDim.z contiguous pieces: piece z (blockIdx.z) sums its entries in list
// order into part[(z nf + b) T + t]; k_bucket_reduce_pieces adds the pieces
// in order.  Enough workgroups to hide the gathers' latency (a bucket can
// hold thousands of entries), and a fixed order.
constexpr int kBredPieces = 32;
__global__ __launch_bounds__(kBlock) void k_bucket_reduce(const double2* scr, int rows, int first, long T,
                                                          const int* ent_start, const int* ent, double2* part) {
    const int b = blockIdx.y, nf = gridDim.y, z = blockIdx.z, P = gridDim.z;
    const long t = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= T) return;
    const long q0 = ent_start[b], len = ent_start[b + 1] - q0;
    const long lo = q0 + len * z / P, hi = q0 + len * (z + 1) / P;
    double2 s = make_double2(0.0, 0.0);
    for (long q = lo; q < hi; ++q) {
        const int code = ent[q];
        const long p = code / 3, role = first + code % 3;
        s = cadd(s, scr[(p * rows + role) * T + t]);
    }
    part[(static_cast<long>(z) * nf + b) * T + t] = s;
}

__global__ __launch_bounds__(kBlock) void k_bucket_reduce_pieces(const double2* part, long T, long Nt,
                                                                 double2* gbar) {
    const int b = blockIdx.y, nf = gridDim.y;
    const long t = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= T) return;
    double2 s = make_double2(0.0, 0.0);
    for (int z = 0; z < kBredPieces; ++z) s = cadd(s, part[(static_cast<long>(z) * nf + b) * T + t]);
    gbar[static_cast<long>(b) * Nt + t] = s;
}

// ---------------------------------------------------------------------------
// TCL2 generator adjoint, the reverse of k_tcl2 (generator.cpp:81-177 with
// diagonal channels).  With P = A masked to bucket b, AdA = P^H P,
// gam = 2 Re Gamma_b(t), S = Im Gamma_b(t) the forward adds per (operator,
// bucket) part gam K (K = dL/dgam, the dissipator direction) and the
// unitary part of H = diag(eps) + hermitize(sum S AdA).  Per time t
// (k_tcl2_adj_t, one workgroup each):
//   Hbar(p,q) = i sum_r Lbar[(r,p),(r,q)] - i sum_r Lbar[(q,r),(p,r)]
//   (row (r1,r2) = r1 N + r2), eps parts Re Hbar(n,n), X = (Hbar + Hbar^H)/2,
//   Gamma_b cotangent (2 sum_parts Re<Lbar,K>, sum_parts Re<X,AdA>).
// Time sums (k_tcl2_adj_w per chunk of times, k_tcl2_adj_wsum over chunks
// in order): W_b = sum_t gam_b Lbar(t), V_b = sum_t S_b X(t) and
// sum_t Re Hbar(n,n); the host forms the operator cotangents from them.
// ---------------------------------------------------------------------------
struct Tcl2AdjArgs {
    const double2* Lbar;   // [T][D^2]
    const double2* gamma;  // [nf][Nt]
    long Nt, T;
    const double2* K;      // [npart][D^2]
    const double2* AdA;    // [npart][N^2]
    const int* part_b;     // [npart] bucket of each part
    int npart, N, nf, order;
    double2* gbar;         // [nf][T]
    double2* X;            // [T][N^2]
    double* epsd;          // [T][N]
    int nchunk;
    long nout;             // nf D^2 + nf N^2 + N
    double2* part;         // [nchunk][nout]
    double2* wsum;         // [nout]: W_b, V_b, eps sums (in .x)
};

// Operator cotangent of every TCL2 part from the time sums W_b (D^2) and
// V_b (N^2) of its bucket: the transposes of the part's K and AdA = P^H P
// terms applied to W_b and V_b,
//   AdAbar(a, c) = V_b(a, c) - 1/2 sum_k W_b[(k N + a) + (k N + c) D]
//                            - 1/2 sum_k W_b[(c N + k) + (a N + k) D],
//   Pbar(x, y) = sum_{r,c} W_b[(r N + x) + (c N + y) D] P(r, c)
//              + sum_{r,c} conj(W_b[(x N + r) + (y N + c) D]) P(r, c)
//              + sum_r AdAbar(r, y) P(x, r) + sum_c conj(AdAbar(y, c)) P(x, c),
// written per part (the host adds Pbar where pair_to_freq = b).  One
// workgroup per part; N^2 <= 1024.
__global__ __launch_bounds__(kBlock) void k_tcl2_ops_parts(const double2* W, const double2* V, const double2* P,
                                                           const int* part_b, int N, double2* Pbar) {
    extern __shared__ double2 shp[];
    const int N2 = N * N, D = N2;
    const long D2 = static_cast<long>(D) * D;
    const long q = blockIdx.x;
    const int b = part_b[q];
    const double2* Wb = W + static_cast<long>(b) * D2;
    const double2* Vb = V + static_cast<long>(b) * N2;
    const double2* Pq = P + q * N2;
    double2* Ps = shp;        // [N2]
    double2* Ab = shp + N2;   // [N2] AdAbar
    for (int e = threadIdx.x; e < N2; e += kBlock) Ps[e] = Pq[e];
    for (int e = threadIdx.x; e < N2; e += kBlock) {
        const int a = e % N, cc = e / N;
        double2 v = Vb[e];
        for (int k = 0; k < N; ++k) v = csub(v, cscale(Wb[(k * N + a) + static_cast<long>(k * N + cc) * D], 0.5));
        for (int k = 0; k < N; ++k) v = csub(v, cscale(Wb[(cc * N + k) + static_cast<long>(a * N + k) * D], 0.5));
        Ab[e] = v;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < N2; e += kBlock) {
        const int x = e % N, y = e / N;
        double2 s = make_double2(0.0, 0.0);
        for (int c = 0; c < N; ++c)
            for (int r = 0; r < N; ++r) s = cadd(s, cmul(Wb[(r * N + x) + static_cast<long>(c * N + y) * D], Ps[r + c * N]));
        for (int c = 0; c < N; ++c)
            for (int r = 0; r < N; ++r)
                s = cadd(s, cmul(cconj(Wb[(x * N + r) + static_cast<long>(y * N + c) * D]), Ps[r + c * N]));
        for (int r = 0; r < N; ++r) s = cadd(s, cmul(Ab[r + y * N], Ps[x + r * N]));
        for (int c = 0; c < N; ++c) s = cadd(s, cmul(cconj(Ab[y + c * N]), Ps[x + c * N]));
        Pbar[q * N2 + e] = s;
    }
}

// K of every TCL2 part (d L / d gam_b for the part's masked operator P):
// K[(r1 N + r2) + (c1 N + c2) D] = conj(P(r1,c1)) P(r2,c2)
//   - [r1 = c1] AdA(r2,c2)/2 - [r2 = c2] AdA(c1,r1)/2.
// Grid: (element blocks of D^2, parts).
__global__ __launch_bounds__(kBlock) void k_tcl2_part_k(const double2* P, const double2* AdA, int N, double2* K) {
    const int N2 = N * N, D = N2;
    const long D2 = static_cast<long>(D) * D;
    const long e = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (e >= D2) return;
    const long q = blockIdx.y;
    const int row = static_cast<int>(e % D), col = static_cast<int>(e / D);
    const int r1 = row / N, r2 = row % N, c1 = col / N, c2 = col % N;
    const double2* Pq = P + q * N2;
    const double2* Aq = AdA + q * N2;
    double2 v = cmul(cconj(Pq[r1 + c1 * N]), Pq[r2 + c2 * N]);
    if (r1 == c1) v = csub(v, cscale(Aq[r2 + c2 * N], 0.5));
    if (r2 == c2) v = csub(v, cscale(Aq[c1 + r1 * N], 0.5));
    K[q * D2 + e] = v;
}

__global__ __launch_bounds__(kBlock) void k_tcl2_adj_t(Tcl2AdjArgs A) {
    __shared__ double wred[4];
    extern __shared__ double2 sh[];
    const int N = A.N, N2 = N * N, D = N2;
    const long D2 = static_cast<long>(D) * D;
    const long t = blockIdx.x;
    const double2* Lb = A.Lbar + t * D2;
    double2* Hb = sh;
    double2* Xb = sh + N2;
    for (int e = threadIdx.x; e < N2; e += kBlock) {
        const int p = e % N, q = e / N;
        double2 h = make_double2(0.0, 0.0);
        for (int r = 0; r < N; ++r) {
            const double2 a = Lb[(r * N + p) + static_cast<long>(r * N + q) * D];
            const double2 b = Lb[(q * N + r) + static_cast<long>(p * N + r) * D];
            h = cadd(h, make_double2(-a.y, a.x));  // + i a
            h = cadd(h, make_double2(b.y, -b.x));  // - i b
        }
        Hb[e] = h;
    }
    __syncthreads();
    for (int n = threadIdx.x; n < N; n += kBlock) A.epsd[t * N + n] = Hb[n + n * N].x;
    if (A.order == 0) return;
    for (int e = threadIdx.x; e < N2; e += kBlock) {
        const int r = e % N, c = e / N;
        const double2 x = cscale(cadd(Hb[e], cconj(Hb[c + r * N])), 0.5);
        Xb[e] = x;
        A.X[t * N2 + e] = x;
    }
    __syncthreads();
    // Gamma_b cotangent, imaginary part (the real part, 2 sum_parts
    // Re<Lbar,K>, comes from k_tcl2_adj_kdot and k_tcl2_adj_gam)
    for (int b = 0; b < A.nf; ++b) {
        double sp = 0.0;
        bool any = false;
        for (int pi = 0; pi < A.npart; ++pi) {
            if (A.part_b[pi] != b) continue;
            any = true;
            const double2* M = A.AdA + static_cast<long>(pi) * N2;
            for (int e = threadIdx.x; e < N2; e += kBlock) {
                const double2 x = Xb[e], m = M[e];
                sp += x.x * m.x + x.y * m.y;
            }
        }
        double sv = 0.0;
        if (any) sv = block_sum(sp, wred);
        if (threadIdx.x == 0) A.gbar[static_cast<long>(b) * A.T + t] = make_double2(0.0, sv);
    }
}

// G[pi][t] = sum_e Re(conj(K_pi[e]) Lbar_t[e]) over e-chunks (blockIdx.z), a
// product of [npart] x [T] over 2 D2 reals.  A workgroup forms 16 parts x 16
// times, each wave 8 x 8 of them: a lane takes every 64th entry, 16 loads for
// 128 fused multiply-adds into 64 sums (the four waves meet in L1), and the
// sums are halved over the lanes until lane q holds pair q.  The chunk sums
// land in part[(z npart + pi) T + t].  Bound by the reads of L2 (a row is read
// once per 16 rows of the other side).  d = 16, 81 parts, 201 times:
// 2.7 -> 0.30 ms (8 x 8 pairs a workgroup from LDS rows in one bank before).
constexpr int kKdTile = 16;       // parts and times of a workgroup
constexpr long kKdChunk = 4096;   // entries of a chunk
__global__ __launch_bounds__(kBlock) void k_tcl2_adj_kdot(const double2* K, const double2* Lbar, long D2, int npart,
                                                          long T, double* part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p0 = blockIdx.x * kKdTile + 8 * (wave & 1);
    const long t0 = static_cast<long>(blockIdx.y) * kKdTile + 8 * (wave >> 1);
    const long e0 = static_cast<long>(blockIdx.z) * kKdChunk, e1 = min(D2, e0 + kKdChunk);
    if (p0 >= npart || t0 >= T) return;
    const double2 *kr[8], *lr[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {  // rows past the end repeat the last one and are not stored
        kr[r] = K + static_cast<long>(min(p0 + r, npart - 1)) * D2;
        lr[r] = Lbar + min(t0 + r, T - 1) * D2;
    }
    double acc[64];
#pragma unroll
    for (int q = 0; q < 64; ++q) acc[q] = 0.0;
    for (long e = e0 + lane; e < e1; e += 64) {
        double2 k[8], l[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            k[r] = kr[r][e];
            l[r] = lr[r][e];
        }
#pragma unroll
        for (int q = 0; q < 64; ++q) acc[q] = fma(l[q % 8].y, k[q / 8].y, fma(l[q % 8].x, k[q / 8].x, acc[q]));
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1)
#pragma unroll
        for (int q = 0; q < m; ++q) {
            const bool up = lane & m;
            const double other = __shfl_xor(up ? acc[q] : acc[q + m], m, 64);
            acc[q] = (up ? acc[q + m] : acc[q]) + other;
        }
    const int pi = p0 + lane / 8;
    const long t = t0 + lane % 8;
    if (pi < npart && t < T) part[(static_cast<long>(blockIdx.z) * npart + pi) * T + t] = acc[0];
}

// gbar[b][t].x = 2 sum over the parts of bucket b (in order) of their
// chunk sums (in order).
__global__ __launch_bounds__(kBlock) void k_tcl2_adj_gam(const double* part, int npart, int nchunk, long T,
                                                         const int* part_b, double2* gbar) {
    const int b = blockIdx.y;
    const long t = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= T) return;
    double g = 0.0;
    for (int pi = 0; pi < npart; ++pi) {
        if (part_b[pi] != b) continue;
        for (int z = 0; z < nchunk; ++z) g += part[(static_cast<long>(z) * npart + pi) * T + t];
    }
    gbar[static_cast<long>(b) * T + t].x = 2.0 * g;
}

// Chunk sums over times of W_b, V_b and the eps parts (grid: outputs x chunks).
__global__ __launch_bounds__(kBlock) void k_tcl2_adj_w(Tcl2AdjArgs A) {
    const long o = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (o >= A.nout) return;
    const int N = A.N, N2 = N * N;
    const long D2 = static_cast<long>(N2) * N2;
    const long per = (A.T + A.nchunk - 1) / A.nchunk;
    const long t0 = blockIdx.y * per, t1 = min(A.T, t0 + per);
    double2 s = make_double2(0.0, 0.0);
    const long nW = A.nf * D2, nV = static_cast<long>(A.nf) * N2;
    if (o < nW) {
        if (A.order != 0) {
            const long b = o / D2, e = o % D2;
            for (long t = t0; t < t1; ++t)
                s = cadd(s, cscale(A.Lbar[t * D2 + e], 2.0 * A.gamma[b * A.Nt + t].x));
        }
    } else if (o < nW + nV) {
        if (A.order != 0) {
            const long b = (o - nW) / N2, e = (o - nW) % N2;
            for (long t = t0; t < t1; ++t) s = cadd(s, cscale(A.X[t * N2 + e], A.gamma[b * A.Nt + t].y));
        }
    } else {
        const long n = o - nW - nV;
        for (long t = t0; t < t1; ++t) s.x += A.epsd[t * N + n];
    }
    A.part[static_cast<long>(blockIdx.y) * A.nout + o] = s;
}

__global__ __launch_bounds__(kBlock) void k_tcl2_adj_wsum(Tcl2AdjArgs A) {
    const long o = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (o >= A.nout) return;
    double2 s = make_double2(0.0, 0.0);
    for (int c = 0; c < A.nchunk; ++c) s = cadd(s, A.part[static_cast<long>(c) * A.nout + o]);
    A.wsum[o] = s;
}

// ---------------------------------------------------------------------------
// Reverse of the bath chain in front of a tape whose Gamma table the device
// produced: Gamma_b(t_k) = (dt/2) sum_{m=1..k} (phi^{m-1} C_{m-1} + phi^m C_m),
// phi = exp(i w_b dt) (gamma.hpp:166-213), of C = (dw/pi) FFT(S), S the
// sampled KMS spectrum of J(w) (correlation_fft.hpp:154-214).  Every sum runs
// in a fixed order, so the cotangents repeat bit for bit.
// ---------------------------------------------------------------------------

// out = a + b elementwise (either may be null: that part is zero).
__global__ __launch_bounds__(kBlock) void k_gbar_sum(const double2* a, const double2* b, long n, double2* out) {
    const long i = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    double2 s = a ? a[i] : make_double2(0.0, 0.0);
    if (b) s = cadd(s, b[i]);
    out[i] = s;
}

// One workgroup per bucket b.  Gamma_b(k) weighs phi^m C_m by dt/2 for m = 0
// (k >= 1) and m = k, by dt for 0 < m < k, so its cotangent is (dt/2) Q_b(m)
// with Q(0) = sum_{k>=1} Gbar(k) and Q(m) = Gbar(m) + 2 sum_{k>m} Gbar(k).
// Writes Q_b [T] and omega_bar_b = (dt/2) Re sum_m conj(Q(m)) (i m dt) phi^m C_m.
// Each thread owns a contiguous run of m; the runs' suffix offsets come from
// one serial pass over the run totals.
__global__ __launch_bounds__(kBlock) void k_trapz_adj_q(const double2* gbar, long T, const double2* C, double dt,
                                                        const double* omegas, double2* Q, double* wbar) {
    __shared__ double2 part[kBlock];
    __shared__ double red[kBlock / 64];
    const int b = blockIdx.x;
    const double2* g = gbar + static_cast<long>(b) * T;
    double2* q = Q + static_cast<long>(b) * T;
    const long seg = (T + kBlock - 1) / kBlock;
    const long m0 = min(T, static_cast<long>(threadIdx.x) * seg), m1 = min(T, m0 + seg);
    double2 s = make_double2(0.0, 0.0);
    for (long m = m1 - 1; m >= m0; --m) s = cadd(s, g[m]);
    part[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double2 run = make_double2(0.0, 0.0);
        for (int i = kBlock - 1; i >= 0; --i) {
            const double2 p = part[i];
            part[i] = run;
            run = cadd(run, p);
        }
    }
    __syncthreads();
    double2 run = part[threadIdx.x];  // sum_{k >= m1} Gbar(k)
    const double w = omegas[b];
    double acc = 0.0;
    for (long m = m1 - 1; m >= m0; --m) {
        const double2 gm = g[m];
        const double2 qm = m == 0 ? run : make_double2(gm.x + 2.0 * run.x, gm.y + 2.0 * run.y);
        q[m] = qm;
        const double md = static_cast<double>(m) * dt;
        const double2 pc = cmul(cexpi(md * w), C[m]);  // phi^m C_m
        acc += md * (qm.y * pc.x - qm.x * pc.y);        // Re(conj(Q) i pc) m dt
        run = cadd(run, gm);
    }
    const double tot = block_sum(acc, red);
    if (threadIdx.x == 0) wbar[b] = 0.5 * dt * tot;
}

// x[m] = conj(C_bar(m)) for m < T, C_bar(m) = (dt/2) sum_b conj(phi_b^m) Q_b(m)
// (buckets in order), and 0 for T <= m < n: the input of the forward FFT that
// gives sum_m C_bar(m) exp(+2 pi i k m / n) as its conjugate.
__global__ __launch_bounds__(kBlock) void k_trapz_adj_c(const double2* Q, long T, int nf, double dt,
                                                        const double* omegas, long n, double2* x) {
    const long m = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (m >= n) return;
    double2 s = make_double2(0.0, 0.0);
    if (m < T) {
        const double md = static_cast<double>(m) * dt;
        for (int b = 0; b < nf; ++b) s = cadd(s, cmul(cconj(cexpi(md * omegas[b])), Q[static_cast<long>(b) * T + m]));
    }
    x[m] = make_double2(0.5 * dt * s.x, -(0.5 * dt * s.y));
}

struct BcfAdjArgs {
    const double2* spec;  // X[k] at ((k mod 2^a) << b) + (k >> a)
    int a, b;
    long nfft;
    double scale;         // dw / pi
    double domega, beta, p0, p1;
    int kind;
    double* part;         // [gridDim.x][3]
};

__device__ __forceinline__ double bcf_adj_sbar(const BcfAdjArgs& A, long k) {
    const long idx = ((k & ((1L << A.a) - 1)) << A.b) + (k >> A.a);
    return A.scale * A.spec[idx].x;
}

// J(w) and dJ/dp0, dJ/dp1 for w > 0.
__device__ __forceinline__ void spectral_J_grad(int kind, double p0, double p1, double w, double& J, double& d0,
                                                double& d1) {
    if (kind == 0) {  // p0 w exp(-w / p1)
        const double e = taco_cr::exp_cr(-w / p1, c_exptab);
        J = p0 * w * e;
        d0 = w * e;
        d1 = J * w / (p1 * p1);
    } else {  // 2 p0 p1 w / (w^2 + p1^2)
        const double den = w * w + p1 * p1;
        J = 2.0 * p0 * p1 * w / den;
        d0 = 2.0 * p1 * w / den;
        d1 = 2.0 * p0 * w * (w * w - p1 * p1) / (den * den);
    }
}

// Per k = 1..nfft/2-1 (a thread each): with Sbar = (dw/pi) Re X the spectrum
// cotangent, kms = exp(-beta w), f = (pi/2) / (1 - kms), S_k = f J and
// S_{nfft-k} = f J kms, the terms of dLoss/d(p0, p1, beta); per-workgroup
// sums (block_sum: a fixed shuffle tree) into part.
__global__ __launch_bounds__(kBlock) void k_bcf_adj_terms(BcfAdjArgs A) {
    __shared__ double red[kBlock / 64];
    constexpr double kPiD = 3.14159265358979323846;
    const long half = A.nfft / 2;
    const long k = 1 + static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    double g0 = 0.0, g1 = 0.0, gb = 0.0;
    if (k < half) {
        const double sk = bcf_adj_sbar(A, k), sm = bcf_adj_sbar(A, A.nfft - k);
        const double w = A.domega * static_cast<double>(k);
        double J, d0, d1;
        spectral_J_grad(A.kind, A.p0, A.p1, w, J, d0, d1);
        const double kms = taco_cr::exp_cr(-A.beta * w, c_exptab);
        const double f = (kPiD / 2.0) / (1.0 - kms);
        const double sp = f * J;
        const double dsp_db = (kPiD / 2.0) * J * (-w * kms) / ((1.0 - kms) * (1.0 - kms));
        g0 = sk * f * d0 + sm * f * kms * d0;
        g1 = sk * f * d1 + sm * f * kms * d1;
        gb = sk * dsp_db + sm * (dsp_db * kms + sp * (-w * kms));
    }
    g0 = block_sum(g0, red);
    g1 = block_sum(g1, red);
    gb = block_sum(gb, red);
    if (threadIdx.x == 0) {
        A.part[3L * blockIdx.x + 0] = g0;
        A.part[3L * blockIdx.x + 1] = g1;
        A.part[3L * blockIdx.x + 2] = gb;
    }
}

// out[0..2] = the workgroup sums in order; out[3] = Sbar_0, out[4] = Sbar_{nfft/2}.
__global__ void k_bcf_adj_final(BcfAdjArgs A, int nblocks, double* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int i = 0; i < nblocks; ++i) {
        s0 += A.part[3L * i + 0];
        s1 += A.part[3L * i + 1];
        s2 += A.part[3L * i + 2];
    }
    out[0] = s0;
    out[1] = s1;
    out[2] = s2;
    out[3] = bcf_adj_sbar(A, 0);
    out[4] = bcf_adj_sbar(A, A.nfft / 2);
}
