// group_fft.hip — phases B and C of the F/C/R passes on register groups.
//
// The forward FFT's last b stages and the inverse's first b stages of a
// residue group {k = k1 mod 2^a} are closed (engine.hip).  Here one workgroup
// of 2^b / 16 threads runs them with the group's values in registers, 16 per
// thread: three radix-2^r passes with two LDS exchanges, the forward values
// kept in registers for every product of the A-job, spectra and results
// straight between registers and memory.  Only the rows t mod 2^b < T of a
// half-inverse feed kept times, so a group writes min(T, 2^b) values and
// phase C combines 2^a of them per kept time.  Every butterfly is the
// reference's u +/- w*x with the stage's table twiddle, as in the tile
// kernels, so the values are bit-identical at every b.
//
// What bounds them (MI355X): phase B moves 5.5-6.2 TB/s past L2 at d = 4, Nfft 2^19
// (1.01 times the algorithmic bytes; a plain copy reaches 4.9), the vector units
// 49-52 % busy; at d = 8, Nfft 2^15, whose spectra stay in L2, 3.2 TB/s and 60 % busy
// (53 % with groups of 2^10): two waves per SIMD, since the forward values and a
// pass's twiddles take the registers of a third, at 1.8-1.9 GHz.  Phase C reads at
// 4.0-4.4 TB/s at d = 4, the rate of a plain copy, and 5.2 at d = 8.
#include "group_fft.hpp"

#include "cr_sincos.hpp"

#pragma clang fp contract(off)

namespace taco_engine {

// A group of 2^LG values on 2^LG / 16 threads (one or two waves, so the
// barriers cost little and four to eight groups share a CU; groups of 2^12
// and 2^13 measured 1.5 and 2 times slower per value).  The stages run as
// passes of radix 2^RL in registers with an LDS exchange between two passes.
template <int LG>
struct Group {
    static constexpr int kNV = 16;
    static constexpr int kNT = 1 << (LG - 4);
    static constexpr int kPass = 3;
    static constexpr int kLds = (1 << LG) + (1 << (LG - 4));  // a pad slot per 16 values
    static __host__ __device__ constexpr int rl(int p) { return p == 0 || (p == 1 && LG == 11) ? 4 : 3; }
    static __host__ __device__ constexpr int s_lo(int p) { return p == 0 ? 1 : s_lo(p - 1) + rl(p - 1); }
};

// base[idx] with a wave-uniform base and a 32-bit byte offset per lane: one
// offset register serves every access that differs by a uniform distance.
__device__ __forceinline__ double2 vload(const double2* base, unsigned idx) {
    return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(base) + idx * 16u);
}
__device__ __forceinline__ void vstore(double2* base, unsigned idx, double2 v) {
    *reinterpret_cast<double2*>(reinterpret_cast<char*>(base) + idx * 16u) = v;
}

__device__ __forceinline__ unsigned lds_at(unsigned pos) { return pos + (pos >> 4); }

// One pass: stages s_lo .. s_lo + RL - 1 (local, 1-based).  Set (k, u0) of a
// thread holds the values at u0 + (k R + m) 2^ub on entry (v[q R + m]) and
// those at u0 + (k + j 2^(s_lo-1)) 2^ub on return (v[q R + j]).
template <int LG, int P>
struct Pass {
    using G = Group<LG>;
    static constexpr int RL = G::rl(P), S = G::s_lo(P), R = 1 << RL, SETS = G::kNV / R;
    static constexpr int UB = LG - S - RL + 1;
    static __device__ __forceinline__ unsigned u0(int q) { return (threadIdx.x + q * G::kNT) & ((1u << UB) - 1); }
    static __device__ __forceinline__ unsigned k(int q) { return (threadIdx.x + q * G::kNT) >> UB; }
    // LDS slots of input m and output j of set q.  The m and j parts carry
    // into no bit of the set's own low four (2^ub > u0, and k R 2^ub or
    // 2^(s_lo-1+ub) clears them), so the padded slots add and the m and j
    // parts are constants.
    static __device__ __forceinline__ unsigned in_slot(int q, int m) {
        return lds_at(u0(q) + ((k(q) * R) << UB)) + lds_at(m << UB);
    }
    static __device__ __forceinline__ unsigned out_slot(int q, int j) {
        return lds_at(u0(q) + (k(q) << UB)) + lds_at(j << (S - 1 + UB));
    }

    static __device__ __forceinline__ void load_tw(double2 (&w)[SETS][R - 1], const double2* __restrict__ tw) {
#pragma unroll
        for (int q = 0; q < SETS; ++q)
#pragma unroll
            for (int i = 0; i < RL; ++i)
#pragma unroll
                for (int j = 0; j < (1 << i); ++j) {
                    const double2* base = tw + ((1 << (S + i - 1)) - 1 + (j << (S - 1)));
                    // pass 0 has k = 0: uniform twiddles
                    w[q][(1 << i) - 1 + j] = P == 0 ? uload2(base) : vload(base, k(q));
                }
    }
    template <bool CONJ>
    static __device__ __forceinline__ void butterflies(double2 (&v)[16], const double2 (&w)[SETS][R - 1], int q) {
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            const int h = R >> (i + 1);
            double2 y[R];
#pragma unroll
            for (int j = 0; j < (1 << i); ++j) {
                double2 t = w[q][(1 << i) - 1 + j];
                if (CONJ) t.y = -t.y;
#pragma unroll
                for (int m = 0; m < h; ++m) {
                    const double2 E = v[q * R + m + 2 * h * j];
                    const double2 x = cmul(t, v[q * R + m + h + 2 * h * j]);
                    y[m + h * j] = cadd(E, x);
                    y[m + h * j + R / 2] = csub(E, x);
                }
            }
#pragma unroll
            for (int m = 0; m < R; ++m) v[q * R + m] = y[m];
        }
    }
    // Output j = 0 alone (the others are past the kept rows).
    template <bool CONJ>
    static __device__ __forceinline__ void butterflies_first(double2 (&v)[16], const double2 (&w)[SETS][R - 1], int q) {
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            const int h = R >> (i + 1);
            double2 t = w[q][(1 << i) - 1];
            if (CONJ) t.y = -t.y;
#pragma unroll
            for (int m = 0; m < h; ++m) v[q * R + m] = cadd(v[q * R + m], cmul(t, v[q * R + m + h]));
        }
    }
};

// Passes P.. of a group FFT.  v holds pass P's inputs; returns the group in
// natural order, v[m] at threadIdx.x + m kNT.  need: positions at or above
// it are not read afterwards (each pass then runs only the sets that feed
// kept ones: a set of index k writes positions from k 2^ub on and reads the
// R 2^ub positions from k R 2^ub).
template <int LG, int P, bool CONJ>
__device__ __forceinline__ void group_passes(double2 (&v)[16], double2* buf, const double2* __restrict__ tw, unsigned need) {
    using G = Group<LG>;
    using A = Pass<LG, P>;
    constexpr bool last = P == G::kPass - 1;
    // Sets of this pass that are needed: walk the bound back from the last pass.
    unsigned kmax = 0;
    {
        unsigned bout = need;
#pragma unroll
        for (int p = G::kPass - 1; p >= P; --p) {
            const int ub = LG - G::s_lo(p) - G::rl(p) + 1;
            kmax = (bout + (1 << ub) - 1) >> ub;
            bout = min(kmax << (ub + G::rl(p)), 1u << LG);
        }
    }
    double2 w[A::SETS][A::R - 1];
    A::load_tw(w, tw);  // in flight over the barrier and the LDS reads
    if constexpr (P > 0) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < A::SETS; ++q)
            if (A::k(q) < kmax)
#pragma unroll
                for (int m = 0; m < A::R; ++m) v[q * A::R + m] = buf[A::in_slot(q, m)];
    }
#pragma unroll
    for (int q = 0; q < A::SETS; ++q)
        if (A::k(q) < kmax) {
            if (last && need <= (1u << (A::S - 1)))
                A::template butterflies_first<CONJ>(v, w, q);
            else
                A::template butterflies<CONJ>(v, w, q);
        }
    if constexpr (last) {
        // set q's output j sits at threadIdx.x + (q + SETS j) kNT
        double2 y[16];
#pragma unroll
        for (int q = 0; q < A::SETS; ++q)
#pragma unroll
            for (int j = 0; j < A::R; ++j) y[q + A::SETS * j] = v[q * A::R + j];
#pragma unroll
        for (int m = 0; m < 16; ++m) v[m] = y[m];
    } else {
        if constexpr (P > 0) __syncthreads();  // every read of this pass is done
#pragma unroll
        for (int q = 0; q < A::SETS; ++q)
            if (A::k(q) < kmax)
#pragma unroll
                for (int j = 0; j < A::R; ++j) buf[A::out_slot(q, j)] = v[q * A::R + j];
        group_passes<LG, P + 1, CONJ>(v, buf, tw, need);
    }
}

// Phase B of one A-job (or spectrum) and one group k1.  SPEC stores the
// forward group; otherwise every live (triple, path) of the A-job takes the
// product with its bucket spectrum (path 0, F: g_mirror(j); path 1, C:
// conj g_j) and the inverse's first b stages.  The forward values stay in
// registers for all of the A-job's products.
template <int LG, bool SPEC>
__global__ __launch_bounds__(Group<LG>::kNT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_group_b(FcrArgs P,
                                                                                                       long njobs) {
    using G = Group<LG>;
    constexpr int NT = G::kNT;
    __shared__ double2 buf[G::kLds];
    const int ngroups = 1 << P.a;
    int job, k1;
    if ((ngroups & 7) == 0) {
        // each XCD keeps a fixed eighth of the groups: its L2 holds their
        // twiddles and spectra
        xcd_map(blockIdx.x, ngroups, job, k1);
    } else {
        // each XCD keeps a contiguous eighth of the A-jobs (sorted by j)
        const long total = njobs << P.a, per = (total + 7) >> 3;
        const long lin = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if ((blockIdx.x >> 3) >= per || lin >= total) return;
        job = static_cast<int>(lin >> P.a);
        k1 = static_cast<int>(lin & (ngroups - 1));
    }
    if constexpr (!SPEC) job = uload(P.bperm + P.a0 + job) - static_cast<int>(P.a0);  // A-job within the chunk
    const long goff = static_cast<long>(k1) << LG;
    const double2* in = P.inter1 + static_cast<long>(job) * P.n + goff;
    double2 v[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) v[m] = vload(in + m * NT, threadIdx.x);
    const long bstride = (1L << LG) - 1;
    group_passes<LG, 0, false>(v, buf, P.twB + static_cast<long>(k1) * bstride, 1 << LG);
    if constexpr (SPEC) {
        double2* out = P.spec + static_cast<long>(job) * P.n + goff;
#pragma unroll
        for (int m = 0; m < 16; ++m) vstore(out + m * NT, threadIdx.x, v[m]);
        return;
    }
    double2 x[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) x[m] = v[m];
    const unsigned need = static_cast<unsigned>(P.Tq);
    const double inv_n = 1.0 / static_cast<double>(P.n);
    const int pend = uload(P.ajob_start + P.a0 + job + 1);
    for (int p = uload(P.ajob_start + P.a0 + job); p < pend; ++p) {
        int i, j, k;
        decode_triple(uload(P.job_tri + p), P.nf, i, j, k);
        const int bF = uload(P.mirror + j);
        const int mask = __builtin_amdgcn_readfirstlane(P.job_mask[p]);
        for (int path = 0; path < 2; ++path) {
            if (!(mask & (1 << path))) continue;
            const double2* sp = P.spec + static_cast<long>(path == 0 ? 2 * bF : 2 * j + 1) * P.n + goff;
#pragma unroll
            for (int m = 0; m < 16; ++m) v[m] = vload(sp + m * NT, threadIdx.x);
#pragma unroll
            for (int m = 0; m < 16; ++m) v[m] = cmul(x[m], v[m]);
            __syncthreads();  // the previous transform's LDS reads are done
            // loaded anew for every product: kept over the loop, the passes'
            // twiddles would take over 200 registers
            long zero = 0;
            asm volatile("" : "+s"(zero));
            group_passes<LG, 0, true>(v, buf, P.twStd + zero, need);
            if (P.a == 0) {  // the whole inverse: no phase C
                double2* out = P.conv + (path * P.cconv + (p - P.comb0)) * P.T;
#pragma unroll
                for (int m = 0; m < 16; ++m) {
                    const unsigned t = threadIdx.x + m * NT;
                    const double2 y = cscale(v[m], inv_n);
                    if (t < need) vstore(out + m * NT, threadIdx.x, make_double2(P.dt * y.x, P.dt * y.y));
                }
            } else {
                double2* out = P.inter2 + (((path * static_cast<long>(P.njobs) + (p - P.job0)) << P.a) + k1) * P.Tq;
#pragma unroll
                for (int m = 0; m < 16; ++m) {
                    const unsigned t = threadIdx.x + m * NT;
                    if (t < need) vstore(out + m * NT, threadIdx.x, v[m]);
                }
            }
        }
    }
}

template <int LG>
static void launch_group_b_lg(const FcrArgs& P, long njobs, bool spec, hipStream_t st) {
    const long total = njobs << P.a;
    const unsigned blocks = static_cast<unsigned>(P.a >= 3 ? total : ((total + 7) / 8) * 8);
    if (spec)
        hipLaunchKernelGGL((k_group_b<LG, true>), dim3(blocks), dim3(Group<LG>::kNT), 0, st, P, njobs);
    else
        hipLaunchKernelGGL((k_group_b<LG, false>), dim3(blocks), dim3(Group<LG>::kNT), 0, st, P, njobs);
}

void launch_group_b(const FcrArgs& P, long njobs, bool spec, hipStream_t st) {
    static_assert(kGroupBitsMin == 10 && kGroupBitsMax == 11, "one case per group size");
    if (P.b == 10)
        launch_group_b_lg<10>(P, njobs, spec, st);
    else
        launch_group_b_lg<11>(P, njobs, spec, st);
}

// Phase C on groups: the inverse's last a stages of the columns
// {t = q mod 2^b}, NP = ceil(T / 2^b) kept rows each, from the 2^a group
// values of a column.  A node of stage b + l is the DFT of the classes
// k1 = r mod 2^(a-l); its value at t is E +/- w O over the classes r and
// r + 2^(a-l) one stage below, w the stage's twiddle at t mod 2^(b+l-1).
// Only the values that feed kept times are formed: min(2^l, NP) per node.
//
// A thread runs the first four stages of one subtree of 16 classes in
// registers (16 reads in flight, coalesced over the columns); for a > 4 the
// 2^(a-4) subtrees of a column sit in one workgroup and finish through LDS,
// where every sign is + (2^4 >= NP).
template <int A1>
__global__ __launch_bounds__(A1 == 4 ? 1024 : 256) void k_group_c(FcrArgs P, int lgS, int lgQ, int NP) {
    constexpr int R = 1 << A1;
    extern __shared__ double2 nodes[];  // [2^lgS subtrees][NP][2^lgQ columns]
    const int jp = blockIdx.x, path = jp / P.njobs, job = jp % P.njobs;
    const int mask = P.job_mask[P.job0 + job];
    if (!(mask & (1 << path))) return;
    const int col = threadIdx.x & ((1 << lgQ) - 1), sub = threadIdx.x >> lgQ;
    const long q = (static_cast<long>(blockIdx.y) << lgQ) + col;
    const bool live = q < P.Tq;
    const long b2 = 1L << P.b;
    double2 v[R];
    if (live) {
        const double2* src = P.inter2 + ((static_cast<long>(jp) << P.a) + sub) * P.Tq + q;
        const long step = P.Tq << lgS;
#pragma unroll
        for (int m = 0; m < R; ++m) v[m] = src[m * step];
        // stage l: y[p] of node m from nodes m and m + R >> l, p < min(2^l, NP)
        // rows; node m's rows sit at v[m + (R >> l) p]
#pragma unroll
        for (int l = 1; l <= A1; ++l) {
            const int h = R >> l, rows = 1 << (l - 1);  // nodes after, rows per node before
            const double2* tw = P.twStd + (static_cast<long>(rows) << P.b) - 1;
            double2 y[R];
#pragma unroll
            for (int p = 0; p < rows; ++p) {
                if (p < NP) {
                    const double2 w = cconj(tw[q + p * b2]);
                    const bool hi = p + rows < NP;
#pragma unroll
                    for (int m = 0; m < h; ++m) {
                        const double2 E = v[m + 2 * h * p], x = cmul(w, v[m + h + 2 * h * p]);
                        y[m + h * p] = cadd(E, x);
                        if (hi) y[m + h * (p + rows)] = csub(E, x);
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < R; ++m) v[m] = y[m];
        }
    }
    const double inv_n = 1.0 / static_cast<double>(P.n);
    double2* out = P.conv + (path * P.cconv + (P.job0 + job - P.comb0)) * P.T;
    if (lgS == 0) {
        if (live)
#pragma unroll
            for (int p = 0; p < R; ++p) {
                const long t = q + p * b2;
                if (p < NP && t < P.T) {
                    const double2 y = cscale(v[p], inv_n);
                    out[t] = make_double2(P.dt * y.x, P.dt * y.y);
                }
            }
        return;
    }
    if (live)
#pragma unroll
        for (int p = 0; p < R; ++p)
            if (p < NP) nodes[((sub * NP + p) << lgQ) + col] = v[p];
    __syncthreads();
    const int rows = NP << lgQ;  // values per subtree
    const int nt = 1 << (lgS + lgQ);
    for (int l = 1; l <= lgS; ++l) {
        const int h = 1 << (lgS - l);  // nodes after this stage
        const double2* tw = P.twStd + (b2 << (A1 + l - 1)) - 1;
        for (int e = threadIdx.x; e < h * rows; e += nt) {
            const int m = e / rows, rest = e - m * rows;
            const long c = (static_cast<long>(blockIdx.y) << lgQ) + (rest & ((1 << lgQ) - 1));
            const long t = c + (rest >> lgQ) * b2;
            if (c >= P.Tq || t >= P.T) continue;
            const double2 E = nodes[e], x = cmul(cconj(tw[t]), nodes[e + h * rows]);
            const double2 y = cadd(E, x);
            if (l < lgS) {
                nodes[e] = y;
            } else {
                const double2 z = cscale(y, inv_n);
                out[t] = make_double2(P.dt * z.x, P.dt * z.y);
            }
        }
        __syncthreads();
    }
}

// Columns and subtrees of a workgroup: 256 threads, 32 columns (512 B runs)
// at least.
static int group_c_cols(int lgS) { return lgS <= 3 ? 8 - lgS : 5; }

bool group_c_fits(const FcrArgs& P) {
    const long NP = (P.T + (1L << P.b) - 1) >> P.b;
    if (P.a <= 4) return true;
    const int lgS = P.a - 4;
    return lgS <= 5 && NP <= 16 && (NP << (lgS + group_c_cols(lgS) + 4)) <= 64 * 1024;
}

void launch_group_c(const FcrArgs& P, hipStream_t st) {
    const int A1 = P.a < 4 ? P.a : 4, lgS = P.a - A1, lgQ = group_c_cols(lgS);
    const int NP = static_cast<int>((P.T + (1L << P.b) - 1) >> P.b);
    const std::size_t lds = lgS ? (static_cast<std::size_t>(NP) << (lgS + lgQ)) * sizeof(double2) : 0;
    const dim3 grid(static_cast<unsigned>(2 * P.njobs), static_cast<unsigned>((P.Tq + (1L << lgQ) - 1) >> lgQ));
    const dim3 block(1u << (lgS + lgQ));
    switch (A1) {
        case 0: hipLaunchKernelGGL(k_group_c<0>, grid, block, lds, st, P, lgS, lgQ, NP); break;
        case 1: hipLaunchKernelGGL(k_group_c<1>, grid, block, lds, st, P, lgS, lgQ, NP); break;
        case 2: hipLaunchKernelGGL(k_group_c<2>, grid, block, lds, st, P, lgS, lgQ, NP); break;
        case 3: hipLaunchKernelGGL(k_group_c<3>, grid, block, lds, st, P, lgS, lgQ, NP); break;
        default: hipLaunchKernelGGL(k_group_c<4>, grid, block, lds, st, P, lgS, lgQ, NP); break;
    }
}

// ---------------------------------------------------------------------------
// Phase A in registers: forward stages 1..a, a <= 8, of the columns
// {t = r mod 2^b}, a thread per column (a <= 4) or 2^(a-4) threads of 16
// values with one LDS exchange.  At most the lower half of a column is
// nonzero (Nin <= n / 2), so stage 1 copies and the upper half is never read.
// Consecutive threads hold consecutive columns: runs of 256 B and more both
// ways.
// ---------------------------------------------------------------------------
__constant__ double c_crtab_a[4 * taco_cr::kTabN];  // table of sincos_cr

hipError_t group_fft_set_table(const double* cr_tab) {
    return hipMemcpyToSymbol(HIP_SYMBOL(c_crtab_a), cr_tab, sizeof(double) * 4 * taco_cr::kTabN, 0,
                             hipMemcpyHostToDevice);
}

template <int A>
struct ColA {
    static constexpr int L1 = A < 4 ? A : 4;   // stages of pass 1
    static constexpr int L2 = A - L1;          // stages of pass 2 (0: none)
    static constexpr int V = 1 << L1;
    static constexpr int H = A == 0 ? 1 : V / 2;
    static constexpr int TPC = 1 << L2;        // threads per column
    static constexpr int COLS = 256 / TPC;     // columns of a workgroup
};

// The column's stages on x[0..H) (position u0 + m 2^L2, u0 = the thread's
// place in its column); stores out[k 2^b + r].
template <int A>
__device__ __forceinline__ void column_stages(double2 (&x)[ColA<A>::V], double2* buf, const double2* __restrict__ tw,
                                              double2* out, int b) {
    using C = ColA<A>;
    constexpr int V = C::V;
    // pass 1: stage 1 has a zero upper half, stages 2..L1 as in Pass (k = 0)
    if constexpr (A > 0) {
#pragma unroll
        for (int m = 0; m < V / 2; ++m) x[m + V / 2] = x[m];
#pragma unroll
        for (int i = 1; i < C::L1; ++i) {
            const int h = V >> (i + 1);
            double2 y[V];
#pragma unroll
            for (int j = 0; j < (1 << i); ++j) {
                const double2 t = uload2(tw + (1 << i) - 1 + j);
#pragma unroll
                for (int m = 0; m < h; ++m) {
                    const double2 E = x[m + 2 * h * j], z = cmul(t, x[m + h + 2 * h * j]);
                    y[m + h * j] = cadd(E, z);
                    y[m + h * j + V / 2] = csub(E, z);
                }
            }
#pragma unroll
            for (int m = 0; m < V; ++m) x[m] = y[m];
        }
    }
    if constexpr (C::L2 == 0) {
#pragma unroll
        for (int k = 0; k < V; ++k) out[static_cast<long>(k) << b] = x[k];
    } else {
        constexpr int R = C::TPC, SETS = 16 / R;
        const int col = threadIdx.x % C::COLS, u = threadIdx.x / C::COLS;
        __syncthreads();  // the previous column's reads are done
#pragma unroll
        for (int j = 0; j < 16; ++j) buf[(j * R + u) * C::COLS + col] = x[j];
        __syncthreads();
        // pass 2: sets k = u + R s of R positions k R + m, stages 5..a
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
            const int k = u + R * s;
            double2 v[R];
#pragma unroll
            for (int m = 0; m < R; ++m) v[m] = buf[(k * R + m) * C::COLS + col];
#pragma unroll
            for (int i = 0; i < C::L2; ++i) {
                const int h = R >> (i + 1);
                double2 y[R];
#pragma unroll
                for (int j = 0; j < (1 << i); ++j) {
                    const double2 t = tw[(16 << i) - 1 + k + 16 * j];
#pragma unroll
                    for (int m = 0; m < h; ++m) {
                        const double2 E = v[m + 2 * h * j], z = cmul(t, v[m + h + 2 * h * j]);
                        y[m + h * j] = cadd(E, z);
                        y[m + h * j + R / 2] = csub(E, z);
                    }
                }
#pragma unroll
                for (int m = 0; m < R; ++m) v[m] = y[m];
            }
#pragma unroll
            for (int j = 0; j < R; ++j) out[static_cast<long>(k + 16 * j) << b] = v[j];
        }
    }
}

// One workgroup per (Omega-class piece, columns): the phases of its columns
// are formed once and applied to the Gamma column g_i of every A-job of the
// piece inside the chunk.  SPEC: the spectra's inputs g_b (even job) and
// conj g_b (odd job) instead.
template <int A, bool SPEC>
__global__ __launch_bounds__(256) void k_column_a(FcrArgs P) {
    using C = ColA<A>;
    extern __shared__ double2 buf[];  // [2^A][COLS] when A > 4
    int cj, cb;
    xcd_map(blockIdx.x, ((1 << P.b) + C::COLS - 1) / C::COLS, cj, cb);
    const int u = threadIdx.x / C::COLS;
    const long r = static_cast<long>(cb) * C::COLS + threadIdx.x % C::COLS;
    const long stride = static_cast<long>(C::TPC) << P.b;       // between a thread's positions
    const long t0 = r + (static_cast<long>(u) << P.b);
    if constexpr (SPEC) {
        const double2* src = P.gamma + static_cast<long>(cj >> 1) * P.Nt;
        double2 x[C::V];
#pragma unroll
        for (int m = 0; m < C::H; ++m) {
            const long t = t0 + m * stride;
            x[m] = t < P.Nin ? src[t] : make_double2(0.0, 0.0);
            if (cj & 1) x[m].y = -x[m].y;
        }
        column_stages<A>(x, buf, P.twStd, P.inter1 + static_cast<long>(cj) * P.n + r, P.b);
    } else {
        const int cls = P.cls0 + cj;
        const long abeg = max(static_cast<long>(uload(P.cls_start + cls)), P.a0);
        const long aend = min(static_cast<long>(uload(P.cls_start + cls + 1)), P.a0 + P.na);
        if (abeg >= aend) return;
        const int pfirst = uload(P.ajob_start + abeg);
        int i, j, k;
        decode_triple(uload(P.job_tri + pfirst), P.nf, i, j, k);
        const double omega = (uload(P.omegas + i) + uload(P.omegas + j)) + uload(P.omegas + k);
        const double2* prow =
            P.ph_tab ? P.ph_tab + static_cast<long>(uload(P.job_row + pfirst)) * P.ph_len : nullptr;
        double2 ph[C::H];
        if (prow) {
#pragma unroll
            for (int m = 0; m < C::H; ++m) {
                const long t = t0 + m * stride;
                ph[m] = t < P.Nin ? cconj(prow[t]) : make_double2(0.0, 0.0);
            }
        } else {
#pragma unroll
            for (int m = 0; m < C::H; ++m) {
                const long t = t0 + m * stride;
                double s, c;
                taco_cr::sincos_cr(omega * (static_cast<double>(t) * P.dt), &s, &c, c_crtab_a);
                ph[m] = make_double2(c, -s);
            }
        }
        for (long aj = abeg; aj < aend; ++aj) {
            const int gi = uload(P.job_tri + uload(P.ajob_start + aj)) / (P.nf * P.nf);
            const double2* src = P.gamma + static_cast<long>(gi) * P.Nt;
            double2 x[C::V];
#pragma unroll
            for (int m = 0; m < C::H; ++m) {
                const long t = t0 + m * stride;
                x[m] = t < P.Nin ? cmul(src[t], ph[m]) : make_double2(0.0, 0.0);
            }
            column_stages<A>(x, buf, P.twStd, P.inter1 + (aj - P.a0) * P.n + r, P.b);
        }
    }
}

bool column_a_fits(const FcrArgs& P) {
    return P.a <= 8 && P.b >= 8 && 2 * P.Nin <= P.n;
}

template <int A>
static void launch_column_a_n(const FcrArgs& P, long njobs, bool spec, hipStream_t st) {
    using C = ColA<A>;
    const std::size_t lds = C::L2 ? (static_cast<std::size_t>(C::COLS) << A) * sizeof(double2) : 0;
    const dim3 grid(static_cast<unsigned>(njobs * ((1L << P.b) / C::COLS)));
    if (spec)
        hipLaunchKernelGGL((k_column_a<A, true>), grid, dim3(256), lds, st, P);
    else
        hipLaunchKernelGGL((k_column_a<A, false>), grid, dim3(256), lds, st, P);
}

void launch_column_a(const FcrArgs& P, long njobs, bool spec, hipStream_t st) {
    switch (P.a) {
        case 0: launch_column_a_n<0>(P, njobs, spec, st); break;
        case 1: launch_column_a_n<1>(P, njobs, spec, st); break;
        case 2: launch_column_a_n<2>(P, njobs, spec, st); break;
        case 3: launch_column_a_n<3>(P, njobs, spec, st); break;
        case 4: launch_column_a_n<4>(P, njobs, spec, st); break;
        case 5: launch_column_a_n<5>(P, njobs, spec, st); break;
        case 6: launch_column_a_n<6>(P, njobs, spec, st); break;
        case 7: launch_column_a_n<7>(P, njobs, spec, st); break;
        default: launch_column_a_n<8>(P, njobs, spec, st); break;
    }
}

}  // namespace taco_engine
