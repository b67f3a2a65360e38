// fcr_device.hpp — device helpers and kernel arguments shared by the F/C/R
// kernels (engine.hip, group_fft.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace taco_engine {

// Reads of kernel-constant data at a wave-uniform address, by scalar loads.
template <class T>
__device__ __forceinline__ T uload(const T* p) {
    return *(const __attribute__((address_space(4))) T*)(unsigned long)(p);
}
__device__ __forceinline__ double2 uload2(const double2* p) {
    const double* d = reinterpret_cast<const double*>(p);
    return make_double2(uload(d), uload(d + 1));
}

// ---------------------------------------------------------------------------
// Device helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
// s + a b and s + conj(a) b with fused multiply-adds.
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 s) {
    s.x = fma(a.x, b.x, s.x);
    s.x = fma(-a.y, b.y, s.x);
    s.y = fma(a.x, b.y, s.y);
    s.y = fma(a.y, b.x, s.y);
    return s;
}
__device__ __forceinline__ double2 cfma_conj(double2 a, double2 b, double2 s) {
    s.x = fma(a.x, b.x, s.x);
    s.x = fma(a.y, b.y, s.x);
    s.y = fma(a.x, b.y, s.y);
    s.y = fma(-a.y, b.x, s.y);
    return s;
}

// Block -> (job, group block).  Workgroups are dispatched to the 8 XCDs
// round-robin by id; when possible each XCD keeps a fixed eighth of the
// group blocks for every job, so its L2 holds only that eighth of the
// per-group twiddle tables.
__device__ __forceinline__ void xcd_map(int bid, int bpj, int& job, int& gb) {
    if ((bpj & 7) == 0) {
        const int x = bid & 7, i = bid >> 3, per = bpj >> 3;
        gb = x + 8 * (i % per);
        job = i / per;
    } else {
        job = bid / bpj;
        gb = bid % bpj;
    }
}

struct FcrArgs {
    const double2* gamma;   // [nf][Nt]
    const double* omegas;   // [nf]
    const int* mirror;      // [nf]
    int nf;
    long Nt;                // Gamma column stride
    long Nin;               // Gamma rows that enter the FFT inputs (Nt, or T in the window mode)
    double dt;
    int L, a, b;
    long n;
    const double2* twStd;   // every stage 1..L, stage-major: T_s[k] at 2^(s-1) - 1 + k
    const double2* twB;     // phase B forward stages, per k1 group
    const double2* twC;     // phase C inverse stages, per q group
    const int* job_tri;     // sorted position -> triple id (triples grouped by equal Omega)
    const unsigned char* job_mask;  // per sorted position: bit0 F needed, bit1 C needed, bit2 R needed
    long nfft_jobs;         // positions [0, nfft_jobs) need FFTs; the rest only R
    const int* ajob_start;  // [nA + 1] first sorted position of each A-job (the triples
                            // of one Omega class with the same i: identical phase-A input)
    const int* cls_start;   // [ncls + 1] first A-job of each Omega-class piece
    const int* bperm;       // phase B processing order: grid slot (per chunk) -> A-job
    long job0;              // first sorted position of the FFT chunk
    int njobs;              // triples in the FFT chunk
    long a0;                // first A-job of the FFT chunk
    int na;                 // A-jobs in the FFT chunk
    int cls0;               // first class piece touching the chunk
    long comb0;             // first sorted position of the combine batch
    long cconv;             // combine-batch capacity (conv slots)
    double2* inter1;        // [njobs][2^a][2^b]
    double2* inter2;        // [2][njobs][2^a][Tq]  half-inverse products, rows t mod 2^b < Tq
    long Tq;                // min(T, 2^b): the rows of a group that feed kept times
    double2* spec;          // [2 nf][2^a][2^b]   spectra of g_b (even) and conj(g_b) (odd)
    double2* conv;          // [2][njobs][T]
    long T;
    // Phase mode TACO_PHASE_LIBM: host table of exp(+i Omega (t dt)), one row
    // of ph_len values per distinct Omega, and the row of each sorted
    // position; null in TACO_PHASE_CR (the kernels evaluate cexpi).
    const double2* ph_tab;
    const int* job_row;
    long ph_len;
};

__device__ __forceinline__ void decode_triple(long tri, int nf, int& i, int& j, int& k) {
    k = static_cast<int>(tri % nf);
    j = static_cast<int>((tri / nf) % nf);
    i = static_cast<int>(tri / (static_cast<long>(nf) * nf));
}

}  // namespace taco_engine
