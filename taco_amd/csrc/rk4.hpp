// rk4.hpp — kernel arguments and launches of the RK4 recursions and their
// reverse (rk4.hip).
#pragma once

#include "fcr_device.hpp"

namespace taco_engine {

constexpr int kRkBlock = 256;  // threads of the general RK4 kernels

// Largest RK4 workgroup: the row-group path at D = 64.
constexpr int kRkBlockMax = 512;

// LDS of the RK4 workgroups: vectors of D, then generators staged nstage at
// a time (column stride D + 1) within the 160 KiB of a CU.
constexpr std::size_t kRkLds = 160 * 1024;

// L0 cotangent parts a thread of the reverse walk carries in registers.
constexpr int kRkCarry = 16;

template <int DT>
struct RowGroup {
    static constexpr int G = DT <= 16 ? 4 : 8;   // lanes per output element
    static constexpr int R = 64 / G;             // output elements per wave
    static constexpr int W = (DT + R - 1) / R;   // waves
    static constexpr int CK = (DT + G - 1) / G;  // terms per lane
    static constexpr int S = DT <= 16 ? 4 : 3;   // generator ring slots (forward)
    static constexpr int SA = 3;                 // ring slots of the reverse walk
};

// Threads of a row-group workgroup for D (0 when D has no row-group path).
__host__ __device__ constexpr int rk4_rows_threads(int D) {
    return D == 4 ? 64 * RowGroup<4>::W
         : D == 9 ? 64 * RowGroup<9>::W
         : D == 16 ? 64 * RowGroup<16>::W
         : D == 25 ? 64 * RowGroup<25>::W
         : D == 36 ? 64 * RowGroup<36>::W
         : D == 49 ? 64 * RowGroup<49>::W
         : D == 64 ? 64 * RowGroup<64>::W
         : 0;
}

// Many independent systems, one workgroup each, in a single launch.
struct Rk4Sys {
    const double2* Ls;   // [steps + 1][D x D]
    int nstage;          // generators staged in LDS at a time (0: read from global)
    const double2* r0;   // [D]
    double2* r;          // [D] final vector
    double2* samples;    // [steps + 1][D]
    long steps;
    double dt;
    int D;
    const double2* Lh = nullptr;  // [steps][D x D] given midpoints, else formed on the fly
    double2* q = nullptr;         // chunked run: [chunks][D x D] products, null: one sequential run
    double2* xs = nullptr;        // chunked run: [chunks][D] first states; wide run: kRkWideVecs x D
    int* plain = nullptr;         // chunked run: [chunks] whether a chunk is stepped (chunk_mild)
    long every = 1;               // sample distance
    long* nsamples = nullptr;
};

struct Rk4AdjArgs {
    const double2* Ls;    // [steps + 1][D * D] generators
    const double2* ck;    // [ceil(steps / K)][D] checkpoint states r_{qK}
    const double2* gbar;  // [steps + 1][D] dLoss/dr_n
    double2* Lbar;        // [steps + 1][D * D]
    double2* seg;         // [steps][4][D] state r_n and stage points u1, u2, u3 of step n
    double2* r0bar;       // [D]
    long steps;
    int D;
    int K;
    double dt;
    int nstage;
    double2* vec = nullptr;        // [steps][4][D] kb1..kb4 of every step (Lbar formed by k_rk4_lbar)
    double2* q = nullptr;          // chunked walk: [chunks][D * D] products,
    double2* lam = nullptr;        // [chunks][D] lam after each chunk's last step (wide walk: kRkWideVecs x D),
    double2* bv = nullptr;         // [chunks][D] constant parts
    int* plain = nullptr;          // [chunks] whether a chunk is stepped (chunk_mild)
};

// Steps of a chunk of the chunked runs.
constexpr int kRkChunk = 16;

// Whether a run of `steps` steps at D is chunked (rk4.hip).  The chunked run
// costs five or six launches and 2 kRkChunk steps of latency whatever its
// length; below 256 steps the plain run (0.5-0.7 us a step at D <= 16) is as
// fast.  At D = 36 the products alone take 0.39 ms, and 320 steps it is (a call
// of 256, 288, 320, 384 and 448 steps: 0.74, 0.78, 0.82, 0.89 and 0.96 ms against
// 0.70, 0.78, 0.86, 1.01 and 1.16 plain).  The reverse has row groups for D <= 16 only.
inline bool rk4_chunked(int D, long steps) {
    return D == 36 ? steps >= 320 : steps >= 256 && (D == 4 || D == 9 || D == 16 || D == 25);
}
inline bool rk4_chunked_walk(int D, long steps) { return D <= 16 && rk4_chunked(D, steps); }
// A chunked run's products, first states (or lam) and flags, in that order, and
// the complex values they take.
inline std::size_t rk4_chunks(long steps) { return static_cast<std::size_t>((steps + kRkChunk - 1) / kRkChunk); }
inline std::size_t rk4_chunk_values(int D, long steps) {
    const std::size_t nch = rk4_chunks(steps);
    return nch * (static_cast<std::size_t>(D) * D + D) + (nch + 3) / 4;
}
inline void rk4_place_chunks(int D, long steps, double2* base, double2*& q, double2*& x, int*& plain) {
    const std::size_t nch = rk4_chunks(steps);
    q = base;
    x = q + nch * D * D;
    plain = reinterpret_cast<int*>(x + nch * D);
}

// Whether runs at D are wide (rk4.hip): two generators do not fit the LDS
// beside the vectors, so one workgroup would read every product's generator
// from memory (D = 256: 18 us a product; a wide product takes 4 us for one
// system or four, and 300 steps gain 1.3 ms at D = 81, 4 ms at D = 144).
inline bool rk4_wide(int D) {
    return D > 64 && (6 * static_cast<std::size_t>(D) + 2 * static_cast<std::size_t>(D) * (D + 1)) * 16 > kRkLds;
}
constexpr int kRkWideVecs = 7;

// Raises the kernels' dynamic LDS limit to kRkLds on the current device.
hipError_t rk4_set_lds_limits();

// One system, row-group path (rk4_rows_threads(D) > 0).
void launch_rk4_rows(int D, const double2* Ls, long steps, double2* r, double dt, long every, double2* samples,
                     long* nsamples, hipStream_t st);
// One system, general path.
void launch_rk4(int D, const double2* Ls, const double2* Lh, long steps, double2* r, double dt, long every,
                double2* samples, long* nsamples, int nstage, int block, std::size_t lds, hipStream_t st);
// nsys systems, one workgroup each.
void launch_rk4_batch(unsigned nsys, const Rk4Sys* sys, int block, std::size_t lds, hipStream_t st);
// Chunked runs of the systems with q set and this D: `one`, or nsys of them on
// the device (arr), of at most max_steps steps; and the chunked walk of `one`
// tape or ntapes tapes.
void launch_rk4_chunked(int D, const Rk4Sys* arr, const Rk4Sys& one, unsigned nsys, long max_steps, hipStream_t st);
void launch_rk4_chunked_walk(int D, const Rk4AdjArgs* arr, const Rk4AdjArgs& one, unsigned ntapes, long steps,
                             hipStream_t st);
// Wide runs (rk4_wide) of `one` or nsys systems of this D (arr), and the
// recompute and walk of `one` tape or ntapes tapes of this D, steps and K.
void launch_rk4_wide(int D, const Rk4Sys* arr, const Rk4Sys& one, unsigned nsys, long max_steps, hipStream_t st);
void launch_rk4_wide_reverse(int D, const Rk4AdjArgs* arr, const Rk4AdjArgs& one, unsigned ntapes, long steps, int K,
                             hipStream_t st);

// Reverse of one tape (A) or of ntapes tapes of one D, steps and K (As on
// the device): the segments' recompute, the walk, the generator cotangents.
void launch_rk4_recompute(const Rk4AdjArgs& A, bool rows, unsigned nseg, std::size_t lds, hipStream_t st);
void launch_rk4_walk(const Rk4AdjArgs& A, bool rows, std::size_t lds, hipStream_t st);
void launch_rk4_lbar(const Rk4AdjArgs& A, hipStream_t st);
void launch_rk4_recompute_multi(const Rk4AdjArgs* As, unsigned ntapes, int D, bool rows, unsigned nseg,
                                std::size_t lds, hipStream_t st);
void launch_rk4_walk_multi(const Rk4AdjArgs* As, unsigned ntapes, int D, bool rows, std::size_t lds, hipStream_t st);
void launch_rk4_lbar_multi(const Rk4AdjArgs* As, unsigned ntapes, int D, long steps, hipStream_t st);

}  // namespace taco_engine
