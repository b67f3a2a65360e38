// group_fft.hpp — launches of the one-workgroup-per-group FFT kernels
// (group_fft.hip) of the F/C/R passes.
#pragma once

#include "fcr_device.hpp"

namespace taco_engine {

constexpr int kGroupBitsMin = 10;  // groups of 2^10 or 2^11 values
constexpr int kGroupBitsMax = 11;
constexpr int kTileBitsMax = 11;   // columns of at most 2^11 classes (phases A and C)

// Copies the table of sincos_cr (cr_sincos.hpp) to the current device.
hipError_t group_fft_set_table(const double* cr_tab);

// Phase A of njobs Omega-class pieces (spec false) or spectra (spec true) on
// registers; column_a_fits: at most 2^8 classes, the input's upper half zero.
bool column_a_fits(const FcrArgs& P);
void launch_column_a(const FcrArgs& P, long njobs, bool spec, hipStream_t st);

// Phase B on groups of 2^P.b values, kGroupBitsMin <= P.b <= kGroupBitsMax:
// njobs A-jobs of the chunk (spec false) or spectra (spec true).
void launch_group_b(const FcrArgs& P, long njobs, bool spec, hipStream_t st);

// Phase C on registers (and LDS past 2^4 classes), whatever phase B ran;
// group_c_fits: its LDS holds the kept rows.
bool group_c_fits(const FcrArgs& P);
void launch_group_c(const FcrArgs& P, hipStream_t st);

}  // namespace taco_engine
