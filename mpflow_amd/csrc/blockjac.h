// Block-diagonal part of the two-level preconditioner (blockjac.hip).
#pragma once

#include "jobs.h"

namespace mpf {

// floats of the inverse blocks of C harmonics on np rows
inline size_t block_inverse_floats(int C, int np) { return (size_t)C * np * kBlkRows; }
// inverse blocks of one mesh (job 0 of the table: its pattern and gather plan at sigma = 1) for
// every harmonic; *bad is set when a block is not positive definite
void launch_block_inverse(const JobDev* d_jobs, int C, int np, float* bloc, int* bad, hipStream_t st);

// The PCG start and update of the listed jobs that have inverse blocks (lane count 2^lg), as k_pcg_init and
// k_pcg_update4: the update leaves z = D^-1/2 B D^-1/2 r in q (A p is not needed any more).
void launch_block_init(const JobDev* d_jobs, const int4* d_tiles, int ntiles, int lg, hipStream_t st);
void launch_block_update(const JobDev* d_jobs, const int4* d_tiles, int ntiles, int iter, int lg, hipStream_t st);

}  // namespace mpf
