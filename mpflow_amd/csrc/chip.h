// On-chip PCG (chip.hip): whole solves of the meshes whose Krylov vectors fit one CU.
#pragma once

#include "jobs.h"

namespace mpf {

// A workgroup keeps one (job, harmonic) and a group of G right-hand-side lanes: p in LDS
// (80 KB), r, x and q in registers, K rows x G lanes per thread.
constexpr int kChipMaxRows = 20480;   // padded rows of the largest mesh (G = 1)
constexpr int kChipMaxWidth = 32;     // padded ELL width (2 bits of 8-slot groups)
constexpr int kChipCus = 256;         // one workgroup each

struct ChipShape {
    int G = 0, K = 0, threads = 0;
    bool hold = false;                // the matrix in registers (padded ELL width 8)
};
// The shape for np padded rows of `width` slots when a solve has `lanes` (job, harmonic, lane)
// triples in all.  Enough lanes to fill the chip: the largest group; fewer: the smallest group
// that keeps every workgroup on a CU of its own.
ChipShape chip_shape(int np, int width, long long lanes);

// Step k of a workgroup of nw wavefronts: the offset of its positions from those of step 0, 64 per
// wavefront.  K is rounded up to an instantiated kernel, so a wavefront's last steps may lie past the
// np rows; their loads, issued ahead of the gather's test, go to step 0's positions.  (As the scalar
// offset of a raw buffer load it is not part of the offset that the bounds check sees: a step past
// the table would read past it.)
__host__ __device__ constexpr int chip_step(int k, int wave, int nw, int np) {
    return (wave + k * nw) * 64 < np ? k * nw * 64 : 0;
}

// polls (about a microsecond each) after which a lane group gives up its wait for the deciding group
constexpr int kLeadPolls = 128;

// gst flags of a lane group
constexpr int kChipCapped = 1, kChipNan = 2, kChipEmpty = 4;

// pos -> row and row -> pos of the chip order: each tile's rows by their place in the node
// bisection (null: row order), 64 positions per aggregate
void launch_chip_order(int np, const uint8_t* tpos, uint16_t* rowof, uint16_t* posof, hipStream_t st);
// column positions of the ELL in chip order: [width / 8][np] x 8 ids of 16 bits; octs[np / 64]:
// 8-slot groups in use per 64 positions
void launch_chip_ids(int np, int width, const int32_t* ids, const uint8_t* gw, const uint16_t* rowof,
                     const uint16_t* posof, uint4* cid, uint8_t* octs, hipStream_t st);
// progress[0, nprogress) = 0, and the values S + alpha_c R of every (job, slice) pair of the
// list: J.cval [C][width / 8][2][np] float4
void launch_chip_pack(const JobDev* d_jobs, const int2* d_js, int njs, int max_np, int* progress, int nprogress,
                      hipStream_t st);
// one phase over `n` items (job, slice, lane group, index of the pair's first group state):
// phase 0 runs every lane group from its start to its own stop test -- under the reference rule
// to the step its pair's deciding group stops at, which that group publishes in progress (zeroed
// by launch_chip_pack; at the pair's first index; waited for `polls` polls a step) -- and phase 1
// takes the groups behind their pair's largest step count (gin) on to it.  gout receives every
// group's (steps, flags).
void launch_chip(const JobDev* d_jobs, const int4* d_items, int n, const ChipShape& c, const int2* gin, int2* gout,
                 int* progress, int polls, int phase, hipStream_t st);

}  // namespace mpf
