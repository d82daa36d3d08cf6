// firk_layout.h -- where the FIRK kernels keep per-interval data.  Plain C++ (the device
// qualifiers aside), shared by the kernels, the host code that sizes the areas, and the host checks.
//
// A wave's lanes own contiguous chunks of an instance's intervals; interval k is the i-th of
// its lane.  Field q of it lies 64 values after field q - 1, and the 64 lanes of a step side by
// side, so that lanes walking their chunks read and write whole 512-byte lines.  (In
// [interval][field] order every access of the wave touched 64 lines.)  An area holds whole
// lines; instances of at most 32 intervals, one per lane, share them.
#pragma once

#include <cstddef>

#ifdef __HIP__
#include <hip/hip_runtime.h>
#define FIRK_HD __host__ __device__ __forceinline__
#else
#define FIRK_HD inline
#endif

namespace bvpdev {

// most intervals of an instance of at most cap nodes; intervals in whole lines
FIRK_HD size_t firk_intervals(int cap) { return cap > 1 ? (size_t)cap - 1 : 1; }
FIRK_HD size_t firk_lines(size_t intervals) { return (intervals + 63) & ~(size_t)63; }

// offset of field 0 of step i of a lane in an area of nf fields (field q: + q * 64)
FIRK_HD size_t firk_cell(int lane, int i, int nf) { return (size_t)i * ((size_t)nf * 64) + lane; }

// instance b's first value in the batch's area of nf fields, and that area's size
FIRK_HD size_t firk_stage_base(size_t b, int cap, int nf) {
    const size_t L = firk_intervals(cap);
    if (L > 32) return b * firk_lines(L) * nf;
    const size_t G = 64 / L;
    return b / G * 64 * nf + b % G * L;
}
FIRK_HD size_t firk_stage_values(size_t n, int cap, int nf) {
    const size_t L = firk_intervals(cap);
    if (L > 32) return n * firk_lines(L) * nf;
    const size_t G = 64 / L;
    return (n + G - 1) / G * 64 * nf;
}

// values of a slot: the correction and a copy of the state at the nodes, then the stage
// correction, a copy of the stages and the condensation records
FIRK_HD size_t firk_aux_values(int cap, int M, int S) {
    return (size_t)cap * (2 * M) + firk_lines(firk_intervals(cap)) * (2 * S * M + S * M * (M + 1));
}

}  // namespace bvpdev
