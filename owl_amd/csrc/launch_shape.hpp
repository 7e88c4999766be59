// Default launch shape and block order of the marching sweeps.
#pragma once
#include <hip/hip_runtime.h>

namespace owl {

// The block this workgroup stands for: workgroups are dealt to the 8 XCDs in
// turn, so workgroup w takes block (w % 8) (n / 8) + w / 8 and each XCD walks
// one contiguous range of blocks, whose halos then meet in its L2 (the last
// n % 8 keep their own).  FSG sweeps of 8 shots of 333 x 171 read 28 + 18 MB
// from beyond the L2 instead of 47 + 36 and take 22.8 + 15.9 us instead of
// 24.8 + 19.8; of 32 shots of 801 x 401, 810 + 547 MB instead of 948 + 685
// for 1-2 %.
__device__ __forceinline__ int xcd_block() {
    const unsigned per = gridDim.x / 8u, w = blockIdx.x;
    return int(w < 8u * per ? (w % 8u) * per + w / 8u : w);
}

// Rows (2D) or planes (3D) that one wavefront marches over, from the number
// of wavefronts the batch has at one row or plane each.  A wavefront's march
// is serial, about 1.5 us a row when few wavefronts share a SIMD, so a small
// batch wants as many wavefronts as it can have; a large one wants longer
// marches, whose fill of the z queue (2R rows) weighs less.  The line is
// where the chip holds about twice the wavefronts that run at once.
// us per step on one MI355X at 2 / 4 / 8 / 32 rows: 2D elastic 301 x 201,
// 1 shot 14 / 17 / 22 / 59, 8 shots 25 / 27 / 33 / 69, 32 shots 59 / 60 / 67 /
// 82; FSG 333 x 171, 8 shots 39 / 39 / 47 / 100; 801 x 401, 32 shots 514 / 477 /
// 478 / 548; 3D elastic 50 x 45 x 40 61 / 57 / 70 / 175, 117 x 90 x 75, 2 shots
// 259 / 248 / 263 / 313; 200 x 200 x 150, 4 shots 2430 / 2264 / 2243 / 2358; 3D
// acoustic (four-wide columns) 50 x 45 x 40 24 / 27 / 39 / 106, 121 x 110 x 93,
// 2 shots 105 / 102 / 110 / 149, 256^3, 16 shots 4499 / 4264 / 4203 / 4458.
inline int default_planes(double wavefronts) {
    constexpr double kEnough = 14000.0;
    if (wavefronts / 8 >= kEnough) return 8;
    if (wavefronts / 4 >= kEnough) return 4;
    return 2;
}

}  // namespace owl
