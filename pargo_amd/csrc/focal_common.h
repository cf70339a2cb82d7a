// focal_common.h -- device helpers shared by the focal (3x3) kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pargo {

// sqrt(2.0) as the reference evaluates it (glibc sqrt is correctly rounded)
// and the double nearest to its reciprocal.
constexpr double kSqrt2 = 0x1.6a09e667f3bcdp+0;
constexpr double kInvSqrt2 = 0x1.6a09e667f3bccp-1;
// The D8 epsilon 0.000001 (apps/hydrology/flowdird8/d8Operator.cpp:3).
constexpr double kD8Eps = 0.000001;

// FP32 D8 filter (focal.hip): RN32(1/sqrt 2) and the thresholds that keep
// the filter's decisions provably those of the FP64 tests.
constexpr float kInvSqrt2f = 0x1.6a09e6p-1f;
constexpr float kD8SureF = 1.0001e-6f;        // K
constexpr float kD8Shrink = 0x1.ffffep-1f;    // 1 - 2^-20
constexpr float kD8FloorF = 0x1.0c6898p-20f;  // the float just below RN32(0.9999e-6)
constexpr float kD8BandMid = 1.5e-6f;         // |M - 1.5e-6| < 0.50025e-6: ambiguous
constexpr float kD8BandHalf = 0.50025e-6f;

// RN(x / kSqrt2) for finite x derived from float32 data (|x| <= 2^129,
// x = 0 or |x| >= 2^-149, so nothing below underflows).
// q0 = RN(x*y) with y = RN(1/s) is within 0.69 ulp of x/s because
// |y*s - 1| = 0.183 * 2^-53; by Markstein's theorem (y within half an ulp
// of 1/s, q0 within one ulp of x/s) r = x - q0*s is exact in one FMA and
// RN(q0 + r*y) is the correctly rounded quotient.  The identity is also
// checked on the host against IEEE division over every binade from 2^-149
// to 2^129 (tests/cpp/gpro_host_test.cpp).
__device__ __forceinline__ double div_sqrt2(double x)
{
    double q0 = x * kInvSqrt2;
    double r = __builtin_fma(-q0, kSqrt2, x);
    return __builtin_fma(r, kInvSqrt2, q0);
}

// Exact float interval test for NoData (see nodata_interval on the host).
__device__ __forceinline__ bool in_interval(float v, float lo, float hi) { return v >= lo && v <= hi; }

// ESRI code -> reference dirType 8 output (median tied window index).
// Built on the host from the reference's rule validDir[len >> 1]
// (d8Operator.cpp:78-88); 255 for code 0 (unused: flat cells are
// resolved before the lookup).
struct D8Lut8 {
    uint8_t v[256];
};

// Workgroups go to the 8 XCDs in turn by linear id.  Renumbers the
// workgroup of a (column block, row strip) grid so that each XCD takes a
// contiguous run of strips, column blocks first: neighbouring strips then
// share their halo rows in that XCD's L2 instead of reading them twice from
// HBM.  A bijection of the grid onto itself.
__device__ __forceinline__ void xcd_strip_order(unsigned &cb, unsigned &strip)
{
    const unsigned gx = gridDim.x, n = gx * gridDim.y, i = blockIdx.y * gx + blockIdx.x;
    const unsigned per = n / 8, rem = n % 8, x = i % 8;
    const unsigned w = x * per + (x < rem ? x : rem) + i / 8;
    cb = w % gx;
    strip = w / gx;
}

// Rows per strip of a kernel whose waves walk strips of `width` columns, for
// a raster of rows x cols: a wave's rows are a serial chain (about 1 us each),
// so a small raster takes the strip that still gives every SIMD four waves
// (4096 waves on 256 CUs), down to single rows, and a larger one the strip
// that gives about five rounds of them, up to `most`; the two halo rows a
// strip reads again come from the caches.  Measured with strips of 16 rows
// before, us for slope / slope + D8 / slope + D8 with the mask:
//   256 x 256     16.4 / 22.7 / 27.6   now  3.6 /  4.7 /  4.5  (1 row)
//   1024 x 1024   16.5 / 23.3 / 28.6        5.7 /  7.4 /  8.0  (1 row)
//   1501 x 2003   17.5 / 25.4 / 30.4        9.5 / 13.2 / 15.5  (3 rows)
//   4096 x 4096   30.4 / 41.9 / 58.8       28.5 / 40.2 / 52.1  (4 rows)
//   7001 x 5003   58.0 / 76.4 / 102.9      52.6 / 71.6 / 97.1  (7 rows)
// At 16384^2 the longest strips stay the fastest (1 row doubles the time).
constexpr long long kStripWaves = 4096;
inline int strip_rows_of(long long work, int most)  // work: rows times strips side by side
{
    const long long n =
        work <= 4 * kStripWaves ? (work + kStripWaves - 1) / kStripWaves : (work + 5 * kStripWaves / 2) / (5 * kStripWaves);
    const long long least = work <= 4 * kStripWaves ? 1 : 4;
    return (int)(n < least ? least : n > most ? most : n);
}
inline long long strip_work(int rows, int cols, int width) { return (long long)rows * ((cols + width - 1) / width); }
inline int strip_rows(int rows, int cols, int width, int most)
{
    return strip_rows_of(strip_work(rows, cols, width), most);
}

}  // namespace pargo
