// Which points a task of SP's staged line solve (sp_lines.inc) holds: index
// arithmetic only, without device code, so that a host program can check it.
#pragma once

namespace npbmz {
namespace sp {

constexpr int kStageLines = 6;  // lines per wave: 10 lanes each, 4 idle

// a / b for 0 <= a < 2^20, inv = 1/b in single precision.
__host__ __device__ __forceinline__ int small_div(int a, float inv) {
  return (int)(((float)a + 0.5f) * inv);
}

// a * b for 0 <= a, b < 2^10.
__host__ __device__ __forceinline__ int small_mul(int a, int b) {
#ifdef __HIP_DEVICE_COMPILE__
  return __mul24(a, b);
#else
  return a * b;
#endif
}

// A task's lines first .. first+cnt-1 of a zone of nx x ny x nz points (at
// least 5 each), their points numbered in memory order: along x the points of
// a line are contiguous, along y and z the lines.  Line numbers are
// line_geom's.
template <int DIR>
struct StagedLines {
  int cnt, nl, across, a0, sa, wrap, st, org;
  float inv_in;
  __host__ __device__ __forceinline__ StagedLines(int nx, int ny, int nz, int first) {
    const int lines = ((DIR == 0 ? ny : nx) - 2) * ((DIR == 2 ? ny : nz) - 2);
    cnt = lines - first < kStageLines ? lines - first : kStageLines;
    nl = DIR == 0 ? nx : DIR == 1 ? ny : nz;
    // line first + li is the one at (a0 + li) mod across, (a0 + li) / across
    // rows above the first one's
    across = (DIR == 0 ? ny : nx) - 2;
    a0 = first % across;
    const int plane = nx * ny, up = DIR == 2 ? nx : plane;
    sa = DIR == 0 ? nx : 1;
    st = DIR == 0 ? 1 : DIR == 1 ? nx : plane;
    wrap = up - across * sa;
    org = sa + (1 + first / across) * up;
    inv_in = 1.0f / (float)(DIR == 0 ? nl : cnt);
  }
  // Element e < cnt * nl (nl < 2^10): its line, its place in it and its point
  // in the zone.
  __host__ __device__ __forceinline__ int at(int e, int& li, int& q) const {
    const int in = DIR == 0 ? nl : cnt;
    const int hi = small_div(e, inv_in), lo = e - small_mul(hi, in);
    li = DIR == 0 ? hi : lo;
    q = DIR == 0 ? lo : hi;
    // by comparisons: w < across + kStageLines - 1 <= 3 across, of any size
    const int w = a0 + li;
    return org + w * sa + (w >= across ? wrap : 0) + (w - across >= across ? wrap : 0) + q * st;
  }
};

}  // namespace sp
}  // namespace npbmz
