// Walks of a grid over an index range whose end may be any int.
#pragma once
#if defined(__HIPCC__)
#define QMCX_HD __host__ __device__
#else
#define QMCX_HD
#endif

namespace qmcx {
// The index `step` after u in [0, end): `end` when it is not below end (u + step may pass INT_MAX there).
QMCX_HD inline int walk_next(int u, int step, int end) { return step < end - u ? u + step : end; }
// a / b rounded up, for a >= 0 up to INT_MAX
QMCX_HD inline int ceil_div(int a, int b) { return a / b + (a % b != 0 ? 1 : 0); }
}  // namespace qmcx
