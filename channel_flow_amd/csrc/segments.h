// Which form the passes along the degree take (columns.hip): in segments, whose
// exchanges cost the same at any size, or one thread per column, whose serial
// chains stream once there are columns enough to hide their latency.
#pragma once

namespace chf {

// By the columns and f32_fields (the mixed form with FFT transforms: u, w, omega_x,
// omega_z and L in FP32), both fixed for a context, so that every kinematics pass of
// a run forms the same bits.  The lines are where the step times (us, segments /
// serial chains) cross; a launch by itself loses from fewer columns on.
//
// Kinematics, FP64: 9216 columns, the launch alone, N = 32 13.2 / 17.1, N = 256 77 / 102;
// steps: 18432 N = 54 517 / 521, 20736 N = 96 964 / 971 and N = 160 1617 / 1607, 23328
// N = 128 1434 / 1443, 24576 N = 96 1137 / 1141 and N = 256 2990 / 2976 (even), 32768
// N = 192 the launch 214 / 154.  Mixed: 16384 N = 128 590 / 595 and N = 192 929 / 939, 24576
// N = 32 266 / 260, N = 192 1510 / 1519, N = 256 2096 / 2061.
inline bool kinematics_in_segments(long ncol, bool f32_fields) { return ncol <= (f32_fields ? 20480 : 24576); }

// h assembly, FP64 steps: 18432 N = 16 195.8 / 196.4 and N = 54 515 / 517, 20736 N = 96 967 /
// 964, 23328 N = 128 1441 / 1434, 24576 N = 96 1144 / 1137, N = 160 1925 / 1917 and N = 256
// 3011 / 2990 (the launch alone 108 / 95).  Mixed, the launch: 16384 N = 256 63 / 88, 24576
// N = 32 16.3 / 18.1 and N = 256 91 / 97.
inline bool hassemble_in_segments(long ncol, bool f32_fields) { return ncol <= (f32_fields ? 24576 : 20480); }

}  // namespace chf
