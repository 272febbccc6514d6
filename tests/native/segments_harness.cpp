// Test harness: C entry points over the rule of channel_flow_amd/csrc/segments.h,
// loaded by tests/test_segments_host.py.
#include "../../channel_flow_amd/csrc/segments.h"

extern "C" int kinematics_c(long ncol, int f32) { return chf::kinematics_in_segments(ncol, f32 != 0); }
extern "C" int hassemble_c(long ncol, int f32) { return chf::hassemble_in_segments(ncol, f32 != 0); }
