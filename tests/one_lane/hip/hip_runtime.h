// One lane of a wavefront on the host: the device code of gagp_amd/csrc
// compiled by g++ with -D__HIPCC__ and this folder on the include path runs as
// a wavefront whose other 63 lanes are off.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

#define __host__
#define __device__
#define __global__

struct OneLane { unsigned x = 0, y = 0, z = 0; };
static const OneLane threadIdx{}, blockIdx{};

using std::signbit;
inline unsigned long long __ballot(int on) { return on != 0; }
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
inline int __ffsll(long long x) { return __builtin_ffsll(x); }
template <class T> inline T __shfl_xor(T x, int, int) { return x; }

// The relative error of the hardware's reciprocal (below 2^-23), set by a test.
static double reciprocal_error = 0;
#define __builtin_amdgcn_rcp(x) ((1.0 + reciprocal_error) / (x))
#define __builtin_amdgcn_readlane(x, lane) ((void)(lane), (x))
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_update_dpp(old, x, control, rows, banks, bound) ((void)(x), (old))  // no lane beside this one
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)
