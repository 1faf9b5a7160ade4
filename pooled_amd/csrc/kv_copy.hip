// Device-to-device copies of cache planes (checkpoint slots) on gfx950; and of outputs that could not be written in place.
//
// A saved or restored session is rows [0, pos) of every layer's K and V (and scales): per tensor n_kv_heads contiguous
// planes at one pitch on either side (the reference's copyBufferToBuffer calls: engine/dense.js:20-47).  One launch covers up
// to PA_COPY_TENSORS tensors: the runtime's pitched copy runs one kernel a tensor, each a few microseconds of ramp-up and
// tail at 3.7 TB/s of traffic.
//
// Bound by HBM.  A workgroup moves one 32 KB piece (256 threads x 8 x 16 bytes, all loads ahead of the stores): small
// enough that the last round of the chip is short, large enough that a piece is several whole DRAM pages.  Measured, 10
// layers of the 2-kv-head shape at 9001 rows (184 MB saved and 184 MB restored, 738 MB of traffic): 359 us on the runtime's
// copies, 126 us here (5.85 TB/s; a plain 1 GiB copy by torch reads 5.2 TB/s).
#include "pa_internal.h"

typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef u4 u4d __attribute__((aligned(8)));       // (planes of an f16 output's columns are 8 bytes aligned)

#define CP_PIECE 2048u      // 16-byte units of a workgroup's piece

__global__ __launch_bounds__(256) void pa_copy_planes_kernel(PaCopyParams p) {
  // workgroup -> (tensor, plane, piece): pieces fastest, so neighbours read neighbouring memory
  uint32_t wg = blockIdx.x, t = 0;
  while (t + 1 < p.n && wg >= p.first[t + 1]) t++;
  wg -= p.first[t];
  const uint32_t units = p.units[t], ppp = (units + CP_PIECE - 1) / CP_PIECE;
  const uint32_t plane = wg / ppp, u0 = (wg - plane * ppp) * CP_PIECE + threadIdx.x;
  const u4* src = (const u4*)((const unsigned char*)p.src[t] + (size_t)plane * p.src_pitch[t]);
  u4d* dst = (u4d*)((unsigned char*)p.dst[t] + (size_t)plane * p.dst_pitch[t]);
  u4 v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = __builtin_nontemporal_load(src + min(u0 + 256u * i, units - 1));
#pragma unroll
  for (int i = 0; i < 8; i++) if (u0 + 256u * i < units) __builtin_nontemporal_store(v[i], dst + u0 + 256u * i);
}

// p.n tensors of n_planes planes each; p.first is filled here
hipError_t pa_launch_copy_planes(PaCopyParams& p, uint32_t n_planes, hipStream_t s) {
  if (p.n == 0) return hipSuccess;
  if (p.n > PA_COPY_TENSORS) return hipErrorInvalidValue;
  uint64_t total = 0;
  for (uint32_t t = 0; t < p.n; t++) {
    if (p.units[t] == 0 || p.units[t] > 0xFFFF0000u) return hipErrorInvalidValue;
    p.first[t] = (uint32_t)total;
    total += (uint64_t)n_planes * ((p.units[t] + CP_PIECE - 1) / CP_PIECE);
    if (total > 0x7FFFFFFFull) return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL(pa_copy_planes_kernel, dim3((uint32_t)total), dim3(256), 0, s, p);
  return hipGetLastError();
}
