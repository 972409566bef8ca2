// The lane-replicated byte-pair code table's fill, shared by the streaming
// decode kernels and the few-token kernels (512-thread workgroups; the table
// itself and its lookups are described in nsmlp_internal.h).
#pragma once

#include "nsmlp_internal.h"

namespace nsmlp {

// Filled by 512 threads in 8 passes of one 16-byte LDS write each: pass ps
// writes entry e = 32 ps + tid / 16, copies 4 (tid % 16) .. +3 (copies 0..31
// decode code_a, 32..63 code_b).  The entry's low half is the code of its high
// nibble (e / 16 = 2 ps + tid / 256), the high half the code of its low nibble
// ((tid / 16) % 16).
struct LutCodes {
  float lo[8];
  float hi;
};

__device__ __forceinline__ void lut_codes_load(const float* code_a, const float* code_b, int tid, LutCodes& c) {
  const float* code = (tid & 15) >= 8 ? code_b : code_a;
#pragma unroll
  for (int ps = 0; ps < 8; ++ps) c.lo[ps] = code[2 * ps + (tid >> 8)];
  c.hi = code[(tid >> 4) & 15];
}

__device__ __forceinline__ void lut_store(uint32_t* lut, const LutCodes& c, int tid) {
  const uint32_t hi = (uint32_t)f2h(c.hi) << 16;
#pragma unroll
  for (int ps = 0; ps < 8; ++ps) {
    const uint32_t v = (uint32_t)f2h(c.lo[ps]) | hi;
    const int e = ps * 32 + (tid >> 4);
    *reinterpret_cast<uint4*>(lut + e * 64 + (tid & 15) * 4) = make_uint4(v, v, v, v);
  }
}

}  // namespace nsmlp
