// The activation table's entries of gate values 2^-9 <= |g| < 2^11 in LDS, for the expert tiles'
// epilogues (20 KB, each sign's run of the 65536-entry table contiguous): gathered from memory, every
// lookup is a cache line of its own.  Values outside the run are read from memory.
#pragma once
#include "contract_act.h"
#include "pp_tile.h"

namespace lsk {

constexpr int kActE0 = 118, kActRun = 20 * 128;  // first biased exponent; entries of a sign
constexpr int kActRunBytes = 2 * kActRun * 4;

// Requests the run into dst (16-byte aligned), 1 KB per instruction dealt to the block's waves; the
// caller waits for the loads and synchronises the block.
LSK_DEV void act_run_load(const float* tab, char* dst, int wave, int waves) {
  const __amdgpu_buffer_rsrc_t rt = make_rsrc(tab, 65536 * 4);
  const int lane = threadIdx.x & 63;
  static_assert(kActRunBytes % 1024 == 0, "whole wave loads");
  for (int g = wave; g < kActRunBytes / 1024; g += waves) {
    const int e = (g * 64 + lane) * 4;       // first entry of the lane's 16 bytes
    const int sign = e >= kActRun ? 1 : 0;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_void_t)(dst + g * 1024), 16,
                                             (sign * 32768 + kActE0 * 128 + e - sign * kActRun) * 4, 0, 0, 0);
  }
}

// tab[g] of a bf16-valued g.
LSK_DEV float act_run_entry(const float* run, const float* tab, float g) {
  const uint32_t bits = __float_as_uint(g) >> 16;
  const uint32_t k = (bits & 0x7fffu) - kActE0 * 128;
  const bool in = k < (uint32_t)kActRun;
  float e = run[in ? (bits >> 15) * kActRun + k : 0];
  if (!in) e = tab[bits];
  return e;
}

}  // namespace lsk
