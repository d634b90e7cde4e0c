// Grouped MX tiles on the block-scaled matrix core of gfx950 (the MoE MXFP4 expert GEMMs with
// per-row activation scales): 128 x 128 tiles, four waves of 64 x 64, K staged 128 elements (four MX
// blocks) at a time, two blocks per CU.
//
// The contract's update needs the exact sum of every 32-wide block before it rounds (mx_tile.h).
// v_mfma_scale_f32_32x32x64_f8f6f4 sums 64 products of six-bit (A) and four-bit (B) floats, each
// 32 with an E8M0 scale of its own, so one MFMA does one MX block: an int8 activation a is two
// six-bit E2M3 planes, sign(a) (|a| >> 4) / 8 and sign(a) (|a| & 15) / 8 (every integer up to 15
// over 8 is an E2M3 value, its magnitude field the integer itself), lanes 0-31 hold the block's
// high plane under the scale 2^7 and lanes 32-63 its low plane under 2^3, and both halves read the
// same 16 bytes of packed E2M1 codes as they lie in memory, under the weight's own E8M0 byte.  From
// a zero accumulator the result is s_b * 2^(kexp - 128) exactly: the products are multiples of
// 2^(kexp - 128) and sum to less than 2^16 of them (checked against binary64 on MI355X over 20 M
// sums with kexp 0 .. 239, 3 M of them at each of 0 .. 19; the accumulator input is not rounded once, so the update stays on the
// VALU).  The update is then one binary32 add per output and block, with no scale to read, no fp4
// conversions and half the matrix-core time of the bf16 form (16 adds of 4 cycles against one MFMA
// of 32 cycles per 32 x 32 outputs and block; bf16: 64).  The adds bound the loop, so the rest of
// it is kept off the VALU: all operands go global -> LDS by direct buffer loads with exact counted
// waits, and a wave whose rows are empty (experts fill few of a tile's 128 rows) skips its strips.
//
// Exponent bytes of 240 and more could overflow the product, so weight sets that hold one (the
// layer's mx_safe) take the bf16 tiles (mx_pp.h); the sums of the smallest are subnormal and exact.
//
// A rows: 48 bytes per block -- [high 0..15][high 16..23, low 16..23][low 0..15], code i of a
// plane at bits 6 i .. 6 i + 5 -- written by the row quantisers (mx.hip).  A lane's six registers
// are one 16-byte and one 8-byte LDS read.  LDS chunks are XOR-swizzled by bits 2 and 3 of the row.
#pragma once
#include <type_traits>

#include "mfma_tile.h"
#include "pp_tile.h"

namespace lsk {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

struct Mx6Cfg {
  static constexpr int BM = 128, BN = 128, kThreads = 256;
  static constexpr int TM = 2, TN = 2;            // 32 x 32 blocks of a wave
  static constexpr int kNB = 4;                   // MX blocks per stage
  static constexpr int kStageA = BM * 48 * kNB;   // two planes of each block
  static constexpr int kStageB = BN * 16 * kNB;
  static constexpr int kStageW = kStageB + BN * 4 * kNB;  // codes and exponents (a byte fills one LDS word)
  static constexpr int kOffW = 2 * kStageA;       // two A stages, then three of codes and exponents
  static constexpr int kRowOff = kOffW + 3 * kStageW;  // the epilogue's row operands [3][BM]
  static constexpr int kSmemBytes = kRowOff + 3 * BM * 4;
  typedef v16f Acc[TM][TN];
};

// Per-thread load plan of one tile: byte offsets of each load slot's row and chunk within a stage
// (kOob: no row), and the slot's block.
struct Mx6Rows {
  uint32_t a[6], b[2], s[2];
  int ab[6], bb[2], sb;
};

template <class FA, class FB, class FS>
LSK_DEV Mx6Rows mx6_rows(FA rowA, FB rowB, FS rowS) {
  const int tid = threadIdx.x;
  Mx6Rows p;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int slot = j * 256 + tid, row = slot / 12;
    const int c = (slot - row * 12) ^ ((row >> 2) & 3);
    const uint32_t r = rowA(row);
    p.a[j] = r == kOob ? kOob : r + 16 * c;
    p.ab[j] = c / 3;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int slot = j * 256 + tid, row = slot >> 2;
    const int c = (slot & 3) ^ ((row >> 2) & 3);
    const uint32_t r = rowB(row), q = rowS(row);
    p.b[j] = r == kOob ? kOob : r + 16 * c;
    p.bb[j] = c;
    p.s[j] = q == kOob ? kOob : q + (slot & 3);
  }
  p.sb = tid & 3;
  return p;
}

// acc += the K / 32 blocks in ascending order.  kTM: 32-row strips of the wave that hold rows (0 ..
// 2); the others' accumulators stay zero.  Waves of one block may run different kTM (the loads and
// barriers are the same).
template <int kTM>
LSK_DEV void mx6_mainloop(Mx6Cfg::Acc& acc, __amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rb,
                          __amdgpu_buffer_rsrc_t rs, const Mx6Rows& rows, int K, int wm, int wn, char* smem) {
  using C = Mx6Cfg;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int nb = K / 32, nk = (nb + C::kNB - 1) / C::kNB;

  // the loads of stage s, activations into slot s & 1, codes and exponents into slot `slot`; TAIL:
  // blocks from nb on read zeros
  auto issue_a = [&](int s, auto tail) {
    constexpr bool kTail = decltype(tail)::value;
    char* st = smem + (s & 1) * C::kStageA;
    const int left = nb - s * C::kNB;
#pragma unroll
    for (int j = 0; j < 6; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t)(st + (j * C::kThreads + wave * 64) * 16), 16,
                                               kTail && rows.ab[j] >= left ? kOob : rows.a[j], s * 48 * C::kNB, 0, 0);
  };
  auto issue_w = [&](int s, int slot, auto tail) {
    constexpr bool kTail = decltype(tail)::value;
    char* st = smem + C::kOffW + slot * C::kStageW;
    const int left = nb - s * C::kNB;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void_t)(st + (j * C::kThreads + wave * 64) * 16), 16,
                                               kTail && rows.bb[j] >= left ? kOob : rows.b[j], s * 16 * C::kNB, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t)(st + C::kStageB + (j * C::kThreads + wave * 64) * 4), 1,
                                               kTail && rows.sb >= left ? kOob : rows.s[j], s * C::kNB, 0, 0);
  };
  auto full = [&](int s) { return (s + 1) * C::kNB <= nb; };
  auto issue_a_any = [&](int s) { full(s) ? issue_a(s, std::false_type{}) : issue_a(s, std::true_type{}); };
  auto issue_w_any = [&](int s, int slot) {
    full(s) ? issue_w(s, slot, std::false_type{}) : issue_w(s, slot, std::true_type{});
  };

  // fragment addresses of row / column r32 of a 32-row block (bits 2 and 3 of the row swizzle it)
  const int r32 = lane & 31, half = lane >> 5, sw = (r32 >> 2) & 3;
  const int offA = (wm * 64 + r32) * 48 * C::kNB, offB = (wn * 64 + r32) * 16 * C::kNB;
  const int offS = C::kStageB + (wn * 64 + r32) * 4 * C::kNB;
  const int sa = half ? 127 + 3 : 127 + 7;
  int aoff[C::kNB][2], boff[C::kNB];  // a block's 16-byte piece of the lane's plane and its 8-byte rest; its codes
#pragma unroll
  for (int b = 0; b < C::kNB; ++b) {
    aoff[b][0] = offA + 16 * ((3 * b + 2 * half) ^ sw);
    aoff[b][1] = offA + 16 * ((3 * b + 1) ^ sw) + 8 * half;
    boff[b] = offB + 16 * (b ^ sw);
  }

  struct Frag {
    v8i a[C::TM], b[C::TN];
  };
  auto read = [&](const char* st, const char* sw_, int b, Frag& f) {
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
      const v4i x = *(const v4i*)(st + aoff[b][0] + i * 32 * 48 * C::kNB);
      const v2i y = *(const v2i*)(st + aoff[b][1] + i * 32 * 48 * C::kNB);
      f.a[i] = v8i{x[0], x[1], x[2], x[3], y[0], y[1], 0, 0};
    }
#pragma unroll
    for (int j = 0; j < C::TN; ++j) {
      const v4i x = *(const v4i*)(sw_ + boff[b] + j * 32 * 16 * C::kNB);
      f.b[j] = v8i{x[0], x[1], x[2], x[3], 0, 0, 0, 0};
    }
  };

  // A stage: a block's fragments are read one block ahead, and the adds of each result run one MFMA
  // behind it, across the blocks (the scheduling barriers keep the compiler from issuing MFMAs
  // together, which needs the registers of all their results and leaves the adds waiting for the
  // first).  BLOCKS: 2 or 4 of the stage's blocks.
  auto compute = [&](const char* st, const char* sw_, auto blocks) {
    constexpr int kBlocks = decltype(blocks)::value, kN = kTM * C::TN;
    const v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16f d[2];
    auto add = [&](int u) {
      v16f& c = acc[u / C::TN][u % C::TN];
#pragma unroll
      for (int r = 0; r < 16; ++r) c[r] = f32_add(c[r], d[u & 1][r]);
      __builtin_amdgcn_sched_barrier(0);
    };
    v4i sb[C::TN];
    Frag f[2];
#pragma unroll
    for (int j = 0; j < C::TN; ++j) sb[j] = *(const v4i*)(sw_ + offS + j * 32 * 4 * C::kNB);
    read(st, sw_, 0, f[0]);
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
      for (int u = 0; u < kN; ++u) {
        d[u & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f[b & 1].a[u / C::TN], f[b & 1].b[u % C::TN], z, 2, 4,
                                                                   0, sa, 0, sb[u % C::TN][b]);
        __builtin_amdgcn_sched_barrier(0);
        if (u == 0 && b + 1 < kBlocks) read(st, sw_, b + 1, f[(b + 1) & 1]);
        if (u > 0 || b > 0) add((u + kN - 1) % kN);
      }
    }
    add(kN - 1);
  };

  // step kt: issue the activations of stage kt + 1 and the codes of stage kt + 2 (AHEAD 2; 1: without
  // the codes; 0: neither), multiply stage kt, wait for stage kt + 1.  The codes run a stage further
  // ahead: an expert's codes come from memory where its rows come from the L2, and the step's last
  // four loads stay in flight across the barrier.  (A last stage's missing blocks add zeros, which
  // leave every accumulator as it is: none is ever -0.)
  int cur = 0;
  auto step = [&](int kt, auto ahead, auto steady) {
    constexpr int kAhead = decltype(ahead)::value;
    const int nxt = cur == 2 ? 0 : cur + 1;
    if constexpr (decltype(steady)::value) {
      issue_a(kt + 1, std::false_type{});
      issue_w(kt + 2, nxt == 2 ? 0 : nxt + 1, std::false_type{});
    } else {
      if constexpr (kAhead > 0) issue_a_any(kt + 1);
      if constexpr (kAhead > 1) issue_w_any(kt + 2, nxt == 2 ? 0 : nxt + 1);
    }
    const char* st = smem + (kt & 1) * C::kStageA;
    const char* sw_ = smem + C::kOffW + cur * C::kStageW;
    if constexpr (kTM > 0) {
      if constexpr (kAhead > 0) {
        compute(st, sw_, std::integral_constant<int, 4>{});
      } else {
        if (nb - kt * C::kNB > 2) compute(st, sw_, std::integral_constant<int, 4>{});
        else compute(st, sw_, std::integral_constant<int, 2>{});
      }
    }
    if constexpr (kAhead > 0) {
      compiler_fence();
      wait_vm<kAhead == 2 ? 4 : 0>();
      phase_barrier();
    }
    cur = nxt;
  };
  issue_a_any(0);
  issue_w_any(0, 0);
  if (nk > 1) issue_w_any(1, 1);
  compiler_fence();
  if (nk > 1) wait_vm<4>();
  else wait_vm<0>();
  phase_barrier();
  int kt = 0;
  for (; kt + 3 < nk; ++kt) step(kt, std::integral_constant<int, 2>{}, std::true_type{});
  if (kt + 2 < nk) step(kt++, std::integral_constant<int, 2>{}, std::false_type{});
  if (kt + 1 < nk) step(kt++, std::integral_constant<int, 1>{}, std::false_type{});
  step(kt, std::integral_constant<int, 0>{}, std::false_type{});
}

}  // namespace lsk
