// Score pass (select_kernel.hpp) for fp32 operands and for caller-given scores, and its plan.
#include "select_kernel.hpp"

namespace asa {

hipError_t launch_select_f32(const SelectParams& p, hipStream_t s) { return launch_type<float>(p, s); }

hipError_t launch_select_scores(const SelectParams& p, hipStream_t s) {
  return launch_r<float, 64, kGivenScores>(p, s);
}

SelectPlan select_plan(const Dims& d, int dtype, bool from_scores, size_t max_lds, int cus) {
  // Rings: 16-bit inputs, hd = D, raw dots (launch_ring).
  const bool raw = !from_scores && d.scale > 0.0f;
  const bool ring = raw && dtype != kElemF32 && d.hd == d.D;
  // Eight waves where the lists leave room for one block per compute unit
  // only: above k = 64, and above k = 42 at d = 128 beside the rings (two
  // 4-wave blocks fit below; 1x16x8192, d = 128, k = 32: 432 against 495 us
  // with eight).  1x8x32768, d = 128, k = 128: 4.9 -> 3.7 ms.  fp32 at
  // d = 128 holds 128 registers of Q and would spill at two waves per SIMD.
  // And where the grid gives each compute unit one block at most, whose
  // waves then are all that the unit runs: this kernel with four against
  // eight waves, 1x4x4096, k = 32: bf16 d = 64 67 -> 45 us, d = 128 79 -> 56,
  // d = 80 80 -> 53, fp16 d = 128 79 -> 56, fp32 d = 64 180 -> 161; 1x2x1500
  // bf16 d = 128 46 -> 33; 16x16 heads of 1x4096, bf16 d = 64 54 -> 48,
  // d = 128 90 -> 92 (each block streams its own K there).  With more blocks
  // two 4-wave ones share a unit.
  const bool few = size_t(d.nQB) * size_t(d.BH) <= size_t(cus);
  const bool wide = raw && (few || d.k > 64 || (d.k > 42 && ring && d.D == 128)) &&
                    !(dtype == kElemF32 && d.D == 128);
  const struct { int waves; bool ring; } tries[] = {{wide ? 8 : 4, ring}, {4, ring}, {4, false}};
  // k + 32 keys per row hold the candidates of random rows with room to
  // spare up to k = 42, and 1.75 k above (the floor's slack grows with k).
  // Where LDS is short (the visible list takes 4 bytes per key block) the
  // first variant that holds k + k / 8 + 16 is taken (random rows list about
  // 1.15 k), else the one that holds most.  Less still works, by overflow
  // rounds that drop cap - k keys each, down to k + 4.
  SelectPlan plan{4, false, -1, 0};
  for (const auto& t : tries) {
    auto bytes = [&](int cap) { return size_t(sel_layout(d.k, cap, d.nKB, t.waves, t.ring ? d.D : 0).total); };
    int cap = d.k + (d.k * 3 / 4 > 32 ? d.k * 3 / 4 : 32);
    while (cap > d.k + 4 && bytes(cap) > max_lds) cap = cap - 4 > d.k + 4 ? cap - 4 : d.k + 4;
    if (bytes(cap) > max_lds) {
      if (plan.cap < 0) plan.needs = bytes(cap);
      continue;
    }
    if (cap > plan.cap) plan = SelectPlan{t.waves, t.ring, cap, 0};
    if (cap >= d.k + d.k / 8 + 16) break;
  }
  return plan;
}

}  // namespace asa
