// Scratch of the three parts of k_mie_homog_tiers (gm_mie.hip): host arithmetic only.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace gm {

// Blocks of the parts for long, middle and short series and the bytes of their slots.
struct HomogParts {
  int64_t big, mid, small;
  size_t bytes;
};

// `want` blocks with slots of the given bytes each, cut to the budget.  The long
// series' part is the one that a launch waits for, so the others give way first, down
// to a sixteenth of the budget between them; a part that is wanted keeps a block.  In
// the 128 MiB of the no-alloc entry, log-distributed to x = 8000, 40k / 200k points: a
// third each 2514 / 11518 us, the short parts' share a third 1484 / 6521, a quarter
// 1352 / 5868, an eighth 1193 / 5120, a sixteenth 1126 / 4808; to x = 2094: 356 / 1694
// with a third each, 189 / 873 (all shares from a quarter down within 5%).
// Where not even a slot of each fits, the long series' part takes every point (mid =
// small = 0).
constexpr size_t kTailShare = 16;
inline HomogParts homog_parts(size_t budget, const HomogParts& want, size_t big_slot,
                              size_t mid_slot, size_t small_slot) {
  HomogParts p = want;
  const size_t tail = (size_t)want.mid * mid_slot + (size_t)want.small * small_slot;
  const size_t all_big = (size_t)want.big * big_slot;
  if (all_big + tail > budget) {
    const size_t left = std::max(budget > all_big ? budget - all_big : 0, budget / kTailShare);
    const double cut = std::min(1.0, (double)left / (double)std::max<size_t>(tail, 1));
    if (p.mid) p.mid = std::max<int64_t>(1, (int64_t)((double)want.mid * cut));
    if (p.small) p.small = std::max<int64_t>(1, (int64_t)((double)want.small * cut));
    const size_t used = (size_t)p.mid * mid_slot + (size_t)p.small * small_slot;
    p.big = std::min<int64_t>(want.big, used < budget ? (int64_t)((budget - used) / big_slot) : 0);
    if (p.big < 1) {
      p.mid = p.small = 0;
      p.big = std::max<int64_t>(1, std::min<int64_t>(want.big, (int64_t)(budget / big_slot)));
    }
  }
  p.bytes = (size_t)p.big * big_slot + (size_t)p.mid * mid_slot + (size_t)p.small * small_slot;
  return p;
}

}  // namespace gm
