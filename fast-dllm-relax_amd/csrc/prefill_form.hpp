// The form of attn_prefill_kernel a launch takes: host code without any GPU header, compiled into attention.hip and
// checked on the CPU (tests/prefill_form_check.cpp).
#pragma once

namespace fdllm {

// Of a kv head's 2 grp query tiles a workgroup takes all twelve (whole; six query heads per kv head) or four, and of
// the nqb = rows / 32 query blocks two (paired) or one.
struct PrefillForm { bool whole, paired; };

// pair: 0 blocks alone, 2 paired with all tiles, 3 paired with four, 1 by size: four tiles alone until their
// workgroups pass one round of the device's compute units by a quarter, then paired (uneven blocks in a second round cost
// more than the pairs' fewer workgroups), all twelve alone once that gives 45/64 of a round (180 workgroups for 256
// units) and paired once the pairs give 7/8.  hpw: the query heads per workgroup, 2 four tiles, 6 all twelve, anything
// else by pair.  Measured (256 units, 1.5B bf16 build_prefix_cache, us per layer; four alone / four paired / twelve alone / twelve paired): 509 rows 109.8 /
// 113.7 / 119.2 / 128.2, 1500 rows 226 / 229 / 245 / 254, 2048 rows 271 / 261 / 282 / 291, 3000 rows 386 / 397 /
// 389 / 398, 4096 rows 494 / 489 / 481 / 487, 6000 rows 762 / 787 / 708 / 716, 8192 rows 1041 / 1025 / 942 / 932.
inline PrefillForm prefill_form(int rows, int nq, int nkv, int cus, int pair, int hpw) {
  const int nqb = (rows + 31) / 32, grp = nq / nkv;
  const bool can_whole = grp == 6 && hpw != 2;
  PrefillForm f{can_whole && (pair == 2 || hpw == 6), pair >= 2};
  if (pair == 1 && !f.whole && 4 * nqb * nkv * ((2 * grp + 3) / 4) > 5 * cus) {
    f.whole = can_whole && 64 * nqb * nkv >= 45 * cus;
    f.paired = !f.whole || 8 * ((nqb + 1) / 2 * nkv) >= 7 * cus;
  }
  return f;
}

}  // namespace fdllm
