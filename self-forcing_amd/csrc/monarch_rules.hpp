// Which way Kbar and Y take between the two steps of the MFMA forward: host arithmetic on the arguments of a pass.
#pragma once

#include "sfm_common.hpp"

namespace sfm {

// Rows of Kbar (and as many of Y) of a pass; with `masked_out` those of visible (query, key) block-frame pairs only: of causal
// blocks of c block-frames, n of them, c * c pairs for each of n (n + 1) / 2.
inline size_t scratch_rows(const MonarchArgs& a, int nunits, bool masked_out) {
    const size_t n = masked_out ? a.na / a.causal : 0;
    const size_t pairs = masked_out ? n * (n + 1) / 2 * a.causal * a.causal : (size_t)a.na * a.nf;
    return pairs * a.b1 * a.b2 * nunits;
}

// Whether step 1 leaves masked pairs out (its kernels for a new chunk do not)
inline bool step1_skips_masked(const MonarchArgs& a) { return a.causal && a.skip_masked && !a.new_kv; }

// From the size on where the memory-side cache holds part of Kbar and Y only, their rows, read once, are read past it: us
// through the caches and past them, 12 heads x 128 of 30 x 52, three frames against 9 (259 MB) 143, 140, 12 (345) 193, 179, in
// half-height blocks (690) 342, 336; 6 heads, 21 frames (302) 155, 146; 40 heads, 21 (2013) 1038, 1002.  Below, they would leave it: 6 heads,
// 12 frames (173 MB) 96.3, 98.6; three frames tied against 21 (201) 146, 149.  Masked pairs count: nine frames of three tied, block-causal, under autograd (165 MiB of
// 247) 465, 460 with their backward.
inline bool step2_past_caches(const MonarchArgs& a, int nunits) {
    return scratch_rows(a, nunits, false) * 4 * a.D >= (size_t)240 << 20;
}

// What a pass writes goes through the caches where they can hold enough of it for the kernel that reads it next, and past them where
// they cannot (written back under that kernel's reads) or where it is little (the L2s give their dirty lines up at the kernel's
// end).  us past the caches and through them, 12 heads x 128 of 30 x 52 unless named: three frames against 3 (86 MB) 67, 63.5,
// 6 (173) 112, 104, 9 (259) 154, 143; three passes at three frames tied (100 and 201) 450, 424; 2 heads, 6 frames (29) 29.4, 29.3;
// 1 head, 3 frames (7) 21.8, 22.9; three frames tied against themselves (29) 44.6, 47.4.
// Too little is less than 40 MiB, and 64 for teams of waves (more than 32 query rows in step 2): 80 random calls of 36 to 70 MiB are 0.988
// times as long with that limit as with 40, block-causal ones 0.982.  Up to 32 rows 51 calls of 40 to 64 take 0.98 times as long
// through the caches.
// Too much depends on the query block-frames, with which the bytes written for each byte of K and V grow.  Since step 2 reads past the
// caches what they hold in part (above), up to five gain as far as 1.1 GiB: three against 10 heads, 21 (480 MiB) 262, 246, 11 heads
// (528) 283, 266, 14 (672) 372, 362; 180 random calls of 280 MiB to 1.1 GiB 0.967 times as long, of 1.1 to 1.5 GiB level.  From six on
// it is too much where step 2 reads past them: of 240 to 364 MiB 1.04 times as long (half-height blocks, 5 heads, 15 frames, 343: 166,
// 184), block-causal ones 1.02, beyond level or longer.  Kbar alone is followed by as many bytes of representatives: two passes, 21
// frames (302) 624, 637.
// Too little is what the pass does write, masked pairs left out; so is too much, up to five query block-frames.
inline bool step1_through_caches(const MonarchArgs& a, int nunits, bool kbar_alone) {
    const size_t written = scratch_rows(a, nunits, step1_skips_masked(a)) * ((kbar_alone ? 2 : 4) * a.D + (a.rb ? 128 : 0));
    const size_t least = a.b1 > 32 && !kbar_alone ? 64 : 40, most = kbar_alone ? 256 : 1100;
    return written >= least << 20 && written <= most << 20 && (kbar_alone || a.na <= 5 || !step2_past_caches(a, nunits));
}

}  // namespace sfm
