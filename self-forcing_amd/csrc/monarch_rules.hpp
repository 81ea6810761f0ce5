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

// What a pass writes goes through the caches where the memory-side one (256 MB) can still hold most of it for the kernel that reads
// it next, and past them where it cannot (written back under that kernel's reads) or where it is little (the L2s give their dirty
// lines up at the kernel's end).  us past the caches and through them, 12 heads x 128 of 30 x 52 unless named: three frames
// against 3 (86 MB) 67, 63.5, 6 (173) 112, 104, 9 (259) 154, 143, 12 (345) 201, 193, 21 (604) 322, 331; 45 x 80, 6 frames (398)
// 245, 242, but level since step 2 reads past them; 12 frames in half-height blocks (690) 341, 376; three passes at three frames
// tied (100 and 201) 450, 424; 2 heads, 6 frames (29) 29.4, 29.3; 1 head, 3 frames (7) 21.8, 22.9; three frames tied against themselves (29) 44.6, 47.4.  Kbar alone is
// followed by as many bytes of representatives: two passes, 21 frames (302) 624, 637.
// Teams of waves (more than 32 query rows in step 2) need 64 MiB: 80 random calls of 36 to 70 are 0.988 times as long with that limit as with 40,
// block-causal ones 0.982 (through the caches, with more than 64 rows, 1.02 times; half-height blocks of 30 x 52, three tied, 4 heads x 64, 55 MiB: 51.5 us, 53.0).  Up to 32 rows 51 calls of 40 to 64 take 0.98 times as long through them.
// What is too little is what the pass does write, masked pairs left out: counted with them, block-causal calls of 25 to 40 MiB took up
// to 4 % longer.  The upper limit counts them: of 240 to 300 MiB without, such calls took 3 % longer through the caches (12 frames
// of 30 x 52, 4 heads, 274 MiB of 439: 173, 182).
inline bool step1_through_caches(const MonarchArgs& a, int nunits, bool kbar_alone) {
    const size_t row = (kbar_alone ? 2 : 4) * a.D + (a.rb ? 128 : 0);
    const size_t least = a.b1 > 32 && !kbar_alone ? 64 : 40;
    return scratch_rows(a, nunits, step1_skips_masked(a)) * row >= least << 20 &&
           scratch_rows(a, nunits, false) * row <= (size_t)(kbar_alone ? 256 : 364) << 20;
}

// From the size on where the memory-side cache holds part of Kbar and Y only, their rows, read once, are read past it: us
// through the caches and past them, 12 heads x 128 of 30 x 52, three frames against 9 (259 MB) 143, 140, 12 (345) 193, 179, in
// half-height blocks (690) 342, 336; 6 heads, 21 frames (302) 155, 146; 40 heads, 21 (2013) 1038, 1002.  Below, they would leave it: 6 heads,
// 12 frames (173 MB) 96.3, 98.6; three frames tied against 21 (201) 146, 149.  Masked pairs count: nine frames of three tied, block-causal, under autograd (165 MiB of
// 247) 465, 460 with their backward.
inline bool step2_past_caches(const MonarchArgs& a, int nunits) {
    return scratch_rows(a, nunits, false) * 4 * a.D >= (size_t)240 << 20;
}

}  // namespace sfm
