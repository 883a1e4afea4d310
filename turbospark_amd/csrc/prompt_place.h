// Which rows of which KV head a workgroup of the prompt attention takes (k_prompt_attn, prompt.hip).  Plain C++, also for the host.
#pragma once

#ifdef __HIP__
#define TSV_BOTH __host__ __device__ __forceinline__
#else
#define TSV_BOTH inline
#endif

namespace tsv {

struct PromptAttnPlace {
    int head, group;  // group g: pairs 128 g .. 128 g + 127 of row and q head of the KV head's
};

// grid: nkv heads times the groups of a head.  The longest rows first, head by head, so that with eight KV heads an XCD has one head's
// K and V in its L2; where everything is in flight at once and a compute unit gets two workgroups (whole: no parts of the context), the
// rows behind the first 256 workgroups' come in the opposite order, a short one beside a long one, each head where it was.  (With all rows
// of one head side by side the two were of one length, and the launch took as long as twice the longest: 8B shape, eight layers, us:
// 2048 rows 8594 -> 8335, 1300 rows 6150 -> 6022, 1500 behind 2000 7820 -> 7698; 64-wide heads, 2000 rows 3148 -> 3058; 1000 rows, one
// workgroup to a compute unit, 4638 -> 4634.  With the heads in the opposite order too, as with the rows alone: 8587 and 8588.)
TSV_BOTH PromptAttnPlace prompt_attn_place(int block, int grid, int nkv, bool whole) {
    const int groups = grid / nkv, first = 256 / nkv;
    int at = block / nkv;
    if (whole && grid > 256 && grid <= 512 && at >= first) at = first + groups - 1 - at;
    return {block % nkv, groups - 1 - at};
}

}  // namespace tsv
