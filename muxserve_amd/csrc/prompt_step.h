// Which prompt steps are one launch (prefill.hip's short form): the rule, for the
// library that launches it and for the operator that chooses between the forms.
#pragma once
#include <algorithm>
#include <cstdint>

namespace mux {

// The waves per workgroup of the launch (one per 32 tokens of the longest prompt), or
// 0 where k is rotated in a launch of its own.
// The short form needs a (prompt, head) to fit one workgroup.  Four waves per
// workgroup where the launch does not fill the chip (two such workgroups per compute
// unit), else as many as the longest prompt needs - unless most prompts would leave
// most of them idle, or hold so few tokens that one row of a wave's 32 is at work (up to
// 1500 (prompt, head)s; two launches / short form: 24 of 4 tokens, 32 heads, 10.6 / 12.4, 40
// of 4 14.5 / 15.6, 24 of 4, 52 heads, 14.4 / 16.0, 16 of 6 14.2 / 12.9; 64 of 2, 32 heads, 18.0 /
// 17.2).  f16, us, two launches (rotation and cache write, attention) /
// rotation of k and the step form / the short form with 1, 2 or 4 waves:
//   32 heads, one prompt of 45 tokens 8.9 / 12.0 / - 10.3 9.0, 16 of 30 16.2 / 14.7 /
//   10.5 - 10.0, 16 of 100 32.0 / 29.9 / - - 21.0, 8 of 128 (40 heads) 26 / 26.7 / - - 18.5;
//   1 wave: 64 of 16 (52 heads) 37.8 / 41.1 / 29.9, 128 of 6 34.5 / 46.3 / 29.5, 200 of 30 110 /
//   99 / 75, 2000 of 1 462 / 540 / 352;
//   2 waves: 64 of 45 51.3 / 48.3 / 41.4, 64 of 64 61.8 / 54.5 / 47.5; 60 and 127 of 6 36.9 / 47.7 /
//   41.6, 32 of 60 and 96 of 6 54.6 / 58.2 / 49.0;
//   4 waves: 64 of 128 131 / 101 / 90, 200 of 100 376 / 317 / 285; 128 and 127 of 20 54.6 / 52.1 /
//   58.0, 128 and 127 of 40 82.8 / 77 / 79.4, 32 of 100 and 32 of 30 (40 heads) 80 / 69 / 64.
// bf16, us, two launches / the short form: 32 heads, one prompt of 20 tokens 8.2 / 7.4, of 45
// 9.7 / 9.4, of 128 12.9 / 12.0, 2 of 91 13.1 / 11.1, 16 of 91 25.8 / 19.3; 52 heads, 8 of 128
// 29.1 / 21.8; 32 heads, 64 of 20 30.7 / 18.0, of 64 55.8 / 48.3, of 91 76.8 / 71.8, of 128 101 /
// 92: the products with the split weights are hidden.
// A few prompts on a few heads are up to a tenth slower as kernels (8 heads, f16, one prompt
// of 70 tokens 9.8 / 10.6, 3 of 33 8.9 / 9.4) and faster as calls, which the host bounds there
// with one launch or two: 32 heads, one prompt of 45 tokens 12.7 / 10.2.
inline int32_t prompt_step_short_waves(const int32_t *prompt_lens_host, int32_t num_prompts, int32_t num_q_heads,
                                       int32_t num_kv_heads) {
  if (!prompt_lens_host || num_prompts <= 0 || num_q_heads != num_kv_heads) return 0;
  int32_t longest = 0;
  int64_t tokens = 0;
  for (int32_t p = 0; p < num_prompts; ++p) {
    longest = std::max(longest, prompt_lens_host[p]);
    tokens += prompt_lens_host[p];
  }
  if (longest > 128) return 0;
  const int64_t groups = static_cast<int64_t>(num_prompts) * num_kv_heads;
  if (groups <= 512) return 4;
  if (longest <= 32) return tokens >= int64_t{6} * num_prompts || groups > 1500 ? 1 : 0;
  if (longest <= 64) return tokens >= int64_t{16} * num_prompts ? 2 : 0;
  return tokens >= int64_t{45} * num_prompts ? 4 : 0;
}

}  // namespace mux
