// Internal interface between linear_recurrence.hip and its chunk-parallel form (chunk_recurrence.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/vlm_hip.h"

#define VLM_CHUNK 64              // tokens per chunk
#define VLM_CHUNK_MIN 17          // segments of at least this many tokens take the chunk-parallel form, where a step runs it
// From which longest segment on a step runs it.  Unrotated fixed decay: 17.  Rotated and gated heads, whose chunks cost a pass over q and k
// or the gates first: where one segment's time by tokens (about 9 + 0.77 a token) crosses that in chunks, us, 12 / 28 heads, rotated (gated is some 10 later on both
// sides): heads of 64, 33 tokens 34 / 34 by tokens, 31 / 34 in chunks; 128, 64 tokens 55 / 55, 56 / 62; 100 tokens 81 / 82, 57 / 63; 256, 100 tokens 90 / 92, 88 / 110;
// 200 tokens 171 / 195, 101 / 126.  (At 17 everywhere short prompts lost by two to five: 32 segments of 18 tokens, 12 heads of 128: 37 by tokens, 120.  The
// lengths are on the device: a caller that knows them and finds a step faster by tokens brings no workspace.)
static inline int vlm_chunk_from(const vlm_recurrence_args* a) { return a->gated != 1 && !a->rot_dims ? VLM_CHUNK_MIN : a->D <= 64 ? 40 : a->D <= 128 ? 72 : 100; }

// what the form keeps at the head of the workspace: rotated q and k, or F (fp64) and the input gate of every (token, head), in whole 16 bytes
static inline long vlm_chunk_prep_floats(const vlm_recurrence_args* a, int ntok) {
  const long n = a->gated == 1 ? 3 * (long)ntok * a->H : a->rot_dims ? 2 * (long)ntok * a->H * a->D : 0;
  return (n + 3) & ~3L;
}

// the raw read-outs and states of the segments of more than max_len tokens (the other segments are left alone)
__attribute__((visibility("hidden"))) int vlm_chunk_recurrence(const vlm_recurrence_args* a, int nseg, int ntok, int max_len, int dtype, hipStream_t st);
