// Shared by the attention kernels (attention.hip, attn_decode.hip).
#pragma once

#include "mfma.h"

namespace ntops {

struct AttnArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* mask;
  void* o;
  int64_t qs[4], ks[4], vs[4], ms[4], os[4];
  int B, Hq, Hkv, Sq, Skv, D;
  int mask_dtype;    // -1: none; NTOPS_BOOL (true = attend), NTOPS_F32 / F16 / BF16 (additive)
  int causal;        // 0: none, 1: upper-left (kv <= q), 2: lower-right (kv <= q + Skv - Sq)
  float scale_log2;  // scale * log2(e)
};

constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float neg_inf() { return -__builtin_huge_valf(); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Chunk slot of 16-byte chunk c of key row r in the V tile ([kv][d] with
// D / 8 chunks per row), conflict-free for the transposing fragment reads.
template <int D>
__device__ __forceinline__ int vslot(int r, int c) {
  if constexpr (D == 128)
    return mnslot(r, c);
  else
    return c ^ (((r >> 1) & 1) << 2);
}

// True when attn_decode serves this problem: 16-bit data whose head dim and
// rows suit the matrix cores, no explicit mask, at most 16 query rows per key
// / value head, and more than kDecodeMinKeys keys -- or any but none, where
// every CU gets a key / value head.
bool attn_decode_serves(const AttnArgs& a);
// Bytes of workspace with which attn_decode splits the keys over more blocks
// (0: one block per key / value head is as good).
int64_t attn_decode_workspace(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Skv, int64_t D);
// Runs it; a missing or short workspace runs one block per key / value head.
int attn_decode(int dtype, const AttnArgs& a, void* workspace, int64_t workspace_bytes, hipStream_t st);

}  // namespace ntops
