// Attention of a few query rows over a long key / value cache (decode):
// O = softmax(Q K^T * scale) V with Sq * (Hq / Hkv) <= 16 query rows per key /
// value head.
//
// Bound by streaming K and V from HBM once, which the 128-row kernel does not
// do: it gives every query head a block, so a grouped-query cache is read once
// per query head (through L2), and a block holds two 64-key tiles at most in
// flight.  Here
//  * a work item is (batch, key / value head, slice of the keys), and the
//    Sq * Hq / Hkv query rows that share the head fill the 16 columns of
//    v_mfma_f32_16x16x32 (S^T = K Q^T, so a lane's scores all belong to one
//    query row and P^T feeds O^T += V^T P^T from registers);
//  * every wave owns its own key tiles (16 KiB of K and V each) in its own
//    part of the LDS, loaded by direct DMA two tiles ahead and refilled as
//    soon as the tile's K, then V, has been read: 32 KiB per wave in flight
//    and no barrier before the final merge of the waves;
//    (16, 32 / 8 heads, 1, 4096, 128) bf16: 145 us in the 128-row kernel, here
//    43.3 us (6.2 TB/s; the K and V bytes at the copy's rate are 40.7 us) and
//    4.7 us of merge.
//  * the slices of a head write fp32 partial (max, sum, O) to the caller's
//    workspace and k_attn_merge combines them in slice order.
#include <algorithm>

#include "attention.h"

namespace ntops {
namespace {

constexpr int kDecodeMaxSplit = 64;
constexpr int kDecodeMinKeys = 256;

// v_mfma_f32_16x16x32: lane l holds row / column l & 15 at k = 8 (l >> 4) ..
// + 7 of A / B, and column l & 15, rows 4 (l >> 4) .. + 3 of the result.
template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same<T, __bf16>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

// Keys of one wave's tile: 8 KiB of K and 8 KiB of V.
template <int D>
constexpr int kDecodeTile = 4096 / D;

// dma16 with the non-temporal hint: every byte of the cache is read once, and
// kept out of the way of the lines still in flight it streams at 6.2 instead
// of 5.5 TB/s ((16, 32 / 8, 1, 4096, 128): 43.3 against 49.3 us).
__device__ __forceinline__ void dma16_stream(u32x4 rsrc, uint32_t lds_dst, uint32_t voffset) {
  asm volatile("buffer_load_dwordx4 %0, %1, 0 offen nt lds"
               :
               : "v"(voffset), "s"(rsrc), "{m0}"(lds_dst)
               : "memory");
}

// Loads of one tile's K (or V) rows: 8 instructions of 1 KiB, the swizzle on
// the global side.
template <int D, bool IS_V>
struct DecodeDma {
  static constexpr int kInst = 8;
  static constexpr int kRows = 512 / D;  // rows per instruction
  u32x4 rsrc;
  uint32_t voff[kInst];

  __device__ __forceinline__ void init(const void* base, int64_t ld, uint32_t extent, int lane, int dt) {
    const uint64_t addr = reinterpret_cast<uint64_t>(base);
    rsrc.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr));
    rsrc.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr >> 32) & 0xffffu);
    rsrc.z = __builtin_amdgcn_readfirstlane(extent);
    rsrc.w = 0x00020000u;
    constexpr int cpr = D / 8;
#pragma unroll
    for (int i = 0; i < kInst; ++i) {
      const int row = i * kRows + lane / cpr;
      const int slot = lane % cpr;
      const int c = IS_V ? vslot<D>(row, slot) : kslot<D>(row, slot);
      voff[i] = c * 8 < dt ? static_cast<uint32_t>(row * ld * 2 + c * 16) : kOOB;
    }
  }
  // tile at byte offset `off` of the head's rows into LDS at `dst`; an empty
  // load (off past every extent) still counts in vmcnt
  __device__ __forceinline__ void issue(uint32_t dst, uint32_t off) const {
#pragma unroll
    for (int i = 0; i < kInst; ++i) {
      // kOOB + kOOB would wrap to 0: keep either one
      dma16_stream(rsrc, dst + i * 1024, (voff[i] | off) & kOOB ? kOOB : voff[i] + off);
    }
  }
};

// Reads of LDS filled by DMA must not move across the wait that orders them.
template <int N>
__device__ __forceinline__ void wait_dma() {
  __builtin_amdgcn_sched_barrier(0);
  wait_vmcnt<N>();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// part: fp32, per query row and slice the unnormalised O row, then (max in
// base 2, sum) pairs; null: one slice, O normalised into a.o.
template <typename T, int D, int NW>
__global__ __launch_bounds__(64 * NW, 1) void k_attn_decode(AttnArgs a, int nsplit, int chunk, float* part) {
  constexpr int NK = kDecodeTile<D>;  // keys per tile
  constexpr int KB = NK / 16;         // 16-key blocks of a tile
  constexpr int KS = D / 32;          // k-steps of S^T = K Q^T
  constexpr int DT = D / 16;          // 16-row tiles of O^T
  extern __shared__ __attribute__((aligned(1024))) char smem[];  // [wave][2 stages][K, V]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4;
  const int64_t blk = block_id();
  if (blk >= static_cast<int64_t>(nsplit) * a.B * a.Hkv) return;  // the tail of a 2-D grid (the whole block)
  const int bh = static_cast<int>(blk / nsplit);
  const int sp = static_cast<int>(blk - static_cast<int64_t>(bh) * nsplit);
  const int b = bh / a.Hkv, hk = bh - b * a.Hkv;
  const int group = a.Hq / a.Hkv;
  const int rows = group * a.Sq;  // <= 16
  // query row of this lane's column: head hk * group + r / Sq, position r % Sq
  const int r = lane & 15;
  const int h = hk * group + r / a.Sq, qi = r % a.Sq;
  const int off = a.causal == 2 ? a.Skv - a.Sq : 0;
  int kv_end = a.Skv, lim = a.Skv, lim_min = a.Skv;
  if (a.causal) {
    kv_end = max(0, min(a.Skv, a.Sq + off));
    lim = min(a.Skv, qi + off + 1);
    lim_min = min(a.Skv, off + 1);
  }

  u32x4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = ks * 32 + 8 * g;
    if (r < rows && d0 < a.D)
      qf[ks] = *reinterpret_cast<const u32x4*>(static_cast<const T*>(a.q) + b * a.qs[0] + h * a.qs[1] + qi * a.qs[2] + d0);
    else
      qf[ks] = u32x4{0, 0, 0, 0};
  }
  // settled here, so that no wait for it is placed among the tile loads
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(qf[ks]));

  DecodeDma<D, false> kd;
  DecodeDma<D, true> vd;
  kd.init(static_cast<const T*>(a.k) + b * a.ks[0] + hk * a.ks[1], a.ks[2],
          static_cast<uint32_t>((static_cast<int64_t>(a.Skv - 1) * a.ks[2] + a.D) * 2), lane, a.D);
  vd.init(static_cast<const T*>(a.v) + b * a.vs[0] + hk * a.vs[1], a.vs[2],
          static_cast<uint32_t>((static_cast<int64_t>(a.Skv - 1) * a.vs[2] + a.D) * 2), lane, a.D);
  const int k0 = sp * chunk, k1 = min(kv_end, k0 + chunk);
  const int nt = (k1 - k0 + NK - 1) / NK;                       // tiles of the slice (<= 0: none)
  const int n = nt > wave ? (nt - wave + NW - 1) / NW : 0;      // of this wave: wave, wave + NW, ...
  char* mine = smem + wave * 32768;
  const uint32_t mine_addr = lds_addr(mine);
  auto key_of = [&](int j) { return k0 + (wave + j * NW) * NK; };
  auto issue_k = [&](int j) {
    kd.issue(mine_addr + (j & 1) * 16384, j < n ? static_cast<uint32_t>(key_of(j) * a.ks[2] * 2) : kOOB);
  };
  auto issue_v = [&](int j) {
    vd.issue(mine_addr + (j & 1) * 16384 + 8192, j < n ? static_cast<uint32_t>(key_of(j) * a.vs[2] * 2) : kOOB);
  };

  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = neg_inf(), l = 0.f;  // running max (base 2) of row r; this lane's part of its sum

  issue_k(0);
  issue_v(0);
  issue_k(1);
  issue_v(1);
  for (int j = 0; j < n; ++j) {
    const char* sk = mine + (j & 1) * 16384;
    const char* sv = sk + 8192;
    wait_dma<24>();  // K of tile j is in; its V and tile j + 1 may be in flight
    f32x4 s[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int row = kb * 16 + (lane & 15);
        const u32x4 kf = *reinterpret_cast<const u32x4*>(sk + row * (D * 2) + kslot<D>(row, ks * 4 + g) * 16);
        s[kb] = mfma16<T>(kf, qf[ks], s[kb]);
      }
    wait_lgkmcnt0();
    issue_k(j + 2);

    // scores of keys kt + 16 kb + 4 g + e
    const int kt = key_of(j);
    float mx = neg_inf();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[kb][e] *= a.scale_log2;
    if (kt + NK > lim_min) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[kb][e] = kt + kb * 16 + 4 * g + e < lim ? s[kb][e] : neg_inf();
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[kb][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == neg_inf() ? 0.f : m_new;  // fully masked so far: P = 0
    if (__any(m_new > m)) {
      const float alpha = fast_exp2(m - m_use);
      l *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[t][e] *= alpha;
      m = m_new;
    }
    u32x4 pf[KB / 2];
#pragma unroll
    for (int p = 0; p < KB / 2; ++p) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] = fast_exp2(s[2 * p + (e >> 2)][e & 3] - m_use);
        l += x[e];
      }
      pf[p] = pack8<T>(x);  // keys 32 p + 4 g + 0..3 and 32 p + 16 + 4 g + 0..3
    }

    wait_dma<24>();  // V of tile j is in
#pragma unroll
    for (int p = 0; p < KB / 2; ++p)
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        // V^T: lane row 16 t + (l & 15) at the keys of pf[p]
        const int i = lane & 15;
        const int col = t * 16 + (i & 3) * 4;
        s16x4 w[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int row = p * 32 + u * 16 + g * 4 + (i >> 2);
          w[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_s16x4_t*)(sv + row * (D * 2) + vslot<D>(row, col >> 3) * 16 + ((col >> 2) & 1) * 8));
        }
        const u32x2 lo = __builtin_bit_cast(u32x2, w[0]), hi = __builtin_bit_cast(u32x2, w[1]);
        o[t] = mfma16<T>(u32x4{lo.x, lo.y, hi.x, hi.y}, pf[p], o[t]);
      }
    wait_lgkmcnt0();
    issue_v(j + 2);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  wait_dma<0>();  // no DMA may land in the LDS the merge reuses
  __syncthreads();

  // merge the waves: per-wave (max, sum) of every row, then O scaled to the
  // block's max
  float* sm = reinterpret_cast<float*>(smem);  // [wave][16] max, [wave][16] sum, then [wave][16][D + 4] O
  float* so = sm + 2 * NW * 16;
  constexpr int LD = D + 4;
  if (g == 0) {
    sm[wave * 16 + r] = m;
    sm[(NW + wave) * 16 + r] = l;
  }
  __syncthreads();
  float mb = sm[r];
#pragma unroll
  for (int w = 1; w < NW; ++w) mb = fmaxf(mb, sm[w * 16 + r]);
  const float f = m == neg_inf() ? 0.f : fast_exp2(m - mb);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) so[(wave * 16 + r) * LD + t * 16 + 4 * g + e] = o[t][e] * f;
  __syncthreads();
  const int64_t nrow = static_cast<int64_t>(a.B) * a.Hq * a.Sq;
  float* part_ml = part + nrow * nsplit * a.D;
  for (int i = threadIdx.x; i < rows * (D / 4); i += 64 * NW) {
    const int row = i / (D / 4), d = (i - row * (D / 4)) * 4;
    if (d >= a.D) continue;
    float mm = sm[row];
#pragma unroll
    for (int w = 1; w < NW; ++w) mm = fmaxf(mm, sm[w * 16 + row]);
    float sum = 0.f;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = sm[w * 16 + row];
      sum += sm[(NW + w) * 16 + row] * (mw == neg_inf() ? 0.f : fast_exp2(mw - mm));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += so[(w * 16 + row) * LD + d + e];
    }
    const int hh = hk * group + row / a.Sq, qq = row % a.Sq;
    if (part) {
      const int64_t at = ((static_cast<int64_t>(b) * a.Hq + hh) * a.Sq + qq) * nsplit + sp;
      if (d == 0) {
        part_ml[2 * at] = mm;
        part_ml[2 * at + 1] = sum;
      }
      *reinterpret_cast<f32x4*>(part + at * a.D + d) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      T w4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) w4[e] = static_cast<T>(v[e] * inv);
      *reinterpret_cast<u32x2*>(static_cast<T*>(a.o) + b * a.os[0] + hh * a.os[1] + qq * a.os[2] + d) =
          __builtin_bit_cast(u32x2, w4);
    }
  }
}

// Combines the slices of every query row in slice order: one wave per row.
template <typename T>
__global__ __launch_bounds__(256) void k_attn_merge(AttnArgs a, int nsplit, const float* part) {
  const int lane = threadIdx.x & 63;
  const int64_t nrow = static_cast<int64_t>(a.B) * a.Hq * a.Sq;
  const int64_t row = block_id() * 4 + (threadIdx.x >> 6);
  if (row >= nrow) return;
  const float* po = part + row * nsplit * a.D;
  const float* ml = part + nrow * nsplit * a.D + 2 * row * nsplit;
  const int d = lane * 2;
  const auto load4 = [&](int s0, float2 (&v)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = s0 + u < nsplit && d < a.D ? *reinterpret_cast<const float2*>(po + static_cast<int64_t>(s0 + u) * a.D + d)
                                        : float2{0.f, 0.f};
  };
  float2 v[4];
  load4(0, v);  // in flight while the weights are formed
  float m = neg_inf(), l = 0.f;
  if (lane < nsplit) {
    m = ml[2 * lane];
    l = ml[2 * lane + 1];
  }
  const float mm = wave_max(m);
  const float w = m == neg_inf() ? 0.f : fast_exp2(m - mm);
  const float sum = wave_sum(l * w);
  float x = 0.f, y = 0.f;
  for (int s0 = 0; s0 < nsplit; s0 += 4) {
    if (s0 > 0) load4(s0, v);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float ws = s0 + u < nsplit ? lane_read(w, s0 + u) : 0.f;
      x += ws * v[u].x;
      y += ws * v[u].y;
    }
  }
  if (d < a.D) {
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    const int q = static_cast<int>(row % a.Sq);
    const int64_t bh = row / a.Sq;
    T* O = static_cast<T*>(a.o) + (bh / a.Hq) * a.os[0] + (bh % a.Hq) * a.os[1] + q * a.os[2];
    T v2[2] = {static_cast<T>(x * inv), static_cast<T>(y * inv)};
    *reinterpret_cast<uint32_t*>(O + d) = __builtin_bit_cast(uint32_t, v2);
  }
}

// Slices of the keys per key / value head, and the keys of each (a multiple
// of every wave's tile).  As many slices as leave at most one two-wave block
// per CU: fewer, longer streams read faster ((7, 32 / 8, 1, 9362, 128): 224
// blocks 46.3 us, 504 blocks 57 us, 280 -- a second round for 24 of them --
// 69.6), and none shorter than four tiles a wave, below which the partial
// results and the merge cost what the slices gain.  With two heads per CU or
// more nothing is split and one-wave blocks, five to a CU, hide each other's
// start ((32, 32, 1, 300, 128): 29.5 against 32.0 us; with fewer heads two
// waves win, (16, 32 / 8, 1, 4096, 128) 47.0 against 68.9).
void decode_split(int64_t heads, int Skv, int D, int& waves, int& nsplit, int& chunk) {
  waves = heads < 2 * cu_count_cached() ? 2 : 1;
  const int step = (D > 64 ? 32 : 64) * waves;
  int64_t n = std::min({static_cast<int64_t>(kDecodeMaxSplit), cu_count_cached() / heads, ceil_div(Skv, 4 * step)});
  if (n <= 2 && Skv <= 8 * step) n = 1;  // two short slices gain what the merge's launch costs
  n = std::max<int64_t>(n, 1);
  chunk = static_cast<int>(ceil_div(ceil_div(Skv, n), step)) * step;
  nsplit = static_cast<int>(ceil_div(Skv, chunk));
}

// Few heads over a short cache stay on the 128-row kernel: four waves share
// the tiles of a head there ((8, 32 / 8, 1, 256, 128): 11.8 us, here 14.6);
// from a head per CU on every byte counts ((32, 32 / 8, 1, 256, 64): 15.6
// against 10.9 us, (32, 32, 1, 256, 128): 34.8 against 28.8).
bool decode_pays(int64_t heads, int64_t Skv) { return Skv > kDecodeMinKeys || heads >= cu_count_cached(); }

template <typename T, int D, int NW>
int launch_decode(const AttnArgs& a, int nsplit, int chunk, float* part, hipStream_t st) {
  constexpr int kLds = NW * 32768;
  static_assert(kLds <= 65536 && (2 * NW * 16 + NW * 16 * (D + 4)) * 4 <= kLds, "LDS");
  const int64_t blocks = static_cast<int64_t>(nsplit) * a.B * a.Hkv;
  note_kernel("sdpa_decode d%d waves%d split%d", D, NW, nsplit);
  hipLaunchKernelGGL((k_attn_decode<T, D, NW>), blocks_2d(blocks), dim3(64 * NW), kLds, st, a, nsplit, chunk,
                     part);
  if (part) {
    const int64_t rows = static_cast<int64_t>(a.B) * a.Hq * a.Sq;
    hipLaunchKernelGGL((k_attn_merge<T>), blocks_2d(ceil_div(rows, 4)), dim3(256), 0, st, a, nsplit, part);
  }
  return check_launch("sdpa");
}

template <typename T>
int run_decode(const AttnArgs& a, void* ws, int64_t ws_bytes, hipStream_t st) {
  int waves, nsplit, chunk;
  decode_split(static_cast<int64_t>(a.B) * a.Hkv, a.Skv, a.D, waves, nsplit, chunk);
  const int64_t need = attn_decode_workspace(a.B, a.Hq, a.Hkv, a.Sq, a.Skv, a.D);
  if (need == 0 || ws == nullptr || ws_bytes < need || !aligned16(ws)) {
    nsplit = 1;
    chunk = a.Skv;
    ws = nullptr;
  }
  float* part = static_cast<float*>(ws);
  if (waves == 1)
    return a.D > 64 ? launch_decode<T, 128, 1>(a, nsplit, chunk, part, st)
                    : launch_decode<T, 64, 1>(a, nsplit, chunk, part, st);
  return a.D > 64 ? launch_decode<T, 128, 2>(a, nsplit, chunk, part, st)
                  : launch_decode<T, 64, 2>(a, nsplit, chunk, part, st);
}

}  // namespace

bool attn_decode_serves(const AttnArgs& a) {
  const auto rows16 = [](const int64_t* s) { return s[3] == 1 && s[2] % 8 == 0 && s[1] % 8 == 0 && s[0] % 8 == 0; };
  const int64_t ld = std::max(a.ks[2], a.vs[2]);
  // (an empty cache has no tile to slice: the general kernel writes its zeros)
  return a.mask_dtype < 0 && a.Skv > 0 && decode_pays(static_cast<int64_t>(a.B) * a.Hkv, a.Skv) &&
         static_cast<int64_t>(a.Sq) * (a.Hq / a.Hkv) <= 16 && a.D % 8 == 0 && a.D <= 128 && rows16(a.qs) &&
         rows16(a.ks) && rows16(a.vs) && a.os[3] == 1 && a.os[2] % 4 == 0 && a.os[1] % 4 == 0 && a.os[0] % 4 == 0 && aligned16(a.q) && aligned16(a.k) &&
         aligned16(a.v) && (reinterpret_cast<uintptr_t>(a.o) & 7u) == 0 && a.ks[2] >= a.D && a.vs[2] >= a.D &&
         (static_cast<int64_t>(a.Skv) + 64) * ld * 2 < 0x7fffffffLL &&
         static_cast<int64_t>(a.B) * a.Hkv <= 0x7fffffffLL / kDecodeMaxSplit;
}

int64_t attn_decode_workspace(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Skv, int64_t D) {
  if (!decode_pays(B * Hkv, Skv) || Sq * (Hq / Hkv) > 16 || D % 8 != 0 || D > 128) return 0;
  int waves, nsplit, chunk;
  decode_split(B * Hkv, static_cast<int>(Skv), static_cast<int>(D), waves, nsplit, chunk);
  return nsplit > 1 ? B * Hq * Sq * nsplit * (D + 2) * 4 : 0;
}

int attn_decode(int dtype, const AttnArgs& a, void* workspace, int64_t workspace_bytes, hipStream_t st) {
  return dtype == NTOPS_BF16 ? run_decode<__bf16>(a, workspace, workspace_bytes, st)
                             : run_decode<_Float16>(a, workspace, workspace_bytes, st);
}

}  // namespace ntops
