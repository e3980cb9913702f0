// Shared by the GEMM kernels (gemm.hip, gemm_large.hip): the problem's
// arguments, operand tile loads and fragments, and the output stores.
#pragma once

#include "mfma.h"

namespace ntops {

struct GemmArgs {
  const void* A;
  const void* B;
  const void* C;
  void* D;
  int64_t sa_b, sa_m, sa_k;
  int64_t sb_b, sb_k, sb_n;
  int64_t sc_b, sc_m, sc_n;
  int64_t sd_b, sd_m, sd_n;
  int M, N, K, batch;
  float alpha, beta;
  int use_c;
  int c_mode;  // epilogue's C access (kCNone / kCStrided / kCVec4 / kCRow), set by set_c_mode
  int staged;  // out is 16-byte aligned with unit column stride and N % 8 == 0
  int ragged;  // out rows are not 8-byte aligned runs with unit column stride: element stores
  int shifted;  // unit column stride, rows not 16-byte aligned: full-tile kernels store shifted 16-byte chunks
  // Split-K (the SPLITK instantiation): block row blockIdx.y takes k in
  // [blockIdx.y * kchunk, min(K, (blockIdx.y + 1) * kchunk)) and writes its
  // fp32 partial tile to part + blockIdx.y * part_stride (rows of N).
  float* part;          // the workspace (null: no split-K)
  int64_t part_bytes;   // its size
  int64_t part_stride;  // M * N
  int kchunk;
  // Implicit convolution operand (used only by the CONV instantiation): B's
  // k-row kg = (c * R + r) * S + s starts at element
  // s * cv_per_s + c * cv_per_c + r * cv_per_r of the batch's B buffer, and
  // its N elements are contiguous from there.
  int cv_rs, cv_r, cv_s;
  int cv_ds, cv_dr, cv_dc;  // BK k-rows expressed as (s, r, c) steps: BK = (dc * R + dr) * S + ds
  int64_t cv_per_s, cv_per_c, cv_per_r;
  // Channels-last convolution operand (CONV == 2): B is K-major with one row
  // per output pixel n of the batch's image, p = n / cl_q, q = n % cl_q,
  // starting at element (p * cl_sh * cl_wp + q * cl_sw) * cl_c of the
  // batch's zero-padded (rows of cl_wp pixels, cl_c channels each) image.
  // k runs over 32-channel blocks, then taps, then the block's channels:
  // k = ((cb * cv_r + r) * cv_s + s) * 32 + ci adds (r * cl_dh * cl_wp +
  // s * cl_dw) * cl_c + 32 * cb + ci, so one K tile is one (block, tap) and
  // the R * S tiles of a block, which read overlapping pixels, follow each
  // other (the reuse stays within L2).
  // The 64-deep kernel (gemm_large.hip) runs over 64-channel blocks instead
  // and divides by multiplication: ceil(2^32 / cl_q), and ceil(2^16 / d) for
  // d = cv_rs and cv_s.
  int cl_q, cl_sh, cl_sw, cl_wp, cl_c, cl_dh, cl_dw;
  uint32_t cl_mq, cl_mrs, cl_ms;
};


// Waits until at most `younger` tiles' worth of this wave's DMA loads
// (loads_per_tile each) are still in flight.
__device__ __forceinline__ void wait_tile(int younger, int loads_per_tile) {
  const int n = younger * loads_per_tile;
  if (n >= 12)
    wait_vmcnt<12>();
  else if (n >= 8)
    wait_vmcnt<8>();
  else if (n >= 6)
    wait_vmcnt<6>();
  else if (n >= 4)
    wait_vmcnt<4>();
  else if (n >= 2)
    wait_vmcnt<2>();
  else
    wait_vmcnt<0>();
}

// Maps a linear workgroup id to (batch, tile_m, tile_n).
__device__ __forceinline__ void tile_of(int pid, int nblocks, int tm_count, int tn_count,
                                        int& bat, int& tm, int& tn) {
  if ((nblocks & 7) == 0) pid = (pid & 7) * (nblocks >> 3) + (pid >> 3);
  const int per_batch = tm_count * tn_count;
  bat = pid / per_batch;
  const int t = pid - bat * per_batch;
  constexpr int kGroupM = 4;  // 4 measured ~0.7 % over 8 and 2 on mm, 16 ~2.5 % below
  const int group_size = kGroupM * tn_count;
  const int g = t / group_size;
  const int first_m = g * kGroupM;
  const int gm = min(tm_count - first_m, kGroupM);
  const int r = t - g * group_size;
  tm = first_m + r % gm;
  tn = r / gm;
}


// One operand's global -> LDS stream for a tile of R rows/columns x BK k.
// The tile is R * BK * 2 bytes: R * BK / 512 one-KiB load instructions,
// spread evenly over the NW waves of the block.
// CONV: 0 a plain operand; 1 the shifted-plane convolution operand (N-major,
// per-lane k-row bases); 2 the channels-last convolution operand (K-major,
// per-lane pixel bases plus one scalar offset per K tile).
template <int R, bool KMAJ, int NW, bool EVEN, int BK, int CONV = 0>
struct TileLoader {
  static_assert(CONV != 1 || !KMAJ, "the shifted-plane convolution operand is N-major");
  static_assert(CONV != 2 || KMAJ, "the channels-last convolution operand is K-major");
  static constexpr int kInst = R * BK / 512 / NW;
  static_assert(kInst * NW * 512 == R * BK, "tile must split evenly over the waves");
  static constexpr int kCprK = BK / 8;  // chunks per row (K-major)
  static constexpr int kCprMN = R / 8;  // chunks per k-row (M/N-major)
  u32x4 rsrc;             // buffer resource (V#) of the operand tile
  uint32_t voff[kInst];   // byte offset of this lane's chunk at k0 = 0
  int lim_row[kInst];     // K-major: tile row; M/N-major: k-row
  int lim_col[kInst];     // K-major: k of the chunk; M/N-major: column of the chunk
  uint32_t k_stride_bytes;
  int lds_base;           // first instruction's LDS offset inside the operand tile
  // implicit convolution (CONV): this lane's k-row of each instruction for
  // the next tile to issue, as (c, r, s) -- advanced by BK per tile
  int cv_c[CONV == 1 ? kInst : 1], cv_r[CONV == 1 ? kInst : 1], cv_s[CONV == 1 ? kInst : 1];
  // channels-last convolution (CONV == 2): the tap (r, s) and first channel
  // c0 of the next K tile to issue
  int cl_r = 0, cl_s = 0, cl_c0 = 0;

  // base: element pointer at the tile origin; ld: row stride (K-major) or
  // k-row stride (M/N-major), in elements; extent_bytes: readable bytes.
  __device__ __forceinline__ void init(const uint16_t* base, int64_t ld, int64_t extent_bytes,
                                       int wave, int lane) {
    const uint64_t addr = reinterpret_cast<uint64_t>(base);
    rsrc.x = static_cast<uint32_t>(addr);
    rsrc.y = static_cast<uint32_t>(addr >> 32) & 0xffffu;  // stride 0, no swizzle
    rsrc.z = static_cast<uint32_t>(extent_bytes);           // num_records (bytes)
    rsrc.w = 0x00020000u;                                   // 32-bit data format
    rsrc.x = __builtin_amdgcn_readfirstlane(rsrc.x);
    rsrc.y = __builtin_amdgcn_readfirstlane(rsrc.y);
    rsrc.z = __builtin_amdgcn_readfirstlane(rsrc.z);
    lds_base = wave * kInst * 1024;
    if constexpr (KMAJ) {
      k_stride_bytes = 2;
      constexpr int rows_per_inst = 1024 / (BK * 2);
#pragma unroll
      for (int i = 0; i < kInst; ++i) {
        const int q = wave * kInst + i;
        const int row = q * rows_per_inst + lane / kCprK;
        const int c = kslot<BK>(row, lane % kCprK);
        voff[i] = static_cast<uint32_t>(row * ld * 2 + c * 16);
        lim_row[i] = row;
        lim_col[i] = c * 8;
      }
    } else {
      k_stride_bytes = static_cast<uint32_t>(ld * 2);
      constexpr int rows_per_inst = 64 / kCprMN;
#pragma unroll
      for (int i = 0; i < kInst; ++i) {
        const int q = wave * kInst + i;
        const int krow = q * rows_per_inst + lane / kCprMN;
        const int c = mnslot(krow, lane % kCprMN);
        voff[i] = static_cast<uint32_t>((CONV == 1 ? 0 : krow * ld * 2) + c * 16);
        lim_row[i] = krow;
        lim_col[i] = c * 8;
      }
    }
  }

  // Channels-last convolution: each instruction's row is output pixel
  // n0 + row; its offset becomes that pixel's element in the padded image
  // (rows past the image's last pixel keep a valid offset and are rejected
  // by lim_row when !EVEN).
  __device__ __forceinline__ void conv_cl_init(const GemmArgs& g, int n0) {
    if constexpr (CONV == 2) {
#pragma unroll
      for (int i = 0; i < kInst; ++i) {
        const int n = min(n0 + lim_row[i], g.N - 1);
        const int p = n / g.cl_q, q = n - p * g.cl_q;
        const int64_t pix = (static_cast<int64_t>(p) * g.cl_sh * g.cl_wp + static_cast<int64_t>(q) * g.cl_sw) * g.cl_c;
        voff[i] = static_cast<uint32_t>(pix * 2 + lim_col[i] * 2);
      }
    }
  }

  // Implicit convolution: the (c, r, s) of each instruction's k-row at
  // k0 = 0 (k-row kg = (c * R + r) * S + s).
  __device__ __forceinline__ void conv_init(const GemmArgs& g) {
    if constexpr (CONV == 1) {
#pragma unroll
      for (int i = 0; i < kInst; ++i) {
        const int kg = lim_row[i];
        cv_c[i] = kg / g.cv_rs;
        const int rs = kg - cv_c[i] * g.cv_rs;
        cv_r[i] = rs / g.cv_s;
        cv_s[i] = rs - cv_r[i] * g.cv_s;
      }
    }
  }

  // Moves the resource to another tile origin with the same leading
  // dimension and extent (the per-lane offsets stay valid).
  __device__ __forceinline__ void rebase(const uint16_t* base) {
    const uint64_t addr = reinterpret_cast<uint64_t>(base);
    rsrc.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr));
    rsrc.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr >> 32) & 0xffffu);
  }

  // Issues the loads of the K tile starting at k0 into LDS at the 32-bit
  // LDS address `lds` (this operand's tile in one LDS stage; the kernels
  // form it from the LDS base once: a generic -> LDS pointer cast per load
  // instruction carries a null test, 3-4 scalar instructions each).
  // `valid` is the number of valid tile rows (K-major) or tile columns
  // (M/N-major); K bounds the k axis.
  // CONV: tiles must be issued in order k0 = 0, BK, 2 BK, ... (each call
  // advances the (c, r, s) state by BK k-rows).
  __device__ __forceinline__ void issue(uint32_t lds, int k0, int valid, int K, const GemmArgs* cv = nullptr) {
    // channels-last: the tile's (channel block, tap) offset in bytes, then
    // advance to the next K tile's: the next tap, after the last tap the
    // next block
    uint32_t cl_off = 0;
    if constexpr (CONV == 2) {
      static_assert(BK == 32, "one K tile is one 32-channel block under one tap");
      cl_off = static_cast<uint32_t>(((cl_r * cv->cl_dh * cv->cl_wp + cl_s * cv->cl_dw) * cv->cl_c + cl_c0) * 2);
      if (++cl_s >= cv->cv_s) {
        cl_s = 0;
        if (++cl_r >= cv->cv_r) {
          cl_r = 0;
          cl_c0 += BK;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kInst; ++i) {
      uint32_t off;
      if constexpr (CONV == 1) {
        // row base of k-row (c, r, s), then advance it by BK k-rows
        const int64_t base = cv_s[i] * cv->cv_per_s + cv_c[i] * cv->cv_per_c + cv_r[i] * cv->cv_per_r;
        off = voff[i] + static_cast<uint32_t>(base * 2);
        cv_s[i] += cv->cv_ds;
        const int cs = cv_s[i] >= cv->cv_s ? 1 : 0;
        cv_s[i] -= cs * cv->cv_s;
        cv_r[i] += cv->cv_dr + cs;
        const int cr = cv_r[i] >= cv->cv_r ? 1 : 0;
        cv_r[i] -= cr * cv->cv_r;
        cv_c[i] += cv->cv_dc + cr;
      } else if constexpr (CONV == 2) {
        off = voff[i] + cl_off;
      } else {
        off = voff[i] + static_cast<uint32_t>(k0) * k_stride_bytes;
      }
      if constexpr (!EVEN) {
        bool ok;
        if constexpr (KMAJ)
          ok = lim_row[i] < valid && k0 + lim_col[i] < K;
        else
          ok = k0 + lim_row[i] < K && lim_col[i] < valid;
        off = ok ? off : kOOB;
      }
      dma16(rsrc, lds + static_cast<uint32_t>(lds_base + i * 1024), off);
    }
  }
};

// Fragment of one 32-row (m or n) x 16 k operand slice for lane `lane`:
// lane l holds row (l & 31), k = 8 * (l >> 5) + 0..7.
template <int R, bool KMAJ, int BK>
__device__ __forceinline__ u32x4 load_frag(const char* tile, int row0, int ks, int lane) {
  if constexpr (KMAJ) {
    const int r = row0 + (lane & 31);
    const int c = ks * 2 + (lane >> 5);
    return *reinterpret_cast<const u32x4*>(tile + r * (BK * 2) + kslot<BK>(r, c) * 16);
  } else {
    // ds_read_b64_tr_b16: within each 16-lane group, source lane i reads
    // 4 elements of k-row kb + i/4 at columns nb + 4 (i % 4) .. +3; output
    // lane j receives column nb + j at k-rows kb .. kb + 3.
    const int i = lane & 15;
    const int n = row0 + ((lane >> 4) & 1) * 16 + (i & 3) * 4;
    const int c = n >> 3, half = (n >> 2) & 1;
    s16x4 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = ks * 16 + (lane >> 5) * 8 + h * 4 + (i >> 2);
      const char* p = tile + k * (R * 2) + mnslot(k, c) * 16 + half * 8;
      v[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p));
    }
    u32x4 r;
    r.x = static_cast<uint16_t>(v[0][0]) | (static_cast<uint32_t>(static_cast<uint16_t>(v[0][1])) << 16);
    r.y = static_cast<uint16_t>(v[0][2]) | (static_cast<uint32_t>(static_cast<uint16_t>(v[0][3])) << 16);
    r.z = static_cast<uint16_t>(v[1][0]) | (static_cast<uint32_t>(static_cast<uint16_t>(v[1][1])) << 16);
    r.w = static_cast<uint16_t>(v[1][2]) | (static_cast<uint32_t>(static_cast<uint16_t>(v[1][3])) << 16);
    return r;
  }
}

// ---- epilogue --------------------------------------------------------------
// With B as the first MFMA operand, lane l of 32x32 tile (i, j) holds output
// row  m = l & 31  and columns  n = 8q + 4(l >> 5) + 0..3  in
// acc[i][j][4q .. 4q+3].  alpha / beta are applied in fp32 and each value is
// rounded once.  (mw, nw) is the wave tile's origin in the output; D and Cp
// already point at the batch's matrices.  The C access mode CM is a template
// parameter so the C test is not a branch per element:
//   kCNone     no C;
//   kCStrided  one load per element (any strides);
//   kCVec4     unit column stride, rows and batches 8-byte aligned: a lane's
//              4 consecutive columns in one 8-byte load (addmm's bias row
//              and full C matrices);
//   kCRow      column stride 0: one value per row (conv2d's bias).
constexpr int kCNone = 0, kCStrided = 1, kCVec4 = 2, kCRow = 3;

// beta * C at (m, n .. n + 3) in fp32 (zeros where `ok` is false, i.e.
// past the output's edge: no load is issued there).
template <typename T, int CM>
__device__ __forceinline__ void c_values(const GemmArgs& g, const T* Cp, int m, int n, bool ok, float (&c)[4]) {
  if constexpr (CM == kCVec4) {
    u32x2 raw = {0u, 0u};
    if (ok) raw = *reinterpret_cast<const u32x2*>(Cp + static_cast<int64_t>(m) * g.sc_m + n);
    const T* t = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] = g.beta * static_cast<float>(t[e]);
  } else if constexpr (CM == kCRow) {
    const float v = ok ? g.beta * static_cast<float>(Cp[static_cast<int64_t>(m) * g.sc_m]) : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      c[e] = (CM == kCStrided && ok) ? g.beta * static_cast<float>(Cp[m * g.sc_m + (n + e) * g.sc_n]) : 0.f;
  }
}

template <typename T, int CM, int TM, int TN>
__device__ __forceinline__ float final_value(const GemmArgs& g, const f32x16 (&acc)[TM][TN], const float (&c)[4],
                                             int i, int j, int q, int e) {
  float v = g.alpha * acc[i][j][4 * q + e];
  if constexpr (CM != kCNone) v += c[e];
  return v;
}

// Staged store: the wave writes its rounded WTM x WTN tile into its own LDS
// region `ep` (rows of WTN * 2 bytes, 16-byte chunk c of row r at slot
// c ^ ((r >> 1) & 7)), reads it back row by row (stage_tile), then streams
// it out with 16-byte stores, 8 lanes per 128-byte row segment, so every L2
// write request is a full line instead of 16 bytes (store_rows: exactly
// WTM / 8 store instructions when EVEN).
template <typename T, int CM, int TM, int TN, int WTM, int WTN, bool EVEN>
__device__ __forceinline__ void stage_tile(const GemmArgs& g, const f32x16 (&acc)[TM][TN], char* ep,
                                           const T* Cp, int mw, int nw, int lane,
                                           u32x4 (&rows)[WTM / 8]) {
  static_assert(WTN * 2 == 128, "staged epilogue assumes 64-column wave tiles");
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = i * 32 + (lane & 31);
    const int m = mw + r;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = j * 32 + q * 8 + (lane >> 5) * 4;
        const int n = nw + col;
        T o[4];
        // N % 4 == 0 on this path, so columns n .. n + 3 are all in or all out
        float cv[4];
        c_values<T, CM>(g, Cp, m, n, EVEN || (m < g.M && n < g.N), cv);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool ok = EVEN || (m < g.M && n + e < g.N);
          o[e] = static_cast<T>(ok ? final_value<T, CM>(g, acc, cv, i, j, q, e) : 0.f);
        }
        const int c = col >> 3, half = (col >> 2) & 1;
        *reinterpret_cast<u32x2*>(ep + r * 128 + ((c ^ ((r >> 1) & 7)) << 4) + half * 8) =
            __builtin_bit_cast(u32x2, o);
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int r0 = 0; r0 < WTM; r0 += 8) {
    const int r = r0 + (lane >> 3), c = lane & 7;
    rows[r0 / 8] = *reinterpret_cast<const u32x4*>(ep + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
  }
}

template <typename T, int WTM, bool EVEN, bool NT>
__device__ __forceinline__ void store_rows(const GemmArgs& g, const u32x4 (&rows)[WTM / 8], T* D,
                                           int mw, int nw, int lane) {
#pragma unroll
  for (int r0 = 0; r0 < WTM; r0 += 8) {
    const int r = r0 + (lane >> 3), c = lane & 7;
    const int m = mw + r;
    const int n = nw + c * 8;
    if (EVEN || (m < g.M && n < g.N)) {
      u32x4* dst = reinterpret_cast<u32x4*>(D + static_cast<int64_t>(m) * g.sd_m + n);
      if constexpr (NT)
        __builtin_nontemporal_store(rows[r0 / 8], dst);
      else
        *dst = rows[r0 / 8];
    }
  }
}

// Staged rows of a 16-bit output whose rows start anywhere (2-byte aligned):
// each wave-tile row segment is 64 columns = 128 bytes at byte address G0 with
// s = G0 % 16.  Lane c of the row's 8 lanes (holding columns 8c .. 8c + 7)
// writes the aligned 16-byte chunk that starts 16 (c + 1) - s bytes into the
// segment (c < 7): the top s bytes of its own chunk and the low 16 - s of the
// next lane's; lane 0 also writes the segment's first (16 - s) / 2 columns and
// lane 7 its last s / 2, element by element.  Every store stays inside the
// segment.  Full tiles only (EVEN): no column of a segment lies past N.
template <typename T, int WTM, bool NT>
__device__ __forceinline__ void store_rows_shifted(const GemmArgs& g, const u32x4 (&rows)[WTM / 8], T* D,
                                                   int mw, int nw, int lane) {
  static_assert(sizeof(T) == 2, "16-bit outputs");
#pragma unroll
  for (int r0 = 0; r0 < WTM; r0 += 8) {
    const int r = r0 + (lane >> 3), c = lane & 7;
    const u32x4 cur = rows[r0 / 8];
    u32x4 nxt;
    nxt.x = static_cast<uint32_t>(__shfl_down(static_cast<int>(cur.x), 1, 8));
    nxt.y = static_cast<uint32_t>(__shfl_down(static_cast<int>(cur.y), 1, 8));
    nxt.z = static_cast<uint32_t>(__shfl_down(static_cast<int>(cur.z), 1, 8));
    nxt.w = static_cast<uint32_t>(__shfl_down(static_cast<int>(cur.w), 1, 8));
    T* seg = D + static_cast<int64_t>(mw + r) * g.sd_m + nw;
    const uint32_t s = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(seg)) & 15u;
    if (s == 0) {
      u32x4* dst = reinterpret_cast<u32x4*>(seg + 8 * c);
      if constexpr (NT)
        __builtin_nontemporal_store(cur, dst);
      else
        *dst = cur;
      continue;
    }
    // (cur | nxt) >> 8 * (16 - s) bits, as 64-bit halves
    const uint64_t x0 = cur.x | (static_cast<uint64_t>(cur.y) << 32), x1 = cur.z | (static_cast<uint64_t>(cur.w) << 32);
    const uint64_t x2 = nxt.x | (static_cast<uint64_t>(nxt.y) << 32), x3 = nxt.z | (static_cast<uint64_t>(nxt.w) << 32);
    const uint32_t sh = 8u * (16u - s);  // 16 .. 112 bits
    uint64_t o0, o1;
    if (sh < 64) {
      o0 = (x0 >> sh) | (x1 << (64 - sh));
      o1 = (x1 >> sh) | (x2 << (64 - sh));
    } else if (sh == 64) {
      o0 = x1;
      o1 = x2;
    } else {
      const uint32_t k = sh - 64;
      o0 = (x1 >> k) | (x2 << (64 - k));
      o1 = (x2 >> k) | (x3 << (64 - k));
    }
    char* base = reinterpret_cast<char*>(seg) - s;  // the 16-byte aligned address below G0
    if (c < 7) {
      const u32x4 v = {static_cast<uint32_t>(o0), static_cast<uint32_t>(o0 >> 32), static_cast<uint32_t>(o1),
                       static_cast<uint32_t>(o1 >> 32)};
      u32x4* dst = reinterpret_cast<u32x4*>(base + 16 * (c + 1));
      if constexpr (NT)
        __builtin_nontemporal_store(v, dst);
      else
        *dst = v;
    }
    auto elem = [&](uint32_t e) -> uint16_t {
      const uint32_t d = e < 2 ? cur.x : e < 4 ? cur.y : e < 6 ? cur.z : cur.w;
      return static_cast<uint16_t>(d >> (16 * (e & 1)));
    };
    uint16_t* seg16 = reinterpret_cast<uint16_t*>(seg);
    if (c == 0)
      for (uint32_t e = 0; e < (16u - s) / 2; ++e) seg16[e] = elem(e);
    if (c == 7)
      for (uint32_t e = 8 - s / 2; e < 8; ++e) seg16[56 + e] = elem(e);
  }
}

template <typename T, int CM, int TM, int TN, int WTM, int WTN, bool EVEN, bool NT>
__device__ __forceinline__ void store_tile_shifted(const GemmArgs& g, const f32x16 (&acc)[TM][TN],
                                                   char* ep, T* D, const T* Cp, int mw, int nw, int lane) {
  u32x4 rows[WTM / 8];
  stage_tile<T, CM, TM, TN, WTM, WTN, EVEN>(g, acc, ep, Cp, mw, nw, lane, rows);
  store_rows_shifted<T, WTM, NT>(g, rows, D, mw, nw, lane);
}

template <typename T, int CM, int TM, int TN, int WTM, int WTN, bool EVEN, bool NT>
__device__ __forceinline__ void store_tile_staged(const GemmArgs& g, const f32x16 (&acc)[TM][TN],
                                                  char* ep, T* D, const T* Cp, int mw, int nw,
                                                  int lane) {
  u32x4 rows[WTM / 8];
  stage_tile<T, CM, TM, TN, WTM, WTN, EVEN>(g, acc, ep, Cp, mw, nw, lane, rows);
  store_rows<T, WTM, EVEN, NT>(g, rows, D, mw, nw, lane);
}

// Direct store: 8-byte stores of each lane's 4 consecutive columns (any
// output row stride that keeps 8-byte alignment), element stores at the edge.
template <typename T, int CM, int TM, int TN, bool EVEN>
__device__ __forceinline__ void store_tile_direct(const GemmArgs& g, const f32x16 (&acc)[TM][TN],
                                                  T* D, const T* Cp, int mw, int nw, int lane) {
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = mw + i * 32 + (lane & 31);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = nw + j * 32 + q * 8 + (lane >> 5) * 4;
        if (g.ragged) {
          // rows of any stride, N of any width: element stores, C read per element
          if (m < g.M) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (n + e < g.N) {
                float cv[4] = {0.f, 0.f, 0.f, 0.f};
                if constexpr (CM != kCNone)
                  cv[e] = g.beta * static_cast<float>(Cp[m * g.sc_m + (n + e) * g.sc_n]);
                D[static_cast<int64_t>(m) * g.sd_m + static_cast<int64_t>(n + e) * g.sd_n] =
                    static_cast<T>(final_value<T, CM>(g, acc, cv, i, j, q, e));
              }
            }
          }
          continue;
        }
        if (!EVEN && m < g.M && n < g.N && n + 3 >= g.N) {
          // the last, partial 4-column group of a row (N % 4 != 0)
#pragma unroll
          for (int e = 0; e < 3; ++e) {
            if (n + e < g.N) {
              float cv[4] = {0.f, 0.f, 0.f, 0.f};
              if constexpr (CM != kCNone)
                cv[e] = g.beta * static_cast<float>(Cp[m * g.sc_m + (n + e) * g.sc_n]);
              D[static_cast<int64_t>(m) * g.sd_m + n + e] = static_cast<T>(final_value<T, CM>(g, acc, cv, i, j, q, e));
            }
          }
          continue;
        }
        if (EVEN || (m < g.M && n + 3 < g.N)) {
          float cv[4];
          c_values<T, CM>(g, Cp, m, n, true, cv);
          T o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = static_cast<T>(final_value<T, CM>(g, acc, cv, i, j, q, e));
          *reinterpret_cast<u32x2*>(D + static_cast<int64_t>(m) * g.sd_m + n) =
              __builtin_bit_cast(u32x2, o);
        }
      }
    }
  }
}

// Output stores marked non-temporal (streamed past L2) per kernel: both
// kernels write their output once (mm 8192 x 14336 bf16: 767 -> 762 us,
// conv2d's implicit GEMM 155.5 -> 152.6 us with them).
constexpr bool kStreamOutMfma = true;
constexpr bool kStreamOutPanel = true;

// Up to 16 rows with a K-major A and B in 16-byte rows, 16 j columns per block
// (gemm_skinny.hip).
int gemm_skinny_dma(int dtype, const GemmArgs& g, int j, hipStream_t st);

// The 256 x 256 persistent kernel (gemm_large.hip): 16-bit products in the
// matrix-core layouts (see run_gemm) that gemm_large_serves.
bool gemm_large_serves(const GemmArgs& g);
// Whether its tiles suit the product's size (k_min: see there).
bool large_tiles_suit(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t k_min);
int gemm_large(int dtype, bool a_kmajor, bool b_kmajor, const GemmArgs& g, hipStream_t st);
// Its channels-last convolution: k in 64-channel blocks; problems that
// conv_large_serves (whatever the number of images in one launch).
int gemm_conv_large(int dtype, GemmArgs g, hipStream_t st);

}  // namespace ntops
