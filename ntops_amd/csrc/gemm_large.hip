// Large 16-bit GEMM (K > 256, sizes by large_tiles_suit): out = alpha A B
// (+ beta times a bias row), any of the four operand layouts, any edges, any
// output layout.
//
// Bound by the matrix cores under the part's power limit, so what counts is
// energy per flop as much as cycles:
//  * v_mfma_f32_16x16x32: the same flops with half the accumulator traffic of
//    32x32x16 (each accumulator is read and written once per 32 k, not 16).
//    The one change took 8192 x 14336 x 4096 with a K-major B from 660 to
//    617 us (8192^3 748 -> 685);
//  * 64-deep K tiles, so a K-major operand's DMA fetches whole 128-byte lines
//    (32-deep ones left the address unit 0.91 busy when both operands are
//    K-major).  Two K tiles of 256 x 256 fill 128 KiB of LDS; to keep loads
//    three phases (about 1.5 us) ahead of their use with only two, a K tile is
//    four half tiles (A0, A1, B0, B1) that are refilled one by one as soon as
//    their last fragment read is over;
//  * the two waves of a SIMD are half a phase apart (ping-pong): in a phase one
//    group of waves reads fragments and issues loads while the other runs 32
//    MFMAs, quadrants (A0, B0), (A1, B0) then (A1, B1), (A0, B1), so that 12 of
//    the 24 fragment reads of a K tile serve two quadrants;
//  * blocks are persistent and nothing is drained between output tiles: the
//    next tile's loads follow the last K tile's, and a finished quadrant is
//    rounded, staged and stored between the MFMAs of the following phases.
//    Memory operations retire in order, so the waits count the stores too.
//    8192 x 50176 x 768 (12 K tiles per output tile): 607 -> 535 us.
// Stores are non-temporal (535 against 625 us there: 32 CUs' outputs fill an
// XCD's L2).  Rows that do not start on 128-byte lines leave partial lines to
// merge: 8192 x 50257 x 768 1020 -> 690 us.
// Same-box pairs, before (32-deep K tiles, one block per tile) and now, bf16:
// 8192 x 14336 x 4096 766 -> 640 us (K-major B; the matrix library 622), 717
// -> 655 (N-major B; 720); 4096^3 108 -> 93; 6000 x 6000 x 4096 388 -> 245.
//
// The channels-last convolution (PixelLoader) runs on the same kernel: a K
// tile is a 64-channel block under one tap, so a pixel's piece is one whole
// 128-byte line (the 32-channel kernel fetched halves of them), and a tile's
// stores leave under the next one's MFMAs.  Whole conv2d calls, bf16 3 x 3:
// (32, 256, 56, 56) to 256 148.7 -> 122.1 us, (32, 128, 56, 56) to 128 75.2 ->
// 64.8, (32, 64, 112, 112) to 128 152.8 -> 136.2.  What is left there is the
// input's copy (19 us) and 416 tiles over 256 CUs: two rounds, 0.8 full.
#include <algorithm>
#include <atomic>

#include "gemm.h"
#include "gemm_tile.h"

namespace ntops {
namespace {

constexpr int kHalf = 128 * 64 * 2;      // bytes of a half tile: 128 rows / columns x 64 k
// LDS: half h of the K tile in buffer b at (2 b + h) * kHalf of A's area, and
// of B's: every fragment read is one per-lane base plus an immediate.
constexpr int kAreaB = 4 * kHalf;
constexpr int kStageOff = 8 * kHalf;             // per wave: 16 rows x 64 rounded outputs
constexpr int kBiasOff = kStageOff + 8 * 2048;   // per wave: the tile's 2 x 64 columns of a bias row
constexpr int kLargeLds = kBiasOff + 8 * 256;

// The lane id through an empty asm: what is computed from it is computed where
// it is used, not hoisted out of the tile loops to sit in registers.
__device__ __forceinline__ int here(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

// v_mfma_f32_16x16x32: lane l holds row / column l & 15 at k = 8 (l >> 4) ..
// + 7 of A / B; of the result column l & 15 and rows 4 (l >> 4) .. + 3.
template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same<T, __bf16>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

// This lane's fragment reads of one operand: TILES slices of 16 rows (or
// columns) of a half tile, 32 k per read.
template <bool KMAJ, int TILES>
struct FragReader {
  // LDS byte addresses at half 0 of buffer 0: per k-step, or per two slices
  // (an M/N-major swizzle leaves the chunk's low two bits alone)
  static constexpr int kBases = KMAJ ? 2 : TILES / 2;
  uint32_t base[kBases];

  // row0: the wave's first row of a half; TILES consecutive 16-row slices
  __device__ __forceinline__ void init(uint32_t area, int row0, int lane) {
    const int g = lane >> 4, i = lane & 15;
    if constexpr (KMAJ) {
      const int r = row0 + i;  // (the slices' rows differ by 16: one swizzle)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        base[ks] = area + static_cast<uint32_t>(r * 128 + kslot<64>(r, ks * 4 + g) * 16);
        asm volatile("" : "+v"(base[ks]));
      }
    } else {
#pragma unroll
      for (int t = 0; t < kBases; ++t) {
        const int n = row0 + t * 32 + (i & 3) * 4;
        const int k = g * 8 + (i >> 2);
        base[t] = area + static_cast<uint32_t>(k * 256 + mnslot(k, n >> 3) * 16 + ((n >> 2) & 1) * 8);
        asm volatile("" : "+v"(base[t]));
      }
    }
  }
  // slice t, k-step ks of the half tile `idx` = 2 buffer + half
  __device__ __forceinline__ u32x4 read(int idx, int t, int ks) const {
    typedef __attribute__((address_space(3))) const u32x4 lds_u32x4_t;
    if constexpr (KMAJ) {
      return *reinterpret_cast<lds_u32x4_t*>(base[ks] + static_cast<uint32_t>(idx * kHalf + t * 2048));
    } else {
      u32x2 v[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        v[h] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4_t*>(
                                             base[t >> 1] + static_cast<uint32_t>(idx * kHalf + (t & 1) * 32 + (ks * 32 + h * 4) * 256))));
      return u32x4{v[0].x, v[0].y, v[1].x, v[1].y};
    }
  }
};

// Loads of an operand's half tiles: 2 instructions of 1 KiB per wave.
template <bool KMAJ>
struct HalfLoader {
  uint32_t voff[2];
  uint32_t kbytes;   // byte distance of consecutive k
  uint32_t lds_off;  // of this wave's first instruction

  __device__ __forceinline__ static int lane_k(int wave, int lane, int i) {
    const int q = wave * 2 + i;
    if constexpr (KMAJ) {
      const int row = q * 8 + lane / 8;
      return kslot<64>(row, lane % 8) * 8;
    } else {
      return q * 4 + lane / 16;
    }
  }
  __device__ __forceinline__ void init(int64_t ld, int wave, int lane) {
    lds_off = static_cast<uint32_t>(wave * 2048);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int q = wave * 2 + i;
      if constexpr (KMAJ)
        voff[i] = static_cast<uint32_t>((q * 8 + lane / 8) * ld * 2 + lane_k(wave, lane, i) * 2);
      else
        voff[i] = static_cast<uint32_t>((q * 4 + lane / 16) * ld * 2 + mnslot(q * 4 + lane / 16, lane % 16) * 16);
    }
    kbytes = static_cast<uint32_t>(KMAJ ? 2 : ld * 2);
  }
  // TAIL: the K tile at k0 may reach past K; its chunks there read as zero.
  template <bool TAIL>
  __device__ __forceinline__ void issue(u32x4 rsrc, uint32_t lds, int k0, int K, int wave, int lane) const {
    // (opaque, so that no sum of a fixed tile's is kept in a register)
    uint32_t koff = static_cast<uint32_t>(k0) * kbytes;
    asm volatile("" : "+s"(koff));
    const int l = TAIL ? here(lane) : 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t off = voff[i] + koff;
      if constexpr (TAIL) off = k0 + lane_k(wave, l, i) < K ? off : kOOB;
      dma16(rsrc, lds + lds_off + i * 1024, off);
    }
  }
};

// The same for a channels-last convolution's pixels (see GemmArgs): a K tile
// is one 64-channel block under one tap, a row one output pixel.
struct PixelLoader {
  uint32_t lds_off;

  // this lane's chunk of its row for instruction i, in elements
  __device__ __forceinline__ static int lane_k(int wave, int lane, int i) {
    return HalfLoader<true>::lane_k(wave, lane, i);
  }
  __device__ __forceinline__ void init(int64_t, int wave, int) { lds_off = static_cast<uint32_t>(wave * 2048); }
  // Byte offset of this lane's chunk of pixel nh + row under the first tap of
  // the first block (pixels past the image read its last one's: columns that
  // are never stored).  n / cl_q by multiplication, exact on the sizes that
  // conv_large_serves takes.
  __device__ __forceinline__ static uint32_t pixel(const GemmArgs& g, int nh, int wave, int lane, int i) {
    const uint32_t n = static_cast<uint32_t>(min(nh + (wave * 2 + i) * 8 + lane / 8, g.N - 1));
    const uint32_t p = __umulhi(n, g.cl_mq);
    const uint32_t col = static_cast<uint32_t>(g.cl_sw) * g.cl_c;
    const uint32_t row = static_cast<uint32_t>(g.cl_sh) * g.cl_wp * g.cl_c;
    return (n * col + p * (row - g.cl_q * col) + lane_k(wave, lane, i)) * 2;
  }
  template <bool TAIL>
  __device__ __forceinline__ void issue(u32x4 rsrc, uint32_t lds, const uint32_t (&pix)[2], int t, const GemmArgs& g) const {
    const uint32_t ut = static_cast<uint32_t>(t);
    const uint32_t cb = (ut * g.cl_mrs) >> 16;  // channel block and tap of the K tile
    const uint32_t tap = ut - cb * g.cv_rs;
    const uint32_t r = (tap * g.cl_ms) >> 16;
    const uint32_t c = tap - r * g.cv_s;
    uint32_t koff = ((r * g.cl_dh * g.cl_wp + c * g.cl_dw) * g.cl_c + cb * 64) * 2;
    asm volatile("" : "+s"(koff));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t off = pix[i] + koff;
      if constexpr (TAIL) off = t * 64 < g.K ? off : kOOB;
      dma16(rsrc, lds + lds_off + i * 1024, off);
    }
  }
};

__device__ __forceinline__ u32x4 make_rsrc(const void* base, int64_t bytes) {
  const uint64_t addr = reinterpret_cast<uint64_t>(base);
  u32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr));
  r.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr >> 32) & 0xffffu);
  r.z = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bytes));
  r.w = 0x00020000u;
  return r;
}

// Resources of an output tile's operand halves (what lies past an edge reads
// as zero, or as some other row's or column's data: such rows and columns of
// the product are never stored); a convolution's pixel offsets.
template <bool CONV>
struct TileRsrc {
  u32x4 a[2], b[2];
  uint32_t pix[CONV ? 2 : 1][2];  // [column half][instruction]
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  wait_vmcnt<(N < 63 ? N : 63)>();
}

// CONV: B is the channels-last convolution operand, the bias a value per row.
template <typename T, bool AK, bool BKM, bool BIAS, bool CONV = false>
__global__ __launch_bounds__(512, 1) void k_gemm_large(GemmArgs g, int total) {
  static_assert(!CONV || (AK && BKM), "the convolution's operands are K-major");
  using Rsrc = TileRsrc<CONV>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;  // 32 rows of a half, 64 columns of a half
  const int grp = wave >> 2;
  const int tm_count = (g.M + 255) / 256, tn_count = (g.N + 255) / 256;
  const int np = (g.K + 127) / 128;  // pairs of K tiles

  // tile `i` of this block: (batch, row, column) or false past the end
  const int nx = (gridDim.x & 7) == 0 ? 8 : 1;
  const int per_x = (total + nx - 1) / nx;
  auto tile_at = [&](int i, int& bat, int& m0, int& n0) __attribute__((always_inline)) {
    const int x = static_cast<int>(blockIdx.x) % nx;
    const int pos = i * (static_cast<int>(gridDim.x) / nx) + static_cast<int>(blockIdx.x) / nx;
    const int id = x * per_x + pos;
    if (pos >= per_x || id >= total) return false;
    const int per_batch = tm_count * tn_count;
    bat = id / per_batch;
    const int t = id - bat * per_batch;
    constexpr int kGroupM = 4;
    const int gsz = kGroupM * tn_count;
    const int gi = t / gsz;
    const int gm = min(tm_count - gi * kGroupM, kGroupM);
    const int r = t - gi * gsz;
    n0 = (r / gm) * 256;
    m0 = (gi * kGroupM + r % gm) * 256;
    return true;
  };
  auto rsrc_of = [&](bool ok, int bat, int m0, int n0) __attribute__((always_inline)) {
    Rsrc r;
    const uint16_t* A = static_cast<const uint16_t*>(g.A) + bat * g.sa_b;
    const uint16_t* B = static_cast<const uint16_t*>(g.B) + bat * g.sb_b;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int mh = m0 + h * 128, nh = n0 + h * 128;
      const int mv = ok ? min(g.M - mh, 128) : 0, nv = ok ? min(g.N - nh, 128) : 0;
      r.a[h] = mv <= 0 ? make_rsrc(g.A, 0)
               : AK    ? make_rsrc(A + static_cast<int64_t>(mh) * g.sa_m, (static_cast<int64_t>(mv - 1) * g.sa_m + g.K) * 2)
                       : make_rsrc(A + mh, (static_cast<int64_t>(g.K - 1) * g.sa_k + mv) * 2);
      if constexpr (CONV) {  // the batch's whole padded image
        r.b[h] = make_rsrc(B, nv > 0 ? g.sb_b * 2 : 0);
#pragma unroll
        for (int i = 0; i < 2; ++i) r.pix[h][i] = PixelLoader::pixel(g, nh, wave, here(lane), i);
        continue;
      }
      r.b[h] = nv <= 0 ? make_rsrc(g.B, 0)
               : BKM   ? make_rsrc(B + static_cast<int64_t>(nh) * g.sb_n, (static_cast<int64_t>(nv - 1) * g.sb_n + g.K) * 2)
                       : make_rsrc(B + nh, (static_cast<int64_t>(g.K - 1) * g.sb_k + nv) * 2);
    }
    return r;
  };

  HalfLoader<AK> la;
  std::conditional_t<CONV, PixelLoader, HalfLoader<BKM>> lb;
  la.init(AK ? g.sa_m : g.sa_k, wave, lane);
  lb.init(BKM ? g.sb_n : g.sb_k, wave, lane);
  const uint32_t smem_addr = lds_addr(smem);

  int bat, m0, n0, nbat = 0, nm0 = 0, nn0 = 0;
  if (!tile_at(0, bat, m0, n0)) return;  // (the whole block)
  Rsrc cur = rsrc_of(true, bat, m0, n0), nxt;

  // loads of half tile `half` of operand A / B of K tile t (buffer t & 1)
  auto dma_a = [&](auto tail, const Rsrc& rs, int half, int t) __attribute__((always_inline)) {
    la.template issue<decltype(tail)::value>(
        rs.a[half], smem_addr + static_cast<uint32_t>(((t & 1) * 2 + half) * kHalf), t * 64, g.K, wave, lane);
  };
  auto dma_b = [&](auto tail, const Rsrc& rs, int half, int t) __attribute__((always_inline)) {
    const uint32_t lds = smem_addr + static_cast<uint32_t>(kAreaB + ((t & 1) * 2 + half) * kHalf);
    if constexpr (CONV)
      lb.template issue<decltype(tail)::value>(rs.b[half], lds, rs.pix[half], t, g);
    else
      lb.template issue<decltype(tail)::value>(rs.b[half], lds, t * 64, g.K, wave, lane);
  };

  // [quadrant][row tile][column tile]; quadrants 00, 10, 11, 01 (row half,
  // column half), 32 x 64 per wave
  f32x4 acc[4][2][4];
  u32x4 ax[4], ay[4], bx[4][2];  // A0, A1, one half of B
  FragReader<AK, 2> fa;
  FragReader<BKM, 4> fb;
  fa.init(smem_addr, wm * 32, lane);
  fb.init(smem_addr + kAreaB, wn * 64, lane);
  auto read_a = [&](u32x4 (&f)[4], int buf, int half) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = fa.read(buf * 2 + half, e & 1, e >> 1);  // [k-step][row tile]
  };
  auto read_b = [&](int buf, int half) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < 4; ++j) bx[j][ks] = fb.read(buf * 2 + half, j, ks);
  };

  // ---- epilogue: a finished quadrant (32 x 64 per wave) is rounded, 16 x 16
  // pieces between the MFMAs of the next K step, into the wave's 2 KiB of
  // staging (16 rows of 128 bytes, chunk c of row r at slot c ^ (r >> 1)) and
  // leaves as 128-byte row segments.  (A wave's LDS operations are in order:
  // the second row tile may be written once the first's reads are issued.)
  const uint32_t ep = smem_addr + static_cast<uint32_t>(kStageOff + wave * 2048);
  const uint32_t bias_lds = smem_addr + static_cast<uint32_t>(kBiasOff + wave * 256);
  int pm0 = 0, pn0 = 0, pbat = 0;  // the tile being stored
  bool pend = false;
  auto row_half = [&](int q) __attribute__((always_inline)) { return q == 1 || q == 2; };
  auto col_half = [&](int q) __attribute__((always_inline)) { return q >= 2; };
  // the bias columns of the tile at n (CONV: rows at m): lanes 0-31 the first half's, 32-63 the
  // second's, two per lane (past N: zero; an odd N's last pair is one dword)
  auto bias_dma = [&](int m, int n) __attribute__((always_inline)) {
    const int l = here(lane);
    const uint32_t off = CONV ? static_cast<uint32_t>((m + (l >> 5) * 128 + wm * 32 + (l & 15) * 2) * 2)
                              : static_cast<uint32_t>((n + (l >> 5) * 128 + wn * 64 + (l & 31) * 2) * 2);
    const u32x4 r = make_rsrc(g.C, (static_cast<int64_t>(CONV ? g.M : g.N) * 2 + 3) & ~3ll);
    asm volatile("buffer_load_dword %0, %1, 0 offen lds" : : "v"(off), "s"(r), "{m0}"(bias_lds) : "memory");
  };
  // LDS address of this lane's 4 columns in column tile 0; column tile ct
  // flips chunk bits 1 and 2: address ^ (ct << 5)
  auto ep_base = [&](int l) __attribute__((always_inline)) {
    const int r = l & 15, c = l >> 5, half = (l >> 4) & 1;
    return ep + static_cast<uint32_t>(r * 128 + ((c ^ (r >> 1)) << 4) + half * 8);
  };
  // the bias values of quadrant q for this lane: per column tile its 4
  // columns', CONV: per row tile its row's
  typedef __attribute__((address_space(3))) const u32x2 lds_cu32x2_t;
  typedef __attribute__((address_space(3))) const uint16_t lds_cu16_t;
  auto bias_of = [&](int q, int l, u32x2 (&bias)[4]) __attribute__((always_inline)) {
    if constexpr (CONV) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
        bias[rt].x = *reinterpret_cast<lds_cu16_t*>(bias_lds + static_cast<uint32_t>(row_half(q) * 128 + rt * 32 + (l & 15) * 2));
    } else {
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
        bias[ct] = *reinterpret_cast<lds_cu32x2_t*>(bias_lds + static_cast<uint32_t>(col_half(q) * 128 + ct * 32 + (l >> 4) * 8));
    }
  };
  // rounds row tile i / 4, column tile i % 4 of quadrant q into the staging
  auto convert = [&](int q, int i, uint32_t base, const u32x2 (&bias)[4]) __attribute__((always_inline)) {
    const int rt = i >> 2, ct = i & 3;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[q][rt][ct][e];
    if constexpr (BIAS) {
      const u32x2 raw = bias[CONV ? rt : ct];
      const T* t = reinterpret_cast<const T*>(&raw);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = g.alpha * v[e] + g.beta * static_cast<float>(t[CONV ? 0 : e]);
    }
    T o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = static_cast<T>(v[e]);
    typedef __attribute__((address_space(3))) u32x2 lds_u32x2_t;
    *reinterpret_cast<lds_u32x2_t*>(base ^ static_cast<uint32_t>(ct << 5)) = __builtin_bit_cast(u32x2, o);
  };
  // (alpha != 1 without a bias: in place, so the usual case carries no multiply)
  auto scale = [&](int q) __attribute__((always_inline)) {
    if constexpr (!BIAS) {
      if (g.alpha != 1.f) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[q][i >> 2][i & 3][e] *= g.alpha;
      }
    }
  };
  // 16 staged rows back, 8 lanes per row: rows l / 8 and l / 8 + 8
  auto load_rows = [&](u32x4 (&rows)[2], int l) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) const u32x4 lds_cu32x4_t;
    const int r = l >> 3, c = l & 7;
    const uint32_t at = ep + static_cast<uint32_t>(r * 128 + ((c ^ (r >> 1)) << 4));
    rows[0] = *reinterpret_cast<lds_cu32x4_t*>(at);
    rows[1] = *reinterpret_cast<lds_cu32x4_t*>((at ^ 64u) + 1024u);
  };
  // Row tile rt of quadrant q to memory: at least 2 store instructions
  // whatever the edges (a lane with nothing to store stores past the
  // resource), which the waits of the following phases count on.  Rows may
  // start at any 2-byte address.
  auto put_rows = [&](const u32x4 (&rows)[2], int q, int rt, int l) __attribute__((always_inline)) {
    const int m = pm0 + row_half(q) * 128 + wm * 32 + rt * 16;
    const int n = pn0 + col_half(q) * 128 + wn * 64;
    const T* D = static_cast<const T*>(g.D) + pbat * g.sd_b + static_cast<int64_t>(m) * g.sd_m +
                 static_cast<int64_t>(n) * g.sd_n;
    const __amdgpu_buffer_rsrc_t r = buffer_rsrc_uniform(D, 0x7fffffffu);
    const int c0 = (l & 7) * 8;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = (l >> 3) + 8 * u;
      const bool in = m + row < g.M;
      const uint32_t off = static_cast<uint32_t>(row) * static_cast<uint32_t>(g.sd_m) * 2;
      if (g.sd_n == 1) {
        const uint32_t at = off + c0 * 2;
        __builtin_amdgcn_raw_buffer_store_b128(rows[u], r, in && n + c0 + 8 <= g.N ? at : kOOB, 0, kBufNT);
        if ((g.N & 7) && pn0 + 256 > g.N) {  // the tile of the row's last, partial chunk
#pragma unroll
          for (int e = 0; e < 7; ++e)
            __builtin_amdgcn_raw_buffer_store_b16(
                static_cast<uint16_t>(rows[u][e >> 1] >> (16 * (e & 1))), r,
                in && n + c0 + 8 > g.N && n + c0 + e < g.N ? at + 2 * e : kOOB, 0, 0);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          __builtin_amdgcn_raw_buffer_store_b16(
              static_cast<uint16_t>(rows[u][e >> 1] >> (16 * (e & 1))), r,
              in && n + c0 + e < g.N ? off + static_cast<uint32_t>(c0 + e) * static_cast<uint32_t>(g.sd_n) * 2 : kOOB, 0, 0);
      }
    }
  };

  // the quadrant's 16 MFMAs; LEAVE: finished quadrant cq leaves between them --
  // its first row tile's rows are stored under its second's conversion, its
  // second's are left in `rows` (put_rows by the caller)
  u32x4 rows[2];
  auto mfma16x = [&](auto first, auto leave, int q, const u32x4 (&af)[4], int cq) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first)::value, LEAVE = decltype(leave)::value;
    int l = 0;
    uint32_t base = 0;
    u32x2 bias[4];
    if constexpr (LEAVE) {
      l = here(lane);
      base = ep_base(l);
      scale(cq);
      if constexpr (BIAS) bias_of(cq, l, bias);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          f32x4 c = acc[q][rt][ct];
          if (FIRST && ks == 0) c = f32x4{0.f, 0.f, 0.f, 0.f};
          acc[q][rt][ct] = mfma16<T>(bx[ct][ks], af[ks * 2 + rt], c);
          if constexpr (LEAVE) {
            const int i = ks * 8 + rt * 4 + ct;  // piece i / 2 after every second MFMA
            if (i & 1) {
              __builtin_amdgcn_sched_barrier(0);
              convert(cq, i >> 1, base, bias);
              if (i == 7) load_rows(rows, l);
              if (i == 11) put_rows(rows, cq, 0, l);
              if (i == 15) load_rows(rows, l);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
  };
  constexpr auto yes = std::true_type{};
  constexpr auto no = std::false_type{};
  // ends a memory phase: its fragments are in registers, and all but the
  // wave's N youngest memory operations are done
  auto end_mem = [&](auto n_tag) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
    __builtin_amdgcn_sched_barrier(0);
    if (N > 8 && pend)
      wait_vm<N>();
    else
      wait_vm<8>();
    wait_lgkmcnt0();
    block_barrier();
    __builtin_amdgcn_s_setprio(1);
  };
  auto end_mfma = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(0);
    block_barrier();
  };
#define NTOPS_W(n) std::integral_constant<int, (n)> {}

  // One K tile (buffer BUF): two phases.  KIND 0: the first K tile of an
  // output tile (quadrants 1 - 3 of the previous one leave), 3: the second,
  // 1: between, 2: the last (quadrant 0 leaves).  Loads issued: B1 of the
  // next K tile (rs1 / t1), then A0, B0, A1 of the one after it (rs2 / t2).
  // The waits allow for the 8 loads issued since the ones the next phase
  // reads, plus the stores among them while a tile leaves (two per put_rows:
  // 4, 8, 5 and 1 of them).
  auto ktile = [&](auto kind_tag, auto buf_tag, auto tail, const Rsrc& rs1, int t1, const Rsrc& rs2,
                   int t2) __attribute__((always_inline)) {
    constexpr int KIND = decltype(kind_tag)::value, BUF = decltype(buf_tag)::value;
    constexpr auto first = std::bool_constant<KIND == 0>{};
    // ---- phase A: quadrants 0 and 1
    read_a(ax, BUF, 0);
    read_b(BUF, 0);
    read_a(ay, BUF, 1);
    dma_b(tail, rs1, 1, t1);
    if constexpr (KIND == 0)
      if (pend) put_rows(rows, 1, 1, here(lane));
    end_mem(NTOPS_W(KIND == 0 ? 16 : KIND == 3 ? 18 : 8));
    if (KIND == 0 && pend) {
      mfma16x(first, yes, 0, ax, 2);
      put_rows(rows, 2, 1, here(lane));
      mfma16x(first, yes, 1, ay, 3);
    } else {
      mfma16x(first, no, 0, ax, 0);
      mfma16x(first, no, 1, ay, 0);
    }
    end_mfma();
    // ---- phase B: quadrants 2 and 3
    read_b(BUF, 1);
    dma_a(tail, rs2, 0, t2);
    dma_b(tail, rs2, 0, t2);
    dma_a(tail, rs2, 1, t2);
    if constexpr (KIND == 0)
      if (pend) put_rows(rows, 3, 1, here(lane));
    end_mem(NTOPS_W(KIND == 0 ? 24 : KIND == 3 ? 10 : 8));
    if constexpr (KIND == 2) {
      pm0 = m0;
      pn0 = n0;
      pbat = bat;
      mfma16x(no, yes, 2, ay, 0);
      put_rows(rows, 0, 1, here(lane));
      mfma16x(no, yes, 3, ax, 1);
    } else {
      mfma16x(first, no, 2, ay, 0);
      mfma16x(first, no, 3, ax, 0);
    }
    end_mfma();
  };

  // prologue: the first K tile and A0, B0, A1 of the second in flight
  dma_a(no, cur, 0, 0);
  dma_b(no, cur, 0, 0);
  dma_a(no, cur, 1, 0);
  dma_b(no, cur, 1, 0);
  dma_a(no, cur, 0, 1);
  dma_b(no, cur, 0, 1);
  dma_a(no, cur, 1, 1);
  wait_vmcnt<8>();
  block_barrier();
  if (grp == 1) block_barrier();

  constexpr auto b0 = NTOPS_W(0);
  constexpr auto b1 = NTOPS_W(1);
  for (int it = 0;; ++it) {
    ktile(NTOPS_W(0), b0, no, cur, 1, cur, 2);
    ktile(NTOPS_W(3), b1, no, cur, 2, cur, 3);
    int t = 2;
    for (; t < 2 * np - 4; t += 2) {
      ktile(NTOPS_W(1), b0, no, cur, t + 1, cur, t + 2);
      ktile(NTOPS_W(1), b1, no, cur, t + 2, cur, t + 3);
    }
    // the loads of the last two K tiles, which may reach past K
    ktile(NTOPS_W(1), b0, yes, cur, t + 1, cur, t + 2);
    ktile(NTOPS_W(1), b1, yes, cur, t + 2, cur, t + 3);
    if constexpr (BIAS) bias_dma(m0, n0);
    const bool more = tile_at(it + 1, nbat, nm0, nn0);
    nxt = rsrc_of(more, nbat, nm0, nn0);
    ktile(NTOPS_W(1), b0, yes, cur, t + 3, nxt, 0);
    ktile(NTOPS_W(2), b1, no, nxt, 0, nxt, 1);
    pend = true;
    if (!more) break;
    cur = nxt;
    m0 = nm0;
    n0 = nn0;
    bat = nbat;
  }
  if (grp == 0) block_barrier();
  put_rows(rows, 1, 1, lane);
#pragma unroll
  for (int q = 2; q < 4; ++q) {
    scale(q);
    u32x2 bias[4];
    if constexpr (BIAS) bias_of(q, lane, bias);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) convert(q, rt * 4 + ct, ep_base(lane), bias);
      load_rows(rows, lane);
      put_rows(rows, q, rt, lane);
    }
  }
  wait_vmcnt<0>();  // no DMA may land after the workgroup ends
}

template <typename T, bool AK, bool BKM, bool BIAS, bool CONV = false>
int launch_large(const GemmArgs& g, hipStream_t st) {
  auto kern = k_gemm_large<T, AK, BKM, BIAS, CONV>;
  static std::atomic<bool> attr_set{false};  // (threads may get here together)
  if (!attr_set.load(std::memory_order_relaxed)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            kLargeLds) != hipSuccess)
      return set_error(NTOPS_ERR_HIP, "gemm: cannot reserve %d bytes of LDS", kLargeLds);
    attr_set.store(true, std::memory_order_relaxed);
  }
  const int64_t total = static_cast<int64_t>((g.M + 255) / 256) * ((g.N + 255) / 256) * g.batch;
  if (total > 0x3fffffffLL) return set_error(NTOPS_ERR_UNSUPPORTED, "gemm: too many tiles");
  const int64_t grid = std::min<int64_t>(total, cu_count_cached());
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(512), kLargeLds, st, g, static_cast<int>(total));
  return check_launch("gemm");
}

template <typename T, bool AK, bool BKM>
int launch_large_c(const GemmArgs& g, hipStream_t st) {
  return g.use_c ? launch_large<T, AK, BKM, true>(g, st) : launch_large<T, AK, BKM, false>(g, st);
}

template <typename T>
int run_large(bool ak, bool bk, const GemmArgs& g, hipStream_t st) {
  if (ak) return bk ? launch_large_c<T, true, true>(g, st) : launch_large_c<T, true, false>(g, st);
  return bk ? launch_large_c<T, false, true>(g, st) : launch_large_c<T, false, false>(g, st);
}

template <typename T>
int run_conv_large(const GemmArgs& g, hipStream_t st) {
  return g.use_c ? launch_large<T, true, true, true, true>(g, st) : launch_large<T, true, true, false, true>(g, st);
}

}  // namespace

bool gemm_large_serves(const GemmArgs& g) {
  const int64_t lim = int64_t(1) << 31;
  // no C, or one bias row for all rows (a C with a value per row or element
  // would be loaded, and waited for, piece by piece: it takes the kernel
  // whose epilogue has all its loads in flight)
  const bool bias_row = g.use_c && g.c_mode == kCVec4 && g.sc_m == 0 && (g.batch == 1 || g.sc_b == 0);
  return g.K > 256 && (!g.use_c || bias_row) && g.sd_m >= 0 && g.sd_n >= 0 &&
         (16 * g.sd_m + 64 * g.sd_n) * 2 < lim && static_cast<int64_t>(g.N) * 2 + 1024 < lim;
}

int gemm_large(int dtype, bool a_kmajor, bool b_kmajor, const GemmArgs& g, hipStream_t st) {
  note_kernel("gemm_large %s %s", a_kmajor ? "A:K" : "A:M", b_kmajor ? "B:K" : "B:N");
  return dtype == NTOPS_BF16 ? run_large<__bf16>(a_kmajor, b_kmajor, g, st)
                             : run_large<_Float16>(a_kmajor, b_kmajor, g, st);
}

// 240 tiles (a round of the GPU's 256 CUs).  Fewer leave CUs idle, but from
// the count where 128 x 128 tiles (two to a CU) need a second round on they
// are still faster: bf16 K-major B, 2560 x 4096 x 4096 (160 tiles) 106.9 -> 70.2
// us, 3584 x 4096 x 4096 (224) 145.7 -> 84.1, 2816 x 3072 x 768 (132) 25.0 ->
// 20.1, 2816 x 3072 x 512 19.4 -> 16.5, N-major within 4 %.  That holds where
// the last row or column of large tiles is half empty or more, too (small ->
// large, K-major B / N-major B): 2050 x 4096 x 512 23.1 -> 16.8 / 23.3 -> 17.5, x
// 1024 37.4 -> 23.3 / 37.5 -> 24.2, x 2040 78.7 -> 43.3 / 68.2 -> 40.6; the
// least, half empty tiles at K = 512, 1152 x 8192 19.2 -> 17.1 / 18.3 -> 18.0
// (M-major A: 20.0 -> 18.2 / 18.9 -> 19.0); convolutions 3 x 3 of 64 channels (40,
// 28 x 28) to 256 37.8 -> 32.3, 1 x 1 of 512 52.8 -> 46.4.  Below K = 512 an
// N-major B starts to lose (x 448: 2560 x 4096 16.8 -> 17.4, 1152 x 8192 17.1 ->
// 18.1), a K-major one still gains (17.6 -> 16.5, 18.0 -> 17.1).  Where the
// small tiles fill seven eighths of their one round, a K of k_min or more
// amortises the large kernel's fill: 2048 x 4096 x 4096 (128) 80.0 -> 65.8, but
// 3584 x 2304 x 768 (126) 19.1 -> 20.0; not with half empty large tiles (a product
// of 128 rows).  Below that the small ones are as fast or faster (768 x 6400 x
// 1600, 75: 34.0 / 32.2; 1024 x 4096 x 4096, 64: 38.7 / 64.5).
bool large_tiles_suit(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t k_min) {
  const int64_t cus = cu_count_cached() > 0 ? cu_count_cached() : 256;
  const int64_t large = ((M + 255) / 256) * ((N + 255) / 256) * batch;
  const int64_t small = ((M + 127) / 128) * ((N + 127) / 128) * batch;
  const bool whole = small == 4 * large;
  return large >= 240 || (small > 2 * cus && K >= 512) || (whole && 4 * small > 7 * cus && K >= k_min);
}

// Where the plain kernel's tiles suit (K > 256), on images whose
// channels are whole 64-deep K tiles, with no bias or a contiguous one.  The
// index divisions by multiplication need
//  * n / Q: ceil(2^32 / Q) is less than Q too large per 2^32, so the quotient
//    is exact where n Q < 2^32 (Q = 1: the factor would not fit);
//  * t / (R S) of K tile t (up to 4 past the last) and tap / S likewise, over
//    2^16.
bool conv_large_serves(int64_t images, int64_t M, int64_t pixels, int64_t C, int64_t R, int64_t S, int64_t Q,
                       int64_t out_ld, const void* bias, int64_t bias_stride) {
  const int64_t rs = R * S;
  const bool bias_ok = bias == nullptr || (bias_stride == 1 && M % 2 == 0 && (reinterpret_cast<uintptr_t>(bias) & 3u) == 0);
  return C % 64 == 0 && C * rs > 256 && bias_ok && Q >= 2 && pixels * Q < (int64_t(1) << 32) &&
         (C / 64 * rs + 4) * rs < 65536 && rs * S < 65536 && out_ld >= 0 && (16 * out_ld + 64) * 2 < (int64_t(1) << 31) &&
         large_tiles_suit(M, pixels, C * rs, images, 1024);
}

int gemm_conv_large(int dtype, GemmArgs g, hipStream_t st) {
  g.cv_rs = g.cv_r * g.cv_s;
  g.cl_mq = static_cast<uint32_t>(((uint64_t(1) << 32) + g.cl_q - 1) / g.cl_q);
  g.cl_mrs = (65536u + g.cv_rs - 1) / g.cv_rs;
  g.cl_ms = (65536u + g.cv_s - 1) / g.cv_s;
  note_kernel("gemm_large A:K B:K conv_cl");
  return dtype == NTOPS_BF16 ? run_conv_large<__bf16>(g, st) : run_conv_large<_Float16>(g, st);
}

}  // namespace ntops
