// Products of up to 16 rows with a large K-major B (decode projections with
// F.linear's weight): out = alpha A B^T' (+ beta C), bound by streaming B once.
//
// The register kernel (k_gemm_skinny in gemm.hip) reads a K-major B in 64-byte
// row pieces and waits for each batch of its loads before the next: 8 x 14336
// x 4096 bf16 28.8 us (4.1 TB/s) there, 22.7 here (5.2 TB/s; 24.8 with
// temporal loads of B, whose lines no other block reads).  Here each
// of a block's four waves owns K steps of its own and streams them through its
// own part of the LDS by direct DMA: rows of 128 bytes or more (whole lines),
// non-temporal, two to three steps (16 to 24 KiB) ahead, no barrier before
// the waves' fp32 partial sums are merged.  A block covers 16 J columns; a
// step is 8 KiB of B (16 J rows of 512 / J bytes) and the matching 16 rows of
// A, so fewer columns mean longer row pieces, not smaller loads.
#include <atomic>

#include "gemm_tile.h"

namespace ntops {
namespace {

constexpr int kSkWaves = 4;

// A and B fragments of one 64-byte column group: lane l holds row / column
// l & 15, its 16 bytes at byte 16 (l >> 4): 32 k of 16-bit data in one MFMA,
// 16 k of fp32 in four (element e of every lane feeds MFMA e).
template <typename T>
__device__ __forceinline__ f32x4 mul16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same<T, __bf16>::value) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  } else if constexpr (std::is_same<T, _Float16>::value) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  } else {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
    return c;
  }
}

// Slot of 16-byte chunk c of tile row r, CPR chunks per row: the 16 rows of a
// fragment read hit 16 different chunk positions of the LDS's 256 bytes.
template <int CPR>
__device__ __forceinline__ int sk_slot(int r, int c) {
  return CPR == 8 ? c ^ ((r >> 1) & 7) : c ^ (r & 15);
}

template <bool NT>
__device__ __forceinline__ void sk_dma(u32x4 rsrc, uint32_t dst, uint32_t off) {
  if constexpr (NT)
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen nt lds" : : "v"(off), "s"(rsrc), "{m0}"(dst) : "memory");
  else
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(off), "s"(rsrc), "{m0}"(dst) : "memory");
}

// One operand's tile: ROWS rows of CPR chunks per step.
template <int ROWS, int CPR, int ES, bool NT>
struct SkLoader {
  static constexpr int kInst = ROWS * CPR / 64;
  static constexpr int kRpi = 64 / CPR;
  u32x4 rsrc;
  uint32_t voff[kInst];
  __device__ __forceinline__ static int chunk_k(int lane, int i) {  // first k of the lane's chunk
    return sk_slot<CPR>(i * kRpi + lane / CPR, lane % CPR) * (16 / ES);
  }
  __device__ __forceinline__ void init(const void* base, int64_t ld, int64_t bytes, int lane) {
    const uint64_t addr = reinterpret_cast<uint64_t>(base);
    rsrc.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr));
    rsrc.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(addr >> 32) & 0xffffu);
    rsrc.z = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bytes));
    rsrc.w = 0x00020000u;
#pragma unroll
    for (int i = 0; i < kInst; ++i)
      voff[i] = static_cast<uint32_t>(((i * kRpi + lane / CPR) * ld + chunk_k(lane, i)) * ES);
  }
  __device__ __forceinline__ void issue(uint32_t dst, int k0, int K, int lane) const {
#pragma unroll
    for (int i = 0; i < kInst; ++i)
      sk_dma<NT>(rsrc, dst + i * 1024,
                 k0 + chunk_k(lane, i) < K ? voff[i] + static_cast<uint32_t>(k0) * ES : kOOB);
  }
};

template <typename T, int J>
__global__ __launch_bounds__(64 * kSkWaves, 1) void k_gemm_skinny_dma(GemmArgs g) {
  constexpr int NW = kSkWaves, ES = sizeof(T);
  constexpr int CPR = 32 / J;             // chunks of a row per step
  constexpr int KS = CPR * 16 / ES;       // k per step
  constexpr int kB = 8192, kA = 8192 / J;  // bytes per step
  constexpr int S = J == 1 ? 2 : 3;       // steps in the ring
  constexpr int kStep = kA + kB;
  using LA = SkLoader<16, CPR, ES, false>;
  using LB = SkLoader<16 * J, CPR, ES, true>;
  constexpr int kInst = LA::kInst + LB::kInst;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * (16 * J);
  const int bat = blockIdx.y;
  const int nv = min(16 * J, g.N - n0);
  const int r16 = lane & 15, q = lane >> 4;

  LA la;
  LB lb;
  la.init(static_cast<const T*>(g.A) + bat * g.sa_b, g.sa_m, (static_cast<int64_t>(g.M - 1) * g.sa_m + g.K) * ES, lane);
  lb.init(static_cast<const T*>(g.B) + bat * g.sb_b + static_cast<int64_t>(n0) * g.sb_n, g.sb_n,
          (static_cast<int64_t>(nv - 1) * g.sb_n + g.K) * ES, lane);
  const int steps = (g.K + KS - 1) / KS;
  const int n = steps > wave ? (steps - wave + NW - 1) / NW : 0;  // this wave's: wave, wave + NW, ...
  char* mine = smem + wave * (S * kStep);
  const uint32_t mine_addr = lds_addr(mine);
  // step j of this wave into ring slot j % S (past the end: empty loads, so
  // that the waits count the same)
  int slot_in = 0;
  auto issue = [&](int j) {
    const int k0 = j < n ? (wave + j * NW) * KS : 0x40000000;
    const uint32_t dst = mine_addr + slot_in * kStep;
    lb.issue(dst, k0, g.K, lane);
    la.issue(dst + kB, k0, g.K, lane);
    slot_in = slot_in + 1 == S ? 0 : slot_in + 1;
  };
  f32x4 acc[J];
#pragma unroll
  for (int j = 0; j < J; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S; ++s) issue(s);
  int slot = 0;
  for (int i = 0; i < n; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<(S - 1) * kInst>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const char* tb = mine + slot * kStep;
    const char* ta = tb + kB;
#pragma unroll
    for (int u = 0; u < CPR / 4; ++u) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(ta + r16 * (CPR * 16) + sk_slot<CPR>(r16, u * 4 + q) * 16);
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int r = j * 16 + r16;
        const u32x4 b = *reinterpret_cast<const u32x4*>(tb + r * (CPR * 16) + sk_slot<CPR>(r, u * 4 + q) * 16);
        acc[j] = mul16<T>(a, b, acc[j]);
      }
    }
    wait_lgkmcnt0();
    issue(i + S);
    slot = slot + 1 == S ? 0 : slot + 1;
  }
  wait_vmcnt<0>();  // no DMA may land in the LDS the merge reuses
  __syncthreads();
  // Lane l holds rows 4 (l >> 4) + r, column 16 j + (l & 15).
  float* red = reinterpret_cast<float*>(smem);  // [wave][j][r][lane]
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[((wave * J + j) * 4 + r) * 64 + lane] = acc[j][r];
  __syncthreads();
  T* D = static_cast<T*>(g.D) + bat * g.sd_b;
  const T* Cp = g.use_c ? static_cast<const T*>(g.C) + bat * g.sc_b : nullptr;
  for (int t = wave; t < J * 4; t += NW) {
    const int j = t >> 2, r = t & 3;
    const int m = q * 4 + r, col = n0 + 16 * j + r16;
    if (m < g.M && col < g.N) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += red[((w * J + j) * 4 + r) * 64 + lane];
      v *= g.alpha;
      if (Cp != nullptr) v += g.beta * static_cast<float>(Cp[m * g.sc_m + col * g.sc_n]);
      D[static_cast<int64_t>(m) * g.sd_m + static_cast<int64_t>(col) * g.sd_n] = static_cast<T>(v);
    }
  }
}

template <typename T, int J>
int launch_sk(const GemmArgs& g, hipStream_t st) {
  constexpr int kLds = kSkWaves * (J == 1 ? 2 : 3) * (8192 + 8192 / J);
  auto kern = k_gemm_skinny_dma<T, J>;
  static std::atomic<bool> attr_set{false};
  if (!attr_set.load(std::memory_order_relaxed)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) !=
        hipSuccess)
      return set_error(NTOPS_ERR_HIP, "gemm: cannot reserve %d bytes of LDS", kLds);
    attr_set.store(true, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL(kern, dim3((g.N + 16 * J - 1) / (16 * J), static_cast<unsigned>(g.batch)), dim3(64 * kSkWaves),
                     kLds, st, g);
  return check_launch("gemm");
}

}  // namespace

int gemm_skinny_dma(int dtype, const GemmArgs& g, int j, hipStream_t st) {
  return dispatch_float16_32(dtype, "gemm", [&](auto tag) {
    using T = decltype(tag);
    return j == 4 ? launch_sk<T, 4>(g, st) : j == 2 ? launch_sk<T, 2>(g, st) : launch_sk<T, 1>(g, st);
  });
}

}  // namespace ntops
