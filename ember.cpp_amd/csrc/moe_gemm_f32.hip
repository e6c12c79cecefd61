// Grouped expert GEMM over F32 stacks on the FP32 matrix cores (v_mfma_f32_32x32x2_f32): F32 operands, F32
// accumulation, for batches of more than a few tokens per expert. The one product the reference has
// (utils.cpp:735-747) with its F32 weights; the decode GEMV (moe_experts.hip) keeps the smallest batches.
//
// Bound: the FP32 matrix rate (v_mfma_f32_32x32x2_f32 back to back: 155 TFLOP/s; the 16x16x4 form reaches
// 114-137) from a few dozen rows per expert on, the weight stream below. Tiles of 64 tokens x 64 weight rows
// (gate/up: 32 gate + 32 up, SwiGLU in the epilogue) x 32 columns, 256 threads: four waves, 2 (M) x 2 (N), one
// 32 x 32 subtile each. FP32 MFMAs take 64 cycles for 4 kFLOP, so neither LDS reads nor the L2 limit so small a
// tile, and it is chosen for balance and registers: ~100 rows per expert give every CU several blocks, three
// at a time, whose waits and epilogues overlap, and the sums below stay in registers (eight waves of a 128-row
// tile, at 128 registers each, spilled, and a reload waits for all the DMA in flight). Both operands go
// straight to LDS (global_load_lds) through a ring of three stages, 16-byte granules XOR-swizzled by row pair
// so that the 16 rows a read pass touches fall on distinct bank groups.
//
// Rounding: an FP32 MFMA is a chain of FMAs, and one chain over all of K drifts with the square root of K,
// which the GEMV's lane-parallel sums do not. So a chain runs over 8 columns only (as the GEMV's do), the eight
// chains of 64 columns are added up, and those sums are accumulated with Kahan's compensation: no more
// roundings deep than the GEMV at any K (layer error against 64 bits 1.6e-7 to 1.7e-7, the GEMV's 1.6e-7 to
// 2.0e-7). The additions are not hidden (FP32 MFMAs and FP32 VALU instructions do not overlap on gfx950: 4 of
// each take the sum of their times; d 1024, d_ff 2816, E 8, 400 tokens, gate/up: MFMAs 47 % of the cycles, vector
// instructions 28 %): 11 of them per 64 columns and output, and a twelfth that keeps infinite sums infinite.
#include <cstdlib>
#include <type_traits>

#include "moe_fmt.hpp"

namespace ember_moe {
using namespace ember_math;

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_f32_t;

constexpr int kF32BM = 64, kF32BK = 32, kF32Rows = 64;  // tokens, columns, weight rows of a tile
constexpr int kF32Threads = 256, kF32Stages = 3;
constexpr int kF32A = kF32BM * kF32BK * 4, kF32B = kF32Rows * kF32BK * 4;  // bytes per stage
constexpr size_t kF32Lds = (size_t)kF32Stages * (kF32A + kF32B);
constexpr int kF32InstA = kF32A / 1024 / 4, kF32InstB = kF32B / 1024 / 4;  // 1 KiB loads per wave and stage
constexpr int kF32Group = 4;  // m-tiles that take one n-tile's weights one after another

__device__ const float4 kF32Zero = {0.0f, 0.0f, 0.0f, 0.0f};  // what columns past K load

template <int N>
__device__ inline void wait_vmcnt_f32() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

template <bool GATED>
__global__ void __launch_bounds__(kF32Threads, 3) gemm_f32_kernel(GemmF32Args g, int NT) {
  constexpr int BN = GATED ? 32 : 64;
  extern __shared__ __align__(16) uint8_t fsm[];

  // block -> (m-tile, n-tile, K part): the W work items in 8 equal runs, one per XCD (block b runs on XCD
  // b % 8); within a run kF32Group m-tiles (mostly one expert's) walk an n-tile together, so its weights
  // come from memory once
  const int M = g.tiles ? *g.n_tiles : (g.T + kF32BM - 1) / kF32BM;
  const int KS = g.ksplit, MG = (M + kF32Group - 1) / kF32Group;
  const int W = MG * kF32Group * NT * KS, C = (W + 7) / 8;
  const int w = (blockIdx.x % 8) * C + blockIdx.x / 8;
  if ((int)(blockIdx.x / 8) >= C || w >= W) return;
  const int mt = w / (kF32Group * NT * KS) * kF32Group + w % kF32Group;
  const int rest = w / kF32Group % (NT * KS);
  const int nt = rest / KS, ks = rest % KS;
  if (mt >= M) return;
  int e = 0, p0, rows;
  if (g.tiles) {
    const int4 t = g.tiles[mt];
    e = t.x;
    p0 = t.y;
    rows = t.z;
  } else {
    const int h = tile_height(g.T, kF32BM);
    p0 = mt * h;
    rows = min(h, g.T - p0);
  }
  if (rows <= 0) return;
  const int n0 = nt * BN, K = g.K, N = g.N;
  const int nk_all = (K + kF32BK - 1) / kF32BK;
  const int kt0 = ks * nk_all / KS, nk = (ks + 1) * nk_all / KS - kt0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, lh = lane >> 5;

  // DMA sources: load j of a wave fills granules 64 (n w + j) + lane; granule gi is row gi / 8, slot gi % 8,
  // holding columns 4 kg .. + 3 of the tile, kg = slot ^ ((row / 2) % 8). Rows past the tile or the matrix
  // repeat the last one (their results are not stored).
  const float* srcA[kF32InstA];
  const float* baseB[kF32InstB];  // (uniform: one load's 8 rows are all gate or all up)
  uint32_t offB[kF32InstB];
  int colA[kF32InstA], colB[kF32InstB];
#pragma unroll
  for (int i = 0; i < kF32InstA; ++i) {
    const int gi = 64 * (kF32InstA * wave + i) + lane, r = gi >> 3;
    colA[i] = 4 * ((gi & 7) ^ ((r >> 1) & 7));
    const int p = p0 + min(r, rows - 1);
    srcA[i] = g.A + (size_t)(g.perm ? g.perm[p] / g.k : p) * K + colA[i];
  }
#pragma unroll
  for (int i = 0; i < kF32InstB; ++i) {
    const int gi = 64 * (kF32InstB * wave + i) + lane, r = gi >> 3;
    colB[i] = 4 * ((gi & 7) ^ ((r >> 1) & 7));
    const bool up = GATED && kF32InstB * wave + i >= 4;
    baseB[i] = (up ? g.W1 : g.W0) + ((int64_t)e * N + n0) * K;
    offB[i] = (uint32_t)min(GATED ? (r & 31) : r, N - 1 - n0) * (uint32_t)K + (uint32_t)colB[i];
  }
  // tile kt of this part; columns past its end (the last tile of K, and the tile that rounds the part up to
  // pairs) come from a block of zeros. NOA: a wave whose activation rows (16 w .. 16 w + 15) lie past the
  // tile's tokens loads none.
  const int kend = min(K, (kt0 + nk) * kF32BK);
  auto dma = [&](const float* p, uint8_t* dst) { __builtin_amdgcn_global_load_lds(p, (lds_void_f32_t*)dst, 16, 0, 0); };
  // WHOLE: every tile of the part is whole and their number even, so nothing is checked (a branch here would
  // also make the compiler keep the chains of one tile for the next: it sinks their additions past it).
  auto issue = [&](int kt, int stage, auto NOAc, auto WHOLEc) {
    constexpr bool whole = decltype(WHOLEc)::value;
    const int k0 = whole ? (kt0 + min(kt, nk - 1)) * kF32BK : (kt0 + kt) * kF32BK;
    uint8_t* st = fsm + stage * (kF32A + kF32B);
    const float* z = reinterpret_cast<const float*>(&kF32Zero);
    if constexpr (!decltype(NOAc)::value) {
#pragma unroll
      for (int i = 0; i < kF32InstA; ++i)
        dma(whole || k0 + colA[i] < kend ? srcA[i] + k0 : z, st + 1024 * (kF32InstA * wave + i));
    }
#pragma unroll
    for (int i = 0; i < kF32InstB; ++i)
      dma(whole || k0 + colB[i] < kend ? baseB[i] + k0 + offB[i] : z, st + kF32A + 1024 * (kF32InstB * wave + i));
  };

  const floatx16 zero = {};
  floatx16 sum = zero, comp = zero, mid = zero, c0 = zero, c1 = zero;

  // this lane's weight row in the tile; gated: the subtile's columns 0 .. 15 are gate rows, 16 .. 31 the up rows
  const int brow = GATED ? 32 * (li >> 4) + 16 * wn + (li & 15) : 32 * wn + li;
  // columns 8 t .. 8 t + 7 of the tile: lane half lh holds 4 lh .. + 3 of them, one per MFMA, in A and B alike
  struct Frags {
    floatx4 a, b;
  };
  const int swz = (li >> 1) & 7;  // (the same for both rows this lane reads: they differ by a multiple of 16)
  auto load = [&](int stage, int t, Frags& f) {
    const uint8_t* st = fsm + stage * (kF32A + kF32B) + 16 * ((2 * t + lh) ^ swz);
    f.a = *reinterpret_cast<const floatx4*>(st + 128 * (32 * wm + li));
    f.b = *reinterpret_cast<const floatx4*>(st + kF32A + 128 * brow);
  };
  auto chain = [&](const Frags& f) {  // 8 columns
    floatx16 c = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[0], f.b[0], zero, 0, 0, 0);
#pragma unroll
    for (int u = 1; u < 4; ++u) c = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[u], f.b[u], c, 0, 0, 0);
    return c;
  };
  auto add = [&](bool first) {  // mid (+)= the two chains of 16 columns
#pragma unroll
    for (int r = 0; r < 16; ++r) mid[r] = first ? c0[r] + c1[r] : mid[r] + (c0[r] + c1[r]);
  };
  // sum += mid + the pair's last two chains, compensated. The compensation of an infinite sum would be Inf - Inf: the
  // clamp (v_med3, whose result for a NaN is its lower bound) keeps it finite and too small to carry a finite v past
  // the largest float, so that an infinite sum stays one, as in the GEMV; it cuts real ones from sums of 2^125 on only
  // (d 1024, d_ff 2816, E 8, 400 tokens 218.7 -> 221.3 us; running the sums of a block with a NaN again without the
  // compensation, 220.4, would keep a second copy of the loop).
  constexpr float kMostComp = 0x1p100f;
  auto fold = [&] {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float v = (mid[r] + (c0[r] + c1[r])) - comp[r], t = sum[r] + v;
      comp[r] = __builtin_amdgcn_fmed3f((t - sum[r]) - v, -kMostComp, kMostComp);
      sum[r] = t;
    }
  };
  // The loop is rotated: the barrier (tile kt + 1 has landed, tile kt is read) sits before the last chain of
  // tile kt, which covers the first reads of tile kt + 1.
  // IDLE: a wave without tokens only loads and keeps the barriers.
  auto k_loop = [&](auto IDLEc, auto NOAc, auto WHOLEc) {
    constexpr bool work = !decltype(IDLEc)::value;
    constexpr int kPer = (decltype(NOAc)::value ? 0 : kF32InstA) + kF32InstB;
    auto barrier = [] {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    auto next = [](int s) { return s == kF32Stages - 1 ? 0 : s + 1; };
    issue(0, 0, NOAc, WHOLEc);
    issue(1, 1, NOAc, WHOLEc);
    wait_vmcnt_f32<kPer>();
    barrier();
    Frags f0, f1;
    int cur = 0, fill = 2;
    if constexpr (work) load(0, 0, f0);
    // (the scheduling barriers keep the compiler from running chains ahead of the additions: their results
    // would not fit the registers of three waves per SIMD)
    auto step = [] { __builtin_amdgcn_sched_barrier(0); };
    auto tile = [&](int kt, bool first) {
      if constexpr (work) {
        load(cur, 1, f1);
        issue(kt + 2, fill, NOAc, WHOLEc);
        step();
        if (first) fold();
        else add(false);
        c0 = chain(f0);
        step();
        load(cur, 2, f0);
        c1 = chain(f1);
        step();
        load(cur, 3, f1);
        add(first);
        c0 = chain(f0);
        step();
      } else {
        issue(kt + 2, fill, NOAc, WHOLEc);
      }
      wait_vmcnt_f32<kPer>();
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads of tile kt are complete
      barrier();
      cur = next(cur);
      fill = next(fill);
      if constexpr (work) {
        load(cur, 0, f0);
        c1 = chain(f1);
        step();
      }
    };
    for (int kt = 0; kt < nk; kt += 2) {  // (the fold in front finishes the pair before, at first zeros)
      tile(kt, true);
      tile(kt + 1, false);
    }
    if constexpr (work) fold();
  };
  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  const bool noa = 16 * wave >= rows;
  const bool idle = 32 * wm >= rows;  // (wave >= 2, so its activation rows lie past the tokens too)
  if (K % kF32BK == 0 && nk % 2 == 0) {
    if (idle) k_loop(Yes{}, Yes{}, Yes{});
    else if (noa) k_loop(No{}, Yes{}, Yes{});
    else k_loop(No{}, No{}, Yes{});
  } else {
    if (idle) k_loop(Yes{}, Yes{}, No{});
    else if (noa) k_loop(No{}, Yes{}, No{});
    else k_loop(No{}, No{}, No{});
  }
  wait_vmcnt_f32<0>();  // no DMA may still target LDS when the block exits

  // lane: column li of the subtile, rows 8 i + 4 lh + r (i, r < 4); gated: up's column sits 16 lanes on
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int m = 32 * wm + 8 * (q >> 2) + 4 * lh + (q & 3);
    if constexpr (GATED) {
      const float u = __shfl_xor(sum[q], 16, 64);
      const int n = n0 + 16 * wn + li;
      if (li < 16 && n < N && m < rows) g.out[(int64_t)(p0 + m) * N + n] = swiglu(sum[q], u);
    } else {
      const int n = n0 + 32 * wn + li;
      if (n < N && m < rows) g.out[ks * g.part_stride + (int64_t)(p0 + m) * N + n] = sum[q];
    }
  }
}

int gemm_f32_ksplit(int mtiles, int N, int K) {
  // parts until every CU has three blocks, each part at least 8 tiles of 32 columns
  const int nt = (N + kF32Rows - 1) / kF32Rows, nk = (K + kF32BK - 1) / kF32BK;
  int ks = 1;
  while (2 * ks <= kMaxKSplit && (int64_t)mtiles * nt * ks < 3 * std::max(1, device_cus()) && nk >= 16 * ks) ks *= 2;
  return ks;
}

int launch_gemm_f32(const GemmF32Args& g, bool gated, int max_mtiles, hipStream_t st) {
  const int BN = gated ? 32 : 64, NT = (g.N + BN - 1) / BN;
  if (max_mtiles <= 0 || NT == 0) return EMBER_OK;
  static const bool ok =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_kernel<true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)kF32Lds) == hipSuccess &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_kernel<false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)kF32Lds) == hipSuccess;
  if (!ok) return EMBER_ERR_LAUNCH;
  const int64_t items = (int64_t)((max_mtiles + kF32Group - 1) / kF32Group) * kF32Group * NT * g.ksplit;
  const unsigned blocks = (unsigned)((items + 7) / 8 * 8);
  if (gated)
    gemm_f32_kernel<true><<<blocks, kF32Threads, kF32Lds, st>>>(g, NT);
  else
    gemm_f32_kernel<false><<<blocks, kF32Threads, kF32Lds, st>>>(g, NT);
  return hipGetLastError() == hipSuccess ? EMBER_OK : EMBER_ERR_LAUNCH;
}

}  // namespace ember_moe
