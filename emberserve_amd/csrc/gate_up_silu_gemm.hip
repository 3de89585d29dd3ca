// Prefill-size gate_up projection with silu_and_mul as its epilogue, for gfx950:
//   out[t, j] = round(round(silu(g)) * u),  g = round(x[t] . W[j]),  u = round(x[t] . W[I + j])
// for t < T, j < I, with W [2I, H] the nn.Linear(H, 2I) weight (gate rows, then up rows).
//
// Reference: Qwen2MLP.forward, emberserve/model/qwen2.py:60-61 (gate_up_proj, then
// ops.silu_and_mul), where the [T, 2I] projection is written and read back. Here it never
// leaves the chip: each workgroup computes a BM-token x (BNG gate + BNG up) column tile with
// bf16/fp16 MFMA (v_mfma_f32_16x16x32) and writes only the [BM, BNG] activation tile. Tiles:
// 256 x 64, 256 x 96 (the last one ragged when 96 does not divide I), 256 x 128, 128 x 128.
//
// Structure:
//   * 8 waves in BM / 64 token groups x 8 / (BM / 64) column groups: each owns 64 tokens of
//     the tile and WC = BNG BM / 512 columns of both the gate and the up half, so it holds
//     (2 WC / 16) x 4 accumulator tiles of 16 x 16;
//   * the tile's operands stream through an LDS ring of "double stages" of 64 k (three for
//     the 256 x 64 and 128 x 128 tiles; for 256 x 96 and 256 x 128, where three would not
//     fit, separate rings of three weight and two x buffers, 160 KiB: 94 instead of 102 us for Qwen3-8B
//     at 256 tokens, the same at 8192): rows of 128
//     bytes (one 64-k line per row), so each direct-to-LDS load (global_load_lds_dwordx4)
//     moves 8 rows x 128 B; 16-byte chunks XOR-swizzled by row & 7 so the fragment reads
//     (one row per lane) spread over the banks. At 256 tokens each workgroup streams its
//     weight rows from HBM once, and the third buffer (two double stages in flight) took the
//     Qwen3-8B call from 91.7 to 70.0 us;
//   * ping-pong: the two waves of each SIMD belong to different groups (grp), and group 1
//     starts one barrier late, so between two barriers one group reads fragments and issues
//     loads while the other runs its MFMAs;
//   * XCD-aware tile order: consecutive workgroups land on different XCDs (round robin), so
//     the order is remapped to give each XCD a contiguous range of tiles, grouped GROUP_M
//     token tiles at a time over a band of column tiles (their weight rows stay in that
//     XCD's L2).
// The k order of every accumulator is the decode kernels' (32-k steps in order, one chain),
// so a token's result is bit-identical to ember_gate_up_silu_packed over whole-slab runs.
// The epilogue is the decode kernels' exact one (expf and a division); v_exp_f32 / v_rcp_f32
// measured 3% faster at 8192 tokens and would give up that identity.
//
// Measured on MI355X (bf16, µs; this kernel at the better column tile / hipBLASLt +
// silu_and_mul): Qwen3-8B 256 tokens 70.0 / 72.6, 8192 tokens 1286 / 1235; Qwen2.5-7B 256
// tokens 110 / 88.5, 8192 tokens 1791 / 1834. Over an unpacked weight the library therefore
// keeps the unfused pair by default at these sizes and runs this kernel when the fused form is
// asked for. Packed weights have a kernel of their own (k_gate_up_silu_gemm_frag, below).
#include <algorithm>
#include <type_traits>

#include "ember_common.h"

#ifndef EMBER_GEMM_GROUP_M
#define EMBER_GEMM_GROUP_M 8
#endif
// Double-stage buffers of the 64-column tile (the 128-column tile's two fill 128 KiB).
#ifndef EMBER_GEMM_SPLIT_RING
#define EMBER_GEMM_SPLIT_RING 1
#endif
#ifndef EMBER_GEMM_NBUF64
#define EMBER_GEMM_NBUF64 3
#endif

namespace ember {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct GemmMfma;
template <>
struct GemmMfma<_Float16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct GemmMfma<__bf16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

constexpr int kGemmRowB = 128;  // LDS row: 64 k of one operand row

__device__ __forceinline__ void gemm_load_lds16(const void* gptr, void* lds_base) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_global_load_lds(gptr, (__attribute__((address_space(3))) void*)(
                                             reinterpret_cast<uintptr_t>(lds_base)), 16, 0, 0);
#else
  (void)gptr;
  (void)lds_base;
#endif
}

// s_waitcnt vmcnt(N) / lgkmcnt(0) alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void gemm_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void gemm_wait_vm0() { gemm_wait_vm<0>(); }
__device__ __forceinline__ void gemm_wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }

// A workgroup barrier with no fence (the waits above are explicit); the asm clobbers keep
// the compiler from moving LDS accesses across it.
__device__ __forceinline__ void gemm_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

struct GemmArgs {
  const void* x;
  int64_t xs;
  const void* w;
  int64_t ws;
  void* out;
  int64_t os;
  int T, H, I;
  // routed experts (MOE kernels only): token tiles are BM-assignment blocks of the
  // block-aligned layout; block b's rows are assignments sorted_ids[b BM + r] (padding:
  // >= num_valid) of expert block_expert[b], x row = assignment / top_k, output row = the
  // assignment; wes = elements between experts' [2I, H] weights
  const int32_t* sorted_ids;
  const int32_t* block_expert;
  int num_valid, top_k, E, ntok;
  int64_t wes;
  uint32_t* err;  // MOE: EMBER_ERR_ROW_INDEX for a valid assignment whose token is >= ntok
  // packed dense weights (the frag kernel): w is the decode kernels' packed array for a grid of
  // pk_G workgroups over pk_total units (pk_total = (I / 64) (H / 64))
  int64_t pk_total, pk_G;
};

template <typename T, int BNG, int BM, bool MOE, bool PK = false>
__global__ void __launch_bounds__(512, 1)
k_gate_up_silu_gemm(GemmArgs a) {
  static_assert(!PK || (MOE && BNG % 64 == 0), "packed experts: tiles of whole 64-row slabs");
  using M = GemmMfma<T>;
  using V8 = typename M::v8;
  static_assert((BM == 256 && (BNG == 64 || BNG == 96 || BNG == 128)) || (BM == 128 && BNG == 128), "tile");
  constexpr int TG = BM / 64;                  // token groups of 64
  constexpr int WC = BNG * TG / 8;             // gate (and up) columns per wave
  constexpr int NT = 2 * WC / 16;              // row tiles per wave: NT / 2 gate, NT / 2 up
  constexpr int WREG = 2 * BNG * kGemmRowB;    // weight region of a double stage
  constexpr int XREG = BM * kGemmRowB;         // x region
  constexpr int DST = WREG + XREG;             // one double stage (64 k)
  constexpr int LOADS = (2 * BNG + BM) / 8 / 8;  // 1 KiB load instructions per wave per double stage
  // Double-stage buffers: NBUF - 1 double stages of loads in flight while one is consumed.
  constexpr int NBUF = 3 * DST <= 160 * 1024 ? EMBER_GEMM_NBUF64 : 2;
  // SPLIT: when three double stages do not fit, the operands get rings of their own: three
  // weight buffers (HBM latency) and two x buffers (mostly L2 hits), 160 KiB in all. Each
  // wave then loads WL weight blocks and LOADS - WL x blocks per double stage.
  constexpr bool SPLIT = EMBER_GEMM_SPLIT_RING != 0 && NBUF == 2 && 3 * WREG + 2 * XREG <= 160 * 1024;
  constexpr int WL = SPLIT ? 2 * BNG / 8 / 8 : 0;
  constexpr int LDS_BYTES = SPLIT ? 3 * WREG + 2 * XREG : NBUF * DST;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = w >> 2;    // ping-pong group: waves w and w + 4 share a SIMD
  const int q = w % TG;      // token group
  const int cg = w / TG;     // column group
  const int n = lane & 15, g = lane >> 4;

  // XCD-aware tile order, then GROUP_M token tiles per band of column tiles
  int mtiles = (a.T + BM - 1) / BM;
  const int ntiles = (a.I + BNG - 1) / BNG;  // the last one ragged when BNG does not divide I
  int pid = blockIdx.x;
  int nb = gridDim.x;
  if (MOE) {
    // The grid covers every block the layout may use, but only the blocks before the first
    // one past the last expert hold work (block_expert is ascending, num_experts after the
    // used blocks). Counted here (one coalesced read of the small table, the same for every
    // workgroup) so that the XCD ranges below split the real tiles evenly instead of
    // leaving the unused blocks' share of the chip idle.
    int used = 0;
    for (int i0 = 0; i0 < mtiles; i0 += kWave) {
      const int i = i0 + lane;
      const bool u = i < mtiles && a.block_expert[i] < a.E;
      used += __builtin_popcountll(__ballot(u));
    }
    mtiles = used;
    nb = used * ntiles;
  }
  {
    const int per = (nb + 7) / 8;
    const int xcd = pid % 8, idx = pid / 8;
    const int full = nb % 8 == 0 ? 8 : nb % 8;
    if (MOE && idx >= (xcd < full ? per : per - 1)) return;  // past this XCD's share of the real tiles
    pid = xcd < full ? xcd * per + idx : full * per + (xcd - full) * (per - 1) + idx;
  }
  constexpr int GM = EMBER_GEMM_GROUP_M;
  const int group = pid / (GM * ntiles);
  const int first_m = group * GM;
  const int gsize = min(mtiles - first_m, GM);
  const int mt = first_m + (pid % (GM * ntiles)) % gsize;
  const int nt = (pid % (GM * ntiles)) / gsize;
  const int m0 = mt * BM, n0 = nt * BNG;

  const T* X = static_cast<const T*>(a.x);
  const T* W = static_cast<const T*>(a.w);
  if (MOE) {
    const int e = a.block_expert[mt];  // uniform
    if (e < 0 || e >= a.E) return;     // past the layout's used blocks
    W += static_cast<int64_t>(e) * a.wes;
  }
  // This wave's load instructions of a double stage: instruction ins moves rows
  // 8 (ins % 32) + lane / 8 of region ins / 32-ish (weight rows first, then x rows); lane l
  // loads 16-byte chunk (l % 8) ^ (row % 8) of its row into slot l of the 1 KiB block.
  const T* src[LOADS];
  int dst[LOADS];
  auto x_src = [&](int xr, int c) {
    int64_t xrow;
    if (MOE) {  // padding assignments read token 0 and store nothing
      const int id = a.sorted_ids[m0 + xr];
      xrow = id >= 0 && id < a.num_valid ? id / a.top_k : 0;
      if (xrow >= a.ntok) {  // a corrupt layout: flag it, read token 0 (the row is stored)
        atomicOr(a.err, EMBER_ERR_ROW_INDEX);
        xrow = 0;
      }
    } else {
      xrow = min(m0 + xr, a.T - 1);  // padded tokens: the last real one
    }
    return X + xrow * a.xs + 8 * c;
  };
  auto w_src = [&](int row, int c) {
    // columns past I (a ragged last tile) read the last real row and store nothing
    const int wr = row < BNG ? min(n0 + row, a.I - 1) : a.I + min(n0 + row - BNG, a.I - 1);
    return W + static_cast<int64_t>(wr) * a.ws + 8 * c;
  };
  // Packed weights: the tile's weight region is its S slabs' 16 KiB units side by side, in
  // the units' own fragment order (1 KiB block ins of slab ins / 16 is bytes
  // [1024 (ins % 16), +1024) of the slab's unit), so every load is 1 KiB of contiguous
  // memory and the fragment reads need no swizzle.
  constexpr int S = PK ? BNG / 64 : 1;
  bool isw[LOADS];  // a weight load (uniform)
  int wsl[LOADS];   // PK: the slab of a weight load
  auto pk_src = [&](int ins) { return W + (ins % 16) * 512 + 8 * lane; };
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    if (SPLIT) {  // block offsets within the operand's own buffer
      const int ins = i < WL ? WL * w + i : (LOADS - WL) * w + (i - WL);
      const int row = 8 * ins + (lane >> 3);
      const int c = (lane & 7) ^ (row & 7);
      isw[i] = i < WL;
      wsl[i] = ins / 16;
      src[i] = i < WL ? (PK ? pk_src(ins) : w_src(row, c)) : x_src(row, c);
      dst[i] = ins * 1024;
    } else {
      const int ins = LOADS * w + i;  // 0 .. 2 BNG / 8 + BM / 8 - 1
      const int row = 8 * ins + (lane >> 3);
      const int c = (lane & 7) ^ (row & 7);
      isw[i] = row < 2 * BNG;  // whole blocks: uniform
      wsl[i] = ins / 16;
      src[i] = isw[i] ? (PK ? pk_src(ins) : w_src(row, c)) : x_src(row - 2 * BNG, c);
      dst[i] = ins * 1024;  // the weight region is rows 0 .. 2 BNG - 1, the x region follows
    }
  }
  const int nd = a.H / 64;  // double stages
  // Routed experts' packed weights are per expert k-major (unit j * slabs + slab of the
  // expert's array), so a stage's S units are adjacent: element offsets of double stage d's.
  int64_t wofs[S];
  auto next_units = [&](int d) {
    constexpr int64_t kUnitElems = 16384 / static_cast<int64_t>(sizeof(T));
#pragma unroll
    for (int ss = 0; ss < S; ++ss)
      wofs[ss] = (static_cast<int64_t>(min(d, nd - 1)) * (a.I / 64) + n0 / 64 + ss) * kUnitElems;
  };
  auto wk = [&](int i, int kk) -> int64_t { return PK ? wofs[wsl[i]] : kk; };
  auto wbuf = [&](int d) { return lds + (SPLIT ? (d % 3) * WREG : (d % NBUF) * DST); };
  auto xbuf = [&](int d) { return lds + (SPLIT ? 3 * WREG + (d % 2) * XREG : (d % NBUF) * DST + WREG); };
  auto issue = [&](int d) {
    const int kk = min(d, nd - 1) * 64;
    if (PK) next_units(d);
    unsigned char* st = lds + (d % NBUF) * DST;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) gemm_load_lds16(src[i] + (isw[i] ? wk(i, kk) : kk), st + dst[i]);
  };
  auto issue_w = [&](int d) {
    const int kk = min(d, nd - 1) * 64;
    if (PK) next_units(d);
#pragma unroll
    for (int i = 0; i < WL; ++i) gemm_load_lds16(src[i] + wk(i, kk), wbuf(d) + dst[i]);
  };
  auto issue_x = [&](int d) {
    const int kk = min(d, nd - 1) * 64;
#pragma unroll
    for (int i = WL; i < LOADS; ++i) gemm_load_lds16(src[i] + kk, xbuf(d) + dst[i]);
  };
  int woff[NT], xoff[4];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (PK) {  // slab c / 64, fragment (row tile (c % 64) / 16, part) of the unit's first k32 half
      const int c = WC * cg + 16 * (t % (NT / 2));
      woff[t] = (c / 64) * 16384 + (((c % 64) / 16) * 2 + (t < NT / 2 ? 0 : 1)) * 1024 + 16 * lane;
    } else {
      woff[t] = ((t < NT / 2 ? 0 : BNG) + WC * cg + 16 * (t % (NT / 2)) + n) * kGemmRowB;
    }
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) xoff[u] = (64 * q + 16 * u + n) * kGemmRowB;
  const int sw = n & 7;  // row % 8 of every fragment row

  f32x4 acc[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  V8 fw[NT], fx[4];

  // vmcnt after which the next double stage has landed: split rings issue x(j + 1), then
  // w(j + 2) at each even step, so all but the last WL loads
  constexpr int kNextLanded = SPLIT ? WL : (NBUF - 2) * LOADS;
  if (SPLIT) {
    issue_w(0);
    issue_x(0);
    issue_w(1);
  } else {
#pragma unroll
    for (int d = 0; d < NBUF - 1; ++d) issue(d);
  }
  gemm_wait_vm<kNextLanded>();
  gemm_barrier();
  // M(s): at an even 32-k stage issue the next loads into free buffers; read this stage's
  // fragments; at an odd stage wait for the next double stage's loads.
  auto mphase = [&](int s, bool even) {
    const int j = s >> 1;
    if (even) {
      if (SPLIT) {
        issue_x(j + 1);
        issue_w(j + 2);
      } else {
        issue(j + NBUF - 1);
      }
    }
    const unsigned char* sw_ = wbuf(j);
    const unsigned char* sx_ = xbuf(j);
    const int co = ((4 * (s & 1) + g) ^ sw) << 4;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      fw[t] = *reinterpret_cast<const V8*>(sw_ + woff[t] + (PK ? (s & 1) * 8192 : co));
#pragma unroll
    for (int u = 0; u < 4; ++u) fx[u] = *reinterpret_cast<const V8*>(sx_ + xoff[u] + co);
    if (!even) gemm_wait_vm<kNextLanded>();  // the next double stage has landed
    gemm_wait_lgkm0();
  };
  // Routed experts: an expert's run is padded to whole blocks at its end, so a wave whose
  // 64 rows start with a padding assignment holds padding only; it still loads its share
  // of the tiles and keeps the barriers, but skips the MFMAs (nothing of it is stored).
  bool live = true;
  if (MOE) {
    const int id0 = a.sorted_ids[m0 + 64 * q];
    live = __builtin_amdgcn_readfirstlane(id0 >= 0 && id0 < a.num_valid ? 1 : 0) != 0;
  }
  auto cphase = [&]() {
    if (MOE && !live) return;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[t][u] = M::run(fw[t], fx[u], acc[t][u]);
  };
  const int nk = 2 * nd;
  if (grp == 1) gemm_barrier();
  for (int s = 0; s < nk; s += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      mphase(s + h, h == 0);
      gemm_barrier();
      cphase();
      gemm_barrier();
    }
  }
  if (grp == 0) gemm_barrier();
  gemm_wait_vm0();

  // Epilogue: lane (n, g) holds rows 4g + r of each 16-row tile for token 16 u + n.
  T* out = static_cast<T*>(a.out);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int tok = m0 + 64 * q + 16 * u + n;
    bool real = tok < a.T;
    if (MOE) {  // the assignment's own output row
      tok = a.sorted_ids[tok];
      real = tok >= 0 && tok < a.num_valid;
    }
    if (real) {
#pragma unroll
      for (int t = 0; t < NT / 2; ++t) {
        const int col = n0 + WC * cg + 16 * t + 4 * g;
        if (col >= a.I) continue;  // a ragged last tile (I a multiple of 16)
        Pack<T, 4> o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float gf = round_to<T>(acc[t][u][r]);
          const float uf = round_to<T>(acc[t + NT / 2][u][r]);
          const float act = round_to<T>(gf / (1.0f + expf(-gf)));
          o.v[r] = half_product<T>(act, uf);
        }
        store_pack<T, 4>(out + static_cast<int64_t>(tok) * a.os + col, o);
      }
    }
  }
}

// ---------------------------------------------------------------- packed weight, dense
//
// k_gate_up_silu_gemm_frag: the GEMM over the decode kernels' packed weight (dense, or an
// expert's: MOE, token tiles of 64 or 128 assignments). Every 1 KiB
// block of the packed layout is one MFMA operand fragment, so the weights go from memory
// straight to registers, one contiguous KiB per load, and only x passes through LDS. With
// both operands in LDS (k_gate_up_silu_gemm) a 256 x (128 + 128) tile reads 192 KB and writes
// 64 KB of LDS per 64 k, the whole of its 128 B/clk beside 2048 cycles of MFMA; here it reads
// 128 and writes 32.
//   * 2 CG waves in two token groups x CG column groups; a wave has BM / 2 tokens x (CW gate +
//     CW up) columns. Waves 2c and 2c + 1 take the two token groups of one column group: they
//     sit on different SIMDs and read the same fragments at about the same time (the second
//     from L1).
//   * weight fragments: a register ring of four 32-k steps, loaded three steps ahead;
//   * x: an LDS ring of four 64-k stages, loaded two stages ahead by buffer loads to LDS (rows
//     of 128 bytes, 16-byte chunks XOR-swizzled by row & 7). The buffer form matters: after a
//     global_load_lds the compiler treats every wait as one for a flat access and drains both
//     counters (vmcnt(0) lgkmcnt(0)), after a buffer load it counts;
//   * x fragments: a register ring of four (six in 192-token, two in 64-token tiles), each
//     refilled behind the MFMAs that used it last;
//   * one barrier per stage, in its middle, where the next step's operands are already in
//     registers: no read waits for it.
// The k order of every accumulator and the epilogue are k_gate_up_silu_gemm's, so the results
// are its bits.
//
// What bounds it: the vector memory path (96 KB per 64 k of the 256 x 128 tile) beside the
// MFMAs. Qwen3-8B, T = 8192, one box: 1353 us; without the weight loads 1171, without the x
// loads 1244, without either 1069, MFMAs and barriers alone 1011. Deeper rings (8 and 16 weight
// steps, 5 to 8 x stages) changed nothing, x staged through registers lost 4-10%.
// Measured against both operands in LDS (us, bf16, the best tile of each | hipBLASLt +
// silu_and_mul): Qwen3-8B 64 tokens 68 -> 41 | 45, 128: 69 -> 46 | 50, 200: 70 -> 60 | 63, 512:
// 115 -> 90 | 92, 8192: 1450 -> 1320 | 1205; Qwen2.5-7B 64: 78 -> 52 | 62, 256: 100 -> 76 | 80,
// 600: 217 -> 174 | 171; Qwen2.5-0.5B 130: 21 -> 12.3 | 12.6, 2000: 62 -> 45 | 70.
// Routed experts (H 2048, I 1408, 64 experts, top-6; without the alignment): 128-row blocks
// at 512 tokens 147 -> 144, 2048: 258 -> 251, 8192: 767 -> 715; 64-row ones at 128 tokens 129,
// 256: 133 (128-row ones 143 before). 256-row blocks stay with k_gate_up_silu_gemm: their
// weights, shared by few blocks, would cross the vector memory path twice (4099 tokens 367,
// here 388).
__device__ __forceinline__ auto gemm_rsrc(const void* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, -1, kBufferWord3);
#else
  return p;
#endif
}
// 16 bytes per lane from base + voff (per lane) + soff (uniform) to lds_base + 16 lane.
template <typename R>
__device__ __forceinline__ void gemm_buffer_lds16(R r, int voff, int soff, void* lds_base) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(
                                                  reinterpret_cast<uintptr_t>(lds_base)), 16, voff, soff, 0, 0);
#else
  (void)r;
  (void)voff;
  (void)soff;
  (void)lds_base;
#endif
}

// Walks the packed units of one 64-row slab in k order: unit t of workgroup b's run while the
// slab's units last. start(b) = b total / G = b q + off with q = total / G, r = total % G,
// off = b r / G: stepping b adds r to the remainder b r % G, so the walk needs no division.
struct SlabWalk {
  int t, b, off, rem, len, left, q, r, G;
  __device__ void init(int slab, int nk, int64_t total, int64_t G_) {
    const int64_t u = static_cast<int64_t>(slab) * nk;
    const int64_t b_ = gu_owner(u, total, G_);
    const int64_t q_ = total / G_;
    const int64_t start = gu_start(b_, total, G_);
    G = __builtin_amdgcn_readfirstlane(static_cast<int>(G_));
    q = __builtin_amdgcn_readfirstlane(static_cast<int>(q_));
    r = __builtin_amdgcn_readfirstlane(static_cast<int>(total % G_));
    b = __builtin_amdgcn_readfirstlane(static_cast<int>(b_));
    t = __builtin_amdgcn_readfirstlane(static_cast<int>(u - start));
    off = __builtin_amdgcn_readfirstlane(static_cast<int>(start - b_ * q_));
    rem = __builtin_amdgcn_readfirstlane(static_cast<int>(b_ * (total % G_) % G_));
    len = q + (rem + r >= G ? 1 : 0);
    left = nk - 1;
  }
  __device__ int pos() const { return t < q ? t * G + b : q * G + off; }
  // Past the slab's last unit it stays there. No branches: they would cut the k loop's body
  // into blocks (and cost registers).
  __device__ void advance() {
    const int step = left > 0 ? 1 : 0;
    left -= step;
    t += step;
    const int wrap = t == len ? 1 : 0;
    t = wrap ? 0 : t;
    b += wrap;
    rem += wrap ? r : 0;
    const int carry = rem >= G ? 1 : 0;
    rem -= carry ? G : 0;
    off += carry;
    len = q + (rem + r >= G ? 1 : 0);
  }
};

template <int V>
using IntC = std::integral_constant<int, V>;

template <typename T, int BM, int CG, int CW, bool MOE>
__global__ void __launch_bounds__(128 * CG, (2 * CG + 3) / 4)
k_gate_up_silu_gemm_frag(GemmArgs a) {
  using M = GemmMfma<T>;
  using V8 = typename M::v8;
  constexpr int BNG = CG * CW;           // gate (and up) columns of the tile
  constexpr int NW = 2 * CG;             // waves
  constexpr int TW = BM / 2;             // tokens per wave
  constexpr int NX = TW / 16;            // x fragments per 32 k
  constexpr int NC = CW / 16;            // 16-column tiles per wave
  constexpr int NF = 2 * NC;             // weight fragments per 32 k
  static_assert(BM % 32 == 0 && (CW == 16 || CW == 32) && 64 % CW == 0, "a wave's columns lie in one slab");
  constexpr int XREG = BM * kGemmRowB;   // one x stage (64 k)
  constexpr int NBUF = 4;                // x ring: two stages of loads in flight
  constexpr int XI = BM / 8;             // x load instructions (8 rows) per stage
  constexpr int XL = (XI + NW - 1) / NW; // ... per wave (the last ones may repeat a row group)
  constexpr int WR = 4;                  // weight fragment ring, in 32-k steps
  constexpr int FX = NX % 4 == 0 ? 4 : NX;  // x fragment ring
  static_assert(NX % FX == 0, "x fragment ring");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NBUF * XREG];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = w & 1;
  const int cg = w >> 1;
  const int n = lane & 15, g = lane >> 4;

  // XCD-aware tile order, then GROUP_M token tiles per band of column tiles
  int mtiles = (a.T + BM - 1) / BM;
  const int ntiles = (a.I + BNG - 1) / BNG;
  int pid = blockIdx.x;
  int nb = gridDim.x;
  if (MOE) {  // only the used blocks share out the chip (see k_gate_up_silu_gemm)
    int used = 0;
    for (int i0 = 0; i0 < mtiles; i0 += kWave) {
      const int i = i0 + lane;
      const bool u = i < mtiles && a.block_expert[i] < a.E;
      used += __builtin_popcountll(__ballot(u));
    }
    mtiles = used;
    nb = used * ntiles;
  }
  {
    const int per = (nb + 7) / 8;
    const int xcd = pid % 8, idx = pid / 8;
    const int full = nb % 8 == 0 ? 8 : nb % 8;
    if (MOE && idx >= (xcd < full ? per : per - 1)) return;
    pid = xcd < full ? xcd * per + idx : full * per + (xcd - full) * (per - 1) + idx;
  }
  constexpr int GM = EMBER_GEMM_GROUP_M;
  const int group = pid / (GM * ntiles);
  const int first_m = group * GM;
  const int gsize = min(mtiles - first_m, GM);
  const int mt = first_m + (pid % (GM * ntiles)) % gsize;
  const int nt = (pid % (GM * ntiles)) / gsize;
  const int m0 = mt * BM, n0 = nt * BNG;

  // x: byte offsets of this lane's 16 bytes from the tile's first row (padded tokens: the last
  // real row); instruction ins moves rows 8 ins .. 8 ins + 7
  const T* X = static_cast<const T*>(a.x) + (MOE ? 0 : static_cast<int64_t>(m0) * a.xs);
  int64_t expert = 0;
  if (MOE) {
    expert = a.block_expert[mt];  // uniform
    if (expert < 0 || expert >= a.E) return;
  }
  const auto xrsrc = gemm_rsrc(X);
  const int nd = a.H / 64;
  int src[XL], dst[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int ins = min(XL * w + i, XI - 1);
    const int xr = 8 * ins + (lane >> 3);
    const int c = (lane & 7) ^ (xr & 7);
    int64_t xrow = min(xr, a.T - 1 - m0);
    if (MOE) {  // padding assignments read token 0 and store nothing
      const int id = a.sorted_ids[m0 + xr];
      xrow = id >= 0 && id < a.num_valid ? id / a.top_k : 0;
      if (xrow >= a.ntok) {  // a corrupt layout: flag it, read token 0 (the row is stored)
        atomicOr(a.err, EMBER_ERR_ROW_INDEX);
        xrow = 0;
      }
    }
    src[i] = static_cast<int>((xrow * a.xs + 8 * c) * static_cast<int64_t>(sizeof(T)));
    dst[i] = ins * 1024;
  }
  auto issue_x = [&](int d) __attribute__((always_inline)) {
    const int kk = min(d, nd - 1) * 64 * static_cast<int>(sizeof(T));
#pragma unroll
    for (int i = 0; i < XL; ++i) gemm_buffer_lds16(xrsrc, src[i], kk, lds + (d % NBUF) * XREG + dst[i]);
  };
  // weights: the wave's first column, the last real ones past I (nothing of those is stored)
  const int c0 = n0 + CW * cg;
  const int cw = min(c0, a.I - CW);
  const unsigned char* W = static_cast<const unsigned char*>(a.w) + ((cw % 64) / 16) * 2048 +
                           expert * a.wes * static_cast<int64_t>(sizeof(T));
  const uint32_t lane16 = 16u * lane;
  // The weights' unit of each stage: the dense packing's place is walked, an expert's units are
  // k-major (unit j slabs + slab).
  SlabWalk walk;
  if (!MOE) walk.init(cw / 64, nd, a.pk_total, a.pk_G);
  const int64_t kstep = MOE ? static_cast<int64_t>(a.I / 64) * 16384 : 0;
  int64_t unit = MOE ? static_cast<int64_t>(cw / 64) * 16384 - kstep : 0;  // byte offset of the current unit
  int left = nd;
  auto next_unit = [&]() __attribute__((always_inline)) {
    if (MOE) {  // past the last stage it stays there
      unit += left > 0 ? kstep : 0;
      --left;
    } else {
      unit = static_cast<int64_t>(walk.pos()) * 16384;
      walk.advance();
    }
  };
  V8 fw[WR][NF];
  auto load_w = [&](V8 (&f)[NF], int half) __attribute__((always_inline)) {
    const unsigned char* p = W + unit + half * 8192;
#pragma unroll
    for (int t = 0; t < NF; ++t) f[t] = *reinterpret_cast<const V8*>(p + t * 1024 + lane16);
  };
  const int sw = n & 7;
  const int xrow0 = (TW * q + n) * kGemmRowB;
  const int xo[2] = {xrow0 + ((g ^ sw) << 4), xrow0 + (((4 + g) ^ sw) << 4)};
  V8 fx[FX];
  auto read_x = [&](int d, int half, int u) __attribute__((always_inline)) {
    fx[u % FX] = *reinterpret_cast<const V8*>(lds + (d % NBUF) * XREG + xo[half] + u * 16 * kGemmRowB);
  };
  f32x4 acc[NF][NX];
#pragma unroll
  for (int t = 0; t < NF; ++t)
#pragma unroll
    for (int u = 0; u < NX; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int i = 0; i < WR - 1; ++i) {  // weight steps 0 .. WR - 2
    if (i % 2 == 0) next_unit();
    load_w(fw[i], i % 2);
  }
#pragma unroll
  for (int d = 0; d < NBUF - 1; ++d) issue_x(d);
  gemm_wait_vm0();
  gemm_barrier();
#pragma unroll
  for (int u = 0; u < FX; ++u) read_x(0, 0, u);

  // Step 2j + H of stage j: load weight step 2j + H + WR - 1, then the MFMAs, each x fragment
  // refilled FX groups ahead (from the next half or the next stage at the end).
  auto step = [&](int j, auto ring, auto half) __attribute__((always_inline)) {
    constexpr int R = decltype(ring)::value, H = decltype(half)::value;
    constexpr int A = H + WR - 1;
    if (A % 2 == 0) next_unit();
    load_w(fw[(R + WR - 1) % WR], A % 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
#pragma unroll
      for (int t = 0; t < NF; ++t) acc[t][u] = M::run(fw[R][t], fx[u % FX], acc[t][u]);
      if (u + FX < NX) read_x(j, H, u + FX);
      else read_x(j + H, 1 - H, u + FX - NX);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // The barrier makes x(j + 1) visible (read from step 2j + 1 on) and frees the buffer of
  // x(j - 1) (last used by the MFMAs of step 2j - 1) for x(j + NBUF - 1). x(j + 1) was loaded
  // before the loop or at the barrier of stage j - NBUF + 2: kYounger loads are younger.
  constexpr int kYounger = 2 * (NBUF - 2) * NF + (NBUF - 3) * XL;
  static_assert(kYounger < 64, "vmcnt");
  auto stage = [&](int j, auto ring) __attribute__((always_inline)) {
    constexpr int R = decltype(ring)::value;
    step(j, IntC<R>{}, IntC<0>{});
    gemm_wait_vm<kYounger>();
    gemm_barrier();
    issue_x(j + NBUF - 1);
    step(j, IntC<(R + 1) % WR>{}, IntC<1>{});
  };
  int j = 0;
  for (; j + 2 <= nd; j += 2) {
    stage(j, IntC<0>{});
    stage(j + 1, IntC<2>{});
  }
  if (j < nd) stage(j, IntC<0>{});
  gemm_wait_vm0();

  // Epilogue: lane (n, g) holds rows 4g + r of each 16-row tile for token 16 u + n.
  if (c0 >= a.I) return;
  T* out = static_cast<T*>(a.out);
#pragma unroll
  for (int u = 0; u < NX; ++u) {
    int tok = m0 + TW * q + 16 * u + n;
    bool real = tok < a.T;
    if (MOE) {  // the assignment's own output row
      tok = a.sorted_ids[tok];
      real = tok >= 0 && tok < a.num_valid;
    }
    if (real) {
#pragma unroll
      for (int t = 0; t < NC; ++t) {
        Pack<T, 4> o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float gf = round_to<T>(acc[2 * t][u][r]);
          const float uf = round_to<T>(acc[2 * t + 1][u][r]);
          const float act = round_to<T>(gf / (1.0f + expf(-gf)));
          o.v[r] = half_product<T>(act, uf);
        }
        store_pack<T, 4>(out + static_cast<int64_t>(tok) * a.os + c0 + 16 * t + 4 * g, o);
      }
    }
  }
}

template <typename T, int BM, int CG, int CW, bool MOE = false>
int launch_frag(const GemmArgs& a, hipStream_t st) {
  const int64_t grid = cdiv(a.T, BM) * cdiv(a.I, CG * CW);
  if (grid > 0x7fffffffLL) return EMBER_EINVAL;
  k_gate_up_silu_gemm_frag<T, BM, CG, CW, MOE><<<dim3(static_cast<uint32_t>(grid)), dim3(128 * CG), 0, st>>>(a);
  return launch_status();
}

// A tile's workgroup takes about as long as the rows it needs, BM x rows and 2 x columns weight
// rows per k: the tile with the fewest rows in all rounds, the smaller on a tie. Measured (bf16,
// us, one round at H = 4096; rows: 224 41-46, 256 45-50, 288 45-56, 320 49-63, 352 55-68, 384 59-73,
// 416 78-82, 448 70-91, 512 84-112): not a strict order. 80-column tiles of 192 and 256 tokens take
// longer than 96-column ones, 128 x 96 longer than 192 x 64. Still the pick is the fastest of the
// sixteen tiles, or within 2%, at 64 to 700 tokens of Qwen3-8B, 64 to 600 of Qwen2.5-7B and 100 to
// 1024 of Qwen2.5-0.5B (2000: 48.2 against 45.0 at 128 x 64). BM + 4 x columns, the rows that the
// loads issue (both token groups load the weights, the second from L1), picks worse: Qwen3-8B 200
// tokens 65 against 60, 256: 68 against 63, 600: 138 against 134, and nowhere better.
// The 192-token tiles: Qwen3-8B 160 tokens 59 -> 53 us, 300: 87 -> 70, 700: 160 -> 141.
void frag_pick_tile(int64_t tokens, int64_t inter, int64_t& token_tile, int64_t& column_tile) {
  const int64_t ncu = std::max(1, device_cu_count());
  int64_t best = INT64_MAX;
  for (int64_t bm : {128, 192, 256})
    for (int64_t cols : {32, 48, 64, 80, 96, 128}) {
      if (bm > 128 && cols == 32) continue;  // four waves of 96 or 128 tokens: slower than their rows
      const int64_t rows = cdiv(cdiv(tokens, bm) * cdiv(inter, cols), ncu) * (bm + 2 * cols);
      if (rows < best) {
        best = rows;
        token_tile = bm;
        column_tile = cols;
      }
    }
}

template <typename T>
int launch_frag_tile(const GemmArgs& a, int64_t token_tile, int64_t column_tile, hipStream_t st) {
  if (token_tile == 128) {
    switch (column_tile) {
      case 32: return launch_frag<T, 128, 2, 16>(a, st);
      case 48: return launch_frag<T, 128, 3, 16>(a, st);
      case 64: return launch_frag<T, 128, 4, 16>(a, st);
      case 80: return launch_frag<T, 128, 5, 16>(a, st);
      case 96: return launch_frag<T, 128, 6, 16>(a, st);
      default: return launch_frag<T, 128, 4, 32>(a, st);
    }
  }
  if (token_tile == 192) {
    switch (column_tile) {
      case 48: return launch_frag<T, 192, 3, 16>(a, st);
      case 64: return launch_frag<T, 192, 4, 16>(a, st);
      case 80: return launch_frag<T, 192, 5, 16>(a, st);
      case 96: return launch_frag<T, 192, 6, 16>(a, st);
      default: return launch_frag<T, 192, 4, 32>(a, st);
    }
  }
  switch (column_tile) {
    case 48: return launch_frag<T, 256, 3, 16>(a, st);
    case 64: return launch_frag<T, 256, 4, 16>(a, st);
    case 80: return launch_frag<T, 256, 5, 16>(a, st);
    case 96: return launch_frag<T, 256, 6, 16>(a, st);
    default: return launch_frag<T, 256, 4, 32>(a, st);
  }
}

// The packed entry points' body: token_tile 0 lets frag_pick_tile choose.
int gemm_packed_core(const void* x, int64_t x_row_stride, const void* packed, int dtype, int64_t tokens,
                     int64_t hidden, int64_t inter, int64_t num_workgroups, int64_t token_tile, int64_t column_tile,
                     void* out, int64_t out_row_stride, void* stream) {
  if (tokens == 0) return EMBER_OK;
  if (tokens < 0 || tokens > (int64_t(1) << 24) || hidden < 64 || hidden % 64 != 0 || hidden > (int64_t(1) << 20) ||
      inter < 64 || inter % 64 != 0 || inter > (int64_t(1) << 28) || num_workgroups < 1)
    return EMBER_EINVAL;
  const bool shape = (token_tile == 256 && (column_tile == 64 || column_tile == 128)) ||
                     (token_tile == 128 && column_tile == 128);
  if (token_tile != 0 && (!shape || inter % column_tile != 0)) return EMBER_EINVAL;
  if (dtype != EMBER_F16 && dtype != EMBER_BF16) return EMBER_EINVAL;
  if (x == nullptr || packed == nullptr || out == nullptr || !aligned16(x) || !aligned16(packed) || !aligned16(out))
    return EMBER_EINVAL;
  if (x_row_stride < hidden || out_row_stride < inter || x_row_stride % 8 != 0 || out_row_stride % 4 != 0)
    return EMBER_EINVAL;
  const int64_t total = (inter / 64) * (hidden / 64);
  if (total > INT32_MAX) return EMBER_EINVAL;  // 32 TiB of weights
  // A tile's rows are addressed by 32-bit offsets: rows farther apart than that allows go in
  // calls of one token.
  constexpr int64_t kMaxStride = int64_t(1) << 22;
  const int64_t per_call = x_row_stride > kMaxStride ? 1 : tokens;
  if (token_tile == 0) frag_pick_tile(per_call, inter, token_tile, column_tile);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  for (int64_t t = 0; t < tokens; t += per_call) {
    const GemmArgs a{static_cast<const char*>(x) + 2 * t * x_row_stride, x_row_stride, packed, 0,
                     static_cast<char*>(out) + 2 * t * out_row_stride, out_row_stride, static_cast<int>(per_call),
                     static_cast<int>(hidden), static_cast<int>(inter), nullptr, nullptr, 0, 1, 0, 0, 0, nullptr,
                     total, num_workgroups < total ? num_workgroups : total};  // the packing's grid
    const int rc = dtype == EMBER_F16 ? launch_frag_tile<_Float16>(a, token_tile, column_tile, st)
                                      : launch_frag_tile<__bf16>(a, token_tile, column_tile, st);
    if (rc != EMBER_OK) return rc;
  }
  return EMBER_OK;
}

template <typename T, int BNG, int BM = 256, bool MOE = false, bool PK = false>
int launch_gemm(const GemmArgs& a, hipStream_t st) {
  const int64_t grid = cdiv(a.T, BM) * cdiv(a.I, BNG);
  if (grid > 0x7fffffffLL) return EMBER_EINVAL;
  hipLaunchKernelGGL((k_gate_up_silu_gemm<T, BNG, BM, MOE, PK>), dim3(static_cast<uint32_t>(grid)), dim3(512), 0, st,
                     a);
  return launch_status();
}

// The tile shapes: (tokens, gate columns) of 256 x 64, 256 x 96, 256 x 128 or 128 x 128;
// every one gives each of the 8 waves 64 tokens x (WC gate + WC up) columns. 96-column
// tiles need I only a multiple of 16 (the last tile may be ragged), the others I a
// multiple of the tile.
template <typename T, bool MOE>
int launch_tile(const GemmArgs& a, int64_t token_tile, int64_t column_tile, hipStream_t st) {
  if (token_tile == 128) return launch_gemm<T, 128, 128, MOE>(a, st);
  if (column_tile == 96) return launch_gemm<T, 96, 256, MOE>(a, st);
  return column_tile == 64 ? launch_gemm<T, 64, 256, MOE>(a, st) : launch_gemm<T, 128, 256, MOE>(a, st);
}

bool gemm_tile_ok(int64_t token_tile, int64_t column_tile, int64_t inter) {
  const bool shape = (token_tile == 256 && (column_tile == 64 || column_tile == 96 || column_tile == 128)) ||
                     (token_tile == 128 && column_tile == 128);
  return shape && inter >= column_tile && inter % (column_tile == 96 ? 16 : column_tile) == 0;
}

}  // namespace
}  // namespace ember

extern "C" int ember_gate_up_silu_gemm(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                       int dtype, int64_t tokens, int64_t hidden, int64_t inter, int64_t token_tile,
                                       int64_t column_tile, void* out, int64_t out_row_stride, void* stream) {
  using namespace ember;
  if (tokens == 0) return EMBER_OK;
  if (tokens < 0 || tokens > (int64_t(1) << 24) || hidden < 64 || hidden % 64 != 0 || hidden > (int64_t(1) << 20) ||
      !gemm_tile_ok(token_tile, column_tile, inter) || inter > (int64_t(1) << 28))
    return EMBER_EINVAL;
  if (dtype != EMBER_F16 && dtype != EMBER_BF16) return EMBER_EINVAL;
  if (x == nullptr || w == nullptr || out == nullptr || !aligned16(x) || !aligned16(w) || !aligned16(out))
    return EMBER_EINVAL;
  if (x_row_stride < hidden || w_row_stride < hidden || out_row_stride < inter || x_row_stride % 8 != 0 ||
      w_row_stride % 8 != 0 || out_row_stride % 4 != 0)
    return EMBER_EINVAL;
  GemmArgs a{x, x_row_stride, w, w_row_stride, out, out_row_stride, static_cast<int>(tokens),
             static_cast<int>(hidden), static_cast<int>(inter), nullptr, nullptr, 0, 1, 0, 0, 0};
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == EMBER_F16) return launch_tile<_Float16, false>(a, token_tile, column_tile, st);
  return launch_tile<__bf16, false>(a, token_tile, column_tile, st);
}

extern "C" int ember_moe_gate_up_silu_gemm(const void* x, int64_t x_row_stride, int64_t num_tokens, const void* w,
                                           int64_t w_expert_stride, int64_t w_row_stride, int dtype,
                                           int64_t num_experts, int64_t hidden, int64_t inter,
                                           const int32_t* sorted_ids, const int32_t* block_expert, int64_t num_blocks,
                                           int64_t block_rows, int64_t num_valid, int64_t top_k, int64_t column_tile,
                                           void* out, int64_t out_row_stride, void* stream) {
  using namespace ember;
  if (num_blocks == 0 || num_valid == 0) return EMBER_OK;
  if (num_blocks < 0 || num_valid < 0 || num_tokens < 1 || top_k < 1 || num_experts < 1 || num_blocks > (1 << 22) ||
      num_valid > INT32_MAX / 2 || num_tokens > INT32_MAX || hidden < 64 || hidden % 64 != 0 ||
      hidden > (int64_t(1) << 20) || !gemm_tile_ok(block_rows, column_tile, inter) || inter > (int64_t(1) << 28))
    return EMBER_EINVAL;
  if (dtype != EMBER_F16 && dtype != EMBER_BF16) return EMBER_EINVAL;
  if (x == nullptr || w == nullptr || out == nullptr || sorted_ids == nullptr || block_expert == nullptr ||
      !aligned16(x) || !aligned16(w) || !aligned16(out))
    return EMBER_EINVAL;
  if (x_row_stride < hidden || w_row_stride < hidden || w_expert_stride < 2 * inter * w_row_stride ||
      out_row_stride < inter || x_row_stride % 8 != 0 || w_row_stride % 8 != 0 || w_expert_stride % 8 != 0 ||
      out_row_stride % 4 != 0)
    return EMBER_EINVAL;
  GemmArgs a{x, x_row_stride, w, w_row_stride, out, out_row_stride, static_cast<int>(num_blocks * block_rows),
             static_cast<int>(hidden), static_cast<int>(inter), sorted_ids, block_expert,
             static_cast<int>(num_valid), static_cast<int>(top_k), static_cast<int>(num_experts),
             static_cast<int>(num_tokens), w_expert_stride, device_error_word()};
  if (a.err == nullptr) return EMBER_ENODEV;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == EMBER_F16) return launch_tile<_Float16, true>(a, block_rows, column_tile, st);
  return launch_tile<__bf16, true>(a, block_rows, column_tile, st);
}

extern "C" int ember_gate_up_silu_gemm_packed(const void* x, int64_t x_row_stride, const void* packed, int dtype,
                                              int64_t tokens, int64_t hidden, int64_t inter, int64_t num_workgroups,
                                              int64_t token_tile, int64_t column_tile, void* out,
                                              int64_t out_row_stride, void* stream) {
  return ember::gemm_packed_core(x, x_row_stride, packed, dtype, tokens, hidden, inter, num_workgroups,
                                 token_tile > 0 ? token_tile : -1, column_tile, out, out_row_stride, stream);
}

extern "C" int ember_gate_up_silu_gemm_packed_auto(const void* x, int64_t x_row_stride, const void* packed, int dtype,
                                                   int64_t tokens, int64_t hidden, int64_t inter,
                                                   int64_t num_workgroups, void* out, int64_t out_row_stride,
                                                   void* stream) {
  return ember::gemm_packed_core(x, x_row_stride, packed, dtype, tokens, hidden, inter, num_workgroups, 0, 0, out,
                                 out_row_stride, stream);
}

namespace ember {
namespace {

// The packed experts' entry points' body; `rows64` admits the 64-row blocks.
int moe_gemm_packed_core(const void* x, int64_t x_row_stride, int64_t num_tokens, const void* packed, int dtype,
                         int64_t num_experts, int64_t hidden, int64_t inter, const int32_t* sorted_ids,
                         const int32_t* block_expert, int64_t num_blocks, int64_t block_rows, int64_t num_valid,
                         int64_t top_k, int64_t column_tile, bool rows64, void* out, int64_t out_row_stride,
                         void* stream) {
  if (num_blocks == 0 || num_valid == 0) return EMBER_OK;
  if (num_blocks < 0 || num_valid < 0 || num_tokens < 1 || top_k < 1 || num_experts < 1 || num_blocks > (1 << 22) ||
      num_valid > INT32_MAX / 2 || num_tokens > INT32_MAX || hidden < 64 || hidden % 64 != 0 ||
      hidden > (int64_t(1) << 20) || inter < 64 || inter > (int64_t(1) << 28))
    return EMBER_EINVAL;
  const bool shape = (rows64 && block_rows == 64 && column_tile == 128) ||
                     (block_rows == 256 && (column_tile == 64 || column_tile == 128)) ||
                     (block_rows == 128 && column_tile == 128);
  if (!shape || inter % column_tile != 0) return EMBER_EINVAL;
  if (dtype != EMBER_F16 && dtype != EMBER_BF16) return EMBER_EINVAL;
  if (x == nullptr || packed == nullptr || out == nullptr || sorted_ids == nullptr || block_expert == nullptr ||
      !aligned16(x) || !aligned16(packed) || !aligned16(out))
    return EMBER_EINVAL;
  if (x_row_stride < hidden || out_row_stride < inter || x_row_stride % 8 != 0 || out_row_stride % 4 != 0)
    return EMBER_EINVAL;
  GemmArgs a{x, x_row_stride, packed, 0, out, out_row_stride, static_cast<int>(num_blocks * block_rows),
             static_cast<int>(hidden), static_cast<int>(inter), sorted_ids, block_expert,
             static_cast<int>(num_valid), static_cast<int>(top_k), static_cast<int>(num_experts),
             static_cast<int>(num_tokens), 2 * inter * hidden, device_error_word(), 0, 1};
  if (a.err == nullptr) return EMBER_ENODEV;
  // the frag kernel addresses x rows by 32-bit offsets
  const bool frag = num_tokens * x_row_stride < (int64_t(1) << 29);
  if (block_rows == 64 && !frag) return EMBER_ETOOBIG;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == EMBER_F16) {
    if (block_rows == 128 && frag) return launch_frag<_Float16, 128, 4, 32, true>(a, st);
    if (block_rows == 64) return launch_frag<_Float16, 64, 4, 32, true>(a, st);
    if (block_rows == 128) return launch_gemm<_Float16, 128, 128, true, true>(a, st);
    return column_tile == 64 ? launch_gemm<_Float16, 64, 256, true, true>(a, st)
                             : launch_gemm<_Float16, 128, 256, true, true>(a, st);
  }
  if (block_rows == 128 && frag) return launch_frag<__bf16, 128, 4, 32, true>(a, st);
  if (block_rows == 64) return launch_frag<__bf16, 64, 4, 32, true>(a, st);
  if (block_rows == 128) return launch_gemm<__bf16, 128, 128, true, true>(a, st);
  return column_tile == 64 ? launch_gemm<__bf16, 64, 256, true, true>(a, st)
                           : launch_gemm<__bf16, 128, 256, true, true>(a, st);
}

}  // namespace
}  // namespace ember

extern "C" int ember_moe_gate_up_silu_gemm_packed(const void* x, int64_t x_row_stride, int64_t num_tokens,
                                                  const void* packed, int dtype, int64_t num_experts, int64_t hidden,
                                                  int64_t inter, const int32_t* sorted_ids,
                                                  const int32_t* block_expert, int64_t num_blocks, int64_t block_rows,
                                                  int64_t num_valid, int64_t top_k, int64_t column_tile, void* out,
                                                  int64_t out_row_stride, void* stream) {
  return ember::moe_gemm_packed_core(x, x_row_stride, num_tokens, packed, dtype, num_experts, hidden, inter, sorted_ids,
                                     block_expert, num_blocks, block_rows, num_valid, top_k, column_tile, false, out,
                                     out_row_stride, stream);
}

extern "C" int ember_moe_gate_up_silu_gemm_packed_rows64(const void* x, int64_t x_row_stride, int64_t num_tokens,
                                                         const void* packed, int dtype, int64_t num_experts,
                                                         int64_t hidden, int64_t inter, const int32_t* sorted_ids,
                                                         const int32_t* block_expert, int64_t num_blocks,
                                                         int64_t num_valid, int64_t top_k, void* out,
                                                         int64_t out_row_stride, void* stream) {
  return ember::moe_gemm_packed_core(x, x_row_stride, num_tokens, packed, dtype, num_experts, hidden, inter, sorted_ids,
                                     block_expert, num_blocks, 64, num_valid, top_k, 128, true, out, out_row_stride,
                                     stream);
}
