// The screened pass 1 of the isotropic and diagonal models' default plans (gfx950), and
// the device-side choice of a call's branches.
#pragma once

#include <algorithm>

#include "fgmm_common.hpp"

namespace fgmm {
namespace {

// 16-feature chunks of the approximate contraction: x (and, for the diagonal model, x^2)
// and the constants' chunk.
constexpr int kScreenWaves = 4;     // waves per workgroup, 64 rows (two 32-row tiles) each
__host__ __device__ constexpr int screen_chunks(int DP, bool DIAG) { return (DIAG ? 2 : 1) * (DP / 16) + 1; }
// Component blocks per LDS stage: two, or one where two stages of two would leave room
// for one workgroup per compute unit only.
__host__ __device__ constexpr int screen_blocks(int DP, bool DIAG) { return DIAG && DP > 96 ? 1 : 2; }
__host__ __device__ constexpr int screen_rs(int DP) { return DP / 2 + 8; }   // bf16 row stride of a staging tile
__host__ __device__ constexpr size_t screen_stage_bytes(int DP, bool DIAG) {
  return (size_t)screen_blocks(DP, DIAG) * screen_chunks(DP, DIAG) * 64 * 16;
}
// Per wave: half of a 32-row tile's columns in bf16 and their partial sums of squares
// (DIAG: x and x^2, and partial sums of x^2 and x^4).
__host__ __device__ constexpr size_t screen_tile_bytes(int DP, bool DIAG) {
  return (DIAG ? 2 : 1) * ((size_t)32 * screen_rs(DP) * 2 + (size_t)32 * (DP / 8 + 1) * 4);
}
// The first stage's operands, then the staging tiles, which the second stage and the
// rows' block bounds (bf16, 64 rows per wave) overlay once the rows are in registers.
__host__ __device__ constexpr size_t screen_lds_bytes(int DP, bool DIAG, int KB) {
  const size_t a = kScreenWaves * screen_tile_bytes(DP, DIAG);
  const size_t b = screen_stage_bytes(DP, DIAG) + (size_t)kScreenWaves * 64 * round_up(KB, 8) * 2;
  return screen_stage_bytes(DP, DIAG) + (a > b ? a : b);
}
// Calls that may screen: at least 4 blocks (with one near block a row, screening B blocks
// leaves 1/B of the exact contraction), two workgroups per compute unit (the rows' block
// bounds in LDS: at most 2816 components at D = 128 and 1792 diagonal ones at D = 96; beyond,
// the exact pass 1 runs) and at least kScreenMinWork (32-row tile, block, chunk) steps.
// Calls that the probe then leaves to the exact pass 1 pay for the probe and two kernels that
// return, 10 to 22 us, where they had no probe before (the default plan without the automatic
// stored branch); N(0, I) rows, K=1024, without and with: at 500,000 steps 305 and 309 us
// (D=128), 345 and 360 us (D=96), 324 and 335 us (D=64), at 250,000 steps 201 and 222, 203
// and 216, 187 and 198 us, at 2,000,000 at most 2% more.  Separated clusters gain at once: at
// 250,000 steps 136 -> 92 us, 130 -> 84 us and 153 -> 99 us, at 500,000 167 -> 101, 192 ->
// 126 and 258 -> 113 us.  So the line lies where the first has become small, well above the
// crossover of the second (between 60,000 and 125,000 steps).
constexpr int64_t kScreenMinWork = 500000;
constexpr int64_t kMaxScreenLdx = (int64_t)4 << 20;   // 64 rows within 32-bit buffer offsets
__host__ inline bool use_screen(int64_t N, int DP, bool DIAG, int KB) {
  return DP <= 128 && KB >= 4 && KB <= kProbeMaxKB && N < ((int64_t)1 << 31) - 256 &&
         cdiv(N, 32) * KB * (screen_chunks(DP, DIAG) - 1) >= kScreenMinWork &&
         screen_lds_bytes(DP, DIAG, KB) <= (size_t)80 * 1024;
}
constexpr int kListBase = 64;   // ints before the first row of the list (entry 0: its length)
// Lists of up to this many 32-row workgroups per compute unit run one tile per workgroup
// (a round of them takes about a quarter of a round of whole workgroups).
constexpr int kFewRounds = 3;
__host__ inline int64_t few_rows(int64_t grid) {
  return 32 * std::min<int64_t>((int64_t)kFewRounds * current_device_cus(), grid);
}
// Bytes of a row's share of its tile's need words, rounded up: the gathering pass 2 after the
// screening reads them through a resource over its slab (cap_slab_rows).
__host__ constexpr size_t screen_word_bytes(int KB, size_t word) { return ((size_t)KB * word + 31) / 32; }

// The screened pass 1 tells near pairs from faint ones.  A pair is near unless its
// responsibility r provably has r, r ||x||, r ||x||^2 <= 2^-kNearGap.  Pass 2 takes the near
// pairs, and then the faint ones of those blocks that hold a component with Nk < kNearNk.
// What it leaves out, the faint pairs of the other components, changes their Nk by at most
// N 2^-72 in absolute value, less than a rounding (N 2^-72 <= 2^-41, against 2^-24 of 2^-10),
// and their other sums by at most N 2^-72 each: an element of mu_acc that is 0 in the near
// rows, or whose terms cancel, loses terms of that size.  A row's terms outside its near
// blocks change no bit of its fp32 log-sum-exp (at most K 2^-72 of it).
constexpr float kNearGap = 72.0f;
constexpr float kNearNk = 0x1p-10f;
// Pass 2 marks, in one word per block (`alive`, zeroed by the prologue), the components
// with Nk >= kNearNk from the near pairs of one partial; the blocks whose word is
// complete need no faint pass.
__device__ __forceinline__ void mark_alive(unsigned* __restrict__ alive, int kb, float nk) {
  const unsigned m = (unsigned)__builtin_amdgcn_ballot_w64(nk >= kNearNk);
  if ((threadIdx.x & 63) == 0 && m != 0u) atomicOr(alive + kb, m);
}

// The norm of the vector of squares, sqrt(sum x^4), from the fp32 sums xs = ||x||^2 and xq =
// sum x^4.  Where fourth powers may have underflowed it is bounded by xs; what xs loses
// itself (x^2 below 2^-126) is under 2^-19 of log-joint for weights up to 1e30.
__device__ __forceinline__ float squares_norm(float xs, float xq) { return xq < 0x1p-100f ? xs : sqrtf(xq); }

// The factor of the row's norm in the screening's error bound (screen_pairs): from an operand
// row's sums of squares, of its rounding errors and of its rounded values.
__device__ __forceinline__ double screen_weight_error(double err_sq, double rounded_sq) {
  return sqrt(err_sq) + 0x1.06p-8 * sqrt(rounded_sq);
}

// The components of a block that weigh something (log_pi > -inf, or NaN) in the screening's
// operands, for the models' prologues (lane c of a half-wave is component c).  A component
// without weight, padding included, repeats the block's first one with weight, so that it
// does not change the row's block maximum; a block of such components only gets the
// constant -inf: it raises no row's lower bound and gets a bit only where no block has one.
// (A finite constant in their place wins once a row's log-joints are all below it.)
struct BlockLive {
  unsigned mask;
  int src;   // the lane to copy from
  __device__ explicit BlockLive(bool live) {
    const int lane = threadIdx.x & 63;
    mask = (unsigned)__builtin_amdgcn_ballot_w64(live);   // the half-waves agree
    src = live || mask == 0u ? lane : (lane & 32) + __builtin_ctz(mask);
  }
  __device__ __forceinline__ uint2 copy(uint2 v) const {
    if (mask == ~0u) return v;   // uniform
    return make_uint2(__shfl(v.x, src), __shfl(v.y, src));
  }
  __device__ __forceinline__ bf16x8 copy(const bf16x8& a) const {
    uint4 w = __builtin_bit_cast(uint4, a);
    const uint2 lo = copy(make_uint2(w.x, w.y)), hi = copy(make_uint2(w.z, w.w));
    return __builtin_bit_cast(bf16x8, make_uint4(lo.x, lo.y, hi.x, hi.y));
  }
  // The same for the constants' chunk, whose second half (g == 1) starts with the constant
  // against the row operand's ones.
  __device__ __forceinline__ bf16x8 constants(bf16x8 a, int g) const {
    if (mask != 0u) return copy(a);
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = (__bf16)0.0f;
    if (g == 1) a[0] = (__bf16)(-INFINITY);
    return a;
  }
};

// How a call's passes run.  The probe's last workgroup sums its counts and writes the
// choice as one word, which every later kernel of the call reads with one scalar load
// (each summing the counts for itself cost 0.5 us a kernel).
enum CallMode { kModeDefault = 0, kModeStored = 1, kModeScreen = 2 };
__device__ __forceinline__ int call_mode(const int* __restrict__ sel) { return sel ? *sel : kModeDefault; }
// What the probe chooses from: up to max_multi sampled rows near several blocks, the
// screened pass 1 (-1: never); else, from min_pairs needed pairs on, the stored branch if
// the call has one.  The callers' max_multi is half of the rows.  Clustered rows with that
// share on the list, screened and exact, us: N=1M K=1024 D=128 2744 and 3217 (0.50 listed),
// N=500K D=96 1013 and 1414 (0.49), N=400K K=300 D=50 399 and 508 (0.53), diagonal N=1M
// K=1024 D=96 3123 and 5257 (0.58), N=500K D=64 906 and 2032 (0.47); the two cross at 0.6
// (isotropic D=128) to 0.95 (diagonal D=64).  Not so where, besides, a few components hold
// many of the rows: the gathering pass 2 takes longer for such a block with logZ formed in it
// (N=1M K=1024 D=128, half of the clusters without a component of their own: 3756 and 2971).
struct ProbeRule {
  int64_t max_multi, min_pairs;
  int stored;
};
// A call's state words: the choice, the probe's count of finished workgroups and (from
// kStateAlive on, screened calls) a word per block (mark_alive); the prologue zeroes the
// last two.  The probe's counts (two per sampled tile: needed pairs, then from
// kProbeTiles on rows near several blocks) are pass 1's only.
constexpr int kStateMode = 0, kStateDone = 1, kStateAlive = 2;
constexpr size_t kProbeBytes = 2 * kProbeTiles * sizeof(unsigned);
__host__ __device__ constexpr size_t state_bytes(int KB) { return (size_t)(kStateAlive + KB) * sizeof(unsigned); }

// The partials a call left: `stored` of them where the stored branch ran, else `n`.
struct PartCount {
  const int* sel;
  int n, stored;
};
__device__ __forceinline__ int part_count(const PartCount& p) {
  return call_mode(p.sel) == kModeStored ? p.stored : p.n;
}

// The end of a probe kernel, run by one wave of each of its ntile workgroups: tile s had
// `pairs` needed pairs and `multi` rows near several blocks (from lane 0).  The last
// workgroup to finish makes the choice.
__device__ __forceinline__ void probe_choose(unsigned* __restrict__ count, unsigned* __restrict__ state, int s,
                                             int ntile, unsigned pairs, unsigned multi, const ProbeRule& rule) {
  const int lane = threadIdx.x & 63;
  unsigned done = 0;
  if (lane == 0) {
    count[s] = pairs;
    count[kProbeTiles + s] = multi;
    __threadfence();
    done = atomicAdd(state + kStateDone, 1u);
  }
  if (__builtin_amdgcn_readfirstlane(done) != (unsigned)ntile - 1u) return;
  // Every count is visible to device-scope loads.
  __threadfence();
  uint64_t t = 0;
  if (lane < ntile)
    t = ((uint64_t)__hip_atomic_load(count + kProbeTiles + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) << 32) |
        __hip_atomic_load(count + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);   // at most 2^20 pairs and 2^11 rows
  if (lane == 0)
    state[kStateMode] = (int64_t)(t >> 32) <= rule.max_multi ? kModeScreen
                        : rule.stored && (int64_t)(t & 0xffffffffu) >= rule.min_pairs ? kModeStored : kModeDefault;
}
// Both probes' second half (1024 threads): from the sampled tile's block maxima R and error
// bounds (rmax, rerr: [block][row]), the pairs with R >= the row's largest less
// kLjNeedGap (those the exact pass 1 would mark) and the rows the screening would find
// near several blocks; then the choice.  row_a, row_b, part, blocks: LDS scratch.
struct ProbeScratch {
  float a[32][33], b[32][33];
  unsigned part[16], blocks[32];
};
__device__ __forceinline__ void probe_finish(const float* rmax, const float* rerr, ProbeScratch& sh, int KB, bool valid,
                                             float nx, bool screen, int s, int ntile, const ProbeRule& rule,
                                             unsigned* __restrict__ count, unsigned* __restrict__ state) {
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, wave = tid >> 6;
  if (tid < 32) sh.blocks[tid] = 0u;
  __syncthreads();
  // Each row's largest maximum R and largest lower bound L: 32 threads a row.
  const int t32 = tid >> 5;
  float R = -INFINITY, L = -INFINITY;
  for (int kb = t32; kb < KB; kb += 32) {
    const float r = rmax[kb * 32 + c];
    R = fmaxf(R, r);
    L = fmaxf(L, r - rerr[kb * 32 + c]);
  }
  sh.a[t32][c] = R;
  sh.b[t32][c] = L;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    R = fmaxf(R, sh.a[j][c]);
    L = fmaxf(L, sh.b[j][c]);
  }
  unsigned need = 0, kept = 0;
  if (valid) {
    const float near_gap = fminf(kLjNeedGap, kNearGap + 2.0f * log2f(1.0f + nx));
    for (int kb = t32; kb < KB; kb += 32) {
      const float r = rmax[kb * 32 + c];
      need += (r - R >= -kLjNeedGap) ? 1u : 0u;
      kept += !(r + rerr[kb * 32 + c] - L < -near_gap) ? 1u : 0u;
    }
    if (screen && kept != 0) atomicAdd(sh.blocks + c, kept);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) need += __shfl_xor(need, o);
  if (lane == 0) sh.part[wave] = need;
  __syncthreads();
  if (wave != 0) return;
  unsigned tot = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) tot += sh.part[w];
  const uint64_t multi = __builtin_amdgcn_ballot_w64(screen && lane < 32 && sh.blocks[c] > 1u);
  probe_choose(count, state, s, ntile, tot, (unsigned)__builtin_popcountll(multi), rule);
}

// ---------------------------------------------------------------------------
// The screened pass 1 (default plans up to D = 128, large calls, selected by the probe).
//
// Where clusters are separated, the exact contraction (seven bf16 steps per 16
// dimensions) of nearly every (row, block) pair only proves that its responsibilities
// are zero.  This kernel proves it with one step: the approximate log-joint
//   iso:  a_nk = sum_d bf16(x_d) bf16(2 b_k mu_kd) - b_k ||x||^2 + C_k
//   diag: a_nk = sum_d bf16(x_d) bf16(2 v_kd) + sum_d bf16(x_d^2) bf16(-w_kd) + C_k
// comes straight out of the matrix cores (the constants are one more chunk of three-way
// splits), a row's block maximum is a maximum of accumulators, and per block (the models'
// prologues form sc_e)
//   |a_nk - ll2_nk| <= E = sc_e.x ||x|| + sc_e.y s + sc_e.z,
// s = ||x||^2 (iso) or the norm of the vector of squares (diag, squares_norm).  With w an
// operand's row and h its rounding to bf16, |x.w - bf16(x).h| <= ||x|| ||w - h|| +
// ||x - bf16(x)|| ||h||, the second of at most 2^-8 ||x|| ||h|| (8 significant bits), so
// ||x||'s factor is ||w - h|| + 0x1.06p-8 ||h|| (screen_weight_error; 0x1.06 for the
// second-order terms and the sum's roundings), s's likewise (diag); the constants' dropped
// split products and their fp32 sums err by under 2^-14 (b ||x||^2 + |C|).  (Bounding
// ||w - h|| by 2^-8 ||w|| too lists a fifth more of the rows at K=300 D=50.)
// With L the largest a - E over all blocks (logZ2 >= L), a block with a + E < L -
// kLjNeedGap holds only responsibilities that are exactly zero, as the need masks of the
// exact pass 1 state; the other blocks get their need bit.  Not-finite values make E
// or a infinite or NaN, and the comparison then keeps the block.
// A row with one near block needs no other block for logZ either: the gathering pass 2
// forms its log-sum-exp there (the pair's bit is set in both words, near and faint).  The
// rest go on a list, which the exact pass 1 then runs.
//
// Bound: matrix steps and VALU, which mostly add up on a SIMD: at D = 128, 9 matrix
// steps (288 cycles) and 31 VALU instructions per (32 rows, block), 58% and 25% of the SIMDs'
// cycles (diagonal, D = 96: 13 and 36, 56% and 19%).  Each operand read from LDS serves two
// 32-row tiles.  Rows are read in whole lines and transposed through LDS (the exact pass
// reads 16-byte pieces of 32 rows per instruction, which at this kernel's length would bound
// it).  N=1M K=1024 D=128 clustered: 0.27 ms, drop-in call 1.75 -> 0.57 ms; N=400K K=300
// D=50: call 0.51 -> 0.28 ms; diagonal N=1M K=1024 D=96 clustered 0.38 ms, call 2.86 ->
// 0.69 ms.
// ---------------------------------------------------------------------------
template <int DP, bool DIAG>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * kScreenWaves, 64 * kScreenWaves),
                          amdgpu_waves_per_eu(DIAG ? 2 : 3, DIAG ? 2 : 3)))
void screen_pairs(const float* __restrict__ X, int64_t ldx, int64_t N, int D, const bf16x8* __restrict__ sc_op,
                const float4* __restrict__ sc_e, int KB, unsigned* __restrict__ need, unsigned* __restrict__ faint, int wstride,
                  int* __restrict__ list, const int* __restrict__ sel) {
  constexpr int NC = screen_chunks(DP, DIAG), NQ = DP / 16;
  constexpr int SB = screen_blocks(DP, DIAG);
  constexpr int BLK = NC * 64;                    // bf16x8 per block
  constexpr int STG = SB * BLK;                   // bf16x8 per stage
  constexpr int RS = screen_rs(DP), V4 = DP / 8;  // float4 per half row
  constexpr int LPT = 32 * V4 / 64;               // float4 per lane and half tile
  if (call_mode(sel) != kModeScreen) return;

  extern __shared__ __align__(16) unsigned char lds_raw[];
  bf16x8* const op0 = reinterpret_cast<bf16x8*>(lds_raw);
  unsigned char* const rest = lds_raw + screen_stage_bytes(DP, DIAG);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, g = lane >> 5;
  unsigned short* const ub_l = reinterpret_cast<unsigned short*>(rest + screen_stage_bytes(DP, DIAG)) +
                               wave * 64 * ((KB + 7) & ~7) + lane;

  // Stage st (blocks SB st ..) into operand buffer st & 1, in 1 KB pieces.
  auto fetch = [&](int st) {
    const int nb = KB - st * SB < SB ? KB - st * SB : SB;
    const DmaSrc r = dma_src(sc_op + (int64_t)st * STG, (uint32_t)(nb * BLK * (int)sizeof(bf16x8)));
    bf16x8* dst = (st & 1) ? reinterpret_cast<bf16x8*>(rest) : op0;
    for (int p = wave; p < nb * NC; p += kScreenWaves)
      lds_dma16(r, dst + p * 64, lane * (int)sizeof(bf16x8), p * 64 * (int)sizeof(bf16x8));
  };
  const int64_t row0 = (int64_t)blockIdx.x * (64 * kScreenWaves) + wave * 64;
  const int64_t row = row0 + lane;
  fetch(0);

  // The wave's two 32-row tiles in halves of the columns: whole 128-byte lines per load,
  // rounded to bf16 into the wave's staging tile and read back as B operands; ||x||^2
  // from the fp32 values.  The next half's loads are in flight meanwhile.
  __bf16* const xt = reinterpret_cast<__bf16*>(rest + wave * screen_tile_bytes(DP, DIAG));
  float* const sq = reinterpret_cast<float*>(xt + (DIAG ? 2 : 1) * 32 * RS);
  bf16x8 xb[2][NC];
  float xs = 0.0f, xq = 0.0f;   // of the lane's own row, row0 + lane: ||x||^2, sum of x^4 (DIAG)
  f32x4 raw[2][LPT];
  // Rows past N lie past the resource and read zeros, as do columns from D on.
  const int64_t rows = N - row0 < 64 ? (N - row0 > 0 ? N - row0 : 0) : 64;
  const buf_rsrc xr = make_rsrc(X + (rows > 0 ? row0 * ldx : 0), (uint32_t)(rows * ldx * (int64_t)sizeof(float)));
  const int rbytes = (int)ldx * (int)sizeof(float);
  auto load = [&](int u, f32x4 (&r)[LPT]) __attribute__((always_inline)) {
    if constexpr (64 % V4 == 0) {   // a lane's column is the same in every load
      const int d0 = (u & 1) * (DP / 2) + 4 * (lane % V4);
      int off = d0 < D ? (32 * (u >> 1) + lane / V4) * rbytes + d0 * 4 : kBufOob;
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        r[i] = buf_load_f32x4(xr, buf_off(off));
        off += (64 / V4) * rbytes;
        if (d0 >= D) off = kBufOob;
      }
    } else {
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        const int idx = i * 64 + lane, d0 = (u & 1) * (DP / 2) + 4 * (idx % V4);
        r[i] = buf_load_f32x4(xr, buf_off(d0 < D ? (32 * (u >> 1) + idx / V4) * rbytes + d0 * 4 : kBufOob));
      }
    }
    if (D & 3) {   // uniform: the columns past D inside the last vector
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        const int d0 = (u & 1) * (DP / 2) + 4 * ((i * 64 + lane) % V4);
        if (d0 + 1 >= D) r[i].y = 0.0f;
        if (d0 + 2 >= D) r[i].z = 0.0f;
        if (d0 + 3 >= D) r[i].w = 0.0f;
      }
    }
  };
  load(0, raw[0]);
  float s = 0.0f, s4 = 0.0f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int t = u >> 1, h = u & 1;
    if (u < 3) load(u + 1, raw[(u + 1) & 1]);
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int idx = i * 64 + lane, rr = idx / V4, v = idx % V4;
      const f32x4 x = raw[u & 1][i];
      const uint2 w = {bf16_pair(f32x2{x.x, x.y}), bf16_pair(f32x2{x.z, x.w})};
      *reinterpret_cast<uint2*>(xt + rr * RS + 4 * v) = w;
      const f32x4 y = x * x;
      sq[rr * (V4 + 1) + v] = (y.x + y.y) + (y.z + y.w);
      if constexpr (DIAG) {
        const uint2 w2 = {bf16_pair(f32x2{y.x, y.y}), bf16_pair(f32x2{y.z, y.w})};
        *reinterpret_cast<uint2*>(xt + (32 + rr) * RS + 4 * v) = w2;
        sq[(32 + rr) * (V4 + 1) + v] = fmaf(y.x, y.x, fmaf(y.y, y.y, fmaf(y.z, y.z, y.w * y.w)));
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (h == 0) s = s4 = 0.0f;
#pragma unroll
    for (int v = 0; v < V4; ++v) {
      s += sq[c * (V4 + 1) + v];
      if constexpr (DIAG) s4 += sq[(32 + c) * (V4 + 1) + v];
    }
#pragma unroll
    for (int q = 0; q < NQ / 2; ++q) {
      xb[t][h * (NQ / 2) + q] = *reinterpret_cast<const bf16x8*>(xt + c * RS + 16 * q + 8 * g);
      if constexpr (DIAG)
        xb[t][NQ + h * (NQ / 2) + q] = *reinterpret_cast<const bf16x8*>(xt + (32 + c) * RS + 16 * q + 8 * g);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (h == 1) {
      if (g == t) {
        xs = s;
        xq = s4;
      }
      // The constants' chunk: ||x||^2's splits in the first half (DIAG: against zeros),
      // ones in the second.
      f32x4 lo = zero4();
      lo.x = DIAG ? 0.0f : s;
      bf16x8 sp[3], a;
      split3_bf16(lo, zero4(), sp);
      const __bf16 one = (__bf16)1.0f, zero = (__bf16)0.0f;
      a[0] = g == 0 ? sp[0][0] : one;
      a[1] = g == 0 ? sp[1][0] : one;
      a[2] = g == 0 ? sp[2][0] : one;
      a[3] = g == 0 ? sp[0][0] : zero;
      a[4] = g == 0 ? sp[1][0] : zero;
      a[5] = g == 0 ? sp[0][0] : zero;
      a[6] = zero;
      a[7] = zero;
      xb[t][NC - 1] = a;
    }
  }
  const float nx = sqrtf(xs), ny = DIAG ? squares_norm(xs, xq) : xs;
  lds_barrier();   // every wave has read its staging tile: the second stage and the bounds may overwrite it

  uint2* const words_l = reinterpret_cast<uint2*>(ub_l - lane);   // 32 blocks' words take 4 blocks' bounds
  for (int kb = KB; kb < ((KB + 7) & ~7); ++kb) ub_l[kb * 64] = 0xff7f;   // the least finite bound

  float L = -INFINITY;
  const int nst = (KB + SB - 1) / SB;
  for (int st = 0; st < nst; ++st) {
    dma_barrier();   // stage st has landed, and every wave is done with stage st - 1
    if (st + 1 < nst) fetch(st + 1);
    const bf16x8* op = ((st & 1) ? reinterpret_cast<const bf16x8*>(rest) : op0) + lane;
#pragma unroll
    for (int j = 0; j < SB; ++j) {
      const int kb = st * SB + j;
      if (kb >= KB) break;
      const float4 e = sc_e[kb];
      // All of the block's operand reads in flight before the first is used.
      bf16x8 a[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) a[q] = op[(j * NC + q) * 64];
      __builtin_amdgcn_sched_barrier(0);
      f32x16 acc[2] = {zero16(), zero16()};
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int q = 0; q < NC; ++q) acc[t] = mfma_bf16(a[q], xb[t][q], acc[t]);
      }
      float m[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        m[t] = acc[t][0];
#pragma unroll
        for (int i = 1; i < 16; ++i) m[t] = fmaxf(m[t], acc[t][i]);
      }
      // Lane l's own row is row l % 32 of tile l / 32; the other half-wave holds half of
      // its block maximum.
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[0]), __float_as_uint(m[1]), false, false);
      const float am = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      const float E = fmaf(e.x, nx, fmaf(e.y, ny, e.z));
      // The bound rounded up to bf16: truncation does it for negative values, and for
      // positive ones after adding 2^-7 of them (one bf16 step or more).
      const float ub = am + E;
      ub_l[kb * 64] = (unsigned short)(__float_as_uint(fmaf(fmaxf(ub, 0.0f), 0x1p-7f, ub)) >> 16);
      L = fmaxf(L, am - E);
    }
  }

  // Need words of the two tiles (each lane reads back the bounds it wrote itself), 32
  // blocks at a time, lane c of half g keeping block kb0 + c of tile g.
  const uint64_t valid = __builtin_amdgcn_ballot_w64(row < N);   // a row past N gets no bit
  const float near_gap = fminf(kLjNeedGap, kNearGap + 2.0f * log2f(1.0f + nx));   // kLjNeedGap if nx is NaN
  uint64_t once = 0, twice = 0;   // rows with at least one, two near blocks
  const int64_t tile = (row0 >> 5) + g;
  for (int kb0 = 0; kb0 < KB; kb0 += 32) {
    unsigned w = 0, wf = 0;
#pragma unroll 1
    for (int j0 = 0; j0 < 32 && kb0 + j0 < KB; j0 += 8) {
      // Eight bounds in flight together (past KB: the fill).
      float ub[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) ub[j] = bf16_bits_to_float(ub_l[(kb0 + j0 + j) * 64]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float u = ub[j] - L;
        const uint64_t b = __builtin_amdgcn_ballot_w64(!(u < -near_gap)) & valid;
        const uint64_t f = __builtin_amdgcn_ballot_w64(!(u < -kLjNeedGap)) & valid & ~b;
        twice |= once & b;
        once |= b;
        if (c == j0 + j) {
          w = g == 0 ? (unsigned)b : (unsigned)(b >> 32);
          wf = g == 0 ? (unsigned)f : (unsigned)(f >> 32);
        }
      }
    }
    // Kept (over the bounds of the blocks just read) until the rows near one block only
    // are known.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    words_l[kb0 * 16 + lane] = make_uint2(w, wf);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const uint64_t one = once & ~twice;
  const uint64_t many = valid & ~one;
  const unsigned own = g == 0 ? (unsigned)one : (unsigned)(one >> 32);
  for (int kb0 = 0; kb0 < KB; kb0 += 32) {
    const uint2 w = words_l[kb0 * 16 + lane];
    if (kb0 + c < KB && tile * 32 < N) {
      need[(tile * KB + kb0 + c) * wstride] = w.x;
      faint[(tile * KB + kb0 + c) * wstride] = w.y | (w.x & own);
    }
  }
  // The workgroup's listed rows: one atomic for all (one per wave, at N=400K
  // K=300 D=50 where most waves have some, serialised on the counter: 110 us for the
  // kernel, 48 us this way).
  int* cnt_l = reinterpret_cast<int*>(lds_raw);   // the first stage's operands have been used
  lds_barrier();
  if (lane == 0) cnt_l[wave] = __builtin_popcountll(many);
  lds_barrier();
  int before = 0, total = 0;
#pragma unroll
  for (int v = 0; v < kScreenWaves; ++v) {
    const int n = cnt_l[v];
    before += v < wave ? n : 0;
    total += n;
  }
  if (total == 0) return;
  if (tid == 0) cnt_l[kScreenWaves] = (int)atomicAdd(reinterpret_cast<unsigned*>(list), (unsigned)total);
  lds_barrier();
  const int pos = cnt_l[kScreenWaves] + before +
                  (int)__builtin_amdgcn_mbcnt_hi((unsigned)(many >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)many, 0u));
  if ((many >> lane) & 1) list[kListBase + pos] = (int)row;
}

}  // namespace
}  // namespace fgmm
