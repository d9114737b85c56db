// The experts' prompt GEMMs on 256-row units: two 128-row tiles of one expert (moe.hip lays them out) by 256 weight rows a workgroup, in
// the two-group schedule of gemm_pingpong.hip — eight waves, two a SIMD, which swap roles every barrier interval: one runs a cluster of 16
// MFMAs, its partner reads the fragments of its own next cluster and asks for two pieces of a later K-tile. See there for the order of
// the stream and why a slot is free when it is refilled. What is different here: both operands are row-major (the step's rows, gathered
// through the plan, and the experts' weights as the weight streams of decode steps read them), so a weight half-tile is 128 rows of
// 128 bytes with the same swizzle as the rows' half-tiles; the units are found from the plan on the device; and an expert's last,
// odd tile runs as 128 rows by 256 weight rows, without the empty half:
//   two phases a K-tile, q0: A0 x B0, q1: A0 x B1; three K-tiles of three half-tiles in LDS (144 KiB). q0 of K-tile t asks for A0 and B0
//   of t + 2, q1 for its B1, into the slots that K-tile t - 1 was read from two phases before; at q1 a wave waits until only
//   the four pieces it asked for in q0 may be on their way, so all of t + 1 has landed.
// 1900 tokens, 2 of 8 experts of 3584, width 4096, against the ring of single tiles: gate and up 343 -> 242 us (0.92 PFLOP/s), down 151 -> 109
// (1.02); 4096 tokens 670 -> 490, 353 -> 257. With weights that stay in the last-level cache 222 and 94: what is left to the 1.4 PFLOP/s of
// packed weights is the weights' way from memory, a second round that is three quarters full, and the activation (8 us a round).
// KIND 0: down; 1: gate and up (B0 gate rows, B1 the up rows of the same columns: they meet in registers); 2: up alone (relu squared).
#include <algorithm>
#include "common.h"
#include "expert_act.h"
#include "launch.h"
#include "pingpong.h"
#include <type_traits>

namespace dlia {

constexpr int kMPLds = 9 * kPPHalf;

template <int V> using mic = std::integral_constant<int, V>;

// tile: first 128-row tile of the unit; pair: the next tile is the expert's too. Every wave looks for itself; ntile >= 1.
struct MoeUnit { int tile, expert; bool pair; };

// mask of the tiles base .. base + 63 that begin a unit (an expert's tiles lie one behind the other); run: where the run in progress began
__device__ __forceinline__ unsigned long long unit_starts(const int* __restrict__ tiles, int ntile, int base, int lane, int& run) {
  const int i = base + lane;
  const int e = i < ntile ? tiles[1 + i] : -1, before = i > 0 && i < ntile ? tiles[i] : -1;
  const unsigned long long first = __ballot(i < ntile && e != before), upto = first & (~0ull >> (63 - lane));
  const int at = upto ? base + 63 - __clzll((long long)upto) : run;
  run = first ? base + 63 - __clzll((long long)first) : run;
  return __ballot(i < ntile && ((i - at) & 1) == 0);
}
__device__ __forceinline__ int count_units(const int* __restrict__ tiles, int ntile, int lane) {
  int n = 0, run = 0;
  for (int base = 0; base < ntile; base += 64) n += __popcll(unit_starts(tiles, ntile, base, lane, run));
  return n;
}
__device__ __forceinline__ MoeUnit find_unit(const int* __restrict__ tiles, int ntile, int lane, int unit) {
  int run = 0, tile = 0;
  for (int base = 0; base < ntile; base += 64) {
    const unsigned long long m = unit_starts(tiles, ntile, base, lane, run);
    const int n = __popcll(m);
    if (unit < n) {
      tile = base + __ffsll((long long)__ballot((m >> lane & 1ull) && __popcll(m & ((1ull << lane) - 1)) == unit)) - 1;
      break;
    }
    unit -= n;
  }
  tile = __builtin_amdgcn_readfirstlane(tile);
  const int e = __builtin_amdgcn_readfirstlane(tiles[1 + tile]);
  return {tile, e, tile + 1 < ntile && __builtin_amdgcn_readfirstlane(tiles[1 + min(tile + 1, ntile - 1)]) == e};
}

template <int KIND>
__global__ __launch_bounds__(kPPThreads, 2) void moe_pingpong_kernel(bf16* __restrict__ act_out, float* __restrict__ y_out,
                                                                     const bf16* __restrict__ a, const bf16* __restrict__ w0,
                                                                     const bf16* __restrict__ w1, const int* __restrict__ tiles,
                                                                     const int* __restrict__ row_tok, int N, int K, long lda, long ldo,
                                                                     float limit, const float* __restrict__ row_w) {
  constexpr bool UP = KIND >= 1, GLU = KIND == 1;
  constexpr int BM = 128, BO = GLU ? 128 : 256;                 // rows of a plan tile; output columns of the workgroup
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, quad = lane >> 4, wr = wave >> 2, wc = wave & 3;
  const int ncol = (N + BO - 1) / BO, ntile = tiles[0];
  if (ntile <= 0) return;
  const int units = __builtin_amdgcn_readfirstlane(count_units(tiles, ntile, lane));
  if ((int)blockIdx.x >= ncol * units) return;
  // every XCD takes a run of the work of its own: two units (mostly of one expert) by one column block after the other
  const int item = xcd_remap(blockIdx.x, ncol * units), band = item / (2 * ncol), high = min(2, units - band * 2);
  const MoeUnit u = find_unit(tiles, ntile, lane, band * 2 + (item - band * 2 * ncol) % high);
  const int cblk = (item - band * 2 * ncol) / high;
  const int n0 = cblk * BO;          // first output column of the workgroup
  const int n = K / 64;                                         // K-tiles
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  // (Every workgroup walks K from its start, as the ring does: begun an eighth further on each XCD, for the memory channels' sake, it took 0 to 2 %
  // less, and a row's bits depended on the step's other rows.)

  // ---- the pieces this wave brings in: rows 16 wave + 8 e + lane / 8 of every half-tile, 16-byte slot XOR-ed with (row / 2) % 8 ----
  // Nothing is masked: a row without a token reads token 0 or its own stale row, a weight row beyond N reads row 0, and neither
  // reaches a result that is kept. (The second piece of a pair is asked for with offset:1024.)
  const char* asrc[2][2];
  const char* bsrc[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int r = 16 * wave + 8 * e + (lane >> 3), slot = (lane & 7) ^ ((r >> 1) & 7);
      const long grow = (long)(u.tile + (u.pair ? h : 0)) * BM + r;
      long arow = grow;
      if constexpr (UP) arow = max(row_tok[grow], 0);
      asrc[h][e] = reinterpret_cast<const char*>(a + arow * lda) + slot * 16 - e * 1024;
      const int col = n0 + (GLU ? 0 : h * 128) + r;
      bsrc[h][e] = reinterpret_cast<const char*>((GLU && h ? w1 : w0) + ((long)u.expert * N + (col < N ? col : 0)) * K) + slot * 16 - e * 1024;
    }
  // half 0 / 1 of the rows (WHICH 0) or of the weights (1), K-tile c, to LDS offset `at`
  auto issue = [&](auto which_c, auto half_c, int c, int at) {
    constexpr int which = decltype(which_c)::value, h = decltype(half_c)::value;
    const long off = (long)min(c, n - 1) * 128;
    const char* const (&s)[2] = which ? bsrc[h] : asrc[h];
    pp_dma_pair(s[0] + off, s[1] + off, lds0 + at + wave * 2048);
  };

  f32x4 acc[2][2][4][2];                         // [row half][column half][16 rows][16 columns]
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[p][q][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 af[4][2], b0[2][2], b1[2][2];
  const int sw = (l15 >> 1) & 7;
  const int xoff = (wr * 64 + l15) * 128, boff = (wc * 32 + l15) * 128;
  const int s0 = (quad ^ sw) << 4, s1 = ((4 + quad) ^ sw) << 4;
  auto read_a = [&](int at) {
    const char* base = smem + at + xoff;
#pragma unroll
    for (int i = 0; i < 4; ++i) { af[i][0] = ld16(base + i * 2048 + s0); af[i][1] = ld16(base + i * 2048 + s1); }
  };
  auto read_b = [&](int at, u32x4 (&bf)[2][2]) {
    const char* base = smem + at + boff;
#pragma unroll
    for (int j = 0; j < 2; ++j) { bf[j][0] = ld16(base + j * 2048 + s0); bf[j][1] = ld16(base + j * 2048 + s1); }
  };
  auto cluster = [&](f32x4 (&c)[4][2], const u32x4 (&bf)[2][2]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) c[i][j] = mfma16(bf[j][kk], af[i][kk], c[i][j]);
    __builtin_amdgcn_s_setprio(0);
  };

  if (u.pair) {
    // K-tile buffer `par` (compile time): A0 B0 B1 A1, 64 KiB
    auto phase = [&](auto q_c, int t, auto par_c) {
      constexpr int q = decltype(q_c)::value, here = decltype(par_c)::value * 4 * kPPHalf, there = 4 * kPPHalf - here;
      if constexpr (q == 3) pp_wait_vm<2>();     // my pieces of K-tile t + 1 have landed (A0 of t + 2 may be on its way)
      if constexpr (q == 0) { read_b(here + kPPHalf, b0); __builtin_amdgcn_sched_barrier(0); read_a(here); }
      if constexpr (q == 1) read_b(here + 2 * kPPHalf, b1);
      if constexpr (q == 2) read_a(here + 3 * kPPHalf);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (q == 0) issue(mic<1>{}, mic<1>{}, t + 1, there + 2 * kPPHalf);
      if constexpr (q == 1) issue(mic<0>{}, mic<1>{}, t + 1, there + 3 * kPPHalf);
      if constexpr (q == 2) issue(mic<0>{}, mic<0>{}, t + 2, here);
      if constexpr (q == 3) issue(mic<1>{}, mic<0>{}, t + 2, here + kPPHalf);
      pp_barrier();
      if constexpr (q == 0) cluster(acc[0][0], b0);
      if constexpr (q == 1) cluster(acc[0][1], b1);
      if constexpr (q == 2) cluster(acc[1][1], b1);
      if constexpr (q == 3) cluster(acc[1][0], b0);
      pp_barrier();
    };
    issue(mic<0>{}, mic<0>{}, 0, 0); issue(mic<1>{}, mic<0>{}, 0, kPPHalf); issue(mic<1>{}, mic<1>{}, 0, 2 * kPPHalf); issue(mic<0>{}, mic<1>{}, 0, 3 * kPPHalf);
    issue(mic<0>{}, mic<0>{}, 1, 4 * kPPHalf); issue(mic<1>{}, mic<0>{}, 1, 5 * kPPHalf);
    pp_wait_vm<4>();                             // K-tile 0 has landed (my pieces)
    pp_barrier();                                // ... and everyone's
    if (wr == 1) pp_barrier();                   // waves 4-7 run one interval behind
    for (int t = 0; t < n; t += 2) {
      phase(mic<0>{}, t, mic<0>{}); phase(mic<1>{}, t, mic<0>{}); phase(mic<2>{}, t, mic<0>{}); phase(mic<3>{}, t, mic<0>{});
      if (t + 1 < n) { phase(mic<0>{}, t + 1, mic<1>{}); phase(mic<1>{}, t + 1, mic<1>{}); phase(mic<2>{}, t + 1, mic<1>{}); phase(mic<3>{}, t + 1, mic<1>{}); }
    }
  } else {
    // K-tile buffer `buf` of three: A0 B0 B1, 48 KiB
    auto phase = [&](auto q_c, int t, auto buf_c) {
      constexpr int q = decltype(q_c)::value, buf = decltype(buf_c)::value, here = buf * 3 * kPPHalf, there = (buf + 2) % 3 * 3 * kPPHalf;
      if constexpr (q == 1) pp_wait_vm<4>();     // all of K-tile t + 1 has landed
      if constexpr (q == 0) { read_b(here + kPPHalf, b0); __builtin_amdgcn_sched_barrier(0); read_a(here); }
      else read_b(here + 2 * kPPHalf, b1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (q == 0) { issue(mic<0>{}, mic<0>{}, t + 2, there); issue(mic<1>{}, mic<0>{}, t + 2, there + kPPHalf); }
      else issue(mic<1>{}, mic<1>{}, t + 2, there + 2 * kPPHalf);
      pp_barrier();
      if constexpr (q == 0) cluster(acc[0][0], b0);
      else cluster(acc[0][1], b1);
      pp_barrier();
    };
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      issue(mic<0>{}, mic<0>{}, c, c * 3 * kPPHalf); issue(mic<1>{}, mic<0>{}, c, (c * 3 + 1) * kPPHalf); issue(mic<1>{}, mic<1>{}, c, (c * 3 + 2) * kPPHalf);
    }
    pp_wait_vm<6>();
    pp_barrier();
    if (wr == 1) pp_barrier();
    for (int t = 0; t < n; t += 3) {
      phase(mic<0>{}, t, mic<0>{}); phase(mic<1>{}, t, mic<0>{});
      if (t + 1 < n) { phase(mic<0>{}, t + 1, mic<1>{}); phase(mic<1>{}, t + 1, mic<1>{}); }
      if (t + 2 < n) { phase(mic<0>{}, t + 2, mic<2>{}); phase(mic<1>{}, t + 2, mic<2>{}); }
    }
  }
  if (wr == 0) pp_barrier();                     // the barrier waves 4-7 took at the start
  pp_wait_vm<0>();                               // every piece has landed: the area is free behind the next barrier

  const long row0 = (long)u.tile * BM;
  const int rows = u.pair ? 2 * BM : BM;
  if constexpr (UP) {
    // activations leave through LDS as 16-byte pieces of whole rows; rows and columns that do not come in such pieces one by one
    constexpr int LDO = BO + 8;
    bf16* o = reinterpret_cast<bf16*>(smem);
    __syncthreads();
#pragma unroll
    for (int hm = 0; hm < 2; ++hm)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (hm && !u.pair) continue;
        const int row = hm * 128 + wr * 64 + i * 16 + l15;
        const float rw = row_w && row_tok[row0 + row] >= 0 ? row_w[row0 + row] : 1.f;      // (padding rows have no weight)
#pragma unroll
        for (int hn = 0; hn < (GLU ? 1 : 2); ++hn)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
              v[r] = GLU ? expert_act(acc[hm][0][i][j][r] * rw, acc[hm][1][i][j][r] * rw, limit) : relu2(acc[hm][hn][i][j][r] * rw);
            *reinterpret_cast<u32x2*>(o + row * LDO + hn * 128 + wc * 32 + j * 16 + quad * 4) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
          }
      }
    __syncthreads();
    const bool wide = N % 8 == 0 && ldo % 8 == 0 && (uintptr_t)act_out % 16 == 0;
    for (int p = tid; p < rows * (BO / 8); p += kPPThreads) {
      const int row = p / (BO / 8), c8 = (p % (BO / 8)) * 8, col = n0 + c8;
      bf16* to = act_out + (row0 + row) * ldo + col;
      if (wide) { if (col < N) st16(to, ld16(o + row * LDO + c8)); }
      else for (int j = 0; j < 8 && col + j < N; ++j) to[j] = o[row * LDO + c8 + j];
    }
  } else {
    const bool wide = N % 4 == 0 && ldo % 4 == 0 && (uintptr_t)y_out % 16 == 0;
#pragma unroll
    for (int hm = 0; hm < 2; ++hm)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (hm && !u.pair) continue;
        float* to = y_out + (row0 + hm * 128 + wr * 64 + i * 16 + l15) * ldo;
#pragma unroll
        for (int hn = 0; hn < 2; ++hn)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int col = n0 + hn * 128 + wc * 32 + j * 16 + quad * 4;
            const f32x4 v = acc[hm][hn][i][j];
            if (wide) { if (col < N) *reinterpret_cast<f32x4*>(to + col) = v; }
            else
              for (int r = 0; r < 4; ++r)
                if (col + r < N) to[col + r] = v[r];
          }
      }
  }
}

}  // namespace dlia

template <int KIND>
static void launch_moe_pingpong(void* act, float* y, const void* a, const void* w0, const void* w1, const int* tiles, const int* row_tok,
                                int max_tiles, int experts, int N, int K, long lda, long ldo, float limit, const float* row_w, hipStream_t stream) {
  static const bool once = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dlia::moe_pingpong_kernel<KIND>), hipFuncAttributeMaxDynamicSharedMemorySize, dlia::kMPLds);
    return true;
  }();
  (void)once;
  // (units at most: every expert has one that is not full; how many there are is known on the device alone, a workgroup without one ends)
  const int units = std::min(max_tiles, (max_tiles + experts + 1) / 2), cols = KIND == 1 ? 128 : 256;
  hipLaunchKernelGGL(dlia::moe_pingpong_kernel<KIND>, dim3((N + cols - 1) / cols * units), dim3(dlia::kPPThreads), dlia::kMPLds, stream,
                     (dlia::bf16*)act, y, (const dlia::bf16*)a, (const dlia::bf16*)w0, (const dlia::bf16*)w1, tiles, row_tok, N, K, lda, ldo, limit, row_w);
}

// Whether a step's 128-row tiles run in pairs here (cols: weight rows of the GEMM, gate and up together): by the rounds over the 256 CUs that
// about max_tiles - experts / 2 - 2 tiles make as they are (256 weight rows, or 128 at 0.62 of the price) and as pairs, an expert's odd tile
// a unit of its own. A round of pairs costs 1.45 of one of single tiles, also where it is not full. 58 GEMMs of 614 to 3669 tokens, 4 to 64 experts,
// K 512 to 4096: 3974 us as single tiles, 3713 all in pairs, 3411 by this rule, 3372 with the better one of each; 2014 tokens, 2 of 16, 4096 x 512
// and 3428, 2 of 32, 1024 x 1792, both down, are taken the wrong way (41 -> 44, 47 -> 53: the rounds depend on how even the routing is).
extern "C" int dlia_moe_pairs(int max_tiles, int experts, int cols, int K) {
  if (K % 64 != 0) return 0;
  const int tiles = std::max(max_tiles - experts / 2 - 2, experts);
  const double units = std::max((double)experts, tiles / 2.0 + experts / 4.0);
  const int c256 = (cols + 255) / 256, c128 = (cols + 127) / 128;
  const double single = std::min((double)((tiles * c256 + 255) / 256), 0.62 * ((tiles * c128 + 255) / 256));
  return 1.45 * std::max(1.0, units * c256 / 256) < single;
}

extern "C" void dlia_moe_pingpong(int kind, void* act, float* y, const void* a, const void* w0, const void* w1, const int* tiles,
                                  const int* row_tok, int max_tiles, int experts, int N, int K, long lda, long ldo, float limit,
                                  const float* row_w, hipStream_t stream) {
  if (kind == 0) launch_moe_pingpong<0>(act, y, a, w0, w1, tiles, row_tok, max_tiles, experts, N, K, lda, ldo, limit, row_w, stream);
  else if (kind == 1) launch_moe_pingpong<1>(act, y, a, w0, w1, tiles, row_tok, max_tiles, experts, N, K, lda, ldo, limit, row_w, stream);
  else launch_moe_pingpong<2>(act, y, a, w0, w1, tiles, row_tok, max_tiles, experts, N, K, lda, ldo, limit, row_w, stream);
}
