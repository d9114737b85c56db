// Routed feed-forward (mixture of experts) without a host round trip: routing, a plan that sorts the step's (token, choice)
// pairs by expert into 32-row tiles, the experts' two GEMMs over those tiles, and the weighted sum per token.
//
//   moe_route    one thread per token. Scores are sigmoids of the fp32 router logits, or their softmax over all router outputs.
//                The choice goes by score + correction[e] when a correction is given. Experts are split into `groups`
//                contiguous blocks of equal size; a block is ranked by its best `group_rank` (1 or 2) choice scores added up;
//                the `keep` best blocks stay; the `top` best experts of those are chosen (equal scores: the lower index),
//                weighted score / (sum + 1e-20) * scale, or score * scale without the division.
//   moe_route_plan   routing and plan together; ONE launch for steps of up to 256 tokens.
//   moe_plan     one workgroup. Pairs whose choice is not a real expert (an identity expert: index >= E) get row -1 and no
//                place in a tile. Counts the pairs per expert, lays the experts' row ranges out one after the other, each
//                padded to whole 32-row tiles, and writes for every padded row its token (or -1), for every pair its row,
//                for every tile its expert; tiles[0] holds the number of tiles. Rows of one expert are in no fixed order:
//                every row is computed on its own, so the order does not reach the results.
//   moe_table_plan  the same plan for every routed layer of a stack whose experts go by the token's id, in ONE launch ahead of the
//                layers: workgroup l reads layer l's table [vocab, top] at the step's ids and lays out its pairs. Where the
//                layers' parts lie in the shared buffers comes from a descriptor per layer (kPlanDesc numbers: table offset, top,
//                experts, offset of the tile list, of the row list, of the pair list, whether 128-row tiles may be used).
//   glu_act      the activation of one expert that runs for every token, from gate | up (| one more number, whose sigmoid
//                multiplies the row) in fp32
//   moe_up       grid (column blocks, tiles): act[row, f] = g s(1.702 g) (u + 1), g = min(x . Wg[e][f], limit),
//                u = clamp(x . Wu[e][f], -limit, limit), x the row's token; with limit <= 0 the plain silu(g) * u.
//                Gate and up accumulate over the same A fragments. Experts without a gate: act = relu(x . Wu[e][f])^2. With
//                weights per row (the plan lays them out) x is the token times its weight: the products are multiplied by it.
//   moe_down     y[row, c] = act[row] . Wd[e][c] in fp32.
//   moe_combine  out[t, :] = sum over the token's choices of weight * y[row, :], in the order of the choices (fp32); a choice
//                without a row (an identity expert) contributes weight * x[t, :].
// Operands are bf16 (16x16x32 MFMA) or fp32 (16x16x4 MFMA, true 32-bit): fragments read straight from the K-contiguous rows in steps
// with few rows, through an LDS ring in prompt steps (128-row tiles; in pairs of an expert's tiles where that fills the chip, moe_pingpong.hip).
#include "common.h"
#include "expert_act.h"
#include "frag.h"
#include <type_traits>
#include <algorithm>
#include "units.h"
#include "launch.h"

namespace dlia {

constexpr int kMoeMaxExperts = 256;
constexpr int kMoeRows = 32;           // rows of a plan tile (steps with few rows), kMoeBigRows for the LDS-tiled kernel
constexpr int kMoeBigRows = 128;

__device__ __forceinline__ void route_token(int t, int* __restrict__ sel, float* __restrict__ wts, const float* __restrict__ logits, long ld,
                                            int E, int top, int groups, int keep, float scale, const float* __restrict__ corr, int softmax,
                                            int group_rank, int renorm) {
  const float* z = logits + (long)t * ld;
  const int per = E / groups;
  float zmax = 0.f, zinv = 1.f;
  if (softmax) {
    zmax = -INFINITY;
    for (int e = 0; e < E; ++e) zmax = fmaxf(zmax, z[e]);
    float sum = 0.f;
    for (int e = 0; e < E; ++e) sum += expf(z[e] - zmax);
    zinv = 1.f / sum;
  }
  auto score = [&](int e) { return softmax ? expf(z[e] - zmax) * zinv : 1.f / (1.f + expf(-z[e])); };
  auto choice = [&](int e) { return corr ? score(e) + corr[e] : score(e); };
  // the groups that stay: `keep` times the best group not yet taken
  unsigned long long gmask[4] = {0ull, 0ull, 0ull, 0ull};
  if (keep >= groups) gmask[0] = gmask[1] = gmask[2] = gmask[3] = ~0ull;      // (all of them: nothing to rank)
  for (int r = 0; r < (keep >= groups ? 0 : keep); ++r) {
    int best = -1; float bs = -INFINITY;
    for (int g = 0; g < groups; ++g) {
      if (gmask[g >> 6] >> (g & 63) & 1ull) continue;
      float a = -INFINITY, b = -INFINITY;             // the block's best two choice scores
      for (int e = g * per; e < (g + 1) * per; ++e) {
        const float s = choice(e);
        if (s > a) { b = a; a = s; } else if (s > b) b = s;
      }
      const float gs = a + (group_rank >= 2 && b > -INFINITY ? b : 0.f);
      if (best < 0 || gs > bs) { bs = gs; best = g; }
    }
    if (best >= 0) gmask[best >> 6] |= 1ull << (best & 63);
  }
  unsigned long long emask[4] = {0ull, 0ull, 0ull, 0ull};
  float total = 0.f;
  for (int r = 0; r < top; ++r) {
    int best = -1; float bs = -INFINITY;
    for (int e = 0; e < E; ++e) {
      const int g = e / per;
      if (!(gmask[g >> 6] >> (g & 63) & 1ull) || (emask[e >> 6] >> (e & 63) & 1ull)) continue;
      const float s = choice(e);
      if (best < 0 || s > bs) { bs = s; best = e; }
    }
    if (best < 0) best = 0;
    emask[best >> 6] |= 1ull << (best & 63);
    const float w = score(best);
    sel[(long)t * top + r] = best;
    wts[(long)t * top + r] = w;
    total += w;
  }
  const float inv = renorm ? scale / (total + 1e-20f) : scale;
  for (int r = 0; r < top; ++r) wts[(long)t * top + r] *= inv;
}

// The same for up to 32 experts in up to 8 groups: the scores, formed once, stay in LDS (a column a thread, `ks` apart), what may be chosen is one
// 32-bit mask, nothing is divided by the group's size. Same choices and weights to the last bit. (64 tokens of 16 experts in 4 groups,
// with the plan: 20.2 -> 10.4 us, 300 of 16 in 2 27 -> 13; the general form evaluates exponentials and divides at every comparison.)
constexpr int kFewExperts = 32, kFewGroups = 8;

__device__ __forceinline__ void route_few(int t, int* __restrict__ sel, float* __restrict__ wts, const float* __restrict__ logits, long ld, int E,
                                          int top, int groups, int keep, float scale, const float* __restrict__ corr, int softmax, int group_rank,
                                          int renorm, float* kept, float* gscore, int ks) {
  const float* z = logits + (long)t * ld;
  const int per = E / groups;
#pragma unroll 8
  for (int e = 0; e < E; ++e) kept[e * ks] = z[e];
  float zmax = 0.f, zinv = 1.f;
  if (softmax) {
    zmax = -INFINITY;
    for (int e = 0; e < E; ++e) zmax = fmaxf(zmax, kept[e * ks]);
    float sum = 0.f;
#pragma unroll 4
    for (int e = 0; e < E; ++e) { const float x = expf(kept[e * ks] - zmax); kept[e * ks] = x; sum += x; }
    zinv = 1.f / sum;
#pragma unroll 4
    for (int e = 0; e < E; ++e) kept[e * ks] *= zinv;
  } else {
#pragma unroll 4
    for (int e = 0; e < E; ++e) kept[e * ks] = 1.f / (1.f + expf(-kept[e * ks]));
  }
  auto choice = [&](int e) { return corr ? kept[e * ks] + corr[e] : kept[e * ks]; };
  unsigned open = ~0u;
  if (keep < groups) {
    for (int g = 0; g < groups; ++g) {
      float a = -INFINITY, b = -INFINITY;             // the block's best two choice scores
      for (int e = g * per; e < (g + 1) * per; ++e) {
        const float s = choice(e);
        if (s > a) { b = a; a = s; } else if (s > b) b = s;
      }
      gscore[g * ks] = a + (group_rank >= 2 && b > -INFINITY ? b : 0.f);
    }
    unsigned taken = 0u;
    open = 0u;
    for (int r = 0; r < keep; ++r) {
      int best = -1; float bs = -INFINITY;
      for (int g = 0; g < groups; ++g) {
        if (taken >> g & 1u) continue;
        const float gs = gscore[g * ks];
        if (best < 0 || gs > bs) { bs = gs; best = g; }
      }
      if (best >= 0) { taken |= 1u << best; open |= ((1u << per) - 1u) << (best * per); }       // (per < 32: more than one group)
    }
  }
  float total = 0.f;
  for (int r = 0; r < top; ++r) {
    int best = -1; float bs = -INFINITY;
    for (int e = 0; e < E; ++e) {
      const float s = choice(e);
      if ((open >> e & 1u) && (best < 0 || s > bs)) { bs = s; best = e; }
    }
    if (best < 0) best = 0;
    open &= ~(1u << best);
    const float w = kept[best * ks];
    sel[(long)t * top + r] = best;
    wts[(long)t * top + r] = w;
    total += w;
  }
  const float inv = renorm ? scale / (total + 1e-20f) : scale;
  for (int r = 0; r < top; ++r) wts[(long)t * top + r] *= inv;
}

__global__ __launch_bounds__(64) void moe_route_kernel(int* __restrict__ sel, float* __restrict__ wts,
                                                       const float* __restrict__ logits, long ld, int T, int E, int top,
                                                       int groups, int keep, float scale, const float* __restrict__ corr,
                                                       int softmax, int group_rank, int renorm) {
  __shared__ float kept[kFewExperts * 64], gscore[kFewGroups * 64];
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t >= T) return;
  if (E <= kFewExperts && groups <= kFewGroups)
    route_few(t, sel, wts, logits, ld, E, top, groups, keep, scale, corr, softmax, group_rank, renorm, kept + threadIdx.x, gscore + threadIdx.x, 64);
  else
    route_token(t, sel, wts, logits, ld, E, top, groups, keep, scale, corr, softmax, group_rank, renorm);
}

// Lays out the pairs of one layer. expert(i): the expert of pair i (i / top is its token). 1024 threads.
// tiles: [0] number of tiles, [1 + i] expert of tile i. row_tok [max_rows], pair_row [pairs].
template <typename Sel>
__device__ __forceinline__ void plan_pairs(int* __restrict__ tiles, int* __restrict__ row_tok, int* __restrict__ pair_row, int pairs,
                                           int top, int E, int max_rows, int tile_rows, int* count, int* start, int* fill, int* ntiles,
                                           Sel expert, const float* __restrict__ wts = nullptr, float* __restrict__ row_w = nullptr) {
  for (int e = threadIdx.x; e < E; e += 1024) { count[e] = 0; fill[e] = 0; }
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += 1024) {
    const int e = expert(i);
    if (e < E) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, nt = 0;
    for (int e = 0; e < E; ++e) {
      start[e] = at;
      const int n = (count[e] + tile_rows - 1) / tile_rows;
      for (int i = 0; i < n; ++i) tiles[1 + nt + i] = e;
      nt += n; at += n * tile_rows;
    }
    tiles[0] = nt;
    *ntiles = nt;
  }
  __syncthreads();
  const int used = *ntiles * tile_rows;
  for (int i = threadIdx.x; i < max_rows; i += 1024) row_tok[i] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += 1024) {
    const int e = expert(i);
    if (e >= E) { pair_row[i] = -1; continue; }                      // (an identity expert: no row)
    const int r = start[e] + atomicAdd(&fill[e], 1);
    if (r < max_rows && r < used) { row_tok[r] = i / top; pair_row[i] = r; if (row_w) row_w[r] = wts[i]; }
  }
}

__global__ __launch_bounds__(1024) void moe_plan_kernel(int* __restrict__ tiles, int* __restrict__ row_tok,
                                                        int* __restrict__ pair_row, const int* __restrict__ sel, int pairs,
                                                        int top, int E, int max_rows, int tile_rows, const float* __restrict__ wts,
                                                        float* __restrict__ row_w) {
  __shared__ int count[kMoeMaxExperts], start[kMoeMaxExperts], fill[kMoeMaxExperts];
  __shared__ int ntiles;
  plan_pairs(tiles, row_tok, pair_row, pairs, top, E, max_rows, tile_rows, count, start, fill, &ntiles, [&](int i) { return sel[i]; }, wts, row_w);
}

// Routing and plan of a step with few tokens in one launch (one workgroup, a thread per token).
__global__ __launch_bounds__(1024) void moe_route_plan_kernel(int* __restrict__ sel, float* __restrict__ wts, const float* __restrict__ logits,
                                                              long ld, int T, int E, int top, int groups, int keep, float scale,
                                                              const float* __restrict__ corr, int softmax, int group_rank, int renorm,
                                                              int* __restrict__ tiles, int* __restrict__ row_tok, int* __restrict__ pair_row,
                                                              int experts, int max_rows, int tile_rows, float* __restrict__ row_w) {
  __shared__ int count[kMoeMaxExperts], start[kMoeMaxExperts], fill[kMoeMaxExperts];
  __shared__ int ntiles;
  __shared__ float kept[kFewExperts * 256], gscore[kFewGroups * 256];
  const bool few = E <= kFewExperts && groups <= kFewGroups && T <= 256;
  for (int t = threadIdx.x; t < T; t += 1024) {
    if (few) route_few(t, sel, wts, logits, ld, E, top, groups, keep, scale, corr, softmax, group_rank, renorm, kept + t, gscore + t, 256);
    else route_token(t, sel, wts, logits, ld, E, top, groups, keep, scale, corr, softmax, group_rank, renorm);
  }
  __threadfence_block();
  __syncthreads();
  plan_pairs(tiles, row_tok, pair_row, T * top, top, experts, max_rows, tile_rows, count, start, fill, &ntiles,
             [&](int i) { return *(volatile const int*)(sel + i); }, wts, row_w);
}

constexpr int kPlanDesc = 8;
constexpr int kTableMaxExperts = 1024;

__global__ __launch_bounds__(1024) void moe_table_plan_kernel(int* __restrict__ tiles, int* __restrict__ row_tok,
                                                              int* __restrict__ pair_row, const int* __restrict__ tables,
                                                              const int* __restrict__ ids, const int* __restrict__ desc, int T, int vocab,
                                                              int big_pairs) {
  __shared__ int count[kTableMaxExperts], start[kTableMaxExperts], fill[kTableMaxExperts];
  __shared__ int ntiles;
  const int* d = desc + blockIdx.x * kPlanDesc;
  const int* table = tables + d[0];
  const int top = d[1], E = d[2], pairs = T * top;
  const int tile_rows = d[6] && pairs >= big_pairs ? kMoeBigRows : kMoeRows;
  plan_pairs(tiles + d[3], row_tok + d[4], pair_row + d[5], pairs, top, E, ((pairs + tile_rows - 1) / tile_rows + E) * tile_rows, tile_rows,
             count, start, fill, &ntiles, [&](int i) {
               int id = ids[i / top];
               id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);     // (as the embedding does: never fault on a bad id)
               const int e = table[(long)id * top + i % top];
               return e < 0 ? 0 : e;
             });
}

// V entries of a row per thread (1900 rows of 3584, bf16 out: 18.1 us with one, 11 with four). LIMITED at compile time: with both forms of the activation in
// sight the compiler evaluates both and selects (256 rows of 8192, one entry a thread, 5.2 -> 6.5 us).
template <typename OT, int V, bool LIMITED>
__global__ __launch_bounds__(256) void glu_act_kernel(OT* __restrict__ act, long lda, const float* __restrict__ z, long ldz, int F,
                                                      float limit, int gated) {
  const long m = blockIdx.y;
  const int c = (blockIdx.x * 256 + threadIdx.x) * V;
  if (c >= F) return;
  const float* zr = z + m * ldz;
  const Unit<V> g = ldu<V>(zr + c), u = ldu<V>(zr + F + c);
  Unit<V> o;
#pragma unroll
  for (int e = 0; e < V; ++e) o.v[e] = LIMITED ? expert_act_limited(g.v[e], u.v[e], limit) : expert_act_free(g.v[e], u.v[e]);
  if (gated) {
    const float all = 1.f / (1.f + expf(-zr[2 * F]));
#pragma unroll
    for (int e = 0; e < V; ++e) o.v[e] *= all;
  }
  stu<V>(act + m * lda + c, o);
}

// Row tiles of the plan: 32 rows. Where experts have several of them and the blocks fill the chip (fp32 prompts above all) a workgroup of four waves covers one
// row tile by 128 (up) or 256 (down) output columns; a wave holds both 16-row halves of the tile against its 32 (64) columns, so
// every fragment it loads feeds two or more MFMAs, and the fragments of the next k-step are on their way while the current ones
// are multiplied.
constexpr int kMoeTile = kMoeRows;

// FAST: K in whole pieces, aligned rows; then no load is masked (a row without a token reads token 0 or its own stale row, a weight row beyond the last reads row 0:
// neither reaches a result that is kept), because a load under a mask is a branch and a wait of its own. Else: steps beyond K load zeros.
template <bool FAST, typename T>
__device__ __forceinline__ u32x4 step_frag(const T* __restrict__ row, int k, int K, bool valid, int vec_ok) {
  if constexpr (FAST) return ld16(row + k);
  else return load_frag<T>(row, k, K, valid, vec_ok);
}

template <typename T, typename OT, int NJ, bool GLU, bool FAST>
__global__ __launch_bounds__(256) void moe_up_kernel(OT* __restrict__ act, const T* __restrict__ x, const T* __restrict__ wg,
                                                     const T* __restrict__ wu, const int* __restrict__ tiles,
                                                     const int* __restrict__ row_tok, int F, int K, long ldx, long lda,
                                                     float limit, int vec_ok, const float* __restrict__ row_w) {
  constexpr int VEC = 16 / sizeof(T), KS = 4 * VEC;
  const int tile = blockIdx.y;
  if (tile >= tiles[0]) return;
  const int e = tiles[1 + tile];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int f0 = (blockIdx.x * 4 + wave) * 16 * NJ;
  if (f0 >= F) return;
  const T* arow[2]; long wrow[NJ]; bool av[2], wv[NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int tok = row_tok[tile * kMoeTile + i * 16 + r16];
    av[i] = tok >= 0;
    arow[i] = x + (long)(av[i] ? tok : 0) * ldx;
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    wv[j] = f0 + j * 16 + r16 < F;
    wrow[j] = ((long)e * F + (wv[j] ? f0 + j * 16 + r16 : 0)) * K;
  }
  f32x4 ag[2][NJ], au[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) { ag[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; au[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
  struct Frags { u32x4 a[2], g[GLU ? NJ : 1], u[NJ]; };
  auto load = [&](Frags& f, int k0) {
    const int k = k0 + kq * VEC;
#pragma unroll
    for (int i = 0; i < 2; ++i) f.a[i] = step_frag<FAST>(arow[i], k, K, av[i], vec_ok);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if constexpr (GLU) f.g[j] = step_frag<FAST>(wg + wrow[j], k, K, wv[j], vec_ok);
      f.u[j] = step_frag<FAST>(wu + wrow[j], k, K, wv[j], vec_ok);
    }
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if constexpr (GLU) ag[i][j] = mma_frag(T{}, f.a[i], f.g[j], ag[i][j]);
        au[i][j] = mma_frag(T{}, f.a[i], f.u[j], au[i][j]);
      }
  };
  Frags fa, fb;
  load(fa, 0);
  for (int k0 = 0; k0 < K; k0 += 2 * KS) {
    if (k0 + KS < K) load(fb, k0 + KS);
    multiply(fa);
    if (k0 + KS < K) {
      if (k0 + 2 * KS < K) load(fa, k0 + 2 * KS);
      multiply(fb);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = f0 + j * 16 + r16;
      if (col >= F) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = tile * kMoeTile + i * 16 + kq * 4 + r;
        const float rw = row_w && row_tok[row] >= 0 ? row_w[row] : 1.f;      // (padding rows have no weight)
        if constexpr (GLU) act[(long)row * lda + col] = (OT)expert_act(ag[i][j][r] * rw, au[i][j][r] * rw, limit);
        else act[(long)row * lda + col] = (OT)relu2(au[i][j][r] * rw);
      }
    }
}

template <typename T, int NJ, bool FAST>
__global__ __launch_bounds__(256) void moe_down_kernel(float* __restrict__ y, const T* __restrict__ act, const T* __restrict__ wd,
                                                       const int* __restrict__ tiles, const int* __restrict__ row_tok,
                                                       int H, int F, long lda, int vec_ok) {
  constexpr int VEC = 16 / sizeof(T), KS = 4 * VEC;
  const int tile = blockIdx.y;
  if (tile >= tiles[0]) return;
  const int e = tiles[1 + tile];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int c0 = (blockIdx.x * 4 + wave) * 16 * NJ;
  if (c0 >= H) return;
  const T* arow[2]; const T* wrow[NJ]; bool av[2], wv[NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    av[i] = row_tok[tile * kMoeTile + i * 16 + r16] >= 0;
    arow[i] = act + (long)(tile * kMoeTile + i * 16 + r16) * lda;
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    wv[j] = c0 + j * 16 + r16 < H;
    wrow[j] = wd + ((long)e * H + (wv[j] ? c0 + j * 16 + r16 : 0)) * F;
  }
  f32x4 acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Frags { u32x4 a[2], w[NJ]; };
  auto load = [&](Frags& f, int k0) {
    const int k = k0 + kq * VEC;
#pragma unroll
    for (int i = 0; i < 2; ++i) f.a[i] = step_frag<FAST>(arow[i], k, F, av[i], vec_ok);
#pragma unroll
    for (int j = 0; j < NJ; ++j) f.w[j] = step_frag<FAST>(wrow[j], k, F, wv[j], vec_ok);
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = mma_frag(T{}, f.a[i], f.w[j], acc[i][j]);
  };
  Frags fa, fb;
  load(fa, 0);
  for (int k0 = 0; k0 < F; k0 += 2 * KS) {
    if (k0 + KS < F) load(fb, k0 + KS);
    multiply(fa);
    if (k0 + KS < F) {
      if (k0 + 2 * KS < F) load(fa, k0 + 2 * KS);
      multiply(fb);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = c0 + j * 16 + r16;
      if (col >= H) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[(long)(tile * kMoeTile + i * 16 + kq * 4 + r) * H + col] = acc[i][j][r];
    }
}

// Few row tiles an expert (decoding): a stream of the experts' weights, KIND 0: down, 1: gated up, 2: squared-ReLU up. A workgroup
// holds the row tile against 16 NJ columns (of gate and up alike) over ALL of K; its four waves take K in turns, U whole k-steps (a
// cache line or two of every row) at a time with the next piece on its way, and their partial tiles meet in LDS, added in the order
// of the waves. Workgroups are many and short, so the chip stays even, and no half of a tile without a token is loaded or
// multiplied. RT 2: the workgroup of an expert's first, third, ... tile takes the one behind it along. Rows of a power of two of bytes put one k of every row on the same memory channels: workgroups begin at different
// places of K and go round. Two column tiles a wave halve the traffic of the token rows, which at 16 rows an expert equals the
// weights'. (Before: 64 columns of a tile in each workgroup, every wave over all of K with its own columns: 448 or 512 workgroups on
// 256 CUs, all on the same channels.) 8 experts, two a token, gate and up [3584, 4096], down [4096, 3584], bf16: 4 tokens 90 -> 51
// and 75 -> 32 us, 64 tokens (470 and 235 MB) 116 -> 95 and 76 -> 50 us (4.9 and 4.7 TB/s), 160 tokens 216 -> 157 and 148 -> 96.
template <typename T, typename OT, int KIND, bool FAST, int NW, int U, int NJ, int RT = 1>
__global__ __launch_bounds__(64 * NW, RT > 1 ? 2 : 1) void moe_stream_kernel(OT* __restrict__ out, const T* __restrict__ x, const T* __restrict__ w0,
                                                             const T* __restrict__ w1, const int* __restrict__ tiles,
                                                             const int* __restrict__ row_tok, int N, int K, long ldx, long ldo, float limit,
                                                             int vec_ok, const float* __restrict__ row_w) {
  constexpr int VEC = 16 / (int)sizeof(T), KS = 4 * VEC, CH = U * KS, NG = KIND == 1 ? 2 : 1;
  constexpr int HM = 2 * RT;                                       // 16-row halves of RT tiles
  __shared__ f32x4 part[NW][HM][NG * NJ][64];
  const int tile = blockIdx.y;
  if (tile >= tiles[0]) return;
  const int e = tiles[1 + tile];
  int follows = 0;                                                 // RT 2: an expert's tiles two at a time, by the workgroup of the first
  if constexpr (RT > 1) {
    int before = 0;
    while (before < tile && tiles[tile - before] == e) ++before;
    if (before & 1) return;
    follows = tile + 1 < tiles[0] && tiles[2 + tile] == e;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int n0 = blockIdx.x * 16 * NJ;
  const int* rows = row_tok + (long)tile * kMoeTile;
  const T* wr[NG * NJ]; bool wv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    wv[j] = n0 + j * 16 + r16 < N;
    const long wrow = ((long)e * N + (wv[j] ? n0 + j * 16 + r16 : 0)) * K;
    wr[j * NG] = w0 + wrow;
    if constexpr (KIND == 1) wr[j * NG + 1] = w1 + wrow;
  }
  const T* ar[HM]; bool av[HM];
#pragma unroll
  for (int i = 0; i < HM; ++i) {
    const int tok = i < 2 || follows ? rows[i * 16 + r16] : -1;
    av[i] = tok >= 0;
    ar[i] = x + (KIND == 0 ? (long)tile * kMoeTile + i * 16 + r16 : (long)(av[i] ? tok : 0)) * ldx;
  }
  int halves = 1;                                                  // with a token (their rows are filled from the front)
#pragma unroll
  for (int i = 1; i < HM; ++i)
    if (__ballot(av[i]) != 0) halves = i + 1;
  f32x4 acc[HM][NG * NJ];
#pragma unroll
  for (int i = 0; i < HM; ++i)
#pragma unroll
    for (int g = 0; g < NG * NJ; ++g) acc[i][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto run = [&](auto halves) {
    constexpr int MI = decltype(halves)::value;
    struct Frags { u32x4 w[U][NG * NJ], a[U][MI]; };
    auto load = [&](Frags& f, int k0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * KS + kq * VEC;
#pragma unroll
        for (int g = 0; g < NG * NJ; ++g) f.w[u][g] = step_frag<FAST>(wr[g], k, K, wv[g / NG], vec_ok);
#pragma unroll
        for (int i = 0; i < MI; ++i) f.a[u][i] = step_frag<FAST>(ar[i], k, K, av[i], vec_ok);
      }
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int g = 0; g < NG * NJ; ++g) acc[i][g] = mma_frag(T{}, f.a[u][i], f.w[u][g], acc[i][g]);
    };
    // Piece c of the wave's share; each workgroup begins elsewhere in K and goes round. A K of no more pieces than waves stays with
    // one of them: its sums are then formed in the order of the wide blocks, so that for such K (up to 512 in 16 bits, 128 in 32) a row's
    // result does not depend on which of the two its step took; for longer K it may, in the last bits. (Steps of few workgroups alone:
    // there a launch is all there is, 4.5 to 5 us either way.)
    const int total = (K + CH - 1) / CH, turn = total > NW ? (blockIdx.x * 4 + e) % total : 0, step = total > NW ? NW : 1;
    if (wave >= step) return;
    auto at = [&](int c) { const int k = c + turn; return (k >= total ? k - total : k) * CH; };
    Frags fa, fb;
    int c = wave;
    if (c < total) load(fa, at(c));
    for (; c < total; c += 2 * step) {
      if (c + step < total) load(fb, at(c + step));
      multiply(fa);
      if (c + step < total) {
        if (c + 2 * step < total) load(fa, at(c + 2 * step));
        multiply(fb);
      }
    }
  };
  if (halves == 1) run(std::integral_constant<int, 1>{});
  else if (RT == 1 || halves == 2) run(std::integral_constant<int, 2>{});
  else if constexpr (RT > 1) {
    if (halves == 3) run(std::integral_constant<int, 3>{});
    else run(std::integral_constant<int, 4>{});
  }
#pragma unroll
  for (int i = 0; i < HM; ++i)
#pragma unroll
    for (int g = 0; g < NG * NJ; ++g) part[wave][i][g][lane] = acc[i][g];
  __syncthreads();
  const int used = follows ? HM : 2;
  for (int q = wave; q < used * NJ; q += NW) {
    const int i = q % used, j = q / used, col = n0 + j * 16 + r16;
    f32x4 s[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      s[g] = part[0][i][j * NG + g][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) s[g] += part[w][i][j * NG + g][lane];
    }
    if (col >= N) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = i * 16 + kq * 4 + r;
      const long at = ((long)tile * kMoeTile + row) * ldo + col;
      if constexpr (KIND == 0) out[at] = s[0][r];
      else {
        const float rw = row_w && rows[row] >= 0 ? row_w[(long)tile * kMoeTile + row] : 1.f;      // (padding rows have no weight)
        if constexpr (KIND == 1) out[at] = (OT)expert_act(s[0][r] * rw, s[NG - 1][r] * rw, limit);
        else out[at] = (OT)relu2(s[0][r] * rw);
      }
    }
  }
}

// Steps with many rows (prompts): 128-row tiles by BN weight rows (256, or 128), eight waves of 64 rows by BN / 4 weight rows each.
// For the up projection the BN weight rows are BN / 2 gate rows and the up rows of the same columns, a wave holding both, so the
// activation is formed in registers. Operands go through a ring of six LDS stages of 32 K-elements (direct LDS loads: 16 rows of
// 64 bytes a piece, rows gathered through the plan for the up projection), four of them on their way. In step t a wave waits for
// stage t + 1, meets the others, asks for that stage's fragments and the loads of stage t + 5, and multiplies the fragments of
// step t, which it has held since the step before: the matrix cores have work the moment the barrier opens. The 16-byte chunk c
// of row r sits at c ^ (r / 2 % 4), so that 8 rows of a fragment read fall on different banks (the swizzle is applied to the
// address each lane loads FROM).
// 1900 tokens, 2 of 8 experts of 3584, width 4096, before -> now: gate and up 433 -> 344 us, down 216 -> 203 (800 tokens: 264 -> 174,
// 112 -> 86). Before: four waves, operands through registers, two steps ahead. With three stages of 64 K-elements and the fragment
// reads behind the barrier: 361 us, matrix cores busy 42 % of a CU's cycles without a bank conflict; with a branch around a step's
// loads: 360, the compiler then waits for the fragments just asked for. 24 KiB of operands arrive per 512 cycles of matrix work.
// bf16, K a multiple of 32 with 16-byte aligned rows (the caller falls back to the register-tiled kernels otherwise).
// KIND 0: down; 1: gate and up; 2: up alone (the square of relu).
constexpr int kBigStages = 6;

template <int KIND, int BN>
__global__ __launch_bounds__(512) void moe_big_kernel(bf16* __restrict__ act_out, float* __restrict__ y_out, const bf16* __restrict__ a,
                                                      const bf16* __restrict__ w0, const bf16* __restrict__ w1,
                                                      const int* __restrict__ tiles, const int* __restrict__ row_tok, int N, int K,
                                                      long lda, long ldo, float limit, const float* __restrict__ row_w) {
  constexpr bool UP = KIND >= 1, GLU = KIND == 1;
  constexpr int BM = kMoeBigRows, P = (BM + BN) / 128, kStage = (BM + BN) * 64;
  constexpr int MT = 4, NT = BN / 64, BO = GLU ? BN / 2 : BN;   // 16-wide tiles of a wave; output columns of the workgroup
  __shared__ __attribute__((aligned(1024))) char lds[kBigStages * kStage];
  // Every XCD takes a run of the work of its own, four row tiles (mostly of one expert) by one column block after the other: the
  // 32 workgroups it runs at a time share 4 row panels and 8 weight panels in its L2 (counters: half of the pieces missed L2 with
  // the column block as the fastest index of the whole grid).
  const int ncol = (N + BO - 1) / BO, ntile = tiles[0];
  if ((int)blockIdx.x >= ncol * ntile) return;
  const int item = xcd_remap(blockIdx.x, ncol * ntile), band = item / (4 * ncol), high = min(4, ntile - band * 4);
  const int tile = band * 4 + (item - band * 4 * ncol) % high, cblk = (item - band * 4 * ncol) / high;
  const int e = tiles[1 + tile];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int n0 = cblk * BO;                                     // first output column of the workgroup
  // the 1 KiB pieces this wave brings in: piece p of a stage holds its rows 16 p .. 16 p + 15 (the step's rows, then the weights').
  // Nothing is masked: a row without a token reads token 0 or its own stale row, a weight row beyond N reads row 0, and neither
  // reaches a result that is kept.
  const bf16* src[P];
  const int chunk = (lane & 3) ^ ((lane >> 3) & 3);
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int row = (wave * P + q) * 16 + (lane >> 2);
    if (row < BM) {
      const int grow = tile * BM + row;
      if constexpr (UP) { const int tok = row_tok[grow]; src[q] = a + (long)(tok >= 0 ? tok : 0) * lda + chunk * 8; }
      else src[q] = a + (long)grow * lda + chunk * 8;
    } else {
      const int w = row - BM;
      const int wr = n0 + (GLU ? (w < BO ? w : w - BO) : w);
      src[q] = (GLU && w >= BO ? w1 : w0) + ((long)e * N + (wr < N ? wr : 0)) * K + chunk * 8;
    }
  }
  const unsigned lds_base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * P * 1024);
  const int nk = K / 32;
  // (stages are asked for in order: the sources walk along)
  auto fetch = [&](int slot) {
    const void* g[P];
#pragma unroll
    for (int q = 0; q < P; ++q) { g[q] = src[q]; src[q] += 32; }
    lds_dma_run<P>(g, lds_base + slot * kStage);
  };
  // a stage has landed when only the `behind` stages after it are still on their way (own pieces; the barrier makes it everybody's)
  auto meet = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 2) * 64, wn = wave & 3;
  // LDS row of a wave's weight tile j: gate tiles first, then the up tiles of the same columns
  auto wrow = [&](int j) { return GLU ? (j < NT / 2 ? wn * (BO / 4) + j * 16 : BO + wn * (BO / 4) + (j - NT / 2) * 16) : wn * (BN / 4) + j * 16; };
  struct Frags { u32x4 a[MT], w[NT]; };
  const int at = r16 * 64 + ((kq ^ ((r16 >> 1) & 3)) << 4);      // (tiles start at multiples of 16 rows: the swizzle is the lane's own)
  auto read = [&](Frags& f, int slot) {
    const char* st = lds + slot * kStage + at;
#pragma unroll
    for (int i = 0; i < MT; ++i) f.a[i] = ld16(st + (wm + i * 16) * 64);
#pragma unroll
    for (int j = 0; j < NT; ++j) f.w[j] = ld16(st + (BM + wrow(j)) * 64);
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = mfma16(f.a[i], f.w[j], acc[i][j]);
  };
#pragma unroll
  for (int s = 0; s < kBigStages - 1; ++s)
    if (s < nk) fetch(s);
  Frags f0, f1;
  if (nk > 4) wait_pieces<4 * P>();
  else wait_pieces<0>();
  meet();
  read(f0, 0);
  // Rounds of six steps, the slots of the ring known at compile time and nothing conditional in them (a branch around the loads
  // makes the compiler wait for the fragments just asked for); what is left goes step by step.
  auto steady = [&](int slot, const Frags& now, Frags& next) {
    wait_pieces<3 * P>();
    meet();
    read(next, (slot + 1) % kBigStages);
    fetch((slot + kBigStages - 1) % kBigStages);                 // (the stage everybody has been done with since the step before)
    multiply(now);
  };
  int t = 0;
  for (; t + 2 * kBigStages - 2 < nk; t += kBigStages) {
    steady(0, f0, f1); steady(1, f1, f0); steady(2, f0, f1);
    steady(3, f1, f0); steady(4, f0, f1); steady(5, f1, f0);
  }
  auto step = [&](int slot, const Frags& now, Frags& next) {
    if (t + 1 < nk) {
      const int behind = nk - 2 - t;
      if (behind >= 3) wait_pieces<3 * P>();
      else if (behind == 2) wait_pieces<2 * P>();
      else if (behind == 1) wait_pieces<P>();
      else wait_pieces<0>();
      meet();
      read(next, (slot + 1) % kBigStages);
      if (t + kBigStages - 1 < nk) fetch((slot + kBigStages - 1) % kBigStages);
    }
    multiply(now);
    ++t;
  };
  for (int slot = 0; t < nk; slot = (slot + 2) % kBigStages) {
    step(slot, f0, f1);
    if (t < nk) step(slot + 1, f1, f0);
  }
  if constexpr (UP) {
    // activations leave through LDS as 16-byte pieces of whole rows (straight from the accumulators a store instruction would
    // write 32 bytes of each of four rows); rows and columns that do not come in such pieces go out one by one
    constexpr int LDO = BO + 8, NO = GLU ? NT / 2 : NT;
    bf16* o = reinterpret_cast<bf16*>(lds);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm + i * 16 + kq * 4 + r;
        const long grow = (long)tile * BM + row;
        const float rw = row_w && row_tok[grow] >= 0 ? row_w[grow] : 1.f;      // (padding rows have no weight)
#pragma unroll
        for (int j = 0; j < NO; ++j) {
          float v;
          if constexpr (GLU) v = expert_act(acc[i][j][r] * rw, acc[i][j + NO][r] * rw, limit);
          else v = relu2(acc[i][j][r] * rw);
          o[row * LDO + wn * (BO / 4) + j * 16 + r16] = (bf16)v;
        }
      }
    __syncthreads();
    const bool wide = N % 8 == 0 && ldo % 8 == 0 && (uintptr_t)act_out % 16 == 0;
    for (int p = threadIdx.x; p < BM * (BO / 8); p += 512) {
      const int row = p / (BO / 8), c8 = (p % (BO / 8)) * 8, col = n0 + c8;
      bf16* to = act_out + ((long)tile * BM + row) * ldo + col;
      if (wide) { if (col < N) st16(to, ld16(o + row * LDO + c8)); }
      else for (int j = 0; j < 8 && col + j < N; ++j) to[j] = o[row * LDO + c8 + j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long row = (long)tile * BM + wm + i * 16 + kq * 4 + r;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int col = n0 + wrow(j) + r16;
          if (col < N) y_out[row * ldo + col] = acc[i][j][r];
        }
      }
  }
}

// V entries of a token's row per thread; the choices' rows and weights are asked for four at a time. (One entry a thread and choice
// after choice, 64 tokens of 4096: 12 us, now 4.8.)
template <int V>
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ out, const float* __restrict__ y,
                                                          const int* __restrict__ pair_row, const float* __restrict__ wts,
                                                          int H, int top, long ldo, const float* __restrict__ x, long ldx) {
  const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * V;
  if constexpr (V == 1) {      // (a loop: with many rows a workgroup each; 4096 rows of 1030 11.9 us, 14.4 with one for every 256 columns)
    for (int i = c; i < H; i += gridDim.y * 256) {
      float s = 0.f;
      for (int r = 0; r < top; ++r) {
        const int row = pair_row[(long)t * top + r];
        s += wts[(long)t * top + r] * (row >= 0 ? y[(long)row * H + i] : (x ? x[(long)t * ldx + i] : 0.f));
      }
      out[(long)t * ldo + i] = s;
    }
    return;
  }
  if (c >= H) return;
  Unit<V> s;
#pragma unroll
  for (int e = 0; e < V; ++e) s.v[e] = 0.f;
#pragma unroll 4
  for (int r = 0; r < top; ++r) {
    const int row = pair_row[(long)t * top + r];
    const float w = wts[(long)t * top + r];
    Unit<V> a;
    if (row >= 0 || x) a = ldu<V>(row >= 0 ? y + (long)row * H + c : x + (long)t * ldx + c);
    else {      // (zeros times the weight: one that is no number shows)
#pragma unroll
      for (int e = 0; e < V; ++e) a.v[e] = 0.f;
    }
#pragma unroll
    for (int e = 0; e < V; ++e) s.v[e] += w * a.v[e];
  }
  stu<V>(out + (long)t * ldo + c, s);
}

}  // namespace dlia

extern "C" void dlia_moe_route(int* sel, float* wts, const float* logits, long ld, int T, int E, int top, int groups, int keep,
                               float scale, const float* corr, int softmax, int group_rank, int renorm, hipStream_t stream) {
  if (T <= 0) return;
  hipLaunchKernelGGL(dlia::moe_route_kernel, dim3((T + 63) / 64), dim3(64), 0, stream, sel, wts, logits, ld, T, E, top, groups,
                     keep, scale, corr, softmax, group_rank, renorm);
}

extern "C" void dlia_moe_plan(int* tiles, int* row_tok, int* pair_row, const int* sel, int pairs, int top, int E, int max_rows,
                              int tile_rows, const float* wts, float* row_w, hipStream_t stream) {
  hipLaunchKernelGGL(dlia::moe_plan_kernel, dim3(1), dim3(1024), 0, stream, tiles, row_tok, pair_row, sel, pairs, top, E, max_rows,
                     tile_rows, wts, row_w);
}

extern "C" void dlia_moe_route_plan(int* sel, float* wts, const float* logits, long ld, int T, int E, int top, int groups, int keep, float scale,
                                    const float* corr, int softmax, int group_rank, int renorm, int* tiles, int* row_tok, int* pair_row,
                                    int experts, int max_rows, int tile_rows, float* row_w, hipStream_t stream) {
  if (T <= 0) return;
  if (T <= 256) {
    hipLaunchKernelGGL(dlia::moe_route_plan_kernel, dim3(1), dim3(1024), 0, stream, sel, wts, logits, ld, T, E, top, groups, keep, scale, corr,
                       softmax, group_rank, renorm, tiles, row_tok, pair_row, experts, max_rows, tile_rows, row_w);
    return;
  }
  dlia_moe_route(sel, wts, logits, ld, T, E, top, groups, keep, scale, corr, softmax, group_rank, renorm, stream);
  dlia_moe_plan(tiles, row_tok, pair_row, sel, T * top, top, experts, max_rows, tile_rows, wts, row_w, stream);
}

template <typename T, typename OT, int NJ>
static void launch_moe_up(void* act, const void* x, const void* wg, const void* wu, const int* tiles, const int* row_tok, int max_tiles,
                          int F, int K, long ldx, long lda, float limit, int ok, const float* row_w, hipStream_t stream) {
  const dim3 grid((F + 64 * NJ - 1) / (64 * NJ), max_tiles);
  const bool fast = ok && K % (64 / (int)sizeof(T)) == 0;
#define DLIA_UP(GLU, FAST)                                                                                                                 \
  hipLaunchKernelGGL((dlia::moe_up_kernel<T, OT, NJ, GLU, FAST>), grid, dim3(256), 0, stream, (OT*)act, (const T*)x, (const T*)wg, (const T*)wu, \
                     tiles, row_tok, F, K, ldx, lda, limit, ok, row_w)
  if (wg) { if (fast) DLIA_UP(true, true); else DLIA_UP(true, false); }
  else { if (fast) DLIA_UP(false, true); else DLIA_UP(false, false); }
#undef DLIA_UP
}
template <typename T, int NJ>
static void launch_moe_down(float* y, const void* act, const void* wd, const int* tiles, const int* row_tok, int max_tiles, int H, int F,
                            long lda, int ok, hipStream_t stream) {
  const dim3 grid((H + 64 * NJ - 1) / (64 * NJ), max_tiles);
  if (ok && F % (64 / (int)sizeof(T)) == 0)
    hipLaunchKernelGGL((dlia::moe_down_kernel<T, NJ, true>), grid, dim3(256), 0, stream, y, (const T*)act, (const T*)wd, tiles, row_tok, H, F, lda, ok);
  else
    hipLaunchKernelGGL((dlia::moe_down_kernel<T, NJ, false>), grid, dim3(256), 0, stream, y, (const T*)act, (const T*)wd, tiles, row_tok, H, F, lda, ok);
}

// (the plan's number of tiles is known on the device alone: max_tiles has one to spare per expert, a workgroup without one ends)
template <int KIND>
static void launch_moe_big(void* act, float* y, const void* a, const void* w0, const void* w1, const int* tiles, const int* row_tok,
                           int max_tiles, int experts, int N, int K, long lda, long ldo, float limit, const float* row_w, hipStream_t stream) {
  // 256 or 128 weight rows by the rounds over the 256 CUs that about max_tiles - experts / 2 row tiles make, one an expert at least (a round of
  // the narrow form costs 0.6 of one of the wide form: 520 tokens, 2 of 8 experts, width and expert 2048: gate and up 41 us wide and 54
  // narrow, down 33 and 23)
  const int cols = KIND == 1 ? 2 * N : N, likely = std::max(max_tiles - experts / 2 - 1, experts);
  if (dlia_moe_pairs(max_tiles, experts, cols, K)) {
    dlia_moe_pingpong(KIND, act, y, a, w0, w1, tiles, row_tok, max_tiles, experts, N, K, lda, ldo, limit, row_w, stream);
    return;
  }
  const int r256 = ((cols + 255) / 256 * likely + 255) / 256, r128 = ((cols + 127) / 128 * likely + 255) / 256;
#define DLIA_BIG(BN)                                                                                                                    \
  hipLaunchKernelGGL((dlia::moe_big_kernel<KIND, BN>), dim3((N + (KIND == 1 ? BN / 2 : BN) - 1) / (KIND == 1 ? BN / 2 : BN) * max_tiles), \
                     dim3(512), 0, stream, (dlia::bf16*)act, y, (const dlia::bf16*)a, (const dlia::bf16*)w0, (const dlia::bf16*)w1, tiles, \
                     row_tok, N, K, lda, ldo, limit, row_w)
  if (r128 * 0.62 < r256) DLIA_BIG(128);
  else DLIA_BIG(256);
#undef DLIA_BIG
}

// About how many row tiles of 32 a step has: its pairs' and half a tile an expert, one an expert at least where there are four pairs for each
static int likely_tiles(int max_tiles, int experts) {
  const int most = max_tiles - experts;
  return std::max(std::min(max_tiles - experts / 2, 32 * most), 8 * most >= experts ? experts : 0);
}

template <typename T, typename OT, int KIND>
static void launch_moe_stream(OT* out, const T* x, const T* w0, const T* w1, const int* tiles, const int* row_tok, int max_tiles, int experts, int N,
                              int K, long ldx, long ldo, float limit, int ok, const float* row_w, hipStream_t stream) {
  // One column tile a wave where the gated kernel would have too few workgroups to fill the chip three a CU, or hardly a row each (2048 x
  // 2048, 64 tokens: 27.6 us against 30.7; 3584 x 4096, 4 tokens: 51 against 58, 64 tokens 101 against 96; by the row tiles there
  // are, not the experts: 2048 x 2048, 300 / 400 tokens in 19 / 25 tiles 86 / 107 us against 70 / 89); fp32 pieces are half as deep and its
  // workgroups last longer (64 tokens: 68 against 60).
#define DLIA_ST(FAST, U, NJ, RT)                                                                                                               \
  hipLaunchKernelGGL((dlia::moe_stream_kernel<T, OT, KIND, FAST, 4, U, NJ, RT>), dim3((N + 16 * NJ - 1) / (16 * NJ), max_tiles), dim3(256), 0, \
                     stream, out, x, w0, w1, tiles, row_tok, N, K, ldx, ldo, limit, ok, row_w)
  if constexpr (KIND == 1 && sizeof(T) == 2)
    if (max_tiles - experts <= 1 || (long)(N + 31) / 32 * likely_tiles(max_tiles, experts) < 768) {
      if (ok && K % (256 / (int)sizeof(T)) == 0) DLIA_ST(true, 4, 1, 1);
      else DLIA_ST(false, 4, 1, 1);
      return;
    }
  // Tiles of one expert two a workgroup from 16 rows an expert on, where some have more than a tile: its weights then come once for 64 rows. us, a tile a
  // workgroup against two, gated 3584 x 4096, two of 8 experts: 96 / 128 / 160 / 200 / 300 tokens 102 / 130 / 153 / 158 / 226 -> 100 / 121 / 127 / 134 / 192, down 61 / 80 / 93 / 102 / 143 ->
  // 61 / 68 / 72 / 83 / 133; with one tile each the same (64 tokens 92, 52). Not in fp32, whose tiles are bound by the matrix rate (a prompt of 300 tokens, one expert of 8
  // taking all of them, the step 4317 -> 4530).
  constexpr int two = sizeof(T) == 2 ? 2 : 1;
  if (ok && K % (128 / (int)sizeof(T)) == 0 && 2 * (max_tiles - experts) >= experts) DLIA_ST(true, 2, 2, two);
  else if (ok && K % (128 / (int)sizeof(T)) == 0) DLIA_ST(true, 2, 2, 1);
  else DLIA_ST(false, 2, 2, 1);
#undef DLIA_ST
}

// Steps that run in wide column blocks (128 columns of gate and up, 256 of the down projection, a workgroup a CU) and not as a stream of the
// weights: experts of more than four tiles, and blocks that fill their rounds over the 256 CUs. A round takes what it takes however few its
// blocks (8 experts, two a token, 2048 x 2048 fp32, down: 96 to 107 us), a stream goes by the rows (0.48 us a block's worth): 700 / 1000 /
// 1400 / 2048 tokens 187 / 303 / 306 / 527 us in blocks and 179 / 250 / 339 / 485 as a stream. Gate and up gain by blocks in a single full
// round alone (1900 tokens, one of 4 experts, 1024 x 512: 60 against 64 us; the above, 1000 / 1400 tokens: 579 / 707 against 421 / 576).
extern "C" int dlia_moe_wide(int max_tiles, int experts, int cols, int down) {
  const long blocks = (long)(max_tiles - experts / 2) * ((cols + (down ? 255 : 127)) / (down ? 256 : 128)), rounds = (blocks + 255) / 256;
  return max_tiles - experts > 4 * experts && blocks * 10 > rounds * 256 * 9 && (down || rounds == 1);
}

// Steps of a short K (kind as in the stream, which leaves such a K to one of a workgroup's four waves and pays for whole pieces): column blocks of
// 64 (1), or the wide ones (2) where experts have more than four tiles, as soon as the stream's workgroups are more than a round or two; before
// that its launch is the shorter one. Stream against blocks, 314 shapes of K up to 512 bf16, 128 fp32, by the stream's workgroups as estimated here:
// gated, above 512 0.93 to 3.7 of the blocks' time, on average 1.35 (32 tokens, one of 32 experts of 4096, K 40: 24 against 6.5 us; 1400 tokens, two of 16
// of 3584, K 200: 105 against 50), in 16 bits 0.76 to 0.9 up to 512 and with whole pieces up to 1024; the other kinds, from 1024 on, 0.92 to 1.39 where K is at most 192 bytes, down
// 0.66 to 1.0 above that, squared ReLU 0.98 to 1.25 with masked pieces; with many tiles the wide ones up to 256 in fp32 too: gated, K 256, 111 against 99 us, down, K 64, 35 against 27.
extern "C" int dlia_moe_short(int max_tiles, int experts, int cols, int K, int f32, int kind) {
  const int bytes = K * (f32 ? 4 : 2), most = max_tiles - experts;
  if (bytes > 1024) return 0;
  const long tiles = likely_tiles(max_tiles, experts);
  const bool narrow = kind == 1 && !f32 && (most <= 1 || (cols + 31) / 32 * tiles < 768);
  const long groups = (narrow ? (cols + 15) / 16 : (cols + 31) / 32) * tiles;
  if (most > 4 * experts && groups >= 4096 && (kind || bytes <= 512)) return 2;
  if (f32 && bytes > 512) return 0;
  if (kind == 1 ? groups <= (narrow && bytes % 256 == 0 ? 1024 : 512) : groups < 1024 || (bytes > 192 && (kind == 0 || bytes % 128 == 0))) return 0;
  return most > 4 * experts ? 2 : 1;
}

template <typename T>
static void moe_up_rows(T* act, const T* x, const T* wg, const T* wu, const int* tiles, const int* row_tok, int max_tiles, int experts, int F, int K,
                        long ldx, long lda, float limit, int ok, const float* row_w, hipStream_t stream) {
  const int few = dlia_moe_short(max_tiles, experts, F, K, sizeof(T) == 4, wg ? 1 : 2);
  if (few == 1) launch_moe_up<T, T, 1>(act, x, wg, wu, tiles, row_tok, max_tiles, F, K, ldx, lda, limit, ok, row_w, stream);
  else if (few || dlia_moe_wide(max_tiles, experts, F, 0)) launch_moe_up<T, T, 2>(act, x, wg, wu, tiles, row_tok, max_tiles, F, K, ldx, lda, limit, ok, row_w, stream);
  else if (wg) launch_moe_stream<T, T, 1>(act, x, wg, wu, tiles, row_tok, max_tiles, experts, F, K, ldx, lda, limit, ok, row_w, stream);
  else launch_moe_stream<T, T, 2>(act, x, wu, nullptr, tiles, row_tok, max_tiles, experts, F, K, ldx, lda, limit, ok, row_w, stream);
}
template <typename T>
static void moe_down_rows(float* y, const T* act, const T* wd, const int* tiles, const int* row_tok, int max_tiles, int experts, int H, int F,
                          long lda, int ok, hipStream_t stream) {
  const int few = dlia_moe_short(max_tiles, experts, H, F, sizeof(T) == 4, 0);
  if (few == 1) launch_moe_down<T, 1>(y, act, wd, tiles, row_tok, max_tiles, H, F, lda, ok, stream);
  else if (few || dlia_moe_wide(max_tiles, experts, H, 1)) launch_moe_down<T, 4>(y, act, wd, tiles, row_tok, max_tiles, H, F, lda, ok, stream);
  else launch_moe_stream<T, float, 0>(y, act, wd, nullptr, tiles, row_tok, max_tiles, experts, H, F, lda, (long)H, 0.f, ok, nullptr, stream);
}

extern "C" void dlia_moe_up(void* act, const void* x, const void* wg, const void* wu, int f32, const int* tiles, const int* row_tok,
                            int max_tiles, int experts, int F, int K, long ldx, long lda, float limit, int tile_rows, const float* row_w,
                            hipStream_t stream) {
  if (max_tiles <= 0) return;
  if (tile_rows == dlia::kMoeBigRows) {
    if (wg) launch_moe_big<1>(act, nullptr, x, wg, wu, tiles, row_tok, max_tiles, experts, F, K, ldx, lda, limit, row_w, stream);
    else launch_moe_big<2>(act, nullptr, x, wu, nullptr, tiles, row_tok, max_tiles, experts, F, K, ldx, lda, limit, row_w, stream);
    return;
  }
  const int vec = f32 ? 4 : 8;
  const int ok = K % vec == 0 && ldx % vec == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)wg % 16 == 0 && (uintptr_t)wu % 16 == 0;
  if (f32)
    moe_up_rows((float*)act, (const float*)x, (const float*)wg, (const float*)wu, tiles, row_tok, max_tiles, experts, F, K, ldx, lda, limit, ok, row_w, stream);
  else
    moe_up_rows((dlia::bf16*)act, (const dlia::bf16*)x, (const dlia::bf16*)wg, (const dlia::bf16*)wu, tiles, row_tok, max_tiles, experts, F, K, ldx, lda,
                limit, ok, row_w, stream);
}

extern "C" void dlia_moe_down(float* y, const void* act, const void* wd, int f32, const int* tiles, const int* row_tok,
                              int max_tiles, int experts, int H, int F, long lda, int tile_rows, hipStream_t stream) {
  if (max_tiles <= 0) return;
  if (tile_rows == dlia::kMoeBigRows) {
    launch_moe_big<0>(nullptr, y, act, wd, nullptr, tiles, row_tok, max_tiles, experts, H, F, lda, (long)H, 0.f, nullptr, stream);
    return;
  }
  const int vec = f32 ? 4 : 8;
  const int ok = F % vec == 0 && lda % vec == 0 && (uintptr_t)act % 16 == 0 && (uintptr_t)wd % 16 == 0;
  if (f32) moe_down_rows(y, (const float*)act, (const float*)wd, tiles, row_tok, max_tiles, experts, H, F, lda, ok, stream);
  else moe_down_rows(y, (const dlia::bf16*)act, (const dlia::bf16*)wd, tiles, row_tok, max_tiles, experts, H, F, lda, ok, stream);
}

extern "C" void dlia_moe_combine(float* out, const float* y, const int* pair_row, const float* wts, int T, int H, int top, long ldo,
                                 const float* x, long ldx, hipStream_t stream) {
  if (T <= 0) return;
  if (H % 4 == 0 && ldo % 4 == 0 && ldx % 4 == 0 && dlia::al16_(out) && dlia::al16_(y) && dlia::al16_(x))
    hipLaunchKernelGGL(dlia::moe_combine_kernel<4>, dim3(T, (H + 1023) / 1024), dim3(256), 0, stream, out, y, pair_row, wts, H, top, ldo, x, ldx);
  else
    hipLaunchKernelGGL(dlia::moe_combine_kernel<1>, dim3(T, T > 1024 ? 1 : (H + 255) / 256), dim3(256), 0, stream, out, y, pair_row, wts, H, top, ldo, x, ldx);
}

extern "C" void dlia_moe_table_plan(int* tiles, int* row_tok, int* pair_row, const int* tables, const int* ids, const int* desc, int layers,
                                    int T, int vocab, int big_pairs, hipStream_t stream) {
  if (layers <= 0) return;
  hipLaunchKernelGGL(dlia::moe_table_plan_kernel, dim3(layers), dim3(1024), 0, stream, tiles, row_tok, pair_row, tables, ids, desc, T, vocab,
                     big_pairs);
}

extern "C" void dlia_glu_act(void* act, int out_f32, long lda, const float* z, long ldz, int M, int F, float limit, int gated, hipStream_t stream) {
  if (M <= 0 || F <= 0) return;
  // (fewer entries are spread over more threads: 16 rows of 2048 2.0 us, 2.1 in fours; 1024 of 96 2.1, 2.35; 64 of 8192 2.3, 2.4; from the line on
  // 256 rows of 2048 2.6, 2.4, 1024 of 3584 7.8, 6.2)
  const bool wide = M >= 128 && F >= 512 && (long)M * F >= 1 << 19 && F % 4 == 0 && ldz % 4 == 0 && lda % 4 == 0 && dlia::al16_(z) && (uintptr_t)act % (out_f32 ? 16 : 8) == 0;
  const dim3 grid(((wide ? F / 4 : F) + 255) / 256, M);
#define DLIA_GLU(OT, V)                                                                                                              \
  do {                                                                                                                              \
    if (limit > 0.f) hipLaunchKernelGGL((dlia::glu_act_kernel<OT, V, true>), grid, dim3(256), 0, stream, (OT*)act, lda, z, ldz, F, limit, gated); \
    else hipLaunchKernelGGL((dlia::glu_act_kernel<OT, V, false>), grid, dim3(256), 0, stream, (OT*)act, lda, z, ldz, F, limit, gated);            \
  } while (0)
  if (out_f32) { if (wide) DLIA_GLU(float, 4); else DLIA_GLU(float, 1); }
  else { if (wide) DLIA_GLU(dlia::bf16, 4); else DLIA_GLU(dlia::bf16, 1); }
#undef DLIA_GLU
}
