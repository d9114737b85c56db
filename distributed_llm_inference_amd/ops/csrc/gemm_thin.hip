// Weight stream for at most 16 rows with the whole of K inside a workgroup: out[M,N] = epi(f(x)[M,K] @ W[N,K]^T), f the RMSNorm of the rows or
// nothing. W is the packed-B image of gemm_skinny.hip.
//
// A decode step of few rows is a chain of launches of 4 to 8 us, each a launch, a trip to memory for x and one for the weights; the bytes
// themselves take 2 to 5 us. Two of the chain's launches a layer were norms, which existed because the GEMM in front of them left K splits to be added
// up: a column block of 128 needs eight of them to fill the chip. Here a workgroup has 16 columns (32 where gate and up meet) and its eight waves
// deal out K, so sums are complete where they are formed: the residual is added in the epilogue, and the next GEMM normalises the rows
// itself while its weights are on their way (every workgroup the same few KB, from L2). The q | k | v projection goes further: its workgroups hold
// the two places of a head that rotate together, and their epilogue is the rotation and the cache write.
// Bound by memory latency at one or two rounds of workgroups, by the weight stream beyond. A TinyLlama layer (hidden 2048, one row, 300 tokens), us a launch:
// norm 4.2, qkv 7, rope 5.1, attention, o 6, norm 4.2, gate / up 13, down 9 -> qkv 5.8, attention, o and down 6.3 on average, gate / up 9.6 (4.8 TB/s);
// 11 layers with the head 556 -> 410 a step, 8 rows 597 -> 474, 12 rows 605 -> 502. Four Llama-3-8B layers, 1 / 4 / 7 rows 446 / 461 / 468 -> 406 / 422 / 441.
// Rows times hidden size is the limit: every workgroup reads all rows, and from 32768 entries on (64 KB of LDS) one workgroup a CU is left
// (8 rows of 4096: 466 either way, 16 of 2048: 614 -> 594 and 617 on two boxes): the callers stay below.
// What helped: rows in LDS instead of registers (a second workgroup a CU: gate / up 13.8 -> 11.2), its second chunk of weights asked for behind the norm
// (11.2 -> 9.6), eight columns a workgroup where there are fewer than 256 (the step 451 -> 433).
#include "common.h"
#include "gemm_common.h"
#include "kv_layout.h"
#include "launch.h"

namespace dlia {

constexpr int kThinRows = 16 * (2048 + 8);      // entries of normalised rows a workgroup keeps at most

// Row t's places d .. d + 3 and D / 2 + d .. of a head of q | k | v: bias, rotation, q to its row, k and v to the paged cache (as rope_kv.hip).
__device__ __forceinline__ void rope_and_store(const ThinRope& p, bf16* __restrict__ q, long ldq, const bf16* __restrict__ bias, int t, int head, int d,
                                               f32x4 lo, f32x4 hi) {
  const int half = p.D >> 1, pos = p.tok_pos[t], seq = p.tok_seq[t], bidx = pos / kBlockTokens, kk = pos % kBlockTokens;
  if (bias) {
    const u32x2 a = *reinterpret_cast<const u32x2*>(bias + head * p.D + d), b = *reinterpret_cast<const u32x2*>(bias + head * p.D + half + d);
    lo += f32x4{bf16_lo(a[0]), bf16_hi(a[0]), bf16_lo(a[1]), bf16_hi(a[1])};
    hi += f32x4{bf16_lo(b[0]), bf16_hi(b[0]), bf16_lo(b[1]), bf16_hi(b[1])};
  }
  if (head < p.Hq + p.Hkv) {
    const long rp = pos < 0 ? 0 : (pos >= p.rope_len ? p.rope_len - 1 : pos);        // table reads stay in bounds
    const f32x4 c = *reinterpret_cast<const f32x4*>(p.cos_t + rp * half + d), s = *reinterpret_cast<const f32x4*>(p.sin_t + rp * half + d);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = lo[r], b = hi[r];
      lo[r] = a * c[r] - b * s[r];
      hi[r] = b * c[r] + a * s[r];
    }
  }
  const u32x2 l2 = {pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3])}, h2 = {pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
  if (head < p.Hq) {
    bf16* to = q + (long)t * ldq + head * p.D + d;
    *reinterpret_cast<u32x2*>(to) = l2;
    *reinterpret_cast<u32x2*>(to + half) = h2;
    return;
  }
  int blk = -1;
  if (pos >= 0 && seq >= 0 && bidx < p.max_blocks) blk = p.block_table[(long)seq * p.max_blocks + bidx];
  if (blk < 0 || blk >= p.num_blocks) return;                    // an unallocated slot is skipped, never a wild store
  const bool is_k = head < p.Hq + p.Hkv;
  bf16* base = reinterpret_cast<bf16*>(p.kv) + kv_head_base(blk, is_k ? head - p.Hq : head - p.Hq - p.Hkv, p.Hkv, p.D, is_k ? 0 : 1);
  if (is_k) {
    *reinterpret_cast<u32x2*>(base + k_elem_off(kk, d, p.D)) = l2;
    *reinterpret_cast<u32x2*>(base + k_elem_off(kk, half + d, p.D)) = h2;
  } else {
    unsigned short* v = reinterpret_cast<unsigned short*>(base);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[v_elem_off(kk, d + r)] = (unsigned short)(l2[r >> 1] >> (16 * (r & 1)));
      v[v_elem_off(kk, half + d + r)] = (unsigned short)(h2[r >> 1] >> (16 * (r & 1)));
    }
  }
}

// U: k-steps of a chunk; a wave has two chunks of weights on their way, asked for before anything else. NORM: the rows go through RMSNorm into LDS, a
// wave a row, while the weights travel (in registers they would keep a second workgroup off the CU); otherwise fragments straight from memory.
template <int NT, int NORM, int EPI, int U, int NW, bool HALF>
__global__ __launch_bounds__(64 * NW, EPI == 4 ? 4 : 2) void gemm_thin_kernel(void* __restrict__ out, long ldo, const bf16* __restrict__ x, long ldx,
                                                            const u32x4* __restrict__ wp, const bf16* __restrict__ nw, float eps,
                                                            const bf16* __restrict__ bias, const bf16* residual, long ldr, int M, int N, int K, ThinRope rope) {
  static_assert((EPI != 4 && EPI != 7) || NT % 2 == 0, "two tiles of the same columns");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4 (*const part)[NT][64] = reinterpret_cast<f32x4 (*)[NT][64]>(smem);          // [NW]
  bf16* const rows = reinterpret_cast<bf16*>(smem + NW * NT * 1024);                // [M][K + 8]: 16 rows of a fragment on different banks
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int l15 = lane & 15, quad = lane >> 4;
  const int KT = K >> 5, per = (KT + NW - 1) / NW;
  const int k0 = min(wave * per, KT - 1), n = max(min(wave * per + per, KT) - wave * per, 0);          // k-steps of this wave
  const int tiles = (N + 15) >> 4;
  // HALF: eight columns of every tile, the other eight lanes of a quad the same ones again
  const int block = HALF ? blockIdx.x >> 1 : blockIdx.x, hc = HALF ? (blockIdx.x & 1) * 8 : 0;
  // EPI 7: a workgroup's two tiles are the places d .. d + 15 of a head and those half a head further on, which rotate together
  const int half_tiles = rope.D >> 5, head = EPI == 7 ? block / half_tiles : 0, place = EPI == 7 ? block % half_tiles : 0;
  auto tile = [&](int j) { return EPI == 7 ? head * 2 * half_tiles + place + j * half_tiles : block * NT + j; };
  const bf16* const xr = NORM ? rows + min(l15, M - 1) * (K + 8) + quad * 8 + k0 * 32 : x + (long)min(l15, M - 1) * ldx + quad * 8 + (long)k0 * 32;
  const unsigned wl = (HALF ? quad * 16 + hc + (l15 & 7) : lane) * 16;
  const char* wr[NT];                                  // (the same for all lanes)
#pragma unroll
  for (int j = 0; j < NT; ++j) wr[j] = reinterpret_cast<const char*>(wp + ((long)min(tile(j), tiles - 1) * KT + k0) * 64);
  f32x4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 wf[2][U][NT], xf[2][NORM ? 1 : U];
  // (past the end of the wave's part: its last k-step again, which is not multiplied)
  auto step = [&](int c, int u) { return max(min(c * U + u, n - 1), 0); };
  auto fetch = [&](int b, int c) {
    if constexpr (!NORM) {
#pragma unroll
      for (int u = 0; u < U; ++u) xf[b][u] = ld16(xr + step(c, u) * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j) wf[b][u][j] = ld16_nt(wr[j] + (long)step(c, u) * 1024 + wl);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mul = [&](int b, int c) {
    auto one = [&](int u) {
      const u32x4 v = NORM ? ld16(xr + (c * U + u) * 32) : xf[b][NORM ? 0 : u];
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = mfma16(wf[b][u][j], v, acc[j]);
    };
    if (c * U + U <= n) {
#pragma unroll
      for (int u = 0; u < U; ++u) one(u);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c * U + u < n) one(u);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // NORM waves a row, up to 2048 entries each
  constexpr int kRow = 4;                              // 16-byte pieces of a row a lane holds
  u32x4 row[NORM ? kRow : 1], factor[NORM ? kRow : 1];
  constexpr int parts = NORM ? NORM : 1, stride = NW / parts;
  const int mine = wave % parts, r0 = wave / parts;
  auto at = [&](int i) { return mine * 2048 + (i * 64 + lane) * 8; };
  auto fetch_row = [&](int r) {
#pragma unroll
    for (int i = 0; i < kRow; ++i) row[i] = ld16(x + (long)min(r, M - 1) * ldx + min(at(i), K - 8));
  };
  if constexpr (NORM) {
    fetch_row(r0);
#pragma unroll
    for (int i = 0; i < kRow; ++i) factor[i] = ld16(nw + min(at(i), K - 8));
    __builtin_amdgcn_sched_barrier(0);
  }
  const int chunks = (n + U - 1) / U;
  fetch(0, 0);
  if constexpr (!NORM || EPI != 4) fetch(1, 1);
  if constexpr (NORM) {
    auto meet = [] {                                   // (no wait for the weights: the barrier is for LDS alone)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    auto squares = [&] {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < kRow; ++i) {
        float f[8];
        unpack8(row[i], f);
        if (at(i) < K) {
#pragma unroll
          for (int e = 0; e < 8; ++e) s += f[e] * f[e];
        }
      }
      return wave_sum(s);
    };
    auto put = [&](int r, float sum) {
      const float rstd = rsqrtf(sum / K + eps);
#pragma unroll
      for (int i = 0; i < kRow; ++i) {
        float f[8], g[8];
        unpack8(row[i], f);
        unpack8(factor[i], g);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = f[e] * rstd * g[e];
        if (at(i) < K) st16(rows + r * (K + 8) + at(i), pack8(f));
      }
    };
    if constexpr (NORM == 1) {
      for (int r = r0; r < M; r += stride) {
        put(r, squares());
        if (r + stride < M) fetch_row(r + stride);
      }
    } else {
      float* const sums = reinterpret_cast<float*>(smem);        // [16][parts], where the tiles meet later
      for (int r = r0; r < M; r += stride) {
        if (r != r0) fetch_row(r);
        const float s = squares();
        if (lane == 0) sums[r * parts + mine] = s;
      }
      meet();
      for (int r = r0; r < M; r += stride) {
        if (M > stride) fetch_row(r);
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < parts; ++q) t += sums[r * parts + q];
        put(r, t);
      }
    }
    meet();
    if constexpr (EPI == 4) fetch(1, 1);
  }
  int c = 0;
  for (; c + 3 < chunks; c += 2) { mul(0, c); fetch(0, c + 2); mul(1, c + 1); fetch(1, c + 3); }
  mul(0, c);
  if (c + 2 < chunks) {
    fetch(0, c + 2);
    mul(1, c + 1);
    mul(0, c + 2);
  } else {
    mul(1, c + 1);                                     // (no such chunk: nothing)
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) part[wave][j][lane] = acc[j];
  __syncthreads();
  constexpr int OUT = EPI == 4 || EPI == 7 ? NT / 2 : NT, IN = NT / OUT;   // (one wave a tile that leaves)
  if (wave >= OUT || l15 >= M || (HALF && quad >= 2)) return;
  f32x4 s[IN];
#pragma unroll
  for (int j = 0; j < IN; ++j) {
    s[j] = part[0][wave * IN + j][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) s[j] += part[w][wave * IN + j][lane];
  }
  if constexpr (EPI == 7) {
    rope_and_store(rope, reinterpret_cast<bf16*>(out), ldo, bias, l15, head, place * 16 + hc + quad * 4, s[0], s[IN - 1]);
    return;
  }
  const int col = (block * OUT + wave) * 16 + hc + quad * 4;
  if (col >= (EPI == 4 ? N >> 1 : N)) return;
  float v[4] = {s[0][0], s[0][1], s[0][2], s[0][3]};
  if constexpr (EPI == 4) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = silu(v[r]) * s[IN - 1][r];
  }
  if (bias) {
    const u32x2 b = *reinterpret_cast<const u32x2*>(bias + col);
    v[0] += bf16_lo(b[0]); v[1] += bf16_hi(b[0]); v[2] += bf16_lo(b[1]); v[3] += bf16_hi(b[1]);
  }
  if constexpr (EPI == 2) {
    const u32x2 b = *reinterpret_cast<const u32x2*>(residual + (long)l15 * ldr + col);
    v[0] += bf16_lo(b[0]); v[1] += bf16_hi(b[0]); v[2] += bf16_lo(b[1]); v[3] += bf16_hi(b[1]);
  }
  store4(out, ldo, l15, col, v, EPI == 6);
}

}  // namespace dlia

using namespace dlia;

template <int NT, int NORM, int EPI, int U, int NW, bool HALF>
static void launch_thin(int workgroups, void* out, long ldo, const void* x, long ldx, const void* wp, const void* norm_w, float eps, const void* bias,
                        const void* residual, long ldr, int M, int N, int K, const ThinRope& rope, hipStream_t stream) {
  constexpr int join = NW * NT * 1024;
  const int lds = join + (NORM ? M * (K + 8) * 2 : 0);
  if constexpr (NORM) {                                 // (more than 64 KiB of dynamic LDS is opt-in, once per kernel)
    static const bool once = [] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_thin_kernel<NT, NORM, EPI, U, NW, HALF>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                join + kThinRows * 2);
      return true;
    }();
    (void)once;
  }
  hipLaunchKernelGGL((gemm_thin_kernel<NT, NORM, EPI, U, NW, HALF>), dim3(workgroups), dim3(64 * NW), lds, stream, out, ldo, (const bf16*)x, ldx, (const u32x4*)wp,
                     (const bf16*)norm_w, eps, (const bf16*)bias, (const bf16*)residual, ldr, M, N, K, rope);
}

extern "C" void dlia_gemm_thin(void* out, long ldo, const void* x, long ldx, const void* wp, const void* norm_w, float eps, const void* bias,
                               const void* residual, long ldr, int M, int N, int K, int epi, const dlia::ThinRope* rope, hipStream_t stream) {
  if (M <= 0 || N <= 0) return;
  const int tiles = (N + 15) / 16;
  const ThinRope none = {};
#define DLIA_THIN(WGS, NT, NORM, EPI, U, NW, H, R) \
  launch_thin<NT, NORM, EPI, U, NW, H>((WGS) << (H), out, ldo, x, ldx, wp, norm_w, eps, bias, residual, ldr, M, N, K, R, stream)
  const bool half = tiles < 256;                       // (columns for every CU)
  const bool wide = K > 2048;
  if (epi == 7) {
    if (wide) DLIA_THIN(tiles / 2, 2, 2, 7, 2, 16, false, *rope);
    else if (half) DLIA_THIN(tiles / 2, 2, 1, 7, 2, 16, true, *rope);
    else DLIA_THIN(tiles / 2, 2, 1, 7, 2, 16, false, *rope);
  } else if (epi == 4) {
    if (wide) DLIA_THIN(tiles / 2, 2, 2, 4, 4, 8, false, none);
    else DLIA_THIN(tiles / 2, 2, 1, 4, 4, 8, false, none);
  } else if (epi == 6) {
    if (wide) DLIA_THIN(tiles, 1, 2, 6, 4, 8, false, none);
    else DLIA_THIN(tiles, 1, 1, 6, 4, 8, false, none);
  } else {
    if (half) DLIA_THIN(tiles, 1, 0, 2, 8, 8, true, none);
    else DLIA_THIN(tiles, 1, 0, 2, 8, 8, false, none);
  }
#undef DLIA_THIN
}
