// Row kernels of stacks whose sublayers read the fp32 residual stream itself and are normed on their OUTPUT only,
//     x <- x + rms(a * ya + b * yb) w,
// and the preparation of an attention mixer's q, k, v between its input projection and the cache.
//
//   post_norm_add   one launch per sublayer boundary: the weighted sum of one or two sublayer outputs is RMS-normed over the
//                   row, scaled by the norm's weight and added to the stream; the stream leaves in the GEMMs' input type
//                   for the next sublayer (the role residual + RMSNorm has for the Llama path). Without outputs it only
//                   converts the stream (the embedding ahead of the first layer).
//   mix_prep        per token, on the fp32 output q | k | v of the input projection: RMS norm of q and of k over the WHOLE
//                   projection (all heads at once, a weight per entry), rotation of the first `dims` entries of every head by
//                   the token's position (pairs (i, i + dims / 2), angles from a table), every value head divided by its root
//                   mean square; k and v rows go to the paged cache, q leaves for the attention kernel. With a head-mixing
//                   matrix M [H, H] (scores of head h are sum_g M[h, g] q_g . k) the mix is carried by the query: q leaves
//                   as H rows of G * d entries, row h holding for every key head c the sum over the heads g of c's group of
//                   M[h, g] q_g, and the keys of all G heads are ONE cache row of G * d entries that every head reads.
// The fused multiply-adds of the sums and of the rotation are written out: which product of a pair is rounded would otherwise change with the
// unrolling, and a stack whose gates are exponential shows it.
// Norm statistics, rotation and the mix are fp32; outputs take the GEMMs' / the cache's type (bf16 or fp32).
#include "common.h"
#include "launch.h"

namespace dlia {

constexpr int kPostBlock = 32;       // tokens per cache block
constexpr int kPostThreads = 256;

// N > 0: rows of up to N * 256 entries in registers, a thread's entries of all operands asked for at once. A few hundred rows are about a
// workgroup a CU, so a launch lasts as long as one row's loads, and a loop that reads an entry, adds and reads the next pays the memory's
// latency for each. Entries are dealt to threads and added in the order of the loop (N = 0, any length), the multiply-adds written out: the same bits.
// Two operands, us a launch: 1 row of 2048 6.5 -> 3.1, 256 of 2048 7.5 -> 3.9, 256 of 1024 4.8 -> 3.2, 256 of 256 2.9 -> 2.65 (with the eight predicated
// loads of the longest rows 3.2; 2048 such rows 4.4 -> 4.2, with eight 5.6), 32 of 4096 9.6 -> 4.4, 2048 of 4096 31.9 -> 20.6. Rows of
// more than 4096 entries stay in the loop (16 entries take 78 registers; more was not tried).
template <typename OT, int N>
__global__ __launch_bounds__(kPostThreads) void post_norm_add_kernel(
    OT* __restrict__ out, long ldo, float* __restrict__ x, long ldx, const float* __restrict__ ya, long ldya,
    const float* __restrict__ yb, long ldyb, float a, float b, const float* __restrict__ w, int H, float eps) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  float* xr = x + (long)t * ldx;
  OT* orow = out ? out + (long)t * ldo : nullptr;
  const float* ar = ya ? ya + (long)t * ldya : nullptr;
  const float* br = yb ? yb + (long)t * ldyb : nullptr;
  if constexpr (N > 0) {
    float v[N], y[N], y2[N], g[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = threadIdx.x + u * kPostThreads;
      const bool in = i < H;
      v[u] = in ? xr[i] : 0.f;
      y[u] = in && ar ? ar[i] : 0.f;
      y2[u] = in && br ? br[i] : 0.f;
      g[u] = in && ar ? w[i] : 0.f;
    }
    if (ar) {
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < N; ++u) {
        y[u] = br ? __builtin_fmaf(b, y2[u], a * y[u]) : a * y[u];
        if ((int)threadIdx.x + u * kPostThreads < H) ss = __builtin_fmaf(y[u], y[u], ss);
      }
      ss = block_sum(ss, scratch);
      const float r = 1.f / sqrtf(ss / H + eps);
#pragma unroll
      for (int u = 0; u < N; ++u) v[u] = __builtin_fmaf(y[u] * r, g[u], v[u]);
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = threadIdx.x + u * kPostThreads;
      if (i >= H) break;
      if (ar) xr[i] = v[u];
      if (out) orow[i] = (OT)v[u];
    }
    return;
  }
  if (ya) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < H; i += kPostThreads) {
      const float y = br ? __builtin_fmaf(b, br[i], a * ar[i]) : a * ar[i];
      ss = __builtin_fmaf(y, y, ss);
    }
    ss = block_sum(ss, scratch);
    const float r = 1.f / sqrtf(ss / H + eps);
    for (int i = threadIdx.x; i < H; i += kPostThreads) {
      const float y = br ? __builtin_fmaf(b, br[i], a * ar[i]) : a * ar[i];
      xr[i] = __builtin_fmaf(y * r, w[i], xr[i]);
    }
  }
  if (!out) return;
  for (int i = threadIdx.x; i < H; i += kPostThreads) orow[i] = (OT)xr[i];      // (each thread re-reads what it wrote itself)
}

template <typename T, typename QT, int NQ, int NK>
__global__ __launch_bounds__(kPostThreads) void mix_prep_kernel(
    const float* __restrict__ z, long ldz, int H, int G, int d, int dv, const float* __restrict__ qw, const float* __restrict__ kw,
    float eps, int dims, const float* __restrict__ cos_t, const float* __restrict__ sin_t, int table_pos, int v_unit,
    const float* __restrict__ mix, QT* __restrict__ q_out, long ldqo, T* __restrict__ kcache, int Gk, T* __restrict__ vcache, int v_t,
    const int* __restrict__ tok_pos, const int* __restrict__ tok_seq, const int* __restrict__ block_table, int max_blocks,
    int num_blocks, int table_rows) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int qn = H * d, kn = G * d, vn = G * dv;
  float* ms = sm;                       // the head mix, transposed: [head mixed in][head], 16-byte rows of eight where H allows
  float* qs = sm + (mix ? H * H : 0);
  float* ks = qs + qn;
  float* scratch = ks + kn;
  const int t = blockIdx.x;
  const float* zr = z + (long)t * ldz;
  // A token's first entries of q and k, their norm weights and the way to its cache row are asked for together, ahead of everything that waits
  // (as in post_norm_add: a launch of some hundred tokens lasts as long as one token's loads). With the mix read 16 bytes at a time and
  // dealt over blockIdx.y, fp32, us a launch: 16 heads of 128 on 4 key heads, 1 token 13.4 -> 7.5, 300 15.8 -> 9.8; 32 heads on 8, 64 tokens
  // 37.7 -> 14.6; without a mix 300 tokens 8.0 -> 7.0, 2048 tokens of 32 heads 40.3 -> 34.6. NQ and NK by the length (predicated loads that nobody
  // needs cost a short row 0.5 us: 4 heads of 64, 64 tokens, 4.3 -> 4.8 with eight, 4.25 with one).
  float q0[NQ], k0[NK], wq[NQ], wk[NK];
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int i = threadIdx.x + u * kPostThreads;
    q0[u] = i < qn ? zr[i] : 0.f;
    wq[u] = qw && i < qn ? qw[i] : 0.f;
  }
#pragma unroll
  for (int u = 0; u < NK; ++u) {
    const int i = threadIdx.x + u * kPostThreads;
    k0[u] = i < kn ? zr[qn + i] : 0.f;
    wk[u] = qw && i < kn ? kw[i] : 0.f;
  }
  const int pos = tok_pos[t], slot = tok_seq[t];
  int blk = -1;
  if (slot >= 0 && slot < table_rows && pos >= 0 && pos / kPostBlock < max_blocks) blk = block_table[(long)slot * max_blocks + pos / kPostBlock];
  // rotation: lanes over the pairs of a vector (a power of two of them, so that a wave takes several short vectors), each with its angle's
  // cosine and sine asked for here, once for all vectors
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int half = dims >> 1, lg = half > 32 ? 6 : half > 16 ? 5 : half > 8 ? 4 : half > 4 ? 3 : half > 2 ? 2 : half > 1 ? 1 : 0;
  const int p0 = lane & ((1 << lg) - 1);
  const bool rotate = dims > 0 && pos >= 0 && pos < table_pos;
  const float* cs = cos_t + (rotate ? (long)pos * half : 0);
  const float* sn = sin_t + (rotate ? (long)pos * half : 0);
  const float c0 = rotate && p0 < half ? cs[p0] : 0.f, s0 = rotate && p0 < half ? sn[p0] : 0.f;
  if (mix)
    for (int i = threadIdx.x; i < H * H; i += kPostThreads) ms[i % H * H + i / H] = mix[i];
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int u = 0; u < NQ; ++u) sq = __builtin_fmaf(q0[u], q0[u], sq);
#pragma unroll
  for (int u = 0; u < NK; ++u) sk = __builtin_fmaf(k0[u], k0[u], sk);
  for (int i = threadIdx.x + NQ * kPostThreads; i < qn; i += kPostThreads) { const float v = zr[i]; qs[i] = v; sq = __builtin_fmaf(v, v, sq); }
  for (int i = threadIdx.x + NK * kPostThreads; i < kn; i += kPostThreads) { const float v = zr[qn + i]; ks[i] = v; sk = __builtin_fmaf(v, v, sk); }
  if (qw) {
    sq = block_sum(sq, scratch);
    sk = block_sum(sk, scratch);
    const float rq = 1.f / sqrtf(sq / qn + eps), rk = 1.f / sqrtf(sk / kn + eps);
#pragma unroll
    for (int u = 0; u < NQ; ++u) q0[u] *= rq * wq[u];
#pragma unroll
    for (int u = 0; u < NK; ++u) k0[u] *= rk * wk[u];
    for (int i = threadIdx.x + NQ * kPostThreads; i < qn; i += kPostThreads) qs[i] *= rq * qw[i];      // (a thread's own entries)
    for (int i = threadIdx.x + NK * kPostThreads; i < kn; i += kPostThreads) ks[i] *= rk * kw[i];
  }
#pragma unroll
  for (int u = 0; u < NQ; ++u)
    if ((int)threadIdx.x + u * kPostThreads < qn) qs[threadIdx.x + u * kPostThreads] = q0[u];
#pragma unroll
  for (int u = 0; u < NK; ++u)
    if ((int)threadIdx.x + u * kPostThreads < kn) ks[threadIdx.x + u * kPostThreads] = k0[u];
  __syncthreads();
  if (rotate) {
    const int each = 64 >> lg;
    for (int vec = wave * each + (lane >> lg); vec < H + G; vec += kPostThreads >> lg) {
      float* v = vec < H ? qs + (long)vec * d : ks + (long)(vec - H) * d;
      for (int p = p0; p < half; p += 1 << lg) {
        const float c = p == p0 ? c0 : cs[p], s = p == p0 ? s0 : sn[p];
        const float e = v[p], f = v[p + half];
        v[p] = __builtin_fmaf(e, c, -(f * s));
        v[p + half] = __builtin_fmaf(f, c, e * s);
      }
    }
  }
  __syncthreads();
  if (q_out) {
    QT* qo = q_out + (long)t * ldqo;
    if (mix) {
      // A thread takes one entry (key head c, place i) of the query rows of eight heads at a time: the group's queries at that place
      // are consecutive over the lanes, the mix comes from LDS (every lane of a wave reads the same address: a broadcast, 16 bytes
      // at once), and a wave's stores cover consecutive entries of one head's row. blockIdx.y deals out the eights.
      const int group = H / G, row = G * d;
      const bool vec8 = H % 8 == 0;
      for (int e = threadIdx.x; e < row; e += kPostThreads) {
        const int c = e / d, i = e % d;
        for (int h0 = 8 * blockIdx.y; h0 < H; h0 += 8 * gridDim.y) {
          float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          for (int j = 0; j < group; ++j) {
            const float qv = qs[(c * group + j) * d + i];
            const float* mr = ms + (c * group + j) * H + h0;
            if (vec8) {
              const f32x4 m0 = *reinterpret_cast<const f32x4*>(mr), m1 = *reinterpret_cast<const f32x4*>(mr + 4);
#pragma unroll
              for (int u = 0; u < 8; ++u) acc[u] = __builtin_fmaf(u < 4 ? m0[u] : m1[u - 4], qv, acc[u]);
            } else {
#pragma unroll
              for (int u = 0; u < 8; ++u)
                if (h0 + u < H) acc[u] = __builtin_fmaf(mr[u], qv, acc[u]);
            }
          }
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (h0 + u < H) qo[(long)(h0 + u) * row + e] = (QT)acc[u];
        }
      }
    } else {
      for (int i = threadIdx.x; i < qn; i += kPostThreads) qo[i] = (QT)qs[i];
    }
  }
  if (blockIdx.y > 0 || blk < 0 || blk >= num_blocks) return;
  const int off = pos % kPostBlock, dk = kn / Gk;
  for (int i = threadIdx.x; i < kn; i += kPostThreads) {
    const int g = i / dk, c = i % dk;
    kcache[(((long)blk * Gk + g) * kPostBlock + off) * dk + c] = (T)ks[i];
  }
  // values: a wave per head; v_t: a block holds them key-contiguous, [head][entry][32 tokens]
  const float* vr = zr + qn + kn;
  for (int g = wave; g < G; g += kPostThreads / 64) {
    float r = 1.f;
    if (v_unit) {
      float ss = 0.f;
      for (int c = lane; c < dv; c += 64) { const float v = vr[g * dv + c]; ss += v * v; }
      ss = wave_sum(ss);
      r = 1.f / sqrtf(ss / dv + eps);
    }
    for (int c = lane; c < dv; c += 64) {
      const float v = vr[g * dv + c] * r;
      if (v_t) vcache[(((long)blk * G + g) * dv + c) * kPostBlock + off] = (T)v;
      else vcache[(((long)blk * G + g) * kPostBlock + off) * dv + c] = (T)v;
    }
  }
  (void)vn;
}

}  // namespace dlia

extern "C" void dlia_post_norm_add(void* out, int out_f32, long ldo, float* x, long ldx, const float* ya, long ldya, const float* yb,
                                   long ldyb, float a, float b, const float* w, int T, int H, float eps, hipStream_t stream) {
  if (T <= 0) return;
#define DLIA_POST(OT, N)                                                                                                      \
  hipLaunchKernelGGL((dlia::post_norm_add_kernel<OT, N>), dim3(T), dim3(dlia::kPostThreads), 0, stream, (OT*)out, ldo, x, ldx, ya, ldya, yb, \
                     ldyb, a, b, w, H, eps)
#define DLIA_POST_ROW(OT)                                                                                                     \
  if (H <= 256) DLIA_POST(OT, 1); else if (H <= 512) DLIA_POST(OT, 2); else if (H <= 1024) DLIA_POST(OT, 4);                  \
  else if (H <= 2048) DLIA_POST(OT, 8); else if (H <= 4096) DLIA_POST(OT, 16); else DLIA_POST(OT, 0)
  if (out_f32 || !out) { DLIA_POST_ROW(float); }
  else { DLIA_POST_ROW(dlia::bf16); }
#undef DLIA_POST_ROW
#undef DLIA_POST
}

extern "C" int dlia_mix_prep(const float* z, long ldz, int T, int H, int G, int d, int dv, const float* qw, const float* kw, float eps,
                             int dims, const float* cos_t, const float* sin_t, int table_pos, int v_unit, const float* mix, void* q_out,
                             int q_f32, long ldqo, void* kcache, int Gk, void* vcache, int v_t, int cache_f32, const int* tok_pos,
                             const int* tok_seq, const int* block_table, int max_blocks, int num_blocks, int table_rows,
                             hipStream_t stream) {
  if (T <= 0) return 0;
  const size_t lds = ((size_t)(H + G) * d + 16 + (mix ? (size_t)H * H : 0)) * sizeof(float);
  if (lds > 65536) return 1;
  // the mixed query rows of few tokens: several workgroups a token, each preparing the token and mixing its share of the heads
  int gy = 1;
  while (mix && q_out && 16 * gy <= H && 2 * gy * T <= 1024) gy *= 2;
#define DLIA_PREP_N(CT, QT, NQ, NK)                                                                                            \
  hipLaunchKernelGGL((dlia::mix_prep_kernel<CT, QT, NQ, NK>), dim3(T, gy), dim3(dlia::kPostThreads), lds, stream, z, ldz, H, G, d, dv, qw, kw, eps, dims, cos_t, sin_t, table_pos, v_unit, mix, (QT*)q_out, ldqo, (CT*)kcache, Gk, (CT*)vcache, v_t, tok_pos, tok_seq, \
                     block_table, max_blocks, num_blocks, table_rows)
#define DLIA_PREP(CT, QT)                                                                                                      \
  do {                                                                                                                         \
    if (H * d <= 256) DLIA_PREP_N(CT, QT, 1, 1); else if (H * d <= 512) DLIA_PREP_N(CT, QT, 2, 1);                             \
    else if (H * d <= 1024) DLIA_PREP_N(CT, QT, 4, 1); else DLIA_PREP_N(CT, QT, 8, 2);                                         \
  } while (0)
  if (cache_f32) {
    if (q_f32) DLIA_PREP(float, float); else return 1;
  } else {
    if (q_f32) DLIA_PREP(dlia::bf16, float); else DLIA_PREP(dlia::bf16, dlia::bf16);
  }
#undef DLIA_PREP
#undef DLIA_PREP_N
  return 0;
}
