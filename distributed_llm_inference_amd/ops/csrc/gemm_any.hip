// GEMM for any shape and for row-major (unpacked) weights: C[M,N] = epilogue(A[M,K] . W[N,K]^T + bias), operands in
// bf16 (MFMA 16x16x32, fp32 accumulation) or in fp32 (MFMA 16x16x4 on fp32 operands: products and sums in true
// 32-bit), output in fp32 or in the operand type.
//
// The packed-weight kernels of this library want K in multiples of 128 and N in multiples of 16; models whose
// widths are not (a 200-wide residual stream, the few-row gate projections of a recurrent mixer) and the fp32 mode run
// here. Both operands are K-contiguous, and an MFMA fragment is 16 bytes of one row per lane: lane l of a 16-row tile
// holds row l % 16 at k-chunk l / 16. Three kernels:
//   gemm_any_rows   up to 16 rows, rows in whole 16-byte pieces, long K: a weight stream
//   gemm_any_tile   K in multiples of 128 bytes, rows in whole 16-byte pieces: tiles staged through LDS
//   gemm_any        everything else: fragments straight from memory, edges by zero fragments and guarded stores
//
// epi 0: + bias (optional). epi 1: gated pair — W's 16-row tiles alternate gate, up (`interleave_gate_up`), the
// wave holds both for the same 16 output columns and writes gelu_tanh(gate) * up, N/2 columns wide.
#include "common.h"
#include "frag.h"
#include "launch.h"

namespace dlia {

// accurate tanh-form GELU for the fp32 path (expf, IEEE division); the bf16 path's fast form is in common.h
__device__ __forceinline__ float gelu_tanh_exact(float x) {
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.f + tanhf(u));
}

// The general form: a workgroup of four waves covers a 64 x 64 tile of C (each wave 32 x 32: two row tiles by two column
// tiles, four MFMAs per k-step); the operand panels it shares are served by L1 / L2. Rows that are not 16-byte aligned take
// an element-wise load.
template <typename T, typename OT, int EPI>
__global__ __launch_bounds__(256) void gemm_any_kernel(OT* __restrict__ C, const T* __restrict__ A, const T* __restrict__ W,
                                                       const float* __restrict__ bias, int M, int N, int K, long lda,
                                                       long ldw, long ldc, int vec_ok, long a_step, long w_step, long c_step) {
  constexpr int VEC = 16 / sizeof(T), KS = 4 * VEC;
  // (blockIdx.z: one of several independent products of equal shape, e.g. the blocks of a block-diagonal matrix)
  A += blockIdx.z * a_step; W += blockIdx.z * w_step; C += blockIdx.z * c_step;
  if (bias) bias += (long)blockIdx.z * N;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int m_base = blockIdx.y * 64 + (wave >> 1) * 32, n_base = blockIdx.x * 64 + (wave & 1) * 32;
  if (m_base >= M || n_base >= N) return;
  const int r16 = lane & 15, kq = lane >> 4;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const T* arow[2]; const T* wrow[2]; bool av[2], wv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = m_base + i * 16 + r16, c = n_base + i * 16 + r16;
    av[i] = r < M; wv[i] = c < N;
    arow[i] = A + (long)(av[i] ? r : 0) * lda;
    wrow[i] = W + (long)(wv[i] ? c : 0) * ldw;
  }
  for (int k0 = 0; k0 < K; k0 += KS) {
    const int k = k0 + kq * VEC;
    u32x4 a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) { a[i] = load_frag<T>(arow[i], k, K, av[i], vec_ok); b[i] = load_frag<T>(wrow[i], k, K, wv[i], vec_ok); }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mma_frag(T{}, a[i], b[j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m_base + i * 16 + kq * 4 + r;
      if (row >= M) continue;
      if constexpr (EPI == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int col = n_base + j * 16 + r16;
          if (col < N) C[(long)row * ldc + col] = (OT)(acc[i][j][r] + (bias ? bias[col] : 0.f));
        }
      } else {
        const int cg = n_base + r16, cu = n_base + 16 + r16;
        if (cu < N) {
          const float g = acc[i][0][r] + (bias ? bias[cg] : 0.f), u = acc[i][1][r] + (bias ? bias[cu] : 0.f);
          const float act = sizeof(T) == 4 ? gelu_tanh_exact(g) : gelu_tanh(g);
          C[(long)row * ldc + (n_base >> 1) + r16] = (OT)(act * u);
        }
      }
    }
}

// all tiles of a k-step: in fp32 one k of the four after the other over ALL tiles, so that the products that wait for the same
// accumulator are MT * NT instructions apart
template <int MT, int NT>
__device__ __forceinline__ void mma_tiles(bf16, const u32x4 (&a)[MT], const u32x4 (&b)[NT], f32x4 (&acc)[MT][NT]) {
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
}
template <int MT, int NT>
__device__ __forceinline__ void mma_tiles(float, const u32x4 (&a)[MT], const u32x4 (&b)[NT], f32x4 (&acc)[MT][NT]) {
  f32x4 af[MT], bf[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) af[i] = __builtin_bit_cast(f32x4, a[i]);
#pragma unroll
  for (int j = 0; j < NT; ++j) bf[j] = __builtin_bit_cast(f32x4, b[j]);
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i][e], bf[j][e], acc[i][j], 0, 0, 0);
}

// A BM x BN tile of C per workgroup, both operand panels through a ring of four LDS stages of 128 bytes of K. The general
// kernel issues its next fragment loads only when the last ones have been used, so every k-step waits for L2; here a wave holds
// the fragments of stage s when the barrier opens, asks for those of stage s + 1 and for the loads of stage s + 4 (into the slot that
// everybody has just read), and multiplies: the matrix cores have work at once. (Before, the fragments were read behind the barrier: the
// table's middle column.) A stage is rows of 128 bytes, written by direct LDS loads (1 KiB = 8 rows a piece, whole cache lines of eight
// rows); the 16-byte chunk c of row r sits at c ^ (r / 2 % 8), so that the 16 rows a fragment read touches fall on different banks, of
// which two rows fill all (the swizzle is applied to the address each lane loads FROM). Rows beyond M or N repeat the last one: their
// products are never stored.
// Bound by the fp32 matrix rate in fp32 (a 64 x 64 tile needs 16 bytes of L2 and 32 of LDS per cycle and CU) and by how evenly
// the tiles fall on the CUs. us, general kernel -> fragments behind the barrier -> this one, fp32: 300 rows, N 8192, K 2048 172 -> 118 -> 99;
// N 2048, K 8192 355 -> 128 -> 111; 1024 rows, N = K = 4096 476 -> 317 -> 277 (124 TFLOP/s), 2048 rows 612 -> 515; 64 rows, N 8192, K 2048
// 27 -> 22. bf16: 1024 rows, N = K = 4096 233 -> 61 -> 50; 32 products of 1900 rows, N 448, K 128 61 -> 35 -> 35, N 128, K 448 54 -> 28 -> 23.
//
// KG > 1: the stages are dealt out to KG groups of four waves with a ring each, whose tiles meet in LDS at the end. One tile
// per CU is one wave per SIMD, and a stage is then mostly waiting (barrier, first fragment read).
constexpr int kAnyStages = 4;
template <typename T, typename OT, int EPI, int BM, int BN, int KG>
__global__ __launch_bounds__(256 * KG) void gemm_any_tile_kernel(OT* __restrict__ C, const T* __restrict__ A, const T* __restrict__ W,
                                                                 const float* __restrict__ bias, int M, int N, int K, long lda,
                                                                 long ldw, long ldc, int wide_out, long a_step, long w_step, long c_step) {
  constexpr int BK = 128 / (int)sizeof(T), VEC = 16 / (int)sizeof(T);
  // waves 2 x 2 over the tile; 48 rows: 1 x 4, and the ring keeps 64 (whole pieces for every wave)
  constexpr int WM = BM == 48 ? 1 : 2, WN = 4 / WM, BMP = BM == 48 ? 64 : BM;
  constexpr int MT = BM / WM / 16, NT = BN / WN / 16;             // 16-wide tiles of a wave
  constexpr int P = (BMP + BN) / 32;                              // pieces per wave and stage
  constexpr int kStage = (BMP + BN) * 128;
  __shared__ __attribute__((aligned(1024))) char lds[KG * kAnyStages * kStage];
  A += blockIdx.z * a_step; W += blockIdx.z * w_step; C += blockIdx.z * c_step;
  if (bias) bias += (long)blockIdx.z * N;
  const int group = threadIdx.x >> 8, wave = (threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int r16 = lane & 15, kq = lane >> 4;
  char* ring = lds + group * (kAnyStages * kStage);
  // the pieces this wave brings in: piece p of a stage holds its rows 8 p .. 8 p + 7 (A's rows, then W's)
  const T* src[P];
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int row = (wave * P + q) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    src[q] = row < BMP ? A + (long)min(m0 + row, M - 1) * lda + chunk * VEC : W + (long)min(n0 + row - BMP, N - 1) * ldw + chunk * VEC;
  }
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)ring + wave * P * 1024;
  // stage i of this group: K-step i KG + group (asked for in order: the sources walk along)
  const int steps = K / BK, nk = (steps - group + KG - 1) / KG, rounds = (steps + KG - 1) / KG;
#pragma unroll
  for (int q = 0; q < P; ++q) src[q] += group * BK;
  auto fetch = [&](int slot) {
    const void* g[P];
#pragma unroll
    for (int q = 0; q < P; ++q) { g[q] = src[q]; src[q] += KG * BK; }
    lds_dma_run<P>(g, __builtin_amdgcn_readfirstlane(lds_base + slot * kStage));
  };
#pragma unroll
  for (int i = 0; i < kAnyStages; ++i)
    if (i < nk) fetch(i);
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
  struct Frags { u32x4 a[2][MT], b[2][NT]; };
  const int at = r16 * 128, sw = (r16 >> 1) & 7;                  // (tiles start at multiples of 16 rows: the swizzle is the lane's own)
  auto read = [&](Frags& f, int slot) {
    const char* st = ring + slot * kStage + at;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = ((kk * 4 + kq) ^ sw) << 4;
#pragma unroll
      for (int i = 0; i < MT; ++i) f.a[kk][i] = ld16(st + (wm + i * 16) * 128 + c);
#pragma unroll
      for (int j = 0; j < NT; ++j) f.b[kk][j] = ld16(st + (BMP + wn + j * 16) * 128 + c);
    }
  };
  // own reads are done and own pieces have landed; the barrier makes it everybody's
  auto meet = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto landed = [&](int behind) {                                 // all but the last `behind` stages asked for
    if (behind >= 3) wait_pieces<3 * P>();
    else if (behind == 2) wait_pieces<2 * P>();
    else if (behind == 1) wait_pieces<P>();
    else wait_pieces<0>();
  };
  Frags f0, f1;
  landed(nk - 1);
  meet();
  read(f0, 0);
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) mma_tiles<MT, NT>(T{}, f.a[kk], f.b[kk], acc);
  };
  // (a group may have one stage less than the others: it then reads a slot that nothing was asked for, and does not multiply it)
  auto step = [&](int s, const Frags& now, Frags& next) {
    landed(nk - 2 - s < 2 ? nk - 2 - s : 2);
    meet();
    read(next, (s + 1) % kAnyStages);
    if (s + kAnyStages < nk) fetch(s % kAnyStages);               // (everybody holds stage s)
    multiply(now);
  };
  // Rounds of four stages with nothing conditional in them (a branch around the loads makes the compiler wait for the fragments just
  // asked for); what is left goes step by step.
  auto steady = [&](int slot, const Frags& now, Frags& next) {
    wait_pieces<2 * P>();
    meet();
    read(next, (slot + 1) % kAnyStages);
    fetch(slot);
    multiply(now);
  };
  static_assert(kAnyStages == 4, "the slots of a round of steps");
  int s = 0;
  const int least = steps / KG;                                   // (stages that every group has)
  for (; s + 2 * kAnyStages - 1 < least; s += kAnyStages) { steady(0, f0, f1); steady(1, f1, f0); steady(2, f0, f1); steady(3, f1, f0); }
  for (; s + 2 < rounds; s += 2) { step(s, f0, f1); step(s + 1, f1, f0); }
  if (s + 1 < rounds) {
    step(s, f0, f1);
    if (KG == 1 || s + 1 < nk) multiply(f1);
  } else if (KG == 1 || s < nk) {
    multiply(f0);
  }
  if constexpr (KG > 1) {
    f32x4* part = reinterpret_cast<f32x4*>(lds);                  // [group - 1][wave][tile][lane]
    __syncthreads();
    if (group) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) part[((((group - 1) * 4 + wave) * MT + i) * NT + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (group) return;
#pragma unroll
    for (int g = 0; g < KG - 1; ++g)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] += part[(((g * 4 + wave) * MT + i) * NT + j) * 64 + lane];
  }
  if constexpr (EPI == 0 && sizeof(OT) == 2 && KG == 1) {
    // 16-bit output: a lane's values are one column of four rows, 32 bytes of a row per store instruction. Through LDS they
    // leave as 16-byte pieces of whole rows.
    if (wide_out) {
      constexpr int LDO = BN + 8;
      OT* o = reinterpret_cast<OT*>(lds);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int col = n0 + wn + j * 16 + r16;
          const float bv = bias && col < N ? bias[col] : 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[(wm + i * 16 + kq * 4 + r) * LDO + wn + j * 16 + r16] = (OT)(acc[i][j][r] + bv);
        }
      __syncthreads();
      for (int e = threadIdx.x; e < BM * (BN / 8); e += 256) {
        const int row = e / (BN / 8), c8 = (e % (BN / 8)) * 8;
        if (m0 + row < M && n0 + c8 < N) st16(C + (long)(m0 + row) * ldc + n0 + c8, ld16(o + row * LDO + c8));
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + wm + i * 16 + kq * 4 + r;
      if (row >= M) continue;
      if constexpr (EPI == 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int col = n0 + wn + j * 16 + r16;
          if (col < N) C[(long)row * ldc + col] = (OT)(acc[i][j][r] + (bias ? bias[col] : 0.f));
        }
      } else {
        static_assert(EPI == 0 || NT == 2, "a wave holds a gate tile and its up tile");
        const int cg = n0 + wn + r16, cu = cg + 16;
        if (cu < N) {
          const float g = acc[i][0][r] + (bias ? bias[cg] : 0.f), u = acc[i][NT - 1][r] + (bias ? bias[cu] : 0.f);
          const float act = sizeof(T) == 4 ? gelu_tanh_exact(g) : gelu_tanh(g);
          C[(long)row * ldc + ((n0 + wn) >> 1) + r16] = (OT)(act * u);
        }
      }
    }
}

// Up to 16 rows: a stream of W. 16 NT columns per workgroup and ALL of K inside it, dealt out to its eight waves 256 bytes of
// every row at a time (whole cache lines), each wave with its next piece on its way while it multiplies the last one;
// the eight partial tiles meet in LDS and are added in the order of the waves. (In the general kernel one wave walks all of K
// with one k-step of loads in flight, and N / 64 workgroups are too few to keep HBM busy.)
template <typename T, typename OT, int EPI, int NT>
__global__ __launch_bounds__(512) void gemm_any_rows_kernel(OT* __restrict__ C, const T* __restrict__ A, const T* __restrict__ W,
                                                            const float* __restrict__ bias, int M, int N, int K, long lda,
                                                            long ldw, long ldc, long a_step, long w_step, long c_step) {
  constexpr int VEC = 16 / (int)sizeof(T), KS = 4 * VEC, U = 4, CH = U * KS, NW = 8;
  __shared__ f32x4 part[NW][NT][64];
  A += blockIdx.z * a_step; W += blockIdx.z * w_step; C += blockIdx.z * c_step;
  if (bias) bias += (long)blockIdx.z * N;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4, n0 = blockIdx.x * 16 * NT;
  const bool av = r16 < M;
  const T* arow = A + (long)(av ? r16 : 0) * lda;
  const T* wrow[NT]; bool wv[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) { const int c = n0 + j * 16 + r16; wv[j] = c < N; wrow[j] = W + (long)(wv[j] ? c : 0) * ldw; }
  f32x4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 w[2][U][NT], a[2][U];
  auto fetch = [&](int to, int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * KS + kq * VEC;
#pragma unroll
      for (int j = 0; j < NT; ++j) w[to][u][j] = load_frag<T>(wrow[j], k, K, wv[j], true);
      a[to][u] = load_frag<T>(arow, k, K, av, true);
    }
  };
  auto mul = [&](int from) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = mma_frag(T{}, a[from][u], w[from][u][j], acc[j]);
  };
  // (chunks beyond K load nothing and multiply zeros)
  int k0 = wave * CH;
  fetch(0, k0);
  for (; k0 < K; k0 += 2 * NW * CH) {
    fetch(1, k0 + NW * CH);
    mul(0);
    fetch(0, k0 + 2 * NW * CH);
    mul(1);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) part[wave][j][lane] = acc[j];
  __syncthreads();
  if (wave >= (EPI == 0 ? NT : 1)) return;                 // one wave per column tile, or for the gate / up pair
  f32x4 s[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    s[j] = part[0][EPI == 0 ? wave : j][lane];
#pragma unroll
    for (int q = 1; q < NW; ++q) s[j] += part[q][EPI == 0 ? wave : j][lane];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = kq * 4 + r;
    if (row >= M) continue;
    if constexpr (EPI == 0) {
      const int col = n0 + wave * 16 + r16;
      if (col < N) C[(long)row * ldc + col] = (OT)(s[0][r] + (bias ? bias[col] : 0.f));
    } else {
      static_assert(EPI == 0 || NT == 2, "a workgroup holds a gate tile and its up tile");
      const int cg = n0 + r16, cu = cg + 16;
      if (cu < N) {
        const float g = s[0][r] + (bias ? bias[cg] : 0.f), u = s[NT - 1][r] + (bias ? bias[cu] : 0.f);
        const float act = sizeof(T) == 4 ? gelu_tanh_exact(g) : gelu_tanh(g);
        C[(long)row * ldc + (n0 >> 1) + r16] = (OT)(act * u);
      }
    }
  }
}

// The unfused form of the gated epilogue, for activations that a packed-weight GEMM left as [M, 2F] (gate columns,
// then up columns, bias already added): act[m, j] = gelu_tanh(gu[m, j]) * gu[m, F + j]. Eight columns per lane.
__global__ __launch_bounds__(256) void gated_gelu_kernel(bf16* __restrict__ act, const bf16* __restrict__ gu, int M, int F,
                                                         long ldg, long lda) {
  const int per_row = F >> 3;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)M * per_row) return;
  const int m = (int)(i / per_row), c = (int)(i % per_row) * 8;
  float g[8], u[8];
  unpack8(ld16(gu + (long)m * ldg + c), g);
  unpack8(ld16(gu + (long)m * ldg + F + c), u);
#pragma unroll
  for (int j = 0; j < 8; ++j) g[j] = gelu_tanh(g[j]) * u[j];
  st16(act + (long)m * lda + c, pack8(g));
}

}  // namespace dlia

// The kernel that a product takes where its rows are in whole 16-byte pieces: 0 the general one, 1 the weight stream, a tile of BM x BN with KG groups
// of waves as 1000 BM + 10 BN + KG. The tile is the one whose rounds over the 256 CUs take least; what a round of each costs relative to 64 x
// 64 is measured (fp32, K 4096: 77, 60, 45 and 25 us; 28 where a CU has one 32 x 32 tile to itself). bf16 chooses by the same numbers: of
// 159 shapes (17 to 2048 rows, N and K 64 to 8192) of either type the tile taken was within 8 % of the best of the four, but for 400 rows,
// N 8192, K 2048 (bf16 40 us where 64 x 64 takes 34, fp32 166 and 152).
extern "C" int dlia_gemm_any_form(int M, int N, int K, int blocks, int f32, int epi, int out_f32) {
  const int bk = f32 ? 32 : 64;
  if (M <= 16 && K >= 8 * bk) return 1;
  if (K % bk) return 0;
  auto rounds = [&](int bm, int bn) { return (int)(((long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * blocks + 255) / 256); };
  const int r66 = rounds(64, 64), r46 = rounds(48, 64), r36 = rounds(32, 64), r33 = rounds(32, 32);
  const double t66 = r66, t46 = epi == 0 ? r46 * 0.77 : 1e30, t36 = r36 * 0.58, t33 = epi == 0 ? (r33 == 1 ? 0.36 : r33 * 0.33) : 1e30;
  // (a single stage and the chip full: the stores are what is left, in fp32 the general kernel's have less in front of them. fp32, 2048 rows, N 4096, K 32
  // 19.1 us, the general kernel 16.4; 16-bit operands, K 64, 32 products of 1900 rows, N 640: fp32 out 65.6, 51.7, 16-bit out the tiles take 0.9 of it over 40 shapes)
  if ((f32 || out_f32) && K == bk && r66 >= 4) return 0;
  const bool split = K >= 16 * bk;             // (below that the rings are filled once or twice: nothing to hide)
  const double best = r66 > 6 ? t66 : fmin(fmin(t66, t46), fmin(t36, t33));        // (with many rounds the last one is small change: 32 products of 1900 rows, N 128, K 448 23 us, in tiles of 48 rows 27)
  if (t66 == best) return split && r66 == 1 ? 64642 : 64641;
  if (t36 == best) return split && r36 == 1 ? 32642 : 32641;
  if (t46 == best) return split && r46 == 1 ? 48642 : 48641;
  return split && r33 == 1 ? 32324 : split && r33 == 2 ? 32322 : 32321;
}

namespace dlia {

#define DLIA_ANY_ARGS (OT*)C, (const T*)A, (const T*)W, bias, M, N, K, lda, ldw, ldc

template <typename T, typename OT, int EPI>
static void launch_any_epi(void* C, const void* A, const void* W, const float* bias, int M, int N, int K, long lda, long ldw, long ldc,
                           hipStream_t stream, int blocks, long a_step, long w_step, long c_step) {
  constexpr int VEC = 16 / sizeof(T);
  const int vec_ok = K % VEC == 0 && lda % VEC == 0 && ldw % VEC == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                     a_step % VEC == 0 && w_step % VEC == 0;
  const int form = vec_ok ? dlia_gemm_any_form(M, N, K, blocks, sizeof(T) == 4, EPI, sizeof(OT) == 4) : 0;
  if (form == 1) {
    constexpr int NT = EPI == 0 ? 1 : 2;
    hipLaunchKernelGGL((gemm_any_rows_kernel<T, OT, EPI, NT>), dim3((N + 16 * NT - 1) / (16 * NT), 1, blocks), dim3(512), 0, stream, DLIA_ANY_ARGS, a_step, w_step, c_step);
    return;
  }
  if (form) {
    const int wide = N % 8 == 0 && ldc % 8 == 0 && c_step % 8 == 0 && (uintptr_t)C % 16 == 0;
#define DLIA_ANY_TILE(BM, BN, KG, E)                                                                                                       \
  hipLaunchKernelGGL((gemm_any_tile_kernel<T, OT, E, BM, BN, KG>), dim3((N + BN - 1) / BN, (M + BM - 1) / BM, blocks), dim3(256 * KG), 0, \
                     stream, DLIA_ANY_ARGS, wide, a_step, w_step, c_step)
    switch (form) {
      case 64642: DLIA_ANY_TILE(64, 64, 2, EPI); break;
      case 64641: DLIA_ANY_TILE(64, 64, 1, EPI); break;
      case 32642: DLIA_ANY_TILE(32, 64, 2, EPI); break;
      case 32641: DLIA_ANY_TILE(32, 64, 1, EPI); break;
      case 48642: DLIA_ANY_TILE(48, 64, 2, 0); break;
      case 48641: DLIA_ANY_TILE(48, 64, 1, 0); break;
      case 32324: DLIA_ANY_TILE(32, 32, 4, 0); break;
      case 32322: DLIA_ANY_TILE(32, 32, 2, 0); break;
      default: DLIA_ANY_TILE(32, 32, 1, 0);
    }
#undef DLIA_ANY_TILE
    return;
  }
  hipLaunchKernelGGL((gemm_any_kernel<T, OT, EPI>), dim3((N + 63) / 64, (M + 63) / 64, blocks), dim3(256), 0, stream, DLIA_ANY_ARGS, vec_ok,
                     a_step, w_step, c_step);
}

template <typename T, typename OT>
static void launch_any(void* C, const void* A, const void* W, const float* bias, int M, int N, int K, long lda, long ldw,
                       long ldc, int epi, hipStream_t stream, int blocks = 1, long a_step = 0, long w_step = 0, long c_step = 0) {
  if (epi == 0) launch_any_epi<T, OT, 0>(C, A, W, bias, M, N, K, lda, ldw, ldc, stream, blocks, a_step, w_step, c_step);
  else launch_any_epi<T, OT, 1>(C, A, W, bias, M, N, K, lda, ldw, ldc, stream, blocks, a_step, w_step, c_step);
}

}  // namespace dlia

extern "C" void dlia_gated_gelu(void* act, const void* gu, int M, int F, long ldg, long lda, hipStream_t stream) {
  if (M <= 0 || F <= 0) return;
  const long n = (long)M * (F >> 3);
  hipLaunchKernelGGL(dlia::gated_gelu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, (dlia::bf16*)act,
                     (const dlia::bf16*)gu, M, F, ldg, lda);
}

extern "C" void dlia_gemm_any(void* C, int out_f32, const void* A, const void* W, int in_f32, const float* bias, int M, int N,
                              int K, long lda, long ldw, long ldc, int epi, hipStream_t stream) {
  if (M <= 0 || N <= 0) return;
  if (in_f32)
    dlia::launch_any<float, float>(C, A, W, bias, M, N, K, lda, ldw, ldc, epi, stream);
  else if (out_f32)
    dlia::launch_any<dlia::bf16, float>(C, A, W, bias, M, N, K, lda, ldw, ldc, epi, stream);
  else
    dlia::launch_any<dlia::bf16, dlia::bf16>(C, A, W, bias, M, N, K, lda, ldw, ldc, epi, stream);
}

extern "C" void dlia_gemm_blocks(void* C, int out_f32, const void* A, const void* W, int in_f32, const float* bias, int M, int N,
                                 int K, long lda, long ldw, long ldc, int blocks, long a_step, long w_step, long c_step,
                                 hipStream_t stream) {
  if (M <= 0 || N <= 0 || blocks <= 0) return;
  if (in_f32)
    dlia::launch_any<float, float>(C, A, W, bias, M, N, K, lda, ldw, ldc, 0, stream, blocks, a_step, w_step, c_step);
  else if (out_f32)
    dlia::launch_any<dlia::bf16, float>(C, A, W, bias, M, N, K, lda, ldw, ldc, 0, stream, blocks, a_step, w_step, c_step);
  else
    dlia::launch_any<dlia::bf16, dlia::bf16>(C, A, W, bias, M, N, K, lda, ldw, ldc, 0, stream, blocks, a_step, w_step, c_step);
}
