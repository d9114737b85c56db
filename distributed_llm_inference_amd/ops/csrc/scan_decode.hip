// One token per sequence through the linear recurrences over a matrix state (the rules of delta_rule.hip and state_scan.hip). A
// decode step reads and writes every sequence's whole state once and does next to nothing with it: what counts is how many of its
// bytes are on their way. A workgroup owns a (head, sequence), asks for the whole state at once and then forms the token's vectors:
//
//   rule 0, generalised delta rule   S <- diag(w) S - (a u) (u^T S) + k v^T;  o = S^T r
//   rule 2, gated delta rule         S <- g S;  S <- S + k (beta (v - S^T k))^T;  o = S^T q
//       square states of 128 (rule 0: of 64 too) in whole 16-byte pieces: thread (row group, 4 columns) holds 16 (4) rows of its
//       columns; the two sums over rows meet in LDS. 32 heads of 128 x 128: 64 sequences (268 MB) rule 0 146 -> 59 us, rule 2 91 -> 59 us;
//       4 sequences 14.2 -> 8.0 and 7.5 -> 6.6 us; one 10.3 -> 6.8 and 6.0 -> 5.3. Rule 2 on states of 64 x 64, 64 x 128 and 128 x 64 stays
//       with the general kernel (a form of this one for any size: 1.1 to 1.6 times its time).
//   rule 1, matrix memory            S <- keep S + put k v^T, the normaliser n as the last column of every row
//       rows of dv + 1 entries are not 16-byte aligned: thread (row group, column), 16 rows in flight; the normaliser's column is
//       a thread's per row. 16 heads of 128 x 129: 64 sequences (135 MB) 85 -> 38 us, 4 sequences 10.5 -> 8.8 us.
// (Calls on states that are not in the caches. The general kernels keep 16 rows of a column per lane and as many lanes
// per column as that takes, so a load instruction touches 64 / R columns of R rows 16 apart: 4-byte accesses, a quarter or an eighth
// of a cache line each. They stay for prompts and other sizes.) A sequence that has more tokens than one all the same runs them in turn.
// Error against 64 bits (relative 2-norm, random states), general kernels -> these: read-outs, rule 0 0.87e-7 .. 0.92e-7 -> 0.55e-7 .. 0.71e-7, rule 1
// 0.89e-7 .. 1.2e-7 -> 0.58e-7 .. 0.74e-7, rule 2 0.93e-7 -> 0.84e-7; states, rule 1 4.1e-8 .. 4.8e-8 -> 3.2e-8 .. 3.9e-8, the others the same. Hence the
// short chains, the 64-bit sums and, in rule 1, the 64-bit products below: with a thread's rows in one 32-bit chain the read-outs had up
// to 1.6 and the memory's states up to 1.8 times the general kernels' error.
#include "units.h"
#include "launch.h"

namespace dlia {

struct DecScanArgs {
  float* o; long ldo;
  const float* x; long ldx;              // q (or r), k, v
  const float* z; long ldz;              // gates
  const float* wz; long ldw;
  float* state; float* mstate;
  const float* b0; const float* b1;
  const int* q_start; const int* ctx; const int* slots;
  int H, per, d, dv, state_rows;
  int col_q, col_k, col_v, col_a, col_b;
  float cap, qscale;
};

constexpr int kDecRows = 16;

template <int RULE, int D>
__global__ __launch_bounds__(256) void scan_decode_kernel(DecScanArgs p) {
  constexpr int CT = D / 4, RG = 256 / CT, ROWS = D / RG;      // threads across the columns, row groups, rows of a thread
  __shared__ float vec[5][D];                        // w, a u, u, k, q (rule 2: k, q)
  __shared__ f32x4 red[2][256];
  __shared__ float scratch[16];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, ct = tid % CT;
  const int t0 = p.q_start[b], t1 = p.q_start[b + 1], slot = p.slots[b];
  if (t1 <= t0 || slot < 0 || slot >= p.state_rows) return;
  bool fresh = p.ctx[b] <= 0;
  int rg = tid / CT;
  float* S = p.state + ((long)slot * p.H + h) * (long)D * D + ct * 4;
  const int hk = h / p.per;
  for (int t = t0; t < t1; ++t) {
    asm volatile("" : "+v"(rg), "+v"(S));            // (nothing is kept from token to token: offsets held over the loop would take the registers)
    f32x4 s[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) s[i] = !fresh ? *reinterpret_cast<const f32x4*>(S + (rg + i * RG) * D) : f32x4{0.f, 0.f, 0.f, 0.f};
    const float* xr = p.x + (long)t * p.ldx;
    const f32x4 v = *reinterpret_cast<const f32x4*>(xr + p.col_v + (long)h * D + ct * 4);
    float g = 1.f, beta = 0.f;
    float k = 0.f, q = 0.f;
    if (tid < D) { k = xr[p.col_k + (long)hk * D + tid]; q = xr[p.col_q + (long)hk * D + tid]; }
    if constexpr (RULE == 0) {
      const float ksq = block_sum(k * k, scratch), inv = rsqrtf(ksq + 1e-6f);
      if (tid < D) {
        const int c = h * D + tid;
        const float a = 1.f / (1.f + expf(-(p.z[(long)t * p.ldz + p.col_a + c] + p.b0[c])));
        const float w = expf(-0.6065306597126334f / (1.f + expf(-(p.wz[(long)t * p.ldw + c] + p.b1[c]))));
        vec[0][tid] = w; vec[1][tid] = a * (k * inv); vec[2][tid] = k * inv; vec[3][tid] = k; vec[4][tid] = q;
      }
    } else {
      const float a = p.z[(long)t * p.ldz + p.col_a + h] + p.b1[h];
      g = expf(-expf(p.b0[h]) * (a > 20.f ? a : log1pf(expf(a))));
      beta = 1.f / (1.f + expf(-p.z[(long)t * p.ldz + p.col_b + h]));
      if (tid < D) { vec[2][tid] = vec[3][tid] = k; vec[4][tid] = q; }
    }
    __syncthreads();
    // (each sum over the rows: two chains in a thread, then the row groups' parts in 64 bits)
    auto groups = [&](const f32x4* parts) {
      f64x4 a = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int i = 0; i < RG; ++i) a += __builtin_convertvector(parts[i * CT + ct], f64x4);
      return __builtin_convertvector(a, f32x4);
    };
    f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      if (RULE == 2) s[i] *= g;
      (i & 1 ? p1 : p0) += s[i] * vec[2][rg + i * RG];
    }
    red[0][tid] = p0 + p1;
    __syncthreads();
    const f32x4 dot = groups(red[0]), u = beta * (v - dot);      // (u: rule 2)
    p0 = p1 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int r = rg + i * RG;
      if constexpr (RULE == 0) s[i] = vec[0][r] * s[i] - vec[1][r] * dot + vec[3][r] * v;
      else s[i] += vec[3][r] * u;
      *reinterpret_cast<f32x4*>(S + r * D) = s[i];
      (i & 1 ? p1 : p0) += vec[4][r] * s[i];
    }
    red[1][tid] = p0 + p1;
    __syncthreads();
    if (tid < CT) *reinterpret_cast<f32x4*>(p.o + (long)t * p.ldo + (long)h * D + tid * 4) = groups(red[1]);
    fresh = false;
  }
}

__global__ __launch_bounds__(1024) void memory_decode_kernel(DecScanArgs p) {
  __shared__ float kv[512], qv[512];
  __shared__ double red[1024];
  __shared__ float scratch[16];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, NT = blockDim.x;
  const int t0 = p.q_start[b], t1 = p.q_start[b + 1], slot = p.slots[b];
  if (t1 <= t0 || slot < 0 || slot >= p.state_rows) return;
  bool fresh = p.ctx[b] <= 0;
  const int d = p.d, dv = p.dv, NC = dv + 1, CT = (dv + 63) / 64 * 64, c = tid % CT, rg = tid / CT;
  int RG = NT / CT;
  float* S = p.state + ((long)slot * p.H + h) * (long)d * NC;
  float* mst = p.mstate + ((long)slot * p.H + h) * 128;
  float s[kDecRows];
  auto load = [&](int r0) {
#pragma unroll
    for (int i = 0; i < kDecRows; ++i) { const int r = r0 + i * RG; s[i] = r < d && c < dv && !fresh ? S[(long)r * NC + c] : 0.f; }
  };
  for (int t = t0; t < t1; ++t) {
    asm volatile("" : "+s"(RG));                     // (as above)
    load(rg);
    const float* xr = p.x + (long)t * p.ldx;
    const float* zr = p.z + (long)t * p.ldz;
    const float m0 = fresh ? 0.f : mst[0];
    const float vc = c < dv ? xr[p.col_v + (long)h * dv + c] : 0.f;
    // the vectors and the normaliser: a thread per row
    const bool row = tid < d;
    const float n0 = row && !fresh ? S[(long)tid * NC + dv] : 0.f;
    const float k = row ? xr[p.col_k + (long)h * d + tid] : 0.f, q = row ? xr[p.col_q + (long)h * d + tid] * p.qscale : 0.f;
    const float fg = p.cap * tanhf((zr[p.col_a + h] + p.b0[p.H + h]) / p.cap);
    float li = p.cap * tanhf((zr[p.col_b + h] + p.b0[h]) / p.cap), lf = fg >= 0.f ? -log1pf(expf(-fg)) : fg - log1pf(expf(fg));
    asm volatile("" : "+v"(li), "+v"(lf));           // (rounded here: fused into one of the sums below and not the other, the maximum's own term would not cancel)
    const float m1 = fmaxf(lf + m0, li), keep = expf(lf + m0 - m1), put = expf(li - m1);
    const float nn = (float)((double)keep * n0 + (double)put * k);
    if (row) { kv[tid] = k; qv[tid] = q; S[(long)tid * NC + dv] = nn; }
    const float nq = block_sum(row ? nn * q : 0.f, scratch);      // (its barriers publish the vectors too)
    // keep s + put k v is rounded once: the products in 64 bits, the sum over the rows in four chains of four, those in 64 bits
    const double v = (double)put * vc, keepd = keep;
    double out = 0.0;
    for (int r0 = rg;;) {
      float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < kDecRows; ++i) {
        const int r = r0 + i * RG;
        if (r >= d || c >= dv) break;
        s[i] = (float)(keepd * s[i] + v * kv[r]);
        part[i & 3] += qv[r] * s[i];
        S[(long)r * NC + c] = s[i];
      }
      out += ((double)part[0] + part[1]) + ((double)part[2] + part[3]);
      r0 += RG * kDecRows;
      if (r0 >= d) break;
      load(r0);
    }
    red[tid] = out;
    __syncthreads();
    float* orow = p.o + (long)t * p.ldo + (long)h * (dv + 2);
    if (tid < CT && c < dv) {
      for (int i = 1; i < RG; ++i) out += red[i * CT + tid];
      orow[c] = (float)out;
    }
    if (tid == 0) { orow[dv] = nq; orow[dv + 1] = expf(-m1); }
    if (tid < 128) mst[tid] = m1;                      // (every copy: this step has one column block)
    fresh = false;
    __syncthreads();                                 // the running maximum, the vectors and the sums of this token
  }
}

}  // namespace dlia

using dlia::DecScanArgs;

// The sizes that take the step kernels. The memory's workgroup owns a (head, sequence) whole, so few of them on wide states leave most of the
// chip without work: 8 heads of 128 x 257, 4 / 6 / 8 sequences 11.2 / 11.6 / 11.9 us against 10.2 / 11.9 / 12.7 of the general kernel's column
// blocks, 2 of 512 x 257, 8 / 24 sequences 28 / 37 against 22 / 64 (64 x 257: 7.7 against 9.9 from one sequence on).
extern "C" int dlia_scan_decode_takes(int rule, long B, int H, int d, int dv) {
  if (B <= 0 || B > 65535) return 0;
  if (rule == 1) return d <= 512 && dv <= 256 && (dv <= 128 || d <= 64 || B * H >= 48);
  return d == dv && (d == 128 || (rule == 0 && d == 64));
}

// Steps of single tokens. 0: launched; 1: sizes or layout that the general kernels take.
extern "C" int dlia_scan_decode(int rule, float* o, long ldo, const float* x, long ldx, const float* z, long ldz, const float* wz, long ldw,
                                float* state, float* mstate, const float* b0, const float* b1, const int* q_start, const int* ctx,
                                const int* slots, int B, int H, int per, int d, int dv, int state_rows, int col_q, int col_k, int col_v, int col_a,
                                int col_b, float cap, float qscale, hipStream_t stream) {
  const DecScanArgs p{o, ldo, x, ldx, z, ldz, wz, ldw, state, mstate, b0, b1, q_start, ctx, slots, H, per, d, dv, state_rows, col_q, col_k, col_v,
                      col_a, col_b, cap, qscale};
  if (!dlia_scan_decode_takes(rule, B, H, d, dv)) return 1;
  auto al = [](const void* q) { return (uintptr_t)q % 16 == 0; };
  if (rule == 1) {
    // Row groups: every row in flight with up to 1024 threads while the chip has fewer workgroups than two a CU, batches of rows with
    // 256 from there on, a thread per row at least. 16 heads of 128 x 129, 4 / 16 / 64 / 160 sequences: 9.1 / 12.0 / 45.8 / 103 us with
    // 1024 threads, 12.3 / 15.9 / 38.3 / 88 with 256.
    const int CT = (dv + 63) / 64 * 64, most = (long)B * H < 512 ? 1024 : 256;
    int rg = (d + dlia::kDecRows - 1) / dlia::kDecRows;
    while (rg > 2 && rg * CT > most) --rg;
    while (rg * CT < d) ++rg;
    hipLaunchKernelGGL(dlia::memory_decode_kernel, dim3(H, B), dim3(CT * (rg < 2 ? 2 : rg)), 0, stream, p);
    return 0;
  }
  if (ldx % 4 || ldo % 4 || col_v % 4 || !al(x) || !al(o) || !al(state)) return 1;
  if (rule == 2) hipLaunchKernelGGL((dlia::scan_decode_kernel<2, 128>), dim3(H, B), dim3(256), 0, stream, p);
  else if (d == 128) hipLaunchKernelGGL((dlia::scan_decode_kernel<0, 128>), dim3(H, B), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((dlia::scan_decode_kernel<0, 64>), dim3(H, B), dim3(256), 0, stream, p);
  return 0;
}
