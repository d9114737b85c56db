// Row kernels of stacks with dynamic-tanh norms and gated residuals; the residual stream is fp32.
//
//   embed_pos32     x[t] = table[ids[t]] + ptable[pos[t]]                          (learned positions)
//   dyt_gate        x += sigmoid(gl + gb) * y;  x += step;  out = tanh(alpha x) w + b     one workgroup per row, one launch
//                   for a sublayer's gated residual add, the vector that opens a pass of a repeated stretch of layers, and the
//                   next sublayer's norm. y is one stream, or the mean of two streams that are RMS-normed over the row first
//                   (y = (rms(ya) wa + rms(yb) wb) / 2). Every part is optional; rows can be gathered for the output.
//   headnorm_gate   per (token, head): v = o / (max(|nq|, em) + 1e-6) when the head's read-out carries its two normaliser
//                   columns [dv | nq | em], then out = v / rms(v) * w[head, :] * sigmoid(gate)
//   unary_act       act = f(x) of an fp32 GEMM output, f the exact GELU x Phi(x) (kind 0) or tanh (kind 1)
//   softcap         logits <- cap tanh(logits / cap), in place
#include "units.h"
#include "launch.h"

namespace dlia {

template <typename TT>
__global__ __launch_bounds__(1024) void embed_pos32_kernel(float* __restrict__ out, const int* __restrict__ ids,
                                                          const int* __restrict__ pos, const TT* __restrict__ table,
                                                          const TT* __restrict__ ptable, int H, int vocab, int max_pos, int vec) {
  const int t = blockIdx.x;
  int id = ids[t], ps = pos[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);   // never fault on a bad id or position
  ps = ps < 0 ? 0 : (ps >= max_pos ? max_pos - 1 : ps);
  const TT* a = table + (long)id * H;
  const TT* b = ptable + (long)ps * H;
  float* dst = out + (long)t * H;
  if (vec) {      // four entries a thread, one pass
    for (int i = threadIdx.x * 4; i < H; i += blockDim.x * 4) {
      Unit<4> u = ldu4(a + i);
      const Unit<4> q = ldu4(b + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) u.v[e] += q.v[e];
      stu<4>(dst + i, u);
    }
    return;
  }
  for (int i = threadIdx.x; i < H; i += blockDim.x) dst[i] = (float)a[i] + (float)b[i];
}

template <typename OT>
__global__ __launch_bounds__(256) void dyt_gate_kernel(
    OT* __restrict__ out, float* __restrict__ x, const float* __restrict__ ya, const float* __restrict__ yb,
    const float* __restrict__ wa, const float* __restrict__ wb, const float* __restrict__ gl, const float* __restrict__ gb,
    const float* __restrict__ step, const float* __restrict__ nw, const float* __restrict__ nb, const int* __restrict__ row_idx,
    int H, long ldx, long ldy, long ldg, long ldo, float alpha, float eps) {
  __shared__ float scratch[16];
  const int orow = blockIdx.x;
  const long irow = row_idx ? row_idx[orow] : orow;
  float* xr = x + irow * ldx;
  if (ya) {
    const float* ar = ya + irow * ldy;
    const float* br = yb ? yb + irow * ldy : nullptr;
    float ra = 1.f, rb = 1.f;
    if (br) {
      float sa = 0.f, sb = 0.f;
      for (int i = threadIdx.x; i < H; i += 256) { const float a = ar[i], b = br[i]; sa += a * a; sb += b * b; }
      sa = block_sum(sa, scratch);
      sb = block_sum(sb, scratch);
      ra = rsqrtf(sa / H + eps); rb = rsqrtf(sb / H + eps);
    }
    const float* gr = gl ? gl + irow * ldg : nullptr;
    for (int i = threadIdx.x; i < H; i += 256) {
      float y = br ? 0.5f * (ar[i] * ra * wa[i] + br[i] * rb * wb[i]) : ar[i];
      if (gr) y *= 1.f / (1.f + expf(-(gr[i] + gb[i])));
      xr[i] += y;
    }
  }
  if (step)
    for (int i = threadIdx.x; i < H; i += 256) xr[i] += step[i];
  if (!out) return;
  // (each thread reads back only the elements it wrote itself)
  OT* outr = out + (long)orow * ldo;
  for (int i = threadIdx.x; i < H; i += 256) outr[i] = (OT)(tanhf(alpha * xr[i]) * nw[i] + nb[i]);
}

// The same for rows in whole 16-byte pieces: the row in registers, once through memory. 64 rows of 4096 behind a parallel mixer:
// 32 -> 6.6 us, behind a feed-forward 17 -> 4.7 us.
template <typename OT, int NR>
__global__ __launch_bounds__(1024) void dyt_gate_row_kernel(
    OT* __restrict__ out, float* __restrict__ x, const float* __restrict__ ya, const float* __restrict__ yb,
    const float* __restrict__ wa, const float* __restrict__ wb, const float* __restrict__ gl, const float* __restrict__ gb,
    const float* __restrict__ step, const float* __restrict__ nw, const float* __restrict__ nb, const int* __restrict__ row_idx,
    int H, long ldx, long ldy, long ldg, long ldo, float alpha, float eps) {
  __shared__ float scratch[16];
  const int orow = blockIdx.x, units = H / 4;
  const long irow = row_idx ? row_idx[orow] : orow;
  float* xr = x + irow * ldx;
  Unit<4> xv[NR];
  row_units<NR>(units, [&](int k, bool, int c) { xv[k] = ldu<4>(xr + c); });
  if (ya) {
    const float* ar = ya + irow * ldy;
    const float* br = yb ? yb + irow * ldy : nullptr;
    const float* gr = gl ? gl + irow * ldg : nullptr;
    Unit<4> av[NR], bv[NR], gv[NR];
    row_units<NR>(units, [&](int k, bool, int c) {
      av[k] = ldu<4>(ar + c);
      if (br) bv[k] = ldu<4>(br + c);
      if (gr) {
        gv[k] = ldu<4>(gr + c);
        const Unit<4> q = ldu<4>(gb + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) gv[k].v[e] = 1.f / (1.f + expf(-(gv[k].v[e] + q.v[e])));
      }
    });
    if (br) {
      float sa = 0.f, sb = 0.f;
      row_units<NR>(units, [&](int k, bool ok, int) {
        if (ok)
#pragma unroll
          for (int e = 0; e < 4; ++e) { sa += av[k].v[e] * av[k].v[e]; sb += bv[k].v[e] * bv[k].v[e]; }
      });
      sa = block_sum(sa, scratch);
      sb = block_sum(sb, scratch);
      const float ra = rsqrtf(sa / H + eps), rb = rsqrtf(sb / H + eps);
      row_units<NR>(units, [&](int k, bool, int c) {
        const Unit<4> p = ldu<4>(wa + c), q = ldu<4>(wb + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) av[k].v[e] = 0.5f * (av[k].v[e] * ra * p.v[e] + bv[k].v[e] * rb * q.v[e]);
      });
    }
    row_units<NR>(units, [&](int k, bool, int) {
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[k].v[e] += gr ? av[k].v[e] * gv[k].v[e] : av[k].v[e];
    });
  }
  if (step)
    row_units<NR>(units, [&](int k, bool, int c) {
      const Unit<4> q = ldu<4>(step + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[k].v[e] += q.v[e];
    });
  if (ya || step) row_units<NR>(units, [&](int k, bool ok, int c) { if (ok) stu<4>(xr + c, xv[k]); });
  if (!out) return;
  OT* outr = out + (long)orow * ldo;
  row_units<NR>(units, [&](int k, bool ok, int c) {
    const Unit<4> w = ldu<4>(nw + c), q = ldu<4>(nb + c);
    Unit<4> o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[e] = tanhf(alpha * xv[k].v[e]) * w.v[e] + q.v[e];
    if (ok) stu<4>(outr + c, o);
  });
}

template <typename OT>
__global__ __launch_bounds__(256) void headnorm_gate_kernel(OT* __restrict__ out, const float* __restrict__ o,
                                                            const float* __restrict__ gate, const float* __restrict__ w,
                                                            int items, int heads, int dv, int extra, long ldo_in, long ldg,
                                                            long ld_out, float eps) {
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= items) return;
  const int t = item / heads, h = item % heads, lane = lane_id();
  const float* orow = o + (long)t * ldo_in + (long)h * (dv + extra);
  const float* grow = gate + (long)t * ldg + (long)h * dv;
  const float den = extra ? 1.f / (fmaxf(fabsf(orow[dv]), orow[dv + 1]) + 1e-6f) : 1.f;
  float s = 0.f;
  for (int i = lane; i < dv; i += 64) { const float v = orow[i] * den; s += v * v; }
  s = wave_sum(s);
  const float r = rsqrtf(s / dv + eps) * den;
  OT* dst = out + (long)t * ld_out + (long)h * dv;
  for (int i = lane; i < dv; i += 64) dst[i] = (OT)(orow[i] * r * w[h * dv + i] / (1.f + expf(-grow[i])));
}

template <typename OT>
__global__ __launch_bounds__(256) void unary_act_kernel(OT* __restrict__ act, const float* __restrict__ z, long n, int F, long ldz,
                                                        long lda, int kind) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const long m = i / F; const int c = (int)(i % F);
  const float x = z[m * ldz + c];
  // 0: exact GELU, 1: tanh, 2: the square of relu, 3: silu(x) times the entry F columns further (gate | up side by side)
  float y;
  if (kind == 0) y = 0.5f * x * (1.f + erff(x * 0.7071067811865476f));
  else if (kind == 1) y = tanhf(x);
  else if (kind == 2) { const float r = fmaxf(x, 0.f); y = r * r; }
  else y = x / (1.f + expf(-x)) * z[m * ldz + c + F];
  act[m * lda + c] = (OT)y;
}

__global__ __launch_bounds__(256) void softcap_kernel(float* __restrict__ z, long n, int V, long ld, float cap) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float* p = z + (i / V) * ld + (i % V);
  *p = cap * tanhf(*p / cap);
}

}  // namespace dlia

extern "C" void dlia_embed_pos32(float* out, const int* ids, const int* pos, const void* table, const void* ptable, int f32, int T,
                                 int H, int vocab, int max_pos, hipStream_t stream) {
  if (T <= 0) return;
  // (many wide rows, where the bytes are the time, keep the walk of single entries: 4096 rows of 8192 32 us, 39 in units of four)
  const int vec = H % 4 == 0 && dlia::al16_(out) && dlia::al16_(table) && dlia::al16_(ptable) && !(T > 2048 && H > 4096);
  const int nt = vec ? dlia::row_shape(T, H).threads : 128;
  if (f32)
    hipLaunchKernelGGL(dlia::embed_pos32_kernel<float>, dim3(T), dim3(nt), 0, stream, out, ids, pos, (const float*)table,
                       (const float*)ptable, H, vocab, max_pos, vec);
  else
    hipLaunchKernelGGL(dlia::embed_pos32_kernel<dlia::bf16>, dim3(T), dim3(nt), 0, stream, out, ids, pos, (const dlia::bf16*)table,
                       (const dlia::bf16*)ptable, H, vocab, max_pos, vec);
}

extern "C" void dlia_dyt_gate(void* out, int out_f32, float* x, const float* ya, const float* yb, const float* wa, const float* wb,
                              const float* gl, const float* gb, const float* step, const float* nw, const float* nb,
                              const int* row_idx, int rows, int H, long ldx, long ldy, long ldg, long ldo, float alpha, float eps,
                              hipStream_t stream) {
  if (rows <= 0) return;
  using dlia::al16_;
  // (one stream of a short row, few rows: a thread's four sigmoids and tanh in a row cost more than the one pass saves, 2.2 -> 2.4 us)
  if ((yb || H > 256 || rows >= 1024) && dlia::row_fits(H) && ldx % 4 == 0 && ldy % 4 == 0 && ldg % 4 == 0 && ldo % 4 == 0 && al16_(out) && al16_(x) && al16_(ya) && al16_(yb) &&
      al16_(wa) && al16_(wb) && al16_(gl) && al16_(gb) && al16_(step) && al16_(nw) && al16_(nb)) {
    // (sigmoids and tanh: threads of one unit up to the 2048 a CU holds; one stream, 513 / 2048 rows of 576 5.6 / 8.6 -> 4.0 / 7.0 us)
    const dlia::RowShape sh = dlia::row_shape(rows, H, 2048);
#define DLIA_ROW(OT, NR) hipLaunchKernelGGL((dlia::dyt_gate_row_kernel<OT, NR>), dim3(rows), dim3(sh.threads), 0, stream, (OT*)out, x, ya, yb, wa, wb, gl, gb, \
                                            step, nw, nb, row_idx, H, ldx, ldy, ldg, ldo, alpha, eps)
    if (out_f32 || !out) { if (sh.nr == 1) DLIA_ROW(float, 1); else DLIA_ROW(float, 4); }
    else { if (sh.nr == 1) DLIA_ROW(dlia::bf16, 1); else DLIA_ROW(dlia::bf16, 4); }
#undef DLIA_ROW
    return;
  }
  if (out_f32 || !out)
    hipLaunchKernelGGL(dlia::dyt_gate_kernel<float>, dim3(rows), dim3(256), 0, stream, (float*)out, x, ya, yb, wa, wb, gl, gb, step,
                       nw, nb, row_idx, H, ldx, ldy, ldg, ldo, alpha, eps);
  else
    hipLaunchKernelGGL(dlia::dyt_gate_kernel<dlia::bf16>, dim3(rows), dim3(256), 0, stream, (dlia::bf16*)out, x, ya, yb, wa, wb, gl,
                       gb, step, nw, nb, row_idx, H, ldx, ldy, ldg, ldo, alpha, eps);
}

extern "C" void dlia_headnorm_gate(void* out, int out_f32, const float* o, const float* gate, const float* w, int T, int heads,
                                   int dv, int extra, long ldo_in, long ldg, long ld_out, float eps, hipStream_t stream) {
  const int items = T * heads;
  if (items <= 0) return;
  if (out_f32)
    hipLaunchKernelGGL(dlia::headnorm_gate_kernel<float>, dim3((items + 3) / 4), dim3(256), 0, stream, (float*)out, o, gate, w, items,
                       heads, dv, extra, ldo_in, ldg, ld_out, eps);
  else
    hipLaunchKernelGGL(dlia::headnorm_gate_kernel<dlia::bf16>, dim3((items + 3) / 4), dim3(256), 0, stream, (dlia::bf16*)out, o, gate,
                       w, items, heads, dv, extra, ldo_in, ldg, ld_out, eps);
}

extern "C" void dlia_unary_act(void* act, int out_f32, const float* z, int M, int F, long ldz, long lda, int kind, hipStream_t stream) {
  const long n = (long)M * F;
  if (n <= 0) return;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (out_f32)
    hipLaunchKernelGGL(dlia::unary_act_kernel<float>, grid, dim3(256), 0, stream, (float*)act, z, n, F, ldz, lda, kind);
  else
    hipLaunchKernelGGL(dlia::unary_act_kernel<dlia::bf16>, grid, dim3(256), 0, stream, (dlia::bf16*)act, z, n, F, ldz, lda, kind);
}

extern "C" void dlia_softcap(float* z, int M, int V, long ld, float cap, hipStream_t stream) {
  const long n = (long)M * V;
  if (n <= 0) return;
  hipLaunchKernelGGL(dlia::softcap_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, z, n, V, ld, cap);
}
