// Single-token recurrent step on the (B,H,D,D) float32 state -- the decode
// step of a model served with GDN-2 layers.  Per (b,h) and token
//   S <- Diag(e^g) S,  pred = (b*k)^T S,  S <- S + k (w*v - pred)^T,
//   o = scale q^T S,
// the chunked forward's math with a chunk of one token (its state and output
// are sanitized like every chunk state and output, gdn2_fwd.py:355-356).  The
// state layout is h0 / h_final's: S[b][h][dk][dv] (gdn2_fwd.py:342).
//
// One 256-thread workgroup per (b,h) and slice of CS state columns: thread (column
// quad c4, row group rg) keeps D CS / 1024 state rows of four columns in registers,
// read and written with 16-byte accesses.  Both column reductions (pred and o)
// run over the rows, so the columns split freely; they are summed over the row
// groups of a wave by lane shuffles, then over the four waves in LDS.  The state
// is read and written once (memory-bound); h_out may alias h_in.
//
// CS: a row of a slice should fill whole 128-byte lines (32 columns), or two
// workgroups -- on different XCDs -- fetch and write back each line.  With 16, 32
// and 64 columns (bfloat16 tokens, D = 128, state updated in place, kernels back to
// back): 32 x 6 (b,h) 11.7, 6.2 and 6.1 us, 128 x 6 28.9, 19.4 and 16.6, 512 x 6
// 95.9, 64.1 and 61.2 us (403 MB, of which the 201 MB state stays in the 256 MB cache;
// written to a new state 78 us, the rate of a copy); 8 x 6 at D = 256 10.7, 6.4 and
// 6.6 us; 2 at D = 64 3.45, 3.75 and 4.40 us.  So: 64 columns from 512 such workgroups
// on (two per CU), 16 where 32 would leave fewer than 32 workgroups.
#include "gdn2_common.h"

namespace gdn2 {

// Sum of x over the lanes of a wave that hold the same column quad (lane mod C4).
template <int C4>
__device__ __forceinline__ f32x4 rowgroup_sum(f32x4 x) {
#pragma unroll
  for (int m = C4; m < 64; m *= 2)
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] += __shfl_xor(x[c], m);
  return x;
}

// Sum over a thread's rows: rows 2j, 2j+1 are accumulated in p[j], then the p[j] are
// added pairwise, so that wider slices (more rows per thread) round no more than
// narrow ones.
template <int N>
__device__ __forceinline__ f32x4 pair_sum(f32x4 (&p)[N]) {
#pragma unroll
  for (int m = 1; m < N; m *= 2)
#pragma unroll
    for (int j = 0; j + m < N; j += 2 * m) p[j] += p[j + m];
  return p[0];
}

template <typename T, typename TG, int D, int CS>
__global__ void __launch_bounds__(256) decode_step(const T* q, const T* k, const T* v,
                                                   const T* w, const T* b, const TG* g,
                                                   float scale, const float* h_in,
                                                   float* h_out, float* out) {
  constexpr int NSL = D / CS;
  constexpr int C4 = CS / 4, RG = 256 / C4, RPT = D / RG;   // row groups, rows per thread
  static_assert(RPT >= 1 && D % RG == 0, "rows must split over the row groups");
  __shared__ float sQ[D], sK[D], sBK[D], sEG[D];
  __shared__ f32x4 sRed[4][C4];   // per wave and column quad
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c4 = tid % C4, rg = tid / C4;
  const size_t bh = blockIdx.x / NSL;
  const int col = (blockIdx.x % NSL) * CS + 4 * c4;   // first of this thread's four columns
  const size_t vo = bh * D;                  // token vectors are (B,H,D) contiguous
  // the state rows and this thread's w, v first: their loads are in flight while
  // the token vectors are gathered into LDS (the step is latency-bound)
  const float* src = h_in ? h_in + bh * D * D : nullptr;
  f32x4 s[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i)
    s[i] = src ? load4f(src + (size_t)(rg * RPT + i) * D + col) : f32x4{0.f, 0.f, 0.f, 0.f};
  float wv4[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) wv4[c] = to_f(w[vo + col + c]) * to_f(v[vo + col + c]);
  for (int i = tid; i < D; i += 256) {
    const float kv = to_f(k[vo + i]);
    sQ[i] = to_f(q[vo + i]);
    sK[i] = kv;
    sBK[i] = to_f(b[vo + i]) * kv;
    sEG[i] = __expf(to_f(g[vo + i]));
  }
  __syncthreads();
  constexpr int NP = (RPT + 1) / 2;
  f32x4 part[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) part[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = rg * RPT + i;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      s[i][c] = sanitize(s[i][c]) * sEG[d];
      part[i / 2][c] += sBK[d] * s[i][c];
    }
  }
  f32x4 pred = rowgroup_sum<C4>(pair_sum(part));
  if (lane < C4) sRed[wave][lane] = pred;
  __syncthreads();
  pred = sRed[0][c4] + sRed[1][c4] + sRed[2][c4] + sRed[3][c4];
  f32x4 delta;
#pragma unroll
  for (int c = 0; c < 4; ++c) delta[c] = wv4[c] - pred[c];
  __syncthreads();  // every thread has read sRed
#pragma unroll
  for (int j = 0; j < NP; ++j) part[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float* dst = h_out + bh * D * D;
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = rg * RPT + i;
    f32x4 nv;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      nv[c] = sanitize(s[i][c] + sK[d] * delta[c]);
      part[i / 2][c] += sQ[d] * nv[c];
    }
    store4(dst + (size_t)d * D + col, nv);
  }
  const f32x4 o = rowgroup_sum<C4>(pair_sum(part));
  if (lane < C4) sRed[wave][lane] = o;
  __syncthreads();
  if (tid < C4) {
    const f32x4 t = sRed[0][tid] + sRed[1][tid] + sRed[2][tid] + sRed[3][tid];
    store4(out + vo + (blockIdx.x % NSL) * CS + 4 * tid, sanitize4(scale * t));
  }
}

template <typename T, typename TG, int D>
hipError_t launch_decode(hipStream_t st, int B, int H, const void* q, const void* k,
                         const void* v, const void* w, const void* b, const void* g,
                         float scale, const float* h_in, float* h_out, float* out) {
  launch_mark(st);
  auto go = [&](auto csc) {
    constexpr int CS = decltype(csc)::value;
    hipLaunchKernelGGL((decode_step<T, TG, D, CS>), dim3((size_t)B * H * (D / CS)), dim3(256), 0,
                       st, (const T*)q, (const T*)k, (const T*)v, (const T*)w, (const T*)b,
                       (const TG*)g, scale, h_in, h_out, out);
  };
  const size_t BH = (size_t)B * H;
  if (BH * (D / 64) >= 512) go(std::integral_constant<int, 64>{});
  else if (BH * (D / 32) >= 32) go(std::integral_constant<int, 32>{});
  else go(std::integral_constant<int, 16>{});
  launch_mark(st);
  return hipGetLastError();
}

#define GDN2_INST_DEC(T, TG, D)                                                            \
  template hipError_t launch_decode<T, TG, D>(hipStream_t, int, int, const void*,         \
                                              const void*, const void*, const void*,      \
                                              const void*, const void*, float,            \
                                              const float*, float*, float*);
GDN2_INST_DEC(float, float, 64)
GDN2_INST_DEC(float, float, 128)
GDN2_INST_DEC(bf16_t, float, 64)
GDN2_INST_DEC(bf16_t, float, 128)
GDN2_INST_DEC(bf16_t, bf16_t, 64)
GDN2_INST_DEC(bf16_t, bf16_t, 128)
GDN2_INST_DEC(float, float, 256)
GDN2_INST_DEC(bf16_t, float, 256)
GDN2_INST_DEC(bf16_t, bf16_t, 256)

// This translation unit's clip bound on the current device (gdn2_set_clip).
hipError_t set_clip_decode(float c) { return set_unit_clip(c); }

}  // namespace gdn2
