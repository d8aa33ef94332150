// Forward state scan (the state half of reference kernel D, gdn2_fwd.py:347-358)
// with its operands streamed from global memory into registers.
//
// Operand-fragment order.  The tiles the scan multiplies by, W [t][d], kg^T
// [d][t] and u^T [e][t], are stored as the 16-byte operand runs of the 16 x 16
// MFMAs that read them: fragment (rt, kk) covers rows 16 rt .. 16 rt + 15 and the
// 32 k positions from 32 kk, lane 16 lg + li of it holds row 16 rt + li and the
// eight k positions {4 lg + r} and {16 + 4 lg + r} (the chained order of kpos in
// gdn2_common.h), and the 64 lanes' runs are 1 KB contiguous.  A wave then loads
// an operand with one 16-byte load per lane and needs no LDS, no layout change
// and no other wave.
#pragma once

#include <type_traits>

#include "gdn2_common.h"
#include "gdn2_layout.h"

namespace gdn2 {

// Element offset of (row, k) of a [R][K] bfloat16 tile in fragment order.
template <int K>
__host__ __device__ constexpr int frag_off(int row, int k) {
  return (((row / 16) * (K / 32) + k / 32) * 64 + ((k % 16) / 4) * 16 + row % 16) * 8 +
         ((k / 16) % 2) * 4 + k % 4;
}

// sanitize of `n` tiles.  The clip binds only outside the domain: one test of the
// wave's largest magnitude (maximum propagates NaN, 0.5 instructions per value
// against 4), the element-wise sanitize only where it can change a value.
// Returns whether a value of this lane was clipped or NaN.
__device__ __forceinline__ bool sanitize_all(f32x4* v, int n, float clip) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < n; ++i) {
    const float x = __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(__builtin_fabsf(v[i][0]), __builtin_fabsf(v[i][1])),
        __builtin_fabsf(v[i][2]));
    m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, __builtin_fabsf(v[i][3])), m);
  }
  const bool over = !(m <= clip);
  if (__builtin_expect(__ballot(over) != 0, 0)) {
#pragma unroll
    for (int i = 0; i < n; ++i) v[i] = sanitize4(v[i]);
  }
  return over;
}

// A tile read with buffer loads: 16 bytes per lane at byte offset voff + soff
// (soff uniform), 0 where that is past `bytes`.  The addresses then cost no vector
// instructions.
using Rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ Rsrc tile_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ uint4 tile_load(Rsrc r, int voff, int soff) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// Wait until at most VM vector memory operations (LG of LDS) of this wave are in
// flight, known to the compiler, which then adds no wait of its own per operand:
// a lone wave issues one instruction per four cycles, waits included.
template <int VM, int LG>
__device__ __forceinline__ void wait_counts() {
  constexpr int V = VM < 63 ? VM : 63;
  __builtin_amdgcn_s_waitcnt((V & 15) | (7 << 4) | (LG << 8) | ((V >> 4) << 14));
}

template <typename T>
struct ScanArgs {
  const T* W;       // [cid] -W in fragment order
  const T* UT;      // [cid] u^T in fragment order
  const T* KgT;     // [cid] kg^T in fragment order
  const float* GL;  // [cid][D] gc_last
  const float* h0;  // nullable, (B,H,D,D)
  int N;            // chunks per (b,h)
  int units;        // (b,h) pairs, times segments or sequences
  int S, L;         // segments per (b,h), chunks per segment (the last may be shorter)
  int summary;      // segment-summary pass (S > 1): writes `seg`, no h^T / v_new^T
  const float* hin; // S > 1 and !summary: segment entry states [bh][S][D][D]
  float* seg;       // summary: [bh][S][2][D][D] = (end state, transition M_seg)
  T* HT;            // [cid][D][D] h_c^T, [cid][D][BT] v_new^T (no output waves)
  T* VnT;
  float* h_final;
  const int* cu;    // variable-length batch (B = 1): unit (h, sequence s) scans chunks
                    // [cu[s], cu[s+1]); h0 / h_final are [s][h][D][D]
  int H;
  // Output waves (NO > 0): o = scale qg h_c + Aqk v_new formed in this kernel
  const T* Qg;
  const T* Aqk;
  float* out;
  float scale;
  int T_len;
  const int* cstart;  // variable-length chunk table (see PrepArgs)
  // Segmented scan (S > 1): `sat` is set to 1 when a clip of the carried state
  // binds in a segmented pass (the segments' affine combination is exact only
  // while none does); a pass with `gate` runs only if *gate is nonzero -- the
  // serial scan that then replaces the segmented result
  int* sat;
  const int* gate;
};

// One workgroup: one unit and 16 CPW value columns: KS state waves (each D / KS
// rows of CPW column tiles of h, fp32 in MFMA accumulators), NO output waves and
// one helper wave.  Per chunk the state waves form v_new = u - W h and
// h <- e^{gl} h + kg^T v_new, two chained products whose other operands each wave
// loaded NSET chunks ahead, straight into registers.  With KS > 1 each wave forms
// its rows' part of W h; the parts are exchanged through LDS (two slots) and
// summed in the same order by every wave.  float32 tiles hold hi and lo fragments
// and the products run in the split form (gdn2_common.h).
// One barrier X(c) per chunk paces the waves and hands tiles over:
//   * the helper brings the lines of a later chunk into L2 (one 4-byte DMA per
//     128-byte line, shared among the unit's column slices, which run on one XCD)
//     and puts e^{g_last}(c) into LDS before X(c);
//   * the output waves form out(c) = scale qg h_c + Aqk v_new between X(c+1) and
//     X(c+2).  h_c is written to LDS before X(c) (three slots), v_new between X(c)
//     and X(c+1) (two slots), both in operand form.
template <typename T, int BT, int D, int KS, int CPW, int NO>
__global__ void __launch_bounds__(64 * (KS + NO + 1)) fwd_scan(ScanArgs<T> a) {
  constexpr bool F32 = sizeof(T) == 4;
  using Op = typename Tr<T>::Op;                  // operands of the output products
  constexpr int PL = F32 ? 2 : 1;                 // hi and lo fragments of a tile
  constexpr int NB = BT / 16, NDT = D / 16, NKT = BT / 32;
  constexpr int NDH = NDT / KS, NKD = NDH / 2;    // row tiles, k-groups of h per wave
  constexpr int NVS = D / (16 * CPW);
  constexpr int FW = NB * NKD * PL, FK = NDH * NKT * PL;   // fragments per wave
  // chunks held in registers ahead: two where they fit (with up to three waves; a
  // fourth brings nothing from a second set: 0.77 against 0.79 us a step)
  constexpr int NSET = FW + FK <= (KS + NO < 3 ? 32 : 16) ? 2 : 1;
  constexpr int UB = F32 ? NB : NKT;              // u^T loads per column tile
  constexpr int NHF = D / Tr<T>::KS, NVF = BT / Tr<T>::KS;   // output operands: h, v_new
  constexpr int OA = NO % 2 == 0 ? 2 : 1, OR = NO / OA;   // output waves: chunks x rows
  constexpr int NBO = NO > 0 ? NB / (OR > 0 ? OR : 1) : 1;   // row blocks per output wave
  static_assert(NDT % (2 * KS) == 0 && (NO == 0 || NB % OR == 0), "waves must split the tiles");
  __shared__ __align__(16) uint4 sH[NO > 0 ? 3 * CPW * NHF * 64 : 1];
  __shared__ __align__(16) uint4 sV[NO > 0 ? 2 * CPW * NVF * 64 : 1];
  __shared__ __align__(16) f32x4 sP[KS > 1 ? 2 * KS * CPW * NB * 64 : 1];
  __shared__ __align__(16) float sEg[2 * D];
  __shared__ __align__(16) float sJunk[64];       // target of the L2 touches

  if (a.gate && *a.gate == 0) return;   // whole workgroups, before any barrier
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Unit u runs on XCD u mod 8 (workgroup ids are dealt round-robin over the
  // XCDs): its column slices share that XCD's L2.  The grid is padded to whole
  // groups of 8 units.
  const int NSL = a.summary ? 2 * NVS : NVS;
  const int slot = blockIdx.x / 8;
  const int unit = (slot / NSL) * 8 + blockIdx.x % 8;
  int vs = slot % NSL;
  if (unit >= a.units) return;
  const int vsl = vs;                        // slice index within the unit
  const int bh = unit / a.S, sg = unit % a.S;
  const bool mslice = vs >= NVS;             // summary pass: columns of M_seg
  if (mslice && sg == 0) return;             // segment 0 starts from h0: no M needed
  if (mslice) vs -= NVS;
  int c0, n;                                 // chunks [c0, c0 + n) of this unit
  if (a.cu) {
    const SeqChunks sc = seq_chunks(a.cu, sg, a.N);
    c0 = sc.c0;
    n = sc.n;
  } else {
    c0 = sg * a.L;
    n = a.N - c0;
    n = n < a.L ? n : a.L;
  }
  n = n > 0 ? n : 0;
  const float clip = g_clip;
  // tiles of chunk c, c clamped to the unit's last chunk (n > 0)
  auto chunk_id = [&](int c) { return (size_t)bh * a.N + c0 + (c < n ? c : n - 1); };

  if (wv == KS + NO) {
    // ---- helper -----------------------------------------------------------------
    constexpr int LINE = 128;
    constexpr int ES = sizeof(T);
    constexpr int LW = BT * D * ES / LINE, LU = 16 * CPW * BT * ES / LINE;
    // Aqk: the fragments on and below the diagonal only (row blocks I, k-groups up
    // to the diagonal block's)
    constexpr int FPG = 16 * Tr<T>::KS * ES / LINE;         // lines per Aqk fragment
    constexpr int JPF = Tr<T>::KS / 16, NVK = NB / JPF;     // blocks per k-group, k-groups
    constexpr int LA = NO > 0 ? JPF * (NVK * (NVK + 1) / 2) * FPG : 0;
    constexpr int LSH = 2 * LW + (NO > 0 ? LW + LA : 0);  // W, kg^T (, q_g, Aqk): all slices
    constexpr int AHEAD = BT >= 128 ? 2 : 4;               // chunks
    const int lws = (LSH + NSL - 1) / NSL;                 // shared lines touched here
    constexpr int LMAX = (LSH + NVS - 1) / NVS + LU;
    constexpr int NTP = (LMAX + 63) / 64;
    auto aqk_line = [](int l) __attribute__((always_inline)) {
      const int f = l / FPG;                                // f-th stored fragment
      int P = 0;                                            // its group of JPF row blocks
#pragma unroll
      for (int g = 1; g < NVK; ++g) P += f >= JPF * (g * (g + 1) / 2) ? 1 : 0;
      const int rem = f - JPF * (P * (P + 1) / 2);
      const int I = P * JPF + (rem >= P + 1 ? 1 : 0), j = rem - (rem >= P + 1 ? P + 1 : 0);
      return (I * NVK + j) * FPG + l % FPG;
    };
    auto touch = [&](int c) __attribute__((always_inline)) {
      const size_t cid = chunk_id(c);
      const char* wsrc = reinterpret_cast<const char*>(a.W + cid * BT * D);
      const char* ksrc = reinterpret_cast<const char*>(a.KgT + cid * D * BT);
      const char* qsrc = reinterpret_cast<const char*>(a.Qg + cid * BT * D);
      const char* asrc = reinterpret_cast<const char*>(a.Aqk + cid * BT * BT);
      const char* usrc =
          reinterpret_cast<const char*>(a.UT + cid * D * BT + (size_t)vs * 16 * CPW * BT);
#pragma unroll
      for (int j = 0; j < NTP; ++j) {
        const int l = j * 64 + lane;
        const int lw = min(vsl * lws + l, LSH - 1);
        const char* src = lw < LW ? wsrc + lw * LINE
                        : lw < 2 * LW ? ksrc + (lw - LW) * LINE
                        : lw < 3 * LW ? qsrc + (lw - 2 * LW) * LINE
                        : asrc + aqk_line(lw - 3 * LW) * LINE;
        if (l >= lws) src = usrc + min(l - lws, LU - 1) * LINE;
        lds_dma4(src, sJunk);
      }
    };
    // e^{g_last}: loaded two chunks ahead of its use, by register set (a copy from
    // set to set would wait for the load)
    constexpr int GPL = D / 64;
    float g0[GPL], g1[GPL];
    auto load_gl = [&](int c, float* g) __attribute__((always_inline)) {
      const float* src = a.GL + chunk_id(c) * D;
#pragma unroll
      for (int j = 0; j < GPL; ++j) g[j] = src[j * 64 + lane];
    };
    auto put_eg = [&](int c, const float* g) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < GPL; ++j) sEg[(c & 1) * D + j * 64 + lane] = __expf(g[j]);
    };
    auto hstep = [&](int c, float* g) __attribute__((always_inline)) {
      put_eg(c + 1, g);
      load_gl(c + 3, g);
      touch(c + AHEAD);
      lds_barrier();  // X(c)
    };
    if (n > 0) {
      load_gl(0, g0);
      put_eg(0, g0);
      load_gl(1, g1);
      load_gl(2, g0);
      for (int c = 1; c < AHEAD; ++c) touch(c);
    }
    lds_barrier();    // E
    int c = 0;
    for (; c + 1 < n; c += 2) {
      hstep(c, g1);
      hstep(c + 1, g0);
    }
    if (c < n) hstep(c, g1);
    wait_vmcnt<0>();  // no DMA into this workgroup's LDS outlives it
    lds_barrier();    // X(n)
    return;
  }

  if constexpr (NO > 0) {
    if (wv >= KS) {
      // ---- output waves ---------------------------------------------------------
      // Wave (oa, orow): chunks oa, oa + OA, ... and every OR-th row block.  With
      // OA = 2 a chunk takes two steps: the products after X(c+1), its stores after
      // X(c+2), so that a wait for the next operands (vector memory operations
      // complete in issue order) meets stores that are three steps old.
      const int oa = OA == 2 ? (wv - KS) % 2 : 0;
      const int orow = OR == 1 ? 0 : (wv - KS) / OA;
      const int hh = bh % a.H, bb = bh / a.H;
      const size_t HD = (size_t)a.H * D;
      auto oblock = [&](int i) { return i % 2 == 0 ? i * OR + orow : i * OR + OR - 1 - orow; };
      constexpr int KC = Tr<T>::KC, JPF = Tr<T>::KS / 16;   // 16-token blocks per v operand
      constexpr int NST = NBO * CPW;                        // stores of a chunk
      Op qf[NBO][NHF], af[NBO][NVF];
      f32x4 acc[CPW][NBO];
      auto q_rsrc = [&](int c) {
        return tile_rsrc(a.Qg + chunk_id(c) * BT * D, BT * D * (int)sizeof(T));
      };
      auto a_rsrc = [&](int c) {
        return tile_rsrc(a.Aqk + chunk_id(c) * BT * BT, BT * BT * (int)sizeof(T));
      };
      auto load_q = [&](Rsrc r, int i, int kg) __attribute__((always_inline)) {
        qf[i][kg] = __builtin_bit_cast(Op, tile_load(r, lane * 16, (oblock(i) * NHF + kg) * 1024));
      };
      // (Aqk blocks right of the diagonal block are never written and not used)
      auto load_a = [&](Rsrc r, int i, int kg) __attribute__((always_inline)) {
        if (JPF * kg <= oblock(i))
          af[i][kg] = __builtin_bit_cast(Op, tile_load(r, lane * 16, (oblock(i) * NVF + kg) * 1024));
      };
      // the products of chunk c, the operands of chunk c + OA loaded behind them
      auto form = [&](int c) __attribute__((always_inline)) {
        const uint4* hs = &sH[(c % 3) * CPW * NHF * 64];
        const uint4* vn = &sV[(c & 1) * CPW * NVF * 64];
        Op ho[CPW][NHF], vo[CPW][NVF];
#pragma unroll
        for (int ct = 0; ct < CPW; ++ct) {
#pragma unroll
          for (int kg = 0; kg < NHF; ++kg)
            ho[ct][kg] = __builtin_bit_cast(Op, hs[(ct * NHF + kg) * 64 + lane]);
#pragma unroll
          for (int kg = 0; kg < NVF; ++kg)
            vo[ct][kg] = __builtin_bit_cast(Op, vn[(ct * NVF + kg) * 64 + lane]);
        }
        wait_counts<NST, 0>();   // chunk c's operands
        const Rsrc rq = q_rsrc(c + OA), ra = a_rsrc(c + OA);
#pragma unroll
        for (int i = 0; i < NBO; ++i) {
          const int It = oblock(i);
          f32x4 x[CPW], y[CPW];
#pragma unroll
          for (int ct = 0; ct < CPW; ++ct) x[ct] = y[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kg = 0; kg < NHF; ++kg) {
#pragma unroll
            for (int ct = 0; ct < CPW; ++ct) mma(x[ct], ho[ct][kg], qf[i][kg]);
            load_q(rq, i, kg);
          }
#pragma unroll
          for (int kg = 0; kg < NVF; ++kg) {
            if (JPF * kg <= It) {
              Op z = af[i][kg];
              if (JPF == 2 && 2 * kg + 1 > It) {   // block 2kg+1 lies right of the diagonal
#pragma unroll
                for (int e = KC / 2; e < KC; ++e) z[e] = (T)0.f;
              }
#pragma unroll
              for (int ct = 0; ct < CPW; ++ct) mma(y[ct], vo[ct][kg], z);
            }
            load_a(ra, i, kg);
          }
#pragma unroll
          for (int ct = 0; ct < CPW; ++ct) acc[ct][i] = x[ct] * a.scale + y[ct];
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      auto put = [&](int c) __attribute__((always_inline)) {
        sanitize_all(&acc[0][0], CPW * NBO, clip);
        const ChunkRows cr = chunk_rows(a.cstart, c0 + c, bb, a.T_len, BT);
        float* obase = a.out + cr.row0 * HD + (size_t)hh * D + vs * 16 * CPW + 4 * lg;
#pragma unroll
        for (int i = 0; i < NBO; ++i) {
          const int t = oblock(i) * 16 + li;
          if (t < cr.valid) {
#pragma unroll
            for (int ct = 0; ct < CPW; ++ct) store4(obase + (size_t)t * HD + ct * 16, acc[ct][i]);
          }
        }
      };
      if (n > 0) {
        const Rsrc rq = q_rsrc(oa), ra = a_rsrc(oa);
#pragma unroll
        for (int i = 0; i < NBO; ++i) {
#pragma unroll
          for (int kg = 0; kg < NHF; ++kg) load_q(rq, i, kg);
#pragma unroll
          for (int kg = 0; kg < NVF; ++kg) load_a(ra, i, kg);
        }
        lds_barrier();  // E
        lds_barrier();  // X(0)
        int c = oa;
        if (oa == 1) lds_barrier();  // X(1)
        for (; c + OA - 1 < n; c += OA) {
          lds_barrier();  // X(c+1)
          form(c);
          if constexpr (OA == 2) lds_barrier();  // X(c+2)
          put(c);
        }
        if (OA == 2 && c < n) {
          lds_barrier();  // X(n)
          form(c);
          put(c);
        }
      } else {
        lds_barrier();  // E
        lds_barrier();  // X(0)
      }
      return;
    }
  }

  // ---- state waves --------------------------------------------------------------
  const int ks = KS > 1 ? wv : 0, row0 = ks * NDH * 16;   // this wave's rows of h
  const int col0 = vs * CPW * 16 + li;                    // column of tile cp: col0 + 16 cp
  f32x4 h[CPW][NDH];
  const float* hsrc = a.cu ? (a.h0 ? a.h0 + ((size_t)sg * a.H + bh) * D * D : nullptr)
                    : (a.S > 1 && !a.summary) ? a.hin + ((size_t)unit) * D * D
                    : (sg == 0 && !mslice && a.h0) ? a.h0 + (size_t)bh * D * D : nullptr;
#pragma unroll
  for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
    for (int i = 0; i < NDH; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + i * 16 + 4 * lg + r, col = col0 + 16 * cp;
        h[cp][i][r] = mslice ? (row == col ? 1.f : 0.f)
                    : hsrc ? sanitize(hsrc[(size_t)row * D + col]) : 0.f;
      }
  const bool track = a.sat != nullptr && !mslice;
  bool bound = false;   // a clip of the state bound (NaN included)

  // Operands: -W rows 16 it of this wave's k-groups (kk-major, as P1 uses them),
  // kg^T rows of its row tiles (q-major)
  bf16x8 Wf[NSET][FW], Kf[NSET][FK];
  uint4 Uf[NSET][CPW][UB];
  constexpr int TILE = BT * D * (int)sizeof(T);
  const int vl16 = lane * 16;
  auto load_w = [&](int s, Rsrc r, int it, int kk) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < PL; ++p)
      Wf[s][(kk * NB + it) * PL + p] = __builtin_bit_cast(
          bf16x8, tile_load(r, vl16, ((it * KS + ks) * NKD + kk) * PL * 1024 + p * 1024));
  };
  auto load_k = [&](int s, Rsrc r, int i, int q) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < PL; ++p)
      Kf[s][(q * NDH + i) * PL + p] = __builtin_bit_cast(
          bf16x8, tile_load(r, vl16, ((ks * NDH + i) * NKT + q) * PL * 1024 + p * 1024));
  };
  auto load_u = [&](int s, Rsrc r, int cp, int q) __attribute__((always_inline)) {
    Uf[s][cp][q] = tile_load(r, vl16, ((vs * CPW + cp) * UB + q) * 1024);
  };
  // The next chunk to load of each tile, advanced up to the unit's last chunk
  const size_t cid0 = chunk_id(0) * BT * D;
  const T *pw = a.W + cid0, *pk = a.KgT + cid0, *pu = a.UT + cid0;
  auto advance = [&](const T*& q, int c) { q += c + 1 < n ? BT * D : 0; };
  // acc += X Y for one 32-deep k step, X a loaded fragment (pair), Y from C tiles
  struct Y { bf16x8 p[PL]; };
  auto make_y = [](const f32x4& t0, const f32x4& t1) __attribute__((always_inline)) {
    Y y;
    if constexpr (F32) {
      const Split8 s = split8(t0, t1);
      y.p[0] = s.hi;
      y.p[1] = s.lo;
    } else {
      y.p[0] = op_from_c(t0, t1, (bf16x8*)nullptr);
    }
    return y;
  };
  auto mul = [](f32x4& acc, const bf16x8* x, const Y& y) __attribute__((always_inline)) {
    if constexpr (F32) mma3(acc, Split8{x[0], x[1]}, Split8{y.p[0], y.p[1]});
    else mma(acc, x[0], y.p[0]);
  };

  // memory operations of a step, in issue order: FW + FU loads (and STH stores of
  // h) in P1, FK loads (and STV stores of v_new) in P3
  constexpr int FU = CPW * UB;
  constexpr int MPW = F32 ? (3 * CPW + 1) / 2 : CPW;   // products per loaded fragment
  constexpr int STH = NO == 0 ? CPW * (F32 ? NDH : NKD) : 0;
  constexpr int STV = NO == 0 ? CPW * (NVF / KS) : 0;
  // bfloat16 u enters the accumulators through MFMA: rows of the identity pick the
  // even (odd) row block of a u operand
  bf16x8 sel[2];
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) sel[o][e] = (bf16_t)(e / 4 == o && 4 * lg + e % 4 == li ? 1.f : 0.f);

  auto step = [&](int c, auto sc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value;
    // ---- P1: v_new = u - W h (this wave's rows), the next W and u on their way ----
    // (e^{g_last} is read first: its LDS latency hides behind the products)
    f32x4 eg[NDH];
#pragma unroll
    for (int i = 0; i < NDH; ++i) eg[i] = load4f(&sEg[(c & 1) * D + row0 + i * 16 + 4 * lg]);
    __builtin_amdgcn_sched_group_barrier(0x100, NDH, 0);   // LDS reads
    wait_counts<NSET == 2 ? 2 * FK + FW + FU + 2 * STV + STH : FK + STV, 15>();   // W(c), u(c)
    const Rsrc rw = tile_rsrc(pw, TILE), ru = tile_rsrc(pu, mslice ? 0 : TILE);
    f32x4 vn[CPW][NB];
#pragma unroll
    for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
      for (int it = 0; it < NB; ++it) {
        vn[cp][it] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (F32) {
          if (ks == 0) vn[cp][it] = __builtin_bit_cast(f32x4, Uf[s][cp][it]);
        } else {   // (with KS > 1 the first wave's part starts from u)
          if (ks == 0) mma(vn[cp][it], sel[it % 2], __builtin_bit_cast(bf16x8, Uf[s][cp][it / 2]));
        }
      }
    Y hy[CPW][NKD];
#pragma unroll
    for (int kk = 0; kk < NKD; ++kk) {
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp) {
        hy[cp][kk] = make_y(h[cp][2 * kk], h[cp][2 * kk + 1]);
        if constexpr (NO > 0) {   // h_c for the output waves: operands, or float32 tiles
          uint4* dst = &sH[(((c % 3) * CPW + cp) * NHF + ks * (NHF / KS)) * 64 + lane];
          if constexpr (F32) {
            dst[2 * kk * 64] = __builtin_bit_cast(uint4, h[cp][2 * kk]);
            dst[(2 * kk + 1) * 64] = __builtin_bit_cast(uint4, h[cp][2 * kk + 1]);
          } else {
            dst[kk * 64] = __builtin_bit_cast(uint4, hy[cp][kk].p[0]);
          }
        }
      }
#pragma unroll
      for (int it = 0; it < NB; ++it) {
#pragma unroll
        for (int cp = 0; cp < CPW; ++cp) mul(vn[cp][it], &Wf[s][(kk * NB + it) * PL], hy[cp][kk]);
        load_w(s, rw, it, kk);
      }
    }
#pragma unroll
    for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
      for (int q = 0; q < UB; ++q) load_u(s, ru, cp, q);
    advance(pw, c + NSET);
    advance(pu, c + NSET);
    if constexpr (NO == 0) {
      if (!a.summary) {
#pragma unroll
        for (int cp = 0; cp < CPW; ++cp) {
          T* hT = a.HT + chunk_id(c) * D * D + (size_t)(col0 + 16 * cp) * D + row0;
          if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < NDH; ++i) store4(hT + i * 16 + 4 * lg, h[cp][i]);
          } else {
#pragma unroll
            for (int kk = 0; kk < NKD; ++kk)
              *reinterpret_cast<bf16x8*>(hT + kk * 32 + 8 * lg) = hy[cp][kk].p[0];
          }
        }
      }
    }
    // e^{g_last} h, behind the products
    wait_counts<63, 0>();
#pragma unroll
    for (int i = 0; i < NDH; ++i)
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
        for (int r = 0; r < 4; ++r) h[cp][i][r] *= eg[i][r];
    if constexpr (KS > 1) {
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
        for (int it = 0; it < NB; ++it)
          sP[(((c & 1) * KS + ks) * CPW + cp) * NB * 64 + it * 64 + lane] = vn[cp][it];
    }
    // one load behind each product: in a burst they would stall the wave at issue
#pragma unroll
    for (int j = 0; j < FW + FU; ++j) {
      __builtin_amdgcn_sched_group_barrier(0x8, MPW, 0);   // MFMA
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);    // load
    }
    lds_barrier();  // X(c)
    // ---- P3: h <- e^{g_last} h + kg^T v_new, the next kg^T on its way ---------------
    wait_counts<NSET == 2 ? 2 * (FW + FU) + FK + 2 * STH + STV : FW + FU + STH, 15>();   // kg^T(c)
    const Rsrc rk = tile_rsrc(pk, TILE);
    advance(pk, c + NSET);
    Y vy[CPW][NKT];
    if constexpr (KS > 1) {
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
        for (int it = 0; it < NB; ++it) {
          auto part = [&](int k) __attribute__((always_inline)) {
            return sP[(((c & 1) * KS + k) * CPW + cp) * NB * 64 + it * 64 + lane];
          };
          f32x4 sum;
          if constexpr (KS == 2) {   // two parts: the same sum in either order
            sum = vn[cp][it] + part(1 - ks);
          } else {
            sum = part(0);
#pragma unroll
            for (int k = 1; k < KS; ++k) sum += part(k);
          }
          vn[cp][it] = sum;
        }
    }
#pragma unroll
    for (int q = 0; q < NKT; ++q) {
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp) vy[cp][q] = make_y(vn[cp][2 * q], vn[cp][2 * q + 1]);
#pragma unroll
      for (int i = 0; i < NDH; ++i) {
#pragma unroll
        for (int cp = 0; cp < CPW; ++cp) mul(h[cp][i], &Kf[s][(q * NDH + i) * PL], vy[cp][q]);
        load_k(s, rk, i, q);
      }
    }
#pragma unroll
    for (int j = 0; j < FK; ++j) {
      __builtin_amdgcn_sched_group_barrier(0x8, MPW, 0);
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
    }
#pragma unroll
    for (int cp = 0; cp < CPW; ++cp) {
      if constexpr (NO > 0) {
#pragma unroll
        for (int j = 0; j < NVF; ++j) {
          if (j % KS != ks) continue;
          uint4 x;
          if constexpr (F32) x = __builtin_bit_cast(uint4, vn[cp][j]);
          else x = __builtin_bit_cast(uint4, vy[cp][j].p[0]);
          sV[(((c & 1) * CPW + cp) * NVF + j) * 64 + lane] = x;
        }
      } else if (!a.summary) {
        T* vT = a.VnT + chunk_id(c) * D * BT + (size_t)(col0 + 16 * cp) * BT;
#pragma unroll
        for (int j = 0; j < NVF; ++j) {
          if (j % KS != ks) continue;
          if constexpr (F32) store4(vT + j * 16 + 4 * lg, vn[cp][j]);
          else *reinterpret_cast<bf16x8*>(vT + j * 32 + 8 * lg) = vy[cp][j].p[0];
        }
      }
    }
    if (!mslice) bound = sanitize_all(&h[0][0], CPW * NDH, clip) || bound;
  };

  if (n > 0) {
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
      const Rsrc rw = tile_rsrc(pw, TILE), rk = tile_rsrc(pk, TILE);
      const Rsrc ru = tile_rsrc(pu, mslice ? 0 : TILE);
#pragma unroll
      for (int kk = 0; kk < NKD; ++kk)
#pragma unroll
        for (int it = 0; it < NB; ++it) load_w(s, rw, it, kk);
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
        for (int q = 0; q < UB; ++q) load_u(s, ru, cp, q);
#pragma unroll
      for (int q = 0; q < NKT; ++q)
#pragma unroll
        for (int i = 0; i < NDH; ++i) load_k(s, rk, i, q);
      advance(pw, s);
      advance(pu, s);
      advance(pk, s);
    }
    lds_barrier();  // E
    if constexpr (NSET == 1) {
      for (int c = 0; c < n; ++c) step(c, std::integral_constant<int, 0>{});
    } else {
      // whole pairs in the loop: a path that skipped the second step would make the
      // compiler wait for that step's loads as well
      int c = 0;
      for (; c + 1 < n; c += 2) {
        step(c, std::integral_constant<int, 0>{});
        step(c + 1, std::integral_constant<int, 1>{});
      }
      if (c < n) step(c, std::integral_constant<int, 0>{});
    }
  } else {
    lds_barrier();  // E
  }
  lds_barrier();  // X(n)
  if (track && __ballot(bound) != 0 && lane == 0) *a.sat = 1;
  float* hout = a.cu ? a.h_final + ((size_t)sg * a.H + bh) * D * D
              : a.summary ? a.seg + ((size_t)unit * 2 + (mslice ? 1 : 0)) * D * D
              : (sg == a.S - 1) ? a.h_final + (size_t)bh * D * D : nullptr;
  if (hout) {
#pragma unroll
    for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
      for (int i = 0; i < NDH; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          hout[(size_t)(row0 + i * 16 + 4 * lg + r) * D + col0 + 16 * cp] = h[cp][i][r];
  }
}

// Workgroups of a scan over `units` units (the padding of the XCD mapping included).
inline unsigned scan_grid(size_t units, int slices) {
  return (unsigned)((units + 7) / 8 * 8 * slices);
}

}  // namespace gdn2
