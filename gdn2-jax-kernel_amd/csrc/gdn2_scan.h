// Forward state scan (the state half of reference kernel D, gdn2_fwd.py:347-358)
// with its operands streamed from global memory into registers.
//
// The tiles the scan multiplies by, W [t][d], kg^T [d][t] and u^T [e][t], are stored
// in the operand-fragment order of gdn2_common.h (float32 W and kg^T as hi and lo
// fragments), so that a wave loads an operand with one 16-byte load per lane, 1 KB
// contiguous per wave, and needs no LDS, no layout change and no other wave.
#pragma once

#include <type_traits>

#include "gdn2_common.h"
#include "gdn2_layout.h"

namespace gdn2 {

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
  const float* hin; // S > 1, final pass: segment entry states [bh][S][D][D]
  float* seg;       // S > 1, summary pass: [bh][S][2][D][D] = (end state, transition M_seg)
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
// one helper wave (SUM: the summary pass of a segmented scan, which writes the
// segments' maps instead of h^T / v_new^T or outputs).  Per chunk the state waves form v_new = u - W h and
// h <- e^{gl} h + kg^T v_new, two chained products whose other operands each wave
// loaded NSET chunks ahead, straight into registers.  With KS > 1 each wave forms
// its rows' part of W h; the parts are exchanged through LDS (two slots) and
// summed in the same order by every wave.  float32 tiles hold hi and lo fragments
// and the products run in the split form (gdn2_common.h).
// One barrier X(c) per chunk paces the waves and hands tiles over:
//   * the helper brings the lines of a later chunk into L2 (TOUCH: one 4-byte DMA
//     per 128-byte line, shared among the unit's column slices, which run on one
//     XCD) and puts e^{g_last}(c) into LDS before X(c);
//   * the output waves form out(c) = scale qg h_c + Aqk v_new between X(c+1) and
//     X(c+2).  h_c is written to LDS before X(c) (three slots), v_new between X(c)
//     and X(c+1) (two slots), both in operand form.
template <typename T, int BT, int D, int KS, int CPW, int NO, bool SUM>
__global__ void __launch_bounds__(64 * (KS + NO + 1), scan_per_cu(sizeof(T), NO))
    fwd_scan(ScanArgs<T> a) {
  constexpr bool F32 = sizeof(T) == 4;
  // Lines of later chunks are brought into L2 ahead of the loads, except where two
  // workgroups share a CU: each then covers the other's waits, and the touches only
  // add traffic (float32 D = 64, 8 x 4096 tokens of 12 heads: 436 us a call without,
  // 440, 442 and 446 two, three and four chunks ahead; bfloat16 summary pass, 131072
  // tokens of 8 heads: 307 against 324 us at chunk 128, 323 against 345 at chunk 64).
  constexpr bool TOUCH = scan_per_cu(sizeof(T), NO) == 1 && !(SUM && KS == 1 && CPW == 2);
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
  constexpr int NSL = SUM ? 2 * NVS : NVS;
  const int slot = blockIdx.x / 8;
  const int unit = (slot / NSL) * 8 + blockIdx.x % 8;
  int vs = slot % NSL;
  if (unit >= a.units) return;
  const int vsl = vs;                        // slice index within the unit
  const int bh = unit / a.S, sg = unit % a.S;
  const bool mslice = SUM && vs >= NVS;      // summary pass: columns of M_seg
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
    // Chunk 128 on a full device: one chunk ahead, W by slice 0 and kg^T by slice 1.
    // The lines of more chunks, or of more tiles, push one another out of the XCD's 4 MB
    // (final pass of 131072 tokens of 8 heads, all tiles shared by all slices: 487 us
    // two chunks ahead, 451 one; W and kg^T only, by four slices 453, by one 457, so
    // 421).  With few units nothing is pushed out (4096 tokens of 6 heads 78 us a call,
    // so 82).
    constexpr bool TWO = BT >= 128 && CPW == 2;
    constexpr int AHEAD = TWO ? 1 : BT >= 128 ? 2 : 4;     // chunks
    static_assert(!TWO || (LW % 64 == 0 && NVS >= 2), "a slice touches a whole tile");
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
      if constexpr (TWO) {
        if (vsl < 2) {
          const char* src = vsl == 0 ? wsrc : ksrc;
#pragma unroll
          for (int j = 0; j < LW / 64; ++j) lds_dma4(src + (j * 64 + lane) * LINE, sJunk);
        }
        return;
      }
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
      if constexpr (TOUCH) touch(c + AHEAD);
      lds_barrier();  // X(c)
    };
    if (n > 0) {
      load_gl(0, g0);
      put_eg(0, g0);
      load_gl(1, g1);
      load_gl(2, g0);
      if constexpr (TOUCH)
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
          f32x4 x[CPW];
#pragma unroll
          for (int ct = 0; ct < CPW; ++ct) x[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kg = 0; kg < NHF; ++kg) {
#pragma unroll
            for (int ct = 0; ct < CPW; ++ct) mma(x[ct], ho[ct][kg], qf[i][kg]);
            load_q(rq, i, kg);
          }
#pragma unroll
          for (int ct = 0; ct < CPW; ++ct) x[ct] *= a.scale;
#pragma unroll
          for (int kg = 0; kg < NVF; ++kg) {
            if (JPF * kg <= It) {
              Op z = af[i][kg];
              if (JPF == 2 && 2 * kg + 1 > It) {   // block 2kg+1 lies right of the diagonal
#pragma unroll
                for (int e = KC / 2; e < KC; ++e) z[e] = (T)0.f;
              }
#pragma unroll
              for (int ct = 0; ct < CPW; ++ct) mma(x[ct], vo[ct][kg], z);
            }
            load_a(ra, i, kg);
          }
#pragma unroll
          for (int ct = 0; ct < CPW; ++ct) acc[ct][i] = x[ct];
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
                    : (a.S > 1 && !SUM) ? a.hin + ((size_t)unit) * D * D
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
  constexpr int STH = NO == 0 && !SUM ? CPW * (F32 ? NDH : NKD) : 0;
  constexpr int STV = NO == 0 && !SUM ? CPW * (NVF / KS) : 0;
  // bfloat16 u enters the accumulators through MFMA: rows of the identity pick the
  // even (odd) row block of a u operand (with KS > 1 in the first wave's part only)
  bf16x8 sel[2];
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) sel[o][e] = (bf16_t)(ks == 0 && e / 4 == o && 4 * lg + e % 4 == li ? 1.f : 0.f);

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
    // bfloat16 accumulates from u; float32 sums W h first and adds u last, a
    // rounding error of W h instead of one of u per product
    f32x4 vn[CPW][NB], u32[CPW][F32 ? NB : 1];
#pragma unroll
    for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
      for (int it = 0; it < NB; ++it) {
        vn[cp][it] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (F32) {
          u32[cp][it] = __builtin_bit_cast(f32x4, Uf[s][cp][it]);
        } else {
          mma(vn[cp][it], sel[it % 2], __builtin_bit_cast(bf16x8, Uf[s][cp][it / 2]));
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
    if constexpr (NO == 0 && !SUM) {
      {
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
    if constexpr (F32) {
#pragma unroll
      for (int cp = 0; cp < CPW; ++cp)
#pragma unroll
        for (int it = 0; it < NB; ++it) vn[cp][it] += u32[cp][it];
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
      // each wave hands on (stores) its share of v_new
      if constexpr (NO > 0 || !SUM) {
        T* vT = a.VnT + chunk_id(c) * D * BT + (size_t)(col0 + 16 * cp) * BT;
#pragma unroll
        for (int jj = 0; jj < NVF / KS; ++jj) {
          auto piece = [&](int j) __attribute__((always_inline)) {
            if constexpr (F32) return __builtin_bit_cast(uint4, vn[cp][j]);
            else return __builtin_bit_cast(uint4, vy[cp][j].p[0]);
          };
          uint4 x = piece(jj * KS);
#pragma unroll
          for (int k = 1; k < KS; ++k) {
            const uint4 y = piece(jj * KS + k);
            x.x = ks == k ? y.x : x.x;
            x.y = ks == k ? y.y : x.y;
            x.z = ks == k ? y.z : x.z;
            x.w = ks == k ? y.w : x.w;
          }
          const int j = jj * KS + ks;
          if constexpr (NO > 0) sV[(((c & 1) * CPW + cp) * NVF + j) * 64 + lane] = x;
          else *reinterpret_cast<uint4*>(vT + (F32 ? j * 16 + 4 * lg : j * 32 + 8 * lg)) = x;
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
              : SUM ? a.seg + ((size_t)unit * 2 + (mslice ? 1 : 0)) * D * D
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

// ---------------------------------------------------------------------------
// The scan of float32 tiles in rows (scan_rows in gdn2_layout.h), where the units
// fill the device or have one or two chunks: one workgroup per unit and 32 value
// columns, which shares each tile through LDS -- two 16-column slices with two
// K-split compute waves each (half of h's rows) and four producer waves.  W and kg^T
// come in the split pair layout (gdn2_common.h), u^T in rows.
//
// While the compute waves work on chunk c, the producers stream chunk c+1 (W,
// kg^T, g_last and this workgroup's u^T rows) into LDS with
// global_load_lds_dwordx4, wait for it and replace g_last by e^{g_last}.  A wave
// that issues that much memory traffic stalls at issue, so the compute waves issue
// none and the traffic is split over four producers.  Barriers per chunk: A (chunk
// c resident), B (u^T of chunk c in registers, its buffer free), X (the parts of
// W h exchanged).  W / kg^T tiles are stored unpadded with the 16-byte chunks of
// row r XOR-permuted by (r mod 16), so the 16 rows an MFMA operand read touches land
// in distinct LDS banks; u^T is gathered straight into the order the compute lanes
// read it (1 KB per wave and row block).
//
// Where two tile buffers do not fit in LDS (D = 256: 128 KB per chunk) the kernel
// runs single-buffered, with a fourth barrier E after the compute waves' last
// reads: the producers refill W and u^T after X(c) (W is read before the exchange)
// and kg^T and g_last after E(c), each move behind the other product, from L2
// through the touch issued one chunk ahead.
template <int BT, int D, bool SUM>
__global__ void __launch_bounds__(512) fwd_state(ScanArgs<float> a) {
  constexpr int NW = 2, KS = 2, NP = 4;              // column slices, K-split, producers
  constexpr int NB = BT / 16, NDT = D / 16;
  constexpr int NVS = D / (16 * NW);
  constexpr int WBYTES = BT * D * 4;   // one tile (W or kg^T)
  constexpr int BUF = 2 * WBYTES;                    // W + kg^T
  constexpr int PIECES = BUF / 1024;                 // 1 KB DMA instructions per chunk
  constexpr int NBUF = 2 * BUF <= 132 * 1024 ? 2 : 1;
  constexpr int NCW = NW * KS;                       // compute waves
  constexpr int NDH = NDT / KS;                      // row tiles of h per compute wave
  static_assert(BUF % 1024 == 0, "tiles must split into 1 KB pieces");
  static_assert(NDT % (2 * KS) == 0 && NB % KS == 0, "the K-split must tile h and v_new");
  __shared__ __align__(16) char sbuf0[BUF];
  __shared__ __align__(16) char sbuf1[NBUF == 2 ? BUF : 16];
  __shared__ __align__(16) uint4 sU[NW * NB * 64];   // u^T in compute-lane order
  __shared__ __align__(16) f32x4 sX[NCW * NB * 64];  // K-split partials of W h
  __shared__ __align__(16) float sGL0[D];
  __shared__ __align__(16) float sGL1[NBUF == 2 ? D : 4];
  __shared__ __align__(16) float sJunk[64];        // target of the L2 touches

  if (a.gate && *a.gate == 0) return;   // whole workgroups, before any barrier
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // A unit is one (b,h) segment; it has NVS column slices (2 NVS in the summary
  // pass, the second NVS carrying M).  Workgroups are dealt round-robin over the
  // 8 XCDs (XCD = id mod 8): all slices of a unit go to one XCD so the W / kg^T
  // tiles they all stream are fetched into that XCD's L2 once.
  constexpr int NSL = SUM ? 2 * NVS : NVS;
  int unit, vs;
  bool one_xcd = false;   // all slices of the unit on this workgroup's XCD
  {
    const int nwg = gridDim.x, id = blockIdx.x;
    const int per_xcd = nwg / 8;
    if (nwg % 8 == 0 && per_xcd % NSL == 0) {
      const int xcd = id % 8, slot = id / 8;
      unit = xcd * (per_xcd / NSL) + slot / NSL;
      vs = slot % NSL;
      one_xcd = true;
    } else {
      unit = id / NSL;
      vs = id % NSL;
    }
  }
  const int bh = unit / a.S, sg = unit % a.S;
  const bool mslice = SUM && vs >= NVS;      // summary pass: columns of M_seg
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

  if (wv >= NCW) {
    // ---- producers ----------------------------------------------------------
    // producer p moves W / kg^T pieces [p PP, (p+1) PP) and u^T blocks q = p mod NP
    constexpr int ROWB_W = D * 4, ROWB_K = BT * 4;
    constexpr int WPIECES = WBYTES / 1024;
    constexpr int PP = PIECES / NP;
    static_assert(PIECES % NP == 0 && (NW * NB) % NP == 0, "work must split evenly");
    const int p = wv - NCW;
    // parts: 1 the W / kg^T tiles and g_last, 2 the u^T blocks, 3 both
    auto issue = [&](int c, char* base, float* gl, int parts = 3) __attribute__((always_inline)) {
      const size_t cid = (size_t)bh * a.N + c0 + c;
      const char* wsrc = reinterpret_cast<const char*>(a.W + cid * BT * D);
      const char* ksrc = reinterpret_cast<const char*>(a.KgT + cid * D * BT);
#pragma unroll
      for (int i = 0; i < ((parts & 1) ? PP : 0); ++i) {
        const int piece = p * PP + i;                      // wave-uniform
        char* dst = base + piece * 1024;
        if (piece < WPIECES) {
          const int ib = piece * 1024 + lane * 16;
          const int r = ib / ROWB_W, pch = (ib % ROWB_W) / 16;
          constexpr int NCH = ROWB_W / 16, M = (NCH < 16 ? NCH : 16) - 1;
          lds_dma16(wsrc + (size_t)r * ROWB_W + ((pch ^ (r & M)) * 16), dst);
        } else {
          const int ib = (piece - WPIECES) * 1024 + lane * 16;
          const int r = ib / ROWB_K, pch = (ib % ROWB_K) / 16;
          constexpr int NCH = ROWB_K / 16, M = (NCH < 16 ? NCH : 16) - 1;
          lds_dma16(ksrc + (size_t)r * ROWB_K + ((pch ^ (r & M)) * 16), dst);
        }
      }
      if ((parts & 1) && p == NP - 1 && lane < D / 4) lds_dma16(a.GL + cid * D + lane * 4, gl);
      if (!(parts & 2)) return;
      // u^T[col][t] for compute wave w, row block q: lane (li, lg) of that wave gets
      // the 16 bytes at u^T[16 w + li][16 q + 4 lg], at sU[(w NB + q) 64 + lane]
      if (mslice) return;  // M columns: u = 0
      const float* usrc = a.UT + cid * D * BT + (size_t)(vs * 16 * NW + li) * BT + 4 * lg;
#pragma unroll
      for (int j = 0; j < NW * NB / NP; ++j) {
        const int q = j * NP + p, w = q / NB, it = q % NB;
        lds_dma16(usrc + (size_t)w * 16 * BT + it * 16, &sU[q * 64]);
      }
    };
    // L2 touch of chunk c: one 4-byte DMA into a junk slot per 128-byte line of
    // everything issue(c) will read, spread over the producers.  Issued one
    // chunk ahead of the DMA, it turns the DMA's HBM latency into L2 latency.
    // The W / kg^T lines are read by every column slice of the unit: when the
    // slices share an XCD (one L2) slice v touches only the v-th share of them
    // (a touch per line and workgroup cost the scan a fifth of its time), every
    // slice its own u^T rows.
    constexpr int LINE = 128;
    constexpr int LW = WBYTES / LINE;                       // lines per W / kg^T tile
    constexpr int LUR = BT * 4 / LINE;         // lines per u^T row
    constexpr int LU = 16 * NW * LUR;                       // this workgroup's u^T rows
    constexpr int LG = (D * 4 + LINE - 1) / LINE;           // g_last
    constexpr int LSH = 2 * LW, LTOT = LSH + LU + LG;
    constexpr int NTP = ((LTOT + 63) / 64 + NP - 1) / NP;   // touch instructions per producer
    const int vsl = vs + (mslice ? NVS : 0);                // slice index within the unit
    const int lws = one_xcd ? (LSH + NSL - 1) / NSL : LSH;  // shared lines touched here
    const int lw0 = one_xcd ? vsl * lws : 0;
    const int ltot = lws + LU + LG;
    auto touch = [&](int c) __attribute__((always_inline)) {
      const size_t cid = (size_t)bh * a.N + c0 + c;
      const char* wsrc = reinterpret_cast<const char*>(a.W + cid * BT * D);
      const char* ksrc = reinterpret_cast<const char*>(a.KgT + cid * D * BT);
      const char* usrc =
          reinterpret_cast<const char*>(a.UT + cid * D * BT + (size_t)vs * 16 * NW * BT);
      const char* gsrc = reinterpret_cast<const char*>(a.GL + cid * D);
#pragma unroll
      for (int j = 0; j < NTP; ++j) {
        int l = (j * NP + p) * 64 + lane;
        l = l < ltot ? l : ltot - 1;
        const int lw = min(lw0 + l, LSH - 1);                   // shared line
        const char* sh = lw < LW ? wsrc + lw * LINE : ksrc + (lw - LW) * LINE;
        const char* src = l < lws ? sh
                        : l < lws + LU ? usrc + (l - lws) * LINE
                        : gsrc + (l - lws - LU) * LINE;
        lds_dma4(src, sJunk);
      }
    };
    // In flight at the top of chunk c: issue(c), then touch(c+1) if c+1 < n.
    auto wait_chunk = [&](int c) __attribute__((always_inline)) {
      if (c + 1 < n) wait_vmcnt<NTP>();
      else wait_vmcnt<0>();
    };
    // The producers' data ordering is the explicit vmcnt wait; a plain barrier
    // (no fence) keeps the compiler from also waiting for the L2 touches.
    auto barrier = []() __attribute__((always_inline)) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    // g_last -> e^{g_last} in place, once per chunk, by the producer that moved it
    auto exp_gl = [&](float* gl) __attribute__((always_inline)) {
      if (p == NP - 1) {
#pragma unroll
        for (int i = 0; i < (D + 63) / 64; ++i)
          if (i * 64 + lane < D) gl[i * 64 + lane] = __expf(gl[i * 64 + lane]);
      }
    };
    if constexpr (NBUF == 1) {
      // One tile buffer: W and u^T of chunk c+1 move in once barrier X(c) has
      // passed (the compute waves are done with W(c) and u^T(c)), kg^T and g_last
      // once E(c) has passed, so each move hides behind the other product of the
      // chain (kg^T v_new of chunk c, then W h of chunk c+1).  Every producer
      // moves the same counts: its share of the W pieces and u^T blocks, then its
      // share of the kg^T pieces and of g_last, which it exponentiates itself.
      constexpr int PPW = WPIECES / NP, PPK = (PIECES - WPIECES) / NP, GQ = D / NP;
      static_assert(WPIECES % NP == 0 && (PIECES - WPIECES) % NP == 0 &&
                        GQ % 4 == 0 && GQ <= 64,
                    "single-buffer split: equal shares per producer");
      auto piece_dma = [&](const char* wsrc, const char* ksrc, int piece) __attribute__((always_inline)) {
        char* dst = sbuf0 + piece * 1024;
        if (piece < WPIECES) {
          const int ib = piece * 1024 + lane * 16;
          const int r = ib / ROWB_W, pch = (ib % ROWB_W) / 16;
          constexpr int NCH = ROWB_W / 16, M = (NCH < 16 ? NCH : 16) - 1;
          lds_dma16(wsrc + (size_t)r * ROWB_W + ((pch ^ (r & M)) * 16), dst);
        } else {
          const int ib = (piece - WPIECES) * 1024 + lane * 16;
          const int r = ib / ROWB_K, pch = (ib % ROWB_K) / 16;
          constexpr int NCH = ROWB_K / 16, M = (NCH < 16 ? NCH : 16) - 1;
          lds_dma16(ksrc + (size_t)r * ROWB_K + ((pch ^ (r & M)) * 16), dst);
        }
      };
      auto issue_w = [&](int c) __attribute__((always_inline)) {
        const size_t cid = (size_t)bh * a.N + c0 + c;
        const char* wsrc = reinterpret_cast<const char*>(a.W + cid * BT * D);
#pragma unroll
        for (int i = 0; i < PPW; ++i) piece_dma(wsrc, nullptr, p * PPW + i);
        if (mslice) return;  // M columns: u = 0
        const float* usrc = a.UT + cid * D * BT + (size_t)(vs * 16 * NW + li) * BT + 4 * lg;
#pragma unroll
        for (int j = 0; j < NW * NB / NP; ++j) {
          const int q = j * NP + p, w = q / NB, it = q % NB;
          lds_dma16(usrc + (size_t)w * 16 * BT + it * 16, &sU[q * 64]);
        }
      };
      auto issue_k = [&](int c) __attribute__((always_inline)) {
        const size_t cid = (size_t)bh * a.N + c0 + c;
        const char* ksrc = reinterpret_cast<const char*>(a.KgT + cid * D * BT);
#pragma unroll
        for (int i = 0; i < PPK; ++i) piece_dma(nullptr, ksrc, WPIECES + p * PPK + i);
        if (lane < GQ / 4) lds_dma16(a.GL + cid * D + p * GQ + lane * 4, sGL0 + p * GQ);
      };
      auto exp_q = [&]() __attribute__((always_inline)) {
        if (lane < GQ) sGL0[p * GQ + lane] = __expf(sGL0[p * GQ + lane]);
      };
      if (n > 0) {
        issue_w(0);
        issue_k(0);
      }
      if (n > 1) touch(1);
      for (int c = 0; c < n; ++c) {
        // in flight here (c > 0): W / u^T of chunk c, then kg^T / g_last of chunk
        // c (PPK + 1), then touch(c+1) if c+1 < n (NTP)
        const bool tch = c + 1 < n;
        if (c == 0) {
          if (tch) wait_vmcnt<NTP>();
          else wait_vmcnt<0>();
          exp_q();
        } else {
          if (tch) wait_vmcnt<PPK + 1 + NTP>();
          else wait_vmcnt<PPK + 1>();
        }
        barrier();  // A(c): W(c), u^T(c) resident
        barrier();  // B(c)
        if (c > 0) {
          if (tch) wait_vmcnt<NTP>();
          else wait_vmcnt<0>();
          exp_q();
        }
        barrier();  // X(c): kg^T(c), e^{g_last(c)} resident; W(c) no longer read
        if (c + 1 < n) issue_w(c + 1);
        barrier();  // E(c): kg^T(c) no longer read
        if (c + 1 < n) {
          issue_k(c + 1);
          if (c + 2 < n) touch(c + 2);
        }
      }
      return;
    }
    if (n > 0) issue(0, sbuf0, sGL0);
    if (n > 1) touch(1);
    // The next chunk's W / kg^T / g_last move once A(c) has passed (their buffer was
    // last read in chunk c-1), its u^T once B(c) has (one u^T buffer, read between
    // A(c) and B(c)); the touch comes last, so waiting for all but the touch waits
    // for both.
    for (int c = 0; c < n; c += 2) {
      wait_chunk(c);
      exp_gl(sGL0);
      barrier();  // A(c)
      if (c + 1 < n) issue(c + 1, sbuf1, sGL1, 1);
      barrier();  // B(c)
      if (c + 1 < n) {
        issue(c + 1, sbuf1, sGL1, 2);
        if (c + 2 < n) touch(c + 2);
        barrier();  // X(c)
        wait_chunk(c + 1);
        exp_gl(sGL1);
        barrier();  // A(c+1)
        if (c + 2 < n) issue(c + 2, sbuf0, sGL0, 1);
        barrier();  // B(c+1)
        if (c + 2 < n) issue(c + 2, sbuf0, sGL0, 2);
        if (c + 3 < n) touch(c + 3);
        barrier();  // X(c+1)
      } else {
        barrier();  // X(c)
      }
    }
    return;
  }

  // ---- compute waves ----------------------------------------------------------
  const int wcol = wv % NW, ks = wv / NW;          // column slice, k-half (K-split)
  const int col = vs * 16 * NW + wcol * 16 + li;
  // element offset of logical (row r, element e) in a tile whose rows hold `re` elements
  auto swz = [](int r, int e, int re) {
    const int nchunk = re / 4, m = (nchunk < 16 ? nchunk : 16) - 1;
    return r * re + (((e / 4) ^ (r & m)) * 4) + (e % 4);
  };

  // entry state: h0 (or 0) for a plain pass and for segment 0 of the summary
  // pass, 0 for later segments of the summary pass, the identity for M slices,
  // the combined entry state in the final segmented pass
  f32x4 h[NDH];   // row tiles at = ks NDH + i of this slice's h
  const float* hsrc = a.cu ? (a.h0 ? a.h0 + ((size_t)sg * a.H + bh) * D * D : nullptr)
                    : (a.S > 1 && !SUM) ? a.hin + ((size_t)unit) * D * D
                    : (sg == 0 && !mslice && a.h0) ? a.h0 + (size_t)bh * D * D : nullptr;
  if (mslice) {
#pragma unroll
    for (int i = 0; i < NDH; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        h[i][r] = ((ks * NDH + i) * 16 + 4 * lg + r == col) ? 1.f : 0.f;
  } else if (hsrc) {
#pragma unroll
    for (int i = 0; i < NDH; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        h[i][r] = sanitize(hsrc[(size_t)((ks * NDH + i) * 16 + 4 * lg + r) * D + col]);
  } else {
#pragma unroll
    for (int i = 0; i < NDH; ++i) h[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // segmented passes: whether a clip of the state bound (NaN included)
  const bool track = a.sat != nullptr && !mslice;
  bool bound = false;

  // One chunk: v_new = u - W h, h <- e^{gl} h + kg^T v_new, with chunk c in `cur`.
  auto step = [&](int c, const char* cur, const float* eglc) __attribute__((always_inline)) {
    const size_t cid = (size_t)bh * a.N + c0 + c;
    __syncthreads();  // A(c)
    f32x4 vn[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const uint4 pc = sU[(wcol * NB + q) * 64 + lane];
      vn[q] = mslice ? f32x4{0.f, 0.f, 0.f, 0.f} : __builtin_bit_cast(f32x4, pc);
    }
    __syncthreads();  // B(c)
    const float* sW = reinterpret_cast<const float*>(cur);
    const float* sK = reinterpret_cast<const float*>(cur + WBYTES);

    if constexpr (!SUM) {
      float* hT = a.HT + cid * D * D + (size_t)col * D;
#pragma unroll
      for (int i = 0; i < NDH; ++i) store4(hT + (ks * NDH + i) * 16 + 4 * lg, h[i]);
      // the stores go out here and below, not among the products (300 against 345 us
      // on 48 (b,h) of 128 chunks at D = 128)
      __builtin_amdgcn_sched_barrier(0);
    }

    // v_new -= W h: h split once per chunk, all row blocks independent (chunks 2p,
    // 2p+1 of a lane are one split pair)
    {
      auto wop = [&](int it, int kk) __attribute__((always_inline)) {
        return load4f(&sW[swz(it * 16 + li, (ks * NDH + kk) * 16 + 4 * lg, D)]);
      };
      f32x4 acc[NB];
      Split8 hs[NDH / 2];
#pragma unroll
      for (int p = 0; p < NDH / 2; ++p) hs[p] = split8(h[2 * p], h[2 * p + 1]);
#pragma unroll
      for (int it = 0; it < NB; ++it) acc[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < NDH / 2; ++p)
#pragma unroll
        for (int it = 0; it < NB; ++it)
          mma3(acc[it], split_read(wop(it, 2 * p), wop(it, 2 * p + 1)), hs[p]);
      // exchange the parts; both waves of the slice sum them in the order of the
      // k-parts, so both form the same v_new
#pragma unroll
      for (int it = 0; it < NB; ++it) sX[(wv * NB + it) * 64 + lane] = acc[it];
      lds_barrier();  // X(c)
#pragma unroll
      for (int it = 0; it < NB; ++it) {
        f32x4 sum = ks == 0 ? acc[it] : sX[(wcol * NB + it) * 64 + lane];
        sum += ks == 1 ? acc[it] : sX[((NW + wcol) * NB + it) * 64 + lane];
        vn[it] -= sum;
      }
    }
    if constexpr (!SUM) {
      float* vT = a.VnT + cid * D * BT + (size_t)col * BT;
#pragma unroll
      for (int it = ks * (NB / KS); it < (ks + 1) * (NB / KS); ++it)
        store4(vT + it * 16 + 4 * lg, vn[it]);
      __builtin_amdgcn_sched_barrier(0);
    }

    // h <- e^{g_last} h + kg^T v_new: v_new split once per chunk, the row tiles of h
    // independent accumulators
    {
#pragma unroll
      for (int i = 0; i < NDH; ++i) {
        const f32x4 egl = load4f(eglc + (ks * NDH + i) * 16 + 4 * lg);
#pragma unroll
        for (int r = 0; r < 4; ++r) h[i][r] *= egl[r];
      }
      auto kop = [&](int i, int kk) __attribute__((always_inline)) {
        return load4f(&sK[swz((ks * NDH + i) * 16 + li, kk * 16 + 4 * lg, BT)]);
      };
      Split8 vs2[NB / 2];
#pragma unroll
      for (int p = 0; p < NB / 2; ++p) vs2[p] = split8(vn[2 * p], vn[2 * p + 1]);
#pragma unroll
      for (int p = 0; p < NB / 2; ++p)
#pragma unroll
        for (int at = 0; at < NDH; ++at)
          mma3(h[at], split_read(kop(at, 2 * p), kop(at, 2 * p + 1)), vs2[p]);
      if (!mslice) {
        if (track) {
#pragma unroll
          for (int at = 0; at < NDH; ++at)
#pragma unroll
            for (int r2 = 0; r2 < 4; ++r2) bound = bound || !(fabsf(h[at][r2]) <= g_clip);
        }
#pragma unroll
        for (int at = 0; at < NDH; ++at)
#pragma unroll
          for (int r2 = 0; r2 < 4; ++r2) h[at][r2] = sanitize(h[at][r2]);
      }
    }
  };

  if constexpr (NBUF == 1) {
    for (int c = 0; c < n; ++c) {
      step(c, sbuf0, sGL0);
      __syncthreads();  // E(c)
    }
  } else {
    for (int c = 0; c < n; c += 2) {
      step(c, sbuf0, sGL0);
      if (c + 1 < n) step(c + 1, sbuf1, sGL1);
    }
  }
  if (track && __ballot(bound) != 0 && lane == 0) *a.sat = 1;
  float* hout = a.cu ? a.h_final + ((size_t)sg * a.H + bh) * D * D
              : SUM ? a.seg + ((size_t)unit * 2 + (mslice ? 1 : 0)) * D * D
              : (sg == a.S - 1) ? a.h_final + (size_t)bh * D * D : nullptr;
  if (hout) {
#pragma unroll
    for (int i = 0; i < NDH; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        hout[(size_t)((ks * NDH + i) * 16 + 4 * lg + r) * D + col] = h[i][r];
  }
}

// ---------------------------------------------------------------------------
// Backward state scan B1 (gdn2_bwd.py:45-80) of float32 tiles in fragments, the
// reverse of fwd_scan for the same few units (scan_rows in gdn2_layout.h):
//   dv_new = dvp + kg dh,   dh <- e^{g_last} dh + scale qg^T do - W^T dv_new.
// Both products contract over the other index than the forward's, so their
// fragments are those of the transposed tiles (frag_transpose below).
struct BScanArgs {
  const float* Kg;    // [cid] kg [t][d] in split fragments
  const float* WT;    // [cid] -W^T [d][t] in split fragments
  const float* GL;    // [cid][D] gc_last
  const float* DVPT;  // [cid][D][BT]  (Aqk^T do)^T
  const float* QDOT;  // [cid][D][D]   (scale qg^T do)^T
  const float* dh_final;  // nullable, (B,H,D,D)
  float* DHT;         // [cid][D][D]   dh_{c+1}^T
  float* DVNT;        // [cid][D][BT]  dv_new^T
  float* dh0;         // (B,H,D,D)
  int N, units;
  const int* cu;      // variable-length batch (B = 1): unit (h, sequence s) scans chunks
                      // [cu[s], cu[s+1]) in reverse; dh_final / dh0 are [s][h][D][D]
  int S, H;           // sequences and heads of a variable-length batch
};

// One workgroup: one unit and 16 value columns of dh, KS state waves (D / KS rows
// each) and a helper wave; loads, the exchange and the barriers E and X(i) as in
// fwd_scan, step i on chunk n-1-i.  dvp and qdot come with the tiles' loads.
template <int BT, int D, int KS>
__global__ void __launch_bounds__(64 * (KS + 1)) bwd_scan(BScanArgs a) {
  constexpr int NB = BT / 16, NDT = D / 16, NKT = BT / 32;
  constexpr int NDH = NDT / KS, NKD = NDH / 2;
  constexpr int NVS = D / 16;
  constexpr int FK = NB * NKD * 2, FW = NDH * NKT * 2;   // fragments of kg, W^T per wave
  constexpr int NSET = FK + FW <= (KS < 3 ? 32 : 16) ? 2 : 1;
  static_assert(NDT % (2 * KS) == 0 && NB % KS == 0, "waves must split the tiles");
  __shared__ __align__(16) f32x4 sP[2 * KS * NB * 64];
  __shared__ __align__(16) float sEg[2 * D];
  __shared__ __align__(16) float sJunk[64];

  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = blockIdx.x / 8;                       // units and slices as in fwd_scan
  const int unit = (slot / NVS) * 8 + blockIdx.x % 8, vs = slot % NVS;
  if (unit >= a.units) return;
  int bh = unit, c0 = 0, n = a.N;
  size_t st_idx = (size_t)unit;          // index of this unit's dh_final / dh0
  if (a.cu) {
    const int sg = unit % a.S;
    bh = unit / a.S;
    const SeqChunks sc = seq_chunks(a.cu, sg, a.N);
    c0 = sc.c0;
    n = sc.n;
    st_idx = (size_t)sg * a.H + bh;
  }
  auto chunk_id = [&](int i) { return (size_t)bh * a.N + c0 + (i < n ? n - 1 - i : 0); };

  if (wv == KS) {
    // ---- helper: L2 touches and e^{g_last}, as in fwd_scan -------------------------
    constexpr int LINE = 128, AHEAD = 3;
    constexpr int LW = BT * D * 4 / LINE, LU = 16 * BT * 4 / LINE, LQ = 16 * D * 4 / LINE;
    constexpr int LSL = 2 * LW / NVS;                    // shared lines touched here
    constexpr int LTOT = LSL + LU + LQ, NTP = (LTOT + 63) / 64;
    static_assert(2 * LW % NVS == 0, "the shared lines must split over the slices");
    auto touch = [&](int i) __attribute__((always_inline)) {
      const size_t cid = chunk_id(i);
      const char* ksrc = reinterpret_cast<const char*>(a.Kg + cid * BT * D);
      const char* wsrc = reinterpret_cast<const char*>(a.WT + cid * BT * D);
      const char* dsrc = reinterpret_cast<const char*>(a.DVPT + cid * D * BT + (size_t)vs * 16 * BT);
      const char* qsrc = reinterpret_cast<const char*>(a.QDOT + cid * D * D + (size_t)vs * 16 * D);
#pragma unroll
      for (int j = 0; j < NTP; ++j) {
        const int l = min(j * 64 + lane, LTOT - 1), lw = vs * LSL + l;
        const char* src = l < LSL ? (lw < LW ? ksrc + lw * LINE : wsrc + (lw - LW) * LINE)
                        : l < LSL + LU ? dsrc + (l - LSL) * LINE : qsrc + (l - LSL - LU) * LINE;
        lds_dma4(src, sJunk);
      }
    };
    constexpr int GPL = D / 64;
    float g0[GPL], g1[GPL];
    auto load_gl = [&](int i, float* g) __attribute__((always_inline)) {
      const float* src = a.GL + chunk_id(i) * D;
#pragma unroll
      for (int j = 0; j < GPL; ++j) g[j] = src[j * 64 + lane];
    };
    auto put_eg = [&](int i, const float* g) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < GPL; ++j) sEg[(i & 1) * D + j * 64 + lane] = __expf(g[j]);
    };
    auto hstep = [&](int i, float* g) __attribute__((always_inline)) {
      put_eg(i + 1, g);
      load_gl(i + 3, g);
      touch(i + AHEAD);
      lds_barrier();  // X(i)
    };
    if (n > 0) {
      load_gl(0, g0);
      put_eg(0, g0);
      load_gl(1, g1);
      load_gl(2, g0);
      for (int i = 1; i < AHEAD; ++i) touch(i);
    }
    lds_barrier();    // E
    int i = 0;
    for (; i + 1 < n; i += 2) {
      hstep(i, g1);
      hstep(i + 1, g0);
    }
    if (i < n) hstep(i, g1);
    wait_vmcnt<0>();  // no DMA into this workgroup's LDS outlives it
    return;
  }

  // ---- state waves --------------------------------------------------------------
  const float clip = g_clip;
  const int ks = wv, row0 = ks * NDH * 16, col = vs * 16 + li;
  f32x4 dh[NDH];
#pragma unroll
  for (int j = 0; j < NDH; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      dh[j][r] = a.dh_final
          ? a.dh_final[(st_idx * D + row0 + j * 16 + 4 * lg + r) * D + col] : 0.f;
  // The last chunk's dh' is dh_final as given: B3 takes it raw (gdn2_pipeline.py:
  // 52-56,105) while the carry starts from its sanitized value (gdn2_bwd.py:53)
  if (n > 0) {
    float* dht = a.DHT + chunk_id(0) * D * D + (size_t)col * D + row0;
#pragma unroll
    for (int j = 0; j < NDH; ++j) store4(dht + j * 16 + 4 * lg, dh[j]);
  }
#pragma unroll
  for (int j = 0; j < NDH; ++j) dh[j] = sanitize4(dh[j]);

  bf16x8 Kf[NSET][FK], Wf[NSET][FW];
  f32x4 Uf[NSET][NB], Qf[NSET][NDH];
  constexpr int TILE = BT * D * 4;
  const int vl16 = lane * 16;
  auto load_k = [&](int s, Rsrc r, int it, int kk) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
      Kf[s][(kk * NB + it) * 2 + p] = __builtin_bit_cast(
          bf16x8, tile_load(r, vl16, ((it * KS + ks) * NKD + kk) * 2048 + p * 1024));
  };
  auto load_w = [&](int s, Rsrc r, int j, int q) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
      Wf[s][(q * NDH + j) * 2 + p] = __builtin_bit_cast(
          bf16x8, tile_load(r, vl16, ((ks * NDH + j) * NKT + q) * 2048 + p * 1024));
  };
  auto k_rsrc = [&](int i) { return tile_rsrc(a.Kg + chunk_id(i) * BT * D, TILE); };
  auto w_rsrc = [&](int i) { return tile_rsrc(a.WT + chunk_id(i) * BT * D, TILE); };
  // dvp^T and qdot rows of this workgroup's columns (row pitch BT and D floats)
  auto load_u = [&](int s, int i) __attribute__((always_inline)) {
    const Rsrc r = tile_rsrc(a.DVPT + chunk_id(i) * BT * D, TILE);
#pragma unroll
    for (int it = 0; it < NB; ++it)
      Uf[s][it] = __builtin_bit_cast(
          f32x4, tile_load(r, (li * BT + 4 * lg) * 4, (vs * 16 * BT + it * 16) * 4));
  };
  auto load_q = [&](int s, int i) __attribute__((always_inline)) {
    const Rsrc r = tile_rsrc(a.QDOT + chunk_id(i) * D * D, D * D * 4);
#pragma unroll
    for (int j = 0; j < NDH; ++j)
      Qf[s][j] = __builtin_bit_cast(
          f32x4, tile_load(r, (li * D + 4 * lg) * 4, (vs * 16 * D + row0 + j * 16) * 4));
  };

  // memory operations of a step, in issue order: FK + NB loads and STH stores in P1,
  // FW + NDH loads and STV stores in P3
  constexpr int STH = NDH, STV = NB / KS;
  auto step = [&](int i, auto sc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value;
    // ---- P1: this wave's part of kg dh ----------------------------------------------
    f32x4 eg[NDH];
#pragma unroll
    for (int j = 0; j < NDH; ++j) eg[j] = load4f(&sEg[(i & 1) * D + row0 + j * 16 + 4 * lg]);
    wait_counts<NSET == 2 ? 2 * (FW + NDH) + FK + NB + 2 * STV + STH : FW + NDH + STV, 15>();
    const Rsrc rk = k_rsrc(i + NSET);
    f32x4 dvn[NB], dvp[NB];
#pragma unroll
    for (int it = 0; it < NB; ++it) {
      dvn[it] = f32x4{0.f, 0.f, 0.f, 0.f};
      dvp[it] = Uf[s][it];
    }
#pragma unroll
    for (int kk = 0; kk < NKD; ++kk) {
      const Split8 y = split8(dh[2 * kk], dh[2 * kk + 1]);
#pragma unroll
      for (int it = 0; it < NB; ++it) {
        mma3(dvn[it], Split8{Kf[s][(kk * NB + it) * 2], Kf[s][(kk * NB + it) * 2 + 1]}, y);
        load_k(s, rk, it, kk);
      }
    }
    load_u(s, i + NSET);
#pragma unroll
    for (int it = 0; it < NB; ++it) sP[((i & 1) * KS + ks) * NB * 64 + it * 64 + lane] = dvn[it];
    if (i > 0) {   // dh_{c+1} (chunk n-1's was stored raw before the scan)
      float* dht = a.DHT + chunk_id(i) * D * D + (size_t)col * D + row0;
#pragma unroll
      for (int j = 0; j < NDH; ++j) store4(dht + j * 16 + 4 * lg, dh[j]);
    }
    lds_barrier();  // X(i)
    // ---- P3: dv_new, then dh ---------------------------------------------------------
#pragma unroll
    for (int it = 0; it < NB; ++it) {
      auto part = [&](int k) __attribute__((always_inline)) {
        return sP[((i & 1) * KS + k) * NB * 64 + it * 64 + lane];
      };
      f32x4 sum;
      if constexpr (KS == 2) {   // two parts: the same sum in either order
        sum = dvn[it] + part(1 - ks);
      } else {
        sum = part(0);
#pragma unroll
        for (int k = 1; k < KS; ++k) sum += part(k);
      }
      dvn[it] = dvp[it] + sum;
    }
    sanitize_all(dvn, NB, clip);
    wait_counts<NSET == 2 ? 2 * (FK + NB) + FW + NDH + 2 * STH + STV : FK + NB + STH, 15>();
    const Rsrc rw = w_rsrc(i + NSET);
    f32x4 acc[NDH];
#pragma unroll
    for (int j = 0; j < NDH; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NKT; ++q) {
      const Split8 y = split8(dvn[2 * q], dvn[2 * q + 1]);
#pragma unroll
      for (int j = 0; j < NDH; ++j) {
        mma3(acc[j], Split8{Wf[s][(q * NDH + j) * 2], Wf[s][(q * NDH + j) * 2 + 1]}, y);
        load_w(s, rw, j, q);
      }
    }
#pragma unroll
    for (int j = 0; j < NDH; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) dh[j][r] = eg[j][r] * dh[j][r] + Qf[s][j][r] + acc[j][r];
    load_q(s, i + NSET);
    // each wave stores its share of dv_new
    float* dvo = a.DVNT + chunk_id(i) * D * BT + (size_t)col * BT;
#pragma unroll
    for (int jj = 0; jj < NB / KS; ++jj) {
      f32x4 x = dvn[jj * KS];
#pragma unroll
      for (int k = 1; k < KS; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = ks == k ? dvn[jj * KS + k][r] : x[r];
      store4(dvo + (jj * KS + ks) * 16 + 4 * lg, x);
    }
    sanitize_all(dh, NDH, clip);
  };

  if (n > 0) {
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
      const Rsrc rk = k_rsrc(s), rw = w_rsrc(s);
#pragma unroll
      for (int kk = 0; kk < NKD; ++kk)
#pragma unroll
        for (int it = 0; it < NB; ++it) load_k(s, rk, it, kk);
      load_u(s, s);
#pragma unroll
      for (int q = 0; q < NKT; ++q)
#pragma unroll
        for (int j = 0; j < NDH; ++j) load_w(s, rw, j, q);
      load_q(s, s);
    }
    lds_barrier();  // E
    if constexpr (NSET == 1) {
      for (int i = 0; i < n; ++i) step(i, std::integral_constant<int, 0>{});
    } else {
      int i = 0;
      for (; i + 1 < n; i += 2) {
        step(i, std::integral_constant<int, 0>{});
        step(i + 1, std::integral_constant<int, 1>{});
      }
      if (i < n) step(i, std::integral_constant<int, 0>{});
    }
  } else {
    lds_barrier();  // E
  }
#pragma unroll
  for (int j = 0; j < NDH; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      a.dh0[(st_idx * D + row0 + j * 16 + 4 * lg + r) * D + col] = dh[j][r];
}

// Split-fragment tiles [R][K] (R K / 512 fragments of hi then lo parts) into those of
// the transposed tiles [K][R], hi and lo moved as they are: workgroup 2 m + part of
// the first half of the grid takes one part of tile m of `a` ([BT][D]), of the second
// half of tile m of `b` ([D][BT]), through LDS in fragment order.
template <int BT, int D>
__global__ void __launch_bounds__(256) frag_transpose(const float* a, float* at, const float* b,
                                                      float* bt, int n) {
  constexpr int ELEMS = BT * D, PIECES = ELEMS / 8;   // 16-byte pieces of one part
  __shared__ __align__(16) bf16_t s[ELEMS];
  const bool second = (int)blockIdx.x >= 2 * n;
  const int id = (int)blockIdx.x - (second ? 2 * n : 0);
  const int part = id & 1;
  const size_t off = (size_t)(id >> 1) * ELEMS * 2;
  const bf16_t* src = reinterpret_cast<const bf16_t*>(second ? b : a) + off;
  bf16_t* dst = reinterpret_cast<bf16_t*>(second ? bt : at) + off;
  for (int i = threadIdx.x; i < PIECES; i += 256)
    *reinterpret_cast<uint4*>(&s[i * 8]) =
        *reinterpret_cast<const uint4*>(src + ((i / 64) * 2 + part) * 512 + (i % 64) * 8);
  __syncthreads();
  auto move = [&](auto kc) __attribute__((always_inline)) {
    constexpr int K = decltype(kc)::value, R = ELEMS / K;   // the source is [R][K]
    for (int i = threadIdx.x; i < PIECES; i += 256) {
      const int f = i / 64, ln = i % 64;
      const int row = (f / (R / 32)) * 16 + ln % 16;        // of the transposed tile
      const int k0 = (f % (R / 32)) * 32 + (ln / 16) * 4;
      bf16x8 x;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = s[frag_off<K>(k0 + (e / 4) * 16 + e % 4, row)];
      *reinterpret_cast<bf16x8*>(dst + (f * 2 + part) * 512 + ln * 8) = x;
    }
  };
  if (second) move(std::integral_constant<int, BT>{});
  else move(std::integral_constant<int, D>{});
}

// Workgroups of a scan over `units` units (the padding of the XCD mapping included).
inline unsigned scan_grid(size_t units, int slices) {
  return (unsigned)((units + 7) / 8 * 8 * slices);
}

}  // namespace gdn2
