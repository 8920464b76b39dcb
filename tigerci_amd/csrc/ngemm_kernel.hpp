// Kernel templates of ngemm.hpp (instantiated by ngemm_f64.hip and
// ngemm_s16.hip).
#pragma once

#include "ngemm.hpp"

namespace tci {

namespace {

typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __attribute__((aligned(16))) u4 nzero[1];

// ---- element types ----------------------------------------------------------
// Swizzle: 16-byte chunk c of LDS row r sits at position c ^ sw(r).  A 128-bit
// LDS read is served 16 lanes at a time, lanes 8q .. 8q+7 with the lanes 16
// further, over 256 bytes of banks (two rows): the 16 x 16 FP64 fragments read
// chunks c, c + 1 of rows r .. r+7 in one pass, the 16 x 16 split fragments
// chunks c, c + 2 of rows r .. r+7, the 32 x 32 ones chunk c of rows r .. r+7
// and r+16 .. r+23.  Each sw makes those sixteen addresses distinct.

// FP64, v_mfma_f64_16x16x4: A[i][k] lane i + 16k, B[k][j] lane j + 16k,
// D[i][j] lane j + 16 (i % 4), register i / 4.  A lane group lg reads the two
// values k = 2 lg, 2 lg + 1 of each run of 8 as one 16-byte chunk and feeds
// them to two MFMAs (the same order of k for both operands).
struct F64T {
  static constexpr int BS = 16;     // block side
  typedef d4 Acc;
  static __device__ __forceinline__ int sw(int r) { return ((r >> 1) & 3) << 1; }
  static __device__ __forceinline__ Acc zero() { return d4{0.0, 0.0, 0.0, 0.0}; }
};

template <int PREC>
struct NV;

template <int PREC>
struct S16T {
  static constexpr int BS = 16;
  typedef f4 Acc;
  typedef typename NV<PREC>::T T16;
  static __device__ __forceinline__ int sw(int r) { return ((r >> 1) & 1) | (((r >> 2) & 1) << 2); }
  static __device__ __forceinline__ Acc zero() { return f4{0.f, 0.f, 0.f, 0.f}; }
};

template <int PREC>
struct S32T {
  static constexpr int BS = 32;
  typedef f16v Acc;
  typedef typename NV<PREC>::T T16;
  static __device__ __forceinline__ int sw(int r) { return ((r >> 1) & 3) | (((r >> 4) & 1) << 2); }
  static __device__ __forceinline__ Acc zero() {
    f16v z;
#pragma unroll
    for (int e = 0; e < 16; ++e) z[e] = 0.f;
    return z;
  }
};

template <>
struct NV<TCI_SIGMA_BF16X3> {
  typedef __bf16 T;
  typedef bf16x8 V;
  static __device__ __forceinline__ f4 mfma(V a, V b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ f16v mfma32(V a, V b, f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct NV<TCI_SIGMA_FP16X3> {
  typedef _Float16 T;
  typedef h8 V;
  static __device__ __forceinline__ f4 mfma(V a, V b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ f16v mfma32(V a, V b, f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};

// ---- staging ------------------------------------------------------------------
// NI loads of one wave for one operand of R rows and NWK k-chunks: load q
// covers 8 rows (lane / 8) of k-chunk sub(q).
// Groups of 8 rows wholly outside the output are not loaded when SKIP is set
// (their LDS rows then hold anything, which only reaches products that are not
// stored); three-stage kernels count their loads in flight and load them all.
template <class TT, int R, int NWK, int NW, bool SKIP>
struct NStage {
  static constexpr int NI = NWK * R / (8 * NW);
  static_assert(NI * 8 * NW == NWK * R, "loads divide evenly over the waves");
  uint32_t off[NI];
  // per-lane byte offsets from the segment's base; rows clamped to `rows`.
  // Gathered rows count from the operand's base, plain ones from the tile's
  // first row.  The map reads are waited for inside their branch: plain
  // segments then pass from one to the next with loads in flight.
  __device__ __forceinline__ void set(int w, int lane, const int32_t* map, int64_t ld, int r0, int rows) {
    uint32_t row[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
      const int ins = w * NI + q, r = (ins % (R / 8)) * 8 + (lane >> 3);
      row[q] = (uint32_t)(min(r0 + r, rows - 1) - r0);
    }
    if (map) {
#pragma unroll
      for (int q = 0; q < NI; ++q) row[q] = (uint32_t)gld(map + r0 + row[q]);
#pragma unroll
      for (int q = 0; q < NI; ++q) asm volatile("" : "+v"(row[q]));
    }
#pragma unroll
    for (int q = 0; q < NI; ++q) {
      const int ins = w * NI + q, sub = ins / (R / 8), r = (ins % (R / 8)) * 8 + (lane >> 3);
      off[q] = row[q] * (uint32_t)ld + (uint32_t)(((lane & 7) ^ TT::sw(r)) * 16 + sub * 128);
    }
  }
  // rem: bytes of k left in the segment from this step on
  __device__ __forceinline__ void issue(int w, int lane, const char* base, int rem, char* lds, int rowbase,
                                        int stride, int valid) const {
    const bool whole = rem >= NWK * 128;
#pragma unroll
    for (int q = 0; q < NI; ++q) {
      const int ins = w * NI + q, sub = ins / (R / 8), r8 = ins % (R / 8);
      if (SKIP && r8 * 8 >= valid) continue;
      char* dst = lds + sub * stride + (rowbase + r8 * 8) * 128;
      if (whole) {
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(base + off[q]),
                                         (void __attribute__((address_space(3)))*)dst, 16, 0, 0);
      } else {
        const int r = r8 * 8 + (lane >> 3);
        const int kb = sub * 128 + ((lane & 7) ^ TT::sw(r)) * 16;
        const char* p = kb < rem ? base + off[q] : (const char*)nzero;
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)p,
                                         (void __attribute__((address_space(3)))*)dst, 16, 0, 0);
      }
    }
  }
};

// ---- one 128-byte k-step of a wave's blocks -----------------------------------
template <class TT, int NWM, int NWN, int BM, int BN>
struct NStep;

template <int NWM, int NWN, int BM, int BN>
struct NStep<F64T, NWM, NWN, BM, BN> {
  template <bool FULL>
  static __device__ __forceinline__ void run(const char* sa, const char* sb, int wr, int wc, int lane, int nbm, int nbn,
                                             d4 (&acc)[BM][BN]) {
    const int li = lane & 15, lg = lane >> 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      d2 a[BM], b[BN];
#pragma unroll
      for (int i = 0; i < BM; ++i) {
        const int r = 16 * (wr + NWM * i) + li;
        a[i] = *reinterpret_cast<const d2*>(sa + r * 128 + (((4 * h + lg) ^ F64T::sw(r)) << 4));
      }
#pragma unroll
      for (int j = 0; j < BN; ++j) {
        const int r = 16 * (wc + NWN * j) + li;
        b[j] = *reinterpret_cast<const d2*>(sb + r * 128 + (((4 * h + lg) ^ F64T::sw(r)) << 4));
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < BM; ++i)
          if (FULL || i < nbm) {
#pragma unroll
            for (int j = 0; j < BN; ++j)
              if (FULL || j < nbn) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
          }
    }
  }
};

template <int PREC, int NWM, int NWN, int BM, int BN>
struct NStep<S16T<PREC>, NWM, NWN, BM, BN> {
  template <bool FULL>
  static __device__ __forceinline__ void run(const char* sa, const char* sb, int wr, int wc, int lane, int nbm, int nbn,
                                             f4 (&acc)[BM][BN]) {
    typedef typename NV<PREC>::V V;
    const int li = lane & 15, lg = lane >> 4;
    V ah[BM], al[BM], bh[BN], bl[BN];
#pragma unroll
    for (int i = 0; i < BM; ++i) {
      const int r = 16 * (wr + NWM * i) + li, s = S16T<PREC>::sw(r);
      ah[i] = *reinterpret_cast<const V*>(sa + r * 128 + (((2 * lg) ^ s) << 4));
      al[i] = *reinterpret_cast<const V*>(sa + r * 128 + (((2 * lg + 1) ^ s) << 4));
    }
#pragma unroll
    for (int j = 0; j < BN; ++j) {
      const int r = 16 * (wc + NWN * j) + li, s = S16T<PREC>::sw(r);
      bh[j] = *reinterpret_cast<const V*>(sb + r * 128 + (((2 * lg) ^ s) << 4));
      bl[j] = *reinterpret_cast<const V*>(sb + r * 128 + (((2 * lg + 1) ^ s) << 4));
    }
    // small terms first; B goes in as the MFMA's first operand, so a lane ends
    // with four consecutive columns of one row
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int i = 0; i < BM; ++i)
        if (FULL || i < nbm) {
#pragma unroll
          for (int j = 0; j < BN; ++j)
            if (FULL || j < nbn)
              acc[i][j] = NV<PREC>::mfma(p == 1 ? bl[j] : bh[j], p == 0 ? al[i] : ah[i], acc[i][j]);
        }
  }
};

template <int PREC, int NWM, int NWN, int BM, int BN>
struct NStep<S32T<PREC>, NWM, NWN, BM, BN> {
  template <bool FULL>
  static __device__ __forceinline__ void run(const char* sa, const char* sb, int wr, int wc, int lane, int nbm, int nbn,
                                             f16v (&acc)[BM][BN]) {
    typedef typename NV<PREC>::V V;
    const int lr = lane & 31, hs = lane >> 5;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = 2 * (2 * h + hs);
      V ah[BM], al[BM], bh[BN], bl[BN];
#pragma unroll
      for (int i = 0; i < BM; ++i) {
        const int r = 32 * (wr + NWM * i) + lr, s = S32T<PREC>::sw(r);
        ah[i] = *reinterpret_cast<const V*>(sa + r * 128 + ((c ^ s) << 4));
        al[i] = *reinterpret_cast<const V*>(sa + r * 128 + (((c + 1) ^ s) << 4));
      }
#pragma unroll
      for (int j = 0; j < BN; ++j) {
        const int r = 32 * (wc + NWN * j) + lr, s = S32T<PREC>::sw(r);
        bh[j] = *reinterpret_cast<const V*>(sb + r * 128 + ((c ^ s) << 4));
        bl[j] = *reinterpret_cast<const V*>(sb + r * 128 + (((c + 1) ^ s) << 4));
      }
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < BM; ++i)
          if (FULL || i < nbm) {
#pragma unroll
            for (int j = 0; j < BN; ++j)
              if (FULL || j < nbn)
                acc[i][j] = NV<PREC>::mfma32(p == 1 ? bl[j] : bh[j], p == 0 ? al[i] : ah[i], acc[i][j]);
          }
    }
  }
};

// ---- epilogue -------------------------------------------------------------------
__device__ __forceinline__ int64_t nrow_off(const Task& t, int row) {
  return t.rdiv ? (int64_t)(row / t.rdiv) * t.rstride + (int64_t)(row % t.rdiv) * t.ldc : (int64_t)row * t.ldc;
}
__device__ __forceinline__ int64_t ncol_off(const Task& t, int col) {
  if (!t.cdiv) return col;
  const int cb = col / t.cdiv;
  return (int64_t)cb * t.cstride + (col - cb * t.cdiv);
}
__device__ __forceinline__ void nput(const Task& t, int64_t o, double v) {
  __attribute__((address_space(1))) double* p = (__attribute__((address_space(1))) double*)(t.C + o);
  *p = t.accumulate ? *p + v : v;
}

template <class TT, int NWM, int NWN, int BM, int BN>
__device__ __forceinline__ void nstore(const Task& t, const float*, const d4 (&acc)[BM][BN], int wr, int wc, int lane) {
  const int li = lane & 15, lg = lane >> 4;
  int64_t co[BN];
#pragma unroll
  for (int j = 0; j < BN; ++j) co[j] = ncol_off(t, t.n0 + 16 * (wc + NWN * j) + li);
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = t.m0 + 16 * (wr + NWM * i) + lg + 4 * r;
      if (row >= t.M) continue;
      const int64_t ro = nrow_off(t, row);
#pragma unroll
      for (int j = 0; j < BN; ++j)
        if (t.n0 + 16 * (wc + NWN * j) + li < t.N) nput(t, ro + co[j], acc[i][j][r]);
    }
}

// four consecutive columns col .. col+3 of one row.  out_split (see NProgram):
// C holds FP32 values.
__device__ __forceinline__ void nput4(const Task& t, int row, int col, const float* v) {
  const int64_t ro = nrow_off(t, row);
  const int cc = t.cdiv ? col % t.cdiv : col;
  const bool whole = t.cdiv ? ((cc & 3) == 0 && cc + 3 < t.cdiv && col + 3 < t.N) : col + 3 < t.N;
  if (t.out_split) {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // ldc is arbitrary
    __attribute__((address_space(1))) float* C = (__attribute__((address_space(1))) float*)t.C;
    if (whole) {
      const f4u o = {v[0], v[1], v[2], v[3]};
      *(__attribute__((address_space(1))) f4u*)(C + ro + ncol_off(t, col)) = o;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (col + r < t.N) C[ro + ncol_off(t, col + r)] = v[r];
    }
    return;
  }
  if (whole) {
    typedef double d4u __attribute__((ext_vector_type(4), aligned(8)));
    __attribute__((address_space(1))) d4u* p = (__attribute__((address_space(1))) d4u*)(t.C + ro + ncol_off(t, col));
    const d4u o = {(double)v[0], (double)v[1], (double)v[2], (double)v[3]};
    if (t.accumulate) *p = *p + o;
    else *p = o;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (col + r < t.N) nput(t, ro + ncol_off(t, col + r), (double)v[r]);
  }
}

template <class TT, int NWM, int NWN, int BM, int BN>
__device__ __forceinline__ void nstore(const Task& t, const float* scales, const f4 (&acc)[BM][BN], int wr, int wc,
                                       int lane) {
  const int li = lane & 15, lg = lane >> 4;
  const float osc = t.oscale >= 0 ? scales[t.oscale] : 1.f;
#pragma unroll
  for (int i = 0; i < BM; ++i) {
    const int row = t.m0 + 16 * (wr + NWM * i) + li;
    if (row >= t.M) continue;
#pragma unroll
    for (int j = 0; j < BN; ++j) {
      const int col = t.n0 + 16 * (wc + NWN * j) + 4 * lg;
      const f4 v = acc[i][j] * osc;
      const float x[4] = {v[0], v[1], v[2], v[3]};
      if (col < t.N) nput4(t, row, col, x);
    }
  }
}

template <class TT, int NWM, int NWN, int BM, int BN>
__device__ __forceinline__ void nstore(const Task& t, const float* scales, const f16v (&acc)[BM][BN], int wr, int wc,
                                       int lane) {
  const int lr = lane & 31, hs = lane >> 5;
  const float osc = t.oscale >= 0 ? scales[t.oscale] : 1.f;
#pragma unroll
  for (int i = 0; i < BM; ++i) {
    const int row = t.m0 + 32 * (wr + NWM * i) + lr;
    if (row >= t.M) continue;
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = t.n0 + 32 * (wc + NWN * j) + 8 * g + 4 * hs;
        const float x[4] = {acc[i][j][4 * g] * osc, acc[i][j][4 * g + 1] * osc, acc[i][j][4 * g + 2] * osc,
                            acc[i][j][4 * g + 3] * osc};
        if (col < t.N) nput4(t, row, col, x);
      }
  }
}

// ---- kernel ---------------------------------------------------------------------
// Column of wave wq.  With 2 x 4 waves, w and w + 4 share a SIMD: the second
// row of waves is rotated by two columns, so that in a ragged tile (say 10
// column blocks: 3, 3, 2, 2) every SIMD gets one long and one short wave.
template <int NWM, int NWN>
__device__ __forceinline__ int nwave_col(int wq) {
  return NWM == 2 && NWN == 4 ? (wq + 2 * (wq >> 2)) & 3 : wq % NWN;
}

template <class TT, int NWM, int NWN, int NWK, int BM, int BN, int NST, bool FULL>
__device__ __forceinline__ void nbody(const Task& t, const NSeg* __restrict__ segs, int64_t J0,
                                      const float* __restrict__ scales, char* sm, int w, int lane, int nbm, int nbn) {
  constexpr int NW = NWM * NWN * NWK;
  constexpr int TM = TT::BS * NWM * BM, TN = TT::BS * NWN * BN;
  constexpr int SUB = (TM + TN) * 128, STG = NWK * SUB;
  typedef NStage<TT, TM, NWK, NW, NST == 2 && !FULL> SA;
  typedef NStage<TT, TN, NWK, NW, NST == 2 && !FULL> SB;
  constexpr int PER = SA::NI + SB::NI;
  static_assert(NST == 2 || (NST == 3 && PER <= 15), "two stages, or three within the vmcnt field");
  const int kg = w / (NWM * NWN), wq = w % (NWM * NWN), wr = wq / NWN, wc = nwave_col<NWM, NWN>(wq);
  typename TT::Acc acc[BM][BN];
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j) acc[i][j] = TT::zero();
  SA la;
  SB lb;
  int seg = t.seg0;
  const char *pa = nullptr, *pb = nullptr;
  int rem = 0, reps = 0;  // bytes left of this pass over the range, passes left
  // first segment with work from `seg` on: sets the load state, false at the end
  auto open = [&]() -> bool {
    while (seg < t.seg1) {
      const NSeg& S = segs[seg];
      rem = (int)S.kbytes;
      if (rem > 0) {
        pa = static_cast<const char*>(S.A) + J0 * S.ja + (S.am ? 0 : (int64_t)t.m0 * S.lda);
        pb = static_cast<const char*>(S.B) + J0 * S.jb + (S.bm ? 0 : (int64_t)t.n0 * S.ldb);
        la.set(w, lane, S.am, S.lda, t.m0, t.M);
        lb.set(w, lane, S.bm, S.ldb, t.n0, t.N);
        reps = (int)S.reps - 1;
        return true;
      }
      seg = __builtin_amdgcn_readfirstlane(seg + 1);
    }
    return false;
  };
  auto issue = [&](char* buf) {
    la.issue(w, lane, pa, rem, buf, 0, SUB, t.M - t.m0);
    lb.issue(w, lane, pb, rem, buf, TM, SUB, t.N - t.n0);
    pa += NWK * 128;
    pb += NWK * 128;
    rem -= NWK * 128;
  };
  auto step = [&]() -> bool {  // is there a further stage to load?
    if (rem > 0) return true;
    if (reps > 0) {  // the same rows again, sa and sb bytes further
      const NSeg& S = segs[seg];
      const int kb = (int)S.kbytes, used = kb - rem;  // rem <= 0: what the last step ran over
      --reps;
      pa += S.sa - used;
      pb += S.sb - used;
      rem = kb;
      return true;
    }
    seg = __builtin_amdgcn_readfirstlane(seg + 1);
    return open();
  };
  bool more = open();
  int ahead = 0;  // stages in flight beyond the current one
  if (more) {
    issue(sm);
    more = step();
    if (NST == 3 && more) {
      issue(sm + STG);
      more = step();
      ahead = 1;
    }
    int cb = 0;
    while (true) {
      if (NST == 3 && ahead) __builtin_amdgcn_s_waitcnt(0x0F70 | PER);  // vmcnt(PER): this stage has landed
      else __builtin_amdgcn_s_waitcnt(0x0F70);                          // vmcnt(0)
      __builtin_amdgcn_s_barrier();  // every wave's loads of this stage are in LDS; the oldest buffer is free
      bool issued = false;
      if (more) {
        issue(sm + (NST == 2 ? cb ^ 1 : (cb + 2) % 3) * STG);
        more = step();
        issued = true;
      }
      const char* sa = sm + cb * STG + kg * SUB;
      if (FULL || (nbm > 0 && nbn > 0))
        NStep<TT, NWM, NWN, BM, BN>::template run<FULL>(sa, sa + TM * 128, wr, wc, lane, nbm, nbn, acc);
      if (!ahead && !issued) break;
      cb = NST == 2 ? cb ^ 1 : (cb + 1) % 3;
      ahead = NST == 3 && issued ? 1 : 0;
    }
  }
  if constexpr (NWK > 1) {  // sum the K-groups in LDS, group 0 stores
    typedef typename TT::Acc Acc;
    __syncthreads();
    Acc* red = reinterpret_cast<Acc*>(sm);
    static_assert((NWK - 1) * NWM * NWN * BM * BN * 64 * (int)sizeof(Acc) <= NST * STG, "reduction fits the stages");
    if (kg > 0)
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j) red[((((kg - 1) * NWM * NWN + wq) * BM + i) * BN + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 0; g < NWK - 1; ++g)
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j) acc[i][j] += red[(((g * NWM * NWN + wq) * BM + i) * BN + j) * 64 + lane];
  }
  nstore<TT, NWM, NWN, BM, BN>(t, scales, acc, wr, wc, lane);
}

// FULL bodies have no block predicates; a wave takes the predicated body when
// part of its blocks lies outside the output (both execute the same loads and
// barriers)
template <class TT, int NWM, int NWN, int NWK, int BM, int BN, int NST, int OCC>
__global__ __launch_bounds__(64 * NWM * NWN * NWK, OCC) void ngemm_kernel(const Task* __restrict__ tasks,
                                                                          const NSeg* __restrict__ segs, int64_t J0,
                                                                          const float* __restrict__ scales, int remap) {
  constexpr int BS = TT::BS, TM = BS * NWM * BM, TN = BS * NWN * BN;
  const Task t = tasks[remap ? xcd_task(blockIdx.x, gridDim.x) : blockIdx.x];
  __shared__ __attribute__((aligned(16))) char sm[NST * NWK * (TM + TN) * 128];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = w % (NWM * NWN), wr = wq / NWN, wc = nwave_col<NWM, NWN>(wq);
  const int nbm = __builtin_amdgcn_readfirstlane(max(0, min(BM, (t.M - t.m0 - BS * wr + BS * NWM - 1) / (BS * NWM))));
  const int nbn = __builtin_amdgcn_readfirstlane(max(0, min(BN, (t.N - t.n0 - BS * wc + BS * NWN - 1) / (BS * NWN))));
  if (nbm == BM && nbn == BN)
    nbody<TT, NWM, NWN, NWK, BM, BN, NST, true>(t, segs, J0, scales, sm, w, lane, nbm, nbn);
  else
    nbody<TT, NWM, NWN, NWK, BM, BN, NST, false>(t, segs, J0, scales, sm, w, lane, nbm, nbn);
}

}  // namespace

}  // namespace tci
