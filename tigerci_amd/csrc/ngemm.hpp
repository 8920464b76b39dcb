// Grouped GEMM over k-contiguous operands with direct global-to-LDS stages:
//   C[tile] (+)= s sum_seg A_seg B_seg^T,   A_seg: M x K,  B_seg: N x K,
// both operands as rows of bytes: FP64 (16 values of k per 128 bytes) or split
// rows (common.hpp: 32 values of k, hi and lo parts, per 128 bytes).  The two
// types share the staging: a k-step is 128 bytes of every row, copied by
// global_load_lds_dwordx4 into LDS rows of 128 bytes whose 16-byte chunks are
// XOR-swizzled on the source side.  Rows may be gathered through a row map, so
// one launch covers pair blocks over local domains without packed copies of
// operands that already have their k contiguous.
//
// What the loop avoids, against a staging that reads its segment descriptor
// and forms 64-bit row addresses for every load: each lane keeps one 32-bit
// offset per load for a whole segment, the segment's base is scalar and moves
// by 128 bytes a step, and nothing between two barriers waits on scalar
// memory, so the loads of the next stage cost a few issue slots and the MFMAs
// follow at once.
//
// Rows beyond M or N load a valid row again (their products are not stored);
// k beyond the segment loads zeros.
//
// Waves: NWM x NWN over the tile, blocks of 16 rows (columns) dealt
// round-robin, so that a ragged tile (a domain below the tile's size) loads
// every wave about equally; NWK groups of waves take alternate 128-byte
// k-chunks of one deeper stage and meet in LDS at the end (small outputs,
// whose few tiles would otherwise run a long chain of dependent k-steps on a
// mostly idle chip).
#pragma once

#include <algorithm>

#include "common.hpp"

namespace tci {

// one value of a split-row chunk: its parts 8 elements apart
__device__ __forceinline__ void put_split1(uint16_t* p, double v, float s, bool f16) {
  const float x = (float)v * s;
  if (f16) {
    const _Float16 h = (_Float16)x;
    const _Float16 l = (_Float16)(x - (float)h);
    p[0] = __builtin_bit_cast(uint16_t, h);
    p[8] = __builtin_bit_cast(uint16_t, l);
  } else {
    const __bf16 h = (__bf16)x;
    const __bf16 l = (__bf16)(x - (float)h);
    p[0] = __builtin_bit_cast(uint16_t, h);
    p[8] = __builtin_bit_cast(uint16_t, l);
  }
}

// One contraction range of a task.  kbytes: valid bytes of k per row, a
// multiple of 16; lda / ldb row strides in bytes (multiples of 16); am / bm
// row maps or null; ja / jb bytes per unit of the launch argument J0.  The range
// is taken `reps` times (at least once), A and B moving by sa and sb bytes from
// one to the next (the Cholesky vectors of one walk): the row offsets stay.
struct NSeg {
  const void* A;
  const void* B;
  const int32_t* am;
  const int32_t* bm;
  int64_t lda, ldb, ja, jb;
  int64_t kbytes;
  int64_t reps, sa, sb;
  int64_t pad_;
};

// Tile shapes (rows x columns; K-groups).
enum NShape {
  N128 = 0,    // 128 x 128, 4 waves, two workgroups per CU
  N192 = 1,    // 192 x 192, 8 waves, one workgroup per CU
  N64 = 2,     // 64 x 64, 4 waves
  N32K4 = 3,   // 32 x 32, 4 waves each on a quarter of k
  N256 = 4,    // split only: 256 x 256 on 32 x 32 MFMAs, 8 waves
  N128x192 = 5 // split only: 128 x 192, 4 waves
};

// A schedule asked for in the environment, "tile/ks" or "tile/ksx" (XCD-contiguous
// order), tile 128, 192, 64, 32k4 and for split products 256 or 128x192: shape
// -1 where the variable is unset or names no tile of this element type.
struct NSchedule {
  int shape = -1, ks = 1, order = 0;
};
NSchedule asked_schedule(const char* env, bool split);

struct NProgram {
  int shape = N128;
  bool split = false;
  int remap = 0;
  double alg_flops = 0.0;
  std::vector<Task> tasks;
  std::vector<NSeg> segs;
  DevBuf d_tasks, d_segs;
  void clear() {
    tasks.clear();
    segs.clear();
  }
  int tm() const { return shape == N192 ? 192 : shape == N64 ? 64 : shape == N32K4 ? 32 : shape == N256 ? 256 : 128; }
  int tn() const { return shape == N128x192 ? 192 : tm(); }
  // adds the tiles of one M x N output; rows / cols of the stored element are
  // offset by the blocking as in GemmProgram.  out32 (split programs, no
  // accumulation): C points to FP32 values, the sums as they were accumulated
  void add(double* C, int64_t ldc, int M, int N, const std::vector<NSeg>& s, bool accumulate, Blocking blk = Blocking(),
           int oscale = -1, bool out32 = false);
  void upload_tables(hipStream_t st);
  void launch(int precision, hipStream_t st, int64_t J0 = 0, const float* scales = nullptr) const;
  std::string kernel_name() const;
};

// May a task address `rows` plain rows of ld_bytes from one tile of `tile` rows?
// A lane holds the distance from the tile's first row, and the place within the
// staged part of a row (at most 512 bytes), as a 32-bit byte offset.
inline bool nrows_addressable(int64_t rows, int64_t tile, int64_t ld_bytes) {
  const int64_t last = std::min(rows, tile) - 1;
  return last <= 0 || ld_bytes <= ((((int64_t)1 << 32) - 512) / last);
}

// segment over rows of elements of `esz` bytes per value of k (8: FP64, 4: split rows)
inline NSeg nseg(const void* A, int64_t lda, const void* B, int64_t ldb, int64_t K, int esz,
                 const int32_t* am = nullptr, const int32_t* bm = nullptr) {
  NSeg s{};
  s.A = A;
  s.B = B;
  s.am = am;
  s.bm = bm;
  s.lda = lda * esz;
  s.ldb = ldb * esz;
  s.kbytes = K * esz;
  s.reps = 1;
  return s;
}

void launch_ngemm64(int shape, const Task* tasks, const NSeg* segs, int64_t ntasks, int64_t J0, hipStream_t st,
                    int remap);
void launch_ngemm16(int precision, int shape, const Task* tasks, const NSeg* segs, int64_t ntasks, int64_t J0,
                    const float* scales, hipStream_t st, int remap);

}  // namespace tci
