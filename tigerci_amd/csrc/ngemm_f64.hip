// FP64 instances of the direct-stage NT GEMM (ngemm_kernel.hpp) and its
// program tables.
#include <algorithm>

#include "ngemm_kernel.hpp"

namespace tci {

void launch_ngemm64(int shape, const Task* tasks, const NSeg* segs, int64_t ntasks, int64_t J0, hipStream_t st,
                    int remap) {
  if (ntasks <= 0) return;
  TCI_REQUIRE(ntasks < ((int64_t)1 << 31), "too many gemm tasks");
  const dim3 g((unsigned)ntasks);
  const float* sc = nullptr;
  switch (shape) {
    case N128:
      hipLaunchKernelGGL((ngemm_kernel<F64T, 2, 2, 1, 4, 4, 2, 2>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N192:
      hipLaunchKernelGGL((ngemm_kernel<F64T, 2, 4, 1, 6, 3, 2, 2>), g, dim3(512), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N64:
      hipLaunchKernelGGL((ngemm_kernel<F64T, 2, 2, 1, 2, 2, 2, 4>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N32K4:
      hipLaunchKernelGGL((ngemm_kernel<F64T, 1, 1, 4, 2, 2, 2, 2>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    default: throw Error(TCI_ERR_ARG, "no FP64 NT GEMM tile of this shape");
  }
  TCI_HIP(hipGetLastError());
}

void NProgram::add(double* C, int64_t ldc, int M, int N, const std::vector<NSeg>& s, bool accumulate, Blocking blk,
                   int oscale, bool out32) {
  if (M <= 0 || N <= 0) return;
  TCI_REQUIRE(oscale < 0 || split, "output scales belong to split programs");
  TCI_REQUIRE(!out32 || (split && !accumulate), "FP32 output needs a split program and no accumulation");
  for (const NSeg& x : s)
    TCI_REQUIRE(x.A && x.B && x.kbytes % 16 == 0 && x.lda % 16 == 0 && x.ldb % 16 == 0 && x.ja % 16 == 0 &&
                    x.jb % 16 == 0 && x.kbytes < ((int64_t)1 << 30) && x.reps >= 1 && x.reps < ((int64_t)1 << 30) && x.sa % 16 == 0 && x.sb % 16 == 0 &&
                    (reinterpret_cast<uintptr_t>(x.A) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(x.B) & 15) == 0,
                "NT GEMM operands need 16-byte aligned rows and ranges");
  // (gathered rows: the caller keeps the operand below 4 GiB)
  for (const NSeg& x : s)
    TCI_REQUIRE((x.am || nrows_addressable(M, tm(), x.lda)) && (x.bm || nrows_addressable(N, tn(), x.ldb)),
                "NT GEMM row stride too large");
  const int seg0 = (int)segs.size();
  for (const NSeg& x : s) segs.push_back(x);
  const int seg1 = (int)segs.size();
  for (int m0 = 0; m0 < M; m0 += tm())
    for (int n0 = 0; n0 < N; n0 += tn()) {
      Task t{};
      t.C = C;
      t.ldc = ldc;
      t.M = M;
      t.N = N;
      t.m0 = m0;
      t.n0 = n0;
      t.seg0 = seg0;
      t.seg1 = seg1;
      t.accumulate = accumulate ? 1 : 0;
      t.out_split = out32 ? 1 : 0;
      t.rdiv = blk.rdiv;
      t.cdiv = blk.cdiv;
      t.rstride = blk.rstride;
      t.cstride = blk.cstride;
      t.oscale = oscale;
      tasks.push_back(t);
    }
}

void NProgram::upload_tables(hipStream_t st) {
  alg_flops = 0.0;
  const double esz = split ? 4.0 : 8.0;
  for (const Task& t : tasks) {
    const double mv = std::min(tm(), t.M - t.m0), nv = std::min(tn(), t.N - t.n0);
    for (int q = t.seg0; q < t.seg1; ++q) alg_flops += 2.0 * mv * nv * (double)segs[q].kbytes / esz * (double)segs[q].reps;
  }
  upload(d_tasks, tasks, st);
  upload(d_segs, segs, st);
}

void NProgram::launch(int precision, hipStream_t st, int64_t J0, const float* scales) const {
  TCI_REQUIRE(split == (precision != TCI_SIGMA_FP64), "NT program launched in another precision than it was built for");
  const int rm = xcd_remap_forced() ? xcd_remap_default() : remap;
  if (split)
    launch_ngemm16(precision, shape, d_tasks.as<Task>(), d_segs.as<NSeg>(), (int64_t)tasks.size(), J0, scales, st, rm);
  else
    launch_ngemm64(shape, d_tasks.as<Task>(), d_segs.as<NSeg>(), (int64_t)tasks.size(), J0, st, rm);
}

std::string NProgram::kernel_name() const {
  return std::string("ngemm_kernel<") + (split ? "split," : "fp64,") + std::to_string(tm()) + "x" +
         std::to_string(tn()) + (shape == N32K4 ? ",k4>" : ">");
}

}  // namespace tci
