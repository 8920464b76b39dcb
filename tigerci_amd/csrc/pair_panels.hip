// Pair-pair terms as per-walk products over packed panels.
//
// For an internal orbital i let K_i be the list of all (k, c) with the walk
// {i, k} strong and c in its domain D_ik: blocks by k, each padded to a
// multiple of 8.  C^{pq} is the walk's dense block (p >= q) or its transpose.
// Panels over K_i, rows a over all virtuals (zero outside the domains):
//   CR_i[a][(k,c)] = C^{ik}[a][c],  CC_i[a][(k,c)] = C^{ki}[a][c],  CT_i = 2 CR_i - CC_i
// (written from C in every sigma) and, once per plan, for every strong ordered
// pair (i, j) over the rows x of D_ij, and for every i over the Cholesky vectors,
//   JP_ij[x][(k,c)] = -(kj|c D_ij[x]),   LP_i[J][(k,c)] = L^J_kc.
// With U[(i,a)][J] = Y[i][J][a] + W[i][J][a],
//   Y[i][J][a] = sum_c L^J_ac s_i^c,  W_i = LP_i CT_i^T  ([i][J][a]),
// the ring and 3-external terms of the walk P = (i, j), rows and columns over
// D_P, are one contraction (Kov = Lov^T Lov puts C~ K into U Lov):
//   R_P += CR_i JP_ij^T + JP_ij CC_i^T + JP_ji CR_j^T + CC_j JP_ji^T
//        + U_i Lov_j + (U_j Lov_i)^T
// and the 3-internal singles terms are two more ranges of it (FP64):
//        + s_i O_ij^T + O_ji s^T,   O_ij[b][k] = -(ki|bj).
// Where the JP_ij of all pairs do not fit, the columns (k, c) run over all
// virtuals instead (wide panels): JP_ij then is the rows D_ij of one JP_j, and
// LP_i one LP, for four N x N matrices (N = n_int n_v) in all.
// All operands have their k contiguous and rows gathered through D_P, so they
// run on the NT GEMM (ngemm.hpp): flops 2 d_P^2 (2 |K_i| + 2 |K_j| + 2 n_chol)
// per walk, the count of the gathered per-walk products, at the rate of the
// dense ones.  Embedding every block in the full virtual space instead
// (4 N^3 + 6 N^2 n_chol, N = n_int n_v) costs 4.4 times the flops at 34
// internal, 192 virtual orbitals with domains of 60 to 192.  W serves U and
// the singles (g += W L): it is computed once.
//
// The 4-internal term sum_Q [(ki|lj) C_Q + (li|kj) C_Q^T] acts on the symmetric
// and antisymmetric parts of C_Q separately, over packed virtual pairs:
//   H+[P][p] = sum_Q h+_PQ X+_Q[p],  H-[P'][q] = sum_Q h-_PQ X-_Q[q],
//   h+- = (ki|lj) +- (li|kj),
// products over k = walk with X+- transposed to [pair][walk].  The final kernel
// (pack_panels_kernel) adds everything of one CSF: K-split partials, S+- of
// the resident ladder, H+-, c0 (ia|jb) and the CSF factors.
#include "plan.hpp"

#include <algorithm>
#include <cstdlib>
#include <string>

namespace tci {

namespace {

constexpr double SQRT2 = 1.41421356237309504880;
constexpr double INV_SQRT2 = 0.70710678118654752440;
constexpr double SQRT3 = 1.73205080756887729353;

__host__ __device__ __forceinline__ int64_t tri(int64_t a) { return a * (a + 1) / 2; }
__device__ __forceinline__ void untri32(int t, int& x, int& y) {  // t = x(x+1)/2 + y, y <= x
  int r = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
  while ((r + 1) * (r + 2) / 2 <= t) ++r;
  while (r * (r + 1) / 2 > t) --r;
  x = r;
  y = t - r * (r + 1) / 2;
}
inline int64_t up(int64_t n, int64_t m) { return (n + m - 1) / m * m; }

constexpr int kMaxKs = 8;  // K-splits of the pair products

// Offsets are in values; a value is 8 bytes (FP64) or 4 (split rows).
struct PanelTab {
  const int32_t* koff;   // [i n_int + k] -> column of block k in panel i, or -1
  const int64_t* ld;     // [i] row stride of panel i
  const int64_t* poff;   // [i] start of panel i (n_v rows)
  const int64_t* jpoff;  // [i n_int + j] start of JP_ij
  const int64_t* lpoff;  // [i] start of LP_i (n_chol rows)
  const int32_t* pairid;
  int wide;              // columns of a block: 0 positions in its domain, 1 virtuals
};

// column, within its block, of position y of the domain D
__device__ __forceinline__ int pcol(const PanelTab& K, const int32_t* __restrict__ D, int y) { return K.wide ? D[y] : y; }

__device__ __forceinline__ uint16_t* srow(void* base, int64_t row_start, int64_t col) {
  return static_cast<uint16_t*>(base) + 2 * row_start + xidx(col);
}

// Eight values of a panel row (its block starts at value `at`), positions y ..
// y + 7 of the domain D of size d, as split parts.  A wide block has them
// together only where D holds eight aligned consecutive virtuals.
__device__ __forceinline__ void put_cols(const PanelTab& K, void* dst, int64_t row, int64_t at,
                                         const int32_t* __restrict__ D, int y, int d, const float (&w)[8], float s, bool f16) {
  if (!K.wide) {
    put_split8(srow(dst, row, at + y), w, s, f16);
    return;
  }
  const int g = D[y];
  if (y + 7 < d && (g & 7) == 0 && D[y + 7] == g + 7) {
    put_split8(srow(dst, row, at + g), w, s, f16);
    return;
  }
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (y + q < d) put_split1(srow(dst, row, at + D[y + q]), w[q], s, f16);
}

// CR, CC and CT of both panels of walk Q from its C block: 32 x 32 tiles, the
// tile and its transpose read once.  Rows outside the domain and padding
// columns are zero from set-up and never written.
template <bool SPLIT>
__global__ __launch_bounds__(256) void panels_kernel(PairTab T, PanelTab K, const double* __restrict__ C, void* CR,
                                                     void* CC, void* CT, const float* scl, const float* sclt, int f16,
                                                     int what) {
  __shared__ double ta[32][33], tb[32][33];
  const int Q = blockIdx.y;
  const int64_t o = T.dom_off[Q];
  const int d = (int)(T.dom_off[Q + 1] - o), nt = (d + 31) >> 5;
  if ((int)blockIdx.x >= nt * nt) return;
  const int x0 = ((int)blockIdx.x / nt) * 32, y0 = ((int)blockIdx.x % nt) * 32;
  const int i = T.pairs[2 * Q], j = T.pairs[2 * Q + 1];
  const double* Cq = C + T.cd_off[Q];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) {
    const int x = x0 + r, y = y0 + tx;
    ta[r][tx] = x < d && y < d ? Cq[(int64_t)x * d + y] : 0.0;     // C^{ij}[x][y]
    const int yr = y0 + r, xc = x0 + tx;
    tb[tx][r] = yr < d && xc < d ? Cq[(int64_t)yr * d + xc] : 0.0;  // C^{ji}[x][y] = C_Q[y][x]
  }
  __syncthreads();
  const int two = i != j ? 2 : 1;
  if (!SPLIT) {
    for (int p = 0; p < two; ++p) {
      const int u = p ? j : i, v = p ? i : j;
      const int64_t base = K.poff[u] + K.koff[u * T.n_int + v], ld = K.ld[u];
      for (int r = ty; r < 32; r += 8) {
        const int x = x0 + r, y = y0 + tx;
        if (x >= d || y >= d) continue;
        const double a = p ? tb[r][tx] : ta[r][tx], b = p ? ta[r][tx] : tb[r][tx];
        const int64_t e = base + (int64_t)T.dom_idx[o + x] * ld + pcol(K, T.dom_idx + o, y);
        static_cast<double*>(CR)[e] = a;
        static_cast<double*>(CC)[e] = b;
        static_cast<double*>(CT)[e] = 2.0 * a - b;
      }
    }
  } else {
    const float s = scale_at(scl), st = scale_at(sclt);
    // 128 chunks of 8 per array (row r, chunk ch); arrays CR, CC (what & 1), CT (what & 2), per panel
    for (int t = threadIdx.x; t < 128 * 3 * two; t += 256) {
      const int arr = (t >> 7) % 3, p = (t >> 7) / 3;
      if (!(what & (arr == 2 ? 2 : 1))) continue;
      const int r = (t & 127) >> 2, c = 8 * (t & 3);
      const int x = x0 + r, y = y0 + c;
      if (x >= d || y >= d) continue;
      const int u = p ? j : i, v = p ? i : j;
      float w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const double a = p ? tb[r][c + q] : ta[r][c + q], b = p ? ta[r][c + q] : tb[r][c + q];
        w[q] = (float)(arr == 0 ? a : arr == 1 ? b : 2.0 * a - b);
      }
      void* dst = arr == 0 ? CR : arr == 1 ? CC : CT;
      put_cols(K, dst, K.poff[u] + (int64_t)T.dom_idx[o + x] * K.ld[u], K.koff[u * T.n_int + v], T.dom_idx + o, y, d, w,
               arr == 2 ? st : s, f16 != 0);
    }
  }
}

// XT+[p(a,b)][Q] = C+_ab, XT-[q(a,b)][Q] = C-_ab of walk Q (0 outside its
// domain), rows of ldw values, from the CI vector (the symmetric part of C_Q
// is its singlet-coupled block, the antisymmetric part its triplet-coupled
// one).  Block: one a, 32 b and 32 walks; the walks' elements are read along b
// and leave through LDS along Q.
template <bool SPLIT>
__device__ __forceinline__ void xt_block(const PairTab& T, const int32_t* __restrict__ pos, const double* __restrict__ x,
                                         void* XTp, void* XTm, int64_t ldw, const float* scl, int f16, int a, int b0,
                                         int Q0, double (&tp)[32][33], double (&tm)[32][33]) {
  const int nv = T.n_v;
  if (b0 > a) return;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int b = b0 + tx;
  for (int r = ty; r < 32; r += 8) {
    const int Q = Q0 + r;
    double vp = 0.0, vm = 0.0;
    if (Q < T.n_pairs && b <= a) {
      const int32_t* ps = pos + (int64_t)Q * nv;
      const int pa = ps[a], pb = ps[b];
      if (pa >= 0 && pb >= 0) {
        const int d = (int)(T.dom_off[Q + 1] - T.dom_off[Q]);
        const bool same = T.pairs[2 * Q] == T.pairs[2 * Q + 1];
        if (pa == pb) {
          vp = same ? x[T.aa_off[Q] + pa] : -x[T.aa_off[Q] + pa] * INV_SQRT2;
        } else {  // domains are sorted: pa > pb
          const int64_t idx = T.ab_off[Q] + (int64_t)pa * (pa - 1) / 2 + pb;
          vp = same ? x[idx] * INV_SQRT2 : -0.5 * x[idx];
          if (!same) vm = -x[idx + (int64_t)d * (d - 1) / 2] * 0.28867513459481288225;  // 1 / (2 sqrt3)
        }
      }
    }
    tp[r][tx] = vp;
    tm[r][tx] = vm;
  }
  __syncthreads();
  if (!SPLIT) {
    for (int r = ty; r < 32; r += 8) {
      const int bb = b0 + r, Q = Q0 + tx;
      if (bb > a || Q >= T.n_pairs) continue;
      static_cast<double*>(XTp)[(tri(a) + bb) * ldw + Q] = tp[tx][r];
      if (bb < a) static_cast<double*>(XTm)[(tri(a - 1) + bb) * ldw + Q] = tm[tx][r];
    }
  } else {
    const int t = threadIdx.x & 127, r = t >> 2, c = 8 * (t & 3);
    const bool minus = threadIdx.x >= 128;
    const int bb = b0 + r;
    if (bb <= a && Q0 + c < T.n_pairs && !(minus && bb == a)) {
      float w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = (float)(minus ? tm[c + q][r] : tp[c + q][r]);
      put_split8(srow(minus ? XTm : XTp, (minus ? tri(a - 1) + bb : tri(a) + bb) * ldw, Q0 + c), w, scale_at(scl),
                 f16 != 0);
    }
  }
}

template <bool SPLIT>
__global__ __launch_bounds__(256) void xt_kernel(PairTab T, const int32_t* __restrict__ pos, const double* __restrict__ x,
                                                 const IoSlot* __restrict__ io, void* XTp, void* XTm, int64_t ldw,
                                                 const float* scl, int f16) {
  if (io) x = io->x;
  __shared__ double tp[32][33], tm[32][33];
  xt_block<SPLIT>(T, pos, x, XTp, XTm, ldw, scl, f16, blockIdx.x, blockIdx.y * 32, blockIdx.z * 32, tp, tm);
}

// Everything a sigma derives from the CI vector alone, in one pass over it:
// the panels, Ct (and C where a term reads it), the rows X+- of the resident
// ladder, s and its transpose, and (blocks past the walks') XT+-.  Block: one walk, one pair of 32 x 32 tiles
// (X >= Y) of the packed triangle; each vector element is read once and both
// orientations leave along rows.  FP64 and bf16x3 (the scales of fp16x3 need
// max|C| first: unpack_kernel, vv_scatter_kernel and panels_kernel there).
// Bound by its writes: 230 us (bf16x3) and 304 us (FP64) at 34/192/1200 (its
// part without XT+- 116 and 157, against 98 + 50 + 100 us for unpack, scatter
// and panels one after the other; XT+- in a launch of its own 95-125), FP64 at
// 10/100/400 15.6 us and at 5/30/175 6.5 us, where XT+- alone took 11 and 5.
struct ExpandOut {
  double *C, *Ct, *s, *sT;  // C null: not needed
  int nk;
  double* sP;               // s with rows of ldw, or null
  int64_t ldw;
  void *CR, *CC, *CT;
  void *Xp, *Xm;            // null: no resident ladder
  int64_t ldp, ldm;         // values
  const int32_t* colm;
  const int32_t* pos;
  void *XTp, *XTm;
  int64_t ldx;              // row stride of XT+-
};

__device__ __forceinline__ void put_bf(uint16_t* p, double v) {
  const float x = (float)v;
  const __bf16 h = (__bf16)x;
  const __bf16 l = (__bf16)(x - (float)h);
  p[0] = __builtin_bit_cast(uint16_t, h);
  p[8] = __builtin_bit_cast(uint16_t, l);
}

template <bool SPLIT>
__global__ __launch_bounds__(256) void expand_kernel(PairTab T, PanelTab K, const double* __restrict__ x,
                                                     const IoSlot* __restrict__ io, ExpandOut O) {
  if (io) x = io->x;
  const int Q = blockIdx.y, n = T.n_int, nv = T.n_v;
  __shared__ double ta[32][33], tb[32][33];  // C[x][y] and C[y][x], x in tile X, y in tile Y
  if (Q > T.n_pairs) {  // XT+-
    const int64_t l = (int64_t)(Q - T.n_pairs - 1) * gridDim.x + blockIdx.x;
    const int nb = (nv + 31) >> 5;
    const int64_t r = l / nv;
    const int z = (int)(r / nb);
    if (z * 32 < T.n_pairs)
      xt_block<SPLIT>(T, O.pos, x, O.XTp, O.XTm, O.ldx, nullptr, 0, (int)(l - r * nv), (int)(r - (int64_t)z * nb) * 32,
                      z * 32, ta, tb);
    return;
  }
  if (Q == T.n_pairs) {  // singles (walks by descending hole)
    const int64_t tot = (int64_t)nv * O.nk;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot; e += (int64_t)gridDim.x * blockDim.x) {
      const int k = (int)(e / nv), a = (int)(e - (int64_t)k * nv);
      const double v = k < n ? x[1 + (int64_t)(n - 1 - k) * nv + a] * INV_SQRT2 : 0.0;
      if (k < n) O.s[e] = v;
      if (k < n && O.sP) O.sP[k * O.ldw + a] = v;
      O.sT[(int64_t)a * O.nk + k] = v;
    }
    return;
  }
  const int64_t o = T.dom_off[Q];
  const int d = (int)(T.dom_off[Q + 1] - o), nt = (d + 31) >> 5;
  if ((int)blockIdx.x >= nt * (nt + 1) / 2) return;
  int X, Y;
  untri32((int)blockIdx.x, X, Y);
  const int x0 = X * 32, y0 = Y * 32;
  const int i = T.pairs[2 * Q], j = T.pairs[2 * Q + 1];
  const int64_t m2 = (int64_t)d * (d - 1) / 2;
  const double *xa = x + T.aa_off[Q], *xb = x + T.ab_off[Q];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  constexpr double INV_2SQRT3 = 0.28867513459481288225;
  const int cm = O.colm[Q];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = ty + 8 * u, xr = x0 + r, yc = y0 + tx;
    double A = 0.0, B = 0.0;
    if (xr < d && yc <= xr) {
      if (xr == yc) {
        A = B = i == j ? xa[xr] : -xa[xr] * INV_SQRT2;
      } else {
        const int64_t idx = (int64_t)xr * (xr - 1) / 2 + yc;
        if (i == j) {
          A = B = xb[idx] * INV_SQRT2;
        } else {
          const double vs = -0.5 * xb[idx], q = xb[m2 + idx] * INV_2SQRT3;
          A = vs - q;
          B = vs + q;
        }
      }
      if (O.Xp) {
        const int gx = T.dom_idx[o + xr], gy = T.dom_idx[o + yc];
        const double vp = xr == yc ? 0.5 * A : 0.5 * (A + B);
        const int64_t kp = tri(gx) + gy;
        if (SPLIT) put_bf(static_cast<uint16_t*>(O.Xp) + 2 * Q * O.ldp + xidx(kp), vp);
        else static_cast<double*>(O.Xp)[Q * O.ldp + kp] = vp;
        if (cm >= 0 && xr != yc) {
          const int64_t km = tri(gx - 1) + gy;
          const double vm = 0.5 * (A - B);
          if (SPLIT) put_bf(static_cast<uint16_t*>(O.Xm) + 2 * cm * O.ldm + xidx(km), vm);
          else static_cast<double*>(O.Xm)[cm * O.ldm + km] = vm;
        }
      }
    }
    ta[r][tx] = A;
    tb[r][tx] = B;
  }
  __syncthreads();
  if (X == Y) {  // fill the upper half of the diagonal tile
    double up[4], lo[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = ty + 8 * u;
      up[u] = tx > r ? tb[tx][r] : ta[r][tx];
      lo[u] = tx > r ? ta[tx][r] : tb[r][tx];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ta[ty + 8 * u][tx] = up[u];
      tb[ty + 8 * u][tx] = lo[u];
    }
    __syncthreads();
  }
  // orientation 0: rows in X, columns in Y, C[row][col] = ta; 1: rows in Y,
  // columns in X, C[row][col] = tb^T (the diagonal tile is whole after 0)
  const int no = X == Y ? 1 : 2;
  for (int w = 0; w < no; ++w) {
    const int r0 = w ? y0 : x0, c0 = w ? x0 : y0;
    double* Cq = O.C ? O.C + T.cd_off[Q] : nullptr;
    double* Ctq = O.Ct + T.cd_off[Q];
    const int two = i != j ? 2 : 1;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = ty + 8 * u, row = r0 + r, col = c0 + tx;
      if (row >= d || col >= d) continue;
      const double a = w ? tb[tx][r] : ta[r][tx], b = w ? ta[tx][r] : tb[r][tx];  // C[row][col], C[col][row]
      const int64_t e = (int64_t)row * d + col;
      if (Cq) Cq[e] = a;
      Ctq[e] = 2.0 * a - b;
      if (!SPLIT) {
        const int64_t g = T.dom_idx[o + row];
        for (int p = 0; p < two; ++p) {
          const int iu = p ? j : i, iv = p ? i : j;
          const int64_t q = K.poff[iu] + K.koff[iu * n + iv] + g * K.ld[iu] + pcol(K, T.dom_idx + o, col);
          const double aa = p ? b : a, bb = p ? a : b;
          static_cast<double*>(O.CR)[q] = aa;
          static_cast<double*>(O.CC)[q] = bb;
          static_cast<double*>(O.CT)[q] = 2.0 * aa - bb;
        }
      }
    }
    if (SPLIT) {
      for (int t = threadIdx.x; t < 128 * 3 * two; t += 256) {
        const int arr = (t >> 7) % 3, p = (t >> 7) / 3;
        const int r = (t & 127) >> 2, c = 8 * (t & 3);
        const int row = r0 + r, col = c0 + c;
        if (row >= d || col >= d) continue;
        const int iu = p ? j : i, iv = p ? i : j;
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          double a = w ? tb[c + q][r] : ta[r][c + q], b = w ? ta[c + q][r] : tb[r][c + q];
          if (p) {
            const double h = a;
            a = b;
            b = h;
          }
          v[q] = col + q < d ? (float)(arr == 0 ? a : arr == 1 ? b : 2.0 * a - b) : 0.f;
        }
        void* dst = arr == 0 ? O.CR : arr == 1 ? O.CC : O.CT;
        put_cols(K, dst, K.poff[iu] + (int64_t)T.dom_idx[o + row] * K.ld[iu], K.koff[iu * n + iv], T.dom_idx + o, col, d,
                 v, 1.f, false);
      }
    }
  }
}

// JP_ij block k: rows x of D_ij, columns c of D_ik.  Grid (k, (i,j)).  F (FP64,
// or null): the off-diagonal virtual Fock elements; block k = j of JP_ij (i >= j)
// multiplies C_ij from both sides, so adding F there (half for i = j, whose
// products come twice) makes F C + C F part of the pair products.
template <bool SPLIT>
__global__ __launch_bounds__(256) void jp_kernel(PairTab T, PanelTab K, const double* __restrict__ Jvv,
                                                 const double* __restrict__ F, void* JP, const float* scl, int f16) {
  const int n = T.n_int, k = blockIdx.x, i = blockIdx.y / n, j = blockIdx.y % n;
  const int P = K.pairid[i * n + j], Q = K.pairid[i * n + k];
  if (P < 0 || Q < 0) return;
  const int64_t oP = T.dom_off[P], oQ = T.dom_off[Q];
  const int dP = (int)(T.dom_off[P + 1] - oP), dQ = (int)(T.dom_off[Q + 1] - oQ);
  const int hi = max(k, j), lo = min(k, j);
  const int64_t nv = T.n_v;
  const double* J = Jvv + ((int64_t)hi * (hi + 1) / 2 + lo) * nv * nv;
  const int64_t ld = K.ld[i], base = K.jpoff[i * n + j];
  const int64_t col = K.koff[i * n + k];
  const float s = SPLIT ? scale_at(scl) : 1.f;
  const int nch = (dQ + 7) >> 3;
  if (SPLIT) {
    for (int t = threadIdx.x; t < dP * nch; t += 256) {
      const int x = t / nch, c = 8 * (t - x * nch);
      const double* row = J + (int64_t)T.dom_idx[oP + x] * nv;
      float w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = c + q < dQ ? (float)-row[T.dom_idx[oQ + c + q]] : 0.f;
      put_split8(srow(JP, base + x * ld, col + c), w, s, f16 != 0);
    }
  } else {
    const double f = F && k == j && i >= j ? (i == j ? 0.5 : 1.0) : 0.0;
    for (int t = threadIdx.x; t < dP * dQ; t += 256) {
      const int x = t / dQ, c = t - x * dQ;
      const int64_t e = (int64_t)T.dom_idx[oP + x] * nv + T.dom_idx[oQ + c];
      double v = -J[e];
      if (f != 0.0) v += f * F[e];
      static_cast<double*>(JP)[base + x * ld + col + c] = v;
    }
  }
}

// LP_i[J][(k,c)] = L^J_kc.  Grid (J, i).
template <bool SPLIT>
__global__ __launch_bounds__(256) void lp_kernel(PairTab T, PanelTab K, const double* __restrict__ Lov, void* LP,
                                                 const float* scl, int f16) {
  const int n = T.n_int, i = blockIdx.y;
  const int64_t J = blockIdx.x, nv = T.n_v;
  const int64_t row = K.lpoff[i] + J * K.ld[i];
  const float s = SPLIT ? scale_at(scl) : 1.f;
  for (int k = 0; k < n; ++k) {
    const int Q = K.pairid[i * n + k];
    if (Q < 0) continue;
    const int64_t o = T.dom_off[Q];
    const int d = (int)(T.dom_off[Q + 1] - o);
    const double* L = Lov + (J * n + k) * nv;
    const int64_t col = K.koff[i * n + k];
    if (SPLIT) {
      for (int c = 8 * (int)threadIdx.x; c < d; c += 8 * 256) {
        float w[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) w[q] = c + q < d ? (float)L[T.dom_idx[o + c + q]] : 0.f;
        put_split8(srow(LP, row, col + c), w, s, f16 != 0);
      }
    } else {
      for (int c = threadIdx.x; c < d; c += 256) static_cast<double*>(LP)[row + col + c] = L[T.dom_idx[o + c]];
    }
  }
}

// The same for wide panels, whose columns (k, c) run over all virtuals of all
// internal orbitals: one JP_j[x][(k,c)] for every i, rows x over all virtuals.
// Half of F goes into block k = j: the walk (i, j) meets it once in JP_j and
// once in JP_i.  Grid (k, j).
template <bool SPLIT>
__global__ __launch_bounds__(256) void jp_wide_kernel(PairTab T, PanelTab K, const double* __restrict__ Jvv,
                                                      const double* __restrict__ F, void* JP, const float* scl, int f16) {
  const int k = blockIdx.x, j = blockIdx.y, nv = T.n_v;
  const int hi = max(k, j), lo = min(k, j);
  const double* J = Jvv + ((int64_t)hi * (hi + 1) / 2 + lo) * nv * nv;
  const int64_t ld = K.ld[j], base = K.jpoff[j], col = (int64_t)k * ((nv + 7) & ~7);
  const float s = SPLIT ? scale_at(scl) : 1.f;
  if (SPLIT) {
    const int nch = (nv + 7) >> 3;
    for (int t = threadIdx.x; t < nv * nch; t += 256) {
      const int x = t / nch, c = 8 * (t - x * nch);
      float w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = c + q < nv ? (float)-J[(int64_t)x * nv + c + q] : 0.f;
      put_split8(srow(JP, base + x * ld, col + c), w, s, f16 != 0);
    }
  } else {
    for (int t = threadIdx.x; t < nv * nv; t += 256) {
      const int x = t / nv, c = t - x * nv;
      static_cast<double*>(JP)[base + x * ld + col + c] = F && k == j ? 0.5 * F[t] - J[t] : -J[t];
    }
  }
}

// ... and one LP[J][(k,c)].  Grid (J, k).
template <bool SPLIT>
__global__ __launch_bounds__(256) void lp_wide_kernel(PairTab T, PanelTab K, const double* __restrict__ Lov, void* LP,
                                                      const float* scl, int f16) {
  const int k = blockIdx.y, nv = T.n_v;
  const int64_t row = (int64_t)blockIdx.x * K.ld[0], col = (int64_t)k * ((nv + 7) & ~7);
  const double* L = Lov + ((int64_t)blockIdx.x * T.n_int + k) * nv;
  const float s = SPLIT ? scale_at(scl) : 1.f;
  if (SPLIT) {
    for (int c = 8 * (int)threadIdx.x; c < nv; c += 8 * 256) {
      float w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = c + q < nv ? (float)L[c + q] : 0.f;
      put_split8(srow(LP, row, col + c), w, s, f16 != 0);
    }
  } else {
    for (int c = threadIdx.x; c < nv; c += 256) static_cast<double*>(LP)[row + col + c] = L[c];
  }
}

// U[(i,a)][J] = Y[i][J][a] + W[i][J][a] (Y null: W alone, for the transposed
// Lov), 32 x 32 tiles through LDS; row stride ldu values.  Grid (J tiles, a
// tiles, i).
template <bool SPLIT>
__global__ __launch_bounds__(256) void u_kernel(const double* __restrict__ Y, const double* __restrict__ W, int n_v,
                                                int64_t n_chol, int64_t wstride_i, int64_t wstride_J, void* U,
                                                int64_t ldu, const float* scl, int f16) {
  __shared__ double tile[32][33];
  const int i = blockIdx.z;
  const int64_t J0 = (int64_t)blockIdx.x * 32;
  const int a0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) {
    const int64_t J = J0 + r;
    const int a = a0 + tx;
    double v = 0.0;
    if (J < n_chol && a < n_v) {
      v = W[i * wstride_i + J * wstride_J + a];
      if (Y) v += Y[(i * n_chol + J) * n_v + a];
    }
    tile[r][tx] = v;
  }
  __syncthreads();
  if (!SPLIT) {
    for (int r = ty; r < 32; r += 8) {
      const int a = a0 + r;
      const int64_t J = J0 + tx;
      if (J < n_chol && a < n_v) static_cast<double*>(U)[((int64_t)i * n_v + a) * ldu + J] = tile[tx][r];
    }
  } else if (threadIdx.x < 128) {
    const int r = threadIdx.x >> 2, c = 8 * (threadIdx.x & 3);
    const int a = a0 + r;
    if (a < n_v && J0 + c < n_chol) {
      float w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = (float)tile[c + q][r];  // zero beyond n_chol
      put_split8(srow(U, ((int64_t)i * n_v + a) * ldu, J0 + c), w, scale_at(scl), f16 != 0);
    }
  }
}

// max |Y + W| into *out (float bits)
__global__ __launch_bounds__(256) void u_absmax_kernel(const double* __restrict__ Y, const double* __restrict__ W,
                                                       int64_t n, int n_v, int pad, unsigned* __restrict__ out) {
  __shared__ float part[4];
  float m = 0.f;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
    m = fmaxf(m, fabsf((float)(Y[e] + W[pad ? e + e / n_v * pad : e])));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_down(m, off, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(out, __float_as_uint(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]))));
}

// split rows of an FP64 matrix (rows x K values, stride ld) into stride ldo values
__global__ void split_matrix_kernel(const double* __restrict__ src, int64_t rows, int64_t K, int64_t ld, void* out,
                                    int64_t ldo, const float* scl, int f16) {
  const float s = scale_at(scl);
  const int64_t nch = (K + 7) >> 3;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < rows * nch; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / nch, c = 8 * (e - r * nch);
    float w[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) w[q] = c + q < K ? (float)src[r * ld + c + q] : 0.f;
    put_split8(srow(out, r * ldo, c), w, s, f16 != 0);
  }
}

// O_ij[b][k] = -(ki|bj) = -O3[k][i][j][b], rows of nk values; grid (i n_int + j)
__global__ __launch_bounds__(256) void o3t_kernel(const double* __restrict__ O3, int n, int nv, int nk,
                                                  double* __restrict__ O) {
  const int i = blockIdx.x / n, j = blockIdx.x % n;
  for (int t = threadIdx.x; t < nv * nk; t += 256) {
    const int k = t / nv, b = t - k * nv;
    O[((int64_t)blockIdx.x * nv + b) * nk + k] = k < n ? -O3[(((int64_t)k * n + i) * n + j) * nv + b] : 0.0;
  }
}

// sT[a][k] = s[k][a], rows of nk values, zero padded
__global__ void st_kernel(const double* __restrict__ s, int n, int nv, int nk, double* __restrict__ sT) {
  const int64_t tot = (int64_t)nv * nk;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot; e += (int64_t)gridDim.x * blockDim.x) {
    const int a = (int)(e / nk), k = (int)(e - (int64_t)a * nk);
    sT[e] = k < n ? s[(int64_t)k * nv + a] : 0.0;
  }
}

// Everything of one CSF of the pair walks: R_P[x][y] and R_P[y][x] from the
// K-split partials (d x d each), the packed S+- and H+-, c0 (ia|jb), and R
// itself when another term went there; then the CSF factors of pack_kernel.
// Block: one walk, one pair of 32 x 32 tiles (X >= Y); the transposed elements
// come through LDS.  blockIdx.y == n_pairs: valence and singles.
struct PackSrc {
  const void* Rp;       // [nrp][sum_d2]
  int64_t rstride;
  int nrp;
  const double* rank;   // [sum_d2] FP64 products next to FP32 partials Rp, or null
  const double* R;      // null: no further terms
  const void* Sp;       // [nsp][n_pairs][np] (nsp = 0: no resident ladder)
  const void* Sm;       // [nsp][ncm][nm]
  int64_t sp_part, sm_part;
  int nsp;
  const double* Hp;     // [n_pairs][np], null: part of S+-
  const double* Hm;     // [ncm][nm]
  int64_t np, nm;
  const int32_t* colm;
  const double* Kov;
};

// TR, TS: FP64, or FP32 where the sums were accumulated in FP32 (split products).
// Bound by the partials it reads: at
// 34/192/1200 (bf16x3) 208 us with all of them in FP64, 165 in FP32.
template <class TR, class TS>
__global__ __launch_bounds__(256) void pack_panels_kernel(PairTab T, PackSrc S, const double* __restrict__ x,
                                                          const double* __restrict__ g,
                                                          const double* __restrict__ sig0, double e_ref, int flags,
                                                          double* __restrict__ sigma, const IoSlot* __restrict__ io) {
  if (io) {
    x = io->x;
    sigma = io->y;
  }
  const bool accum = (flags & TCI_ACCUMULATE) != 0;
  const double eadd = (flags & TCI_ADD_EREF) ? e_ref : 0.0;
  const int P = blockIdx.y, no = T.n_int, nv = T.n_v;
  if (P == T.n_pairs) {
    const int64_t n = 1 + (int64_t)no * nv;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
      double v;
      if (k == 0) {
        v = *sig0 + eadd * x[0];
      } else {
        const int64_t w = (k - 1) / nv;  // N-1 walk rank: hole no - 1 - w
        const int i = no - 1 - (int)w, a = (int)(k - 1 - w * nv);
        v = SQRT2 * g[(int64_t)i * nv + a] + (T.eps[no + a] - T.eps[i] + eadd) * x[k];
      }
      sigma[k] = accum ? sigma[k] + v : v;
    }
    return;
  }
  const int64_t off = T.dom_off[P];
  const int d = (int)(T.dom_off[P + 1] - off), nt = (d + 31) >> 5;
  if ((int)blockIdx.x >= nt * (nt + 1) / 2) return;
  int X, Yt;
  untri32((int)blockIdx.x, X, Yt);
  const int x0 = X * 32, y0 = Yt * 32;
  const int i = T.pairs[2 * P], j = T.pairs[2 * P + 1];
  const int64_t niv = (int64_t)no * nv, m2 = (int64_t)d * (d - 1) / 2;
  const TR* Rp = static_cast<const TR*>(S.Rp) + T.cd_off[P];
  const double* rank = S.rank ? S.rank + T.cd_off[P] : nullptr;
  const TS *Sp = static_cast<const TS*>(S.Sp), *Sm = static_cast<const TS*>(S.Sm);
  const double* R = S.R ? S.R + T.cd_off[P] : nullptr;
  const int32_t* D = T.dom_idx + off;
  const int cm = S.colm[P];
  const double c0 = x[0], ei = T.eps[i], ej = T.eps[j];
  __shared__ double tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  // elements [r + 8 u][c] (u < 4) without the packed parts, four rows' loads
  // in flight together
  auto elems = [&](int r, int rmax, int c, bool cok, double (&v)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = 0.0;
    if (!cok) return;
    int64_t e[4];
    const int64_t kc = (int64_t)j * nv + D[c];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int rr = min(r + 8 * u, rmax);
      e[u] = (int64_t)rr * d + c;
      v[u] = c0 * S.Kov[((int64_t)i * nv + D[rr]) * niv + kc];
    }
#pragma unroll 2
    for (int q = 0; q < S.nrp; ++q)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] += (double)Rp[q * S.rstride + e[u]];
    if (rank)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] += rank[e[u]];
    if (R)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] += R[e[u]];
  };
  double v[4];
  elems(y0 + ty, d - 1, x0 + tx, x0 + tx < d, v);
#pragma unroll
  for (int u = 0; u < 4; ++u) tile[ty + 8 * u][tx] = v[u];
  __syncthreads();
  const int yc = y0 + tx;
  if (yc >= d) return;
  elems(x0 + ty, d - 1, yc, true, v);
  const int gy = D[yc];
  double sp[4], sm[4];
  int gx[4];
  int64_t p[4], m[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    // clamped where the element lies outside (above the diagonal, beyond d):
    // the loads stay in bounds and nothing is stored
    const int xr = max(min(x0 + ty + 8 * u, d - 1), yc);
    gx[u] = D[xr];  // domains are sorted: gx >= gy
    p[u] = P * S.np + tri(gx[u]) + gy;
    m[u] = cm >= 0 && gx[u] != gy ? cm * S.nm + tri(gx[u] - 1) + gy : -1;
    sp[u] = S.Hp ? S.Hp[p[u]] : 0.0;
    sm[u] = S.Hm && m[u] >= 0 ? S.Hm[m[u]] : 0.0;
  }
#pragma unroll 2
  for (int q = 0; q < S.nsp; ++q)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      sp[u] += (double)Sp[q * S.sp_part + p[u]];
      if (m[u] >= 0) sm[u] += (double)Sm[q * S.sm_part + m[u]];
    }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int xr = x0 + ty + 8 * u;
    if (xr >= d || yc > xr) continue;
    const double A = v[u] + sp[u] + sm[u], B = tile[tx][ty + 8 * u] + sp[u] - sm[u];
    const double fock = T.eps[no + gx[u]] + T.eps[no + gy] - ei - ej + eadd;
    auto put = [&](int64_t k, double w) {
      w += fock * x[k];
      sigma[k] = accum ? sigma[k] + w : w;
    };
    if (xr == yc) {
      put(T.aa_off[P] + xr, i == j ? A : -SQRT2 * A);
    } else {
      const int64_t k = T.ab_off[P] + (int64_t)xr * (xr - 1) / 2 + yc;
      if (i == j) {
        put(k, (A + B) * INV_SQRT2);
      } else {  // aa and singlet CSFs with a minus sign (see pack_kernel)
        put(k, -(A + B));
        put(k + m2, SQRT3 * (B - A));
      }
    }
  }
}

// fp16x3 scales of the panel products: mode 0 (slots 11, 12) for W from
// max|C|; mode 1 (slots 6, 5) for the pair products and the 4-internal product
// from max|C| and max|U|
__global__ void panel_scales_kernel(int mode, const unsigned* __restrict__ mx, float* __restrict__ sc) {
  if (threadIdx.x != 0) return;
  const float mc = __uint_as_float(mx[0]);
  const float m = mode == 0 ? 3.f * mc : fmaxf(3.f * mc, __uint_as_float(mx[1]));
  const float s = m > 0.f ? ldexpf(1.f, 13 - ilogbf(m)) : 1.f;
  if (mode == 0) {
    sc[11] = s;
    sc[12] = 1.f / (sc[0] * s);
  } else {
    sc[6] = s;
    sc[5] = 1.f / (sc[0] * s);
  }
}
__global__ void zero_word_kernel(unsigned* p) {
  if (threadIdx.x == 0) *p = 0u;
}

inline unsigned gsz(int64_t work, unsigned cap = 16384) {
  return (unsigned)std::min<int64_t>(std::max<int64_t>(cdiv(work, 256), 1), cap);
}

PanelTab ptab(const tci_plan& P) {
  const auto& Z = P.pp;
  return PanelTab{Z.koff.as<int32_t>(), Z.ld.as<int64_t>(), Z.poff.as<int64_t>(), Z.jpoff.as<int64_t>(),
                  Z.lpoff.as<int64_t>(), Z.pairid.as<int32_t>(), Z.wide ? 1 : 0};
}

// JP and LP of one element type from the integrals
template <bool SPLIT>
void fill_jp_lp(tci_plan& P, tci_plan::PairPanels::Set& F, const double* Fvv, const float* scl, int f16, hipStream_t st) {
  const int n = P.n_int;
  const PanelTab K = ptab(P);
  const dim3 lg((unsigned)P.n_chol, n), b(256);
  if (P.pp.wide) {
    hipLaunchKernelGGL(jp_wide_kernel<SPLIT>, dim3(n, n), b, 0, st, P.tab, K, P.Jvv.as<double>(), Fvv, F.JP.p, scl, f16);
    hipLaunchKernelGGL(lp_wide_kernel<SPLIT>, lg, b, 0, st, P.tab, K, P.Lov.as<double>(), F.LP.p, scl, f16);
  } else {
    hipLaunchKernelGGL(jp_kernel<SPLIT>, dim3(n, n * n), b, 0, st, P.tab, K, P.Jvv.as<double>(), Fvv, F.JP.p, scl, f16);
    hipLaunchKernelGGL(lp_kernel<SPLIT>, lg, b, 0, st, P.tab, K, P.Lov.as<double>(), F.LP.p, scl, f16);
  }
  TCI_HIP(hipGetLastError());
}

void zero(DevBuf& b, size_t bytes, hipStream_t st) {
  b.alloc((size_t)up((int64_t)std::max<size_t>(bytes, 16), 16));
  launch_fill(b.as<double>(), (int64_t)(b.bytes / 8), 0.0, st);
}

constexpr int kAsked = 16;  // modes from here on: one tile shape for all

// tile shape of a d x d pair block under a tiling mode: 0 by size (64, 128,
// 192, in split precision 256; 128-wide tiles above), 1 all 128, 2 all 64, 3 all
// 32 x 32 in four K-groups.  A block on one tile reads its panels once: at
// 16/203/811 (fp16x3) 0.76 ms on 256 x 256 tiles, 0.83 on 128 x 128
int shape_of(int mode, int d, bool split) {
  if (mode >= kAsked) return mode - kAsked;
  if (mode == 3) return N32K4;
  if (mode == 2 || d <= 64) return N64;
  if (mode == 1 || d <= 128) return N128;
  return d <= 192 ? N192 : split && d <= 256 ? N256 : N128;
}
constexpr int kShapes = 6;

}  // namespace

// Layout of the panels: 0 none (gathered products), 1 columns over the domains,
// 2 wide (columns over all virtuals).
//
// Panels over the domains hold |K_i| columns for n_v rows three times, for every
// ordered strong pair's domain once (JP) and for n_chol rows once (LP): JP grows
// as n_int^3 d^2, 72 GB at about 50 full domains of 200.  Beyond that the wide
// ones share JP and LP between the internal orbitals (4 N^2 values, N = n_int
// n_v) for products of K = N.  They are taken while their flops stay below 2.5
// times the gathered products' (domains of a quarter of the virtuals and more):
// the NT GEMM runs at 42-58 TF (FP64), the gathered products at 15-28.  Sigma at
// 60/200/600, gathered -> wide: full domains 2938 -> 234 ms (FP64), 2901 -> 42.5
// (bf16x3); domains of 100-200 1180 -> 150 and 1145 -> 34 ms.
int panels_choose(const tci_plan& P) {
  if (P.n_pairs == 0) return 0;
  const char* env = std::getenv("TCI_DENSE_PAIRS");
  if (env && env[0] == '0') return 0;
  const int n = P.n_int;
  if (n > 255) return 0;  // grids of n_int^2 rows
  const double nv = P.n_v, nc = (double)P.n_chol, np = (double)tri(P.n_v), nw = (double)up(P.n_pairs, 16);
  const double ldw = (double)up(n * up(P.n_v, 8), 16);  // row stride of a wide panel
  double vals = 0.0, kmax = 0.0, f_gather = 0.0, f_wide = 2.0 * n * nc * nv * ldw;
  for (int i = 0; i < n; ++i) {
    double kp = 0.0, rows = 3.0 * nv + nc;
    for (int k = 0; k < n; ++k) {
      const int Q = P.pairid[(size_t)i * n + k];
      if (Q < 0) continue;
      const double d = (double)(P.h_dom_off[Q + 1] - P.h_dom_off[Q]);
      kp += (double)up((int64_t)d, 8);
      rows += d;
    }
    vals += (kp + 16.0) * rows;
    kmax = std::max(kmax, kp + 16.0);
  }
  for (int Q = 0; Q < P.n_pairs; ++Q) {
    const double d = (double)(P.h_dom_off[Q + 1] - P.h_dom_off[Q]);
    for (int e = 0; e < 2; ++e)
      for (int k = 0; k < n; ++k) {
        const int R = P.pairid[(size_t)P.h_pairs[2 * Q + e] * n + k];
        if (R >= 0) f_gather += 6.0 * d * d * (double)(P.h_dom_off[R + 1] - P.h_dom_off[R]);
      }
    f_gather += 4.0 * d * d * nc + 2.0 * d * nv * nc;
    f_wide += 2.0 * d * d * (4.0 * ldw + 2.0 * nc);
  }
  // XT+-, H+-, the 4- and 3-internal factors, U and LovT
  const double common = 2.0 * np * nw + 2.0 * np * P.n_pairs + 2.0 * nw * P.n_pairs + (double)n * n * nv * (n + 1) +
                        2.0 * n * nv * (nc + 16.0);
  size_t freeb = 0, totalb = 0;
  if (hipMemGetInfo(&freeb, &totalb) != hipSuccess) return 0;
  // FP64 and one split copy and the K-split partials, with room left for the
  // ladder's smallest form (T' of a chunk in either precision); gathered rows
  // are addressed by 32-bit byte offsets from a panel
  auto fits = [&](double v, double k) {
    const double need = 12.0 * (v + common) + 8.0 * 9.0 * (double)P.sum_d2;
    return need <= 72.0e9 && need + 24.0e9 <= (double)freeb && 8.0 * k * nv < 4.0e9 && 8.0 * (nc + 16.0) * nv < 4.0e9;
  };
  const bool force = env && env[0] == '2';
  if (!force && fits(vals, kmax)) return 1;
  return fits((4.0 * n * nv + nc) * ldw, ldw) && (force || f_wide <= 2.5 * f_gather) ? 2 : 0;
}

// Do the pair terms of a split build run in split precision?  Where products
// over whole pair blocks (6 N^3 + 4 N^2 n_chol flops, N = n_int n_v) cost at most
// eight times the per-walk ones, i.e. the domains fill a good part of the
// virtual space.  Elsewhere (small domains in a wide space) the pair terms are a few
// percent of the ladder's work: they stay FP64, and the split error is the
// ladder's alone.
bool panels_split_rule(const tci_plan& P) {
  const double N = (double)P.n_int * P.n_v;
  if (8.0 * (6.0 * N * N + 3.0 * P.n_pairs * (double)P.n_v * P.n_v) > 48.0e9 || N >= 46340.0) return false;
  const char* env = std::getenv("TCI_DENSE_PAIRS");
  if (env && (env[0] == '1' || env[0] == '2')) return true;
  double f = 0.0;
  for (int Q = 0; Q < P.n_pairs; ++Q) {
    const double d = (double)(P.h_dom_off[Q + 1] - P.h_dom_off[Q]);
    for (int e = 0; e < 2; ++e)
      for (int k = 0; k < P.n_int; ++k) {
        const int R = P.pairid[(size_t)P.h_pairs[2 * Q + e] * P.n_int + k];
        if (R >= 0) f += 6.0 * d * d * (double)(P.h_dom_off[R + 1] - P.h_dom_off[R]);
      }
    f += 4.0 * d * d * (double)P.n_chol + 2.0 * d * P.n_v * (double)P.n_chol;
  }
  return 6.0 * N * N * N + 4.0 * N * N * (double)P.n_chol <= 8.0 * f;
}

void panels_build(tci_plan& P, const std::vector<double>& o4, hipStream_t st) {
  auto& Z = P.pp;
  Z.split = panels_split_rule(P);
  const int n = P.n_int, nv = P.n_v, np_w = P.n_pairs;
  Z.h_koff.assign((size_t)n * n, -1);
  Z.h_ld.assign(n, 0);
  Z.h_poff.assign(n, 0);
  Z.h_lpoff.assign(n, 0);
  Z.h_jpoff.assign((size_t)n * n, 0);
  Z.n_panel = Z.n_jp = Z.n_lp = 0;
  for (int i = 0; i < n; ++i) {
    int64_t w = 0;
    if (Z.wide) {  // JP_j for every i at j, one LP
      w = n * up(nv, 8);
      Z.h_ld[i] = std::max<int64_t>(up(w, 16), 16);
      Z.h_poff[i] = Z.n_panel;
      Z.n_panel += nv * Z.h_ld[i];
      for (int k = 0; k < n; ++k) {
        if (P.pairid[(size_t)i * n + k] >= 0) Z.h_koff[(size_t)i * n + k] = (int32_t)(k * up(nv, 8));
        Z.h_jpoff[(size_t)i * n + k] = k * nv * Z.h_ld[i];
      }
      Z.n_jp = Z.n_panel;
      Z.n_lp = P.n_chol * Z.h_ld[i];
      continue;
    }
    for (int k = 0; k < n; ++k) {
      const int Q = P.pairid[(size_t)i * n + k];
      if (Q < 0) continue;
      Z.h_koff[(size_t)i * n + k] = (int32_t)w;
      w += up(P.h_dom_off[Q + 1] - P.h_dom_off[Q], 8);
    }
    Z.h_ld[i] = std::max<int64_t>(up(w, 16), 16);
    Z.h_poff[i] = Z.n_panel;
    Z.n_panel += nv * Z.h_ld[i];
    Z.h_lpoff[i] = Z.n_lp;
    Z.n_lp += P.n_chol * Z.h_ld[i];
    for (int j = 0; j < n; ++j) {
      const int Q = P.pairid[(size_t)i * n + j];
      if (Q < 0) continue;
      Z.h_jpoff[(size_t)i * n + j] = Z.n_jp;
      Z.n_jp += (P.h_dom_off[Q + 1] - P.h_dom_off[Q]) * Z.h_ld[i];
    }
  }
  upload(Z.koff, Z.h_koff, st);
  upload(Z.ld, Z.h_ld, st);
  upload(Z.poff, Z.h_poff, st);
  upload(Z.lpoff, Z.h_lpoff, st);
  upload(Z.jpoff, Z.h_jpoff, st);
  upload(Z.pairid, P.pairid, st);
  Z.np = tri(nv);
  Z.nm = tri(nv - 1);
  Z.ldw = up(np_w, 16);
  Z.ldu = up(P.n_chol, 16);
  std::vector<int32_t> colm(np_w, -1);
  Z.ncm = 0;
  for (int Q = 0; Q < np_w; ++Q)
    if (P.h_pairs[2 * Q] != P.h_pairs[2 * Q + 1]) colm[Q] = Z.ncm++;
  upload(Z.colm, colm, st);
  // 4-internal coefficients (o4[((k n + i) n + l) n + j] = (ki|lj))
  std::vector<double> hp((size_t)np_w * Z.ldw, 0.0), hm((size_t)std::max(Z.ncm, 1) * Z.ldw, 0.0);
  for (int X = 0; X < np_w; ++X) {
    const size_t i = P.h_pairs[2 * X], j = P.h_pairs[2 * X + 1];
    for (int Q = 0; Q < np_w; ++Q) {
      const size_t k = P.h_pairs[2 * Q], l = P.h_pairs[2 * Q + 1];
      const double a = o4[((k * n + i) * n + l) * n + j], b = k != l ? o4[((l * n + i) * n + k) * n + j] : 0.0;
      hp[(size_t)X * Z.ldw + Q] = a + b;
      if (colm[X] >= 0 && k != l) hm[(size_t)colm[X] * Z.ldw + Q] = a - b;
    }
  }
  upload(Z.holeP, hp, st);
  upload(Z.holeM, hm, st);
  Z.Hp.alloc((size_t)np_w * Z.np * 8);
  Z.Hm.alloc((size_t)std::max(Z.ncm, 1) * std::max<int64_t>(Z.nm, 1) * 8);
  // 3-internal singles factors
  Z.nk = (int)up(n, 2);
  Z.O3T.alloc((size_t)n * n * nv * Z.nk * 8);
  hipLaunchKernelGGL(o3t_kernel, dim3((unsigned)(n * n)), dim3(256), 0, st, P.O3.as<double>(), n, nv, Z.nk,
                     Z.O3T.as<double>());
  Z.sTp.alloc((size_t)nv * Z.nk * 8);
  // one buffer for every schedule of both element types: the programs keep its
  // address (kMaxKs partials and the 3-internal products of a split sigma)
  Z.Rp.alloc((size_t)(kMaxKs + 1) * P.sum_d2 * 8);
  // FP64 operands
  auto& F = Z.f64;
  for (DevBuf* b : {&F.CR, &F.CC, &F.CT}) zero(*b, (size_t)Z.n_panel * 8, st);
  zero(F.JP, (size_t)Z.n_jp * 8, st);
  zero(F.LP, (size_t)Z.n_lp * 8, st);
  zero(F.U, (size_t)n * nv * Z.ldu * 8, st);
  zero(F.LovT, (size_t)n * nv * Z.ldu * 8, st);
  zero(F.XTp, (size_t)Z.np * Z.ldw * 8, st);
  zero(F.XTm, (size_t)std::max<int64_t>(Z.nm, 1) * Z.ldw * 8, st);
  fill_jp_lp<false>(P, F, P.has_fvv ? P.Fvvp.as<double>() : nullptr, nullptr, 0, st);
  // LovT[(i,a)][J] = Lov[J][(i,a)]
  hipLaunchKernelGGL(u_kernel<false>, dim3((unsigned)cdiv(P.n_chol, 32), (unsigned)cdiv(nv, 32), n), dim3(256), 0, st,
                     nullptr, P.Lov.as<double>(), nv, P.n_chol, (int64_t)nv, (int64_t)n * nv, F.LovT.p, Z.ldu, nullptr, 0);
  TCI_HIP(hipGetLastError());
}

// Split copies of the constant operands (scale slot 0) and zeroed panels.
void panels_build_split(tci_plan& P, hipStream_t st) {
  auto& Z = P.pp;
  auto& F = Z.s16;
  const int n = P.n_int, nv = P.n_v;
  const int f16 = P.mx.prec == TCI_SIGMA_FP16X3 ? 1 : 0;
  const float* s0 = P.mx.scales.as<float>();
  for (DevBuf* b : {&F.CR, &F.CC, &F.CT}) zero(*b, (size_t)Z.n_panel * 4, st);
  zero(F.JP, (size_t)Z.n_jp * 4, st);
  zero(F.LP, (size_t)Z.n_lp * 4, st);
  zero(F.U, (size_t)n * nv * Z.ldu * 4, st);
  zero(F.LovT, (size_t)n * nv * Z.ldu * 4, st);
  zero(F.XTp, (size_t)Z.np * Z.ldw * 4, st);
  zero(F.XTm, (size_t)std::max<int64_t>(Z.nm, 1) * Z.ldw * 4, st);
  zero(F.hP, (size_t)P.n_pairs * Z.ldw * 4, st);
  zero(F.hM, (size_t)std::max(Z.ncm, 1) * Z.ldw * 4, st);
  fill_jp_lp<true>(P, F, nullptr, s0, f16, st);
  hipLaunchKernelGGL(u_kernel<true>, dim3((unsigned)cdiv(P.n_chol, 32), (unsigned)cdiv(nv, 32), n), dim3(256), 0, st,
                     nullptr, P.Lov.as<double>(), nv, P.n_chol, (int64_t)nv, (int64_t)n * nv, F.LovT.p, Z.ldu, s0, f16);
  hipLaunchKernelGGL(split_matrix_kernel, dim3(gsz(P.n_pairs * Z.ldw / 8)), dim3(256), 0, st, Z.holeP.as<double>(),
                     (int64_t)P.n_pairs, Z.ldw, Z.ldw, F.hP.p, Z.ldw, s0, f16);
  hipLaunchKernelGGL(split_matrix_kernel, dim3(gsz(std::max(Z.ncm, 1) * Z.ldw / 8)), dim3(256), 0, st,
                     Z.holeM.as<double>(), (int64_t)std::max(Z.ncm, 1), Z.ldw, Z.ldw, F.hM.p, Z.ldw, s0, f16);
  TCI_HIP(hipGetLastError());
  for (DevBuf* b : {&F.CR, &F.CC, &F.CT, &F.JP, &F.LP, &F.U, &F.LovT, &F.XTp, &F.XTm, &F.hP, &F.hM})
    P.mx.bytes += (int64_t)b->bytes;
}

// W of every internal orbital.
void add_w(tci_plan& P, NProgram& g, bool split) {
  auto& Z = P.pp;
  auto& F = split ? Z.s16 : Z.f64;
  const int n = P.n_int, nv = P.n_v, es = split ? 4 : 8;
  auto at = [&](const DevBuf& b, int64_t values) { return static_cast<const char*>(b.p) + values * es; };
  for (int i = 0; i < n; ++i)
    g.add(P.W.as<double>() + (int64_t)i * P.n_chol * P.ldw, P.ldw, (int)P.n_chol, nv,
            {nseg(at(F.LP, Z.h_lpoff[i]), Z.h_ld[i], at(F.CT, Z.h_poff[i]), Z.h_ld[i], Z.h_ld[i], es)}, false,
            Blocking(), split ? 12 : -1);
}

void panels_w_program(tci_plan& P, bool split, int shape, hipStream_t st) {
  NProgram& g = (split ? P.pp.s16 : P.pp.f64).W;
  g.clear();
  g.split = split;
  g.shape = shape;
  add_w(P, g, split);
  g.upload_tables(st);
}

// Programs of one element type: the 4-internal product over packed pairs, and
// the pair products with `mode` (shape_of), `ks` K-splits and `order` (0:
// walks by descending domain, so that the smallest tasks fill the tail of the
// launch; 1: walks in plan order, dealt XCD-contiguously, so that the walks of
// one i share its panels in an L2); for a split type also the FP64 3-internal
// products.
// With `into` the pair products' tasks go there instead (its shape is set).
void panels_programs(tci_plan& P, bool split, int mode, int ks, int order, hipStream_t st, NProgram* into = nullptr) {
  auto& Z = P.pp;
  auto& F = split ? Z.s16 : Z.f64;
  const int n = P.n_int, nv = P.n_v, es = split ? 4 : 8;
  auto at = [&](const DevBuf& b, int64_t values) { return static_cast<const char*>(b.p) + values * es; };
  if (!into) {
  F.hole.clear();
  F.hole.split = split;
  // large tiles when they fill the chip
  auto fill = [](int64_t m, int64_t nn, int64_t cnt, int t) { return cdiv(m, t) * cdiv(nn, t) * cnt; };
  F.hole.shape = fill(P.n_pairs, Z.np, 2, 128) >= 512 ? N128 : fill(P.n_pairs, Z.np, 2, 64) >= 256 ? N64 : N32K4;
  const void* hP = split ? F.hP.p : Z.holeP.p;
  const void* hM = split ? F.hM.p : Z.holeM.p;
  F.hole.add(Z.Hp.as<double>(), Z.np, P.n_pairs, (int)Z.np, {nseg(hP, Z.ldw, F.XTp.p, Z.ldw, Z.ldw, es)}, false,
             Blocking(), split ? 5 : -1);
  if (Z.ncm > 0 && Z.nm > 0)
    F.hole.add(Z.Hm.as<double>(), Z.nm, Z.ncm, (int)Z.nm, {nseg(hM, Z.ldw, F.XTm.p, Z.ldw, Z.ldw, es)}, false,
               Blocking(), split ? 5 : -1);
  F.hole.upload_tables(st);
  }
  // pair products
  F.ks = ks;
  if (!into) {
    F.pair.clear();
    F.pair.resize(kShapes);
  }
  for (int s = 0; s < (into ? 0 : kShapes); ++s) {
    F.pair[s].split = split;
    F.pair[s].shape = s;
    F.pair[s].remap = order;
  }
  TCI_REQUIRE(ks >= 1 && ks <= kMaxKs, "K-splits of the pair products out of range");
  if (split) Z.rank.clear();
  Z.rank.shape = P.dmax <= 64 ? N64 : N128;
  std::vector<int> walks(P.n_pairs);
  for (int Q = 0; Q < P.n_pairs; ++Q) walks[Q] = Q;
  if (order == 0)
    std::stable_sort(walks.begin(), walks.end(), [&](int a, int b) {
      return P.h_dom_off[a + 1] - P.h_dom_off[a] > P.h_dom_off[b + 1] - P.h_dom_off[b];
    });
  for (int Q : walks) {
    const int i = P.h_pairs[2 * Q], j = P.h_pairs[2 * Q + 1];
    const int d = (int)(P.h_dom_off[Q + 1] - P.h_dom_off[Q]);
    const int32_t* D = P.dom_idx.as<int32_t>() + P.h_dom_off[Q];
    const int64_t li = Z.h_ld[i], lj = Z.h_ld[j];
    const char *CRi = at(F.CR, Z.h_poff[i]), *CRj = at(F.CR, Z.h_poff[j]), *CCi = at(F.CC, Z.h_poff[i]),
               *CCj = at(F.CC, Z.h_poff[j]);
    const char *Jij = at(F.JP, Z.h_jpoff[(size_t)i * n + j]), *Jji = at(F.JP, Z.h_jpoff[(size_t)j * n + i]);
    const char *Ui = at(F.U, (int64_t)i * nv * Z.ldu), *Uj = at(F.U, (int64_t)j * nv * Z.ldu);
    const char *Li = at(F.LovT, (int64_t)i * nv * Z.ldu), *Lj = at(F.LovT, (int64_t)j * nv * Z.ldu);
    // the two ranges that read one JP run interleaved in chunks of k, so that
    // its second read finds it in cache
    std::vector<NSeg> sg;
    auto two = [&](const NSeg& u, const NSeg& v) {
      constexpr int64_t chunk = 4096;  // bytes of k: 512 FP64 values, 1024 split ones
      for (int64_t k = 0; k < u.kbytes; k += chunk)
        for (const NSeg* q : {&u, &v}) {
          NSeg c = *q;
          c.A = static_cast<const char*>(q->A) + k;
          c.B = static_cast<const char*>(q->B) + k;
          c.kbytes = std::min(chunk, q->kbytes - k);
          sg.push_back(c);
        }
    };
    const int32_t* DJ = Z.wide ? D : nullptr;  // rows of JP: all virtuals, or the walk's own
    two(nseg(CRi, li, Jij, li, li, es, D, DJ), nseg(Jij, li, CCi, li, li, es, DJ, D));
    two(nseg(Jji, lj, CRj, lj, lj, es, DJ, D), nseg(CCj, lj, Jji, lj, lj, es, D, DJ));
    sg.push_back(nseg(Ui, Z.ldu, Lj, Z.ldu, Z.ldu, es, D, D));
    sg.push_back(nseg(Li, Z.ldu, Uj, Z.ldu, Z.ldu, es, D, D));
    const double* Oij = Z.O3T.as<double>() + ((int64_t)i * n + j) * nv * Z.nk;
    const double* Oji = Z.O3T.as<double>() + ((int64_t)j * n + i) * nv * Z.nk;
    const NSeg r1 = nseg(Z.sTp.p, Z.nk, Oij, Z.nk, Z.nk, 8, D, D), r2 = nseg(Oji, Z.nk, Z.sTp.p, Z.nk, Z.nk, 8, D, D);
    if (split) {
      Z.rank.add(Z.Rp.as<double>() + (int64_t)kMaxKs * P.sum_d2 + P.h_cd_off[Q], d, d, d, {r1, r2}, false);
    } else {
      sg.push_back(r1);
      sg.push_back(r2);
    }
    int64_t tot = 0;
    for (const NSeg& s : sg) tot += s.kbytes;
    NProgram& g = into ? *into : F.pair[shape_of(mode, d, split)];
    for (int s = 0; s < ks; ++s) {
      const int64_t b0 = (tot * s / ks) & ~(int64_t)127, b1 = s + 1 == ks ? tot : (tot * (s + 1) / ks) & ~(int64_t)127;
      std::vector<NSeg> part;
      int64_t pos = 0;
      for (const NSeg& q : sg) {
        const int64_t u = std::max(b0, pos), v = std::min(b1, pos + q.kbytes);
        if (u < v) {
          NSeg c = q;
          c.A = static_cast<const char*>(q.A) + (u - pos);
          c.B = static_cast<const char*>(q.B) + (u - pos);
          c.kbytes = v - u;
          part.push_back(c);
        }
        pos += q.kbytes;
      }
      const int64_t o = (int64_t)s * P.sum_d2 + P.h_cd_off[Q];
      double* Rout = split ? reinterpret_cast<double*>(Z.Rp.as<float>() + o) : Z.Rp.as<double>() + o;
      g.add(Rout, d, d, d, part, false, Blocking(), split ? 5 : -1, split);
    }
  }
  if (into) return;
  for (auto& g : F.pair) g.upload_tables(st);
  if (split) Z.rank.upload_tables(st);
}

// Times tilings and K-splits of the pair products and keeps the fastest.
void panels_tune(tci_plan& P, int precision, hipStream_t st) {
  const bool split = precision != TCI_SIGMA_FP64;
  auto& Z = P.pp;
  auto& F = split ? Z.s16 : Z.f64;
  const float* sc = P.mx.scales.as<float>();
  // split types keep an FP32 chain no longer than about a quarter of the
  // contraction (the partial sums meet in FP64)
  const int kmin = split ? 4 : 1;
  auto wrule = [&] {
    auto fill = [&](int t) { return cdiv(P.n_chol, t) * cdiv(P.n_v, t) * P.n_int; };
    return fill(128) >= 512 ? N128 : fill(64) >= 256 ? N64 : N32K4;
  };
  const NSchedule asked = asked_schedule("TCI_PANEL_TILE", split);
  if (asked.shape >= 0) {
    panels_w_program(P, split, asked.shape, st);
    panels_programs(P, split, kAsked + asked.shape, std::min(std::max(kmin, asked.ks), kMaxKs), asked.order, st);
    return;
  }
  if (!autotune_enabled()) {
    panels_w_program(P, split, wrule(), st);
    panels_programs(P, split, 0, kmin, 0, st);
    return;
  }
  if (split && Z.tuned_mode >= 0) {  // tuned for the other split precision: same tiles, same sums
    panels_w_program(P, split, Z.tuned_w, st);
    panels_programs(P, split, Z.tuned_mode, Z.tuned_ks, Z.tuned_order, st);
    return;
  }
  // operands of a random vector (scales of fp16x3 included) before the timing
  panels_w_program(P, split, wrule(), st);
  panels_programs(P, split, 0, kmin, 0, st);
  DevBuf xr;
  P.tune_vector(xr, st);
  if (precision == TCI_SIGMA_FP16X3)
    launch_split_scales(1, P.C.as<double>(), P.sum_d2, P.mx.maxbits.as<unsigned>(), 0, P.mx.scales.as<float>(),
                        (float)P.dmax, st);
  P.run_Y(precision, st, false);
  panels_terms(P, precision, false, xr.as<double>(), nullptr, st);
  TCI_HIP(hipStreamSynchronize(st));
  static const char* mname[4] = {"by size", "128", "64", "32k4"};
  double tiles128 = 0.0;
  for (int Q = 0; Q < P.n_pairs; ++Q) {
    const int64_t c = cdiv(P.h_dom_off[Q + 1] - P.h_dom_off[Q], 128);
    tiles128 += (double)(c * c);
  }
  std::string log = std::string(split ? "split" : "fp64") + (Z.wide ? " wide pair panels: W" : " pair panels: W");
  double best = 1e300;
  int bw = N128;
  std::vector<int> wshapes = {N128, N192, N64};
  if (split) wshapes.push_back(N128x192);
  if (wrule() == N32K4) wshapes.push_back(N32K4);
  for (int sh : wshapes) {
    panels_w_program(P, split, sh, st);
    const double ms = time_ms(st, 2, [&] { F.W.launch(precision, st, 0, sc); });
    log += " " + std::to_string(F.W.tm()) + "x" + std::to_string(F.W.tn()) + ":" + fmt_ms(ms);
    if (ms < best * 0.98) {
      best = ms;
      bw = sh;
    }
  }
  panels_w_program(P, split, bw, st);
  log += "; products";
  best = 1e300;
  int bm = 0, bk = kmin, bo = 0;
  for (int mode = 0; mode < 4; ++mode) {
    if (mode == 3 && tiles128 > 256) continue;  // enough tiles without K-groups
    if (mode == 2 && tiles128 > 4096) continue;
    for (int ks : {1, 2, 4, 8}) {
      if (ks < kmin || (ks > kmin && tiles128 * ks > 8192)) continue;
      for (int o = 0; o < (xcd_remap_forced() ? 1 : 2); ++o) {
        panels_programs(P, split, mode, ks, o, st);
        const double ms = time_ms(st, 2, [&] {
          for (const auto& g : F.pair)
            if (!g.tasks.empty()) g.launch(precision, st, 0, sc);
        });
        log += std::string(" ") + mname[mode] + "/" + std::to_string(ks) + (o ? "x:" : ":") + fmt_ms(ms);
        if (ms < best * 0.98) {
          best = ms;
          bm = mode;
          bk = ks;
          bo = o;
        }
      }
    }
  }
  panels_programs(P, split, bm, bk, bo, st);
  if (split) {
    Z.tuned_mode = bm;
    Z.tuned_ks = bk;
    Z.tuned_order = bo;
    Z.tuned_w = bw;
  }
  P.tuning += log + " -> W " + std::to_string(F.W.tm()) + "x" + std::to_string(F.W.tn()) + ", " + mname[bm] + "/" +
              std::to_string(bk) + (bo ? "x" : "") + "\n";
  TCI_HIP(hipStreamSynchronize(st));
}

// Small FP64 builds: S+-, W and Y do not depend on each other and none fills
// the chip, so they go out as one launch on small tiles; likewise the pair
// products and gW.  Kept where the one launch beats the separate ones: at
// 5/30/175 the first group takes 12 us instead of 35, the second 12 instead of 25.
void panels_merge(tci_plan& P, hipStream_t st) {
  auto& Z = P.pp;
  auto& F = Z.f64;
  Z.m1on = Z.m2on = false;
  double fl = F.W.alg_flops;
  for (const auto& g : F.pair) fl += g.alg_flops;
  // TCI_MERGE=tile/ks merges both groups so (64 or 32k4), =0 neither
  const NSchedule asked = asked_schedule("TCI_MERGE", false);
  const bool force = asked.shape == N64 || asked.shape == N32K4;
  const char* env = std::getenv("TCI_MERGE");
  if (!P.vv.fp64 || (env && env[0] == '0')) return;
  if (!force && (!autotune_enabled() || fl + P.vv.g64.alg_flops > 4.0e10)) return;
  const bool sing = P.singles_nt();
  const bool gw = !P.nprogGW.tasks.empty();
  Z.m1_singles = sing;
  Z.m2_singles = gw;
  std::string log = "fp64 merged launches:";
  const int kp0 = F.ks;
  // S, W, Y
  double t0 = time_ms(st, 3, [&] {
    P.vv.g64.launch(TCI_SIGMA_FP64, st);
    F.W.launch(TCI_SIGMA_FP64, st);
    if (sing) P.nprogY.launch(TCI_SIGMA_FP64, st);
  });
  log += " S, W, Y separate:" + fmt_ms(t0);
  double best = t0 * 0.98;
  int bs = -1, bk = 1;
  auto build1 = [&](int sh, int ks) {
    Z.m1.clear();
    Z.m1.shape = sh;
    vv_add_products(P, Z.m1, false, ks);
    add_w(P, Z.m1, false);
    if (sing) P.add_singles_Y(Z.m1);
    Z.m1.upload_tables(st);
  };
  const int64_t kmin = P.vv.ncm > 0 ? std::min(P.vv.np, P.vv.nm) : P.vv.np;
  if (force) {
    best = 0.0;
    bs = asked.shape;
    bk = (int)std::max<int64_t>(1, std::min<int64_t>({(int64_t)asked.ks, 4, kmin / 64}));
  }
  for (int sh : {(int)N64, (int)N32K4})
    for (int ks : {1, 2, 4}) {
      if (force || (ks > 1 && ks > kmin / 64)) continue;
      build1(sh, ks);
      const double ms = time_ms(st, 3, [&] { Z.m1.launch(TCI_SIGMA_FP64, st); });
      log += std::string(sh == N64 ? " 64/" : " 32k4/") + std::to_string(ks) + ":" + fmt_ms(ms);
      if (ms < best) {
        best = ms;
        bs = sh;
        bk = ks;
      }
    }
  if (bs >= 0) {
    build1(bs, bk);
    Z.m1on = true;
    Z.m1_ks = bk;
  } else {
    Z.m1.clear();
  }
  // pair products, gW
  t0 = time_ms(st, 3, [&] {
    for (const auto& g : F.pair)
      if (!g.tasks.empty()) g.launch(TCI_SIGMA_FP64, st);
    if (gw) P.nprogGW.launch(TCI_SIGMA_FP64, st);
  });
  log += "; pairs, gW separate:" + fmt_ms(t0);
  best = t0 * 0.98;
  bs = -1;
  if (force) {
    best = 0.0;
    bs = asked.shape;
    bk = std::min(asked.ks, kMaxKs);
  }
  auto build2 = [&](int sh, int ks) {
    Z.m2.clear();
    Z.m2.shape = sh;
    panels_programs(P, false, 0, ks, 0, st, &Z.m2);
    if (gw) P.add_singles_GW(Z.m2);
    Z.m2.upload_tables(st);
  };
  for (int sh : {(int)N64, (int)N32K4})
    for (int ks : {1, 2, 4, 8}) {
      if (force) continue;
      build2(sh, ks);
      const double ms = time_ms(st, 3, [&] { Z.m2.launch(TCI_SIGMA_FP64, st); });
      log += std::string(sh == N64 ? " 64/" : " 32k4/") + std::to_string(ks) + ":" + fmt_ms(ms);
      if (ms < best) {
        best = ms;
        bs = sh;
        bk = ks;
      }
    }
  if (bs >= 0) {
    build2(bs, bk);
    Z.m2on = true;
    Z.m2_ks = bk;
  } else {
    Z.m2.clear();
  }
  F.ks = kp0;  // of the separate programs, which split builds may run
  P.tuning += log + " -> " + (Z.m1on ? "merged " : "separate ") + (Z.m2on ? "merged" : "separate") + "\n";
  TCI_HIP(hipStreamSynchronize(st));
}

// arithmetic of the pair terms in a build of this precision
int panels_precision(const tci_plan& P, int precision) {
  return precision != TCI_SIGMA_FP64 && P.pp.split ? precision : (int)TCI_SIGMA_FP64;
}

// Are the virtual Fock products part of the pair products (FP64 ones only: split
// operands would round F)?  A launch of their own took 114 us of 1.54 ms at
// 13/151/607.
bool panels_hold_fock(const tci_plan& P, int precision) {
  return P.pp.on && panels_precision(P, precision) == TCI_SIGMA_FP64;
}

// Is the 4-internal product a K-range of the resident ladder's product?  Then
// its operand XT+- is written before the ladder and no H+- exists.  Not where
// the two differ in arithmetic or (fp16x3) in their scales.
bool panels_hole_in_ladder(const tci_plan& P, int precision) {
  return P.pp.on && panels_precision(P, precision) == precision &&
         (precision == TCI_SIGMA_FP64 ? P.vv.fp64 : precision == TCI_SIGMA_BF16X3 && P.vv.split);
}

// One pass over the CI vector for everything the build reads of it (FP64 and
// bf16x3); false where the separate kernels are needed.
bool panels_expand(tci_plan& P, int precision, const double* x, const IoSlot* io, hipStream_t st) {
  if (!P.pp.on) return false;
  auto& Z = P.pp;
  const bool vv = precision != TCI_SIGMA_FP64 ? P.vv.split : P.vv.fp64;
  const int pp = panels_precision(P, precision);
  if (pp == TCI_SIGMA_FP16X3 || (vv && pp != precision)) return false;
  const bool split = pp != TCI_SIGMA_FP64;
  auto& F = split ? Z.s16 : Z.f64;
  ExpandOut O{};
  // C itself is read by the Cholesky-direct ladders and the virtual Fock products
  O.C = !vv || (P.has_fvv && split) ? P.C.as<double>() : nullptr;
  O.Ct = P.Ct.as<double>();
  O.s = P.s.as<double>();
  O.sT = Z.sTp.as<double>();
  O.nk = Z.nk;
  O.sP = P.sP.as<double>();
  O.ldw = P.ldw;
  O.CR = F.CR.p;
  O.CC = F.CC.p;
  O.CT = F.CT.p;
  if (vv) {
    O.Xp = split ? P.vv.Xpx.p : P.vv.Xp.p;
    O.Xm = split ? P.vv.Xmx.p : P.vv.Xm.p;
    O.ldp = split ? xpad(Z.np) : up(Z.np, 2);
    O.ldm = split ? xpad(Z.nm) : up(Z.nm, 2);
  }
  O.colm = Z.colm.as<int32_t>();
  const int nt = (P.dmax + 31) / 32;
  O.pos = P.pos.as<int32_t>();
  O.XTp = F.XTp.p;
  O.XTm = F.XTm.p;
  O.ldx = Z.ldw;
  // blocks of XT+-, in rows of the grid's width (at most 32768 rows)
  const int64_t nxt = (int64_t)P.n_v * cdiv(P.n_v, 32) * cdiv(P.n_pairs, 32);
  const int64_t gx = std::max<int64_t>({(int64_t)nt * (nt + 1) / 2, 4, cdiv(nxt, 32768)});
  const dim3 g((unsigned)gx, (unsigned)(P.n_pairs + 1 + cdiv(nxt, gx)));
  const PanelTab K = ptab(P);
  if (split) hipLaunchKernelGGL(expand_kernel<true>, g, dim3(256), 0, st, P.tab, K, x, io, O);
  else hipLaunchKernelGGL(expand_kernel<false>, g, dim3(256), 0, st, P.tab, K, x, io, O);
  TCI_HIP(hipGetLastError());
  return true;
}

// XT+- from the CI vector (needs no scale but that of fp16x3's pair products)
void panels_xt(tci_plan& P, int precision, const double* x, const IoSlot* io, hipStream_t st) {
  auto& Z = P.pp;
  precision = panels_precision(P, precision);
  const bool split = precision != TCI_SIGMA_FP64;
  const int f16 = precision == TCI_SIGMA_FP16X3 ? 1 : 0;
  const dim3 g((unsigned)P.n_v, (unsigned)cdiv(P.n_v, 32), (unsigned)cdiv(P.n_pairs, 32));
  if (split)
    hipLaunchKernelGGL(xt_kernel<true>, g, dim3(256), 0, st, P.tab, P.pos.as<int32_t>(), x, io, Z.s16.XTp.p, Z.s16.XTm.p,
                       Z.ldw, P.mx.scales.as<float>() + 6, f16);
  else
    hipLaunchKernelGGL(xt_kernel<false>, g, dim3(256), 0, st, P.tab, P.pos.as<int32_t>(), x, io,
                       Z.f64.XTp.p, Z.f64.XTm.p, Z.ldw, nullptr, 0);
  TCI_HIP(hipGetLastError());
}

// Pair terms of one sigma into the K-split partials and H+-; needs Y, and C and
// s unless panels_expand has written the panels (`expanded`).
void panels_terms(tci_plan& P, int build, bool expanded, const double* x, const IoSlot* io, hipStream_t st) {
  auto& Z = P.pp;
  const int precision = panels_precision(P, build);
  const bool split = precision != TCI_SIGMA_FP64;
  auto& F = split ? Z.s16 : Z.f64;
  const int n = P.n_int, nv = P.n_v;
  const int f16 = precision == TCI_SIGMA_FP16X3 ? 1 : 0;
  const std::string pn = precision == TCI_SIGMA_FP64 ? "fp64" : (f16 ? "fp16x3" : "bf16x3");
  float* sc = split ? P.mx.scales.as<float>() : nullptr;
  unsigned* mx = f16 ? P.mx.maxbits.as<unsigned>() : nullptr;
  const PanelTab K = ptab(P);
  const int nt = (P.dmax + 31) / 32;
  auto run = [&](const std::string& role, const NProgram& g, int prec) {
    if (!g.tasks.empty()) P.kt_run(pn + " " + role, g, build, st, [&] { g.launch(prec, st, 0, sc); });
  };
  auto panels = [&](int what) {
    const dim3 g(nt * nt, P.n_pairs);
    if (split)
      hipLaunchKernelGGL(panels_kernel<true>, g, dim3(256), 0, st, P.tab, K, P.C.as<double>(), F.CR.p, F.CC.p, F.CT.p,
                         sc + 6, sc + (f16 ? 11 : 6), f16, what);
    else
      hipLaunchKernelGGL(panels_kernel<false>, g, dim3(256), 0, st, P.tab, K, P.C.as<double>(), F.CR.p, F.CC.p, F.CT.p,
                         nullptr, nullptr, 0, 3);
  };
  int e0 = -1;
  if (!expanded) {
    e0 = P.kt_begin(st);
    if (f16) hipLaunchKernelGGL(panel_scales_kernel, dim3(1), dim3(64), 0, st, 0, mx, sc);
    panels(f16 ? 2 : 3);  // fp16x3: the scale of CR and CC waits for max|U|
    hipLaunchKernelGGL(st_kernel, dim3(gsz((int64_t)nv * Z.nk)), dim3(256), 0, st, P.s.as<double>(), n, nv, Z.nk,
                       Z.sTp.as<double>());
    TCI_HIP(hipGetLastError());
    P.kt_end(e0, pn + " pair panels", 0.0, build, st);
  }
  if (build != TCI_SIGMA_FP64 || !Z.m1on) run("pair product W", F.W, precision);
  e0 = P.kt_begin(st);
  if (f16) {
    hipLaunchKernelGGL(zero_word_kernel, dim3(1), dim3(64), 0, st, mx + 1);
    hipLaunchKernelGGL(u_absmax_kernel, dim3(gsz((int64_t)n * nv * P.n_chol, 1024)), dim3(256), 0, st,
                       P.Y.as<double>(), P.W.as<double>(), (int64_t)n * nv * P.n_chol, nv, (int)(P.ldw - nv), mx + 1);
    hipLaunchKernelGGL(panel_scales_kernel, dim3(1), dim3(64), 0, st, 1, mx, sc);
    panels(1);
  }
  const dim3 gu((unsigned)cdiv(P.n_chol, 32), (unsigned)cdiv(nv, 32), n);
  if (split) {
    hipLaunchKernelGGL(u_kernel<true>, gu, dim3(256), 0, st, P.Y.as<double>(), P.W.as<double>(), nv, P.n_chol,
                       P.n_chol * P.ldw, P.ldw, F.U.p, Z.ldu, sc + 6, f16);
  } else {
    hipLaunchKernelGGL(u_kernel<false>, gu, dim3(256), 0, st, P.Y.as<double>(), P.W.as<double>(), nv, P.n_chol,
                       P.n_chol * P.ldw, P.ldw, F.U.p, Z.ldu, nullptr, 0);
  }
  TCI_HIP(hipGetLastError());
  const bool hole = !panels_hole_in_ladder(P, build);
  if (hole && !expanded) panels_xt(P, precision, x, io, st);
  P.kt_end(e0, pn + " pair panels", 0.0, build, st);
  if (build == TCI_SIGMA_FP64 && Z.m2on) {
    run("pair products, gW", Z.m2, precision);
  } else {
    for (const auto& g : F.pair) run("pair products", g, precision);
  }
  if (split && !Z.rank.tasks.empty())
    P.kt_run(pn + " 3-internal products", Z.rank, build, st, [&] { Z.rank.launch(TCI_SIGMA_FP64, st); });
  if (hole) run("4-internal product", F.hole, precision);
}

// sigma from the pair terms' partials, the ladder (packed S+- when `packed`,
// otherwise R) and the singles
void panels_pack(tci_plan& P, int precision, bool packed, bool use_r, const double* x, const IoSlot* io, int flags,
                 double* y, hipStream_t st) {
  auto& Z = P.pp;
  const bool split = precision != TCI_SIGMA_FP64, psplit = split && Z.split;
  PackSrc S{};
  S.Rp = Z.Rp.p;
  S.rstride = P.sum_d2;
  // an FP64 build may have merged its pair products on another K-split
  S.nrp = psplit ? Z.s16.ks : split || !Z.m2on ? Z.f64.ks : Z.m2_ks;
  S.rank = psplit ? Z.Rp.as<double>() + (int64_t)kMaxKs * P.sum_d2 : nullptr;
  S.R = use_r ? P.R.as<double>() : nullptr;
  S.np = Z.np;
  S.nm = Z.nm;
  if (packed) {
    S.nsp = split ? P.vv.ksx : Z.m1on ? Z.m1_ks : P.vv.ks;
    S.Sp = P.vv.Sp.p;
    S.Sm = P.vv.Sm.p;
    S.sp_part = (int64_t)P.n_pairs * Z.np;
    S.sm_part = (int64_t)std::max(Z.ncm, 1) * Z.nm;
  }
  if (!panels_hole_in_ladder(P, precision)) {
    S.Hp = Z.Hp.as<double>();
    S.Hm = Z.Hm.as<double>();
  }
  S.colm = Z.colm.as<int32_t>();
  S.Kov = P.Kov.as<double>();
  const int nt = (P.dmax + 31) / 32;
  auto pack = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)std::max<int64_t>(nt * (nt + 1) / 2, 4), P.n_pairs + 1), dim3(256), 0, st,
                       P.tab, S, x, P.g.as<double>(), P.sig0.as<double>(), P.e_ref, flags, y, io);
  };
  if (psplit) packed ? pack(pack_panels_kernel<float, float>) : pack(pack_panels_kernel<float, double>);
  else if (split && packed) pack(pack_panels_kernel<double, float>);
  else pack(pack_panels_kernel<double, double>);
  TCI_HIP(hipGetLastError());
}

int64_t panels_device_bytes(const tci_plan& P) {
  const auto& Z = P.pp;
  int64_t b = 0;
  for (const auto* F : {&Z.f64, &Z.s16})
    for (const DevBuf* x : {&F->CR, &F->CC, &F->CT, &F->JP, &F->LP, &F->U, &F->LovT, &F->XTp, &F->XTm, &F->hP, &F->hM})
      b += (int64_t)x->bytes;
  for (const DevBuf* x : {&Z.koff, &Z.ld, &Z.poff, &Z.jpoff, &Z.lpoff, &Z.pairid, &Z.colm, &Z.holeP, &Z.holeM, &Z.Hp,
                          &Z.Hm, &Z.O3T, &Z.sTp, &Z.Rp})
    b += (int64_t)x->bytes;
  return b;
}

}  // namespace tci
