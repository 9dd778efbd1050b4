// gfx950 kernels of the frontal subdomain factors (doug_fronts.hpp): scatter
// of the matrix entries, the factorisation height by height, and the solves.
#include "doug_tile.hpp"
#include "doug_front_kernels.hpp"

namespace doug {

namespace {

// Pointers out of a descriptor are generic: as global ones their loads do not
// count as LDS accesses.
template <typename U>
using Global = const U __attribute__((address_space(1))) *;
template <typename U>
__device__ __forceinline__ Global<U> global(const U* p) {
  return reinterpret_cast<Global<U>>(reinterpret_cast<uint64_t>(p));
}

// A value that is the same in every lane, in a scalar register.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// element (row, col) of a panel of H rows (host: front_elem)
template <typename T>
__device__ __forceinline__ int panel_elem(int H, int row, int col) {
  const int g = col >> 2, j = col & 3, base = 4 * (g * H - 2 * g * (g - 1));
  if (sizeof(T) == 4) return base + 4 * (row - 4 * g) + j;
  return base + (j >> 1) * 2 * (H - 4 * g) + 2 * (row - 4 * g) + (j & 1);
}

__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// ------------------------------------------------------------------------
// set-up
// ------------------------------------------------------------------------

// The lower entries of each subdomain's matrix into its zeroed panels; A must
// hold no (i, j) pair twice.
template <typename T>
__global__ __launch_bounds__(256) void k_front_scatter(T* __restrict__ tiles, const FrontSub* __restrict__ subs,
                                                       const int32_t* __restrict__ inds,
                                                       const int32_t* __restrict__ occ_ptr,
                                                       const int32_t* __restrict__ occ_pos,
                                                       const int32_t* __restrict__ a_ptr,
                                                       const int32_t* __restrict__ a_col,
                                                       const double* __restrict__ a_val) {
  const FrontSub s = subs[blockIdx.x];
  const int s0 = (int)s.vec;
  for (int p = blockIdx.y * 256 + threadIdx.x; p < s.n; p += 256 * gridDim.y) {
    const int g = inds[s0 + p];
    for (int e = a_ptr[g]; e < a_ptr[g + 1]; e++) {
      const int q = local_col(occ_ptr, occ_pos, a_col[e], s0, s.n);
      if (q < 0 || q > p) continue;
      const Front f = s.fronts[s.colfront[q]];
      int row = p - f.c0;
      if (row >= f.k) {  // a boundary row: its place in the ascending list
        const uint16_t* rp = s.rpos + f.row0;
        int lo = f.k, hi = f.k + f.m;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (rp[mid] <= p) lo = mid;
          else hi = mid;
        }
        row = lo;
      }
      tiles[s.base + f.pan + panel_elem<T>(f.k + f.m, row, q - f.c0)] = (T)a_val[e];
    }
  }
}

// Cholesky factor of a k x k block (k <= 32) at As (row stride LDX, lower
// part) and D = L^-1 at Bs, zeros right of the diagonal, by one wavefront in
// registers: lane r holds row r, a column step broadcasts the pivot column's
// entries through scalar registers (v_readlane), so that a step waits on no
// LDS access or cross-lane permute.  D by rows, x L = e_r, last column first.
// As ends with L.  A non-positive pivot is replaced by 1 and reported as `id`.
template <typename T, int LDX>
__device__ __forceinline__ void wave_factor_invert(T* As, T* Bs, int k, int lane, int id, int* flag) {
  constexpr int KB = 32;
  T v[KB];
  const int r = lane & 31;
#pragma unroll
  for (int c = 0; c < KB; c++) v[c] = As[r * LDX + c];
  T rinv = (T)0;  // lane r: 1 / L_rr
#pragma unroll
  for (int c = 0; c < KB; c++)
    if (c < k) {
      T piv = lane_value(v[c], c);
      if (!(piv > (T)0)) {
        if (lane == 0) atomicCAS(flag, 0, id);
        piv = (T)1;
      }
      const T sc = rsqrt(piv);
      rinv = lane == c ? sc : rinv;
      v[c] = lane == c ? piv * sc : v[c] * sc;
#pragma unroll
      for (int q0 = c + 1 - (c + 1) % 8; q0 < KB; q0 += 8)
        if (q0 < k) {
#pragma unroll
          for (int q = q0; q < q0 + 8; q++)
            if (q > c) v[q] = v[q] - v[c] * lane_value(v[c], q);
        }
    }
  if (lane < k) {
#pragma unroll
    for (int c = 0; c < KB; c++)
      if (c < k) As[lane * LDX + c] = c <= lane ? v[c] : (T)0;
  }
  if (sizeof(T) == 8) wave_lds_sync();
  T x[KB];
#pragma unroll
  for (int c = 0; c < KB; c++) x[c] = lane == c ? (T)1 : (T)0;
#pragma unroll
  for (int c = KB - 1; c >= 0; c--)
    if (c < k) {
      x[c] = x[c] * lane_value(rinv, c);
      // L's row c: from its lane (FP32), or from LDS where two sets of rows
      // would take too many registers
#pragma unroll
      for (int j = 0; j < c; j++) x[j] = x[j] - x[c] * (sizeof(T) == 4 ? lane_value(v[j], c) : As[c * LDX + j]);
    }
  if (lane < k) {
#pragma unroll
    for (int c = 0; c < KB; c++)
      if (c < k) Bs[lane * LDX + c] = c <= lane ? x[c] : (T)0;
  }
}

// A child's update matrix as the parent reads it.
template <typename T>
struct Child {
  const T* s;
  int m, u;  // rows, work index of its first update entry
  // row of the child that record x (half c) names, -1 if none
  __device__ __forceinline__ int row(uint32_t x, int c, int none) const {
    const int i = c == 0 ? (int)(x & 0xffffu) : (int)(x >> 16);
    return i != none ? i - u : -1;
  }
  // entry (i, j), or entry 0 where either is missing; see kept()
  __device__ __forceinline__ T read(int i, int j) const { return s[(uint32_t)(i >= 0 && j >= 0 ? i * m + j : 0)]; }
};
template <typename T>
__device__ __forceinline__ T kept(T x, int i, int j) {
  return i >= 0 && j >= 0 ? x : (T)0;
}

// One front of height h per workgroup of NW wavefronts (its children's update
// matrices are complete), fronts of at most 16 NB columns, or with NB = 4
// those of more than 32.  The pivot block and its inverse D in LDS; then each
// wavefront takes 16 boundary rows at a time, L_RS = F_RS D^T, kept in the
// panel; then 32x32 tiles of the update matrix F_RR - L_RS L_RS^T, their
// operands read from the panel (through L2) straight into the matrix cores'
// registers; and last C = L_RS D over L_RS.  Only three workgroup barriers
// follow the pivot block, and LDS holds nothing but that block, so that many
// fronts are in flight per CU: the work is bound by the latency of short
// dependent steps, not by arithmetic or bandwidth.  Whole factorisation, 512
// subdomains of 5440 unknowns: 11.7 ms in FP64 and 8.7 ms in FP32 (11.9 and
// 7.4 ms for the envelope factor with its 2.7 times as many entries); 64 of
// 3900 in two dimensions: 1.5 ms (4.7 ms).
template <typename T, int NB, int NW>
__global__ __launch_bounds__(64 * NW) void k_front_factor(T* tiles, T* schur, const FrontSub* __restrict__ subs,
                                                          int h, int* __restrict__ flag) {
  constexpr int KB = 16 * NB, LDX = KB + 1, NG = 4 * NB;
  __shared__ T As[KB * LDX];
  __shared__ T Bs[KB * LDX];
  __shared__ int mc[2][KB];  // rows of the children for the pivot columns
  typedef typename Mma<T>::v4 V;
  const FrontSub s = subs[blockIdx.x];
  if (h >= s.nheights) return;
  const int fi = s.hptr[h] + blockIdx.y;
  if (fi >= s.hptr[h + 1]) return;
  const Front f = s.fronts[s.hlist[fi]];
  const int k = uniform(f.k), m = uniform(f.m), H = k + m, ng = (k + 3) >> 2, n = s.n;
  if (NB == 4 ? k <= 32 : k > KB) return;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  T* pan = tiles + s.base + uniform(f.pan);
  T* S = schur + s.sch + uniform(f.sch);
  const Global<uint32_t> src = global(s.src) + uniform(f.row0);
  Child<T> kid[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const int i = uniform(f.child[c]);
    const Front q = s.fronts[max(i, 0)];
    kid[c] = Child<T>{schur + s.sch + uniform(q.sch), i >= 0 ? uniform(q.m) : 0, uniform(q.u)};
  }
  const bool grown = kid[0].m > 0 || kid[1].m > 0;
  if (t < KB) {
    const uint32_t x = t < k ? src[t] : 0u;
#pragma unroll
    for (int c = 0; c < 2; c++) mc[c][t] = t < k && kid[c].m > 0 ? kid[c].row(x, c, n) : -1;
  }
  if (k > 0) {
    // pivot block: the lower entries of the matrix, the children's, ones on
    // the diagonal past the last column.  Every thread's loads are issued
    // before the first is used.
    constexpr int PER = KB * KB / (64 * NW) > 0 ? KB * KB / (64 * NW) : 1;
    if (grown) __syncthreads();
    T v[PER], u[2][PER];
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int e = t + 64 * NW * q, r = e / KB, c = e % KB;
      v[q] = pan[(uint32_t)(r < k && c <= r ? panel_elem<T>(H, r, c) : 0)];
    }
#pragma unroll
    for (int x = 0; x < 2; x++) {
      if (kid[x].m > 0) {
#pragma unroll
        for (int q = 0; q < PER; q++) {
          const int e = t + 64 * NW * q, r = e / KB, c = e % KB;
          u[x][q] = kid[x].read(c <= r ? mc[x][min(r, KB - 1)] : -1, mc[x][c]);
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
          const int e = t + 64 * NW * q, r = e / KB, c = e % KB;
          u[x][q] = kept(u[x][q], c <= r ? mc[x][min(r, KB - 1)] : -1, mc[x][c]);
        }
      } else {
#pragma unroll
        for (int q = 0; q < PER; q++) u[x][q] = (T)0;
      }
    }
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int e = t + 64 * NW * q, r = e / KB, c = e % KB;
      const T x = r < k && c <= r ? v[q] : r == c ? (T)1 : (T)0;
      if (r < KB) {
        As[r * LDX + c] = x + (u[0][q] + u[1][q]);
        Bs[r * LDX + c] = (T)0;
      }
    }
    __syncthreads();
    // halves of 32 columns; in between, the second half's block minus
    // L_21 L_21^T with L_21 = A_21 D_1^T, and last D_21 = -D_2 (L_21 D_1), one
    // 16x16 block of them per wavefront
    const int I = (w >> 1) & 1, J = w & 1;
    auto block = [&](const T* X, const T* Y, bool yt) {  // 16x16 block (I, J) of a 32x32 product
      V a = V{0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 8; q++)
        a = Mma<T>::op(X[(16 * I + li) * LDX + 4 * q + lk],
                       yt ? Y[(16 * J + li) * LDX + 4 * q + lk] : Y[(4 * q + lk) * LDX + 16 * J + li], a);
      return a;
    };
#pragma unroll 1
    for (int b = 0; b < (NB == 4 ? 2 : 1); b++) {
      const int o = 32 * b;
      if (w == 0)
        wave_factor_invert<T, LDX>(As + o * LDX + o, Bs + o * LDX + o, min(k - o, 32), lane, (int)blockIdx.x + 1,
                                   flag);
      if (NB == 2 || b == 1) break;
      __syncthreads();
      T* A21 = As + 32 * LDX;
      V a = block(A21, Bs, true);
      __syncthreads();
      if (w < 4)
#pragma unroll
        for (int q = 0; q < 4; q++) A21[(16 * I + Mma<T>::row(lane, q)) * LDX + 16 * J + li] = a[q];
      __syncthreads();
      a = block(A21, A21, true);
      if (w < 4)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          T* e = A21 + 32 + (16 * I + Mma<T>::row(lane, q)) * LDX + 16 * J + li;
          *e = *e - a[q];
        }
      __syncthreads();
    }
    __syncthreads();
    if (NB == 4) {
      V a = block(As + 32 * LDX, Bs, false);  // L_21 D_1
      __syncthreads();
      if (w < 4)
#pragma unroll
        for (int q = 0; q < 4; q++) As[(32 + 16 * I + Mma<T>::row(lane, q)) * LDX + 16 * J + li] = a[q];
      __syncthreads();
      a = block(Bs + 32 * LDX + 32, As + 32 * LDX, false);
      if (w < 4)
#pragma unroll
        for (int q = 0; q < 4; q++) Bs[(32 + 16 * I + Mma<T>::row(lane, q)) * LDX + 16 * J + li] = -a[q];
      __syncthreads();
    }
    // D over the pivot block
    for (int e = t; e < k * 4 * ng; e += 64 * NW) {
      const int r = (e >> 2) % k, c = 4 * ((e >> 2) / k) + (e & 3);
      if (c < 4 * ((r >> 2) + 1)) pan[panel_elem<T>(H, r, c)] = c <= r ? Bs[r * LDX + c] : (T)0;
    }
  }
  if (m == 0) return;
  if (k == 0) __syncthreads();
  // L_RS, 16 rows per wavefront at a time (columns past the last one meet
  // zeros of D)
  if (k > 0)
    for (int r0 = 16 * w; r0 < m; r0 += 16 * NW) {
      const int row = min(k + r0 + li, H - 1);
      const uint32_t x = src[(uint32_t)row];
      V acc[NB];
#pragma unroll
      for (int q = 0; q < NB; q++) acc[q] = V{0, 0, 0, 0};
#pragma unroll
      for (int q0 = 0; q0 < NG; q0 += 8)
        if (q0 < ng) {
          T a[8], b[2][8];
#pragma unroll
          for (int q = 0; q < 8; q++) a[q] = pan[(uint32_t)panel_elem<T>(H, row, 4 * min(q0 + q, ng - 1) + lk)];
#pragma unroll
          for (int c = 0; c < 2; c++)
            if (kid[c].m > 0) {
              const int i = kid[c].row(x, c, n);
              int j[8];
#pragma unroll
              for (int q = 0; q < 8; q++) j[q] = mc[c][4 * (q0 + q) + lk];
#pragma unroll
              for (int q = 0; q < 8; q++) b[c][q] = kid[c].read(i, j[q]);
#pragma unroll
              for (int q = 0; q < 8; q++) b[c][q] = kept(b[c][q], i, j[q]);
            } else {
#pragma unroll
              for (int q = 0; q < 8; q++) b[c][q] = (T)0;
            }
#pragma unroll
          for (int q = 0; q < 8; q++) {
            const T e = a[q] + (b[0][q] + b[1][q]);
#pragma unroll
            for (int c = 0; c < NB; c++)
              if (4 * (q0 + q) < 16 * (c + 1))  // D is lower triangular
                acc[c] = Mma<T>::op(e, Bs[(16 * c + li) * LDX + 4 * (q0 + q) + lk], acc[c]);
          }
        }
#pragma unroll
      for (int c = 0; c < NB; c++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int ro = k + r0 + Mma<T>::row(lane, q), co = 16 * c + li;
          if (ro < H && co < 4 * ng) pan[(uint32_t)panel_elem<T>(H, ro, co)] = acc[c][q];
        }
    }
  __syncthreads();
  // update matrix, 32x32 tiles of its lower part
  const int nt = (m + 31) >> 5;
  for (int e = w; e < nt * (nt + 1) / 2; e += NW) {
    int I = (int)((sqrtf(8.0f * e + 1.0f) - 1.0f) * 0.5f);
    while ((I + 1) * (I + 2) / 2 <= e) I++;
    while (I * (I + 1) / 2 > e) I--;
    const int J = e - I * (I + 1) / 2;
    V acc[2][2];
    zero_acc(acc);
    uint32_t xc[2], xr[2][4];
#pragma unroll
    for (int y = 0; y < 2; y++) xc[y] = src[(uint32_t)min(k + 32 * J + 16 * y + li, H - 1)];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int q = 0; q < 4; q++) xr[x][q] = src[(uint32_t)min(k + 32 * I + 16 * x + Mma<T>::row(lane, q), H - 1)];
#pragma unroll
    for (int q0 = 0; q0 < NG; q0 += 8)
      if (q0 < ng) {
        T a[2][8], b[2][8];
#pragma unroll
        for (int x = 0; x < 2; x++) {
          const int ra = min(k + 32 * I + 16 * x + li, H - 1), rb = min(k + 32 * J + 16 * x + li, H - 1);
#pragma unroll
          for (int q = 0; q < 8; q++) {
            const int c = 4 * min(q0 + q, ng - 1) + lk;
            a[x][q] = pan[(uint32_t)panel_elem<T>(H, ra, c)];
            b[x][q] = pan[(uint32_t)panel_elem<T>(H, rb, c)];
          }
        }
#pragma unroll
        for (int q = 0; q < 8; q++) {
          const T a0 = q0 + q < ng ? a[0][q] : (T)0, a1 = q0 + q < ng ? a[1][q] : (T)0;
          acc[0][0] = Mma<T>::op(a0, b[0][q], acc[0][0]);
          acc[0][1] = Mma<T>::op(a0, b[1][q], acc[0][1]);
          acc[1][0] = Mma<T>::op(a1, b[0][q], acc[1][0]);
          acc[1][1] = Mma<T>::op(a1, b[1][q], acc[1][1]);
        }
      }
#pragma unroll
    for (int x = 0; x < 2; x++) {
      T v[2][2][4];
#pragma unroll
      for (int c = 0; c < 2; c++)
        if (kid[c].m > 0) {
          int i[4], j[2];
#pragma unroll
          for (int q = 0; q < 4; q++) i[q] = kid[c].row(xr[x][q], c, n);
#pragma unroll
          for (int y = 0; y < 2; y++) j[y] = kid[c].row(xc[y], c, n);
#pragma unroll
          for (int y = 0; y < 2; y++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[c][y][q] = kid[c].read(j[y] <= i[q] ? i[q] : -1, j[y]);
#pragma unroll
          for (int y = 0; y < 2; y++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[c][y][q] = kept(v[c][y][q], i[q], j[y]);
        } else {
#pragma unroll
          for (int y = 0; y < 2; y++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[c][y][q] = (T)0;
        }
#pragma unroll
      for (int y = 0; y < 2; y++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int row = 32 * I + 16 * x + Mma<T>::row(lane, q), col = 32 * J + 16 * y + li;
          if (row < m && col <= row) S[(uint32_t)(row * m + col)] = (v[0][y][q] + v[1][y][q]) - acc[x][y][q];
        }
    }
  }
  if (k == 0) return;
  __syncthreads();
  // C = L_RS D over L_RS
  for (int r0 = 16 * w; r0 < m; r0 += 16 * NW) {
    const int row = min(k + r0 + li, H - 1);
    T a[NG];
#pragma unroll
    for (int q = 0; q < NG; q++) a[q] = pan[(uint32_t)panel_elem<T>(H, row, 4 * min(q, ng - 1) + lk)];
    V acc[NB];
#pragma unroll
    for (int c = 0; c < NB; c++) acc[c] = V{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < NG; q++)
#pragma unroll
      for (int c = 0; c < NB; c++)
        if (4 * q + 3 >= 16 * c) acc[c] = Mma<T>::op(a[q], Bs[(4 * q + lk) * LDX + 16 * c + li], acc[c]);
#pragma unroll
    for (int c = 0; c < NB; c++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int ro = k + r0 + Mma<T>::row(lane, q), co = 16 * c + li;
        if (ro < H && co < 4 * ng) pan[(uint32_t)panel_elem<T>(H, ro, co)] = acc[c][q];
      }
  }
}

// ------------------------------------------------------------------------
// solve, one right-hand side
// ------------------------------------------------------------------------

// A lane's 32-bit value as another lane of its row of 16 sees it (DPP).
template <int CTRL>
__device__ __forceinline__ float lane_swap(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double lane_swap(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E;        // quad_perm
constexpr int kDppXor8 = 0x128, kDppXor7 = 0x141;      // row_ror:8, row_half_mirror
constexpr int kDppRor4 = 0x124;                        // row_ror:4

// a + b after half the lanes have exchanged them: lanes of the lower half
// (of each 64, or of each 32) return a's sum over the two halves, the others b's.
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int CTRL>
__device__ __forceinline__ float fold_row(float a, float b, bool hi) {
  const float keep = hi ? b : a, send = hi ? a : b;
  return keep + lane_swap<CTRL>(send);
}

// v[0..31] summed over the 64 lanes: lane l returns the sum of entry l / 2.
// Each halving hands one half of the entries to the other half of the lanes;
// all exchanges are register-to-register.
__device__ __forceinline__ float reduce_scatter(float (&v)[32], int lane) {
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = fold32(v[q], v[q + 16]);
#pragma unroll
  for (int q = 0; q < 8; q++) v[q] = fold16(v[q], v[q + 8]);
#pragma unroll
  for (int q = 0; q < 4; q++) v[q] = fold_row<kDppXor8>(v[q], v[q + 4], lane & 8);
#pragma unroll
  for (int q = 0; q < 2; q++) v[q] = fold_row<kDppXor7>(v[q], v[q + 2], lane & 4);
  v[0] = fold_row<kDppXor2>(v[0], v[1], lane & 2);
  return v[0] + lane_swap<kDppXor1>(v[0]);
}

// Workgroup barrier that orders LDS alone: loads of panels already issued for
// the units behind it stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The work lists are read through the constant address space: the barriers'
// fences would otherwise send these uniform loads down the vector path.
typedef const FrontUnit __attribute__((address_space(4))) * UnitPtr;
__device__ __forceinline__ UnitPtr unit_list(const FrontUnit* p) {
  return reinterpret_cast<UnitPtr>(reinterpret_cast<uint64_t>(p));
}
__device__ __forceinline__ int list_at(const int32_t* p, int i) {
  typedef const int32_t __attribute__((address_space(4))) * P;
  return __builtin_amdgcn_readfirstlane(reinterpret_cast<P>(reinterpret_cast<uint64_t>(p))[i]);
}
__device__ __forceinline__ FrontUnit unit_at(UnitPtr p) {
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  typedef const v4 __attribute__((address_space(4))) * P4;
  const P4 q = (P4)p;
  const v4 a = q[0], b = q[1];
  FrontUnit u;
  u.pan = (int32_t)a[0];
  u.row0 = (int32_t)a[1];
  u.h = (uint16_t)a[2];
  u.k = (uint16_t)(a[2] >> 16);
  u.c0 = (uint16_t)a[3];
  u.u = (uint16_t)(a[3] >> 16);
  u.g0 = (uint8_t)b[0];
  u.g1 = (uint8_t)(b[0] >> 8);
  u.chunk = (uint8_t)(b[0] >> 16);
  u.flags = (uint8_t)(b[0] >> 24);
  u.nbar = (uint16_t)b[1];
  return u;
}

// The four entries of column group g in one row: the panel is streamed once
// per pass, so its loads are non-temporal.
typedef float F4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ F4 load_quad(const float* pan, int H, int g, int row) {
  // 32-bit offsets from a uniform base keep the addresses in one register
  const uint32_t o = 16u * (uint32_t)(row + g * (H - 2 * g - 2));
  return __builtin_nontemporal_load(reinterpret_cast<const F4*>(reinterpret_cast<const char*>(pan) + o));
}

// The loads of one unit: its panel rows, the row records of its rows (lane =
// row) and, forward, those of the front's columns (lane = column).  Always
// the same number of loads (a group or row past the end repeats the last
// one), so that the next unit's stay in flight while this one is used.
struct UnitLoad {
  F4 v[kFrontUnitGroups32];
  uint32_t r, c;
};
__device__ __forceinline__ void load_panel(UnitLoad& b, const float* pan, const FrontUnit& d, int rc) {
#pragma unroll
  for (int q = 0; q < kFrontUnitGroups32; q++) {
    const int g = min(d.g0 + q, d.g1 - 1);
    b.v[q] = load_quad(pan, d.h, g, max(rc, 4 * g));
  }
}

// Forward and backward substitution for one subdomain per workgroup, in FP32;
// the right-hand side is gathered from (and the solution written to) FP64
// vectors.  The work vector (positions, then update vectors
// or the top fronts' solution) lives in LDS.  Nothing when *skip is set.
// Forward: one front's panel times its right-hand side, a lane per row, the
// columns' values broadcast from the lanes that gathered them.  Backward: the
// panel's transpose times [y; -x], a lane per row, the columns' sums reduced
// over the lanes at the end.
// Each pass streams the panels once, which bounds it where there are hundreds
// of subdomains (512 of 5440 unknowns: 2.2 GB in 493 us, 4.5 TB/s; envelopes,
// 6 GB in 879 us).  Hence the unit lists: a wavefront's next panel rows are
// always on their way, across barriers too, and the leaves' subtrees run side
// by side without any.
//
// Where subdomains are at most half as many as the CUs, two, four or eight
// workgroups share one, each with subtrees of its own: stage 1 takes these
// forward, stage 2 the few fronts above them in both directions and stage 3
// the subtrees backward; y and the updates in between go through global
// memory (as doubles, unrounded).  Stage 0 is all of it in one workgroup.
// 64 subdomains of 5250 unknowns: 181 us (248 us in one workgroup each); of
// 4300 in two dimensions 75 us (103); 4 of 4224: 57 us (95).
// The matrix-core form below has been measured in FP64 only, where it gave 3 to
// 9 %.  Here another order of the sums also moves the iteration counts of some
// systems by one (8 of 384 inputs between fronts and envelopes).
enum { kWhole = 0, kSubtreesForward = 1, kApex = 2, kSubtreesBackward = 3 };
template <int NW, int STAGE>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_front_solve(
    const float* __restrict__ tiles, const FrontSub* __restrict__ subs, int groups,
    const int32_t* __restrict__ inds, const double* __restrict__ rhs, double* updates, double* sol,
    const double* skip) {
  if (skip && *skip != 0.0) return;
  typedef float T;
  constexpr int UG = kFrontUnitGroups32;
  extern __shared__ __align__(16) unsigned char front_dyn[];
  T* L = reinterpret_cast<T*>(front_dyn);
  constexpr bool kGroup = STAGE == kSubtreesForward || STAGE == kSubtreesBackward;
  const int grp = kGroup ? (int)blockIdx.x % groups : 0;
  const FrontSub s = subs[kGroup ? (int)blockIdx.x / groups : (int)blockIdx.x];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const T* base = tiles + s.base;
  const int n = s.n, top0 = s.top0;
  if (n == 0) return;
  const Global<uint32_t> src = global(s.src);
  const Global<uint16_t> rpos = global(s.rpos);
  T* X = L + n - top0;  // solution at the positions from top0 on
  // this workgroup's positions: [p0, p1), and its subtrees' top fronts [p2, p3)
  const int apex0 = STAGE == kWhole ? n : list_at(s.gtop, groups);
  const int p0 = kGroup ? list_at(s.gpos, grp) : STAGE == kApex ? apex0 : 0;
  const int p1 = kGroup ? list_at(s.gpos, grp + 1) : n;
  const int p2 = kGroup ? list_at(s.gtop, grp) : n, p3 = kGroup ? list_at(s.gtop, grp + 1) : n;
  auto own = [&](auto&& f) {
    for (int p = p0 + t; p < p1; p += 64 * NW) f(p);
    for (int p = p2 + t; p < p3; p += 64 * NW) f(p);
  };
  if (STAGE == kSubtreesBackward) {
    own([&](int p) { L[p] = (T)sol[s.vec + p]; });
    for (int p = apex0 + t; p < n; p += 64 * NW) X[p] = (T)sol[s.vec + p];
  } else {
    own([&](int p) { L[p] = (T)rhs[inds[s.vec + p]]; });
    if (t == 0) L[n] = (T)0;
  }
  if (STAGE == kApex)
    for (int q = t; q < list_at(s.uoff, groups); q += 64 * NW) L[s.uidx[q]] = (T)updates[s.ub + q];
  lds_barrier();
  if constexpr (STAGE != kSubtreesBackward) {
    const UnitPtr units = unit_list(STAGE == kSubtreesForward ? s.bunits_f : s.units_f);
    const int32_t* list = STAGE == kSubtreesForward ? s.blist_f + NW * grp : s.list_f;
    int u0 = list_at(list, w);
    const int last = list_at(list, w + 1) - 1;
    T fv = (T)0, a[4] = {(T)0, (T)0, (T)0, (T)0};
    // y of a front that several wavefronts share: its right-hand side is
    // still read by the others, so it is written behind the next barrier
    T pend = (T)0;
    int pend_at = -1;
    auto load = [&](UnitLoad& b, const FrontUnit& d) {
      const int rc = min(64 * d.chunk + lane, d.h - 1);
      b.c = src[(uint32_t)(d.row0 + min(lane, d.h - 1))];
      b.r = src[(uint32_t)(d.row0 + rc)];
      load_panel(b, base + d.pan, d, rc);
    };
    auto work = [&](const UnitLoad& b, const FrontUnit& d) {
      {
        const int row = 64 * d.chunk + lane, k = d.k;
        if (d.flags & FU_FIRST) {
          fv = (T)0;
          if (lane < k) fv = L[d.c0 + lane] + (L[b.c & 0xffffu] + L[b.c >> 16]);
        }
        if (d.flags & FU_BEGIN) a[0] = a[1] = a[2] = a[3] = (T)0;
#pragma unroll
        for (int q = 0; q < UG; q++) {
          const bool in = row >= 4 * (d.g0 + q);  // right of the diagonal there is nothing
#pragma unroll
          for (int j = 0; j < 4; j++)
            a[j] = __builtin_fmaf(in ? b.v[q][j] : (T)0, lane_value(fv, 4 * (d.g0 + q) + j), a[j]);
        }
        if (d.flags & FU_END) {
          const T r = (a[0] + a[1]) + (a[2] + a[3]);
          if (row < k) {
            if (d.flags & FU_WHOLE) {
              L[d.c0 + row] = r;
            } else {
              pend = r;
              pend_at = d.c0 + row;
            }
          } else if (row < d.h) {
            L[d.u + row - k] = (L[b.r & 0xffffu] + L[b.r >> 16]) - r;
          }
          wave_lds_sync();
        }
      }
      for (int q = 0; q < d.nbar; q++) {
        lds_barrier();
        if (pend_at >= 0) L[pend_at] = pend;
        pend_at = -1;
      }
    };
    UnitLoad b0, b1;
    FrontUnit d0{};
    if (u0 < last) {  // a subdomain may have no fronts above its subtrees
      d0 = unit_at(units + u0);
      load(b0, d0);
    }
    for (; u0 < last; u0 += 2) {  // two units a turn: lists have even lengths
      const FrontUnit d1 = unit_at(units + u0 + 1);
      load(b1, d1);
      work(b0, d0);
      d0 = unit_at(units + min(u0 + 2, last));
      load(b0, d0);
      work(b1, d1);
    }
  }
  if (STAGE == kSubtreesForward) {
    lds_barrier();
    own([&](int p) { sol[s.vec + p] = (double)L[p]; });
    for (int q = list_at(s.uoff, grp) + t; q < list_at(s.uoff, grp + 1); q += 64 * NW)
      updates[s.ub + q] = (double)L[s.uidx[q]];
    return;
  }
  if (STAGE != kSubtreesBackward) lds_barrier();
  if constexpr (STAGE != kSubtreesForward) {
    const UnitPtr units = unit_list(STAGE == kSubtreesBackward ? s.bunits_b : s.units_b);
    const int32_t* list = STAGE == kSubtreesBackward ? s.blist_b + NW * grp : s.list_b;
    int u0 = list_at(list, w);
    const int last = list_at(list, w + 1) - 1;
    T y0 = (T)0, acc[4 * UG];
#pragma unroll
    for (int q = 0; q < 4 * UG; q++) acc[q] = (T)0;
    auto load = [&](UnitLoad& b, const FrontUnit& d) {
      const int rc = min(64 * d.chunk + lane, d.h - 1);
      b.r = rpos[(uint32_t)(d.row0 + rc)];
      load_panel(b, base + d.pan, d, rc);
    };
    auto work = [&](const UnitLoad& b, const FrontUnit& d) {
      {
        const int row = 64 * d.chunk + lane, k = d.k;
        T x = y0;
        if (d.chunk != 0 || (d.flags & FU_FIRST)) {
          const int p = (int)b.r;
          x = L[row >= k && p >= top0 ? n + p - top0 : p];
          x = row < k ? x : row < d.h ? -x : (T)0;
          if (d.chunk == 0) y0 = x;  // holds every y of the front (k <= 64)
        }
        if (d.flags & FU_BEGIN) {
#pragma unroll
          for (int q = 0; q < 4 * UG; q++) acc[q] = (T)0;
        }
#pragma unroll
        for (int q = 0; q < UG; q++) {
          const T xq = row >= 4 * (d.g0 + q) ? x : (T)0;
#pragma unroll
          for (int j = 0; j < 4; j++) acc[4 * q + j] = __builtin_fmaf(b.v[q][j], xq, acc[4 * q + j]);
        }
        if (d.flags & FU_END) {
          const T r = reduce_scatter(acc, lane);
          constexpr int per = 64 / (4 * UG);
          const int col = 4 * d.g0 + lane / per;
          if (lane % per == 0 && col < k && col < 4 * d.g1) (d.c0 < top0 ? L : X)[d.c0 + col] = r;
          wave_lds_sync();
        }
      }
      for (int q = 0; q < d.nbar; q++) lds_barrier();
    };
    UnitLoad b0, b1;
    FrontUnit d0{};
    if (u0 < last) {  // a subdomain may have no fronts above its subtrees
      d0 = unit_at(units + u0);
      load(b0, d0);
    }
    for (; u0 < last; u0 += 2) {  // two units a turn: lists have even lengths
      const FrontUnit d1 = unit_at(units + u0 + 1);
      load(b1, d1);
      work(b0, d0);
      d0 = unit_at(units + min(u0 + 2, last));
      load(b0, d0);
      work(b1, d1);
    }
  }
  lds_barrier();
  own([&](int p) { sol[s.vec + p] = (double)(p < top0 ? L[p] : X[p]); });
}

// ---- FP64: the same on the matrix cores ----
//
// v_mfma_f64_4x4x4 takes A[i][k] of block b from lane i + 4 b + 16 k, B[k][j]
// from lane j + 4 b + 16 k, and holds D[i][j] in lane j + 4 b + 16 i.  One
// column of B is enough here; all four are the same.
__device__ __forceinline__ double mma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ double pick4(const double (&v)[4], int i) {
  const double a = (i & 1) ? v[1] : v[0], b = (i & 1) ? v[3] : v[2];
  return (i & 2) ? b : a;
}

// A unit's descriptor on its way through the vector path: fetched ahead of the
// loads that the units before it issue, it is there when they still are not.
struct RawUnit {
  uint32_t a __attribute__((ext_vector_type(4)));
  uint32_t b __attribute__((ext_vector_type(2)));
};
__device__ __forceinline__ RawUnit raw_unit(const FrontUnit* p, int i) {
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  typedef uint32_t v2 __attribute__((ext_vector_type(2)));
  const Global<v4> q = global(reinterpret_cast<const v4*>(p));
  RawUnit r;
  r.a = q[(uint32_t)(2 * i)];
  r.b = *(const v2 __attribute__((address_space(1)))*)(q + (uint32_t)(2 * i + 1));
  return r;
}
__device__ __forceinline__ FrontUnit unit_of(const RawUnit& r) {
  const uint32_t a2 = uniform(r.a[2]), a3 = uniform(r.a[3]), b0 = uniform(r.b[0]);
  FrontUnit u;
  u.pan = uniform(r.a[0]);
  u.row0 = uniform(r.a[1]);
  u.h = (uint16_t)a2;
  u.k = (uint16_t)(a2 >> 16);
  u.c0 = (uint16_t)a3;
  u.u = (uint16_t)(a3 >> 16);
  u.g0 = (uint8_t)b0;
  u.g1 = (uint8_t)(b0 >> 8);
  u.chunk = (uint8_t)(b0 >> 16);
  u.flags = (uint8_t)(b0 >> 24);
  u.nbar = (uint16_t)uniform(r.b[1]);
  return u;
}

// The units of one wavefront, two a turn (lists have even lengths): the loads
// of the unit after next are issued as soon as a unit's registers are free,
// before its barriers.
template <typename Load, typename F, typename G, typename H>
__device__ __forceinline__ void walk_units(const FrontUnit* units, int u, int end, F&& load, G&& work, H&& barriers) {
  if (u >= end) return;
  Load q0, q1;
  RawUnit r0 = raw_unit(units, u), r1 = raw_unit(units, u + 1);
  FrontUnit d0 = unit_of(r0), d1 = unit_of(r1);
  r0 = raw_unit(units, min(u + 2, end - 1));
  load(q0, d0);
  __builtin_amdgcn_sched_barrier(0);
  r1 = raw_unit(units, min(u + 3, end - 1));
  load(q1, d1);
  __builtin_amdgcn_sched_barrier(0);
  for (; u < end; u += 2) {
    work(q0, d0);
    int n = d0.nbar;
    d0 = unit_of(r0);
    r0 = raw_unit(units, min(u + 4, end - 1));
    load(q0, d0);
    __builtin_amdgcn_sched_barrier(0);
    barriers(n);
    work(q1, d1);
    n = d1.nbar;
    d1 = unit_of(r1);
    r1 = raw_unit(units, min(u + 5, end - 1));
    load(q1, d1);
    __builtin_amdgcn_sched_barrier(0);
    barriers(n);
  }
}

// Byte offset in an FP64 panel of H rows of the columns 4 g + 2 j, 4 g + 2 j + 1
// of a row.
__device__ __forceinline__ uint32_t panel_offset(int H, int g, int j, int row) {
  return 16u * (uint32_t)(2 * g * H - 4 * g * (g - 1) + row - 4 * g + (j ? H - 4 * g : 0));
}
typedef double Two __attribute__((ext_vector_type(2)));
// Buffer loads of a panel: an offset past its end gives zeros and loads nothing.
typedef uint32_t U4 __attribute__((ext_vector_type(4)));
constexpr uint32_t kNothing = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t panel_buffer(const double* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, bytes, 0x00027000);
}
__device__ __forceinline__ Two panel_load(__amdgpu_buffer_rsrc_t b, uint32_t offset) {
  const U4 v = __builtin_amdgcn_raw_buffer_load_b128(b, (int)offset, 0, 0);
  return __builtin_bit_cast(Two, v);
}

// Bytes of a panel's first g1 column groups.
__device__ __forceinline__ int panel_bytes(int H, int g1) { return 32 * (g1 * H - 2 * g1 * (g1 - 1)); }

// A product step takes 16 rows of four columns, so that a unit of 64 rows and
// 16 columns is 16 of them, with neither broadcasts (forward) nor sums over
// lanes (backward): in the vector form above these cost more than the
// products.  A 16-byte load gives a lane two columns of a row, one for each of
// two steps: forward of row l % 16 the pair l / 16 of eight columns, backward
// of row 4 (l / 4 % 4) + l / 16 the pair l % 4.  The operands that all rows
// (columns) share go through 64 entries of LDS per wavefront behind the work
// vector.  Lanes outside the front, or right of its diagonal, load nothing and
// get zeros: what bounds the kernel where subdomains are few is the 64 bytes a
// cycle that a CU loads, and half of a unit is such lanes on average.
// 512 subdomains of 5440 unknowns: 803 us, 5.6 TB/s, bound by HBM (the vector
// form 804, envelopes 1735); 343 of 4600: 395 us (414, 950).
//
// The stages are those of the vector form.  64 subdomains of 4300
// unknowns in two dimensions: 35 + 38 + 34 us (171 us in one workgroup each,
// the vector form 188, envelopes 709); 4 of 4224: 15 + 30 + 17 us (110, 113,
// 302).
template <int NW, int STAGE>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_front_solve_mma(
    const double* __restrict__ tiles, const FrontSub* __restrict__ subs, int groups, int maxwork,
    const int32_t* __restrict__ inds, const double* __restrict__ rhs, double* updates, double* sol,
    const double* skip) {
  if (skip && *skip != 0.0) return;
  constexpr int UG = kFrontUnitGroups64;
  extern __shared__ __align__(16) unsigned char front_dyn[];
  double* L = reinterpret_cast<double*>(front_dyn);
  constexpr bool kGroup = STAGE == kSubtreesForward || STAGE == kSubtreesBackward;
  const int grp = kGroup ? (int)blockIdx.x % groups : 0;
  const FrontSub s = subs[kGroup ? (int)blockIdx.x / groups : (int)blockIdx.x];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lo = lane & 3, mid = (lane >> 2) & 3, hi = lane >> 4;
  double* stage = L + maxwork + 64 * w;  // maxwork is even: 16-byte pieces
  const double* base = tiles + s.base;
  const int n = s.n, top0 = s.top0;
  if (n == 0) return;
  const Global<uint32_t> src = global(s.src);
  const Global<uint16_t> rpos = global(s.rpos);
  double* X = L + n - top0;  // solution at the positions from top0 on
  // this workgroup's positions: [p0, p1), and its subtrees' top fronts [p2, p3)
  const int apex0 = STAGE == kWhole ? n : list_at(s.gtop, groups);
  const int p0 = kGroup ? list_at(s.gpos, grp) : STAGE == kApex ? apex0 : 0;
  const int p1 = kGroup ? list_at(s.gpos, grp + 1) : n;
  const int p2 = kGroup ? list_at(s.gtop, grp) : n, p3 = kGroup ? list_at(s.gtop, grp + 1) : n;
  auto own = [&](auto&& f) {
    for (int p = p0 + t; p < p1; p += 64 * NW) f(p);
    for (int p = p2 + t; p < p3; p += 64 * NW) f(p);
  };
  if (STAGE == kSubtreesBackward) {
    own([&](int p) { L[p] = sol[s.vec + p]; });
    for (int p = apex0 + t; p < n; p += 64 * NW) X[p] = sol[s.vec + p];
  } else {
    own([&](int p) { L[p] = rhs[inds[s.vec + p]]; });
    if (t == 0) L[n] = 0.0;
  }
  if (STAGE == kApex)
    for (int q = t; q < list_at(s.uoff, groups); q += 64 * NW) L[s.uidx[q]] = updates[s.ub + q];
  lds_barrier();
  struct Load {
    Two a[UG / 2][4];
    uint32_t r, c;
  };
  if constexpr (STAGE != kSubtreesBackward) {
    // y of a front that several wavefronts share: its right-hand side is
    // still read by the others, so it is written behind the next barrier
    double acc[4] = {0.0, 0.0, 0.0, 0.0}, pend = 0.0;
    int pend_at = -1;
    const int mine = 16 * lo + 4 * mid + hi;  // the row of a chunk whose sum this lane ends with
    auto load = [&](Load& q, const FrontUnit& d) {
      const auto pan = panel_buffer(base + d.pan, panel_bytes(d.h, d.g1));
#pragma unroll
      for (int x = 0; x < UG / 2; x++) {
        const int g = d.g0 + 2 * x + (hi >> 1), row = 64 * d.chunk + (lane & 15);
        const uint32_t o = panel_offset(d.h, g, hi & 1, row);
        const int first = g < d.g1 ? 4 * g : d.h;
#pragma unroll
        for (int y = 0; y < 4; y++)
          q.a[x][y] = panel_load(pan, row + 16 * y >= first && row + 16 * y < d.h ? o + 256u * y : kNothing);
      }
      q.c = src[(uint32_t)(d.row0 + min(lane, d.h - 1))];
      q.r = src[(uint32_t)(d.row0 + min(64 * d.chunk + mine, d.h - 1))];
    };
    auto work = [&](const Load& q, const FrontUnit& d) {
      const int k = d.k;
      if (d.flags & FU_FIRST) {
        double f = 0.0;
        if (lane < k) f = L[d.c0 + lane] + (L[q.c & 0xffffu] + L[q.c >> 16]);
        stage[lane] = f;
        wave_lds_sync();
      }
      if (d.flags & FU_BEGIN) acc[0] = acc[1] = acc[2] = acc[3] = 0.0;
      const int left = d.h - 64 * d.chunk;
#pragma unroll
      for (int x = 0; x < UG / 2; x++)
        if (x == 0 || d.g0 + 2 * x < d.g1) {
          const int g = d.g0 + 2 * x + (hi >> 1);  // past g1 there are zeros in `stage`
          const Two f = *reinterpret_cast<const Two*>(stage + 4 * g + 2 * (hi & 1));
#pragma unroll
          for (int y = 0; y < 4; y++)
            if (y == 0 || 16 * y < left) {
              const Two a = q.a[x][y];
              acc[y] = mma4(a[0], f[0], acc[y]);
              acc[y] = mma4(a[1], f[1], acc[y]);
            }
        }
      if (d.flags & FU_END) {
        const int row = 64 * d.chunk + mine;
        const double r = pick4(acc, lo);
        if (row < k) {
          if (d.flags & FU_WHOLE) {
            L[d.c0 + row] = r;
          } else {
            pend = r;
            pend_at = d.c0 + row;
          }
        } else if (row < d.h) {
          L[d.u + row - k] = (L[q.r & 0xffffu] + L[q.r >> 16]) - r;
        }
        wave_lds_sync();
      }
    };
    auto barriers = [&](int count) {
      for (int i = 0; i < count; i++) {
        lds_barrier();
        if (pend_at >= 0) L[pend_at] = pend;
        pend_at = -1;
      }
    };
    const int32_t* list = STAGE == kSubtreesForward ? s.blist_f + NW * grp : s.list_f;
    walk_units<Load>(STAGE == kSubtreesForward ? s.bunits_f : s.units_f, list_at(list, w), list_at(list, w + 1), load,
                     work, barriers);
  }
  if (STAGE == kSubtreesForward) {
    lds_barrier();
    own([&](int p) { sol[s.vec + p] = L[p]; });
    for (int q = list_at(s.uoff, grp) + t; q < list_at(s.uoff, grp + 1); q += 64 * NW) updates[s.ub + q] = L[s.uidx[q]];
    return;
  }
  if (STAGE != kSubtreesBackward) lds_barrier();
  if constexpr (STAGE != kSubtreesForward) {
    double acc[UG] = {0.0, 0.0, 0.0, 0.0}, y0 = 0.0;
    auto load = [&](Load& q, const FrontUnit& d) {
      const auto pan = panel_buffer(base + d.pan, panel_bytes(d.h, d.g1));
#pragma unroll
      for (int x = 0; x < UG / 2; x++) {
        const int g = d.g0 + 2 * x + (lo >> 1), row = 64 * d.chunk + 4 * mid + hi;
        const uint32_t o = panel_offset(d.h, g, lo & 1, row);
        const int first = g < d.g1 ? 4 * g : d.h;
#pragma unroll
        for (int y = 0; y < 4; y++)
          q.a[x][y] = panel_load(pan, row + 16 * y >= first && row + 16 * y < d.h ? o + 256u * y : kNothing);
      }
      q.r = rpos[(uint32_t)(d.row0 + min(64 * d.chunk + lane, d.h - 1))];
    };
    auto work = [&](const Load& q, const FrontUnit& d) {
      const int k = d.k;
      {
        const int row = 64 * d.chunk + lane;
        double x = y0;
        if (d.chunk != 0 || (d.flags & FU_FIRST)) {
          const int p = (int)q.r;
          x = L[row >= k && p >= top0 ? n + p - top0 : p];
          x = row < k ? x : row < d.h ? -x : 0.0;
          if (d.chunk == 0) y0 = x;  // holds every y of the front (k <= 64)
        }
        stage[lane] = x;
        wave_lds_sync();
      }
      if (d.flags & FU_BEGIN) {
#pragma unroll
        for (int x = 0; x < UG; x++) acc[x] = 0.0;
      }
      const int left = d.h - 64 * d.chunk;
#pragma unroll
      for (int y = 0; y < 4; y++)
        if (y == 0 || 16 * y < left) {
          const double v = stage[16 * y + 4 * mid + hi];
#pragma unroll
          for (int x = 0; x < UG / 2; x++) {
            const Two a = q.a[x][y];
            acc[2 * x] = mma4(a[0], v, acc[2 * x]);
            acc[2 * x + 1] = mma4(a[1], v, acc[2 * x + 1]);
          }
        }
      wave_lds_sync();
      if (d.flags & FU_END) {
        double r = pick4(acc, lo);
        r += lane_swap<kDppXor8>(r);
        r += lane_swap<kDppRor4>(r);
        const int col = 4 * d.g0 + 8 * (lo >> 1) + 2 * hi + (lo & 1);
        if (mid == 0 && col < k && col < 4 * d.g1) (d.c0 < top0 ? L : X)[d.c0 + col] = r;
        wave_lds_sync();
      }
    };
    auto barriers = [&](int count) {
      for (int i = 0; i < count; i++) lds_barrier();
    };
    const int32_t* list = STAGE == kSubtreesBackward ? s.blist_b + NW * grp : s.list_b;
    walk_units<Load>(STAGE == kSubtreesBackward ? s.bunits_b : s.units_b, list_at(list, w), list_at(list, w + 1), load,
                     work, barriers);
  }
  lds_barrier();
  own([&](int p) { sol[s.vec + p] = p < top0 ? L[p] : X[p]; });
}

}  // namespace

template <typename T>
void launch_front_scatter(T* tiles, const FrontSub* subs, int nsub, const int32_t* inds, const int32_t* occ_ptr,
                          const int32_t* occ_pos, const int32_t* a_ptr, const int32_t* a_col, const double* a_val,
                          hipStream_t st) {
  if (nsub <= 0) return;
  hipLaunchKernelGGL(k_front_scatter<T>, dim3(nsub, 4), dim3(256), 0, st, tiles, subs, inds, occ_ptr, occ_pos,
                     a_ptr, a_col, a_val);
}

template <typename T>
void launch_front_factor(T* tiles, T* schur, const FrontSub* subs, int nsub, int h, int maxcount, bool wide, int* flag,
                         hipStream_t st) {
  if (nsub <= 0 || maxcount <= 0) return;
  const dim3 g(nsub, maxcount);
  // One wavefront per small front where there are thousands: the pivot block
  // is a chain that only one wavefront works on (512 subdomains of 5440
  // unknowns, FP64: 11.7 ms in all, 13.2 ms with four wavefronts throughout).
  // Sixteen per wide front where there are fewer than the GPU has room for at
  // four (the same, 343 subdomains: 5.9 ms, 6.1 ms without).
  const int64_t fronts = (int64_t)maxcount * nsub;
  if (fronts > 4096)
    hipLaunchKernelGGL((k_front_factor<T, 2, 1>), g, dim3(64), 0, st, tiles, schur, subs, h, flag);
  else
    hipLaunchKernelGGL((k_front_factor<T, 2, 4>), g, dim3(256), 0, st, tiles, schur, subs, h, flag);
  if (wide && fronts > 512)
    hipLaunchKernelGGL((k_front_factor<T, 4, 4>), g, dim3(256), 0, st, tiles, schur, subs, h, flag);
  else if (wide)
    hipLaunchKernelGGL((k_front_factor<T, 4, 16>), g, dim3(1024), 0, st, tiles, schur, subs, h, flag);
}

// LDS of a solve by nw wavefronts
template <typename T>
static int front_solve_lds(int nw, int maxwork) {
  return (maxwork + (sizeof(T) == 8 ? 64 * nw : 0)) * (int)sizeof(T);
}

template <typename T>
hipError_t prepare_front_solve() {
  auto allow = [](auto... kernels) {
    hipError_t first = hipSuccess;
    for (hipError_t e : {allow_lds(kernels, kLdsBytes)...})
      if (first == hipSuccess) first = e;
    return first;
  };
  if constexpr (sizeof(T) == 8)
    return allow(&k_front_solve_mma<8, kWhole>, &k_front_solve_mma<16, kWhole>,
                 &k_front_solve_mma<16, kSubtreesForward>, &k_front_solve_mma<16, kApex>,
                 &k_front_solve_mma<16, kSubtreesBackward>);
  else
    return allow(&k_front_solve<8, kWhole>, &k_front_solve<16, kWhole>, &k_front_solve<16, kSubtreesForward>,
                 &k_front_solve<16, kApex>, &k_front_solve<16, kSubtreesBackward>);
}

template <typename T>
void launch_front_solve(const T* tiles, const FrontSub* subs, int nsub, int nw, int groups, int maxwork,
                        const int32_t* inds, const double* r, double* updates, double* sol, hipStream_t st,
                        const double* skip) {
  if (nsub <= 0) return;
  const size_t lds = (size_t)front_solve_lds<T>(nw, maxwork);
  const dim3 b(64 * nw);
  auto go = [&](auto whole8, auto whole, auto forward, auto apex, auto backward, auto... work) {
    auto one = [&](auto kernel, int blocks) {
      hipLaunchKernelGGL(kernel, dim3(blocks), b, lds, st, tiles, subs, groups, work..., inds, r, updates, sol, skip);
    };
    if (groups > 1) {  // nw is 16
      one(forward, nsub * groups);
      one(apex, nsub);
      one(backward, nsub * groups);
    } else {
      one(nw == 16 ? whole : whole8, nsub);
    }
  };
  if constexpr (sizeof(T) == 8)
    go(&k_front_solve_mma<8, kWhole>, &k_front_solve_mma<16, kWhole>, &k_front_solve_mma<16, kSubtreesForward>,
       &k_front_solve_mma<16, kApex>, &k_front_solve_mma<16, kSubtreesBackward>, maxwork);
  else
    go(&k_front_solve<8, kWhole>, &k_front_solve<16, kWhole>, &k_front_solve<16, kSubtreesForward>,
       &k_front_solve<16, kApex>, &k_front_solve<16, kSubtreesBackward>);
}

#define DOUG_INSTANTIATE_FRONTS(T)                                                                              \
  template void launch_front_scatter<T>(T*, const FrontSub*, int, const int32_t*, const int32_t*,               \
                                        const int32_t*, const int32_t*, const int32_t*, const double*,          \
                                        hipStream_t);                                                           \
  template void launch_front_factor<T>(T*, T*, const FrontSub*, int, int, int, bool, int*, hipStream_t);        \
  template hipError_t prepare_front_solve<T>();                                                                 \
  template void launch_front_solve<T>(const T*, const FrontSub*, int, int, int, int, const int32_t*,            \
                                      const double*, double*, double*, hipStream_t, const double*);
DOUG_INSTANTIATE_FRONTS(double)
DOUG_INSTANTIATE_FRONTS(float)
#undef DOUG_INSTANTIATE_FRONTS

}  // namespace doug
