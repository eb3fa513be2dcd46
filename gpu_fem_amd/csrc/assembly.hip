// MITC4 Jacobian / residual / energy assembly kernels (gfx950).
//
// Replaces add_jacobian_gpu (include/base/elem_group.cuh:101-211), the
// residual path add_residual_cpu (include/base/elem_group.h:40-79) and
// add_energy (assembler.h:198-229).
//
// The default kernels (jacobian_mfma_kernel, tangent_kernel, residual_kernel)
// take four elements a wavefront, see there.  Layout of jacobian_kernel
// (GPUFEM_ASSEMBLY=element): one 64-lane workgroup per element.
//   stage 1  lanes 0-3: node frames; lanes 4-8: tying-point geometry
//   stage 2  lanes 0-3: quadrature frames; lanes 4-8: tying normals
//   stage 3  lanes 0-23: column j of B_q (4 x 9) and D_q = detXd C B_q -> LDS
//   stage 4  all 64 lanes: a 3x3 tile of K_e = sum_q B_q^T D_q (8x8 tiles)
//   stage 5  scatter through elemIndMap (global FP64 atomics), residual
//            R_e = K_e u_e reduced through LDS.
#include <cstdlib>
#include <string>

#include <vector>

#include "common.h"
#include "mitc4.h"
#include "symbolic.h"

struct gf_asm_plan_s {
  gf_context ctx = nullptr;
  int nelems = 0, ncolors = 0;
  std::vector<int> color_ptr;
  int* elems = nullptr;  // elements in colour-major order (device)
  int* mask = nullptr;   // first-touch masks in the same order (device)
  bool zero_k = false, zero_res = false;  // untouched K blocks / rows exist
  int nnzb = 0, nnodes = 0;
};

namespace gf {
namespace {

struct ElemLDS {
  double X[12];
  double u[24];
  double data[4];
  mitc4::Geom g;
  double B[4][9][24];
  double D[4][9][24];
  double rpart[8][24];  // residual partial sums per tile column J
};

__device__ __forceinline__ void load_element(ElemLDS& s, int e, int lane,
                                             const int* conn,
                                             const double* xpts,
                                             const double* vars,
                                             const double* data) {
  if (lane < 12) {
    const int a = lane / 3, k = lane % 3;
    s.X[lane] = xpts[3 * (size_t)conn[4 * (size_t)e + a] + k];
  } else if (lane < 36) {
    const int i = lane - 12, a = i / 6, k = i % 6;
    s.u[i] = vars ? vars[6 * (size_t)conn[4 * (size_t)e + a] + k] : 0.0;
  } else if (lane < 40) {
    s.data[lane - 36] = data[4 * (size_t)e + (lane - 36)];
  }
}

__device__ __forceinline__ void element_geometry(ElemLDS& s, int lane) {
  if (lane < 4) {
    mitc4::geom_node(lane, s.X, s.g);
  } else if (lane < 9) {
    mitc4::geom_tying_x(lane - 4, s.X, s.g);
  }
  __syncthreads();
  if (lane < 4) {
    mitc4::geom_quad(lane, s.X, s.g);
  } else if (lane < 9) {
    mitc4::geom_tying_n(lane - 4, s.g);
  }
  __syncthreads();
}

__device__ __forceinline__ void element_bd(ElemLDS& s, int lane) {
  if (lane < 24) {
    mitc4::BColumnPrep prep;
    mitc4::b_column_prep(lane, s.g, prep);
#pragma unroll 1
    for (int q = 0; q < 4; q++) {
      double col[9], st[9];
      mitc4::b_column_q(lane, q, s.g, prep, col);
      mitc4::stress(s.data, col, st);
      const double sc = s.g.scale[q];
#pragma unroll
      for (int k = 0; k < 9; k++) {
        s.B[q][k][lane] = col[k];
        s.D[q][k][lane] = sc * st[k];
      }
    }
  }
  __syncthreads();
}

// 3x3 tile (rows 3I.., cols 3J..) of K_e
__device__ __forceinline__ void element_tile(const ElemLDS& s, int I, int J,
                                             double acc[3][3]) {
#pragma unroll
  for (int r = 0; r < 3; r++)
#pragma unroll
    for (int c = 0; c < 3; c++) acc[r][c] = 0.0;
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const double b0 = s.B[q][k][3 * I], b1 = s.B[q][k][3 * I + 1],
                   b2 = s.B[q][k][3 * I + 2];
      const double d0 = s.D[q][k][3 * J], d1 = s.D[q][k][3 * J + 1],
                   d2 = s.D[q][k][3 * J + 2];
      acc[0][0] += b0 * d0;
      acc[0][1] += b0 * d1;
      acc[0][2] += b0 * d2;
      acc[1][0] += b1 * d0;
      acc[1][1] += b1 * d1;
      acc[1][2] += b1 * d2;
      acc[2][0] += b2 * d0;
      acc[2][1] += b2 * d1;
      acc[2][2] += b2 * d2;
    }
}

// kColored = false: every contribution is an FP64 atomic add (K and res
// zeroed by the caller).  kColored = true: the launch covers one colour of
// an element colouring (no two elements of a colour share a node), so no two
// lanes of the launch touch the same K entry or residual entry; each
// contribution is a plain store when the element is the first to touch the
// block (first-touch mask, bits 4a+b for K blocks, 16+a for residual rows)
// and a plain read-add-write otherwise.  No atomics and no zeroing pass.
template <bool kColored>
__global__ void __launch_bounds__(64)
    jacobian_kernel(int nelems, const int* __restrict__ elem_list,
                    const int* __restrict__ first_mask,
                    const int* __restrict__ conn,
                    const double* __restrict__ xpts,
                    const double* __restrict__ vars,
                    const double* __restrict__ data,
                    const int* __restrict__ elem_ind_map,
                    const int* __restrict__ perm, double* kvals, double* res) {
  __shared__ ElemLDS s;
  if ((int)blockIdx.x >= nelems) return;
  const int e = kColored ? elem_list[blockIdx.x] : (int)blockIdx.x;
  const int mask = kColored ? first_mask[blockIdx.x] : 0;
  const int lane = threadIdx.x;
  load_element(s, e, lane, conn, xpts, vars, data);
  __syncthreads();
  element_geometry(s, lane);
  element_bd(s, lane);
  const int I = lane / 8, J = lane % 8;
  double acc[3][3];
  element_tile(s, I, J, acc);
  // scatter: tile rows belong to node a = I/2, local rows 3*(I%2)..
  const int a = I / 2, b = J / 2, r0 = 3 * (I % 2), c0 = 3 * (J % 2);
  const size_t blk = (size_t)elem_ind_map[16 * (size_t)e + 4 * a + b];
  double* dst = kvals + 36 * blk;
  const bool first = (mask >> (4 * a + b)) & 1;
#pragma unroll
  for (int r = 0; r < 3; r++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      double* d = &dst[6 * (r0 + r) + c0 + c];
      if (!kColored)
        unsafeAtomicAdd(d, acc[r][c]);
      else
        *d = first ? acc[r][c] : *d + acc[r][c];
    }
  if (res) {
    double p0 = 0, p1 = 0, p2 = 0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double uc = s.u[3 * J + c];
      p0 += acc[0][c] * uc;
      p1 += acc[1][c] * uc;
      p2 += acc[2][c] * uc;
    }
    s.rpart[J][3 * I] = p0;
    s.rpart[J][3 * I + 1] = p1;
    s.rpart[J][3 * I + 2] = p2;
    __syncthreads();
    if (lane < 24) {
      double r = 0.0;
#pragma unroll
      for (int j = 0; j < 8; j++) r += s.rpart[j][lane];
      const int node = conn[4 * (size_t)e + lane / 6];
      const int row = perm ? perm[node] : node;
      double* d = &res[6 * (size_t)row + lane % 6];
      if (!kColored)
        unsafeAtomicAdd(d, r);
      else
        *d = ((mask >> (16 + lane / 6)) & 1) ? r : *d + r;
    }
  }
}

// ---------------------------------------------------------------------------
// Two elements per 64-lane wavefront (32 lanes each), quadrature points
// streamed through LDS: per point the element's lanes 0-23 form column j of
// B_q and D_q = detXd C B_q (the column's tying-strain part is formed once
// and kept in registers), then every lane adds two 3x3 tiles of
// B_q^T D_q.  LDS per element holds the geometry and one point's B and D
// (6.2 KB), so a compute unit keeps about three times more elements in
// flight than with all four points' B and D resident.  Scatter as in
// jacobian_kernel (atomic, or colour-ordered stores / read-add-writes).
struct ElemSlotQ {
  double X[12];
  double u[24];
  double data[4];
  mitc4::Geom g;
  double B[9][24];
  double D[9][24];
};

template <bool kColored>
__global__ void __launch_bounds__(64)
    jacobian2_kernel(int nelems, const int* __restrict__ elem_list,
                     const int* __restrict__ first_mask,
                     const int* __restrict__ conn,
                     const double* __restrict__ xpts,
                     const double* __restrict__ vars,
                     const double* __restrict__ data,
                     const int* __restrict__ elem_ind_map,
                     const int* __restrict__ perm, double* kvals,
                     double* res) {
  __shared__ ElemSlotQ S[2];
  __shared__ double rp[2][8][24];  // residual partials per tile column
  const int half = threadIdx.x / 32, l = threadIdx.x % 32;
  const int slot = blockIdx.x * 2 + half;
  const bool valid = slot < nelems;
  const int e = valid ? (kColored ? elem_list[slot] : slot) : 0;
  const int mask = (kColored && valid) ? first_mask[slot] : 0;
  ElemSlotQ& s = S[half];
  if (valid) {
    for (int v = l; v < 40; v += 32) {
      if (v < 12) {
        s.X[v] = xpts[3 * (size_t)conn[4 * (size_t)e + v / 3] + v % 3];
      } else if (v < 36) {
        const int i = v - 12;
        s.u[i] = vars ? vars[6 * (size_t)conn[4 * (size_t)e + i / 6] + i % 6]
                      : 0.0;
      } else {
        s.data[v - 36] = data[4 * (size_t)e + (v - 36)];
      }
    }
  }
  __syncthreads();
  if (valid) {
    if (l < 4)
      mitc4::geom_node(l, s.X, s.g);
    else if (l < 9)
      mitc4::geom_tying_x(l - 4, s.X, s.g);
  }
  __syncthreads();
  if (valid) {
    if (l < 4)
      mitc4::geom_quad(l, s.X, s.g);
    else if (l < 9)
      mitc4::geom_tying_n(l - 4, s.g);
  }
  __syncthreads();
  // tiles (I, J) and (I + 4, J) of the 8 x 8 tile grid
  const int I0 = l / 8, J = l % 8;
  double acc[2][3][3];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int c = 0; c < 3; c++) acc[h][r][c] = 0.0;
  mitc4::BColumnPrep prep;
  if (valid && l < 24) mitc4::b_column_prep(l, s.g, prep);
#pragma unroll 1
  for (int q = 0; q < 4; q++) {
    if (valid && l < 24) {
      double col[9], st[9];
      mitc4::b_column_q(l, q, s.g, prep, col);
      mitc4::stress(s.data, col, st);
      const double sc = s.g.scale[q];
#pragma unroll
      for (int k = 0; k < 9; k++) {
        s.B[k][l] = col[k];
        s.D[k][l] = sc * st[k];
      }
    }
    __syncthreads();
    if (valid) {
#pragma unroll
      for (int k = 0; k < 9; k++) {
        const double d0 = s.D[k][3 * J], d1 = s.D[k][3 * J + 1],
                     d2 = s.D[k][3 * J + 2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int I = I0 + 4 * h;
          const double b0 = s.B[k][3 * I], b1 = s.B[k][3 * I + 1],
                       b2 = s.B[k][3 * I + 2];
          acc[h][0][0] += b0 * d0;
          acc[h][0][1] += b0 * d1;
          acc[h][0][2] += b0 * d2;
          acc[h][1][0] += b1 * d0;
          acc[h][1][1] += b1 * d1;
          acc[h][1][2] += b1 * d2;
          acc[h][2][0] += b2 * d0;
          acc[h][2][1] += b2 * d1;
          acc[h][2][2] += b2 * d2;
        }
      }
    }
    __syncthreads();
  }
  if (valid) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int I = I0 + 4 * h;
      const int a = I / 2, b = J / 2, r0 = 3 * (I % 2), c0 = 3 * (J % 2);
      double* dst = kvals + 36 * (size_t)elem_ind_map[16 * (size_t)e + 4 * a + b];
      const bool first = (mask >> (4 * a + b)) & 1;
#pragma unroll
      for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
          double* d = &dst[6 * (r0 + r) + c0 + c];
          if (!kColored)
            unsafeAtomicAdd(d, acc[h][r][c]);
          else
            *d = first ? acc[h][r][c] : *d + acc[h][r][c];
        }
    }
  }
  if (!res) return;  // uniform across the workgroup
  if (valid) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int I = I0 + 4 * h;
#pragma unroll
      for (int r = 0; r < 3; r++) {
        double v = 0.0;
#pragma unroll
        for (int c = 0; c < 3; c++) v += acc[h][r][c] * s.u[3 * J + c];
        rp[half][J][3 * I + r] = v;
      }
    }
  }
  __syncthreads();
  if (valid && l < 24) {
    double v = 0.0;
#pragma unroll
    for (int j = 0; j < 8; j++) v += rp[half][j][l];
    const int node = conn[4 * (size_t)e + l / 6];
    const int row = perm ? perm[node] : node;
    double* d = &res[6 * (size_t)row + l % 6];
    if (!kColored)
      unsafeAtomicAdd(d, v);
    else
      *d = ((mask >> (16 + l / 6)) & 1) ? v : *d + v;
  }
}

// ---------------------------------------------------------------------------
// Batched Jacobian: six elements per 64-lane wavefront, ten lanes per
// element.  Lane l of an element owns one of the ten node-pair blocks
// (a <= b) of the symmetric K_e and keeps its 6x6 sum in registers; the
// quadrature points are streamed: per point the element's ten lanes form the
// 24 columns of B_q and D_q = detXd C B_q into LDS (two or three columns per
// lane) and every lane adds B_q[:,a]^T D_q[:,b] to its block.  Block (b, a)
// is the transpose of (a, b).  LDS per element: geometry, one quadrature
// point's B and D, the element residual.
constexpr int kElemsPerWave = 6;
constexpr int kLanesPerElem = 10;

struct ElemSlot {
  double X[12];
  double u[24];
  double data[4];
  mitc4::Geom g;
  double B[9][24];
  double D[9][24];
  double res[24];
};

// block index l (0..9) -> (a, b), a <= b
__device__ __forceinline__ void pair_of(int l, int& a, int& b) {
  a = l < 4 ? 0 : l < 7 ? 1 : l < 9 ? 2 : 3;
  b = a + (l - (a == 0 ? 0 : a == 1 ? 4 : a == 2 ? 7 : 9));
}

__global__ void __launch_bounds__(64)
    jacobian_batched_kernel(int nelems, const int* __restrict__ conn,
                            const double* __restrict__ xpts,
                            const double* __restrict__ vars,
                            const double* __restrict__ data,
                            const int* __restrict__ elem_ind_map,
                            const int* __restrict__ perm, double* kvals,
                            double* res) {
  __shared__ ElemSlot S[kElemsPerWave];
  const int lane = threadIdx.x;
  const int es = lane / kLanesPerElem;
  const int l = lane % kLanesPerElem;
  const int e = blockIdx.x * kElemsPerWave + es;
  const bool valid = es < kElemsPerWave && e < nelems;
  ElemSlot& s = S[es < kElemsPerWave ? es : 0];
  if (valid) {
    for (int v = l; v < 40; v += kLanesPerElem) {
      if (v < 12) {
        s.X[v] = xpts[3 * (size_t)conn[4 * (size_t)e + v / 3] + v % 3];
      } else if (v < 36) {
        const int i = v - 12;
        s.u[i] = vars ? vars[6 * (size_t)conn[4 * (size_t)e + i / 6] + i % 6]
                      : 0.0;
      } else {
        s.data[v - 36] = data[4 * (size_t)e + (v - 36)];
      }
    }
    for (int v = l; v < 24; v += kLanesPerElem) s.res[v] = 0.0;
  }
  __syncthreads();
  if (valid) {
    if (l < 4)
      mitc4::geom_node(l, s.X, s.g);
    else if (l < 9)
      mitc4::geom_tying_x(l - 4, s.X, s.g);
  }
  __syncthreads();
  if (valid) {
    if (l < 4)
      mitc4::geom_quad(l, s.X, s.g);
    else if (l < 9)
      mitc4::geom_tying_n(l - 4, s.g);
  }
  __syncthreads();
  int a, b;
  pair_of(l, a, b);
  double acc[6][6];
#pragma unroll
  for (int r = 0; r < 6; r++)
#pragma unroll
    for (int c = 0; c < 6; c++) acc[r][c] = 0.0;
#pragma unroll 1
  for (int q = 0; q < 4; q++) {
    if (valid) {
#pragma unroll 1
      for (int j = l; j < 24; j += kLanesPerElem) {
        mitc4::BColumnPrep prep;
        mitc4::b_column_prep(j, s.g, prep);
        double col[9], st[9];
        mitc4::b_column_q(j, q, s.g, prep, col);
        mitc4::stress(s.data, col, st);
        const double sc = s.g.scale[q];
#pragma unroll
        for (int k = 0; k < 9; k++) {
          s.B[k][j] = col[k];
          s.D[k][j] = sc * st[k];
        }
      }
    }
    __syncthreads();
    if (valid) {
#pragma unroll
      for (int k = 0; k < 9; k++) {
        double ba[6], db[6];
#pragma unroll
        for (int r = 0; r < 6; r++) ba[r] = s.B[k][6 * a + r];
#pragma unroll
        for (int c = 0; c < 6; c++) db[c] = s.D[k][6 * b + c];
#pragma unroll
        for (int r = 0; r < 6; r++)
#pragma unroll
          for (int c = 0; c < 6; c++) acc[r][c] += ba[r] * db[c];
      }
    }
    __syncthreads();
  }
  if (valid) {
    const size_t blk = (size_t)elem_ind_map[16 * (size_t)e + 4 * a + b];
    double* dst = kvals + 36 * blk;
#pragma unroll
    for (int r = 0; r < 6; r++)
#pragma unroll
      for (int c = 0; c < 6; c++) unsafeAtomicAdd(&dst[6 * r + c], acc[r][c]);
    if (a != b) {
      const size_t blt = (size_t)elem_ind_map[16 * (size_t)e + 4 * b + a];
      double* dt = kvals + 36 * blt;
#pragma unroll
      for (int r = 0; r < 6; r++)
#pragma unroll
        for (int c = 0; c < 6; c++)
          unsafeAtomicAdd(&dt[6 * c + r], acc[r][c]);
    }
  }
  if (!res) return;  // uniform across the workgroup
  if (valid) {
    // R_e = K_e u_e: rows of node a from block (a, b), rows of node b from
    // its transpose
#pragma unroll
    for (int r = 0; r < 6; r++) {
      double v = 0.0;
#pragma unroll
      for (int c = 0; c < 6; c++) v += acc[r][c] * s.u[6 * b + c];
      atomicAdd(&s.res[6 * a + r], v);
    }
    if (a != b) {
#pragma unroll
      for (int c = 0; c < 6; c++) {
        double v = 0.0;
#pragma unroll
        for (int r = 0; r < 6; r++) v += acc[r][c] * s.u[6 * a + r];
        atomicAdd(&s.res[6 * b + c], v);
      }
    }
  }
  __syncthreads();
  if (valid) {
    for (int v = l; v < 24; v += kLanesPerElem) {
      const int node = conn[4 * (size_t)e + v / 6];
      const int row = perm ? perm[node] : node;
      unsafeAtomicAdd(&res[6 * (size_t)row + v % 6], s.res[v]);
    }
  }
}

// ---------------------------------------------------------------------------
// FP64 MFMA Jacobian: four elements per 64-lane wavefront, one per 16-lane
// block of v_mfma_f64_4x4x4_4b_f64 (four independent 4x4x4 products per
// instruction).  K_e = sum_q detXd_q B_q^T C B_q is one 24 x 24 x 36 product
// with the 36 = 9 strains x 4 quadrature points stacked strain-major: k-block
// s (4 wide) holds strain s at the four points.  Tile (I, J) of the product
// is taken over the nodes, K_e[6a + I][6b + J] for a, b = 0..3: the lane
// (a, q) of an element (its A row a and k index q, see MfmaLane) forms the
// six columns 6a + k of node a at point q in registers -- the MFMA A operand
// A[a][q] = B_q[s][6a + I] and the B operand D[q][b] = detXd_q (C B_q)[s]
// [6b + J] -- so B and D never pass through LDS, which DOF a column is of is
// known at compile time, and the node's and the point's frames are formed in
// the lane itself: only the node normals and drill vectors go through LDS.
// With column 4J + i in the lane instead (DOF and node both of the lane), the
// two kinds of columns diverge and index arrays at run time, and geometry
// and column parts went through 20 KB of LDS a wavefront in four steps on 4,
// 5 or 16 of 64 lanes: 400 x 400 plate, colour-ordered, 4 x 182 us; so
// 85, 110, 140 and 145 us.  What bounds it: the first colour, all stores, the
// chain of loads and frames at two wavefronts a SIMD (75 us without the
// scatter; three do not fit 54 + 21 doubles); the later colours also the adds'
// read-modify-writes of K (as plain stores 76 us; as loads and stores 157 to
// 180).
// Only the 21 tiles I <= J are formed (K_e is symmetric): 9 x 21 MFMAs per
// four elements, 24,192 flops per element.  K_e is then staged in LDS (lane
// (a, b) holds half of block (a, b) and half of (b, a)) and
// written as whole 6 x 6 blocks, consecutive lanes on consecutive entries
// of a block: plain stores (first element of the colour order to touch the
// block) and FP64 adds without return.  In the colour-ordered launches no
// two elements of a launch share a node, so each add is ordered by the
// launch sequence and the sum is deterministic; the uncoloured entry point
// adds in any order.
constexpr int kMfmaElems = 4;  // elements per wavefront (MFMA blocks)
// doubles from one 6 x 6 block to the next in LDS: with 36 the 16 blocks of an
// element would start on 8 of the 32 pairs of banks
constexpr int kBlkStride = 37;

struct ElemData {
  double X[12];
  double u[24];
  double data[4];
  double fn[4][3], dv[4][3], dw[4][3];
};
union ElemMfma {
  ElemData d;
  double Ke[16 * kBlkStride];  // block 4a + b, row-major 6 x 6
};

// detXd C (stress of a2d/a2disotropicshellstress.h:13-51) applied to the
// strain column e[0..8]; the weight of the point is in the moduli.
struct StressRows {
  double m0, m1, mg, b0, b1, bg, d0, d1, dg, As;
  __device__ __forceinline__ void init(const double d[4], double sc) {
    const double E = d[0], nu = d[1], t = d[2], to = d[3];
    const double Q0 = E / (1.0 - nu * nu), G = E / 2.0 / (1.0 + nu);
    const double am = sc * t, ab = -sc * t * t * to;
    const double ad = sc * (t * t * t / 12.0 + t * t * t * to * to);
    m0 = am * Q0;
    m1 = am * (nu * Q0);
    mg = am * G;
    b0 = ab * Q0;
    b1 = ab * (nu * Q0);
    bg = ab * G;
    d0 = ad * Q0;
    d1 = ad * (nu * Q0);
    dg = ad * G;
    As = sc * ((5.0 / 6.0) * t * G);
  }
  __device__ __forceinline__ double row(int s, const double e[9]) const {
    switch (s) {
      case 0: return m0 * e[0] + m1 * e[1] + b0 * e[3] + b1 * e[4];
      case 1: return m1 * e[0] + m0 * e[1] + b1 * e[3] + b0 * e[4];
      case 2: return mg * e[2] + bg * e[5];
      case 3: return b0 * e[0] + b1 * e[1] + d0 * e[3] + d1 * e[4];
      case 4: return b1 * e[0] + b0 * e[1] + d1 * e[3] + d0 * e[4];
      case 5: return bg * e[2] + dg * e[5];
      case 6: return As * e[6];
      case 7: return As * e[7];
      default: return 10.0 * As * e[8];
    }
  }
};

#ifndef GPUFEM_MFMA_MINWAVES
#define GPUFEM_MFMA_MINWAVES 2
#endif
// A lane's place in the four-elements-per-wavefront layout.  Lane layout of
// v_mfma_f64_4x4x4_4b_f64 on gfx950 (measured): the block of lane L is
// (L / 4) % 4; its A operand is A[L % 4][L / 16], its B operand
// B[L / 16][L % 4] and its result D[L / 16][L % 4].  So a lane forms the
// columns of node a = L % 4 at point q = L / 16, and receives node block
// (q, a) of the product.  Blocks past the last element take element 0's
// data, and nothing of theirs is written.
struct MfmaLane {
  int grp, a, q, slot, e, node;
  bool valid;
  __device__ __forceinline__ MfmaLane(int nelems, const int* elem_list,
                                      const int* conn) {
    const int lane = threadIdx.x;
    grp = (lane >> 2) & 3;
    a = lane & 3;
    q = lane >> 4;
    slot = blockIdx.x * kMfmaElems + grp;
    valid = slot < nelems;
    e = !valid ? 0 : elem_list ? elem_list[slot] : slot;
    node = conn[4 * (size_t)e + a];
  }
};

// Sum over the four lanes of a quad (the nodes of an element at one point).
template <int kCtrl>
__device__ __forceinline__ double quad_perm(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, kCtrl, 0xf, 0xf, true);
  const int hi =
      __builtin_amdgcn_mov_dpp((int)(b >> 32), kCtrl, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double quad_sum(double v) {
  v += quad_perm<0xb1>(v);         // lanes 1, 0, 3, 2
  return v + quad_perm<0x4e>(v);   // lanes 2, 3, 0, 1
}
// Sum over the four points of an element (lanes 16 apart).
__device__ __forceinline__ double point_sum(double v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The lane's columns and what else the kernels need of its node and point.
struct LaneColumns {
  double B[6][9];
  double nf[3];
  mitc4::NodePoint np;
  StressRows C;
};
__device__ __forceinline__ void mfma_columns(ElemData& s, const MfmaLane& L,
                                             const double* xpts,
                                             const double* vars,
                                             const double* data,
                                             LaneColumns& c) {
  if (L.q < 3) s.X[3 * L.a + L.q] = xpts[3 * (size_t)L.node + L.q];
  if (vars) {
    s.u[6 * L.a + L.q] = vars[6 * (size_t)L.node + L.q];
    if (L.q < 2) s.u[6 * L.a + 4 + L.q] = vars[6 * (size_t)L.node + 4 + L.q];
  }
  if (L.q == 3) s.data[L.a] = data[4 * (size_t)L.e + L.a];
  __syncthreads();
  double nd[3], dv[3], dw[3];
  mitc4::node_frame(L.a, s.X, c.nf, nd, dv, dw);
  if (L.q == 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      s.fn[L.a][k] = c.nf[k];
      s.dv[L.a][k] = dv[k];
      s.dw[L.a][k] = dw[k];
    }
  }
  __syncthreads();
  double A[9], Z[9], T[6];
  c.C.init(s.data, mitc4::quad_frame(L.q, s.X, s.fn, A, Z, T));
  c.np.init(L.a, L.q, A, Z);
  mitc4::node_columns_q(L.a, L.q, s.X, s.fn, s.dv, s.dw, c.nf, nd, A, T, c.np,
                        c.B);
}

// Upper tiles of K_e: acc[t] of lane (q, a) is K_e[6q + I][6a + J].
__device__ __forceinline__ void mfma_product(const LaneColumns& c,
                                             double (&acc)[21]) {
#pragma unroll
  for (int t = 0; t < 21; t++) acc[t] = 0.0;
#pragma unroll
  for (int st = 0; st < 9; st++) {
    double d[6];
#pragma unroll
    for (int J = 0; J < 6; J++) d[J] = c.C.row(st, c.B[J]);
    int t = 0;
#pragma unroll
    for (int I = 0; I < 6; I++)
#pragma unroll
      for (int J = I; J < 6; J++, t++)
        acc[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(c.B[I][st], d[J], acc[t],
                                                    0, 0, 0);
  }
}

// K_e of the wavefront's elements: staged in LDS (over the element data) and
// added to its blocks.
template <bool kColored>
__device__ __forceinline__ void mfma_scatter(ElemMfma* S, const MfmaLane& L,
                                             const double (&acc)[21],
                                             int nelems, int own_dst,
                                             int* s_dst, double* kvals) {
  __syncthreads();  // element data no longer read
  {
    s_dst[16 * L.grp + 4 * L.q + L.a] = own_dst;
    double* k1 = &S[L.grp].Ke[kBlkStride * (4 * L.q + L.a)];
    double* k2 = &S[L.grp].Ke[kBlkStride * (4 * L.a + L.q)];
    int t = 0;
#pragma unroll
    for (int I = 0; I < 6; I++)
#pragma unroll
      for (int J = I; J < 6; J++, t++) {
        k1[6 * I + J] = acc[t];
        if (J != I) k2[6 * J + I] = acc[t];
      }
  }
  __syncthreads();
  // entry rc of block nb of the wavefront's 64, 64 entries further each time
  const int nblk = 16 * min(kMfmaElems, nelems - (int)blockIdx.x * kMfmaElems);
  const double* ke = &S[0].Ke[0];
  int nb = threadIdx.x >= 36, rc = (int)threadIdx.x - 36 * nb;
#pragma unroll 4
  for (int it = 0; it < 36; it++) {
    if (nb < nblk) {
      const double v = ke[kBlkStride * nb + rc];
      const int dst = s_dst[nb];
      // colour-ordered: no other element of this launch touches the block,
      // so the add without return is ordered by the launches alone (the same
      // sum, bit for bit, as a read-add-write, without the read's latency)
      if (kColored && dst < 0)
        kvals[36 * (size_t)~dst + rc] = v;
      else
        unsafeAtomicAdd(&kvals[36 * (size_t)dst + rc], v);
    }
    nb += 1;
    rc += 28;
    if (rc >= 36) {
      rc -= 36;
      nb += 1;
    }
  }
}

// Where block 4q + a of the lane's element goes: its block of K,
// complemented if the element is the first to touch it.
template <bool kColored>
__device__ __forceinline__ int mfma_dst(const MfmaLane& L,
                                        const int* elem_ind_map, int mask) {
  const int ab = 4 * L.q + L.a;
  const int b = elem_ind_map[16 * (size_t)L.e + ab];
  return kColored && ((mask >> ab) & 1) ? ~b : b;
}

// B u of the lane's point and its stress, detXd C (B u).
__device__ __forceinline__ void point_strain(const ElemData& s,
                                             const MfmaLane& L,
                                             const LaneColumns& c,
                                             double (&E)[9]) {
#pragma unroll
  for (int st = 0; st < 9; st++) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 6; k++) v += c.B[k][st] * s.u[6 * L.a + k];
    E[st] = quad_sum(v);
  }
}
__device__ __forceinline__ void point_stress(const LaneColumns& c,
                                             const double (&E)[9],
                                             double (&St)[9]) {
#pragma unroll
  for (int st = 0; st < 9; st++) St[st] = c.C.row(st, E);
}
// Energy of the wavefront's elements.
__device__ __forceinline__ void mfma_energy(const MfmaLane& L,
                                            const double (&E)[9],
                                            const double (&St)[9],
                                            double* energy) {
  double es = 0.0;
#pragma unroll
  for (int st = 0; st < 9; st++) es += E[st] * St[st];
  es = wave_sum(L.valid && L.a == 0 ? 0.5 * es : 0.0);
  if (threadIdx.x == 0) unsafeAtomicAdd(energy, es);
}
// R_e = sum_q B_q^T S_q into res: point q's lanes write DOFs q and 4 + q.
template <bool kColored>
__device__ __forceinline__ void mfma_residual(const MfmaLane& L,
                                              const LaneColumns& c,
                                              const double (&St)[9],
                                              const int* perm, int mask,
                                              double* res) {
  double own[2] = {0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 6; k++) {
    double v = 0.0;
#pragma unroll
    for (int st = 0; st < 9; st++) v += c.B[k][st] * St[st];
    v = point_sum(v);
    if (k % 4 == L.q) own[k / 4] = v;
  }
  if (!L.valid) return;
  const int row = perm ? perm[L.node] : L.node;
  const bool first = kColored && ((mask >> (16 + L.a)) & 1);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int k = 4 * h + L.q;
    if (k >= 6) continue;
    double* d = &res[6 * (size_t)row + k];
    if (!kColored)
      unsafeAtomicAdd(d, own[h]);
    else
      *d = first ? own[h] : *d + own[h];
  }
}

template <bool kColored>
__global__ void __launch_bounds__(64, GPUFEM_MFMA_MINWAVES)
    jacobian_mfma_kernel(int nelems, const int* __restrict__ elem_list,
                         const int* __restrict__ first_mask,
                         const int* __restrict__ conn,
                         const double* __restrict__ xpts,
                         const double* __restrict__ vars,
                         const double* __restrict__ data,
                         const int* __restrict__ elem_ind_map,
                         const int* __restrict__ perm, double* kvals,
                         double* res) {
  __shared__ ElemMfma S[kMfmaElems];
  __shared__ int s_dst[16 * kMfmaElems];
  const MfmaLane L(nelems, kColored ? elem_list : nullptr, conn);
  ElemData& s = S[L.grp].d;
  const int mask = kColored && L.valid ? first_mask[L.slot] : 0;
  const int dst = mfma_dst<kColored>(L, elem_ind_map, mask);
  LaneColumns c;
  mfma_columns(s, L, xpts, vars, data, c);
  if (res) {  // uniform; vars null: u = 0
    double E[9], St[9];
#pragma unroll
    for (int st = 0; st < 9; st++) E[st] = 0.0;
    if (vars) point_strain(s, L, c, E);
    point_stress(c, E, St);
    mfma_residual<kColored>(L, c, St, perm, mask, res);
  }
  double acc[21];
  mfma_product(c, acc);
  mfma_scatter<kColored>(S, L, acc, nelems, dst, s_dst, kvals);
}

// ---------------------------------------------------------------------------
// Nonlinear MITC4 (IsotropicShell<..., isNonlinear = true>, physics.h:6-17):
// NonlinearShellStrainCore (a2d/a2dshellstrain.h:72-93) adds to the bending
// strains the quadratic terms of the local displacement gradients u0x, u1x
// (basis.h:470-492),
//   e3 += u0x(:,0).u1x(:,0),  e4 += u0x(:,1).u1x(:,1),
//   e5 += u0x(:,0).u1x(:,1) + u1x(:,0).u0x(:,1);
// the tying strains and the director stay linear (physics.h:214-219,
// 286-300).  With G0, G1 the maps of the element DOFs to the entries
// (r, c < 2) of u0x, u1x (mitc4::NodePoint), B_q(u) = dE_q/du and
// S_q = detXd_q C E_q(u):
//   R_e(u) = sum_q B_q(u)^T S_q                         (the gradient of
//   U = sum_q 1/2 detXd_q E^T C E, physics.h:18-36),
//   K_e(u) = sum_q detXd_q B_q(u)^T C B_q(u) + G0^T W_q G1 + G1^T W_q G0,
// W_q holding S_q's bending stresses on the gradient-entry pairs each
// quadratic term multiplies: K_e is the exact Hessian of U.  (The
// reference's own nonlinear Jacobian routes its displacement gradients'
// second-order terms into the residual, elem_group.h:286-289, and
// overwrites the u0x sensitivity with the u1x one, basis.h:565-567.)
// Layout and scatter as in jacobian_mfma_kernel; R_e into res (6 perm[node] +
// k), the energy into *energy; kvals, res or energy may be null.
// All entries of G0 and G1 of node a are t_r[k] or (fn_a x t_r)[k] times the
// four pairs of scalars of NodePoint, and the t_r are orthonormal: sums over
// r of products of gradient entries do not need the frame.  With D_c the global vectors sum_a su_c u_a +
// ru_c (q_a x fn_a) of u0x (and of sz, rz for u1x), sum_r u0x_rc u1x_rc' =
// D0_c . D1_c'; the columns of B(u) take D0 and D1 alone; and the last two
// terms of K_e are, for nodes a and b, three scalars
//   SS, SR, RR = sum_q sum_c (pu_c (W pz)_c + pz_c (W pu)_c),  p = s or r,
// times I, the cross-product matrix of fn_b and (fn_a . fn_b) I - fn_b fn_a^T:
// 12 MFMAs instead of the 252 of the 24 x 24 x 48 product.
// 131,328-node cylinder (131,072 elements), colour-ordered K and R: 3.31 ms
// with one element a wavefront and 3 x 3 tiles through LDS, 0.47 ms so (the
// four colours 85, 150, 100 and 136 us; bound as jacobian_mfma_kernel).
template <bool kColored>
__global__ void __launch_bounds__(64, GPUFEM_MFMA_MINWAVES)
    tangent_kernel(int nelems, const int* __restrict__ elem_list,
                   const int* __restrict__ first_mask,
                   const int* __restrict__ conn,
                   const double* __restrict__ xpts,
                   const double* __restrict__ vars,
                   const double* __restrict__ data,
                   const int* __restrict__ elem_ind_map,
                   const int* __restrict__ perm, double* kvals, double* res,
                   double* energy) {
  __shared__ ElemMfma S[kMfmaElems];
  __shared__ int s_dst[16 * kMfmaElems];
  const MfmaLane L(nelems, kColored ? elem_list : nullptr, conn);
  ElemData& s = S[L.grp].d;
  const int mask = kColored && L.valid ? first_mask[L.slot] : 0;
  const int dst = kvals ? mfma_dst<kColored>(L, elem_ind_map, mask) : 0;
  LaneColumns c;
  mfma_columns(s, L, xpts, vars, data, c);
  double E[9], St[9];
  point_strain(s, L, c, E);
  const mitc4::NodePoint& np = c.np;
  {
    double D0[2][3], D1[2][3];  // global gradient vectors of u0x, u1x
    const double* u = &s.u[6 * L.a];
    const double th[3] = {u[3], u[4], u[5]};
    double d[3];
    mitc4::cross(th, c.nf, d);
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int m = 0; m < 2; m++) {
        D0[m][k] = quad_sum(np.su[m] * u[k] + np.ru[m] * d[k]);
        D1[m][k] = quad_sum(np.sz[m] * u[k] + np.rz[m] * d[k]);
      }
    E[3] += mitc4::dot3(D0[0], D1[0]);
    E[4] += mitc4::dot3(D0[1], D1[1]);
    E[5] += mitc4::dot3(D0[0], D1[1]) + mitc4::dot3(D1[0], D0[1]);
    // dE/du: the quadratic terms' derivative, per DOF of node a
    double w[3][3], v[3][3];  // rows 3..5, displacements and directors
#pragma unroll
    for (int k = 0; k < 3; k++) {
      w[0][k] = np.su[0] * D1[0][k] + np.sz[0] * D0[0][k];
      w[1][k] = np.su[1] * D1[1][k] + np.sz[1] * D0[1][k];
      w[2][k] = np.su[0] * D1[1][k] + np.sz[1] * D0[0][k] +
                np.sz[0] * D0[1][k] + np.su[1] * D1[0][k];
      v[0][k] = np.ru[0] * D1[0][k] + np.rz[0] * D0[0][k];
      v[1][k] = np.ru[1] * D1[1][k] + np.rz[1] * D0[1][k];
      v[2][k] = np.ru[0] * D1[1][k] + np.rz[1] * D0[0][k] +
                np.rz[0] * D0[1][k] + np.ru[1] * D1[0][k];
    }
#pragma unroll
    for (int m = 0; m < 3; m++) {
      double f[3];
      mitc4::cross(c.nf, v[m], f);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        c.B[k][3 + m] += w[m][k];
        c.B[3 + k][3 + m] += f[k];
      }
    }
  }
  point_stress(c, E, St);
  if (energy) mfma_energy(L, E, St, energy);  // uniform
  if (res) mfma_residual<kColored>(L, c, St, perm, mask, res);
  if (!kvals) return;  // uniform across the workgroup
  double acc[21];
  mfma_product(c, acc);
  double ss = 0.0, sr = 0.0, rr = 0.0;
#pragma unroll
  for (int m = 0; m < 2; m++) {
    const double w0 = m ? St[5] : St[3], w1 = m ? St[4] : St[5];
    const double wsz = w0 * np.sz[0] + w1 * np.sz[1];
    const double wsu = w0 * np.su[0] + w1 * np.su[1];
    const double wrz = w0 * np.rz[0] + w1 * np.rz[1];
    const double wru = w0 * np.ru[0] + w1 * np.ru[1];
    ss = __builtin_amdgcn_mfma_f64_4x4x4f64(np.su[m], wsz, ss, 0, 0, 0);
    sr = __builtin_amdgcn_mfma_f64_4x4x4f64(np.su[m], wrz, sr, 0, 0, 0);
    rr = __builtin_amdgcn_mfma_f64_4x4x4f64(np.ru[m], wrz, rr, 0, 0, 0);
    ss = __builtin_amdgcn_mfma_f64_4x4x4f64(np.sz[m], wsu, ss, 0, 0, 0);
    sr = __builtin_amdgcn_mfma_f64_4x4x4f64(np.sz[m], wru, sr, 0, 0, 0);
    rr = __builtin_amdgcn_mfma_f64_4x4x4f64(np.rz[m], wru, rr, 0, 0, 0);
  }
  // the lane's result is block (q, a): rows of node q, columns of node a
  const double* fq = s.fn[L.q];
  const double* fa = c.nf;
  const double fqa = mitc4::dot3(fq, fa);
  int t = 0;
#pragma unroll
  for (int I = 0; I < 6; I++)
#pragma unroll
    for (int J = I; J < 6; J++, t++) {
      if (J < 3) {
        if (I == J) acc[t] += ss;
      } else if (I < 3) {
        // sum_r t_r[k] (fn x t_r)[l] = eps_lmk fn[m]
        const int k = I, l = J - 3;
        if (l == (k + 1) % 3) acc[t] += sr * fa[3 - k - l];
        if (l == (k + 2) % 3) acc[t] -= sr * fa[3 - k - l];
      } else {
        const int k = I - 3, l = J - 3;
        acc[t] += rr * ((k == l ? fqa : 0.0) - fa[k] * fq[l]);
      }
    }
  mfma_scatter<kColored>(S, L, acc, nelems, dst, s_dst, kvals);
}

// Residual, R_e = sum_q B_q^T (detXd C B_q u), or energy, U = sum_e sum_q 1/2
// detXd (B_q u) . C (B_q u), in the layout of jacobian_mfma_kernel.
// 131 x 257 cylinder (33,667 elements), residual: 197 us with one element a
// wavefront and B and D through LDS, 31 us so.
template <bool kEnergy>
__global__ void __launch_bounds__(64, GPUFEM_MFMA_MINWAVES)
    residual_kernel(int nelems, const int* __restrict__ conn,
                    const double* __restrict__ xpts,
                    const double* __restrict__ vars,
                    const double* __restrict__ data,
                    const int* __restrict__ perm, double* out) {
  __shared__ ElemData S[kMfmaElems];
  const MfmaLane L(nelems, nullptr, conn);
  ElemData& s = S[L.grp];
  LaneColumns c;
  mfma_columns(s, L, xpts, vars, data, c);
  double E[9], St[9];
  point_strain(s, L, c, E);
  point_stress(c, E, St);
  if constexpr (kEnergy)
    mfma_energy(L, E, St, out);
  else
    mfma_residual<false>(L, c, St, perm, 0, out);
}

}  // namespace
}  // namespace gf

namespace {
// Jacobian kernel: the FP64 MFMA kernel by default; GPUFEM_ASSEMBLY=scalar
// selects the two-elements-per-wavefront scalar kernel (jacobian2_kernel),
// =element the one-element-per-wavefront kernel, =batched the
// six-elements-per-wavefront one (atomic entry point only)
enum { kAsmMfma = 0, kAsmElement = 1, kAsmBatched = 2, kAsmScalar = 3 };
int assembly_variant() {
  static const int v = [] {
    const char* e = getenv("GPUFEM_ASSEMBLY");
    if (e && std::string(e) == "element") return (int)kAsmElement;
    if (e && std::string(e) == "batched") return (int)kAsmBatched;
    if (e && std::string(e) == "scalar") return (int)kAsmScalar;
    return (int)kAsmMfma;
  }();
  return v;
}
}  // namespace

extern "C" {

int gf_assemble_jacobian_mitc4_f64(gf_context ctx, int nelems, int nnodes,
                                   const int* conn, const double* xpts,
                                   const double* vars, const double* data,
                                   const int* elem_ind_map, const int* perm,
                                   double* kvals, double* res) {
  if (!ctx || nelems < 0 || nnodes <= 0 || !conn || !xpts || !data ||
      !elem_ind_map || !kvals)
    return gf::set_error(ctx, GF_ERR_INVALID, "assemble_jacobian: bad args");
  if (nelems == 0) return GF_OK;
  if (assembly_variant() == kAsmMfma) {
    hipLaunchKernelGGL(gf::jacobian_mfma_kernel<false>,
                       dim3(gf::div_up(nelems, gf::kMfmaElems)), dim3(64), 0,
                       ctx->stream, nelems, (const int*)nullptr,
                       (const int*)nullptr, conn, xpts, vars, data,
                       elem_ind_map, perm, kvals, res);
    return gf::check_launch(ctx, "jacobian_mfma_kernel");
  }
  if (assembly_variant() == kAsmElement) {
    hipLaunchKernelGGL(gf::jacobian_kernel<false>, dim3(nelems), dim3(64), 0,
                       ctx->stream, nelems, (const int*)nullptr,
                       (const int*)nullptr, conn, xpts, vars, data,
                       elem_ind_map, perm, kvals, res);
    return gf::check_launch(ctx, "jacobian_kernel");
  }
  if (assembly_variant() == kAsmScalar) {
    hipLaunchKernelGGL(gf::jacobian2_kernel<false>,
                       dim3(gf::div_up(nelems, 2)), dim3(64), 0, ctx->stream,
                       nelems, (const int*)nullptr, (const int*)nullptr, conn,
                       xpts, vars, data, elem_ind_map, perm, kvals, res);
    return gf::check_launch(ctx, "jacobian2_kernel");
  }
  hipLaunchKernelGGL(gf::jacobian_batched_kernel,
                     dim3(gf::div_up(nelems, gf::kElemsPerWave)), dim3(64), 0,
                     ctx->stream, nelems, conn, xpts, vars, data, elem_ind_map,
                     perm, kvals, res);
  return gf::check_launch(ctx, "jacobian_batched_kernel");
}


int gf_asm_plan_create(gf_context ctx, int nelems, int nnodes,
                       const int* conn, const int* elem_ind_map, int nnzb,
                       gf_asm_plan* out) {
  if (!ctx || nelems <= 0 || nnodes <= 0 || !conn || !elem_ind_map ||
      nnzb <= 0 || !out)
    return gf::set_error(ctx, GF_ERR_INVALID, "asm_plan_create: bad args");
  auto* pl = new gf_asm_plan_s;
  pl->ctx = ctx;
  pl->nelems = nelems;
  pl->nnzb = nnzb;
  pl->nnodes = nnodes;
  std::vector<int> elems;
  gf::element_coloring(nelems, nnodes, 4, conn, pl->color_ptr, elems);
  pl->ncolors = (int)pl->color_ptr.size() - 1;
  // first-touch masks in processing order (colour-major)
  std::vector<int> mask(nelems, 0);
  std::vector<char> kt(nnzb, 0), rt(nnodes, 0);
  for (int p = 0; p < nelems; p++) {
    const int e = elems[p];
    int m = 0;
    for (int ab = 0; ab < 16; ab++) {
      const int blk = elem_ind_map[16 * (size_t)e + ab];
      if (blk < 0 || blk >= nnzb) {
        delete pl;
        return gf::set_error(ctx, GF_ERR_INVALID,
                             "asm_plan_create: element %d maps outside K", e);
      }
      if (!kt[blk]) {
        kt[blk] = 1;
        m |= 1 << ab;
      }
    }
    for (int a = 0; a < 4; a++) {
      const int nd = conn[4 * (size_t)e + a];
      if (!rt[nd]) {
        rt[nd] = 1;
        m |= 1 << (16 + a);
      }
    }
    mask[p] = m;
  }
  for (int k = 0; k < nnzb && !pl->zero_k; k++) pl->zero_k = !kt[k];
  for (int i = 0; i < nnodes && !pl->zero_res; i++) pl->zero_res = !rt[i];
  int st = gf::dmalloc(ctx, (void**)&pl->elems, sizeof(int) * nelems);
  if (!st) st = gf::dmalloc(ctx, (void**)&pl->mask, sizeof(int) * nelems);
  if (st) {
    gf_asm_plan_destroy(pl);
    return st;
  }
  // copies on the context's stream (a plain hipMemcpy would also wait for
  // the other streams of the device); the host vectors live until the sync
  if (hipMemcpyAsync(pl->elems, elems.data(), sizeof(int) * nelems,
                     hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
      hipMemcpyAsync(pl->mask, mask.data(), sizeof(int) * nelems,
                     hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
      hipStreamSynchronize(ctx->stream) != hipSuccess) {
    gf_asm_plan_destroy(pl);
    return gf::set_error(ctx, GF_ERR_DEVICE, "asm_plan_create: upload");
  }
  *out = pl;
  return GF_OK;
}

int gf_asm_plan_destroy(gf_asm_plan pl) {
  if (!pl) return GF_OK;
  gf::dfree(pl->ctx, pl->elems);
  gf::dfree(pl->ctx, pl->mask);
  delete pl;
  return GF_OK;
}

int gf_asm_plan_colors(gf_asm_plan pl) { return pl ? pl->ncolors : -1; }

int gf_assemble_jacobian_colored_f64(gf_context ctx, gf_asm_plan pl,
                                     const int* conn, const double* xpts,
                                     const double* vars, const double* data,
                                     const int* elem_ind_map, const int* perm,
                                     double* kvals, double* res) {
  if (!ctx || !pl || !conn || !xpts || !data || !elem_ind_map || !kvals)
    return gf::set_error(ctx, GF_ERR_INVALID, "assemble_colored: bad args");
  if (pl->zero_k)
    GF_HIP(ctx, hipMemsetAsync(kvals, 0, sizeof(double) * 36 * (size_t)pl->nnzb,
                               ctx->stream));
  if (res && pl->zero_res)
    GF_HIP(ctx, hipMemsetAsync(res, 0, sizeof(double) * 6 * (size_t)pl->nnodes,
                               ctx->stream));
  for (int c = 0; c < pl->ncolors; c++) {
    const int c0 = pl->color_ptr[c], cnt = pl->color_ptr[c + 1] - c0;
    if (assembly_variant() == kAsmMfma)
      hipLaunchKernelGGL(gf::jacobian_mfma_kernel<true>,
                         dim3(gf::div_up(cnt, gf::kMfmaElems)), dim3(64), 0,
                         ctx->stream, cnt, pl->elems + c0, pl->mask + c0,
                         conn, xpts, vars, data, elem_ind_map, perm, kvals,
                         res);
    else if (assembly_variant() == kAsmElement)
      hipLaunchKernelGGL(gf::jacobian_kernel<true>, dim3(cnt), dim3(64), 0,
                         ctx->stream, cnt, pl->elems + c0, pl->mask + c0,
                         conn, xpts, vars, data, elem_ind_map, perm, kvals,
                         res);
    else
      hipLaunchKernelGGL(gf::jacobian2_kernel<true>, dim3(gf::div_up(cnt, 2)),
                         dim3(64), 0, ctx->stream, cnt, pl->elems + c0,
                         pl->mask + c0, conn, xpts, vars, data, elem_ind_map,
                         perm, kvals, res);
  }
  return gf::check_launch(ctx, "jacobian_kernel<colored>");
}

int gf_assemble_tangent_mitc4_f64(gf_context ctx, int nelems, int nnodes,
                                  const int* conn, const double* xpts,
                                  const double* vars, const double* data,
                                  const int* elem_ind_map, const int* perm,
                                  double* kvals, double* res,
                                  double* energy) {
  if (!ctx || nelems < 0 || nnodes <= 0 || !conn || !xpts || !vars ||
      !data || (kvals && !elem_ind_map))
    return gf::set_error(ctx, GF_ERR_INVALID, "assemble_tangent: bad args");
  if (energy)
    GF_HIP(ctx, hipMemsetAsync(energy, 0, sizeof(double), ctx->stream));
  if (nelems == 0) return GF_OK;
  hipLaunchKernelGGL(gf::tangent_kernel<false>,
                     dim3(gf::div_up(nelems, gf::kMfmaElems)), dim3(64), 0,
                     ctx->stream, nelems, (const int*)nullptr,
                     (const int*)nullptr, conn, xpts, vars, data, elem_ind_map,
                     perm, kvals, res, energy);
  return gf::check_launch(ctx, "tangent_kernel");
}

int gf_assemble_tangent_colored_f64(gf_context ctx, gf_asm_plan pl,
                                    const int* conn, const double* xpts,
                                    const double* vars, const double* data,
                                    const int* elem_ind_map, const int* perm,
                                    double* kvals, double* res) {
  if (!ctx || !pl || !conn || !xpts || !vars || !data || !elem_ind_map ||
      !kvals)
    return gf::set_error(ctx, GF_ERR_INVALID, "assemble_tangent_colored: bad args");
  if (pl->zero_k)
    GF_HIP(ctx, hipMemsetAsync(kvals, 0, sizeof(double) * 36 * (size_t)pl->nnzb,
                               ctx->stream));
  if (res && pl->zero_res)
    GF_HIP(ctx, hipMemsetAsync(res, 0, sizeof(double) * 6 * (size_t)pl->nnodes,
                               ctx->stream));
  for (int c = 0; c < pl->ncolors; c++) {
    const int c0 = pl->color_ptr[c], cnt = pl->color_ptr[c + 1] - c0;
    hipLaunchKernelGGL(gf::tangent_kernel<true>,
                       dim3(gf::div_up(cnt, gf::kMfmaElems)), dim3(64), 0,
                       ctx->stream, cnt, pl->elems + c0, pl->mask + c0, conn,
                       xpts, vars, data, elem_ind_map, perm, kvals, res,
                       (double*)nullptr);
  }
  return gf::check_launch(ctx, "tangent_kernel<colored>");
}

int gf_assemble_residual_mitc4_f64(gf_context ctx, int nelems, int nnodes,
                                   const int* conn, const double* xpts,
                                   const double* vars, const double* data,
                                   const int* perm, double* res) {
  if (!ctx || nelems < 0 || nnodes <= 0 || !conn || !xpts || !vars ||
      !data || !res)
    return gf::set_error(ctx, GF_ERR_INVALID, "assemble_residual: bad args");
  if (nelems == 0) return GF_OK;
  hipLaunchKernelGGL(gf::residual_kernel<false>,
                     dim3(gf::div_up(nelems, gf::kMfmaElems)), dim3(64), 0,
                     ctx->stream, nelems, conn, xpts, vars, data, perm, res);
  return gf::check_launch(ctx, "residual_kernel");
}

int gf_energy_mitc4_f64(gf_context ctx, int nelems, const int* conn,
                        const double* xpts, const double* vars,
                        const double* data, double* energy) {
  if (!ctx || nelems < 0 || !conn || !xpts || !vars || !data || !energy)
    return gf::set_error(ctx, GF_ERR_INVALID, "energy: bad args");
  GF_HIP(ctx, hipMemsetAsync(energy, 0, sizeof(double), ctx->stream));
  if (nelems == 0) return GF_OK;
  hipLaunchKernelGGL(gf::residual_kernel<true>,
                     dim3(gf::div_up(nelems, gf::kMfmaElems)), dim3(64), 0,
                     ctx->stream, nelems, conn, xpts, vars, data,
                     (const int*)nullptr, energy);
  return gf::check_launch(ctx, "energy_kernel");
}

}  // extern "C"
