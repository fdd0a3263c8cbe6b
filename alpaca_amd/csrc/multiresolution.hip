// Multiresolution operators of ALPACA between parent and child blocks held in
// one pool of haloed blocks on gfx950: conservative averaging of a child into
// its parent (Multiresolution::Average, multiresolution.h:94-167; of its jump
// surfaces, AverageJumpBuffer, multiresolution.cpp:47-131), Harten's
// fifth-order prediction of a parent into a child (Multiresolution::
// Prediction, multiresolution.cpp:146-292) and the L-infinity wavelet detail
// with the remeshing decision (ChildNeedsRemeshing<Norm::Linfinity>,
// multiresolution.cpp:299-323; RemeshingDecision, :408-428).
//
// Every expression keeps the reference's operation order and the translation
// unit is built without contraction, so the results are the reference's bits;
// std::min/std::max picks (first extreme, NaN comparisons false) are spelled
// out so that non-finite inputs propagate as they do there.
//
// Work decomposition.  A link names (child block, parent block, sibling
// position, child level).  Averaging is one thread per two parent cells
// written (adjacent along the fastest axis, so the child reads of neighbouring
// threads are contiguous 16-byte accesses).  Prediction and details stage the
// parent's stencil window -- the predicted parent cells plus two on each side, at
// most 16 per axis (32 KiB of doubles in 3D) -- in LDS; a thread predicts the
// children of one parent cell in 2D, of two adjacent along z in 3D.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "fv_device.h"

namespace alpaca {
namespace mr {
namespace {

constexpr int kThreads = 256;         // averaging
constexpr int kStencilThreads = 192;  // 2D prediction of large ranges, 2D details
constexpr int kMaxLevels = 32;

// LDS layout of a parent stencil window: [W][W][W] doubles in 3D, [W][W] in
// 2D, whatever part of it a range fills, so that every stencil offset is a
// compile-time constant.  W = 16 holds any window; W = 12 the windows of
// ranges of at most 8 predicted parent cells per axis (jump halo slabs, the
// internal cells).
template <int DIM, int W> struct LdsW {
  static constexpr int SX = DIM == 3 ? W * W : W;
  static constexpr int SY = DIM == 3 ? W : 1;
  static constexpr int SIZE = W * SX;
};
template <int DIM> using Lds = LdsW<DIM, 16>;

// ConsistencyManagedSum, three and four values (mathematical_functions.h:79-91,
// 115-124): 0.5 (min + max) of the three pairings s1, s2, s3, where std::min
// and std::max over the initializer list keep the first extreme and never
// pick a NaN by comparison.  The hardware minimum/maximum (one instruction
// each) pick the same value whenever s1 is not NaN:
//  * a NaN among s2, s3 is skipped by both (std: the comparison is false);
//  * ties: a rounded sum is -0 only when both addends are -0, so the s_i are
//    zeros of one sign or of none -- equal values are the same bits.
// When s1 is NaN, std keeps it for both extremes and the result is NaN.
__device__ __forceinline__ double cms_pick(double s1, double s2, double s3) {
  double const mn = __builtin_fmin(__builtin_fmin(s1, s2), s3);
  double const mx = __builtin_fmax(__builtin_fmax(s1, s2), s3);
  double const r = 0.5 * (mn + mx);
  return s1 != s1 ? s1 : r;
}
__device__ __forceinline__ double cms3(double a, double b, double c) {
  return cms_pick((a + b) + c, (a + c) + b, (b + c) + a);
}
__device__ __forceinline__ double cms4(double a, double b, double c, double d) {
  return cms_pick((a + b) + (c + d), (a + c) + (b + d), (a + d) + (b + c));
}
// DimensionAwareConsistencyManagedSum (mathematical_functions.h:98-108).
template <int DIM> __device__ __forceinline__ double dams(double a, double b, double c) {
  if constexpr (DIM == 2) {
    (void)c;
    return a + b;
  } else {
    return cms3(a, b, c);
  }
}

template <int DIM> __device__ __forceinline__ bool link_ok(const alpaca_mr_link &l, int nblocks) {
  return l.child >= 0 && l.child < nblocks && l.parent >= 0 && l.parent < nblocks &&
         l.child != l.parent && l.position >= 0 && l.position < (1 << DIM);
}

// ---------------------------------------------------------------- averaging

// Parent internal cells covered by one child: IC/2 per axis, starting at HS
// (low child) or TC/2 (high child) (xyz_look_up_table_, multiresolution.h:
// 35-45); child cells from HS in steps of two.  Each thread writes two parent
// cells adjacent along the fastest axis (k in 3D, j in 2D) and reads the four
// contiguous child cells under them per child row as two 16-byte loads; every
// such pair starts at an even element offset of a block (16-byte aligned).
template <int DIM> struct AvgShape {
  static constexpr int H = kIC / 2;                  // parent cells per axis
  static constexpr int PAIRS = DIM == 3 ? H * H * (H / 2) : H * (H / 2);  // threads per field
};

template <int DIM>
__global__ __launch_bounds__(kThreads) void average_kernel(double *__restrict__ blocks, int nblocks,
                                                           const alpaca_mr_link *__restrict__ links,
                                                           int nlinks) {
  using D = Dims<DIM>;
  constexpr int H = AvgShape<DIM>::H;
  constexpr int PAIRS = AvgShape<DIM>::PAIRS;
  constexpr int SX = D::SX, SY = D::SY;
  size_t const t = (size_t)blockIdx.x * kThreads + threadIdx.x;
  if (t >= (size_t)nlinks * D::NE * PAIRS) return;
  int const r = int(t % PAIRS);
  int const e = int((t / PAIRS) % D::NE);
  alpaca_mr_link const l = links[t / ((size_t)PAIRS * D::NE)];
  if (!link_ok<DIM>(l, nblocks)) return;
  const double *c = blocks + (size_t)l.child * D::BLOCK + (size_t)e * D::FIELD;
  double *p = blocks + (size_t)l.parent * D::BLOCK + (size_t)e * D::FIELD;
  int const x0 = (l.position & 1) ? kTC / 2 : kHS;
  int const y0 = (l.position & 2) ? kTC / 2 : kHS;
  if constexpr (DIM == 2) {
    int const i = r / (H / 2), j = 2 * (r % (H / 2));
    const double *q = c + (kHS + 2 * i) * SX + (kHS + 2 * j) * SY;
    double2 const a0 = *reinterpret_cast<const double2 *>(q);           // (ci,   cj..cj+1)
    double2 const a1 = *reinterpret_cast<const double2 *>(q + 2);       // (ci,   cj+2..cj+3)
    double2 const b0 = *reinterpret_cast<const double2 *>(q + SX);      // (ci+1, cj..cj+1)
    double2 const b1 = *reinterpret_cast<const double2 *>(q + SX + 2);  // (ci+1, cj+2..cj+3)
    double2 out;
    out.x = ((a0.x + b0.y) + (b0.x + a0.y)) * 0.25;
    out.y = ((a1.x + b1.y) + (b1.x + a1.y)) * 0.25;
    *reinterpret_cast<double2 *>(p + (x0 + i) * SX + (y0 + j) * SY) = out;
  } else {
    int const i = r / (H * H / 2), j = (r / (H / 2)) % H, k = 2 * (r % (H / 2));
    int const z0 = (l.position & 4) ? kTC / 2 : kHS;
    const double *q = c + (kHS + 2 * i) * SX + (kHS + 2 * j) * SY + kHS + 2 * k;
    // Rows (dx, dy) of four child cells along k.
    double2 const r00a = *reinterpret_cast<const double2 *>(q);
    double2 const r00b = *reinterpret_cast<const double2 *>(q + 2);
    double2 const r01a = *reinterpret_cast<const double2 *>(q + SY);
    double2 const r01b = *reinterpret_cast<const double2 *>(q + SY + 2);
    double2 const r10a = *reinterpret_cast<const double2 *>(q + SX);
    double2 const r10b = *reinterpret_cast<const double2 *>(q + SX + 2);
    double2 const r11a = *reinterpret_cast<const double2 *>(q + SX + SY);
    double2 const r11b = *reinterpret_cast<const double2 *>(q + SX + SY + 2);
    double2 out;
    out.x = 0.125 * cms4(r00a.x + r11a.y, r00a.y + r11a.x, r01a.x + r10a.y, r01a.y + r10a.x);
    out.y = 0.125 * cms4(r00b.x + r11b.y, r00b.y + r11b.x, r01b.x + r10b.y, r01b.y + r10b.x);
    *reinterpret_cast<double2 *>(p + (x0 + i) * SX + (y0 + j) * SY + z0 + k) = out;
  }
}

// ------------------------------------------------------- jump surfaces

// Multiresolution::AverageJumpBuffer (multiresolution.cpp:47-131) on jump
// surfaces [6][NE][IC][ICZ] per block (SurfaceBuffer, block.h:34-41: East,
// West, North, South, Top, Bottom).  One thread per parent face entry of
// every face a child may touch; a child touches the high face of an axis when
// its bit of that axis is set, the low face otherwise, and covers the quarter
// (half in 2D) of it starting at IC/2 times its bits of the face's transverse
// axes.  The average is ADDED to the parent's value.
template <int DIM>
__global__ __launch_bounds__(kThreads) void average_jump_kernel(double *__restrict__ surfaces,
                                                                int nblocks,
                                                                const alpaca_mr_link *__restrict__ links,
                                                                int nlinks) {
  constexpr int NE = Dims<DIM>::NE;
  constexpr int ICZ = DIM == 3 ? kIC : 1;
  constexpr int HJ = DIM == 3 ? kIC / 2 : 1;      // parent entries along the second index
  constexpr int ENTRIES = NE * (kIC / 2) * HJ;    // per face
  constexpr int FACE = NE * kIC * ICZ;            // doubles per face
  constexpr int BLOCK = 6 * FACE;                 // doubles per block's surfaces
  size_t const t = (size_t)blockIdx.x * kThreads + threadIdx.x;
  if (t >= (size_t)nlinks * DIM * ENTRIES) return;
  int const r = int(t % ENTRIES);
  int const axis = int((t / ENTRIES) % DIM);
  alpaca_mr_link const l = links[t / ((size_t)ENTRIES * DIM)];
  if (!link_ok<DIM>(l, nblocks)) return;
  // The face of this axis the child touches: East/North/Top (2 axis) when its
  // bit is set, West/South/Bottom (2 axis + 1) otherwise.
  int const loc = 2 * axis + (((l.position >> axis) & 1) ? 0 : 1);
  int const t1 = axis == 0 ? 1 : 0, t2 = axis == 2 ? 1 : 2;
  int const s1 = ((l.position >> t1) & 1) * (kIC / 2);
  int const s2 = DIM == 3 ? ((l.position >> t2) & 1) * (kIC / 2) : 0;
  int const e = r / ((kIC / 2) * HJ), i = (r / HJ) % (kIC / 2), j = r % HJ;
  const double *q = surfaces + (size_t)l.child * BLOCK + loc * FACE + (e * kIC + 2 * i) * ICZ +
                    (DIM == 3 ? 2 * j : 0);
  double v;
  if constexpr (DIM == 2)
    v = (q[0] + q[ICZ]) * 0.5;
  else
    v = ((q[0] + q[ICZ + 1]) + (q[ICZ] + q[1])) * 0.25;
  surfaces[(size_t)l.parent * BLOCK + loc * FACE + (e * kIC + s1 + i) * ICZ + s2 + j] += v;
}

// --------------------------------------------------------------- prediction

// Window of parent cells a prediction reads along one axis: the predicted
// parent cells [p0, p0 + n) (n = count / 2, p0 = start / 2 + 2 for the low
// child, start / 2 + TC / 2 - 2 for the high one; PIOLCH/PIOHCH,
// compile_time_constants.h:598-608) and two more on each side.
struct Range {
  int start[3];
  int count[3];  // predicted parent cells per axis (child count / 2)
};

constexpr double kC0 = -22.0 / 128.0, kC1 = 3.0 / 128.0;
constexpr double kC00 = kC0 * kC0, kC01 = kC0 * kC1, kC10 = kC01, kC11 = kC1 * kC1;
constexpr double kC000 = kC00 * kC0, kC001 = kC00 * kC1, kC010 = kC001, kC011 = kC0 * kC11;
constexpr double kC100 = kC001, kC101 = kC011, kC110 = kC011, kC111 = kC1 * kC11;

// The predicted children of a parent cell from its value p and its
// polynomial's terms: out[dx | dy << 1 | dz << 2].
template <int DIM>
__device__ __forceinline__ void form_children(double p, double Qx, double Qy, double Qz, double Qxy,
                                              double Qxz, double Qyz, double Qxyz,
                                              double out[1 << DIM]) {
  out[0] = p + dams<DIM>(Qx, Qy, Qz) + dams<DIM>(Qxy, Qxz, Qyz) + Qxyz;
  out[1] = p + dams<DIM>(-Qx, Qy, Qz) + dams<DIM>(-Qxy, -Qxz, Qyz) - Qxyz;
  out[2] = p + dams<DIM>(Qx, -Qy, Qz) + dams<DIM>(-Qxy, Qxz, -Qyz) - Qxyz;
  out[3] = p + dams<DIM>(-Qx, -Qy, Qz) + dams<DIM>(Qxy, -Qxz, -Qyz) + Qxyz;
  if constexpr (DIM == 3) {
    out[4] = p + cms3(Qx, Qy, -Qz) + cms3(Qxy, -Qxz, -Qyz) - Qxyz;
    out[5] = p + cms3(-Qx, Qy, -Qz) + cms3(-Qxy, Qxz, -Qyz) + Qxyz;
    out[6] = p + cms3(Qx, -Qy, -Qz) + cms3(-Qxy, -Qxz, Qyz) + Qxyz;
    out[7] = p + cms3(-Qx, -Qy, -Qz) + cms3(Qxy, Qxz, Qyz) - Qxyz;
  }
}

// 2D: the predicted children of the parent cell at LDS index `o` of a window.
// The z terms are the reference's zero-initialised Qz, Qxz, Qyz, Qxyz, and
// enter the sums as such (their signs matter for signed zeros).
template <typename L = Lds<2>>
__device__ __forceinline__ void predict_cell(const double *__restrict__ s, int o, double out[4]) {
#define P(a, b) s[o + (a) * L::SX + (b) * L::SY]
  double const Qx = kC0 * (P(1, 0) - P(-1, 0)) + kC1 * (P(2, 0) - P(-2, 0));
  double const Qy = kC0 * (P(0, 1) - P(0, -1)) + kC1 * (P(0, 2) - P(0, -2));
  double const Qxy = (kC00 * ((P(1, 1) + P(-1, -1)) - (P(-1, 1) + P(1, -1))) +
                      kC11 * ((P(2, 2) + P(-2, -2)) - (P(-2, 2) + P(2, -2)))) +
                     (kC01 * ((P(1, 2) + P(-1, -2)) - (P(-1, 2) + P(1, -2))) +
                      kC10 * ((P(2, 1) + P(-2, -1)) - (P(-2, 1) + P(2, -1))));
  form_children<2>(P(0, 0), Qx, Qy, 0.0, Qxy, 0.0, 0.0, 0.0, out);
#undef P
}

// Makes the values be formed here.
__device__ __forceinline__ void formed(double &a, double &b) { asm volatile("" : "+v"(a), "+v"(b)); }

// 3D: the predicted children of the two parent cells at LDS indices o and
// o + 1 (o even).  Both stencils lie in 25 rows of six values along z, each read
// once by three 16-byte accesses, in the order in which the terms use them: 600
// bytes of LDS a cell.  The fences make the compiler form a group's results
// before the next group's rows are read (it moves both otherwise, and 100
// registers spill).
// (A thread per cell read 125 values, 1000 bytes, as
// 8-byte accesses: LDS-bound, 7600 cycles per wavefront of cells where the 428
// FP64 instructions issue in 1700.)
template <typename L>
__device__ __forceinline__ void predict_pair(const double *__restrict__ s, int o,
                                             double (&out)[2][8]) {
  struct Row {
    double v[6];
    __device__ __forceinline__ Row(const double *q) {
      double2 const a = reinterpret_cast<const double2 *>(q)[0];
      double2 const b = reinterpret_cast<const double2 *>(q)[1];
      double2 const c = reinterpret_cast<const double2 *>(q)[2];
      v[0] = a.x, v[1] = a.y, v[2] = b.x, v[3] = b.y, v[4] = c.x, v[5] = c.y;
    }
  };
  auto row = [s, o](int a, int b) { return Row(s + (o - 2 + a * L::SX + b * L::SY)); };
  double Qx[2], Qy[2], Qz[2], Qxy[2], Qxz[2], Qyz[2], Qxyz[2], p[2];
  {
    // The four antisymmetric differences over the corners (+-a, +-b, +-c),
    // c = 1, 2, and the diagonal difference of the rows (+-a, +-b).
    struct Corner {
      double g[2][2], d[2];
    };
    auto corner = [&row](int a, int b) {
      Row const pp = row(a, b), mm = row(-a, -b), mp = row(-a, b), pm = row(a, -b);
      Corner k;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        int const z = n + 2;
        k.d[n] = (pp.v[z] + mm.v[z]) - (mp.v[z] + pm.v[z]);
#pragma unroll
        for (int c = 1; c <= 2; ++c)
          k.g[n][c - 1] = cms4(pp.v[z + c] - mm.v[z - c], mm.v[z + c] - pp.v[z - c],
                               pm.v[z - c] - mp.v[z + c], mp.v[z - c] - pm.v[z + c]);
      }
#pragma unroll
      for (int n = 0; n < 2; ++n) formed(k.g[n][0], k.g[n][1]), formed(k.d[n], k.g[n][1]);
      __builtin_amdgcn_sched_barrier(0);
      return k;
    };
    double q0[2], q1[2], xy[2];
    {
      Corner const k11 = corner(1, 1);
      Corner const k22 = corner(2, 2);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        xy[n] = kC00 * k11.d[n] + kC11 * k22.d[n];
        q0[n] = kC000 * k11.g[n][0] + kC111 * k22.g[n][1];
        q1[n] = kC001 * k11.g[n][1] + kC110 * k22.g[n][0];
      }
    }
    Corner const k12 = corner(1, 2);
    Corner const k21 = corner(2, 1);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      Qxy[n] = xy[n] + (kC01 * k12.d[n] + kC10 * k21.d[n]);
      Qxyz[n] = cms4(q0[n], q1[n], kC011 * k12.g[n][1] + kC100 * k21.g[n][0],
                     kC010 * k12.g[n][0] + kC101 * k21.g[n][1]);
    }
  }
  // The planes of an axis and z.
  auto plane = [&row](int a, int b, double (&Q)[2], double (&Qd)[2]) {
    Row const p1 = row(a, b), m1 = row(-a, -b), p2 = row(2 * a, 2 * b), m2 = row(-2 * a, -2 * b);
    auto diag = [](const Row &p, const Row &m, int z, int c) {
      return (p.v[z + c] + m.v[z - c]) - (m.v[z + c] + p.v[z - c]);
    };
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      int const z = n + 2;
      Q[n] = kC0 * (p1.v[z] - m1.v[z]) + kC1 * (p2.v[z] - m2.v[z]);
      Qd[n] = (kC00 * diag(p1, m1, z, 1) + kC11 * diag(p2, m2, z, 2)) +
              (kC01 * diag(p1, m1, z, 2) + kC10 * diag(p2, m2, z, 1));
      formed(Q[n], Qd[n]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  plane(1, 0, Qx, Qxz);
  plane(0, 1, Qy, Qyz);
  Row const line = row(0, 0);
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    int const z = n + 2;
    Qz[n] = kC0 * (line.v[z + 1] - line.v[z - 1]) + kC1 * (line.v[z + 2] - line.v[z - 2]);
    p[n] = line.v[z];
    form_children<3>(p[n], Qx[n], Qy[n], Qz[n], Qxy[n], Qxz[n], Qyz[n], Qxyz[n], out[n]);
  }
}

// Window geometry of one link: first parent cell of the window per axis and
// its extent (at most 16).
template <int DIM> struct Window {
  int p0[3];  // first window cell (predicted cell - 2) per axis
  int w[3];   // window extent per axis
  __device__ Window(const Range &r, int position) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      int const off = ((position >> a) & 1) ? kTC / 2 - kHS / 2 : kHS / 2;
      bool const live = a < DIM;
      p0[a] = live ? r.start[a] / 2 + off - 2 : 0;
      w[a] = live ? r.count[a] + 4 : 1;
    }
  }
  // LDS index of predicted parent cell (a, b, c) (counted from the range's
  // first predicted cell).
  template <typename L = Lds<DIM>> __device__ static int centre(int a, int b, int c) {
    return (a + 2) * L::SX + (b + 2) * L::SY + (DIM == 3 ? c + 2 : 0);
  }
};

// One 2D field's parent window into LDS.
__device__ __forceinline__ void stage_window2(double *s, const double *__restrict__ field,
                                              const Window<2> &win) {
  using D = Dims<2>;
  for (int t = threadIdx.x; t < win.w[0] * win.w[1]; t += kStencilThreads) {
    int const a = t / win.w[1], b = t % win.w[1];
    s[a * Lds<2>::SX + b * Lds<2>::SY] = field[(win.p0[0] + a) * D::SX + (win.p0[1] + b) * D::SY];
  }
}

// Child cells (2a + dx, 2b + dy, 2c + dz) from `q`, the child's cell
// (2a, 2b, 2c): the two cells adjacent along the fastest axis (dz in 3D, dy in
// 2D) are one 16-byte access (the offset is even: aligned).
template <int DIM> __device__ __forceinline__ void store_children(double *q, const double v[1 << DIM]) {
  using D = Dims<DIM>;
  if constexpr (DIM == 3) {
    *reinterpret_cast<double2 *>(q) = make_double2(v[0], v[4]);
    *reinterpret_cast<double2 *>(q + D::SX) = make_double2(v[1], v[5]);
    *reinterpret_cast<double2 *>(q + D::SY) = make_double2(v[2], v[6]);
    *reinterpret_cast<double2 *>(q + D::SX + D::SY) = make_double2(v[3], v[7]);
  } else {
    *reinterpret_cast<double2 *>(q) = make_double2(v[0], v[2]);
    *reinterpret_cast<double2 *>(q + D::SX) = make_double2(v[1], v[3]);
  }
}
template <int DIM> __device__ __forceinline__ void load_children(const double *q, double x[1 << DIM]) {
  using D = Dims<DIM>;
  if constexpr (DIM == 3) {
    double2 const a = *reinterpret_cast<const double2 *>(q);
    double2 const b = *reinterpret_cast<const double2 *>(q + D::SX);
    double2 const c = *reinterpret_cast<const double2 *>(q + D::SY);
    double2 const d = *reinterpret_cast<const double2 *>(q + D::SX + D::SY);
    x[0] = a.x, x[4] = a.y, x[1] = b.x, x[5] = b.y, x[2] = c.x, x[6] = c.y, x[3] = d.x, x[7] = d.y;
  } else {
    double2 const a = *reinterpret_cast<const double2 *>(q);
    double2 const b = *reinterpret_cast<const double2 *>(q + D::SX);
    x[0] = a.x, x[2] = a.y, x[1] = b.x, x[3] = b.y;
  }
}

// 2D: predicts range r (at most 8 predicted parent cells per axis) of every
// equation of child l.child from its parent, in one workgroup of a wavefront per
// equation: each loads its field's window (at most 144 cells) and predicts at most
// one parent cell per lane.  The caller's early exits are uniform over the
// workgroup.  12,000 links' internal cells 40 us, halo slabs 36 us; 56 and 71
// with a workgroup walking the equations, a barrier each.
constexpr int kPredict2Threads = 64 * Dims<2>::NE;
using Lds2 = LdsW<2, 12>;

__device__ __forceinline__ void predict_range2(double *s, double *__restrict__ blocks,
                                               const alpaca_mr_link &l, const Range &r) {
  using D = Dims<2>;
  Window<2> const win(r, l.position);
  int const e = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double *w = s + e * Lds2::SIZE;
  const double *field = blocks + (size_t)l.parent * D::BLOCK + (size_t)e * D::FIELD;
  int const n = win.w[0] * win.w[1];
  constexpr int K = (Lds2::SIZE + 63) / 64;
  double v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    int const t = lane + 64 * k;
    if (t < n) v[k] = field[(win.p0[0] + t / win.w[1]) * D::SX + (win.p0[1] + t % win.w[1]) * D::SY];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    int const t = lane + 64 * k;
    if (t < n) w[(t / win.w[1]) * Lds2::SX + (t % win.w[1]) * Lds2::SY] = v[k];
  }
  __syncthreads();
  if (lane >= r.count[0] * r.count[1]) return;
  int const a = lane / r.count[1], b = lane % r.count[1];
  double c[4];
  predict_cell<Lds2>(w, Window<2>::centre<Lds2>(a, b, 0), c);
  store_children<2>(blocks + (size_t)l.child * D::BLOCK + (size_t)e * D::FIELD +
                        (r.start[0] + 2 * a) * D::SX + (r.start[1] + 2 * b) * D::SY,
                    c);
}

// Ranges whose window fits the 12-cell layout: at most 8 predicted parent
// cells per axis.
__host__ __device__ inline bool small_window(const Range &r) {
  return r.count[0] <= 8 && r.count[1] <= 8 && r.count[2] <= 8;
}

// 2D ranges with small windows: one workgroup per link, every equation.
__global__ __launch_bounds__(kPredict2Threads) void prediction2_kernel(
    double *__restrict__ blocks, int nblocks, const alpaca_mr_link *__restrict__ links, Range r) {
  __shared__ double s[Dims<2>::NE * Lds2::SIZE];
  alpaca_mr_link const l = links[blockIdx.x];
  if (!link_ok<2>(l, nblocks)) return;
  predict_range2(s, blocks, l, r);
}

// 2D ranges with larger windows: one workgroup per (link, equation).  FULL: the whole
// block (12 predicted parent cells per axis, known at compile time).
template <bool FULL>
__global__ __launch_bounds__(kStencilThreads) __attribute__((amdgpu_waves_per_eu(4, 8))) void prediction2_range_kernel(
    double *__restrict__ blocks, int nblocks, const alpaca_mr_link *__restrict__ links, Range r) {
  using D = Dims<2>;
  __shared__ double s[Lds<2>::SIZE];
  if constexpr (FULL) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      r.start[a] = 0;
      r.count[a] = kTC / 2;
    }
  }
  int const e = blockIdx.x % D::NE;
  alpaca_mr_link const l = links[blockIdx.x / D::NE];
  if (!link_ok<2>(l, nblocks)) return;  // uniform over the workgroup
  stage_window2(s, blocks + (size_t)l.parent * D::BLOCK + (size_t)e * D::FIELD,
                Window<2>(r, l.position));
  __syncthreads();
  double *child = blocks + (size_t)l.child * D::BLOCK + (size_t)e * D::FIELD;
  for (int t = threadIdx.x; t < r.count[0] * r.count[1]; t += kStencilThreads) {
    int const a = t / r.count[1], b = t % r.count[1];
    double v[4];
    predict_cell(s, Window<2>::centre(a, b, 0), v);
    store_children<2>(child + (r.start[0] + 2 * a) * D::SX + (r.start[1] + 2 * b) * D::SY, v);
  }
}

// The halo slab of a location (CommunicationTypes::GetStartIndicesHaloRecv and
// GetHaloSize, communication_types.h:76-132,190-197): per axis, direction +1
// gives the cells [IC+HS, TC), -1 gives [0, HS), 0 the internal cells
// [HS, HS+IC) (in 2D the single z cell).  False for a location outside the
// enum or, in 2D, one with a Top/Bottom part.
template <int DIM> __device__ __forceinline__ bool location_range(int loc, Range &r) {
  if (loc < 0 || loc >= 26) return false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    int const d = kLocationDir[loc][a];
    if (DIM == 2 && a == 2) {
      if (d != 0) return false;
      r.start[2] = 0;
      r.count[2] = 1;
    } else {
      r.start[a] = d > 0 ? kIC + kHS : (d < 0 ? 0 : kHS);
      r.count[a] = (d != 0 ? kHS : kIC) / 2;
    }
  }
  return true;
}

// UpdateMaterialJumpNoMpi (internal_halo_manager.cpp:231-262) for a batch:
// link i's child gets the halo slab of location locations[i] predicted from
// its parent (every equation), one workgroup per link.
__global__ __launch_bounds__(kPredict2Threads) void jump_halo2_kernel(
    double *__restrict__ blocks, int nblocks, const alpaca_mr_link *__restrict__ links,
    const int *__restrict__ locations) {
  __shared__ double s[Dims<2>::NE * Lds2::SIZE];
  alpaca_mr_link const l = links[blockIdx.x];
  Range r;
  if (!link_ok<2>(l, nblocks) || !location_range<2>(locations[blockIdx.x], r)) return;
  predict_range2(s, blocks, l, r);
}

// ------------------------------------------------------------ 3D predictions

// Quotients of numbers below 4096 by a divisor up to 256 that is the same for
// the whole workgroup: n * ceil(2^21 / d) >> 21 is exact there, both factors fit
// 24 bits, and the product 32 where n < 4096 and d >= 5, or n < 1024.
struct SmallDiv {
  unsigned d, m;
  __device__ __forceinline__ explicit SmallDiv(int by)
      : d((unsigned)by), m(((1u << 21) + d - 1) / d) {}
  __device__ __forceinline__ int quotient(int n) const { return int(__umul24((unsigned)n, m) >> 21); }
};

// One field's parent window of NT threads into LDS (layout L).  N > 0: the
// window of N predicted parent cells per axis.  Loads are issued eight at a time.
template <int NT, int N, typename L>
__device__ __forceinline__ void stage_window3(double *s, const double *__restrict__ field,
                                              const Window<3> &win, int tid) {
  using D = Dims<3>;
  int const w1 = N ? N + 4 : win.w[1], w2 = N ? N + 4 : win.w[2];
  int const n = N ? (N + 4) * (N + 4) * (N + 4) : win.w[0] * w1 * w2;
  SmallDiv const by2(w2), by1(w1);
  const double *base = field + win.p0[0] * D::SX + win.p0[1] * D::SY + win.p0[2];
  constexpr int K = 8;
  for (int first = tid; first < n; first += K * NT) {
    double v[K];
    int to[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      int const t = first + k * NT;
      int const row = N ? t / (N + 4) : by2.quotient(t);
      int const a = N ? row / (N + 4) : by1.quotient(row);
      int const b = row - a * w1, c = t - row * w2;
      to[k] = a * L::SX + b * L::SY + c;
      if (t < n) v[k] = base[a * D::SX + b * D::SY + c];
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (first + k * NT < n) s[to[k]] = v[k];
  }
}

// Children of a pair of parent cells (c even) from `q`, the child's cell
// (2a, 2b, 2c): four adjacent doubles per row, or the first two alone.
__device__ __forceinline__ void store_pair(double *q, const double (&v)[2][8], bool second) {
  store_children<3>(q, v[0]);
  if (second) store_children<3>(q + 2, v[1]);
}

// One field of one link by NT threads: the window into s, then the pairs of
// predicted parent cells along z.  N > 0: N predicted cells per axis.
template <int NT, int W, int N, typename F>
__device__ __forceinline__ void for_pairs(const Range &r, int tid, const F &f) {
  using L = LdsW<3, W>;
  int const c1 = N ? N : r.count[1], pz = N ? N / 2 : (r.count[2] + 1) / 2;
  int const tasks = N ? N * N * (N / 2) : r.count[0] * c1 * pz;
  SmallDiv const byz(pz), byy(c1);
  for (int t = tid; t < tasks; t += NT) {
    int a, b, c;
    if constexpr (N == 8 && W == 12) {
      // Four threads read 16 consecutive banks of a window row; rows b and b + 2
      // and planes a and a + 1 of this layout lie 16 and 32 banks further, so a
      // quarter wavefront of these four rows reads without bank conflicts.
      c = 2 * (t & 3);
      b = ((t >> 2) & 1) * 2 + ((t >> 4) & 1) + ((t >> 5) & 1) * 4;
      a = ((t >> 3) & 1) + 2 * (t >> 6);
    } else {
      int const q = N ? t / (N / 2) : byz.quotient(t);
      a = N ? q / N : byy.quotient(q);
      b = q - a * c1;
      c = 2 * (t - q * pz);
    }
    f(a, b, c, Window<3>::template centre<L>(a, b, c));
  }
}

template <int NT, int W, int N, bool EDGES = false>
__device__ __forceinline__ void predict_field3(double *s, double *__restrict__ blocks,
                                               const alpaca_mr_link &l, int e, const Range &r,
                                               int tid) {
  using D = Dims<3>;
  using L = LdsW<3, W>;
  Window<3> const win(r, l.position);
  double *child = blocks + (size_t)l.child * D::BLOCK + (size_t)e * D::FIELD;
  // EDGES: the internal cells of a child row cover its first and last 64-byte segment
  // in part, and a partial write of a segment that is in no cache is a
  // read-modify-write in memory, so both are read first (the values are not used).
  double edge[2];
  if constexpr (EDGES) {
    static_assert(N == 8 && NT == kIC * kIC, "one child row per thread");
    const double *q = child + (kHS + tid / kIC) * D::SX + (kHS + tid % kIC) * D::SY;
    edge[0] = q[0];
    edge[1] = q[kTC - 1];
  }
  stage_window3<NT, N, L>(s, blocks + (size_t)l.parent * D::BLOCK + (size_t)e * D::FIELD, win, tid);
  if constexpr (EDGES) asm volatile("" ::"v"(edge[0]), "v"(edge[1]));
  __syncthreads();
  for_pairs<NT, W, N>(r, tid, [&](int a, int b, int c, int o) {
    double v[2][8];
    predict_pair<L>(s, o, v);
    store_pair(child + (r.start[0] + 2 * a) * D::SX + (r.start[1] + 2 * b) * D::SY + r.start[2] + 2 * c,
               v, c + 1 < r.count[2]);
  });
}

// One workgroup per (link, equation), the equations and siblings of a parent
// on one XCD.  N = 8 (the internal cells): 256 threads, one pair each; N = 12 (the
// whole block): 448 threads, two each; N = 0: any other of at most 8 cells per axis.
// A workgroup stages one field, so others' arithmetic covers its loads.  Bound by the
// writes: without them 2560 links' internal cells take 118 us.
template <int W, int N> constexpr int kPredictThreads = W == 12 ? 256 : 448;

// Links whose children's internal rows (16 x 16 of three 64-byte segments, five
// equations) fill the 256 MB memory-side cache.  Above, a row's edges are read first:
// 2400 links 329 us without, 285 us with, warm, and 1600 links 212 and 194 cold (2560 as
// whole rows would take 177).  Below, the reads only add to the writes: 960 links 66
// without, 97 with, warm, and 124 and 126 cold, 320 links 27 and 36, and 36 and 43.
constexpr int kEdgeLinks = (256 << 20) / (5 * kIC * kIC * 192);

template <int W, int N, bool EDGES = false>
__global__ __launch_bounds__((kPredictThreads<W, N>)) __attribute__((amdgpu_waves_per_eu(4, 8))) void prediction3_kernel(
    double *__restrict__ blocks, int nblocks, const alpaca_mr_link *__restrict__ links, Range r) {
  constexpr int NE = Dims<3>::NE;
  __shared__ __align__(16) double s[LdsW<3, W>::SIZE];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  alpaca_mr_link const l = links[g / NE];
  if (!link_ok<3>(l, nblocks)) return;
  if constexpr (N > 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) r.count[a] = N;
  }
  predict_field3<kPredictThreads<W, N>, W, N, EDGES>(s, blocks, l, int(g % NE), r, threadIdx.x);
}

// Ranges of more than 8 predicted cells along an axis, but for the whole block: as
// prediction3_kernel, with LDS for the part of the layout that the range's window
// reaches.  A range of few pairs is one load, one barrier and one pair deep, and what
// counts is how many of its workgroups a CU holds: with the whole layout (32 KB) and
// 448 threads it held two.  960 links, us, with a workgroup of 192 threads a thread per
// cell, with 448 threads, and so: 1 x 1 x 12 parent cells 23.4, 37.0, 20.2, 2 x 2 x 12 25.9,
// 36.9, 19.2, 4 x 4 x 12 45.2, 47.7, 33.8, 9 x 9 x 9 190, 141, 148, 11 x 11 x 11 279, 208, 218.
constexpr int kRangeThreads = 256;
constexpr size_t range_lds_bytes(const Range &r) {
  return sizeof(double) *
         ((r.count[0] + 3) * Lds<3>::SX + (r.count[1] + 3) * Lds<3>::SY + Lds<3>::SY);
}

__global__ __launch_bounds__(kRangeThreads) __attribute__((amdgpu_waves_per_eu(4, 8))) void prediction3_range_kernel(
    double *__restrict__ blocks, int nblocks, const alpaca_mr_link *__restrict__ links, Range r) {
  constexpr int NE = Dims<3>::NE;
  extern __shared__ __align__(16) double window[];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  alpaca_mr_link const l = links[g / NE];
  if (!link_ok<3>(l, nblocks)) return;
  predict_field3<kRangeThreads, 16, 0>(window, blocks, l, int(g % NE), r, threadIdx.x);
}

// The jump halos of 3D links (jump_halo2_kernel in 2D): a slab has at most 64 pairs of
// parent cells, so one wavefront per (link, equation).
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) void jump_halo3_kernel(double *__restrict__ blocks, int nblocks,
                                                        const alpaca_mr_link *__restrict__ links,
                                                        const int *__restrict__ locations) {
  constexpr int NE = Dims<3>::NE;
  __shared__ __align__(16) double s[LdsW<3, 12>::SIZE];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  alpaca_mr_link const l = links[g / NE];
  Range r;
  if (!link_ok<3>(l, nblocks) || !location_range<3>(locations[g / NE], r)) return;
  predict_field3<64, 12, 0>(s, blocks, l, int(g % NE), r, threadIdx.x);
}

// ------------------------------------------------------------------ details

struct Thresholds {
  double eps[kMaxLevels];  // coarsening threshold per level
  int nlevels;
};

// One workgroup per link: over Mass and Energy (the wavelet equations,
// field_setup.h:243-247) and every child cell, halo included, the relative
// detail between the child and the parent's prediction over the whole block,
// ChildNeedsRemeshing<N> (multiresolution.cpp:299-398):
//   NORM 0 (Linfinity): the largest |exact - predicted| / |exact|;
//   NORM 1 (Lone): per equation the sum of |exact - predicted| / |exact|
//                  times 1/(TC^2 TCZ), the largest over the equations;
//   NORM 2 (Ltwo): per equation sqrt(sum of ((exact - predicted)/exact)^2)
//                  times 1/(TC^2 TCZ), the largest over the equations.
// std::max(max_detail, x) drops a NaN x, so every running maximum is a
// non-NaN value >= +0 and the hardware maximum (which skips a NaN operand)
// picks the same value; for L-infinity the order of the reduction does not
// matter (the quotients of absolute values are never -0).  The L-one and
// L-two sums are reduced as a tree (lanes, then waves) instead of the
// reference's cell order: they agree to rounding, and a NaN or infinite term
// gives a NaN or infinite sum either way.
// The two fields' windows are staged together (64 KB in 3D, two workgroups of
// seven wavefronts per CU: 3456 children in two pairs of parent cells a thread
// and field, 96% of the threads at work); a pair's child cells are read before its
// prediction is formed.
template <int DIM> constexpr int kDetailThreads = DIM == 3 ? 448 : 192;

// A child's relative detail between its value x and the prediction v.
template <int NORM> __device__ __forceinline__ void add_detail(double x, double v, double &m, double &acc) {
  if constexpr (NORM == 0) {
    m = __builtin_fmax(m, __builtin_fabs(x - v) / __builtin_fabs(x));
  } else if constexpr (NORM == 1) {
    acc += __builtin_fabs(x - v) / __builtin_fabs(x);
  } else {
    double const q = (x - v) / x;
    acc = acc + q * q;
  }
}

template <int DIM, int NORM>
__global__ __launch_bounds__(kDetailThreads<DIM>) __attribute__((amdgpu_waves_per_eu(4, 8))) void details_kernel(
    const double *__restrict__ blocks, int nblocks, const alpaca_mr_link *__restrict__ links,
    Thresholds th, double *__restrict__ details, int *__restrict__ decisions) {
  using D = Dims<DIM>;
  constexpr int NT = kDetailThreads<DIM>;
  constexpr int H = kTC / 2;
  constexpr int kWaves = NT / 64;
  constexpr double kOneNumberOfCells = 1.0 / double(kTC * kTC * D::TZ);
  __shared__ __align__(16) double s[2][Lds<DIM>::SIZE];
  __shared__ double part[2][kWaves];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  alpaca_mr_link const l = links[g];
  if (!link_ok<DIM>(l, nblocks)) {
    if (threadIdx.x == 0) {
      details[g] = __builtin_nan("");
      if (decisions) decisions[g] = -1;
    }
    return;
  }
  Range const full{{0, 0, 0}, {H, H, DIM == 3 ? H : 1}};
  Window<DIM> const win(full, l.position);
#pragma unroll
  for (int e = kMass; e <= kEnergy; ++e) {
    const double *field = blocks + (size_t)l.parent * D::BLOCK + (size_t)e * D::FIELD;
    if constexpr (DIM == 3)
      stage_window3<NT, H, Lds<3>>(s[e], field, win, threadIdx.x);
    else
      stage_window2(s[e], field, win);
  }
  __syncthreads();
  double m = 0.0;
#pragma unroll 1
  for (int e = kMass; e <= kEnergy; ++e) {
    const double *child = blocks + (size_t)l.child * D::BLOCK + (size_t)e * D::FIELD;
    double acc = 0.0;
    if constexpr (DIM == 3) {
      for_pairs<NT, 16, H>(full, threadIdx.x, [&](int a, int b, int c, int o) {
        const double *q = child + 2 * a * D::SX + 2 * b * D::SY + 2 * c;
        double x[2][8], v[2][8];
        load_children<3>(q, x[0]);
        load_children<3>(q + 2, x[1]);
        predict_pair<Lds<3>>(s[e], o, v);
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int n = 0; n < 8; ++n) add_detail<NORM>(x[k][n], v[k][n], m, acc);
      });
    } else {
      for (int t = threadIdx.x; t < H * H; t += NT) {
        int const a = t / H, b = t % H;
        double x[4], v[4];
        predict_cell(s[e], Window<2>::centre(a, b, 0), v);
        load_children<2>(child + 2 * a * D::SX + 2 * b * D::SY, x);
#pragma unroll
        for (int n = 0; n < 4; ++n) add_detail<NORM>(x[n], v[n], m, acc);
      }
    }
    if constexpr (NORM != 0) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
      if ((threadIdx.x & 63) == 0) part[e][threadIdx.x >> 6] = acc;
    }
  }
  if constexpr (NORM == 0) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = __builtin_fmax(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) part[0][threadIdx.x >> 6] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if constexpr (NORM == 0) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) m = __builtin_fmax(part[0][w], m);
    } else {
#pragma unroll
      for (int e = kMass; e <= kEnergy; ++e) {
        double sum = part[e][0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) sum += part[e][w];
        double const val =
            NORM == 1 ? sum * kOneNumberOfCells : __builtin_sqrt(sum) * kOneNumberOfCells;
        m = __builtin_fmax(m, val);
      }
    }
    details[g] = m;
    if (decisions) {
      int dec = -1;
      if (l.level >= 0 && l.level < th.nlevels) {
        // RemeshingDecision (multiresolution.cpp:408-428): Coarse 2,
        // Refine 1, Neutral 0 (remesh_identifier.h:29).
        double const eps_coarsen = th.eps[l.level];
        double const eps_refine = eps_coarsen * 32.0;
        dec = m <= eps_coarsen ? 2 : (m >= eps_refine ? 1 : 0);
      }
      decisions[g] = dec;
    }
  }
}

int hip_status(hipError_t e) { return e == hipSuccess ? ALPACA_OK : ALPACA_ERR_HIP; }

bool bad_sizes(int dim, int nblocks, int nlinks) {
  return (dim != 2 && dim != 3) || nblocks < 1 || nblocks > kMaxBlocks || nlinks < 0 ||
         nlinks > kMaxBlocks;
}

template <int DIM> int average_impl(double *blocks, int nblocks, const alpaca_mr_link *links,
                                    int nlinks, hipStream_t s) {
  size_t const total = (size_t)nlinks * Dims<DIM>::NE * AvgShape<DIM>::PAIRS;
  dim3 grid((unsigned)((total + kThreads - 1) / kThreads));
  hipLaunchKernelGGL((average_kernel<DIM>), grid, dim3(kThreads), 0, s, blocks, nblocks, links, nlinks);
  return hip_status(hipGetLastError());
}

template <int DIM> int average_jump_impl(double *surfaces, int nblocks, const alpaca_mr_link *links,
                                         int nlinks, hipStream_t s) {
  size_t const total = (size_t)nlinks * DIM * Dims<DIM>::NE * (kIC / 2) * (DIM == 3 ? kIC / 2 : 1);
  dim3 grid((unsigned)((total + kThreads - 1) / kThreads));
  hipLaunchKernelGGL((average_jump_kernel<DIM>), grid, dim3(kThreads), 0, s, surfaces, nblocks, links,
                     nlinks);
  return hip_status(hipGetLastError());
}

// f(first, n) over all links in launches of at most as many as the hardware can count
// the threads of (below 2^32), `threads` a link.
template <typename F> void in_launches(int nlinks, int threads, const F &f) {
  int const most = int(0xffffffffu / (unsigned)threads);
  for (long long first = 0; first < nlinks; first += most)
    f(int(first), (int)std::min<long long>(most, nlinks - first));
}

template <int DIM> int prediction_impl(double *blocks, int nblocks, const alpaca_mr_link *links,
                                       int nlinks, const Range &r, hipStream_t s) {
  constexpr int NE = Dims<DIM>::NE;
  auto all = [&r](int n) {
    return r.count[0] == n && r.count[1] == n && r.count[2] == (DIM == 3 ? n : 1);
  };
  // `groups` workgroups of nt threads and lds bytes per link.
  auto launch = [&](auto kernel, int groups, int nt, size_t lds = 0) {
    in_launches(nlinks, groups * nt, [&](int first, int n) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)n * groups), dim3(nt), lds, s, blocks, nblocks,
                         links + first, r);
    });
  };
  if constexpr (DIM == 3) {
    if (all(8) && r.start[0] == kHS && r.start[1] == kHS && r.start[2] == kHS)
      launch(nlinks > kEdgeLinks ? prediction3_kernel<12, 8, true> : prediction3_kernel<12, 8>, NE,
             kPredictThreads<12, 8>);
    else if (all(12))
      launch(prediction3_kernel<16, 12>, NE, kPredictThreads<16, 12>);
    else if (small_window(r))
      launch(prediction3_kernel<12, 0>, NE, kPredictThreads<12, 0>);
    else
      launch(prediction3_range_kernel, NE, kRangeThreads, range_lds_bytes(r));
  } else if (small_window(r)) {
    launch(prediction2_kernel, 1, kPredict2Threads);
  } else if (all(12)) {
    launch(prediction2_range_kernel<true>, NE, kStencilThreads);
  } else {
    launch(prediction2_range_kernel<false>, NE, kStencilThreads);
  }
  return hip_status(hipGetLastError());
}

template <int DIM> int jump_halo_impl(double *blocks, int nblocks, const alpaca_mr_link *links,
                                      const int *locations, int nlinks, hipStream_t s) {
  constexpr int groups = DIM == 3 ? Dims<3>::NE : 1, nt = DIM == 3 ? 64 : kPredict2Threads;
  in_launches(nlinks, groups * nt, [&](int first, int n) {
    hipLaunchKernelGGL(DIM == 3 ? jump_halo3_kernel : jump_halo2_kernel, dim3((unsigned)n * groups),
                       dim3(nt), 0, s, blocks, nblocks, links + first, locations + first);
  });
  return hip_status(hipGetLastError());
}

template <int DIM> int details_impl(const double *blocks, int nblocks, const alpaca_mr_link *links,
                                    int nlinks, int norm, const Thresholds &th, double *details,
                                    int *decisions, hipStream_t s) {
  auto kernel = norm == ALPACA_MR_NORM_L1   ? details_kernel<DIM, 1>
                : norm == ALPACA_MR_NORM_L2 ? details_kernel<DIM, 2>
                                            : details_kernel<DIM, 0>;
  in_launches(nlinks, kDetailThreads<DIM>, [&](int first, int n) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(kDetailThreads<DIM>), 0, s, blocks, nblocks,
                       links + first, th, details + first, decisions ? decisions + first : nullptr);
  });
  return hip_status(hipGetLastError());
}

}  // namespace
}  // namespace mr
}  // namespace alpaca

using namespace alpaca;

extern "C" {

int alpaca_mr_average(int dim, double *d_blocks, int nblocks, const alpaca_mr_link *d_links,
                      int nlinks, void *stream) {
  if (mr::bad_sizes(dim, nblocks, nlinks) || !d_blocks || (nlinks > 0 && !d_links))
    return ALPACA_ERR_INVALID;
  if (reinterpret_cast<uintptr_t>(d_blocks) % 16) return ALPACA_ERR_INVALID;  // 16-byte accesses
  if (nlinks == 0) return ALPACA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dim == 2) return mr::average_impl<2>(d_blocks, nblocks, d_links, nlinks, s);
  return mr::average_impl<3>(d_blocks, nblocks, d_links, nlinks, s);
}

int alpaca_mr_average_jump_buffers(int dim, double *d_surfaces, int nblocks,
                                   const alpaca_mr_link *d_links, int nlinks, void *stream) {
  if (mr::bad_sizes(dim, nblocks, nlinks) || !d_surfaces ||
      (nlinks > 0 && !d_links))
    return ALPACA_ERR_INVALID;
  if (nlinks == 0) return ALPACA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dim == 2) return mr::average_jump_impl<2>(d_surfaces, nblocks, d_links, nlinks, s);
  return mr::average_jump_impl<3>(d_surfaces, nblocks, d_links, nlinks, s);
}

int alpaca_mr_prediction(int dim, double *d_blocks, int nblocks, const alpaca_mr_link *d_links,
                         int nlinks, const int *range, void *stream) {
  if (mr::bad_sizes(dim, nblocks, nlinks) || !d_blocks || !range ||
      (nlinks > 0 && !d_links))
    return ALPACA_ERR_INVALID;
  if (reinterpret_cast<uintptr_t>(d_blocks) % 16) return ALPACA_ERR_INVALID;  // 16-byte accesses
  mr::Range r{{0, 0, 0}, {1, 1, 1}};
  for (int a = 0; a < dim; ++a) {
    int const start = range[2 * a], count = range[2 * a + 1];
    // Even start (the reference's own precondition, multiresolution.cpp:154-
    // 159) and inside the block: every parent cell read, start / 2 + 2 - 2 up
    // to start / 2 + count / 2 + TC / 2 - 2 + 1, then lies in [0, TC).
    if (start < 0 || count < 0 || (start & 1) || start + count > kTC) return ALPACA_ERR_INVALID;
    r.start[a] = start;
    r.count[a] = count / 2;
  }
  if (nlinks == 0 || r.count[0] == 0 || r.count[1] == 0 || r.count[2] == 0)
    return ALPACA_OK;  // nothing to predict
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dim == 2) return mr::prediction_impl<2>(d_blocks, nblocks, d_links, nlinks, r, s);
  return mr::prediction_impl<3>(d_blocks, nblocks, d_links, nlinks, r, s);
}

int alpaca_mr_jump_halo_update(int dim, double *d_blocks, int nblocks,
                               const alpaca_mr_link *d_links, const int *d_locations, int nlinks,
                               void *stream) {
  if (mr::bad_sizes(dim, nblocks, nlinks) || !d_blocks ||
      (nlinks > 0 && (!d_links || !d_locations)))
    return ALPACA_ERR_INVALID;
  if (reinterpret_cast<uintptr_t>(d_blocks) % 16) return ALPACA_ERR_INVALID;  // 16-byte accesses
  if (nlinks == 0) return ALPACA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dim == 2) return mr::jump_halo_impl<2>(d_blocks, nblocks, d_links, d_locations, nlinks, s);
  return mr::jump_halo_impl<3>(d_blocks, nblocks, d_links, d_locations, nlinks, s);
}

int alpaca_mr_child_needs_remeshing(int dim, const double *d_blocks, int nblocks,
                                    const alpaca_mr_link *d_links, int nlinks, int norm,
                                    const double *eps_coarsen, int nlevels, double *d_details,
                                    int *d_decisions, void *stream) {
  if (mr::bad_sizes(dim, nblocks, nlinks) || !d_blocks ||
      (norm != ALPACA_MR_NORM_LINF && norm != ALPACA_MR_NORM_L1 && norm != ALPACA_MR_NORM_L2) ||
      (nlinks > 0 && (!d_links || !d_details)) || nlevels < 0 || nlevels > mr::kMaxLevels ||
      (nlevels > 0 && !eps_coarsen) || (d_decisions && nlevels == 0))
    return ALPACA_ERR_INVALID;
  if (reinterpret_cast<uintptr_t>(d_blocks) % 16) return ALPACA_ERR_INVALID;  // 16-byte accesses
  if (nlinks == 0) return ALPACA_OK;
  mr::Thresholds th;
  std::memset(&th, 0, sizeof(th));
  th.nlevels = nlevels;
  for (int i = 0; i < nlevels; ++i) th.eps[i] = eps_coarsen[i];
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dim == 2)
    return mr::details_impl<2>(d_blocks, nblocks, d_links, nlinks, norm, th, d_details,
                               d_decisions, s);
  return mr::details_impl<3>(d_blocks, nblocks, d_links, nlinks, norm, th, d_details,
                             d_decisions, s);
}

}  // extern "C"
