// Fused SSP-RK3 stage kernel, included into alpaca::exact and alpaca::fast
// (see fv_device.h).
//
// One workgroup per (leaf block, tile of TX x TY x TZ internal cells):
//   1. every face of the tile (all directions) is computed from the haloed
//      Average buffer — a flat loop whose per-direction ranges are padded to
//      64 so each wavefront works on a single direction — and its flux is
//      kept in LDS (in R: FP32 in the mixed form);
//   2. after one barrier each thread forms the flux divergence of its cells
//      in FP64 with the reference's ConsistencyManagedSum (space_solver.cpp:
//      131-153), applies the RK combination in FP64 (time_integrator.h:98-113,
//      434-457), writes the new state and pushes it into the face halo slabs
//      of the neighbouring blocks (internal_halo_manager.cpp:439-466) or, on a
//      zero-gradient or symmetry side, into its own halo
//      (boundary_constants.h:169-253);
//   3. on the last stage it also reduces the CFL signal of the new state
//      (modular_algorithm_assembler.cpp:1840-1869) for the next time step.

__device__ __forceinline__ double wave_max64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = smax(v, __shfl_xor(v, o, 64));
  return v;
}

// Writes the new values v of internal cell c3 of block blk of the job's case
// into the halo slabs that read them: the neighbours' slabs across each near
// face, or the block's own slab on a zero-gradient side (the first or last
// internal layer fills all four halo layers) or a symmetry side (the cell at
// internal depth c fills the halo layer at depth c, the face-normal momentum
// negated).  A workgroup's cells lie in one block, so each destination block is
// uniform over the wavefront and addressed by a buffer resource; the cell's
// offset is formed once for all equations.
template <int DIM>
__device__ __forceinline__ void push_halos(const TileJob &j, int blk, const int *bc3, const int *c3,
                                           const double *v) {
  using D = Dims<DIM>;
  constexpr int NE = D::NE;
  int const cell = (c3[0] + kHS) * D::SX + (c3[1] + kHS) * D::SY + (DIM == 3 ? c3[2] + kHS : 0);
  auto block = [&j](int b) {
    return BlockReader<DIM>(j.out + (size_t)__builtin_amdgcn_readfirstlane(b) * D::BLOCK);
  };
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    int const S = d == 0 ? D::SX : (d == 1 ? D::SY : D::SZ);
    int const c = c3[d];
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) {
      if (hi ? c < kIC - kHS : c >= kHS) continue;
      bool const edge = hi ? bc3[d] == j.nb[d] - 1 : bc3[d] == 0;
      if (!edge || j.bc[d] == ALPACA_BC_PERIODIC) {
        int nb3[3] = {bc3[0], bc3[1], bc3[2]};
        nb3[d] = hi ? (edge ? 0 : bc3[d] + 1) : (edge ? j.nb[d] - 1 : bc3[d] - 1);
        BlockReader<DIM> const w = block(j.base + (nb3[0] * j.nb[1] + nb3[1]) * j.nb[2] + nb3[2]);
        int const at = cell + (hi ? -kIC : kIC) * S;
#pragma unroll
        for (int e = 0; e < NE; ++e) w.store(v[e], at, e);
      } else if (j.bc[d] == ALPACA_BC_SYMMETRY) {
        BlockReader<DIM> const w = block(blk);
        int const at = cell + ((hi ? 2 * kIC - 1 : -1) - 2 * c) * S;
#pragma unroll
        for (int e = 0; e < NE; ++e) w.store(e == kMomX + d ? -1.0 * v[e] : v[e], at, e);
      } else if (c == (hi ? kIC - 1 : 0)) {
        BlockReader<DIM> const w = block(blk);
#pragma unroll
        for (int h = 1; h <= kHS; ++h)
#pragma unroll
          for (int e = 0; e < NE; ++e) w.store(v[e], cell + (hi ? h : -h) * S, e);
      }
    }
  }
}

// The step of a stage a cell takes: RK coefficients times the time step and
// the block's place in its grid.
struct StageStep {
  double m0, m1, cdt;
  int bc3[3];
  __device__ __forceinline__ StageStep(const TileJob &j, int blk_local) {
    int const stage = j.stage;
    m0 = stage == 0 ? 1.0 : (stage == 1 ? 0.25 : 2.0 / 3.0);
    m1 = stage == 0 ? 0.0 : (stage == 1 ? 0.75 : 1.0 / 3.0);
    double const cs = stage == 0 ? 1.0 : (stage == 1 ? 0.25 : 2.0 / 3.0);
    cdt = cs * (0.0 + j.state->dt);
    bc3[0] = blk_local / (j.nb[1] * j.nb[2]);
    bc3[1] = (blk_local / j.nb[2]) % j.nb[1];
    bc3[2] = blk_local % j.nb[2];
  }
};

// One internal cell c3 of block blk: the divergence of its flux differences
// (diff gives them per equation), the RK combination, the new value written
// and pushed into the halos that read it, and on the last stage the cell's
// CFL signal.
template <int DIM, typename DIFF>
__device__ __forceinline__ void stage_cell(const TileJob &j, const StageStep &st, int blk,
                                           const int *c3, const DIFF &diff, double &sig,
                                           bool &bad) {
  using D = Dims<DIM>;
  constexpr int NE = D::NE;
  size_t const first = (size_t)__builtin_amdgcn_readfirstlane(blk) * D::BLOCK;
  BlockReader<DIM> const avg(j.avg + first), out(j.out + first);
  int const cell = (c3[0] + kHS) * D::SX + (c3[1] + kHS) * D::SY + (DIM == 3 ? c3[2] + kHS : 0);
  constexpr int B = (int)sizeof(double);
  double u[NE], ini[NE], v[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) u[e] = avg(cell * B, e * D::FIELD * B);
  if (j.stage > 0) {
    BlockReader<DIM> const init(j.init + first);
#pragma unroll
    for (int e = 0; e < NE; ++e) ini[e] = init(cell * B, e * D::FIELD * B);
  } else if (j.init_copy) {
    BlockReader<DIM> const copy(j.init_copy + first);
#pragma unroll
    for (int e = 0; e < NE; ++e) copy.store(u[e], cell, e);
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    double dX, dY, dZ = 0.0;
    diff(e, dX, dY, dZ);
    double const rhs = 0.0 + (0.0 + dams<DIM>(dX, dY, dZ) * j.inv_dx);
    double const base = j.stage == 0 ? u[e] : st.m0 * u[e] + st.m1 * ini[e];
    v[e] = base + st.cdt * rhs;
    bad |= !__builtin_isfinite(v[e]);
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) out.store(v[e], cell, e);
  push_halos<DIM>(j, blk, st.bc3, c3, v);
  if (j.signal) {
    // The CFL signal is FP64 without contraction in every mode, so a step's
    // dt does not depend on which kernel reduced the signal.
    exact::Prim<double> p;
    exact::cons_to_prim<DIM>(j.gamma, j.b, v, p);
    double const cso = exact::eos_sos(j.gamma, j.b, p.rho, p.p);
    double sum;
    if constexpr (DIM == 2)
      sum = (__builtin_fabs(p.vel[0]) + cso) + (__builtin_fabs(p.vel[1]) + cso);
    else
      sum = exact::cms3(__builtin_fabs(p.vel[0]) + cso, __builtin_fabs(p.vel[1]) + cso,
                        __builtin_fabs(p.vel[2]) + cso);
    sig = smax(sig, sum);
  }
}

// Raises the record's CFL signal to sig.  Atomics of a launch on the one
// address follow each other at about 10.6 ns each, so a workgroup sends one,
// and only if sig exceeds what the record holds already.
__device__ __forceinline__ void raise_signal(alpaca_case_state *state, double sig) {
  auto *p = reinterpret_cast<unsigned long long *>(&state->smax);
  auto const bits = (unsigned long long)__double_as_longlong(sig);
  if (bits > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, bits);
}

// After a workgroup's cells: the CFL signal into the case record or, without
// an atomic, into the workgroup's place of `partials`; the non-finite flag.  All
// NT threads of the workgroup must call it.  (One atomic per wavefront made the
// last stage of 64 2D blocks 19.2 us, one per workgroup 11 to 14 us, 8.3 without.)
template <int NT>
__device__ __forceinline__ void stage_finish(const TileJob &j, double sig, bool bad) {
  if (j.signal) {
    __shared__ double part[NT / 64];
    sig = wave_max64(sig);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sig;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < NT / 64; ++w) sig = smax(sig, part[w]);
      if (j.partials)
        j.partials[blockIdx.x] = sig;
      else
        raise_signal(j.state, sig);
    }
  }
  if (bad) atomicOr(&j.state->flags, kFlagNonFinite);
}

template <int DIM, int TX, int TY, int TZ> struct TileShape {
  static constexpr int TZe = DIM == 3 ? TZ : 1;
  static constexpr int NTX = kIC / TX, NTY = kIC / TY, NTZ = DIM == 3 ? kIC / TZ : 1;
  static constexpr int TILES = NTX * NTY * NTZ;
  static constexpr int NFX = (TX + 1) * TY * TZe;
  static constexpr int NFY = TX * (TY + 1) * TZe;
  static constexpr int NFZ = DIM == 3 ? TX * TY * (TZ + 1) : 0;
  static constexpr int PX = round_up64(NFX), PY = round_up64(NFY), PZ = round_up64(NFZ);
  static constexpr int CELLS = TX * TY * TZe;
  static constexpr int LDS = (DIM + 2) * (NFX + NFY + NFZ);  // reals
};

// Face fluxes of one tile (first cell x0, y0, z0 of block bb) into LDS:
// every face of the tile, a flat loop whose per-direction ranges are padded
// to 64 so each wavefront works on a single direction.
template <int DIM, int FLUX, typename R, int TX, int TY, int TZ, int NT>
__device__ __forceinline__ void tile_faces(int tid, const double *__restrict__ bb, int x0, int y0,
                                           int z0, double gamma, double b, R *lds) {
  using D = Dims<DIM>;
  using T = TileShape<DIM, TX, TY, TZ>;
  constexpr int NE = D::NE;
  constexpr int TZe = T::TZe;
  constexpr int NFX = T::NFX, NFY = T::NFY, NFZ = T::NFZ;
  constexpr int PX = T::PX, PY = T::PY, PZ = T::PZ;
  R *FX = lds;
  R *FY = lds + NE * NFX;
  R *FZ = FY + NE * NFY;
  int const zh = DIM == 3 ? kHS : 0;  // halo offset along z
  for (int f = tid; f < PX + PY + PZ; f += NT) {
    R fl[NE];
    if (f < PX) {
      if (f < NFX) {
        int const k = f % TZe, jj = (f / TZe) % TY, ia = f / (TZe * TY);
        stencil_flux<DIM, 0, FLUX, R>(bb, x0 + ia + kHS - 1, y0 + jj + kHS, z0 + k + zh, gamma, b,
                                      fl);
#pragma unroll
        for (int e = 0; e < NE; ++e) FX[e * NFX + f] = fl[e];
      }
    } else if (f < PX + PY) {
      int const r = f - PX;
      if (r < NFY) {
        int const k = r % TZe, ja = (r / TZe) % (TY + 1), i = r / (TZe * (TY + 1));
        stencil_flux<DIM, 1, FLUX, R>(bb, x0 + i + kHS, y0 + ja + kHS - 1, z0 + k + zh, gamma, b,
                                      fl);
#pragma unroll
        for (int e = 0; e < NE; ++e) FY[e * NFY + r] = fl[e];
      }
    } else {
      if constexpr (DIM == 3) {
        int const r = f - PX - PY;
        if (r < NFZ) {
          int const ka = r % (TZ + 1), jj = (r / (TZ + 1)) % TY, i = r / ((TZ + 1) * TY);
          stencil_flux<DIM, 2, FLUX, R>(bb, x0 + i + kHS, y0 + jj + kHS, z0 + ka + kHS - 1, gamma,
                                        b, fl);
#pragma unroll
          for (int e = 0; e < NE; ++e) FZ[e * NFZ + r] = fl[e];
        }
      }
    }
  }
}

// The boundary-flux save of SpaceSolver::UpdateFluxes (space_solver.cpp:160-182):
// the fluxes of a tile's faces on the block's boundary added into the block's
// jump-flux surfaces ([6][NE][IC][ICZ]: East, West, North, South, Top, Bottom).
// From LDS, after the barrier: in the face loop nearly every wavefront of y and z
// faces held a few boundary faces and waited for their surface values (440
// blocks, exact HLLC: 497 us, 461 here).
template <int DIM, typename R, int TX, int TY, int TZ, int NT>
__device__ __forceinline__ void save_boundary(int tid, int x0, int y0, int z0, const R *lds,
                                              double *jump) {
  using D = Dims<DIM>;
  using T = TileShape<DIM, TX, TY, TZ>;
  constexpr int NE = D::NE, TZe = T::TZe, ICZ = D::ICZ;
  const R *FX = lds, *FY = lds + NE * T::NFX, *FZ = FY + NE * T::NFY;
  // One side: n1 x n2 entries from (a0, c0), the flux of (p, q) at first + p s1 + q s2.
  auto side = [&](int loc, int n1, int n2, int a0, int c0, const R *first, int s1, int s2, int field) {
    for (int t = tid; t < NE * n1 * n2; t += NT) {
      int const e = t / (n1 * n2), p = (t / n2) % n1, q = t % n2;
      jump[((loc * NE + e) * kIC + a0 + p) * ICZ + c0 + q] += double(first[e * field + p * s1 + q * s2]);
    }
  };
  if (x0 + TX == kIC) side(0, TY, TZe, y0, z0, FX + TX * TY * TZe, TZe, 1, T::NFX);
  if (x0 == 0) side(1, TY, TZe, y0, z0, FX, TZe, 1, T::NFX);
  if (y0 + TY == kIC) side(2, TX, TZe, x0, z0, FY + TY * TZe, (TY + 1) * TZe, 1, T::NFY);
  if (y0 == 0) side(3, TX, TZe, x0, z0, FY, (TY + 1) * TZe, 1, T::NFY);
  if constexpr (DIM == 3) {
    if (z0 + TZ == kIC) side(4, TX, TY, x0, y0, FZ + TZ, TY * (TZ + 1), TZ + 1, T::NFZ);
    if (z0 == 0) side(5, TX, TY, x0, y0, FZ, TY * (TZ + 1), TZ + 1, T::NFZ);
  }
}

// One tile of one block: faces into LDS, barrier, divergence + RK + halo
// push (+ CFL signal).  blk_local is the block's index within its case.
// All threads of the workgroup must call it (it contains a barrier).
// tid is the thread's index in the workgroup.
template <int DIM, int FLUX, typename R, int TX, int TY, int TZ, int NT>
__device__ __forceinline__ void stage_tile(int tid, const TileJob &j, int blk_local, int tile,
                                           R *lds) {
  using D = Dims<DIM>;
  using T = TileShape<DIM, TX, TY, TZ>;
  constexpr int NE = D::NE;
  constexpr int TZe = T::TZe, NTY = T::NTY, NTZ = T::NTZ;
  constexpr int NFX = T::NFX, NFY = T::NFY, NFZ = T::NFZ;
  R *FX = lds;
  R *FY = lds + NE * NFX;
  R *FZ = FY + NE * NFY;
  int const blk = j.base + blk_local;
  int const z0 = DIM == 3 ? (tile % NTZ) * TZ : 0;
  int const y0 = ((tile / NTZ) % NTY) * TY;
  int const x0 = (tile / (NTZ * NTY)) * TX;
  const double *bb = j.avg + (size_t)blk * D::BLOCK;

  // 1. Face fluxes of the tile into LDS.
  tile_faces<DIM, FLUX, R, TX, TY, TZ, NT>(tid, bb, x0, y0, z0, j.gamma, j.b, lds);
  __syncthreads();

  // 2. Divergence + RK combination + halo push (+ CFL signal).
  StageStep const st(j, blk_local);
  double sig = 0.0;
  bool bad = false;
  for (int c = tid; c < T::CELLS; c += NT) {
    int const kk = c % TZe, jj = (c / TZe) % TY, ii = c / (TZe * TY);
    int const c3[3] = {x0 + ii, y0 + jj, z0 + kk};
    auto diff = [&](int e, double &dX, double &dY, double &dZ) {
      dX = double(FX[e * NFX + (ii * TY + jj) * TZe + kk]) -
           double(FX[e * NFX + ((ii + 1) * TY + jj) * TZe + kk]);
      dY = double(FY[e * NFY + (ii * (TY + 1) + jj) * TZe + kk]) -
           double(FY[e * NFY + (ii * (TY + 1) + jj + 1) * TZe + kk]);
      if constexpr (DIM == 3)
        dZ = double(FZ[e * NFZ + (ii * TY + jj) * (TZ + 1) + kk]) -
             double(FZ[e * NFZ + (ii * TY + jj) * (TZ + 1) + kk + 1]);
    };
    stage_cell<DIM>(j, st, blk, c3, diff, sig, bad);
  }
  stage_finish<NT>(j, sig, bad);
}

// ------------------------------------------------------- plane marching ---
// 3D, large cases: one workgroup of 256 threads per slab of SX = 8 planes of a
// block, thread (j, k) owning the column of cells (x0 .. x0+7, j, k).  Plane
// by plane each thread computes the low y face, the low z face and the high x
// face of its cell; the x flux stays in registers as the next plane's low
// one, the y and z fluxes of the plane go through LDS.  The faces that close
// the slab at j = 16 and k = 16 (8 planes x 16 each: two whole waves per
// direction) are computed before the first plane, by the same code: p = -1
// runs the y body in waves 0 and 1, the z body in waves 2 and 3, and the x
// body on the slab's first face.  So every wave computes 26 units of 64 faces
// for 24 units of cells (8.3% more faces than cells; 8^3 tiles compute 12.5%
// more in 27 units over 4 waves), and the values the Roe average takes from a
// cell are formed once per cell (1.5 times, with the slab's rim) instead of
// six to seven times.
//
// LDS, in units of 256 values: Q (NQ per buffer, two buffers: the plane's
// packed cell quantities, the next plane's written by the x faces), HQ (NQ:
// those of the halo cells at j = -1 and k = -1, all planes), FZ, EX (the closing
// fluxes) and two buffers of FY (NE each): 70 KB in FP64, two workgroups per
// CU as the registers allow.  Before plane 0 the two Q buffers hold the
// quantities of the cells left and right of the closing faces.
//
// Bound by FP64 issue with a share of L2 misses.  256^3, one stage, against the
// 8^3 tiles: HLLC exact 4.10 -> 3.95 ms, FMA (tiles of 512 threads) 2.36 -> 2.32 ms,
// Roe exact 5.01 -> 4.70 ms, FMA 2.84 -> 2.79 ms.  The mixed HLLC form gains nothing (it
// runs 3 or 4 waves per SIMD either way and pays the barrier).  A wavefront
// marching an 8^3 tile by itself, without barriers, was slower (one step, HLLC
// exact 13.3 ms against 12.06, FMA 9.96 ms against 7.46): its waves drift apart
// and their planes no longer share the caches (1.3e8 L2 misses a launch).
struct MarchShape {
  static constexpr int SX = 8;
  static constexpr int SLABS = kIC / SX;
  static constexpr int PLANE = kIC * kIC;  // cells of a plane = threads
  static constexpr int NQ = kPackedQ;
  static constexpr int NE = 5;
  static constexpr int LDS = (3 * NQ + 4 * NE) * PLANE;
  static_assert(SX * 2 * kIC == PLANE, "one halo cell and one closing face per thread");
};

// Barrier of the workgroup that orders LDS accesses only: outstanding global
// stores are not waited for (no thread reads what another one stored).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Makes `off` available only once a and b are formed.
__device__ __forceinline__ void after(int &off, double a, double b) {
  asm volatile("" : "+v"(off) : "v"(a), "v"(b));
}

template <int FLUX>
__device__ __forceinline__ void stage_march(const TileJob &j, int blk_local, int slab, double *lds) {
  using R = double;
  using D = Dims<3>;
  using M = MarchShape;
  constexpr int NE = M::NE, P = M::PLANE, SX = M::SX, NQ = M::NQ;
  int const tid = threadIdx.x;
  int const wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int const x0 = slab * SX;
  int const blk = j.base + blk_local;
  const double *bb = j.avg + (size_t)blk * D::BLOCK;
  BlockReader<3> const rd(bb);
  R *Q = lds, *HQ = lds + 2 * NQ * P, *FZ = HQ + NQ * P, *EX = FZ + NE * P, *FY2 = EX + NE * P;
  // Packed quantities of the cell at halo offset `off` into q.
  auto keep = [&](int off, R *q) {
    double c[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) c[e] = rd(off * (int)sizeof(double), e * D::FIELD * (int)sizeof(double));
    store_packed<3, P>(j.gamma, j.b, c, q);
  };
  // Halo offset of thread t's cell in plane p, and of the cell left of its
  // closing face (threads 0-127 the y side, 128-255 the z side; plane
  // (t >> 4) & 7, position t & 15 along the other axis).
  auto here = [x0](int t, int p) {
    return (x0 + p + kHS) * D::SX + (t / kIC + kHS) * D::SY + t % kIC + kHS;
  };
  auto closing = [x0](int t, bool zside) {
    int const row = (x0 + ((t >> 4) & 7) + kHS) * D::SX;
    return zside ? row + ((t & 15) + kHS) * D::SY + kHS + kIC - 1
                 : row + (kHS + kIC - 1) * D::SY + (t & 15) + kHS;
  };
  // Quantities left and right of the closing faces (t = 0, 1) and of the rim
  // cells at j = -1 and k = -1 (t = 2).
#pragma unroll 1
  for (int t = 0; t < 3; ++t) {
    bool const zside = tid >= P / 2;
    int const step = zside ? 1 : D::SY;
    keep(closing(tid, zside) + (t == 2 ? -kIC : t) * step, Q + t * NQ * P + tid);
  }
  __syncthreads();
  StageStep const st(j, blk_local);
  double sig = 0.0;
  bool bad = false;
  R fx[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) fx[e] = R(0.0);
  // FV: the stencil of the next face is read while this face's Riemann problem
  // is solved, whose registers leave room for it.
  constexpr bool AHEAD = FLUX == 0;
  // The contracted FP64 form also keeps the column's cells p-2 .. p+2 in
  // registers for the x faces (203 VGPRs).  Reading them again for each of the
  // six faces that use a cell misses the XCD's 4 MB L2, which the 64 slabs in
  // flight fill (256^3: 9.4e7 L2 misses a launch against 3.8e7 for tiles; the
  // step takes 7.27 ms with the reads and 6.82 ms with the column).  The exact
  // form has no registers for it (111 spilled: 13.8 ms instead of 12.0).
  constexpr bool COLUMN = AHEAD && kLean<R>;
  double U[6][NE], X[6][NE];
  int p = -1;
  if constexpr (AHEAD) load_stencil<3>(rd, closing(tid, false), D::SY, U);
  if constexpr (COLUMN) load_stencil<3>(rd, here(tid, p), D::SX, X);
#pragma unroll 1
  for (; p < SX; ++p) {
    // The thread's indices pass through empty asm statements, so that no
    // address is formed ahead of the loop and held in registers through it
    // (and the first pass stays in the loop: one copy of each face body).
    asm volatile("" : "+s"(p));
    bool const inner = p >= 0;
    R *FY = FY2 + (p & 1) * NE * P;
    if (inner || wave < 2) {
      int t = tid;
      asm volatile("" : "+v"(t));
      int const yj = t / kIC, yk = t % kIC;
      const R *q = Q + (p & 1) * NQ * P;
      R fl[NE];
      KeptQ<3, P> const qs{inner ? (yj > 0 ? q + t - kIC : HQ + p * kIC + yk) : Q + t,
                              inner ? q + t : Q + NQ * P + t};
      if constexpr (AHEAD) {
        R cl[NE], cr[NE], skipped;
        fv_reconstruct<3, 1, R>(j.gamma, U, qs, cl, cr, skipped);
        int off = here(t, p) - 1;
        after(off, cl[NE - 1], cr[NE - 1]);
        load_stencil<3>(rd, off, 1, U);
        fv_riemann<3, 1, R>(j.gamma, j.b, cl, cr, skipped, fl);
      } else {
        int const off = inner ? here(t, p) - D::SY : closing(t, false);
        face_flux<3, 1, FLUX, R>(j.gamma, j.b, bb, off, qs, fl);
      }
      R *o = (inner ? FY : EX) + t;
#pragma unroll
      for (int e = 0; e < NE; ++e) o[e * P] = fl[e];
    }
    if (inner || wave >= 2) {
      int t = tid;
      asm volatile("" : "+v"(t));
      int const zj = t / kIC, zk = t % kIC;
      const R *q = Q + (p & 1) * NQ * P;
      R fl[NE];
      KeptQ<3, P> const qs{inner ? (zk > 0 ? q + t - 1 : HQ + P / 2 + p * kIC + zj) : Q + t,
                              inner ? q + t : Q + NQ * P + t};
      if constexpr (AHEAD) {
        if (!inner) load_stencil<3>(rd, closing(t, true), 1, U);
        R cl[NE], cr[NE], skipped;
        fv_reconstruct<3, 2, R>(j.gamma, U, qs, cl, cr, skipped);
        int off = here(t, p);
        after(off, cl[NE - 1], cr[NE - 1]);
        if constexpr (COLUMN)
          load_cell<3>(rd, off + 3 * D::SX, X[5]);
        else
          load_stencil<3>(rd, off, D::SX, U);
        fv_riemann<3, 2, R>(j.gamma, j.b, cl, cr, skipped, fl);
      } else {
        int const off = inner ? here(t, p) - 1 : closing(t, true);
        face_flux<3, 2, FLUX, R>(j.gamma, j.b, bb, off, qs, fl);
      }
      R *o = (inner ? FZ : EX) + t;
#pragma unroll
      for (int e = 0; e < NE; ++e) o[e * P] = fl[e];
    }
    R fh[NE];
    {
      int t = tid;
      asm volatile("" : "+v"(t));
      if (!inner) {
        lds_barrier();  // the closing faces have read both Q buffers
        keep(here(t, p), Q + NQ * P + t);
        if constexpr (AHEAD && !COLUMN) load_stencil<3>(rd, here(t, p), D::SX, U);
      }
      KeptThenFormedQ<3, P> const qs{j.gamma, j.b, Q + (p & 1) * NQ * P + t,
                                        Q + ((p + 1) & 1) * NQ * P + t};
      if constexpr (AHEAD) {
        R cl[NE], cr[NE], skipped;
        fv_reconstruct<3, 0, R>(j.gamma, COLUMN ? X : U, qs, cl, cr, skipped);
        if constexpr (COLUMN) {
#pragma unroll
          for (int m = 0; m < 5; ++m)
#pragma unroll
            for (int e = 0; e < NE; ++e) X[m][e] = X[m + 1][e];
        }
        int off = here(t, p) + D::SX - D::SY;
        after(off, cl[NE - 1], cr[NE - 1]);
        load_stencil<3>(rd, off, D::SY, U);
        fv_riemann<3, 0, R>(j.gamma, j.b, cl, cr, skipped, fh);
      } else {
        face_flux<3, 0, FLUX, R>(j.gamma, j.b, bb, here(t, p), qs, fh);
      }
    }
    // The plane's y fluxes and the next plane's quantities.  The z fluxes pass
    // between lanes of one wave, and the y fluxes have two buffers, so one
    // barrier per plane is enough.
    lds_barrier();
    if (inner) {
      int t = tid;
      asm volatile("" : "+v"(t));
      int const cj = t / kIC, ck = t % kIC;
      int const c3[3] = {x0 + p, cj, ck};
      const R *yh = cj < kIC - 1 ? FY + t + kIC : EX + p * kIC + ck;
      const R *zh = ck < kIC - 1 ? FZ + t + 1 : EX + P / 2 + p * kIC + cj;
      auto diff = [&](int e, double &dX, double &dY, double &dZ) {
        dX = double(fx[e]) - double(fh[e]);
        dY = double(FY[e * P + t]) - double(yh[e * P]);
        dZ = double(FZ[e * P + t]) - double(zh[e * P]);
      };
      stage_cell<3>(j, st, blk, c3, diff, sig, bad);
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) fx[e] = fh[e];
  }
  stage_finish<P>(j, sig, bad);
}

// Waves per SIMD the register allocator is held to.  The FP64 2D kernels fit 3
// waves without spilling; the exact 3D flux-splitting kernels need 211 to 217
// VGPRs (2 waves).
template <int DIM, int FLUX, typename R>
constexpr int kMinWaves = !std::is_same<R, double>::value ? 1
                          : DIM == 2 ? 3 : (FLUX == 1 && !kFastArith ? 2 : 1);

// And at most, in the persistent batch kernel.  The 2D mixed flux-splitting form fits 4,
// but with two wavefronts per workgroup its workgroups then gather on some SIMDs, four
// wavefronts there and two on others, and a stage waits for those.  Held to 3 (one step,
// 16x16 cells, us): 1300 blocks 167 -> 144, 1536 174 -> 149, 3072 319 -> 273, 8192 824 ->
// 694; 1024 and fewer the same.
template <int DIM, int FLUX, typename R, int NT>
constexpr int kBatchMaxWaves = DIM == 2 && FLUX == 1 && std::is_same<R, float>::value && NT == 128 ? 3 : 8;

// The job of a single case's stage.
__device__ __forceinline__ TileJob stage_job(const double *avg, const double *init, double *out,
                                             alpaca_case_state *state, const StageArgs &a) {
  TileJob j;
  j.avg = avg;
  j.init = init;
  j.out = out;
  j.state = state;
  j.init_copy = a.init_copy;
  j.base = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    j.nb[d] = a.nb[d];
    j.bc[d] = a.bc[d];
  }
  j.gamma = a.gamma;
  j.b = a.b;
  j.inv_dx = a.inv_dx;
  j.stage = a.stage;
  j.signal = a.signal;
  j.partials = a.partials;
  return j;
}

// Single case: one workgroup per (block, tile).
template <int DIM, int FLUX, typename R, int TX, int TY, int TZ, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(kMinWaves<DIM, FLUX, R>, 8))) void stage_kernel(const double *__restrict__ avg,
                                                   const double *init, double *out,
                                                   alpaca_case_state *state, StageArgs a) {
  using T = TileShape<DIM, TX, TY, TZ>;
  static_assert(NT % 64 == 0, "whole wavefronts");
  __shared__ R lds[T::LDS];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  int const blk = g / T::TILES;
  if (blk >= a.nblocks) return;  // uniform over the workgroup
  if (a.guard && (state->flags & kFlagDone)) return;
  TileJob const j = stage_job(avg, init, out, state, a);
  stage_tile<DIM, FLUX, R, TX, TY, TZ, NT>(threadIdx.x, j, blk, g % T::TILES, lds);
}

// Single 3D case by plane marching: one workgroup per (block, slab).
template <int FLUX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kMinWaves<3, FLUX, double>, 8))) void march_stage_kernel(
    const double *__restrict__ avg, const double *init, double *out, alpaca_case_state *state,
    StageArgs a) {
  constexpr unsigned SLABS = MarchShape::SLABS;
  __shared__ double lds[MarchShape::LDS];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  int const blk = g / SLABS;
  if (blk >= a.nblocks) return;  // uniform over the workgroup
  if (a.guard && (state->flags & kFlagDone)) return;
  TileJob const j = stage_job(avg, init, out, state, a);
  stage_march<FLUX>(j, blk, g % SLABS, lds);
}

// Large 2D cases: one workgroup of 192 threads per two blocks adjacent in
// memory.  A block has 272 faces per direction, 4.25 wavefronts, so a block by itself
// takes 10 units of 64 faces; two take 18, six for each of three wavefronts, and
// the four workgroups that the LDS of a CU holds are the 12 wavefronts its
// registers hold.  A wavefront's faces may lie in both blocks, its cells lie in one.
// 2048^2 cells, one stage: exact HLLC 550 -> 529 us against a block per workgroup,
// exact Roe 806 -> 755 us.
constexpr int kPairThreads = 192;

template <int FLUX, typename R>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(kMinWaves<2, FLUX, R>, 8))) void pair_stage_kernel(
    const double *__restrict__ avg, const double *init, double *out, alpaca_case_state *state,
    StageArgs a) {
  using D = Dims<2>;
  constexpr int NE = D::NE, NT = kPairThreads;
  constexpr int NF = (kIC + 1) * kIC;  // faces of a block per direction
  constexpr int P = round_up64(2 * NF);
  __shared__ R lds[2 * NE * 2 * NF];
  R *FX = lds, *FY = lds + NE * 2 * NF;
  int const pair = 2 * int(xcd_remap_group(blockIdx.x, gridDim.x));
  if (pair >= a.nblocks) return;  // uniform over the workgroup
  if (a.guard && (state->flags & kFlagDone)) return;
  TileJob const j = stage_job(avg, init, out, state, a);
  int const faces = pair + 1 < a.nblocks ? 2 * NF : NF;
  const double *bb = avg + (size_t)pair * D::BLOCK;
  FormedQ<2, R> const qs{a.gamma, a.b};
  for (int f = threadIdx.x; f < 2 * P; f += NT) {
    bool const y = f >= P;  // uniform over the wavefront
    int const r = y ? f - P : f;
    if (r >= faces) continue;
    int const second = r >= NF, q = second ? r - NF : r;
    R fl[NE];
    if (!y) {  // [17][16]
      int const off = (q / kIC + kHS - 1) * D::SX + (q % kIC + kHS) * D::SY;
      face_flux<2, 0, FLUX, R>(a.gamma, a.b, bb, off + second * D::BLOCK, qs, fl);
    } else {  // [16][17]
      int const off = (q / (kIC + 1) + kHS) * D::SX + (q % (kIC + 1) + kHS - 1) * D::SY;
      face_flux<2, 1, FLUX, R>(a.gamma, a.b, bb, off + second * D::BLOCK, qs, fl);
    }
    R *o = (y ? FY : FX) + r;
#pragma unroll
    for (int e = 0; e < NE; ++e) o[e * 2 * NF] = fl[e];
  }
  __syncthreads();
  double sig = 0.0;
  bool bad = false;
  int const cells = faces / NF * D::CELLS;
  for (int c = threadIdx.x; c < cells; c += NT) {
    int const second = __builtin_amdgcn_readfirstlane(c / D::CELLS);
    int const ii = c / kIC % kIC, jj = c % kIC;
    int const c3[3] = {ii, jj, 0};
    const R *fx = FX + second * NF + ii * kIC + jj, *fy = FY + second * NF + ii * (kIC + 1) + jj;
    auto diff = [&](int e, double &dX, double &dY, double &) {
      dX = double(fx[e * 2 * NF]) - double(fx[e * 2 * NF + kIC]);
      dY = double(fy[e * 2 * NF]) - double(fy[e * 2 * NF + 1]);
    };
    stage_cell<2>(j, StageStep(j, pair + second), pair + second, c3, diff, sig, bad);
  }
  stage_finish<NT>(j, sig, bad);
}

// Right-hand side of n blocks (SpaceSolver::UpdateFluxes, space_solver.cpp:
// 50-182): those listed of a pool, or, without a list, blocks 0 .. n-1.  One
// workgroup per (block, tile): the tile's faces into LDS, those on the block's
// boundary also added into its jump-flux surfaces (jump not null); after the
// barrier each internal cell's flux
// divergence (ConsistencyManagedSum, space_solver.cpp:131-153) is written to
// the block's right-hand-side buffer, and the tile's share of the block's
// halo cells is set to zero (the whole output block is written, as by the
// per-block right-hand side that the reference clears first).  In 2D the Top and Bottom surfaces receive += 0.0,
// as from the reference's zeroed z face array.  List entries outside
// [0, capacity) are skipped (uniformly over the workgroup).
template <int DIM, int FLUX, typename R, int TX, int TY, int TZ, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(kMinWaves<DIM, FLUX, R>, 8))) void rhs_tile_kernel(
    const double *__restrict__ avg, double *__restrict__ rhs, double *__restrict__ jump,
    const int *__restrict__ list, int n, int capacity, double gamma, double b, double inv_dx) {
  using D = Dims<DIM>;
  using T = TileShape<DIM, TX, TY, TZ>;
  constexpr int NE = D::NE;
  constexpr int TZe = T::TZe, NTY = T::NTY, NTZ = T::NTZ;
  constexpr int NFX = T::NFX, NFY = T::NFY, NFZ = T::NFZ;
  constexpr int ICZ = D::ICZ;
  constexpr int SURF = 6 * NE * kIC * ICZ;  // doubles per SurfaceBuffer
  __shared__ R lds[T::LDS];
  unsigned const g = xcd_remap_group(blockIdx.x, gridDim.x);
  int const item = int(g / T::TILES), tile = int(g % T::TILES);
  if (item >= n) return;
  int const blk = list ? list[item] : item;
  if (blk < 0 || blk >= capacity) return;  // uniform over the workgroup
  int const z0 = DIM == 3 ? (tile % NTZ) * TZ : 0;
  int const y0 = ((tile / NTZ) % NTY) * TY;
  int const x0 = (tile / (NTZ * NTY)) * TX;
  double *jb = jump ? jump + (size_t)blk * SURF : nullptr;
  tile_faces<DIM, FLUX, R, TX, TY, TZ, NT>(threadIdx.x, avg + (size_t)blk * D::BLOCK, x0, y0, z0, gamma,
                                           b, lds);
  if (DIM == 2 && jb && tile == 0) {  // one workgroup per block: others' would race
    for (int t = threadIdx.x; t < 2 * NE * kIC; t += NT) jb[4 * NE * kIC + t] += 0.0;
  }
  __syncthreads();
  if (jb) save_boundary<DIM, R, TX, TY, TZ, NT>(threadIdx.x, x0, y0, z0, lds, jb);
  const R *FX = lds;
  const R *FY = lds + NE * NFX;
  const R *FZ = FY + NE * NFY;
  double *out = rhs + (size_t)blk * D::BLOCK;
  for (int c = threadIdx.x; c < T::CELLS; c += NT) {
    int const kk = c % TZe, jj = (c / TZe) % TY, ii = c / (TZe * TY);
    int const cell = (x0 + ii + kHS) * D::SX + (y0 + jj + kHS) * D::SY +
                     (DIM == 3 ? z0 + kk + kHS : 0);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      double const dX = double(FX[e * NFX + (ii * TY + jj) * TZe + kk]) -
                        double(FX[e * NFX + ((ii + 1) * TY + jj) * TZe + kk]);
      double const dY = double(FY[e * NFY + (ii * (TY + 1) + jj) * TZe + kk]) -
                        double(FY[e * NFY + (ii * (TY + 1) + jj + 1) * TZe + kk]);
      double dZ = 0.0;
      if constexpr (DIM == 3)
        dZ = double(FZ[e * NFZ + (ii * TY + jj) * (TZ + 1) + kk]) -
             double(FZ[e * NFZ + (ii * TY + jj) * (TZ + 1) + kk + 1]);
      out[e * D::FIELD + cell] = 0.0 + (0.0 + dams<DIM>(dX, dY, dZ) * inv_dx);
    }
  }
  // The tile's share of the halo cells: positions [tile * FIELD / TILES, ...).
  constexpr int SHARE = D::FIELD / T::TILES;
  static_assert(SHARE * T::TILES == D::FIELD, "halo shares cover the block");
  for (int q = threadIdx.x; q < SHARE; q += NT) {
    int const r = tile * SHARE + q;
    int const i = r / D::SX, j = (r / D::SY) % kTC, k = DIM == 3 ? r % kTC : kHS;
    bool const inside = i >= kHS && i < kHS + kIC && j >= kHS && j < kHS + kIC &&
                        k >= kHS && k < kHS + kIC;
    if (!inside) {
#pragma unroll
      for (int e = 0; e < NE; ++e) out[e * D::FIELD + r] = 0.0;
    }
  }
}

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ int in_sgpr(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double in_sgpr(double v) {
  long long const b = __double_as_longlong(v);
  unsigned const lo = __builtin_amdgcn_readfirstlane((int)b);
  unsigned const hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Every tile of every listed block of every case of an ensemble, one
// persistent kernel per RK stage: the grid is sized to the device and each
// workgroup walks the work list (read from device memory, so a captured
// graph of the step stays valid when the list changes).  Work units are
// split into 8 contiguous ranges, one per XCD (group g runs on XCD g % 8),
// so a case's blocks share an L2.  Units of stopped cases are skipped.
template <int DIM, int FLUX, typename R, int TX, int TY, int TZ, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(kMinWaves<DIM, FLUX, R>, kBatchMaxWaves<DIM, FLUX, R, NT>))) void batch_stage_kernel(
    const double *__restrict__ avg, const double *init, double *out, const CaseSlot *slots,
    alpaca_case_state *states, const WorkItem *items, const int *n_items, int stage) {
  using T = TileShape<DIM, TX, TY, TZ>;
  __shared__ R lds[T::LDS];
  __shared__ int skip;
  constexpr unsigned kXcd = 8;
  unsigned const n = unsigned(*n_items);
  unsigned const groups = gridDim.x;
  // Work items are dealt to the 8 XCDs round-robin (item k to XCD k % 8; the
  // hardware deals workgroups round-robin too, so blockIdx % 8 is the XCD),
  // all tiles of an item staying on one XCD's L2.  Round-robin rather than
  // contiguous ranges keeps the XCDs balanced when the active cases cluster
  // in the list (finished cases are skipped); within an XCD the workgroups
  // stride over its items' tiles.
  unsigned const xcd = blockIdx.x % kXcd;
  unsigned const per_xcd = groups / kXcd;  // grid is a multiple of 8
  unsigned const m = blockIdx.x / kXcd;
  unsigned const items_here = n > xcd ? (n - xcd + kXcd - 1) / kXcd : 0u;
  unsigned const units_here = items_here * T::TILES;
  for (unsigned w = m; w < units_here; w += per_xcd) {
    unsigned const u = (xcd + kXcd * (w / T::TILES)) * T::TILES + w % T::TILES;
    WorkItem it = items[u / T::TILES];
    it.case_id = in_sgpr(it.case_id);
    it.block = in_sgpr(it.block);
    alpaca_case_state *st = states + it.case_id;
    // Another workgroup may flag the case during this stage: decide once per
    // workgroup so every thread takes the same branch around the barriers.
    if (threadIdx.x == 0) skip = (__atomic_load_n(&st->flags, __ATOMIC_RELAXED) & kFlagsStop()) != 0;
    __syncthreads();
    bool const stop = skip;
    __syncthreads();
    if (stop) continue;
    CaseSlot const &cs = slots[it.case_id];
    TileJob j;
    j.avg = avg;
    j.init = init;
    j.out = out;
    j.state = st;
    j.init_copy = nullptr;
    j.base = in_sgpr(cs.base);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      j.nb[d] = in_sgpr(cs.nb[d]);
      j.bc[d] = in_sgpr(cs.bc[d]);
    }
    j.gamma = in_sgpr(cs.gamma);
    j.b = in_sgpr(cs.b);
    j.inv_dx = in_sgpr(cs.inv_dx);
    j.stage = stage;
    j.signal = stage == 2;
    j.partials = nullptr;
    // Through an empty asm statement, so that nothing that follows from the
    // thread's index is formed ahead of the loop and held through it.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    stage_tile<DIM, FLUX, R, TX, TY, TZ, NT>(tid, j, it.block, u % T::TILES, lds);
    __syncthreads();  // LDS is reused by the next unit
  }
}
