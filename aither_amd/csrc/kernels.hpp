// Device kernels of the hot path.  Launch geometry and data layout:
//
//  * state W: SoA per variable, ghost padded (ni+2g)(nj+2g)(nk+2g), i fastest;
//  * residual, spectral radius, dt, diagonal, du, time-level states: SoA over
//    physical cells, i fastest;
//  * face vectors: one double4 (unit normal, magnitude) per physical face.
#pragma once

#include <type_traits>

#include "device_math.hpp"

namespace ath {

struct BcStateDev;

// The device pointers of a block point to global memory.  In the device pass
// they carry the global address space, so that the compiler emits global
// loads and stores rather than flat ones: a flat access also counts against
// the LDS wait counter, so every wait for LDS would wait for outstanding
// global loads as well.  The host pass sees plain pointers of the same size.
#ifdef __HIP_DEVICE_COMPILE__
#define ATH_GLOBAL __attribute__((address_space(1)))
#else
#define ATH_GLOBAL
#endif
// a device allocation as a block's pointer
template <typename T>
__host__ __device__ inline ATH_GLOBAL T *Dev(T *p) {
  return (ATH_GLOBAL T *)p;
}

// Records of the pencil sweeps: pencils of kPW x kPW columns, kPenLanes lanes
// a record (one hyperplane step of one pencil, or several where the block is
// thinner than a pencil: DevBlock::pln)
constexpr int kPW = 8;
constexpr int kPenLanes = kPW * kPW;
constexpr int kPenS = 11;      // per-relax values of a cell: W, right-hand side, D^-1 (and viscosity)

struct DevBlock {
  int ni, nj, nk, g;
  int NI, NJ;
  long npad, ncell;
  double ATH_GLOBAL *W;             // 5 * npad
  const double ATH_GLOBAL *cw;      // 3 * npad
  const double4 ATH_GLOBAL *fa[3];  // physical faces per direction
  const double ATH_GLOBAL *vol;     // ncell
  double ATH_GLOBAL *R;             // 5 * ncell
  double ATH_GLOBAL *sr, *dt, *A;   // ncell
  double ATH_GLOBAL *Ainv;          // ncell (FP64 operator)
  float ATH_GLOBAL *Ainv32;         // ncell (FP32 operator)
  double ATH_GLOBAL *consN, *consNm1;  // 5 * ncell
  double ATH_GLOBAL *x;             // 5 * ncell (FP64 operator)
  float ATH_GLOBAL *x32;            // 5 * ncell (FP32 operator)
  double ATH_GLOBAL *xold;          // 5 * ncell, DP-LUR Jacobi copy
  float ATH_GLOBAL *xold32;
  // LU-SGS: the pencil sweep's inputs in the order the sweep takes them.
  // Pencils run along axis pl, pa x pb of them along the axes pl + 1 and
  // pl + 2 (mod 3), pns steps stored for each in prec records, which hold each
  // value 64 lanes at a time (KPencilFaces, KResidual, KPencilPrep, KBlockDiag,
  // KPencilOther).  A step has 2^pln lanes, 2^pla of them along the first cut
  // axis (the pencil's width or the block's, rounded up to a power of two), a
  // record 64 >> pln steps: a 256 x 256 x 1 block takes 8 lanes a step, where 64
  // would make eight times the memory.  pns = 0 and null pointers without it.
  int pl, pa, pb, pns;
  int pla, pln, prec;
  int dtile;  // the block diagonal's tile, an index of kDiagTile
  double ATH_GLOBAL *skF;  // face data, both sides
  double ATH_GLOBAL *skS;  // scalar: state, right-hand side, D^-1 (and viscosity);
                           // block: state, right-hand side (viscosity, conductivity, velocity gradient)
  double ATH_GLOBAL *skX;  // forward du (operator precision)
  double ATH_GLOBAL *skO;  // other-side sums of a full sweep (operator precision), null with one sweep
  // block matrix solvers: main diagonal after AddDiagonalTerms, 25 * ncell,
  // entry (r, c) of cell p at (5 r + c) ncell + p; its inverse in the layout
  // of InverseBase (LU-SGS: the pencil sweep's records; DP-LUR: 8 x 8 x 4
  // tiles, one tile's values of one entry 256 consecutive doubles).  The
  // off-diagonal blocks are formed where they are used (NeighbourBlock).
  double ATH_GLOBAL *Ab, *Abi;
  float ATH_GLOBAL *Abi32;       // FP32 operator: Abi rounded to float, same layout
  int tni, tnj, tnk;  // tile grid of the layout
  // block solvers with the viscous terms: the velocity gradient the viscous
  // pass formed at every physical face of direction d, 9 * faces(d), entry q
  // of face f at q * faces(d) + f; the thin-shear-layer part of the block
  // diagonal reads it back (and forms the face state, viscosity and
  // conductivity again from the cells, with the same functions)
  double ATH_GLOBAL *fvis[3];
  // off-diagonal product of the ghost neighbour across each boundary face
  // that lies on an interblock connection (zero on other faces), per sweep
  // pass; null when the block has no connection.  5 * nbf, SoA.
  double ATH_GLOBAL *bt;            // FP64 operator
  float ATH_GLOBAL *bt32;           // FP32 operator
  long nbf;              // boundary faces: 2 (nj nk + nk ni + ni nj)
  // viscous cases only
  double ATH_GLOBAL *T, *mu;               // padded: temperature, viscosity
  double ATH_GLOBAL *kc;                   // padded: conductivity before scaling (block solvers only)
  const double4 ATH_GLOBAL *faP[3];        // padded faces (ghost faces included)
  const double ATH_GLOBAL *volP;           // padded volumes
  const double ATH_GLOBAL *c2c[3];         // physical faces: centre-to-centre distance projected on the normal
  const unsigned char ATH_GLOBAL *wallf;   // per boundary face (BtSlot order): 1 on a viscousWall patch
  double ATH_GLOBAL *vgrad;                // block solvers: padded cell velocity gradient, 9 * npad, d v_c / d x_r at (3 r + c) npad
  // viscous block solvers: per cell, 1 where the inviscid face states reach
  // a viscousWall ghost cell (null when the block has none)
  const unsigned char ATH_GLOBAL *invPark;
  long cellBase;         // cell offset of this block within its case (L-inf index)
  int blockId;           // block index within its case
  // per case: the CFL number of the current iteration, the device error bits
  // (1 nonphysical state, 4 singular block diagonal) and the boundary states
  // by tag
  const double ATH_GLOBAL *cfl;
  int ATH_GLOBAL *flag;
  const BcStateDev ATH_GLOBAL *states;
};

// laminar viscous terms: Sutherland transport (src/transport.cpp:29-176),
// its nondimensional scaling mu_ref / (rho_ref a_ref L_ref), Prandtl number
// 4 gamma / (9 gamma - 5), and the viscous CFL coefficient
struct ViscParams {
  int on, recon4;
  double vscale, prandtl, coeff, tRef, muRef, kNonDim;
  double c1, s1, c2, s2;  // Sutherland C1, S of viscosity, then of conductivity
};

struct Params {
  Gas gas;
  ViscParams visc;
  double kappa;
  double theta, zeta, relax, dualCFL;
  double dtFixed;  // nondimensional global time step, <= 0 for local dt
  int implicit, multilevel, initMatrix, explicitEuler;
  int block;  // matrixSolver blusgs / bdplur: 5x5 main diagonal and off-diagonals
  int fp32;   // the scalar implicit operator runs in FP32: the residual stage writes Ainv32, else Ainv
  int roeJac; // inviscidFluxJacobian approximateRoe: the off-diagonals are Roe flux changes (FP64)
  int rhsOnce; // the relax writes the right-hand side and the state in sweep order (the block pencil sweep reads them)
  int prep;      // the inviscid residual kernel writes the scalar pencil sweep's records (KPencilPrep's)
  int rhsInDiag; // the block diagonal forms that right-hand side (the relax does not)
};

// ---------------------------------------------------------------------------
// laminar viscous helpers

// idealGas::Temperature (src/eos.cpp:54-60)
__device__ __forceinline__ double TempOf(const GasT<double> &g, double rho, double p) {
  const double rhoR = 0.0 + rho * g.R;
  return Div(p, rhoR);
}
// sutherland::SpeciesViscosity / SpeciesConductivity (src/transport.cpp:
// 97-117), nondimensional; t^1.5 correctly rounded
__device__ __forceinline__ double SutherlandMu(const ViscParams &v, double t) {
  const double temp = t * v.tRef;
  const double mu = Div(v.c1 * Pow15CR(temp), temp + v.s1);
  return Div(mu, v.muRef);
}
__device__ __forceinline__ double SutherlandK(const ViscParams &v, double t) {
  const double temp = t * v.tRef;
  const double k = Div(v.c2 * Pow15CR(temp), temp + v.s2);
  return Div(k, v.kNonDim);
}
// max(4/(3 rho), gamma/rho) and NondimScaling (mu / Pr + mut / Prt), mut = 0
// (include/spectralRadius.hpp:93-151)
template <typename T>
__device__ __forceinline__ T ViscFaceSR(const GasT<T> &g, const T W[5], T mag, T dist, T mu,
                                        const ViscParams &v) {
  const T rho = T(0) + W[0];
  const T a = Div(T(4), T(3) * rho), bq = Div(g.gamma, rho);
  const T maxTerm = a < bq ? bq : a;
  const T viscTerm = T(v.vscale) * (Div(mu, T(v.prandtl)) + T(0) / T(0.9));
  return Div(mag, dist) * maxTerm * viscTerm;
}
__device__ __forceinline__ double ViscCellSR(const GasT<double> &g, const double W[5], double magL,
                                             double magR, double vol, double mu, const ViscParams &v) {
  const double fMag = 0.5 * (magL + magR);
  const double rho = 0.0 + W[0];
  const double a = Div(4.0, 3.0 * rho), bq = Div(g.gamma, rho);
  const double maxTerm = a < bq ? bq : a;
  const double viscTerm = v.vscale * (Div(mu, v.prandtl) + 0.0 / 0.9);
  return Div(maxTerm * viscTerm * fMag * fMag, vol);
}

struct BcStateDev {
  double p, rho, u, v, w, p0, t0, dx, dy, dz;
  double tw;  // viscousWall: wall temperature when iso
  int iso;
  int flux;   // viscousWall: a given heat flux qw
  double qw;
};

struct BcTask {
  int dir, r1s, n1, r2s, n2, r3;
  int gC, srcC, stype, bctype, layer, state;
  long base;
};

__device__ __forceinline__ long PadIdx(const DevBlock &b, int i, int j, int k) {
  return (long)(i + b.g) + (long)(j + b.g) * b.NI + (long)(k + b.g) * b.NI * b.NJ;
}
__device__ __forceinline__ long FaceIdx(const DevBlock &b, int d, int i, int j, int k) {
  const int FI = b.ni + (d == 0), FJ = b.nj + (d == 1);
  return (long)i + (long)j * FI + (long)k * FI * FJ;
}
// slot of a boundary face: surfaces in the order i-lower, i-upper, j-lower,
// j-upper, k-lower, k-upper; within a surface of normal axis d the face
// (c1, c2) along axes d+1, d+2 (mod 3) is at c1 + N(d+1) c2
__device__ __forceinline__ long BtSlot(const DevBlock &b, int d, int upper, int i, int j, int k) {
  const long sI = (long)b.nj * b.nk, sJ = (long)b.nk * b.ni, sK = (long)b.ni * b.nj;
  if (d == 0) return upper * sI + j + (long)b.nj * k;
  if (d == 1) return 2 * sI + upper * sJ + k + (long)b.nk * i;
  return 2 * sI + 2 * sJ + upper * sK + i + (long)b.ni * j;
}
// record (of a pencil's) and first lane of step s
__host__ __device__ __forceinline__ int StepRecord(const DevBlock &b, int s, int &lane) {
  const int sh = 6 - b.pln;
  lane = (s & ((1 << sh) - 1)) << b.pln;
  return s >> sh;
}
// record and lane of cell (i, j, k) in the pencil sweep's arrays
__host__ __device__ __forceinline__ long PencilRecord(const DevBlock &b, int i, int j, int k, int &lane) {
  const int ca = b.pl == 0 ? j : (b.pl == 1 ? k : i), cb = b.pl == 0 ? k : (b.pl == 1 ? i : j),
            cc = b.pl == 0 ? i : (b.pl == 1 ? j : k);
  const int la = ca % kPW, lb = cb % kPW;
  const int r = StepRecord(b, la + lb + cc, lane);
  lane += la + (lb << b.pla);
  return (long)(ca / kPW + b.pa * (cb / kPW)) * b.prec + r;
}
// Values in LDS go 16 bytes a lane: a 16-byte read takes 13 cycles of the
// LDS pipe for a wave, two 8-byte reads 33.  Value q of a lane's record is
// v[q % kVecN] of its vector q / kVecN.
template <typename T>
struct alignas(16) LdsVec {
  T v[16 / sizeof(T)];
};
template <typename T>
constexpr int kVecN = 16 / (int)sizeof(T);
template <typename T>
constexpr int Vecs(int n) { return (n + kVecN<T> - 1) / kVecN<T>; }

// n consecutive values written as whole vectors, zeros behind them
template <typename T, int N>
__device__ __forceinline__ void PutVecs(T *p, const T *v) {
#pragma unroll
  for (int q = 0; q < Vecs<T>(N); ++q) {
    LdsVec<T> w;
#pragma unroll
    for (int r = 0; r < kVecN<T>; ++r) w.v[r] = q * kVecN<T> + r < N ? v[q * kVecN<T> + r] : T(0);
    ((LdsVec<T> *)p)[q] = w;
  }
}
// layout of the block solvers' inverse diagonal: entry q of cell (i, j, k) at
// InverseBase + q * stride.  In the pencil sweep's records a cell's 25 values
// are consecutive, padded to whole 16-byte vectors (an odd number of them, so
// that a record copied to LDS is read without bank conflicts).
template <typename T>
constexpr int kInv = Vecs<T>(25) * kVecN<T>;
static_assert(Vecs<float>(25) % 2 == 1 && Vecs<double>(25) % 2 == 1, "bank spread of a record in LDS");
template <typename T>
__host__ __device__ __forceinline__ long InverseBase(const DevBlock &b, int i, int j, int k, int &stride) {
  if (b.pns) {
    int lane;
    const long rec = PencilRecord(b, i, j, k, lane);
    stride = 1;
    return (rec * kPenLanes + lane) * kInv<T>;
  }
  const long tile = (long)(i >> 3) + (long)b.tni * ((j >> 3) + (long)b.tnj * (k >> 2));
  stride = 256;
  return tile * (25 * 256) + ((i & 7) + 8 * ((j & 7) + 8 * (k & 3)));
}
__device__ __forceinline__ void Map3(int dir, int d3, int d1, int d2, int &i, int &j, int &k) {
  if (dir == 0) { i = d3; j = d1; k = d2; }
  else if (dir == 1) { i = d2; j = d3; k = d1; }
  else { i = d1; j = d2; k = d3; }
}

// ---------------------------------------------------------------------------
// boundary ghost cells: GetGhostState (src/ghostStates.cpp:62-689, inviscid
// branches) and ExtrapolateHoldMixture (:691-709), driven by
// procBlock::AssignInviscidGhostCells (src/procBlock.cpp:2449-2529).  One
// thread per (surface patch cell, layer); every layer depends only on interior
// cells, so all layers of all surfaces run in one launch.

__device__ inline void ExtrapHold(const double bnd[5], double factor, const double in[5],
                                  double out[5]) {
  const double ghostRho = factor * bnd[0] - in[0];
  if (ghostRho <= 0.0) {
    for (int e = 0; e < 5; ++e) out[e] = bnd[e];
    return;
  }
  const double mf = bnd[0] / bnd[0];
  for (int e = 0; e < 5; ++e) out[e] = factor * bnd[e] - in[e];
  out[0] = Dmax(ghostRho * mf, 0.0);
}

__device__ inline void GhostState(const GasT<double> &g, const double in[5], int bctype,
                                  double ax, double ay, double az, int stype, int layer,
                                  const BcStateDev *s, double gh[5]) {
  for (int e = 0; e < 5; ++e) gh[e] = in[e];
  const bool lower = (stype % 2 == 1);
  const double nx = lower ? -1.0 * ax : ax, ny = lower ? -1.0 * ay : ay,
               nz = lower ? -1.0 * az : az;
  if (bctype == 0) {  // slipWall
    const double vn = (in[1] * nx + in[2] * ny) + in[3] * nz;
    gh[1] = in[1] - (nx * 2.0) * vn;
    gh[2] = in[2] - (ny * 2.0) * vn;
    gh[3] = in[3] - (nz * 2.0) * vn;
  } else if (bctype == 1) {  // characteristic
    const double fs[5] = {s->rho * 1.0, s->u, s->v, s->w, s->p};
    const double vn = (in[1] * nx + in[2] * ny) + in[3] * nz;
    const double c = SoS(g, in[0], in[4]);
    const double mach = fabs(vn) / c;
    if (mach >= 1.0 && vn < 0.0) {
      for (int e = 0; e < 5; ++e) gh[e] = fs[e];
    } else if (mach >= 1.0) {
      // supersonic outflow: interior values
    } else if (vn < 0.0) {
      const double rc = in[0] * c;
      const double dv = ((fs[1] - in[1]) * nx + (fs[2] - in[2]) * ny) + (fs[3] - in[3]) * nz;
      gh[4] = 0.5 * (fs[4] + in[4] - rc * dv);
      const double dp = fs[4] - gh[4];
      const double rho = fs[0] - dp / (c * c);
      gh[0] = rho * (fs[0] / fs[0]);
      gh[1] = fs[1] - nx * dp / rc;
      gh[2] = fs[2] - ny * dp / rc;
      gh[3] = fs[3] - nz * dp / rc;
    } else {
      const double rc = in[0] * c;
      const double dp = in[4] - fs[4];
      const double rho = in[0] - dp / (c * c);
      gh[0] = rho * (in[0] / in[0]);
      gh[1] = in[1] + nx * dp / rc;
      gh[2] = in[2] + ny * dp / rc;
      gh[3] = in[3] + nz * dp / rc;
      gh[4] = fs[4];
    }
    double t[5];
    ExtrapHold(gh, 2.0, in, t);
    if (layer > 1) ExtrapHold(t, (double)layer, in, gh);
    else for (int e = 0; e < 5; ++e) gh[e] = t[e];
  } else if (bctype == 2) {  // supersonicInflow
    gh[0] = s->rho * 1.0;
    gh[1] = s->u;
    gh[2] = s->v;
    gh[3] = s->w;
    gh[4] = s->p;
  } else if (bctype == 3) {  // supersonicOutflow
    if (layer > 1)
      for (int e = 0; e < 5; ++e) gh[e] = (double)layer * gh[e] - in[e];
  } else if (bctype == 4) {  // stagnationInlet
    const double gm1 = g.gamma - 1.0;
    const double vn = (in[1] * nx + in[2] * ny) + in[3] * nz;
    const double c = SoS(g, in[0], in[4]);
    const double rNeg = vn - 2.0 * c / gm1;
    const double vmag2 = (in[1] * in[1] + in[2] * in[2]) + in[3] * in[3];
    const double cosT = -1.0 * vn / sqrt(vmag2);
    const double stag = c * c + 0.5 * gm1 * vmag2;
    const double sosB = -1.0 * rNeg * gm1 / (gm1 * cosT * cosT + 2.0) *
                        (1.0 + cosT * sqrt((gm1 * cosT * cosT + 2.0) * stag / (gm1 * rNeg * rNeg) -
                                           0.5 * gm1));
    const double ratio = sosB * sosB / stag;
    const double tb = s->t0 * ratio;
    const double pb = s->p0 * PowCR(ratio, g.gamma / gm1);
    const double vb = sqrt(2.0 / gm1 * (s->t0 - tb));
    gh[0] = (pb / (g.R * tb)) * 1.0;
    gh[1] = vb * s->dx;
    gh[2] = vb * s->dy;
    gh[3] = vb * s->dz;
    gh[4] = pb;
    double t[5];
    ExtrapHold(gh, 2.0, in, t);
    if (layer > 1) ExtrapHold(t, (double)layer, in, gh);
    else for (int e = 0; e < 5; ++e) gh[e] = t[e];
  } else if (bctype == 5) {  // pressureOutlet (reflecting)
    const double c = SoS(g, in[0], in[4]);
    const double rc = in[0] * c;
    gh[4] = s->p;
    const double dp = in[4] - gh[4];
    gh[0] = (in[0] - dp / (c * c)) * (in[0] / in[0]);
    gh[1] = in[1] + nx * dp / rc;
    gh[2] = in[2] + ny * dp / rc;
    gh[3] = in[3] + nz * dp / rc;
    const double gvn = (gh[1] * nx + gh[2] * ny) + gh[3] * nz;
    if (gvn / SoS(g, gh[0], gh[4]) >= 1.0)
      for (int e = 0; e < 5; ++e) gh[e] = in[e];
    for (int e = 0; e < 5; ++e) gh[e] = 2.0 * gh[e] - in[e];
    if (layer > 1)
      for (int e = 0; e < 5; ++e) gh[e] = (double)layer * gh[e] - in[e];
  }
}

// Ghost-cell work of every block in one launch: per block, its task list,
// the global index of its first item (a ghost cell, an edge line or a wall
// cell) and its item count; thread t works on the item of the last block
// whose first item is at or before t.
struct BlockTasks {
  const void *tasks;
  long first, count;
  int ntasks;  // tasks in the list (boundary patches)
  int per;     // tasks per item (edge lines)
};
__device__ __forceinline__ int FindTaskBlock(const BlockTasks *bt, int nb, long t) {
  int lo = 0, hi = nb - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (bt[mid].first <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ void __launch_bounds__(256) KBoundary(const DevBlock *__restrict__ blocks,
                                                 const BlockTasks *__restrict__ bt, int nb, long total,
                                                 Gas gas) {
  const long tg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tg >= total) return;
  const int wb = FindTaskBlock(bt, nb, tg);
  const DevBlock &b = blocks[wb];
  const BcTask *__restrict__ tasks = static_cast<const BcTask *>(bt[wb].tasks);
  const int ntasks = bt[wb].ntasks;
  const long t = tg - bt[wb].first;
  int q = 0;
  while (q + 1 < ntasks && tasks[q + 1].base <= t) ++q;
  const BcTask tk = tasks[q];
  const long loc = t - tk.base;
  const int q1 = (int)(loc % tk.n1), q2 = (int)(loc / tk.n1);
  int fi, fj, fk, ci, cj, ck, gi, gj, gk;
  Map3(tk.dir, tk.r3, tk.r1s + q1, tk.r2s + q2, fi, fj, fk);
  Map3(tk.dir, tk.srcC, tk.r1s + q1, tk.r2s + q2, ci, cj, ck);
  Map3(tk.dir, tk.gC, tk.r1s + q1, tk.r2s + q2, gi, gj, gk);
  const double4 a = b.fa[tk.dir][FaceIdx(b, tk.dir, fi, fj, fk)];
  const long src = PadIdx(b, ci, cj, ck), dst = PadIdx(b, gi, gj, gk);
  double in[5], gh[5];
  for (int e = 0; e < 5; ++e) in[e] = b.W[e * b.npad + src];
  const GasT<double> g = Cast<double>(gas);
  GhostState(g, in, tk.bctype, a.x, a.y, a.z, tk.stype, tk.layer,
             tk.state >= 0 ? &b.states[tk.state] : nullptr, gh);
  for (int e = 0; e < 5; ++e) b.W[e * b.npad + dst] = gh[e];
}

// ---------------------------------------------------------------------------
// fused residual: procBlock::CalcInvFluxI/J/K (src/procBlock.cpp:384-769),
// CalcBlockTimeStep (:782-820), linearSolver::AddDiagonalTerms + Invert
// (src/linearSolver.cpp:146-188).
//
// One workgroup per 8x8x4 tile of cells.  The workgroup evaluates every face
// flux that touches the tile exactly once (896 faces: 288 i, 288 j, 320 k),
// keeps F*|A| in LDS, then each thread assembles its cell's residual in the
// reference's accumulation order (-F_i,lo +F_i,hi -F_j,lo +F_j,hi -F_k,lo
// +F_k,hi), the cell spectral radius (i, j, k order), dt, the scalar diagonal
// and its inverse.
constexpr int kTI = 8, kTJ = 8, kTK = 4;
constexpr int kNFI = (kTI + 1) * kTJ * kTK;
constexpr int kNFJ = kTI * (kTJ + 1) * kTK;
constexpr int kNFK = kTI * kTJ * (kTK + 1);
constexpr int kNF = kNFI + kNFJ + kNFK;

// reconstructed lower (WL) and upper (WR) states of the face (i, j, k) of
// direction d (src/procBlock.cpp:384-437)
template <int RECON, int LIM>
__device__ __forceinline__ void FaceStates(const DevBlock &b, double kappa, int d, int i, int j, int k,
                                           double WL[5], double WR[5]) {
  const long s = d == 0 ? 1 : (d == 1 ? (long)b.NI : (long)b.NI * b.NJ);
  const long c0 = PadIdx(b, i, j, k);  // upper cell of the face
  if (RECON == 0) {
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      WL[e] = b.W[e * b.npad + c0 - s];
      WR[e] = b.W[e * b.npad + c0];
    }
  } else if (RECON >= 2) {
    // src/procBlock.cpp:416-430: the lower state from cells -3..+1 around
    // the face, the upper state from +2..-2
    const double *cw = b.cw + d * b.npad;
    double wc[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) wc[q] = cw[c0 + (q - 3) * s];
    const double wl[5] = {wc[0], wc[1], wc[2], wc[3], wc[4]};
    const double wr[5] = {wc[5], wc[4], wc[3], wc[2], wc[1]};
    const WenoGeom GL = MakeWenoGeom(wl), GR = MakeWenoGeom(wr);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const double *We = b.W + e * b.npad + c0;
      double u[6];
#pragma unroll
      for (int q = 0; q < 6; ++q) u[q] = We[(q - 3) * s];
      WL[e] = Weno<RECON == 3>(GL, wl, u[0], u[1], u[2], u[3], u[4]);
      WR[e] = Weno<RECON == 3>(GR, wr, u[5], u[4], u[3], u[2], u[1]);
    }
  } else {
    const double *cw = b.cw + d * b.npad;
    const double wm2 = cw[c0 - 2 * s], wm1 = cw[c0 - s], w0 = cw[c0], wp1 = cw[c0 + s];
    const Divisor<double> byC = MakeDivisor(wm1 + w0);  // the sum is that of w0 + wm1
    const double dPL = Quot(wm1 + wm1, byC), dML = Div(wm1 + wm1, wm1 + wm2);
    const double dPR = Quot(w0 + w0, byC), dMR = Div(w0 + w0, w0 + wp1);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const double *We = b.W + e * b.npad;
      const double um2 = We[c0 - 2 * s], um1 = We[c0 - s], u0 = We[c0], up1 = We[c0 + s];
      WL[e] = Muscl<LIM>(um2, um1, u0, kappa, dPL, dML);
      WR[e] = Muscl<LIM>(up1, u0, um1, kappa, dPR, dMR);
    }
  }
}

// one side of FaceStates: the lower state WL (upper == false) or the upper
// state WR of face (i, j, k) of direction d, with the same arithmetic
template <int RECON, int LIM>
__device__ __forceinline__ void FaceSide(const DevBlock &b, double kappa, int d, int i, int j, int k, bool upper,
                                         double Wout[5]) {
  const long s = d == 0 ? 1 : (d == 1 ? (long)b.NI : (long)b.NI * b.NJ);
  const long c0 = PadIdx(b, i, j, k);
  if (RECON == 0) {
#pragma unroll
    for (int e = 0; e < 5; ++e) Wout[e] = b.W[e * b.npad + c0 - (upper ? 0 : s)];
  } else if (RECON >= 2) {
    const double *cw = b.cw + d * b.npad;
    double wc[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) wc[q] = cw[c0 + (q - 3) * s];
    const double w5[5] = {upper ? wc[5] : wc[0], upper ? wc[4] : wc[1], upper ? wc[3] : wc[2],
                          upper ? wc[2] : wc[3], upper ? wc[1] : wc[4]};
    const WenoGeom G = MakeWenoGeom(w5);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const double *We = b.W + e * b.npad + c0;
      double u[6];
#pragma unroll
      for (int q = 0; q < 6; ++q) u[q] = We[(q - 3) * s];
      Wout[e] = upper ? Weno<RECON == 3>(G, w5, u[5], u[4], u[3], u[2], u[1])
                      : Weno<RECON == 3>(G, w5, u[0], u[1], u[2], u[3], u[4]);
    }
  } else {
    const double *cw = b.cw + d * b.npad;
    const double wm2 = cw[c0 - 2 * s], wm1 = cw[c0 - s], w0 = cw[c0], wp1 = cw[c0 + s];
    if (!upper) {
      const double dPL = Div(wm1 + wm1, wm1 + w0), dML = Div(wm1 + wm1, wm1 + wm2);
#pragma unroll
      for (int e = 0; e < 5; ++e) {
        const double *We = b.W + e * b.npad;
        Wout[e] = Muscl<LIM>(We[c0 - 2 * s], We[c0 - s], We[c0], kappa, dPL, dML);
      }
    } else {
      const double dPR = Div(w0 + w0, w0 + wm1), dMR = Div(w0 + w0, w0 + wp1);
#pragma unroll
      for (int e = 0; e < 5; ++e) {
        const double *We = b.W + e * b.npad;
        Wout[e] = Muscl<LIM>(We[c0 + s], We[c0], We[c0 - s], kappa, dPR, dMR);
      }
    }
  }
}

template <int RECON, int LIM, int FLUX>
__device__ __forceinline__ void FaceFlux(const DevBlock &b, const GasT<double> &g, double kappa,
                                         int d, int i, int j, int k, double F[5]) {
  double WL[5], WR[5];
  FaceStates<RECON, LIM>(b, kappa, d, i, j, k, WL, WR);
  const double4 a = b.fa[d][FaceIdx(b, d, i, j, k)];
  if (FLUX == 0) RoeFlux(g, WL, WR, a.x, a.y, a.z, F);
  else AusmFlux(g, WL, WR, a.x, a.y, a.z, F);
#pragma unroll
  for (int e = 0; e < 5; ++e) F[e] = F[e] * a.w;
}

// CalcCellDt (src/procBlock.cpp:782-820) and AddDiagonalTerms + Invert
// (src/linearSolver.cpp:146-188) for one cell; `sr` is the cell spectral
// radius, `Ad` the accumulated main diagonal
__device__ __forceinline__ void CellTail(const DevBlock &b, const Params &P, long p, double vol, double sr,
                                         double Ad, double *dtOut = nullptr, double *ainvOut = nullptr) {
  b.sr[p] = sr;
  const double dt = P.dtFixed > 0.0 ? P.dtFixed : (*b.cfl) * Div(vol, Dmax(sr, 0.0));
  b.dt[p] = dt;
  if (dtOut) *dtOut = dt;
  if (P.implicit && !P.block) {
    double dvt = Div(vol * (1.0 + P.zeta), dt * P.theta);
    if (P.dualCFL > 0.0) dvt += Div(Dmax(sr, 0.0), P.dualCFL);
    double A = Ad * P.relax;
    A += dvt;
    b.A[p] = A;
    const double ainv = Div(1.0, A);
    if (ainvOut) *ainvOut = P.fp32 ? double((float)ainv) : ainv;
    if (!P.fp32) {
      if (b.Ainv) b.Ainv[p] = ainv;
    } else if (b.Ainv32) {
      b.Ainv32[p] = (float)ainv;
    }
  }
}

// Workgroups are dealt to the eight XCDs in turn (workgroup n to XCD n mod
// 8), and each XCD has its own L2.  Renumbering them so that every XCD
// receives one contiguous range of the work keeps neighbouring tiles, which
// read the same stencil data, in one L2.  A bijection of [0, N) for any N.
__device__ __forceinline__ unsigned XcdRemap(unsigned n, unsigned N) {
  const unsigned q = N / 8u, r = N % 8u, x = n % 8u, l = n / 8u;
  return x * q + min(x, r) + l;
}

// One launch over every block.  Per block, its grid of work units (tiles or
// ranges of cells) and the global index of its first unit; workgroup n, after
// the XCD renumbering, takes unit n of the concatenation, so each XCD works
// on one contiguous range of units across the blocks.
struct BlockMap {
  const DevBlock *blocks;
  const int4 *units;  // per block: (ux, uy, uz, first unit), ux uy uz units
  int nb;
};
struct Unit {
  const DevBlock *b;
  int x, y, z;      // the unit within its block's grid
  unsigned local;   // index within the block (x fastest)
  unsigned global;  // index in the concatenation
};
__device__ __forceinline__ Unit MapUnit(const BlockMap &m) {
  const unsigned n = XcdRemap(blockIdx.x, gridDim.x);
  int lo = 0, hi = m.nb - 1;  // the last block whose first unit is <= n
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((unsigned)m.units[mid].w <= n) lo = mid;
    else hi = mid - 1;
  }
  const int4 u = m.units[lo];
  const unsigned l = n - (unsigned)u.w;
  return {m.blocks + lo, (int)(l % (unsigned)u.x), (int)((l / (unsigned)u.x) % (unsigned)u.y),
          (int)(l / ((unsigned)u.x * (unsigned)u.y)), l, n};
}

// b = -R/theta + forcing + SolDeltaNm1 - SolDeltaMmN
// (src/linearSolver.cpp:360-378, src/procBlock.cpp:1010-1034); forcing is
// zero on the single grid level
// the same from values already loaded (cNm1 is read only when multilevel)
__device__ __forceinline__ void RhsFrom(const Params &P, const double W[5], double vol, double dt,
                                        const double R[5], const double cN[5], const double cNm1[5],
                                        double out[5]) {
#pragma clang fp contract(off)
  const GasT<double> g = Cast<double>(P.gas);
  double U[5];
  PrimToCons(g, W, U);
  const Divisor<double> byDt = MakeDivisor(dt * P.theta);
  const double coeff = Quot(vol * (1.0 + P.zeta), byDt);
  const double thetaInv = 1.0 / P.theta;
  const double c2 = P.multilevel ? Quot(vol * P.zeta, byDt) : 0.0;
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    const double nm1 = P.multilevel ? c2 * (cN[e] - cNm1[e]) : 0.0;
    const double mmn = coeff * (U[e] - cN[e]);
    double v = -thetaInv * R[e];
    out[e] = (v + nm1) - mmn;
  }
}

__device__ __forceinline__ void Rhs(const DevBlock &b, const Params &P, long p, long c,
                                    double out[5]) {
  double W[5], R[5], cN[5], cNm1[5] = {0, 0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    W[e] = b.W[e * b.npad + c];
    R[e] = b.R[e * b.ncell + p];
    cN[e] = b.consN[e * b.ncell + p];
    if (P.multilevel) cNm1[e] = b.consNm1[e * b.ncell + p];
  }
  RhsFrom(P, W, b.vol[p], b.dt[p], R, cN, cNm1, out);
}

// A tile of 256 cells and the axis its block's pencils run along
struct CellTile {
  int pl, n[3];
};
// the tiles' cells (i fastest) by their place in the pencil sweep's records:
// pencil, step, lane
template <int N>
struct TileOrder {
  unsigned char cell[N][256];
};
template <int N>
constexpr TileOrder<N> MakeTileOrder(const CellTile (&tile)[N]) {
  TileOrder<N> o{};
  for (int q = 0; q < N; ++q) {
    const int c = tile[q].pl, a = (c + 1) % 3, b = (c + 2) % 3;
    const int tc = tile[q].n[c], ta = tile[q].n[a], tb = tile[q].n[b];
    int n = 0;
    for (int b0 = 0; b0 < tb; b0 += kPW)
      for (int a0 = 0; a0 < ta; a0 += kPW)
        for (int key = 0; key < (tc + 2 * kPW) * kPenLanes; ++key) {  // step * kPenLanes + lane
          const int la = key % kPW, lb = key / kPW % kPW, cc = key / kPenLanes - la - lb;
          if (cc < 0 || cc >= tc || a0 + la >= ta || b0 + lb >= tb) continue;
          int x[3] = {0, 0, 0};
          x[c] = cc;
          x[a] = a0 + la;
          x[b] = b0 + lb;
          o.cell[q][n++] = (unsigned char)(x[0] + tile[q].n[0] * (x[1] + tile[q].n[1] * x[2]));
        }
  }
  return o;
}
constexpr CellTile kCellTile[3] = {{0, {kTI, kTJ, kTK}}, {1, {kTI, kTJ, kTK}}, {2, {kTI, kTJ, kTK}}};
__constant__ const TileOrder<3> kCellOrder = MakeTileOrder(kCellTile);

template <int RECON, int LIM, int FLUX>
__global__ void __launch_bounds__(256) KResidual(BlockMap M, Params P) {
  __shared__ double sF[5][kNF];
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const int i0 = U.x * kTI, j0 = U.y * kTJ, k0 = U.z * kTK;
  const GasT<double> g = Cast<double>(P.gas);
  for (int f = threadIdx.x; f < kNF; f += blockDim.x) {
    int d, li, lj, lk;
    if (f < kNFI) {
      d = 0; li = f % (kTI + 1); lj = (f / (kTI + 1)) % kTJ; lk = f / ((kTI + 1) * kTJ);
    } else if (f < kNFI + kNFJ) {
      const int q = f - kNFI;
      d = 1; li = q % kTI; lj = (q / kTI) % (kTJ + 1); lk = q / (kTI * (kTJ + 1));
    } else {
      const int q = f - kNFI - kNFJ;
      d = 2; li = q % kTI; lj = (q / kTI) % kTJ; lk = q / (kTI * kTJ);
    }
    const int i = i0 + li, j = j0 + lj, k = k0 + lk;
    const bool ok = (i < b.ni + (d == 0)) && (j < b.nj + (d == 1)) && (k < b.nk + (d == 2));
    if (ok) {
      double F[5];
      FaceFlux<RECON, LIM, FLUX>(b, g, P.kappa, d, i, j, k, F);
#pragma unroll
      for (int e = 0; e < 5; ++e) sF[e][f] = F[e];
    }
  }
  __syncthreads();
  const int li = threadIdx.x % kTI, lj = (threadIdx.x / kTI) % kTJ, lk = threadIdx.x / (kTI * kTJ);
  const int i = i0 + li, j = j0 + lj, k = k0 + lk;
  const bool cell = i < b.ni && j < b.nj && k < b.nk, prep = P.prep && b.pns;
  if (!cell && !prep) return;
  double W[5], R[5], rb[5], ainv;
  if (cell) {
    const int fi = lk * (kTI + 1) * kTJ + lj * (kTI + 1) + li;
    const int fj = kNFI + lk * kTI * (kTJ + 1) + lj * kTI + li;
    const int fk = kNFI + kNFJ + lk * kTI * kTJ + lj * kTI + li;
    const long p = (long)i + (long)j * b.ni + (long)k * b.ni * b.nj;
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      double r = -sF[e][fi];
      r += sF[e][fi + 1];
      r -= sF[e][fj];
      r += sF[e][fj + kTI];
      r -= sF[e][fk];
      r += sF[e][fk + kTI * kTJ];
      b.R[e * b.ncell + p] = R[e] = r;
    }
    const long c = PadIdx(b, i, j, k);
#pragma unroll
    for (int e = 0; e < 5; ++e) W[e] = b.W[e * b.npad + c];
    const double rho = W[0], u = W[1], v = W[2], w = W[3], pr = W[4];
    const double li_ = InvCellSpecRad(g, rho, u, v, w, pr, b.fa[0][FaceIdx(b, 0, i, j, k)],
                                      b.fa[0][FaceIdx(b, 0, i + 1, j, k)]);
    const double lj_ = InvCellSpecRad(g, rho, u, v, w, pr, b.fa[1][FaceIdx(b, 1, i, j, k)],
                                      b.fa[1][FaceIdx(b, 1, i, j + 1, k)]);
    const double lk_ = InvCellSpecRad(g, rho, u, v, w, pr, b.fa[2][FaceIdx(b, 2, i, j, k)],
                                      b.fa[2][FaceIdx(b, 2, i, j, k + 1)]);
    const double sr = (li_ + lj_) + lk_;
    if (P.visc.on) {
      // the viscous pass adds its spectral radii and forms dt and the diagonal
      b.sr[p] = sr;
      return;
    }
    double dt;
    const double vol = b.vol[p];
    CellTail(b, P, p, vol, sr, sr, &dt, &ainv);
    if (prep) {
      double cN[5], cNm1[5] = {0, 0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 5; ++e) {
        cN[e] = b.consN[e * b.ncell + p];
        if (P.multilevel) cNm1[e] = b.consNm1[e * b.ncell + p];
      }
      RhsFrom(P, W, vol, dt, R, cN, cNm1, rb);
    }
  }
  if (!prep) return;
  // the pencil sweep's records of the tile (KPencilPrep's values), through LDS
  // in their order.  Everything but U^n is at hand here: an iteration of 64^3
  // cells 522 us with KPencilPrep (23 us, gathers) in the relax, 506 so; of
  // the eight served cases 393 and 370.
  __syncthreads();
  double(*sh)[256] = (double(*)[256])sF;
  const int tid = threadIdx.x;
  if (cell) {
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      sh[e][tid] = W[e];
      sh[5 + e][tid] = rb[e];
    }
    sh[10][tid] = ainv;
  }
  __syncthreads();
  const int src = kCellOrder.cell[b.pl][tid];
  const int oi = i0 + src % kTI, oj = j0 + src / kTI % kTJ, ok = k0 + src / (kTI * kTJ);
  if (oi >= b.ni || oj >= b.nj || ok >= b.nk) return;
  int lane;
  const long rec = PencilRecord(b, oi, oj, ok, lane);
  double *o = b.skS + rec * kPenS * kPenLanes + lane;
#pragma unroll
  for (int e = 0; e < kPenS; ++e) o[e * kPenLanes] = sh[e][src];
}

// ---------------------------------------------------------------------------
// laminar viscous residual: procBlock::CalcResidualNoSource's viscous branch
// (src/procBlock.cpp:6126-6138)

__device__ __forceinline__ long FacePadIdx(const DevBlock &b, int d, int i, int j, int k) {
  const int FI = b.NI + (d == 0), FJ = b.NJ + (d == 1);
  return (long)(i + b.g) + (long)(j + b.g) * FI + (long)(k + b.g) * FI * FJ;
}

// one ghost cell on a block edge (AssignInviscidGhostCellsEdge,
// src/procBlock.cpp:2565-2714, and AssignViscousGhostCellsEdge, :2874-3030):
// action 0 / 1 reflects q2 / q3 across the slip wall of unit normal n,
// 2 averages q2 and q3, 3 copies q3, 4 copies q2, 5 leaves the cell
struct EdgeTask {
  long gq, q2, q3;
  double nx, ny, nz;
  int action, stype, layer, pad;
};

// one thread per edge line; its tasks run in the reference's layer order
__global__ void __launch_bounds__(64) KEdgeGhosts(const DevBlock *__restrict__ blocks,
                                                  const BlockTasks *__restrict__ bt, int nb, long total, Gas gas) {
  const long tg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tg >= total) return;
  const int wb = FindTaskBlock(bt, nb, tg);
  const DevBlock &b = blocks[wb];
  const EdgeTask *__restrict__ tasks = static_cast<const EdgeTask *>(bt[wb].tasks);
  const int perLine = bt[wb].per;
  const long line = tg - bt[wb].first;
  const GasT<double> g = Cast<double>(gas);
  for (int q = 0; q < perLine; ++q) {
    const EdgeTask t = tasks[(long)line * perLine + q];
    if (t.action == 5) continue;
    double a[5], c[5], gh[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      a[e] = b.W[e * b.npad + t.q2];
      c[e] = b.W[e * b.npad + t.q3];
    }
    if (t.action == 0) GhostState(g, a, 0, t.nx, t.ny, t.nz, t.stype, t.layer, nullptr, gh);
    else if (t.action == 1) GhostState(g, c, 0, t.nx, t.ny, t.nz, t.stype, t.layer, nullptr, gh);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const double v = t.action <= 1 ? gh[e] : (t.action == 2 ? 0.5 * (a[e] + c[e]) : (t.action == 3 ? c[e] : a[e]));
      b.W[e * b.npad + t.gq] = v;
    }
  }
}

// GetGhostState, viscousWall, low-Re treatment (src/ghostStates.cpp:126-145,
// 185-190): velocity mirrored about the wall velocity; an isothermal wall sets
// the density from the mirrored temperature at the interior pressure
struct WallTask {
  long src, dst;
  int state, pad;
  double wd;  // wall distance of the wall-adjacent cell (heat-flux walls)
};

__global__ void __launch_bounds__(256) KViscWall(const DevBlock *__restrict__ blocks,
                                                 const BlockTasks *__restrict__ bt, int nb, long total,
                                                 Gas gas, ViscParams vp) {
  const long tg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tg >= total) return;
  const int wb = FindTaskBlock(bt, nb, tg);
  const DevBlock &b = blocks[wb];
  const WallTask *__restrict__ tasks = static_cast<const WallTask *>(bt[wb].tasks);
  const WallTask w = tasks[tg - bt[wb].first];
  const BcStateDev *s = w.state >= 0 ? &b.states[w.state] : nullptr;
  double in[5], gh[5];
#pragma unroll
  for (int e = 0; e < 5; ++e) gh[e] = in[e] = b.W[e * b.npad + w.src];
  const double vx = s ? s->u : 0.0, vy = s ? s->v : 0.0, vz = s ? s->w : 0.0;
  gh[1] = 2.0 * vx - in[1];
  gh[2] = 2.0 * vy - in[2];
  gh[3] = 2.0 * vz - in[3];
  if (s && s->iso) {
    const GasT<double> g = Cast<double>(gas);
    const double tGhost = 2.0 * s->tw - TempOf(g, in[0], in[4]);
    const double R = 0.0 + 1.0 * g.R;
    gh[0] = (gh[4] / (R * tGhost)) * (in[0] / (0.0 + in[0]));
  } else if (s && s->flux) {
    // constant heat flux, low-Re treatment (src/ghostStates.cpp:228-238):
    // the interior temperature less q / k times twice the wall distance of
    // the wall-adjacent cell, k = Sutherland conductivity times the scaling
    const GasT<double> g = Cast<double>(gas);
    const double t = TempOf(g, in[0], in[4]);
    const double kappa = SutherlandK(vp, t) * vp.vscale;
    const double tGhost = TempOf(g, in[0], in[4]) - s->qw / kappa * 2.0 * w.wd;
    const double R = 0.0 + 1.0 * g.R;
    gh[0] = (gh[4] / (R * tGhost)) * (in[0] / (0.0 + in[0]));
  }
#pragma unroll
  for (int e = 0; e < 5; ++e) b.W[e * b.npad + w.dst] = gh[e];
}

// UpdateAuxillaryVariables (src/procBlock.cpp:6171-6189): temperature and
// viscosity of every cell but the block corners
__global__ void __launch_bounds__(256) KAux(BlockMap M, Params P) {
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const long q = (long)U.local * blockDim.x + threadIdx.x;
  if (q >= b.npad) return;
  const int i = (int)(q % b.NI) - b.g, j = (int)((q / b.NI) % b.NJ) - b.g, k = (int)(q / ((long)b.NI * b.NJ)) - b.g;
  const bool corner = (i < 0 || i >= b.ni) && (j < 0 || j >= b.nj) && (k < 0 || k >= b.nk);
  if (corner) return;
  const double t = TempOf(Cast<double>(P.gas), b.W[q], b.W[4 * b.npad + q]);
  b.T[q] = t;
  b.mu[q] = SutherlandMu(P.visc, t);
  if (b.kc) b.kc[q] = SutherlandK(P.visc, t);  // read by the block Jacobians
}

// The cell values the viscous face terms read (velocity components and
// temperature, padded volume, state, viscosity), from the block's padded
// arrays (CellsG) or staged in LDS for a box of cells (CellsL: eight arrays
// of n cells, rho, u, v, w, p, T, volume, viscosity, the box's cell (i0, j0,
// k0) first).  The values are the same doubles either way.
struct CellsG {
  const DevBlock &b;
  __device__ __forceinline__ long At(int i, int j, int k) const { return PadIdx(b, i, j, k); }
  __device__ __forceinline__ double Var(int v, long c) const { return (v < 3 ? b.W + (v + 1) * b.npad : b.T)[c]; }
  __device__ __forceinline__ double Vol(long c) const { return b.volP[c]; }
  __device__ __forceinline__ double State(int e, long c) const { return b.W[e * b.npad + c]; }
  __device__ __forceinline__ double Mu(long c) const { return b.mu[c]; }
};
struct CellsL {
  const double *s;
  int i0, j0, k0, sx, sy, n;
  __device__ __forceinline__ long At(int i, int j, int k) const {
    return (i - i0) + sx * ((j - j0) + (long)sy * (k - k0));
  }
  __device__ __forceinline__ double Var(int v, long c) const { return s[(v < 3 ? v + 1 : 5) * n + c]; }
  __device__ __forceinline__ double Vol(long c) const { return s[6 * n + c]; }
  __device__ __forceinline__ double State(int e, long c) const { return s[e * n + c]; }
  __device__ __forceinline__ double Mu(long c) const { return s[7 * n + c]; }
};

// CalcGradsI/J/K at a face (src/procBlock.cpp:5173-5788) with VectorGradGG /
// ScalarGradGG (src/utility.cpp:59-188): Green-Gauss over the control volume
// spanning the face's lower cell L and upper cell U; velocity gradient
// vg[r][c] = d v_c / d x_r, temperature gradient tg
template <class C>
__device__ __forceinline__ void FaceGrads(const DevBlock &b, const C &cv, int d, int i, int j, int k,
                                          double vg[3][3], double tg[3]) {
  const int L[3] = {i - (d == 0), j - (d == 1), k - (d == 2)}, U[3] = {i, j, k};
  const long cL = cv.At(L[0], L[1], L[2]), cU = cv.At(U[0], U[1], U[2]);
  const double vol = 0.5 * (cv.Vol(cL) + cv.Vol(cU));
  // Green-Gauss over the control volume's three face pairs: each entry is
  // the sum, left to right, of +vu au - vl al for the pairs q = 0, 1, 2, so
  // it is accumulated one pair at a time
  double acc[3][4];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int eq[3] = {q == 0, q == 1, q == 2};
    const double4 *F = b.faP[q];
    double4 f1, f2, f3, f4;
    if (q == d) {
      f1 = F[FacePadIdx(b, q, U[0], U[1], U[2])];
      f2 = F[FacePadIdx(b, q, U[0] + eq[0], U[1] + eq[1], U[2] + eq[2])];
      f3 = f1;
      f4 = F[FacePadIdx(b, q, L[0], L[1], L[2])];
    } else {
      f1 = F[FacePadIdx(b, q, U[0] + eq[0], U[1] + eq[1], U[2] + eq[2])];
      f2 = F[FacePadIdx(b, q, L[0] + eq[0], L[1] + eq[1], L[2] + eq[2])];
      f3 = F[FacePadIdx(b, q, U[0], U[1], U[2])];
      f4 = F[FacePadIdx(b, q, L[0], L[1], L[2])];
    }
    double au[3], al[3];
    au[0] = 0.5 * (f1.x * f1.w + f2.x * f2.w);
    au[1] = 0.5 * (f1.y * f1.w + f2.y * f2.w);
    au[2] = 0.5 * (f1.z * f1.w + f2.z * f2.w);
    al[0] = 0.5 * (f3.x * f3.w + f4.x * f4.w);
    al[1] = 0.5 * (f3.y * f3.w + f4.y * f4.w);
    al[2] = 0.5 * (f3.z * f3.w + f4.z * f4.w);
    // face values of the pair: three velocity components, then temperature
    const long uP = cv.At(U[0] + eq[0], U[1] + eq[1], U[2] + eq[2]);
    const long lP = cv.At(L[0] + eq[0], L[1] + eq[1], L[2] + eq[2]);
    const long uM = cv.At(U[0] - eq[0], U[1] - eq[1], U[2] - eq[2]);
    const long lM = cv.At(L[0] - eq[0], L[1] - eq[1], L[2] - eq[2]);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const double xl = cv.Var(v, cL), xu = cv.Var(v, cU);
      double vu, vl;
      if (q == d) {
        vu = xu;
        vl = xl;
      } else {
        vu = 0.25 * (xl + xu + cv.Var(v, uP) + cv.Var(v, lP));
        vl = 0.25 * (xl + xu + cv.Var(v, uM) + cv.Var(v, lM));
      }
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        if (q == 0) acc[r][v] = vu * au[r] - vl * al[r];
        else acc[r][v] = acc[r][v] + vu * au[r] - vl * al[r];
      }
    }
  }
  const double invVol = Div(1.0, vol);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
#pragma unroll
    for (int c = 0; c < 3; ++c) vg[r][c] = acc[r][c] * invVol;
    tg[r] = acc[r][3] * invVol;
  }
}

// viscous flux through face (d, i, j, k) times its area: central or
// fourth-order face state and viscosity (include/reconstruction.hpp:314-349),
// viscousFlux::CalcFlux / CalcWallFlux (src/viscousFlux.cpp:58-188),
// TauNormal (src/utility.cpp:426-436); the wall form has no +0 species term
// (the fourth-order state reads the cells two away from the face, which a
// staged box does not hold: it always reads the block's arrays)
template <bool R4, class C>
__device__ __forceinline__ void ViscFaceState(const DevBlock &b, const C &cv, int d, int i, int j, int k,
                                              double Wf[5], double &muF) {
#pragma clang fp contract(off)
  const long s = d == 0 ? 1 : (d == 1 ? (long)b.NI : (long)b.NI * b.NJ);
  const long cU = PadIdx(b, i, j, k), cL = cU - s;
  const double *cw = b.cw + d * b.npad;
  if (!R4) {
    const double w[2] = {cw[cL], cw[cU]};
    const double c0 = LagrangeCoeffN<2, 1, 0, 0>(w, 0), c1 = LagrangeCoeffN<2, 1, 0, 0>(w, 1);
    const long vU = cv.At(i, j, k), vL = cv.At(i - (d == 0), j - (d == 1), k - (d == 2));
#pragma unroll
    for (int e = 0; e < 5; ++e) Wf[e] = c0 * cv.State(e, vU) + c1 * cv.State(e, vL);
    muF = c0 * cv.Mu(vU) + c1 * cv.Mu(vL);
  } else {
    const long cLL = cL - s, cUU = cU + s;
    const double w[4] = {cw[cLL], cw[cL], cw[cU], cw[cUU]};
    double c[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) c[q] = LagrangeCoeffN<4, 3, 1, 1>(w, q);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const double *We = b.W + e * b.npad;
      Wf[e] = c[0] * We[cLL] + c[1] * We[cL] + c[2] * We[cU] + c[3] * We[cUU];
    }
    muF = c[0] * b.mu[cLL] + c[1] * b.mu[cL] + c[2] * b.mu[cU] + c[3] * b.mu[cUU];
  }
}

template <bool R4>
__device__ __forceinline__ void ViscFaceState(const DevBlock &b, int d, int i, int j, int k, double Wf[5],
                                              double &muF) {
  ViscFaceState<R4>(b, CellsG{b}, d, i, j, k, Wf, muF);
}

template <bool R4, class C>
__device__ __forceinline__ void ViscFaceFlux(const DevBlock &b, const C &cv, const Params &P, int d, int i, int j,
                                             int k, double F[5]) {
#pragma clang fp contract(off)
  const GasT<double> g = Cast<double>(P.gas);
  double vg[3][3], tg[3];
  FaceGrads(b, cv, d, i, j, k, vg, tg);
  const int n3 = d == 0 ? b.ni : (d == 1 ? b.nj : b.nk);
  const int f3 = d == 0 ? i : (d == 1 ? j : k);
  const bool wall = (f3 == 0 || f3 == n3) && b.wallf[BtSlot(b, d, f3 == 0 ? 0 : 1, i, j, k)];
  double Wf[5], muF;
  ViscFaceState<R4>(b, cv, d, i, j, k, Wf, muF);
  const long fq = FaceIdx(b, d, i, j, k);
  const double4 a = b.fa[d][fq];
  const double n[3] = {a.x, a.y, a.z};
  const double mu = P.visc.vscale * muF, mut = P.visc.vscale * 0.0;
  const double lambda = 0.0 - (2.0 / 3.0) * (mu + mut);
  const double trace = vg[0][0] + vg[1][1] + vg[2][2];
  double tau[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double s0 = vg[r][0] + vg[0][r], s1 = vg[r][1] + vg[1][r], s2 = vg[r][2] + vg[2][r];
    const double sa = s0 * n[0] + s1 * n[1] + s2 * n[2];
    tau[r] = lambda * trace * n[r] + (mu + mut) * sa;
  }
  const double t = TempOf(g, Wf[0], Wf[4]);
  const double kLam = SutherlandK(P.visc, t);
  const double kk = kLam * P.visc.vscale;
  const double kt = mut * g.cps / 0.9;
  if (b.fvis[0]) {
    const long nf = (long)(b.ni + (d == 0)) * (b.nj + (d == 1)) * (b.nk + (d == 2));
    double *o = b.fvis[d];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) o[(r * 3 + c) * nf + fq] = vg[r][c];
  }
  const double tv = tau[0] * Wf[1] + tau[1] * Wf[2] + tau[2] * Wf[3];
  const double q = (kk + kt) * (tg[0] * n[0] + tg[1] * n[1] + tg[2] * n[2]);
  F[0] = 0.0 * a.w;
  F[1] = tau[0] * a.w;
  F[2] = tau[1] * a.w;
  F[3] = tau[2] * a.w;
  F[4] = (wall ? tv + q : tv + q + 0.0) * a.w;
}

// fluxJacobian::ApproxTSLJacobian (include/fluxJacobian.hpp:666-758) for a
// laminar single species (diffusion coefficient 0, mass fraction 1), times
// DelprimitiveDelConservative (:612-662) on the right (MatrixMultiply,
// src/matrix.cpp:186-199).  `left` gives the shear term the lower cell's
// sign; vg is the velocity gradient d v_c / d x_r at [3 r + c].
// kLam is Sutherland's conductivity at the state's temperature before the
// nondimensional scaling (formed once per cell or face by the kernels that
// hold it).
__device__ __forceinline__ void TSLJacobian(const GasT<double> &g, const ViscParams &vp, const double W[5],
                                            double muLam, double kLam, double4 a, double dist, bool left,
                                            const double vg[9], double out[25]) {
#pragma clang fp contract(off)
  const double t = TempOf(g, W[0], W[4]);
  const double mu = vp.vscale * muLam, mut = vp.vscale * 0.0;
  const double nx = a.x, ny = a.y, nz = a.z;
  const double u = W[1], v = W[2], w = W[3];
  const double vn = (u * nx + v * ny) + w * nz;
  const double rho = W[0];  // (one species: the reference's sum from +0 is the same for rho > 0)
  const double k = kLam * vp.vscale;
  const double kt = mut * g.cps / 0.9;
  // TauNormal (src/utility.cpp:426-436)
  const double lambda = 0.0 - (2.0 / 3.0) * (mu + mut);
  const double trace = vg[0] + vg[4] + vg[8];
  const double n[3] = {nx, ny, nz};
  double tau[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double s0 = vg[r * 3 + 0] + vg[r], s1 = vg[r * 3 + 1] + vg[3 + r], s2 = vg[r * 3 + 2] + vg[6 + r];
    const double sa = s0 * n[0] + s1 * n[1] + s2 * n[2];
    tau[r] = lambda * trace * n[r] + (mu + mut) * sa;
  }
  const double fac = left ? -1.0 : 1.0;
  const double third = 1.0 / 3.0;
  const double mr = (mu + mut) * rho;
  double J[25];
#pragma unroll
  for (int q = 0; q < 25; ++q) J[q] = 0.0;
  const Divisor<double> byMr = MakeDivisor(mr);
  // (J[0], the species' diffusion term 0 (1 - rho_s / rho) / mr, is zero with one
  // species, and so is what it adds to J[20])
  J[20] = Quot(-(k + kt) * t, byMr);
  const double sh = Div(fac * 0.5 * dist, mu + mut);
  J[6] = third * nx * nx + 1.0;
  J[11] = third * nx * ny;
  J[16] = third * nx * nz;
  J[21] = sh * tau[0] + third * nx * vn + u;
  J[7] = third * ny * nx;
  J[12] = third * ny * ny + 1.0;
  J[17] = third * ny * nz;
  J[22] = sh * tau[1] + third * ny * vn + v;
  J[8] = third * nz * nx;
  J[13] = third * nz * ny;
  J[18] = third * nz * nz + 1.0;
  J[23] = sh * tau[2] + third * nz * vn + w;
  J[24] = Quot(k + kt, byMr);
  const double f = Div(a.w * (mu + mut), dist);
#pragma unroll
  for (int q = 0; q < 25; ++q) J[q] *= f;
  // DelprimitiveDelConservative: its nonzero entries (row-major index)
  const double gm1 = g.gamma - 1.0;
  const double invRho = Div(1.0, rho);
  const double p5 = -invRho * u, p10 = -invRho * v, p15 = -invRho * w;
  const double p20 = 0.5 * gm1 * ((u * u + v * v) + w * w);
  const double p6 = invRho, p12 = invRho, p18 = invRho;
  const double p21 = -gm1 * u, p22 = -gm1 * v, p23 = -gm1 * w, p24 = gm1;
  // J times it, the row-by-column sums from +0 of the 5x5x5 product with the
  // products of structural zeros left out: row 0 of J is +-0, so is its
  // first and last column in rows 1-3, and the product matrix is zero off
  // its first column, diagonal and last row.  A sum from +0 of finite terms
  // is never -0 and is unchanged by adding +-0, so each entry equals the
  // full product's bit for bit.
#pragma unroll
  for (int q = 0; q < 25; ++q) out[q] = 0.0;
#pragma unroll
  for (int r = 1; r < 4; ++r) {
    out[r * 5 + 0] = (J[r * 5 + 1] * p5 + J[r * 5 + 2] * p10) + J[r * 5 + 3] * p15;
    out[r * 5 + 1] = J[r * 5 + 1] * p6;
    out[r * 5 + 2] = J[r * 5 + 2] * p12;
    out[r * 5 + 3] = J[r * 5 + 3] * p18;
  }
  out[20] = (((J[20] + J[21] * p5) + J[22] * p10) + J[23] * p15) + J[24] * p20;
  out[21] = J[21] * p6 + J[24] * p21;
  out[22] = J[22] * p12 + J[24] * p22;
  out[23] = J[23] * p18 + J[24] * p23;
  out[24] = J[24] * p24;
}

// procBlock::CalcViscFluxI/J/K (src/procBlock.cpp:1233-2135), laminar.  The
// same 8x8x4 tiling as KResidual: every viscous face flux of the tile once
// into LDS, then each cell adds them to its residual in the reference's order
// (+Fv_i,lo -Fv_i,hi +Fv_j,lo -Fv_j,hi +Fv_k,lo -Fv_k,hi), adds the viscous
// spectral radii (i, j, k) to its spectral radius (times the viscous CFL
// coefficient) and twice them to its diagonal, then forms dt and A.
constexpr int kVX = kTI + 2, kVY = kTJ + 2, kVZ = kTK + 2, kVN = kVX * kVY * kVZ;
template <bool R4>
__global__ void __launch_bounds__(256) KViscFlux(BlockMap M, Params P) {
  __shared__ double sF[5][kNF];
  // the tile's cells and one layer around them: every cell a face gradient
  // or a central face state of the tile reads
  __shared__ double sC[8][kVN];
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const int i0 = U.x * kTI, j0 = U.y * kTJ, k0 = U.z * kTK;
  for (int q = threadIdx.x; q < kVN; q += blockDim.x) {
    const int i = i0 - 1 + q % kVX, j = j0 - 1 + (q / kVX) % kVY, k = k0 - 1 + q / (kVX * kVY);
    // positions past a partial tile's padded extent are never read
    if (i < b.ni + b.g && j < b.nj + b.g && k < b.nk + b.g) {
      const long c = PadIdx(b, i, j, k);
#pragma unroll
      for (int e = 0; e < 5; ++e) sC[e][q] = b.W[e * b.npad + c];
      sC[5][q] = b.T[c];
      sC[6][q] = b.volP[c];
      sC[7][q] = b.mu[c];
    }
  }
  __syncthreads();
  const CellsL cv{&sC[0][0], i0 - 1, j0 - 1, k0 - 1, kVX, kVY, kVN};
  for (int f = threadIdx.x; f < kNF; f += blockDim.x) {
    int d, li, lj, lk;
    if (f < kNFI) {
      d = 0; li = f % (kTI + 1); lj = (f / (kTI + 1)) % kTJ; lk = f / ((kTI + 1) * kTJ);
    } else if (f < kNFI + kNFJ) {
      const int q = f - kNFI;
      d = 1; li = q % kTI; lj = (q / kTI) % (kTJ + 1); lk = q / (kTI * (kTJ + 1));
    } else {
      const int q = f - kNFI - kNFJ;
      d = 2; li = q % kTI; lj = (q / kTI) % kTJ; lk = q / (kTI * kTJ);
    }
    const int i = i0 + li, j = j0 + lj, k = k0 + lk;
    const bool ok = (i < b.ni + (d == 0)) && (j < b.nj + (d == 1)) && (k < b.nk + (d == 2));
    if (ok) {
      double F[5];
      ViscFaceFlux<R4>(b, cv, P, d, i, j, k, F);
#pragma unroll
      for (int e = 0; e < 5; ++e) sF[e][f] = F[e];
    }
  }
  __syncthreads();
  const int li = threadIdx.x % kTI, lj = (threadIdx.x / kTI) % kTJ, lk = threadIdx.x / (kTI * kTJ);
  const int i = i0 + li, j = j0 + lj, k = k0 + lk;
  if (i >= b.ni || j >= b.nj || k >= b.nk) return;
  const int fi = lk * (kTI + 1) * kTJ + lj * (kTI + 1) + li;
  const int fj = kNFI + lk * kTI * (kTJ + 1) + lj * kTI + li;
  const int fk = kNFI + kNFJ + lk * kTI * kTJ + lj * kTI + li;
  const long p = (long)i + (long)j * b.ni + (long)k * b.ni * b.nj;
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    double r = b.R[e * b.ncell + p];
    r += sF[e][fi];
    r -= sF[e][fi + 1];
    r += sF[e][fj];
    r -= sF[e][fj + kTI];
    r += sF[e][fk];
    r -= sF[e][fk + kTI * kTJ];
    b.R[e * b.ncell + p] = r;
  }
  const GasT<double> g = Cast<double>(P.gas);
  const long c = PadIdx(b, i, j, k);
  double W[5];
#pragma unroll
  for (int e = 0; e < 5; ++e) W[e] = b.W[e * b.npad + c];
  const double vol = b.vol[p], mu = b.mu[c];
  double sr = b.sr[p], Ad = sr;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int ei = d == 0, ej = d == 1, ek = d == 2;
    const double v = ViscCellSR(g, W, b.fa[d][FaceIdx(b, d, i, j, k)].w,
                                b.fa[d][FaceIdx(b, d, i + ei, j + ej, k + ek)].w, vol, mu, P.visc);
    sr += v * P.visc.coeff;
    if (P.implicit) Ad += 2.0 * v;
  }
  CellTail(b, P, p, vol, sr, Ad);
}
// ---------------------------------------------------------------------------
// implicit operator

// values of a block solver's record: state, right-hand side, and with the
// viscous terms viscosity, conductivity and velocity gradient
__host__ __device__ constexpr int BlockRecord(bool viscous) { return viscous ? 21 : 10; }

// The block diagonal's tiles.  Each record takes a cell's values 512 bytes apart, its lanes from as many rows, so
// stores straight from the cells are single words: KBlockDiag on 1.03M cells
// 800 us.  Through LDS in the records' order they are runs of up to eight lanes:
// 534 us (8 x 8 x 4 tiles 554, 16 x 8 x 1 590, a wave's 8 x 8 cells 803),
// against 395 us without any records, which the sweep's two passes (508 -> 353
// us) and the initialisation gone from the relax pay for.  The first tile of an
// axis is the one for blocks thick along every axis; a tile chosen by that axis
// alone left 8 of 256 threads with a cell where ni = 1 and k is longest (the
// rule is DiagTile's, beside the launches).
constexpr int kDiagTiles = 11;
constexpr CellTile kDiagTile[kDiagTiles] = {
    {0, {32, 8, 1}}, {1, {8, 8, 4}},  {2, {32, 1, 8}}, {0, {32, 1, 8}},  {0, {256, 1, 1}}, {1, {8, 32, 1}},
    {1, {1, 32, 8}}, {1, {1, 256, 1}}, {2, {8, 4, 8}}, {2, {1, 8, 32}}, {2, {1, 1, 256}}};
__constant__ const TileOrder<kDiagTiles> kTileOrder = MakeTileOrder(kDiagTile);
constexpr int Log2(int n) { return n > 1 ? 1 + Log2(n / 2) : 0; }
struct TileShift {
  unsigned char i[kDiagTiles], j[kDiagTiles], k[kDiagTiles];
};
constexpr TileShift MakeTileShift() {
  TileShift s{};
  for (int q = 0; q < kDiagTiles; ++q) {
    s.i[q] = (unsigned char)Log2(kDiagTile[q].n[0]);
    s.j[q] = (unsigned char)Log2(kDiagTile[q].n[1]);
    s.k[q] = (unsigned char)Log2(kDiagTile[q].n[2]);
  }
  return s;
}
__constant__ const TileShift kTileShift = MakeTileShift();
// cell `t` of tile U
__device__ __forceinline__ void DiagCell(const DevBlock &b, const Unit &U, int t, int &i, int &j, int &k) {
  const int si = kTileShift.i[b.dtile], sj = kTileShift.j[b.dtile], sk = kTileShift.k[b.dtile];
  i = (U.x << si) + (t & ((1 << si) - 1));
  j = (U.y << sj) + ((t >> si) & ((1 << sj) - 1));
  k = (U.z << sk) + (t >> (si + sj));
}

// Block main diagonal (src/procBlock.cpp:449-486, 588-625, 726-763):
// every face adds the Rusanov Jacobian of its lower state to its lower cell
// and subtracts that of its upper state from its upper cell, faces in i, j, k
// order, so a cell sees -J(face i-) +J(face i+) -J(j-) +J(j+) -J(k-) +J(k+)
// from a zero matrix.  Then AddDiagonalTerms (src/linearSolver.cpp:146-171)
// and the Gauss-Jordan inverse (src/linearSolver.cpp:173-184).  One thread per
// cell of a tile, after the residual kernels have written sr and dt.  A zero pivot sets
// bit 4 of `flag`.
//
// MODE 0: the inviscid sum, then AddDiagonalTerms and the inverse.
// With the viscous terms the inviscid sum must see the inviscid ghost states
// (a viscousWall is a slip wall there).  The cells whose face states reach a
// viscousWall ghost (`invPark`) form it right after the inviscid residual
// kernel and park it in Ab (MODE 1); after the viscous pass MODE 2 (central)
// or 3 (fourth-order face states) takes the parked sum or forms the sum
// itself (every other cell: its face states read no ghost cell that the
// viscous pass changes, so the sum is the same bits), adds the viscous
// faces' thin-shear-layer Jacobians, the cell as upper cell adding
// (src/procBlock.cpp:1467-1474) and as lower cell subtracting (:1416-1424),
// stores the cell velocity gradient, a sixth of each face's in the same order
// (:1396-1414, 1427-1436), and finishes.  Bound by latency: two waves a SIMD (its
// registers), VALU 38 % busy, 1.75 GB at 3.4 TB/s on the 1.03M-cell channel.
template <int RECON, int LIM, int MODE>
__global__ void __launch_bounds__(MODE == 1 ? 128 : 256, MODE == 3 && RECON < 2 ? 2 : 1) KBlockDiag(BlockMap M, Params P) {
#pragma clang fp contract(off)
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const int tid = threadIdx.x;
  const bool tiled = MODE != 1 && b.pns;
  long p = (long)U.local * blockDim.x + tid;
  int i, j, k;
  if (tiled) {
    DiagCell(b, U, tid, i, j, k);
    p = i + (long)b.ni * (j + (long)b.nj * k);
  } else {
    i = (int)(p % b.ni);
    j = (int)((p / b.ni) % b.nj);
    k = (int)(p / ((long)b.ni * b.nj));
  }
  const bool cell = i < b.ni && j < b.nj && k < b.nk;
  if (!tiled && !cell) return;
  const long c = PadIdx(b, i, j, k);
  const bool parked = MODE >= 1 && cell && b.invPark && b.invPark[p];
  if (MODE == 1 && !parked) return;
  if (cell) {
    const GasT<double> g = Cast<double>(P.gas);
    double D[25];
#pragma unroll
    for (int q = 0; q < 25; ++q) D[q] = MODE >= 2 && parked ? b.Ab[q * b.ncell + p] : 0.0;
    if (!(MODE >= 2 && parked)) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        // the cell is the upper cell of its lower face (upper state WR) and the
        // lower cell of its upper face (lower state WL): one side of each
        double Wf[5], J[25];
        FaceSide<RECON, LIM>(b, P.kappa, d, i, j, k, true, Wf);
        double4 a = b.fa[d][FaceIdx(b, d, i, j, k)];
        RusanovJacobian<double>(g, Wf, a.x, a.y, a.z, a.w, false, J);
#pragma unroll
        for (int q = 0; q < 25; ++q) D[q] = D[q] - J[q];
        const int ui = i + (d == 0), uj = j + (d == 1), uk = k + (d == 2);
        FaceSide<RECON, LIM>(b, P.kappa, d, ui, uj, uk, false, Wf);
        a = b.fa[d][FaceIdx(b, d, ui, uj, uk)];
        RusanovJacobian<double>(g, Wf, a.x, a.y, a.z, a.w, true, J);
#pragma unroll
        for (int q = 0; q < 25; ++q) D[q] = D[q] + J[q];
      }
    }
    if (MODE == 1) {
#pragma unroll
      for (int q = 0; q < 25; ++q) b.Ab[q * b.ncell + p] = D[q];
      return;
    }
    if (MODE >= 2) {
      constexpr double sixth = 1.0 / 6.0;
      double G[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) G[q] = 0.0;
#pragma unroll 1
      for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int side = 0; side < 2; ++side) {
          const int fi = i + (side && d == 0), fj = j + (side && d == 1), fk = k + (side && d == 2);
          const long fq = FaceIdx(b, d, fi, fj, fk);
          const long nf = (long)(b.ni + (d == 0)) * (b.nj + (d == 1)) * (b.nk + (d == 2));
          // the face's gradient as the viscous pass formed it; its state,
          // viscosity and conductivity formed again, as that pass forms them
          const double *fv = b.fvis[d];
          double vgr[9], Wf[5], J[25], muF;
#pragma unroll
          for (int q = 0; q < 9; ++q) vgr[q] = fv[q * nf + fq];
          ViscFaceState<MODE == 3>(b, d, fi, fj, fk, Wf, muF);
          const double kF = SutherlandK(P.visc, TempOf(g, Wf[0], Wf[4]));
          TSLJacobian(g, P.visc, Wf, muF, kF, b.fa[d][fq], b.c2c[d][fq], side == 1, vgr, J);
#pragma unroll
          for (int q = 0; q < 25; ++q) D[q] = side ? D[q] - J[q] : D[q] + J[q];
#pragma unroll
          for (int q = 0; q < 9; ++q) G[q] += sixth * vgr[q];
        }
      }
#pragma unroll
      for (int q = 0; q < 9; ++q) b.vgrad[q * b.npad + c] = G[q];
    }
    const double sr = b.sr[p];
    double dvt = Div(b.vol[p] * (1.0 + P.zeta), b.dt[p] * P.theta);
    if (P.dualCFL > 0.0) dvt += Div(Dmax(sr, 0.0), P.dualCFL);
#pragma unroll
    for (int q = 0; q < 5; ++q) D[q * 6] *= P.relax;
#pragma unroll
    for (int q = 0; q < 5; ++q) D[q * 6] += dvt;
#pragma unroll
    for (int q = 0; q < 25; ++q) b.Ab[q * b.ncell + p] = D[q];
    double I[25];
    if (!GJInverse5<double>(D, I)) atomicOr(b.flag, 4);
    int stride;
    const long ib = InverseBase<double>(b, i, j, k, stride), ib32 = InverseBase<float>(b, i, j, k, stride);
    float If[25];
#pragma unroll
    for (int q = 0; q < 25; ++q) If[q] = float(I[q]);
    const bool f32 = P.fp32 && b.Abi32;
    if (b.pns) {
      PutVecs<double, 25>(b.Abi + ib, I);
      if (f32) PutVecs<float, 25>(b.Abi32 + ib32, If);
    } else {
#pragma unroll
      for (int q = 0; q < 25; ++q) b.Abi[ib + (long)q * stride] = I[q];
      if (f32) {
#pragma unroll
        for (int q = 0; q < 25; ++q) b.Abi32[ib32 + (long)q * stride] = If[q];
      }
    }
  }
  if (!b.pns) return;
  // what the pencil sweep forms the off-diagonal blocks and the right-hand
  // side from; this thread writes cell (oi, oj, ok)
  constexpr int nr = BlockRecord(MODE >= 2);
  __shared__ double sh[nr][256];
  if (cell) {
#pragma unroll
    for (int e = 0; e < 5; ++e) sh[e][tid] = b.W[e * b.npad + c];
    if (P.rhsInDiag) {
      // the initialisation of a one-sweep relax, from the values at hand
      double rb[5];
      Rhs(b, P, p, c, rb);
#pragma unroll
      for (int e = 0; e < 5; ++e) sh[5 + e][tid] = rb[e];
    }
    if constexpr (MODE >= 2) {
      sh[10][tid] = b.mu[c];
      sh[11][tid] = b.kc[c];
#pragma unroll
      for (int q = 0; q < 9; ++q) sh[12 + q][tid] = b.vgrad[q * b.npad + c];
    }
  }
  __syncthreads();
  const int src = kTileOrder.cell[b.dtile][tid];
  int oi, oj, ok, lane;
  DiagCell(b, U, src, oi, oj, ok);
  if (oi >= b.ni || oj >= b.nj || ok >= b.nk) return;
  double *o = b.skS + PencilRecord(b, oi, oj, ok, lane) * nr * kPenLanes;
  o += lane;
#pragma unroll
  for (int e = 0; e < nr; ++e)
    if (e < 5 || e >= 10 || P.rhsInDiag) o[e * kPenLanes] = sh[e][src];
}

// RusanovBlockOffDiagonal (src/fluxJacobian.cpp:164-194): the neighbour's
// Rusanov Jacobian; with the viscous terms (vp != null) its thin-shear-layer
// Jacobian from the neighbour's state, viscosity `mu` and cell velocity
// gradient `vg`, at the face's projected centre distance, subtracted for a
// lower (positive) and added for an upper neighbour
template <typename T>
__device__ __forceinline__ void BlockOffDiag(const GasT<T> &g, const T W[5], const T du[5], double4 a,
                                             bool positive, T out[5], const ViscParams *vp = nullptr,
                                             double mu = 0.0, double kLam = 0.0, double dist = 1.0,
                                             const double *vg = nullptr) {
  T J[25];
  RusanovJacobian<T>(g, W, T(a.x), T(a.y), T(a.z), T(a.w), positive, J);
  if (vp && vp->on) {
    const GasT<double> gd = {double(g.R), double(g.gamma), double(g.cps), double(g.cvs)};
    double Wd[5], V[25];
#pragma unroll
    for (int e = 0; e < 5; ++e) Wd[e] = double(W[e]);
    TSLJacobian(gd, *vp, Wd, mu, kLam, a, dist, positive, vg, V);
#pragma unroll
    for (int q = 0; q < 25; ++q) J[q] = positive ? J[q] - T(V[q]) : J[q] + T(V[q]);
  }
  BlockMult<T>(J, du, out);
}

// The off-diagonal block of cell (i, j, k) for its neighbour across
// direction d (upper: the neighbour at +1, else at -1), the matrix that
// RusanovBlockOffDiagonal (src/fluxJacobian.cpp:164-194) forms: the
// neighbour's Rusanov Jacobian at the shared face, with the neighbour's
// thin-shear-layer Jacobian (its cell velocity gradient, viscosity and
// conductivity, the face's projected centre distance) subtracted for a lower
// and added for an upper neighbour.  Formed where it is used, from the same
// inputs in the same order, so every user sees the same bits.
__device__ __forceinline__ void NeighbourBlock(const DevBlock &b, const GasT<double> &g, const ViscParams &vp,
                                               int d, bool upper, int i, int j, int k, double J[25]) {
#pragma clang fp contract(off)
  const int s = upper ? 1 : -1;
  const int ni = i + (d == 0 ? s : 0), nj = j + (d == 1 ? s : 0), nk = k + (d == 2 ? s : 0);
  const long f = upper ? FaceIdx(b, d, ni, nj, nk) : FaceIdx(b, d, i, j, k);
  const double4 a = b.fa[d][f];
  const long c = PadIdx(b, ni, nj, nk);
  double W[5];
#pragma unroll
  for (int e = 0; e < 5; ++e) W[e] = b.W[e * b.npad + c];
  const bool positive = !upper;
  RusanovJacobian<double>(g, W, a.x, a.y, a.z, a.w, positive, J);
  if (vp.on) {
    double vg[9], V[25];
#pragma unroll
    for (int q = 0; q < 9; ++q) vg[q] = b.vgrad[q * b.npad + c];
    TSLJacobian(g, vp, W, b.mu[c], b.kc[c], a, b.c2c[d][f], positive, vg, V);
#pragma unroll
    for (int q = 0; q < 25; ++q) J[q] = positive ? J[q] - V[q] : J[q] + V[q];
  }
}

// BlockMult with the matrix read entry by entry from global memory (entry q
// at M[q * stride + idx]), in the same order of operations
template <typename T, typename MT>
__device__ __forceinline__ void BlockMultG(const MT *__restrict__ M, long stride, long idx, const T v[5],
                                           T out[5]) {
  // all 25 loads issued before the arithmetic
  T m[25];
#pragma unroll
  for (int q = 0; q < 25; ++q) m[q] = T(M[q * stride + idx]);
  BlockMult<T>(m, v, out);
}

// block product with the cell's main diagonal Ab (cell-major layout)
template <typename T>
__device__ __forceinline__ void CellBlockMult(const DevBlock &b, const double *M, long p, const T v[5], T out[5]) {
  BlockMultG<T, double>(M, b.ncell, p, v, out);
}
// block product with the cell's inverse diagonal (Abi)
template <typename T, typename MT>
__device__ __forceinline__ void InverseMult(const DevBlock &b, const MT *M, int i, int j, int k, const T v[5],
                                            T out[5]) {
  int stride;
  const long base = InverseBase<MT>(b, i, j, k, stride);
  BlockMultG<T>(M, stride, base, v, out);
}

template <typename T>
struct OpBuf;
template <>
struct OpBuf<double> {
  static __device__ __forceinline__ double *Bt(const DevBlock &b) { return b.bt; }
  static __device__ __forceinline__ double *X(const DevBlock &b) { return b.x; }
  static __device__ __forceinline__ double *Xold(const DevBlock &b) { return b.xold; }
  static __device__ __forceinline__ const double *Ainv(const DevBlock &b) { return b.Ainv; }
  static __device__ __forceinline__ const double *Abi(const DevBlock &b) { return b.Abi; }
};
template <>
struct OpBuf<float> {
  static __device__ __forceinline__ float *Bt(const DevBlock &b) { return b.bt32; }
  static __device__ __forceinline__ float *X(const DevBlock &b) { return b.x32; }
  static __device__ __forceinline__ float *Xold(const DevBlock &b) { return b.xold32; }
  static __device__ __forceinline__ const float *Ainv(const DevBlock &b) { return b.Ainv32; }
  static __device__ __forceinline__ const float *Abi(const DevBlock &b) { return b.Abi32; }
};

// sum over the lower (upper == false) or upper neighbours of the Rusanov
// off-diagonal products: procBlock::ImplicitLower / ImplicitUpper
// (src/procBlock.cpp:1056-1161), neighbours in i, j, k order.  A ghost
// neighbour counts only across a connection (src/procBlock.cpp:1064, 1078,
// 1092); its product is the precomputed boundary term, zero elsewhere, and
// adding +0 leaves the sum unchanged (it starts at +0 and never becomes -0).
template <typename T>
__device__ __forceinline__ void OffDiagSum(const DevBlock &b, const GasT<T> &g, const ViscParams &vp,
                                           const T *x, int i, int j, int k, bool upper, T out[5],
                                           int block = 0, int roe = 0, const Gas *gas64 = nullptr) {
  // the block and Roe products are formed in FP64, with the FP64 gas
  const GasT<double> gd = gas64 ? Cast<double>(*gas64)
                                : GasT<double>{double(g.R), double(g.gamma), double(g.cps), double(g.cvs)};
#pragma unroll
  for (int e = 0; e < 5; ++e) out[e] = T(0);
  const T *bt = OpBuf<T>::Bt(b);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int s = upper ? 1 : -1;
    const int ni = i + (d == 0 ? s : 0), nj = j + (d == 1 ? s : 0), nk = k + (d == 2 ? s : 0);
    if (ni < 0 || nj < 0 || nk < 0 || ni >= b.ni || nj >= b.nj || nk >= b.nk) {
      if (bt) {
        const long q = BtSlot(b, d, upper ? 1 : 0, i, j, k);
#pragma unroll
        for (int e = 0; e < 5; ++e) out[e] += bt[e * b.nbf + q];
      }
      continue;
    }
    const long fq = upper ? FaceIdx(b, d, ni, nj, nk) : FaceIdx(b, d, i, j, k);
    const double4 a = b.fa[d][fq];
    const long c = PadIdx(b, ni, nj, nk);
    const long q = (long)ni + (long)nj * b.ni + (long)nk * b.ni * b.nj;
    T W[5], du[5], o[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      W[e] = T(b.W[e * b.npad + c]);
      du[e] = x[e * b.ncell + q];
    }
    if (block) {
      double J[25];
      NeighbourBlock(b, gd, vp, d, upper, i, j, k, J);
      T m[25];
#pragma unroll
      for (int q = 0; q < 25; ++q) m[q] = T(J[q]);
      BlockMult<T>(m, du, o);
    } else if (roe) {
      // RoeOffDiagonal: the cell's own state is the other side of the face
      const long cc = PadIdx(b, i, j, k);
      double Wd[5], Wn[5], dd[5], od[5];
#pragma unroll
      for (int e = 0; e < 5; ++e) {
        Wd[e] = b.W[e * b.npad + cc];
        Wn[e] = double(W[e]);
        dd[e] = double(du[e]);
      }
      RoeOffDiag(gd, Wn, Wd, dd, a, !upper, od);
#pragma unroll
      for (int e = 0; e < 5; ++e) o[e] = T(od[e]);
    } else {
      const T lv = vp.on ? ViscFaceSR<T>(g, W, T(a.w), T(b.c2c[d][fq]), T(b.mu[c]), vp) : T(0);
      ScalarOffDiag<T>(g, W, du, T(a.x), T(a.y), T(a.z), T(a.w), !upper, o, vp.on != 0, lv);
    }
#pragma unroll
    for (int e = 0; e < 5; ++e) out[e] += o[e];
  }
}

// InitializeMatrixUpdate (src/linearSolver.cpp:111-144)
template <typename T>
__global__ void __launch_bounds__(256) KInitUpdate(BlockMap M, Params P) {
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const long p = (long)U.local * blockDim.x + threadIdx.x;
  if (p >= b.ncell) return;
  T *x = OpBuf<T>::X(b);
  if (!P.initMatrix && !P.rhsOnce) {
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = T(0);
    return;
  }
  const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
  double rb[5];
  Rhs(b, P, p, PadIdx(b, i, j, k), rb);
  if (P.rhsOnce) {
    // the block pencil sweep's right-hand side, fixed for the relax (FP64; the
    // operator rounds it to its precision), and the state it runs from
    int lane;
    const long rec = PencilRecord(b, i, j, k, lane), c = PadIdx(b, i, j, k);
    double *o = b.skS + rec * BlockRecord(P.visc.on) * kPenLanes + lane;
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      o[e * kPenLanes] = b.W[e * b.npad + c];
      o[(5 + e) * kPenLanes] = rb[e];
    }
  }
  if (!P.initMatrix) {
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = T(0);
    return;
  }
  if (P.block) {
    T v[5], o[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) v[e] = T(rb[e]);
    InverseMult<T>(b, OpBuf<T>::Abi(b), i, j, k, v, o);
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = o[e];
    return;
  }
  const T ainv = OpBuf<T>::Ainv(b)[p];
#pragma unroll
  for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = T(rb[e]) * ainv;
}

// lusgs::LUSGS_Forward over one hyperplane (src/linearSolver.cpp:341-383)
template <typename T>
__global__ void __launch_bounds__(64) KLusgsForward(DevBlock b, Params P,
                                                    const int *__restrict__ cells, int n,
                                                    int useUpper) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const long p = cells[t];
  const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
  const GasT<T> g = Cast<T>(P.gas);
  T *x = OpBuf<T>::X(b);
  T L[5];
  OffDiagSum<T>(b, g, P.visc, x, i, j, k, false, L, P.block, P.roeJac, &P.gas);
  if (useUpper) {
    T U[5];
    OffDiagSum<T>(b, g, P.visc, x, i, j, k, true, U, P.block, P.roeJac, &P.gas);
#pragma unroll
    for (int e = 0; e < 5; ++e) L[e] -= U[e];
  }
  double rb[5];
  Rhs(b, P, p, PadIdx(b, i, j, k), rb);
  if (P.block) {
    T v[5], o[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) v[e] = T(rb[e]) + L[e];
    InverseMult<T>(b, OpBuf<T>::Abi(b), i, j, k, v, o);
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = o[e];
    return;
  }
  const T ainv = OpBuf<T>::Ainv(b)[p];
#pragma unroll
  for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = (T(rb[e]) + L[e]) * ainv;
}

// lusgs::LUSGS_Backward over one hyperplane (src/linearSolver.cpp:385-428)
template <typename T>
__global__ void __launch_bounds__(64) KLusgsBackward(DevBlock b, Params P,
                                                     const int *__restrict__ cells, int n,
                                                     int full) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const long p = cells[t];
  const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
  const GasT<T> g = Cast<T>(P.gas);
  T *x = OpBuf<T>::X(b);
  T U[5];
  OffDiagSum<T>(b, g, P.visc, x, i, j, k, true, U, P.block, P.roeJac, &P.gas);
  if (P.block) {
    T v[5], o[5];
    if (full) {
      T L[5];
      OffDiagSum<T>(b, g, P.visc, x, i, j, k, false, L, P.block, P.roeJac, &P.gas);
      double rb[5];
      Rhs(b, P, p, PadIdx(b, i, j, k), rb);
#pragma unroll
      for (int e = 0; e < 5; ++e) v[e] = (T(rb[e]) + L[e]) - U[e];
      InverseMult<T>(b, OpBuf<T>::Abi(b), i, j, k, v, o);
#pragma unroll
      for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = o[e];
    } else {
      InverseMult<T>(b, OpBuf<T>::Abi(b), i, j, k, U, o);
#pragma unroll
      for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = x[e * b.ncell + p] - o[e];
    }
    return;
  }
  const T ainv = OpBuf<T>::Ainv(b)[p];
  if (full) {
    T L[5];
    OffDiagSum<T>(b, g, P.visc, x, i, j, k, false, L, 0, P.roeJac);
    double rb[5];
    Rhs(b, P, p, PadIdx(b, i, j, k), rb);
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = ((T(rb[e]) + L[e]) - U[e]) * ainv;
  } else {
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = x[e * b.ncell + p] - U[e] * ainv;
  }
}

// dplur::DPLUR Jacobi sweep (src/linearSolver.cpp:473-507): reads the copy
// xold, writes x
template <typename T>
__global__ void __launch_bounds__(256) KDplur(DevBlock b, Params P) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= b.ncell) return;
  const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
  const GasT<T> g = Cast<T>(P.gas);
  const T *xo = OpBuf<T>::Xold(b);
  T L[5], U[5];
  OffDiagSum<T>(b, g, P.visc, xo, i, j, k, false, L, P.block, P.roeJac, &P.gas);
  OffDiagSum<T>(b, g, P.visc, xo, i, j, k, true, U, P.block, P.roeJac, &P.gas);
  double rb[5];
  Rhs(b, P, p, PadIdx(b, i, j, k), rb);
  T *x = OpBuf<T>::X(b);
  if (P.block) {
    T v[5], o[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) v[e] = (T(rb[e]) + T(0)) + (L[e] - U[e]);
    InverseMult<T>(b, OpBuf<T>::Abi(b), i, j, k, v, o);
#pragma unroll
    for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = o[e];
    return;
  }
  const T ainv = OpBuf<T>::Ainv(b)[p];
#pragma unroll
  for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = ((T(rb[e]) + T(0)) + (L[e] - U[e])) * ainv;
}

template <typename T>
__global__ void __launch_bounds__(256) KCopyUpdate(DevBlock b) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= 5 * b.ncell) return;
  OpBuf<T>::Xold(b)[p] = OpBuf<T>::X(b)[p];
}

// ---------------------------------------------------------------------------
// deterministic reductions: each workgroup reduces its 256 values in a fixed
// tree and writes one partial; a single-workgroup kernel sums the partials in
// index order.

constexpr int kRedThreads = 256;
constexpr int kNormSlots = 7;  // 5 x sum R^2, linf value, matrix-residual sum

struct Partial {
  double l2[5];
  double linf;
  long long linfIdx;  // ((cellBase + p) * 5 + e), -1 if none
  double mres;
};

__device__ __forceinline__ bool LinfBetter(double v, long long idx, double bv, long long bidx) {
  if (idx < 0) return false;
  if (bidx < 0) return true;
  return v > bv || (v == bv && idx < bidx);
}

// linearSolver::Residual / AXmB (src/linearSolver.cpp:58-109), squared and
// summed as in mgSolution::CycleAtLevel (src/mgSolution.cpp:197-206)
template <typename T>
__global__ void __launch_bounds__(kRedThreads) KMatrixResidual(BlockMap M, Params P,
                                                               Partial *part) {
  __shared__ double s[kRedThreads];
  // the partial of unit n covers the same cells whichever XCD runs it
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const unsigned n = U.global;
  const long p = (long)U.local * blockDim.x + threadIdx.x;
  double acc = 0.0;
  if (p < b.ncell) {
    const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
    const GasT<T> g = Cast<T>(P.gas);
    const T *x = OpBuf<T>::X(b);
    T L[5], U[5];
    OffDiagSum<T>(b, g, P.visc, x, i, j, k, false, L, P.block, P.roeJac, &P.gas);
    OffDiagSum<T>(b, g, P.visc, x, i, j, k, true, U, P.block, P.roeJac, &P.gas);
    double rb[5];
    Rhs(b, P, p, PadIdx(b, i, j, k), rb);
    const double A = P.block ? 0.0 : b.A[p];
    double axb[5] = {0, 0, 0, 0, 0};
    if (P.block) {
      double xv[5];
#pragma unroll
      for (int e = 0; e < 5; ++e) xv[e] = (double)x[e * b.ncell + p];
      CellBlockMult<double>(b, b.Ab, p, xv, axb);
    }
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const double ax = P.block ? axb[e] : (double)x[e * b.ncell + p] * A;
      const double axmb = (ax - (double)(L[e] - U[e])) - rb[e];
      const double r = 0.0 - axmb;
      acc += r * r;
    }
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kRedThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[n].mres = s[0];
}

// Norms of a workgroup in the tree of halving strides (thread t takes t + w,
// w = 128, ..., 1): the first two levels through LDS, the others within the first
// wave, whose lane 0 has the result.  With eight levels and barriers KUpdate took
// 26.0 us on 96^3 cells, 6.1 on 40^3; so 23.7 and 5.5.
__device__ __forceinline__ void TreeNorms(double l2[5], double &m, double &bv, long long &bi) {
  __shared__ double s[8][kRedThreads];
  const int t = threadIdx.x;
  auto put = [&] {
#pragma unroll
    for (int e = 0; e < 5; ++e) s[e][t] = l2[e];
    s[5][t] = m;
    s[6][t] = bv;
    s[7][t] = __longlong_as_double(bi);
  };
  auto take = [&](const double o[8]) {
#pragma unroll
    for (int e = 0; e < 5; ++e) l2[e] += o[e];
    m += o[5];
    if (LinfBetter(o[6], __double_as_longlong(o[7]), bv, bi)) {
      bv = o[6];
      bi = __double_as_longlong(o[7]);
    }
  };
  static_assert(kRedThreads == 256, "two levels through LDS");
  double o[8];
  if (t >= 128) put();
  __syncthreads();
  if (t < 128) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = s[e][t + 128];
    take(o);
    if (t >= 64) put();
  }
  __syncthreads();
  if (t >= 64) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = s[e][t + 64];
  take(o);
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) {
    const double own[8] = {l2[0], l2[1], l2[2], l2[3], l2[4], m, bv, __longlong_as_double(bi)};
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = __shfl_down(own[e], w);
    take(o);
  }
}

// procBlock::UpdateBlock (src/procBlock.cpp:826-871) with
// ImplicitTimeAdvance (:902-916) or ExplicitEulerTimeAdvance (:880-896)
template <typename T>
__global__ void __launch_bounds__(kRedThreads) KUpdate(BlockMap M, Params P, Partial *part) {
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const long p = (long)U.local * blockDim.x + threadIdx.x;
  double l2[5] = {0, 0, 0, 0, 0};
  double bv = 0.0;
  long long bi = -1;
  if (p < b.ncell) {
    const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
    const long c = PadIdx(b, i, j, k);
    const GasT<double> g = Cast<double>(P.gas);
    double W[5], Wn[5], R[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      W[e] = b.W[e * b.npad + c];
      R[e] = b.R[e * b.ncell + p];
    }
    if (P.explicitEuler) {
      double U[5];
      PrimToCons(g, W, U);
      const double f = Div(b.dt[p], b.vol[p]);
#pragma unroll
      for (int e = 0; e < 5; ++e) U[e] -= f * R[e];
      ConsToPrim(g, U, Wn);
    } else {
      const T *x = OpBuf<T>::X(b);
      double du[5];
#pragma unroll
      for (int e = 0; e < 5; ++e) du[e] = (double)x[e * b.ncell + p];
      UpdatePrim(g, W, du, Wn);
    }
#pragma unroll
    for (int e = 0; e < 5; ++e) b.W[e * b.npad + c] = Wn[e];
    if (!(Wn[0] > 0.0) || !(Wn[4] > 0.0)) atomicOr(b.flag, 1);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      l2[e] = R[e] * R[e];
      if (R[e] > bv) {  // strict '>' from 0: first maximum wins
        bv = R[e];
        bi = (long long)(b.cellBase + p) * 5 + e;
      }
    }
  }
  double m = 0.0;
  TreeNorms(l2, m, bv, bi);
  if (threadIdx.x == 0) {
    Partial &o = part[U.global];
#pragma unroll
    for (int e = 0; e < 5; ++e) o.l2[e] = l2[e];
    o.linf = bv;
    o.linfIdx = bi;
  }
}

// the norms of one case: its partials are [first, first + n) (its blocks'
// 256-cell units, in block order), written to its history ring
struct NormCase {
  int first, n;
  double *hist;
  int *counter;
};

// one workgroup per case: sums the case's partials in index order (a tree
// that depends only on the case's own partial count, so a case's norms do
// not depend on which other cases share the launch); writes the next slot
// of the case's ring = {l2[5], linf, linfIdx (as bits), mres}
__global__ void __launch_bounds__(kRedThreads) KReduceNorms(const Partial *__restrict__ allPart,
                                                           const NormCase *__restrict__ cases,
                                                           int withMres) {
  const NormCase nc = cases[blockIdx.x];
  const Partial *part = allPart + nc.first;
  const int n = nc.n;
  double *hist = nc.hist;
  int *counter = nc.counter;
  double l2[5] = {0, 0, 0, 0, 0}, m = 0.0, bv = 0.0;
  long long bi = -1;
  for (int q = threadIdx.x; q < n; q += kRedThreads) {
#pragma unroll
    for (int e = 0; e < 5; ++e) l2[e] += part[q].l2[e];
    if (withMres) m += part[q].mres;
    if (LinfBetter(part[q].linf, part[q].linfIdx, bv, bi)) {
      bv = part[q].linf;
      bi = part[q].linfIdx;
    }
  }
  TreeNorms(l2, m, bv, bi);
  if (threadIdx.x == 0) {
    const int slot = *counter;
    double *o = hist + (long)slot * 8;
#pragma unroll
    for (int e = 0; e < 5; ++e) o[e] = l2[e];
    o[5] = bv;
    o[6] = __longlong_as_double(bi);
    o[7] = m;
    *counter = slot + 1;
  }
}

__global__ void KSetScalar(double *dst, double v) { *dst = v; }
__global__ void KSetInt(int *dst, int v) { *dst = v; }

// input::CalcCFL (src/input.cpp:647-649) of every case of a group at its own
// outer step, which then advances by one
struct CflCase {
  double start, step, max;
  double *cfl;
  int *nn;
};
// restart every case's norm ring at slot 0
__global__ void KZeroCounters(const NormCase *__restrict__ cs, int n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) *cs[q].counter = 0;
}

__device__ __forceinline__ void CaseCfl(const CflCase &c) {
  const int nn = *c.nn;
  const double v = c.start + nn * c.step;
  *c.cfl = (c.max < v) ? c.max : v;
  *c.nn = nn + 1;
}
__global__ void KCaseCfl(const CflCase *__restrict__ cs, int n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) CaseCfl(cs[q]);
}

// StoreOldSolution (src/procBlock.cpp:1037-1053).  The first workgroup also
// sets the step's CFL number, one case's (`cfl`) or a group's (`cs`): a launch of
// its own is 4.4 us of an iteration of 285 us (40^3 cells).
__global__ void __launch_bounds__(256) KBeginStep(BlockMap M, Params P, int copyNm1, double *cfl, double cflValue,
                                                  const CflCase *__restrict__ cs, int ncs) {
#pragma clang fp contract(off)
  if (blockIdx.x == 0) {
    if (cfl && threadIdx.x == 0) *cfl = cflValue;
    for (int q = threadIdx.x; q < ncs; q += blockDim.x) CaseCfl(cs[q]);
  }
  const Unit Un = MapUnit(M);
  const DevBlock &b = *Un.b;
  const long p = (long)Un.local * blockDim.x + threadIdx.x;
  if (p >= b.ncell) return;
  const int i = (int)(p % b.ni), j = (int)((p / b.ni) % b.nj), k = (int)(p / ((long)b.ni * b.nj));
  const long c = PadIdx(b, i, j, k);
  const GasT<double> g = Cast<double>(P.gas);
  const double W[5] = {b.W[c], b.W[b.npad + c], b.W[2 * b.npad + c], b.W[3 * b.npad + c],
                       b.W[4 * b.npad + c]};
  double U[5];
  PrimToCons(g, W, U);
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    b.consN[e * b.ncell + p] = U[e];
    if (copyNm1) b.consNm1[e * b.ncell + p] = U[e];
  }
}

// AssignSolToTimeNm1 after the last nonlinear iteration (src/gridLevel.cpp:424-428)
__global__ void __launch_bounds__(256) KCopyNm1(DevBlock b) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= 5 * b.ncell) return;
  b.consNm1[p] = b.consN[p];
}

// The state of a block's physical cells between the padded SoA layout and the
// callers' AoS one (five values a cell, i fastest), through the block's
// scratch `xold`: one thread a cell.  A host loop over five strided arrays
// took 12 ns a cell each way; these take 0.04 ns and leave the copy of 40 B a
// cell over the host link.
__global__ void __launch_bounds__(256) KPackState(const DevBlock b, int unpack) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= b.ncell) return;
  const long c = PadIdx(b, (int)(p % b.ni), (int)((p / b.ni) % b.nj), (int)(p / ((long)b.ni * b.nj)));
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    if (unpack) b.W[e * b.npad + c] = b.xold[5 * p + e];
    else b.xold[5 * p + e] = b.W[e * b.npad + c];
  }
}

// batch face-flux evaluation used by the parity tests
__global__ void __launch_bounds__(256) KEvalFlux(int flux, Gas gas, const double *WL,
                                                 const double *WR, const double *n, int count,
                                                 double *F) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const GasT<double> g = Cast<double>(gas);
  double L[5], R[5], out[5];
  for (int e = 0; e < 5; ++e) {
    L[e] = WL[5 * t + e];
    R[e] = WR[5 * t + e];
  }
  if (flux == 0) RoeFlux(g, L, R, n[3 * t], n[3 * t + 1], n[3 * t + 2], out);
  else AusmFlux(g, L, R, n[3 * t], n[3 * t + 1], n[3 * t + 2], out);
  for (int e = 0; e < 5; ++e) F[5 * t + e] = out[e];
}

}  // namespace ath

namespace ath {

// ---------------------------------------------------------------------------
// Publishing a sweep's du to other workgroups.
//
// A workgroup publishes a tile's du by storing it and then a flag that other
// workgroups poll; they read the du after an agent-scope acquire.  An
// agent-scope release on this target writes back the XCD's L2 and then waits
// for the wave's stores: the write-back is there for stores that are not
// coherent at agent scope, and it cost about 100 us of each 760 us pass of a
// tile sweep.  The sweeps therefore store with agent-scope atomic stores
// (written through to the agent's point of coherence), the tiled one waits for
// each wave's own stores to complete and only then stores the flag; no
// write-back is needed for stores that are already coherent.  (The pencil
// sweeps' messages carry their own validity.)
template <typename T>
__device__ __forceinline__ void StoreCoherent(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// wait until every store the wave issued has completed
__device__ __forceinline__ void WaitStores() { __builtin_amdgcn_s_waitcnt(0); }

// ---------------------------------------------------------------------------
// tiled, dataflow-synchronised LU-SGS sweep (lusgs::LUSGS_Forward/Backward,
// src/linearSolver.cpp:341-428).
//
// The hyperplane order of HyperplaneReorder (src/utility.cpp:377-398) is one
// topological order of the Gauss-Seidel dependencies (a cell needs its lower
// neighbours in the forward sweep, its upper neighbours in the backward
// sweep); any other topological order gives the same result bit for bit.
// This kernel uses a blocked one: the block is cut into kLT = 8x8x4 tiles,
// tiles are taken in tile-hyperplane order from an atomic ticket by
// persistent workgroups, and a tile starts once the (at most three) tiles it
// depends on have published their du.  Inside a tile the workgroup walks the
// 18 intra-tile hyperplanes with LDS-resident state, du, right-hand side and
// face vectors.  Cross-tile visibility: du is stored agent-coherent and the
// per-tile flag, carrying the sweep's epoch, is stored once those stores have
// completed (StoreCoherent / WaitStores); readers acquire at agent scope.
// Every wait is bounded and reports through `err` instead of hanging.
constexpr int kLTI = 8, kLTJ = 8, kLTK = 4;
constexpr int kLT = kLTI * kLTJ * kLTK;  // 256 cells, one per thread
constexpr int kLTPlanes = kLTI + kLTJ + kLTK - 2;
constexpr int kHaloI = kLTJ * kLTK, kHaloJ = kLTI * kLTK, kHaloK = kLTI * kLTJ;
constexpr int kHalo = kHaloI + kHaloJ + kHaloK;
constexpr long kSpinLimit = 1L << 20;

struct SweepCtl {
  int *ticket;      // reset to 0 before each sweep
  int *epoch;       // incremented before each sweep
  int *flags;       // one per tile, holds the epoch of its last publication
  int *err;         // bit 1: a dependency wait exceeded the spin limit
  const int4 *tiles;  // (a, b, c, -) in tile-hyperplane order
  int ntiles, ta, tb, tc;  // tile count and tile grid dims
};

__global__ void KSweepPrologue(SweepCtl s) {
  *s.ticket = 0;
  *s.epoch = *s.epoch + 1;
}

__device__ __forceinline__ int TileId(const SweepCtl &s, int a, int b, int c) {
  return a + s.ta * (b + s.tb * c);
}

// off-diagonal product of one neighbour: state/du from LDS or global
template <typename T>
__device__ __forceinline__ void NbOffDiag(const GasT<T> &g, const double *Wnb, const T *du,
                                          double4 a, bool positive, T out[5],
                                          const ViscParams *vp = nullptr, double dist = 1.0,
                                          double mu = 0.0) {
  T W[5], d[5];
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    W[e] = T(Wnb[e]);
    d[e] = du[e];
  }
  const bool visc = vp && vp->on;
  const T lv = visc ? ViscFaceSR<T>(g, W, T(a.w), T(dist), T(mu), *vp) : T(0);
  ScalarOffDiag<T>(g, W, d, T(a.x), T(a.y), T(a.z), T(a.w), positive, out, visc, lv);
}

// ---------------------------------------------------------------------------
// interblock connections

// ghost cell <- partner interior cell, all layers (SwapStateSlice,
// src/procBlock.cpp:3050-3055; sources are interior cells, so the swaps are
// independent of each other)
struct HaloTask {
  int dst, src;
  long dpad, spad;
};

__global__ void __launch_bounds__(256) KHaloState(const DevBlock *__restrict__ blocks,
                                                  const HaloTask *__restrict__ tasks, int n) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const HaloTask h = tasks[t];
  const DevBlock &A = blocks[h.dst], &B = blocks[h.src];
#pragma unroll
  for (int e = 0; e < 5; ++e) A.W[e * A.npad + h.dpad] = B.W[e * B.npad + h.spad];
}

// ghost cell velocity gradients <- partner interior cells
// (SwapEddyViscAndGradients, src/gridLevel.cpp:385-387), block solvers with
// the viscous terms
__global__ void __launch_bounds__(256) KHaloGrad(const DevBlock *__restrict__ blocks,
                                                 const HaloTask *__restrict__ tasks, int n) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const HaloTask h = tasks[t];
  const DevBlock &A = blocks[h.dst], &B = blocks[h.src];
#pragma unroll
  for (int q = 0; q < 9; ++q) A.vgrad[q * A.npad + h.dpad] = B.vgrad[q * B.npad + h.spad];
}

// the off-diagonal product of the ghost neighbour across one connection
// face, from the partner's current du (SwapImplicitUpdate before each pass,
// src/linearSolver.cpp:444-463, then OffDiagonal with the ghost state)
struct ConnTask {
  int blk, src, d, upper;
  long gpad, scell, face, slot;
};

template <typename T>
__global__ void __launch_bounds__(256) KConnTerms(const DevBlock *__restrict__ blocks,
                                                  const ConnTask *__restrict__ tasks, int n, Params P) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const ConnTask c = tasks[t];
  const DevBlock &A = blocks[c.blk], &B = blocks[c.src];
  const T *xb = OpBuf<T>::X(B);
  double Wn[5];
  T dn[5], o[5];
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    Wn[e] = A.W[e * A.npad + c.gpad];
    dn[e] = xb[e * B.ncell + c.scell];
  }
  if (P.block) {
    // the block is formed in FP64 from the FP64 state (with either operator
    // precision)
    double dd[5], od[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) dd[e] = double(dn[e]);
    if (P.visc.on) {
      double vgn[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) vgn[q] = A.vgrad[q * A.npad + c.gpad];
      BlockOffDiag<double>(Cast<double>(P.gas), Wn, dd, A.fa[c.d][c.face], c.upper == 0, od, &P.visc,
                           A.mu[c.gpad], A.kc[c.gpad], A.c2c[c.d][c.face], vgn);
    } else {
      BlockOffDiag<double>(Cast<double>(P.gas), Wn, dd, A.fa[c.d][c.face], c.upper == 0, od);
    }
#pragma unroll
    for (int e = 0; e < 5; ++e) o[e] = T(od[e]);
  } else if (P.roeJac) {
    // RoeOffDiagonal with the interior cell next to the ghost as the other
    // side (a lower ghost lies below it, an upper ghost above)
    const long s = c.d == 0 ? 1 : (c.d == 1 ? (long)A.NI : (long)A.NI * A.NJ);
    const long ci = c.upper ? c.gpad - s : c.gpad + s;
    double Wd[5], dd[5], od[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      Wd[e] = A.W[e * A.npad + ci];
      dd[e] = double(dn[e]);
    }
    RoeOffDiag(Cast<double>(P.gas), Wn, Wd, dd, A.fa[c.d][c.face], c.upper == 0, od);
#pragma unroll
    for (int e = 0; e < 5; ++e) o[e] = T(od[e]);
  } else if (P.visc.on)
    NbOffDiag<T>(Cast<T>(P.gas), Wn, dn, A.fa[c.d][c.face], c.upper == 0, o, &P.visc, A.c2c[c.d][c.face],
                 A.mu[c.gpad]);
  else
    NbOffDiag<T>(Cast<T>(P.gas), Wn, dn, A.fa[c.d][c.face], c.upper == 0, o);
  T *bt = OpBuf<T>::Bt(A);
#pragma unroll
  for (int e = 0; e < 5; ++e) bt[e * A.nbf + c.slot] = o[e];
}

template <typename T, bool FWD>
__global__ void __launch_bounds__(kLT) KLusgsTile(DevBlock b, Params P, SweepCtl s, int full) {
  __shared__ double sW[5][kLT];
  __shared__ T sX[5][kLT];
  __shared__ double sFa[3][4][kLT];  // face shared with the dependency neighbour
  __shared__ double sHW[5][kHalo];   // halo (outside-tile dependency) state
  __shared__ T sHX[5][kHalo];        // halo du
  __shared__ int sTicket;
  __shared__ int sEpoch;

  const int tid = threadIdx.x;
  const int li = tid % kLTI, lj = (tid / kLTI) % kLTJ, lk = tid / (kLTI * kLTJ);
  const GasT<T> g = Cast<T>(P.gas);
  T *x = OpBuf<T>::X(b);
  const T *ainvG = OpBuf<T>::Ainv(b);
  const int sgn = FWD ? -1 : 1;  // direction of the dependency neighbours

  // Thread 0 owns the ticket and the flag.  Exactly one `tid == 0` block
  // sits between two barriers at the end of each pass (publish the tile,
  // fetch the next ticket); with separate blocks on both sides of the loop's
  // back edge the compiler may merge them into a lane-0-only path around the
  // loop header, leaving the other lanes to pass the header barrier with a
  // stale ticket.
  if (tid == 0) {
    sTicket = __hip_atomic_fetch_add(s.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sEpoch = __hip_atomic_load(s.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const int epoch = sEpoch;
  for (;;) {
    const int t = sTicket;
    if (t >= s.ntiles) break;
    const int4 tl = s.tiles[FWD ? t : s.ntiles - 1 - t];
    const int i = tl.x * kLTI + li, j = tl.y * kLTJ + lj, k = tl.z * kLTK + lk;
    const bool valid = i < b.ni && j < b.nj && k < b.nk;
    const long p = (long)i + (long)j * b.ni + (long)k * b.ni * b.nj;

    // --- static data (independent of du) before the dependency wait; the
    // right-hand side and D^-1 of the thread's own cell stay in registers
    double rb[5] = {0, 0, 0, 0, 0};
    T ainv = T(0);
    if (valid) {
      const long c = PadIdx(b, i, j, k);
#pragma unroll
      for (int e = 0; e < 5; ++e) sW[e][tid] = b.W[e * b.npad + c];
      if (FWD || full) Rhs(b, P, p, c, rb);
      ainv = ainvG[p];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        // forward: the cell's lower face; backward: its upper face
        const int fi = i + (FWD ? 0 : (d == 0)), fj = j + (FWD ? 0 : (d == 1)),
                  fk = k + (FWD ? 0 : (d == 2));
        const int n3 = d == 0 ? b.ni : (d == 1 ? b.nj : b.nk);
        const int f3 = d == 0 ? fi : (d == 1 ? fj : fk);
        double4 a = make_double4(0, 0, 0, 0);
        if (f3 > 0 && f3 < n3) a = b.fa[d][FaceIdx(b, d, fi, fj, fk)];
        sFa[d][0][tid] = a.x;
        sFa[d][1][tid] = a.y;
        sFa[d][2][tid] = a.z;
        sFa[d][3][tid] = a.w;
      }
    }
    // halo state: dependency neighbours just outside the tile
    {
      const int di = FWD ? -1 : kLTI, dj = FWD ? -1 : kLTJ, dk = FWD ? -1 : kLTK;
      if (tid < kHalo) {
        int hi, hj, hk;
        if (tid < kHaloI) { hi = di; hj = tid % kLTJ; hk = tid / kLTJ; }
        else if (tid < kHaloI + kHaloJ) { const int q = tid - kHaloI; hi = q % kLTI; hj = dj; hk = q / kLTI; }
        else { const int q = tid - kHaloI - kHaloJ; hi = q % kLTI; hj = q / kLTI; hk = dk; }
        const int gi = tl.x * kLTI + hi, gj = tl.y * kLTJ + hj, gk = tl.z * kLTK + hk;
        if (gi >= 0 && gj >= 0 && gk >= 0 && gi < b.ni && gj < b.nj && gk < b.nk) {
          const long c = PadIdx(b, gi, gj, gk);
#pragma unroll
          for (int e = 0; e < 5; ++e) sHW[e][tid] = b.W[e * b.npad + c];
        }
      }
    }

    // --- wait for the tiles this one depends on
    if (tid == 0) {
      const int deps[3][3] = {{tl.x + sgn, tl.y, tl.z}, {tl.x, tl.y + sgn, tl.z}, {tl.x, tl.y, tl.z + sgn}};
      for (int q = 0; q < 3; ++q) {
        const int a = deps[q][0], bb = deps[q][1], cc = deps[q][2];
        if (a < 0 || bb < 0 || cc < 0 || a >= s.ta || bb >= s.tb || cc >= s.tc) continue;
        const int id = TileId(s, a, bb, cc);
        long spins = 0;
        while (__hip_atomic_load(&s.flags[id], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < epoch) {
          // once any wait of the launch has timed out, stop waiting at all
          if ((++spins & 255) == 0 &&
              (__hip_atomic_load(s.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 2))
            break;
          if (spins > kSpinLimit) {
            __hip_atomic_fetch_or(s.err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      // one acquire for the workgroup, ordered before every wave's halo
      // loads by the barrier
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();

    // halo du, published by the dependency tiles
    {
      const int di = FWD ? -1 : kLTI, dj = FWD ? -1 : kLTJ, dk = FWD ? -1 : kLTK;
      if (tid < kHalo) {
        int hi, hj, hk;
        if (tid < kHaloI) { hi = di; hj = tid % kLTJ; hk = tid / kLTJ; }
        else if (tid < kHaloI + kHaloJ) { const int q = tid - kHaloI; hi = q % kLTI; hj = dj; hk = q / kLTI; }
        else { const int q = tid - kHaloI - kHaloJ; hi = q % kLTI; hj = q / kLTI; hk = dk; }
        const int gi = tl.x * kLTI + hi, gj = tl.y * kLTJ + hj, gk = tl.z * kLTK + hk;
        if (gi >= 0 && gj >= 0 && gk >= 0 && gi < b.ni && gj < b.nj && gk < b.nk) {
          const long q = (long)gi + (long)gj * b.ni + (long)gk * b.ni * b.nj;
#pragma unroll
          for (int e = 0; e < 5; ++e) sHX[e][tid] = x[e * b.ncell + q];
        }
      }
    }
    if (!FWD && valid) {
#pragma unroll
      for (int e = 0; e < 5; ++e) sX[e][tid] = x[e * b.ncell + p];  // forward result
    }
    __syncthreads();

    // --- intra-tile hyperplanes
    const int plane = li + lj + lk;
    for (int st = 0; st < kLTPlanes; ++st) {
      const int pl = FWD ? st : kLTPlanes - 1 - st;
      if (valid && plane == pl) {
        T D[5];  // dependency-side sum: L (forward) or U (backward)
#pragma unroll
        for (int e = 0; e < 5; ++e) D[e] = T(0);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int gi = i + (d == 0 ? sgn : 0), gj = j + (d == 1 ? sgn : 0), gk = k + (d == 2 ? sgn : 0);
          if (gi < 0 || gj < 0 || gk < 0 || gi >= b.ni || gj >= b.nj || gk >= b.nk) {
            // ghost neighbour: the connection term (zero off connections)
            const T *bt = OpBuf<T>::Bt(b);
            if (bt) {
              const long q = BtSlot(b, d, FWD ? 0 : 1, i, j, k);
#pragma unroll
              for (int e = 0; e < 5; ++e) D[e] += bt[e * b.nbf + q];
            }
            continue;
          }
          const int l3 = d == 0 ? li : (d == 1 ? lj : lk);
          const int L3 = d == 0 ? kLTI : (d == 1 ? kLTJ : kLTK);
          const bool inTile = FWD ? (l3 > 0) : (l3 < L3 - 1);
          double Wn[5];
          T dn[5];
          if (inTile) {
            const int nt = tid + sgn * (d == 0 ? 1 : (d == 1 ? kLTI : kLTI * kLTJ));
#pragma unroll
            for (int e = 0; e < 5; ++e) {
              Wn[e] = sW[e][nt];
              dn[e] = sX[e][nt];
            }
          } else {
            const int h = d == 0 ? lj + kLTJ * lk : (d == 1 ? kHaloI + li + kLTI * lk : kHaloI + kHaloJ + li + kLTI * lj);
#pragma unroll
            for (int e = 0; e < 5; ++e) {
              Wn[e] = sHW[e][h];
              dn[e] = sHX[e][h];
            }
          }
          const double4 a = make_double4(sFa[d][0][tid], sFa[d][1][tid], sFa[d][2][tid], sFa[d][3][tid]);
          T o[5];
          if (P.visc.on) {
            const long fq = FWD ? FaceIdx(b, d, i, j, k) : FaceIdx(b, d, gi, gj, gk);
            NbOffDiag<T>(g, Wn, dn, a, FWD, o, &P.visc, b.c2c[d][fq], b.mu[PadIdx(b, gi, gj, gk)]);
          } else {
            NbOffDiag<T>(g, Wn, dn, a, FWD, o);
          }
#pragma unroll
          for (int e = 0; e < 5; ++e) D[e] += o[e];
        }
        T xn[5];
        if (full) {
          // the other side, from the previous sweep's values in global memory
          T O[5];
          OffDiagSum<T>(b, g, P.visc, x, i, j, k, FWD, O);
          if (FWD) {
#pragma unroll
            for (int e = 0; e < 5; ++e) xn[e] = (T(rb[e]) + (D[e] - O[e])) * ainv;
          } else {
#pragma unroll
            for (int e = 0; e < 5; ++e) xn[e] = ((T(rb[e]) + O[e]) - D[e]) * ainv;
          }
        } else if (FWD) {
#pragma unroll
          for (int e = 0; e < 5; ++e) xn[e] = (T(rb[e]) + D[e]) * ainv;
        } else {
#pragma unroll
          for (int e = 0; e < 5; ++e) xn[e] = sX[e][tid] - D[e] * ainv;
        }
#pragma unroll
        for (int e = 0; e < 5; ++e) {
          sX[e][tid] = xn[e];
          StoreCoherent(&x[e * b.ncell + p], xn[e]);
        }
      }
      __syncthreads();
    }

    // --- publish: every wave's du stores have completed before the barrier,
    // and thread 0 stores the flag after it; the same thread takes the next
    // ticket
    WaitStores();
    __syncthreads();
    if (tid == 0) {
      __hip_atomic_store(&s.flags[TileId(s, tl.x, tl.y, tl.z)], epoch, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      sTicket = __hip_atomic_fetch_add(s.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Pencil-wavefront LU-SGS sweep (scalar operator).
//
// The block is cut into kPW x kPW columns ("pencils") that run the whole
// extent of its longest axis C; A = C + 1 and B = C + 2 (mod 3) are the axes
// of the cut.  One workgroup owns a pencil; lane l of its compute wave stands
// for the column (la, lb) = (l % kPW, l / kPW).  At pencil step s the lanes
// update the cells of the local hyperplane la + lb + c = s (forward; mirrored
// in the backward pass, whose step s is the forward step ns - 1 - s), so a
// pencil of full width walks nc + 2 kPW - 2 steps.  The longest axis gives
// the fewest column handoffs and the fewest idle steps.
//
// What bounds it is the dependency chain of na + nb + nc - 2 hyperplanes, not
// memory or arithmetic, so the kernel is laid out to make one step of that
// chain short:
//
//  * A cell's products are formed by the cell itself.  The off-diagonal
//    product that a cell's neighbour adds (RusanovScalarOffDiagonal,
//    src/fluxJacobian.cpp:122-162) takes this cell's state and du and the
//    shared face only.  The lane that has just formed du therefore forms its
//    three outgoing products (three faces) with one U + du -> primitive
//    conversion and one enthalpy, where the neighbours together would do it
//    three times; it hands products, not du, to the next step.  One wave does
//    a whole step and needs no other wave's result of the same step.
//  * The inputs lie in the order the sweep takes them (DevBlock::skS, skF):
//    step by step, 64 lanes of one value contiguous, so that a stager's loads
//    are whole lines.  In the natural layout the 64 cells of a hyperplane lie
//    in different lines and each load fetches 64 of them.
//  * Products cross a pencil face as self-validating messages: the receiving
//    pencil polls the eight lanes' values themselves (every slot holds the
//    all-ones pattern until its value arrives), which saves the wait for the
//    stores' completion, the progress flag and the acquire.  The two
//    directions have slots of their own, and each pass empties the other's.
//
// Waves of a workgroup: the compute wave; a halo wave that polls the next
// step's messages into an LDS ring (or reads the connection terms on a block
// face); a send wave that stores the messages of the step just done; and
// kStagers waves that form, up to kPenSlots steps ahead, everything of the
// products that does not depend on du (U, F(W), the normal, half the face
// area, the spectral radius term) in LDS slots.  They synchronise through
// step counters in LDS, each with one writer.
//
// Pencils are taken from an atomic ticket in pencil-hyperplane order, so a
// pencil only ever waits on pencils whose workgroups are already running: no
// co-residency assumption.  The ticket counts on from launch to launch
// (every launch takes exactly nent of them).  Every wait is bounded.
//
// Measured per pass on a 64^3 block, against a sweep that handed du from an
// owner wave to three neighbour waves and published progress counts: FP64 785
// -> 185 us, FP32 790 -> 164 us.  A step takes 0.80 us (0.47 us of it
// the compute wave's arithmetic, the rest its LDS and store instructions,
// which hold the wave's issue for 13-29 cycles each), a handoff 1.6 us more
// than its step.  Three compute waves, one per outgoing product, took 0.82 us
// a step (the exchange between them costs what the arithmetic saves).
constexpr int kStagers = 4;
constexpr int kPenSlots = kStagers;
constexpr int kPenWaves = 3 + kStagers;
constexpr int kProdRing = 4;   // steps of products kept in LDS for the send wave (a power of two)
constexpr int kHaloRing = 8;   // steps of halo products in LDS
constexpr int kMsg = 5 * kPW;  // values of one message
constexpr int kPenF = 12;      // values of a cell's three faces on one side: unit normal, area (and centre distance)
constexpr int kLdsSpinLimit = 1 << 24;
static_assert(kHaloRing * kPW == kPenLanes, "halo ring layout");

// the pencils of every block in one launch: entry t = (a, b, block, first
// message step of the block), ordered by pencil hyperplane a + b, then block,
// then b, a.  A pencil depends only on pencils of its own block one
// hyperplane lower (forward; higher in the backward pass, which takes the
// entries in reverse), all of which hold earlier tickets.
struct PencilGroup {
  unsigned long long *ticket;
  int *err;             // bit 1: a dependency wait exceeded the spin limit
  const int4 *entries;
  int nent;             // pencils of all blocks
  void *msg[2];         // of the forward and backward passes: per pencil 2 faces x pns steps x kMsg
                        // operator words, all ones when empty
  const DevBlock *blocks;
};

__device__ __forceinline__ int AxisN(const DevBlock &b, int d) { return d == 0 ? b.ni : (d == 1 ? b.nj : b.nk); }
// pencil width (cells) along a cut axis of n cells
__device__ __forceinline__ int PenWidth(int n, int a) { return min(kPW, n - a * kPW); }

template <typename T>
__device__ __forceinline__ T CoherentLoad(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the empty message slot: all bits one, a NaN that no product is stored as
__device__ __forceinline__ bool IsEmpty(double v) { return __double_as_longlong(v) == -1LL; }
__device__ __forceinline__ bool IsEmpty(float v) { return __float_as_int(v) == -1; }
// (a product could hold that pattern only as a NaN handed down from an input)
template <typename T>
__device__ __forceinline__ T NotEmpty(T v) {
  return IsEmpty(v) ? T(__builtin_nan("")) : v;
}
template <typename T>
__device__ __forceinline__ T EmptySlot();
template <>
__device__ __forceinline__ double EmptySlot<double>() { return __longlong_as_double(-1LL); }
template <>
__device__ __forceinline__ float EmptySlot<float>() { return __int_as_float(-1); }

// the cell of a lane of a record of the sweep-ordered arrays
struct PenCell {
  bool active;
  int i, j, k;
};
__device__ __forceinline__ PenCell PencilCell(const DevBlock &b, long rec, int lane) {
  const int pid = (int)(rec / b.prec), s = ((int)(rec % b.prec) << (6 - b.pln)) + (lane >> b.pln);
  const int a = pid % b.pa, bb = pid / b.pa;
  const int na = AxisN(b, (b.pl + 1) % 3), nb = AxisN(b, (b.pl + 2) % 3), nc = AxisN(b, b.pl);
  const int l = lane & ((1 << b.pln) - 1), la = l & ((1 << b.pla) - 1), lb = l >> b.pla, c = s - la - lb;
  PenCell r;
  r.active = la < PenWidth(na, a) && lb < PenWidth(nb, bb) && c >= 0 && c < nc;
  Map3(b.pl, c, a * kPW + la, bb * kPW + lb, r.i, r.j, r.k);
  return r;
}
__device__ __forceinline__ long Records(const DevBlock &b) { return (long)b.pa * b.pb * b.prec; }

// The face data of every pencil record, laid out once per case: side 0 the
// lower faces (what the backward pass's products cross), side 1 the upper
// ones (forward), axes in the order A, B, C.  Records of idle lanes, which the
// sweep reads and whose results it drops, start from zeros.
__global__ void __launch_bounds__(256) KPencilFaces(const DevBlock b, int visc, int nS) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = (int)(t % kPenLanes);
  const long rec = t / kPenLanes, nrec = Records(b);
  if (rec >= nrec) return;
  const PenCell c = PencilCell(b, rec, lane);
  const int nF = kPenF + (visc ? 3 : 0);
  if (!c.active) {
    for (int q = 0; q < nF; ++q)
      b.skF[(rec * nF + q) * kPenLanes + lane] = b.skF[((nrec + rec) * nF + q) * kPenLanes + lane] = 0.0;
    for (int q = 0; q < nS; ++q) b.skS[(rec * nS + q) * kPenLanes + lane] = 0.0;
    for (int q = 0; q < 5; ++q) {
      b.skX[(rec * 5 + q) * kPenLanes + lane] = 0.0;
      if (b.skO) b.skO[(rec * 5 + q) * kPenLanes + lane] = 0.0;
    }
    return;
  }
  for (int side = 0; side < 2; ++side)
    for (int q = 0; q < 3; ++q) {
      const int d = (b.pl + 1 + q) % 3;
      const long f = FaceIdx(b, d, c.i + (side && d == 0), c.j + (side && d == 1), c.k + (side && d == 2));
      const double4 a = (d == 0 ? b.fa[0] : (d == 1 ? b.fa[1] : b.fa[2]))[f];
      double *o = b.skF + ((side * nrec + rec) * nF + 4 * q) * kPenLanes + lane;
      o[0] = a.x;
      o[kPenLanes] = a.y;
      o[2 * kPenLanes] = a.z;
      o[3 * kPenLanes] = a.w;
      if (visc)
        b.skF[((side * nrec + rec) * nF + kPenF + q) * kPenLanes + lane] =
            (d == 0 ? b.c2c[0] : (d == 1 ? b.c2c[1] : b.c2c[2]))[f];
    }
}

// The inputs of a relax in sweep order: the state, the right-hand side
// (which the sweeps do not change), D^-1 and, with the viscous terms, the
// viscosity of every cell
template <typename T>
__global__ void __launch_bounds__(256) KPencilPrep(BlockMap M, Params P) {
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const long t = (long)U.local * blockDim.x + threadIdx.x;
  const int lane = (int)(t % kPenLanes);
  const long rec = t / kPenLanes;
  if (rec >= Records(b)) return;
  const PenCell q = PencilCell(b, rec, lane);
  if (!q.active) return;
  const long p = (long)q.i + (long)q.j * b.ni + (long)q.k * b.ni * b.nj, c = PadIdx(b, q.i, q.j, q.k);
  const int nS = kPenS + (P.visc.on ? 1 : 0);
  double *o = b.skS + rec * nS * kPenLanes + lane;
  double rb[5];
  Rhs(b, P, p, c, rb);
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    o[e * kPenLanes] = b.W[e * b.npad + c];
    o[(5 + e) * kPenLanes] = rb[e];
  }
  o[10 * kPenLanes] = double(OpBuf<T>::Ainv(b)[p]);
  if (P.visc.on) o[kPenS * kPenLanes] = b.mu[c];
}

// A full sweep's other-side sums (OffDiagSum over the upper neighbours in a
// forward pass, the lower ones in a backward pass), formed before the pass:
// none of the du they read is written by the pass before the cell itself is
// updated, so the values are those the sweep would form in place.
template <typename T, bool FWD>
__global__ void __launch_bounds__(256) KPencilOther(BlockMap M, Params P) {
  const Unit U = MapUnit(M);
  const DevBlock &b = *U.b;
  const long t = (long)U.local * blockDim.x + threadIdx.x;
  const int lane = (int)(t % kPenLanes);
  const long rec = t / kPenLanes;
  if (rec >= Records(b)) return;
  const PenCell q = PencilCell(b, rec, lane);
  if (!q.active) return;
  T O[5];
  OffDiagSum<T>(b, Cast<T>(P.gas), P.visc, OpBuf<T>::X(b), q.i, q.j, q.k, FWD, O, P.block, 0, &P.gas);
  T *o = (T *)b.skO + rec * 5 * kPenLanes + lane;
#pragma unroll
  for (int e = 0; e < 5; ++e) o[e * kPenLanes] = O[e];
}

// everything of one step that does not depend on this sweep's du.  Early:
// right-hand side or the cell's forward du (5), D^-1, state
// (5: conservative, or primitive for the FP32 operator's flux change), the
// other-side sum of a full sweep (5).  Late, for the face of each axis A, B,
// C: unit normal (3), 0.5 |A|, the spectral radius term, then FP64: F(W)
// through the face (5), FP32: v.n there and rho E + p.
template <typename T, bool FULL>
constexpr int kEarly = FULL ? 16 : 11;
template <typename T>
constexpr int kLate = sizeof(T) == 8 ? 10 : 7;
template <typename T, bool FULL>
struct PenSlot {
  LdsVec<T> early[Vecs<T>(kEarly<T, FULL>)][kPenLanes];
  LdsVec<T> late[3][Vecs<T>(kLate<T>)][kPenLanes];
};
// n values of a lane from / to its vectors
template <typename T, int N, int STRIDE = kPenLanes>
__device__ __forceinline__ void LdsGet(const LdsVec<T> *p, T *v) {
#pragma unroll
  for (int q = 0; q < Vecs<T>(N); ++q) {
    const LdsVec<T> w = p[q * STRIDE];
#pragma unroll
    for (int r = 0; r < kVecN<T>; ++r)
      if (q * kVecN<T> + r < N) v[q * kVecN<T> + r] = w.v[r];
  }
}
template <typename T, int N>
__device__ __forceinline__ void LdsPut(LdsVec<T> *p, const T *v) {
#pragma unroll
  for (int q = 0; q < Vecs<T>(N); ++q) {
    LdsVec<T> w;
#pragma unroll
    for (int r = 0; r < kVecN<T>; ++r) w.v[r] = q * kVecN<T> + r < N ? v[q * kVecN<T> + r] : T(0);
    p[q * kPenLanes] = w;
  }
}

// what links the steps and the waves of a pencil
template <typename T>
struct PenLink {
  // the products across axes A and B: of the last kProdRing steps, a lane
  // each, and those that enter through the pencil's faces: entry q of step s
  // in column kPW (s mod kHaloRing) + q
  LdsVec<T> prod[kProdRing][2][Vecs<T>(5)][kPenLanes];
  LdsVec<T> halo[2][Vecs<T>(5)][kPenLanes];
  int haloReady;  // steps whose halo products are in the ring
  int xReady;     // steps the compute wave has finished
  int sentReady;  // steps whose outgoing products have been sent
  int ticket;
};
template <typename T, bool FULL>
struct PenShared {
  PenSlot<T, FULL> slot[kPenSlots];
  PenLink<T> link;
  int stageReady[kPenSlots];  // slot j holds step stageReady[j] - 1
};

__device__ __forceinline__ int LdsLoad(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// a counter read without waiting for it, to be tested later (an acquire fence
// comes between the test and the reads of what it covers)
__device__ __forceinline__ int LdsPeek(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// publish a step counter for the whole wave.  A wave's LDS operations complete
// in order, so every LDS read and write it issued before is done when another
// wave sees the count; no wait is needed.  The wave barrier is a convergent
// point the compiler cannot duplicate into a lane-divergent branch, the fence
// keeps it from moving LDS accesses across, and one lane stores the count.
__device__ __forceinline__ void LdsPost(int *p, int v) {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  if (__lane_id() == 0) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// wait until an LDS counter reaches `need`; uniform across the wave.  Waves
// that run ahead sleep between polls (polls take LDS cycles from the compute
// wave); the compute wave does not.
template <int SLEEP = 8>
__device__ __forceinline__ void LdsWait(const int *p, int need, int *err) {
  int spins = 0;
  while (__builtin_amdgcn_readfirstlane(LdsLoad(p)) < need) {
    if (++spins > kLdsSpinLimit) {
      __hip_atomic_fetch_or(err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
    if (SLEEP) __builtin_amdgcn_s_sleep(SLEEP);
  }
}

// a workgroup's pencil
struct Pencil {
  int a, b;             // position in the pencil grid
  int pid;              // number within the block
  int C, na, nb;        // axis the pencil runs along, the block's cells across it
  int wa, wb, nc, ns;   // widths, length, steps
  long rec;             // first record of the pencil
  long nrec;            // records of the block
  long msg;             // first message step of the block
  bool toA, toB;        // a pencil lies downstream across A, across B
  bool from[2];         // a pencil lies upstream across A, across B
};
// the next pencil of the launch for this workgroup: every thread gets it
// after the barrier that follows
__device__ __forceinline__ int PencilTicket(const PencilGroup &G) {
  return (int)(__hip_atomic_fetch_add(G.ticket, 1ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) %
               (unsigned long long)G.nent);
}
template <bool FWD>
__device__ __forceinline__ Pencil MakePencil(const DevBlock &b, int4 ent) {
  constexpr int sgn = FWD ? -1 : 1;
  Pencil p;
  p.a = ent.x;
  p.b = ent.y;
  p.pid = p.a + b.pa * p.b;
  p.C = b.pl;
  p.na = AxisN(b, (b.pl + 1) % 3);
  p.nb = AxisN(b, (b.pl + 2) % 3);
  p.wa = PenWidth(p.na, p.a);
  p.wb = PenWidth(p.nb, p.b);
  p.nc = AxisN(b, b.pl);
  p.ns = p.wa + p.wb + p.nc - 2;
  p.rec = (long)p.pid * b.prec;
  p.nrec = Records(b);
  p.msg = ent.w;
  p.toA = p.a - sgn >= 0 && p.a - sgn < b.pa;
  p.toB = p.b - sgn >= 0 && p.b - sgn < b.pb;
  p.from[0] = p.a + sgn >= 0 && p.a + sgn < b.pa;
  p.from[1] = p.b + sgn >= 0 && p.b + sgn < b.pb;
  return p;
}
// a column's lane among those of a step in the records; columns that the
// records do not have read the first one's values, and their results are dropped
__device__ __forceinline__ int RecordLane(const DevBlock &b, int lane) {
  const int la = lane % kPW, lb = lane / kPW;
  return (la >> b.pla) == 0 && (lb >> (b.pln - b.pla)) == 0 ? la + (lb << b.pla) : 0;
}
// record of pencil p's step s, and the column's lane in it
__device__ __forceinline__ long StepAt(const DevBlock &b, const Pencil &p, int s, int recLane, int &lane) {
  int l0;
  const long rec = p.rec + StepRecord(b, s, l0);
  lane = l0 + recLane;
  return rec;
}
// f(axis, whether a record is one step) with both known to the compiler.  Where
// records hold several steps the columns without lanes of their own must not
// store; the test costs a whole step's pass 3 % (48^3, two sweeps: 140 -> 144 us).
template <typename F>
__device__ __forceinline__ void PencilAxis(const DevBlock &b, const Pencil &p, F f) {
  auto with = [&](auto c) {
    if (b.pln == 6) f(c, std::true_type{});
    else f(c, std::false_type{});
  };
  if (p.C == 0) with(std::integral_constant<int, 0>{});
  else if (p.C == 1) with(std::integral_constant<int, 1>{});
  else with(std::integral_constant<int, 2>{});
}
// messages of pencil (pa, pb) of the block through its face f (0 A, 1 B)
template <typename T, bool FWD>
__device__ __forceinline__ T *Messages(const PencilGroup &G, const DevBlock &b, const Pencil &p, int pa, int pb,
                                       int f) {
  return (T *)G.msg[FWD ? 0 : 1] + (p.msg + ((long)(pa + b.pa * pb) * 2 + f) * b.pns) * kMsg;
}

// The send wave: lane = (value e, entry q); entry q of face A is the row
// lb = q, of face B the row la = q.
template <typename T, bool FWD>
__device__ __forceinline__ void PenSend(const PencilGroup &G, const DevBlock &b, const Pencil &p, PenLink<T> &ln,
                                        int lane) {
  if (!p.toA && !p.toB) return;
  constexpr int sgn = FWD ? -1 : 1;
  const int e = lane / kPW, q = lane % kPW;
  // the columns whose products leave the pencil, and their first steps
  const int cA = (FWD ? p.wa - 1 : 0) + kPW * q, cB = q + kPW * (FWD ? p.wb - 1 : 0);
  const int offA = FWD ? p.wa - 1 + q : p.wa - 1 + p.wb - 1 - q, offB = FWD ? q + p.wb - 1 : p.wa - 1 - q + p.wb - 1;
  const bool useA = p.toA && e < 5 && q < p.wb, useB = p.toB && e < 5 && q < p.wa;
  // the receiver's step lags by this pencil's width less one
  T *mA = p.toA ? Messages<T, FWD>(G, b, p, p.a - sgn, p.b, 0) + e * kPW + q - (long)(p.wa - 1) * kMsg : nullptr;
  T *mB = p.toB ? Messages<T, FWD>(G, b, p, p.a, p.b - sgn, 1) + e * kPW + q - (long)(p.wb - 1) * kMsg : nullptr;
  const int ev = e < 5 ? e / kVecN<T> : 0, er = e % kVecN<T>;
  for (int st = 0; st < p.ns; ++st) {
    LdsWait<1>(&ln.xReady, st + 1, G.err);
    const T vA = ln.prod[st & (kProdRing - 1)][0][ev][cA].v[er], vB = ln.prod[st & (kProdRing - 1)][1][ev][cB].v[er];
    // (no wait for the stores of the steps before)
    asm volatile("" ::"v"(vA), "v"(vB));
    LdsPost(&ln.sentReady, st + 1);
    const int kA = st - offA, kB = st - offB;
    if (useA && kA >= 0 && kA < p.nc) StoreCoherent(mA + (long)st * kMsg, NotEmpty(vA));
    if (useB && kB >= 0 && kB < p.nc) StoreCoherent(mB + (long)st * kMsg, NotEmpty(vB));
  }
}

// The halo wave: the products that enter through the pencil's faces, polled
// from the messages of the pencils upstream; on a block face the connection
// terms `bt` (zero off connections, null for none).  One step at a time: a
// poll of two or four steps lasts as long as its slowest load.
template <typename T, bool FWD>
__device__ __forceinline__ void PenHalo(const PencilGroup &G, const DevBlock &b, const Pencil &p, PenLink<T> &ln,
                                        int lane, const T *bt) {
  const int e = lane / kPW, q = lane % kPW;
  const int w[2] = {p.wb, p.wa};
  const T *in[2];
  int off[2];
  bool use[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    in[f] = Messages<T, FWD>(G, b, p, p.a, p.b, f) + min(lane, kMsg - 1);
    off[f] = FWD ? q : w[f] - 1 - q;
    use[f] = e < 5 && q < w[f];
  }
  bool dead = false;
  for (int st = 0; st < p.ns; ++st) {
    LdsWait<1>(&ln.xReady, st + 1 - kHaloRing, G.err);
    T v[2];
    for (int spins = 0;;) {
      bool empty = false;
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        v[f] = p.from[f] ? CoherentLoad(in[f]) : T(0);
        empty |= use[f] && (unsigned)(st - off[f]) < (unsigned)p.nc && IsEmpty(v[f]) && p.from[f];
      }
      if (dead || !__any(empty)) break;
      if (((++spins & 255) == 0 && (__builtin_amdgcn_readfirstlane(CoherentLoad(G.err)) & 2)) || spins > kSpinLimit) {
        // a wait of this launch has timed out: stop waiting at all
        __hip_atomic_fetch_or(G.err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        dead = true;
      }
    }
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int kk = st - off[f];
      if (bt && !p.from[f] && use[f] && kk >= 0 && kk < p.nc) {
        int i, j, k;
        const int edgeA = FWD ? 0 : p.na - 1, edgeB = FWD ? 0 : p.nb - 1;
        Map3(p.C, FWD ? kk : p.nc - 1 - kk, f == 0 ? edgeA : p.a * kPW + q, f == 0 ? p.b * kPW + q : edgeB, i, j, k);
        v[f] = bt[e * b.nbf + BtSlot(b, (p.C + 1 + f) % 3, FWD ? 0 : 1, i, j, k)];
      }
      if (e < 5) ln.halo[f][e / kVecN<T>][kPW * (st % kHaloRing) + q].v[e % kVecN<T>] = v[f];
      in[f] += kMsg;
    }
    LdsPost(&ln.haloReady, st + 1);
  }
}

// empty this pencil's message slots of the other direction's pass (thread t
// of n)
template <typename T, bool FWD>
__device__ __forceinline__ void PenEmpty(const PencilGroup &G, const DevBlock &b, const Pencil &p, int t, int n) {
  T *const old = Messages<T, !FWD>(G, b, p, p.a, p.b, 0);
  for (long q = t; q < 2L * b.pns * kMsg; q += n) old[q] = EmptySlot<T>();
}

// the connection term across C of a lane's first cell (zero off connections)
template <typename T, bool FWD>
__device__ __forceinline__ void PenFirst(const DevBlock &b, const Pencil &p, int lane, const T *bt, T out[5]) {
  const int la = lane % kPW, lb = lane / kPW;
  const bool conn = bt && la < p.wa && lb < p.wb;
  int i, j, k;
  Map3(p.C, FWD ? 0 : p.nc - 1, p.a * kPW + la, p.b * kPW + lb, i, j, k);
  const long q = conn ? BtSlot(b, p.C, FWD ? 0 : 1, i, j, k) : 0;
#pragma unroll
  for (int e = 0; e < 5; ++e) out[e] = conn ? bt[e * b.nbf + q] : T(0);
}

// one step's slot from the sweep-ordered inputs
template <typename T, bool FWD, bool FULL>
__device__ __forceinline__ void PenStage(const DevBlock &b, const Params &P, const Pencil &pen,
                                         PenSlot<T, FULL> &sl, int lane, int recLane, int st, const int *xReady,
                                         int *err) {
  const GasT<T> g = Cast<T>(P.gas);
  int rl;
  const long rec = StepAt(b, pen, FWD ? st : pen.ns - 1 - st, recLane, rl);
  const int nS = kPenS + (P.visc.on ? 1 : 0), nF = kPenF + (P.visc.on ? 3 : 0);
  const double *S = b.skS + rec * nS * kPenLanes + rl;
  const double *F = b.skF + ((FWD ? pen.nrec : 0) + rec) * nF * kPenLanes + rl;
  // every load before the wait for the slot
  T W[5], fa[12], early[kEarly<T, FULL>];
#pragma unroll
  for (int e = 0; e < 5; ++e) W[e] = T(S[e * kPenLanes]);
#pragma unroll
  for (int q = 0; q < 12; ++q) fa[q] = T(F[q * kPenLanes]);
  if (FWD || FULL) {
#pragma unroll
    for (int e = 0; e < 5; ++e) early[e] = T(S[(5 + e) * kPenLanes]);
  } else {
    const T *X = (const T *)b.skX + rec * 5 * kPenLanes + rl;
#pragma unroll
    for (int e = 0; e < 5; ++e) early[e] = X[e * kPenLanes];
  }
  early[5] = T(S[10 * kPenLanes]);
  if constexpr (FULL) {
    const T *o = (const T *)b.skO + rec * 5 * kPenLanes + rl;
#pragma unroll
    for (int e = 0; e < 5; ++e) early[11 + e] = o[e * kPenLanes];
  }
  T mu = T(0), dist[3] = {T(1), T(1), T(1)};
  if (P.visc.on) {
    mu = T(S[kPenS * kPenLanes]);
#pragma unroll
    for (int q = 0; q < 3; ++q) dist[q] = T(F[(kPenF + q) * kPenLanes]);
  }
  T late[3][kLate<T>];
  if constexpr (sizeof(T) == 8) {
    PrimToCons(g, W, &early[6]);
  } else {
#pragma unroll
    for (int e = 0; e < 5; ++e) early[6 + e] = W[e];
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const T nx = fa[4 * q], ny = fa[4 * q + 1], nz = fa[4 * q + 2], mag = fa[4 * q + 3];
    T lam = T(0.5) * mag * (fabs((W[1] * nx + W[2] * ny) + W[3] * nz) + SoS(g, W[0], W[4]));
    if (P.visc.on) lam += ViscFaceSR<T>(g, W, mag, dist[q], mu, P.visc);
    late[q][0] = nx;
    late[q][1] = ny;
    late[q][2] = nz;
    late[q][3] = T(0.5) * mag;
    late[q][4] = lam;
    if constexpr (sizeof(T) == 8) {
      PhysFlux(g, W, nx, ny, nz, &late[q][5]);
    } else {
      late[q][5] = (W[1] * nx + W[2] * ny) + W[3] * nz;
      late[q][6] = EnergyPlusP(g, W);
    }
  }
  // the slot is free once the compute wave has finished step st - kPenSlots
  LdsWait(xReady, st - kPenSlots + 1, err);
  LdsPut<T, kEarly<T, FULL>>(&sl.early[0][lane], early);
#pragma unroll
  for (int q = 0; q < 3; ++q) LdsPut<T, kLate<T>>(&sl.late[q][0][lane], late[q]);
}

// Where a pass writes its sweep-ordered output of step st.  The
// dependency-side sums of a full pass are the other-side sums of the next: its
// cells' neighbours on that side still have this pass's du then, so without
// connections (whose ghost du changes in between) only the first full pass of a
// relax needs KPencilOther.  The stager reads a step's values before the compute
// wave writes them.  40 iterations of two sweeps, 48^3 viscous cells: 34.6 ms with
// KPencilOther before each pass, 30.7 so.
template <typename T, bool FWD, bool FULL>
__device__ __forceinline__ T *PenStore(const DevBlock &b, const Pencil &pen, int st, int recLane) {
  int rl;
  const long rec = StepAt(b, pen, FWD ? st : pen.ns - 1 - st, recLane, rl);
  return (FULL ? (T *)b.skO : (T *)b.skX) + rec * 5 * kPenLanes + rl;
}

// The compute wave.  A wave issues one instruction in 4.6 cycles whatever it
// depends on, so a step costs its instruction count plus what it waits for,
// and it is ordered so that it waits for nothing: each value of the next step
// is read from LDS as soon as this step has used the last one, between the
// arithmetic; the counters are read well before they are tested; the products
// across B and A go into LDS (where the next step's lanes and the send wave
// take them) before the one across C, which stays in the lane's registers, is
// formed.
template <typename T, bool FWD, bool FULL, int C, bool WHOLE>
__device__ __forceinline__ void PenCompute(const DevBlock &b, const Params &P, const Pencil &pen,
                                           PenShared<T, FULL> &sh, int lane, int store, int *err) {
  constexpr int sgn = FWD ? -1 : 1;  // direction of the dependency neighbours
  constexpr int V5 = Vecs<T>(5);
  PenLink<T> &ln = sh.link;
  const bool sends = pen.toA || pen.toB;
  const GasT<T> g = Cast<T>(P.gas);
  const auto byCvs = MakeDivisor(g.cvs);
  const int ns = pen.ns, nc = pen.nc;
  const int la = lane % kPW, lb = lane / kPW;
  const bool col = la < pen.wa && lb < pen.wb;
  const int off = FWD ? la + lb : (pen.wa - 1 - la) + (pen.wb - 1 - lb);
  const bool firstA = FWD ? la == 0 : la == pen.wa - 1, firstB = FWD ? lb == 0 : lb == pen.wb - 1;
  // where the lane's incoming products lie: the neighbour lane's of the step
  // before, or the halo ring's
  const int nlA = min(max(lane + sgn, 0), kPenLanes - 1), nlB = min(max(lane + sgn * kPW, 0), kPenLanes - 1);
  const LdsVec<T> *const inA = firstA ? &ln.halo[0][0][lb] : &ln.prod[0][0][0][nlA];
  const LdsVec<T> *const inB = firstB ? &ln.halo[1][0][la] : &ln.prod[0][1][0][nlB];
  constexpr int kProdStep = 2 * V5 * kPenLanes;  // vectors of one step of the product ring
  const int gA = pen.a * kPW + la, gB = pen.b * kPW + lb;
  T oC[5];
  PenFirst<T, FWD>(b, pen, lane, OpBuf<T>::Bt(b), oC);
  // du in the natural layout: a lane's cells follow each other along C
  T *const x = OpBuf<T>::X(b);
  int i0, j0, k0;
  Map3(C, FWD ? -off : nc - 1 + off, gA, gB, i0, j0, k0);
  const int sC = -sgn * (C == 0 ? 1 : (C == 1 ? b.ni : b.ni * b.nj));
  int p = i0 + j0 * b.ni + k0 * b.ni * b.nj;  // cell of step st (of the active steps)
  // one-sweep forward pass: du for the backward pass; full pass: the
  // dependency-side sums for the next pass (PenStore)
  const int recLane = RecordLane(b, lane);
  T *Xs = PenStore<T, FWD, FULL>(b, pen, 0, recLane);
  T xA[5], xB[5], S[5], early[kEarly<T, FULL>], late[3][kLate<T>];
  int next = 1;  // slot of the next step
  LdsWait<0>(&sh.stageReady[0], 1, err);
  LdsWait<0>(&ln.haloReady, 1, err);
  int stage = LdsPeek(&sh.stageReady[next]), halo, sent;
  LdsGet<T, kEarly<T, FULL>>(&sh.slot[0].early[0][lane], early);
  LdsGet<T, 5>(inA, xA);
  LdsGet<T, 5>(inB, xB);
#pragma unroll
  for (int q = 0; q < 2; ++q) LdsGet<T, kLate<T>>(&sh.slot[0].late[q][0][lane], late[q]);
  const PenSlot<T, FULL> *cur = &sh.slot[0];
  // The loop from a cache line's start on: without it a pass takes up to 2 %
  // longer along one axis or another as the code before it changes (57 x 49 x 38
  // FP64 along i 141 against 139 us, 40^3 FP32 105 against 103).
  asm volatile(".p2align 6");
  for (int st = 0; st < ns; ++st) {
    const bool more = st + 1 < ns;
    __builtin_amdgcn_sched_barrier(0);
    LdsGet<T, kLate<T>>(&cur->late[2][0][lane], late[2]);
    // the dependency-side sum in the order of ImplicitLower / ImplicitUpper
    // (i, j, k); products of absent neighbours are +0 and leave it unchanged
    // (it starts at +0 and is never -0)
    T xn[5], Un[5], W0[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const T o0 = C == 2 ? xA[e] : (C == 0 ? oC[e] : xB[e]), o1 = C == 2 ? xB[e] : (C == 0 ? xA[e] : oC[e]),
              o2 = C == 2 ? oC[e] : (C == 0 ? xB[e] : xA[e]);
      const T D = ((T(0) + o0) + o1) + o2, v = early[e], ainv = early[5];
      S[e] = D;
      if constexpr (FULL) xn[e] = FWD ? (v + (D - early[11 + e])) * ainv : ((v + early[11 + e]) - D) * ainv;
      else xn[e] = FWD ? (v + D) * ainv : v - D * ainv;
      W0[e] = early[6 + e];
      Un[e] = W0[e] + xn[e];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more && __builtin_amdgcn_readfirstlane(stage) < st + 2) LdsWait<0>(&sh.stageReady[next], st + 2, err);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const PenSlot<T, FULL> &sl = sh.slot[next];
    LdsGet<T, kEarly<T, FULL>>(&sl.early[0][lane], early);
    next = next + 1 == kPenSlots ? 0 : next + 1;
    stage = LdsPeek(&sh.stageReady[next]);
    sent = LdsPeek(&ln.sentReady);
    // the updated state
    T Wu[5], H = T(0);
    StateChange<T> ch;
    if constexpr (sizeof(T) == 8) ConsToPrimH(g, byCvs, Un, Wu, H);
    else ch = ChangeOf(g, W0, xn);
    // the outgoing product across axis q
    auto product = [&](int q, T o[5]) {
      if constexpr (sizeof(T) == 8) {
        PhysFluxH(Wu, H, late[q][0], late[q][1], late[q][2], o);
#pragma unroll
        for (int e = 0; e < 5; ++e) o[e] = o[e] - late[q][5 + e];
      } else {
        ChangeThrough(ch, W0[0], xn[4], late[q][5], late[q][6], late[q][0], late[q][1], late[q][2], o);
      }
#pragma unroll
      for (int e = 0; e < 5; ++e) {
        const T fc = late[q][3] * o[e];
        o[e] = FWD ? fc + xn[e] * late[q][4] : fc - xn[e] * late[q][4];
      }
    };
    // the product ring's place is free once its products have been sent
    if (sends && __builtin_amdgcn_readfirstlane(sent) < st + 1 - kProdRing)
      LdsWait<0>(&ln.sentReady, st + 1 - kProdRing, err);
    LdsVec<T> *const out = &ln.prod[st & (kProdRing - 1)][0][0][lane];
    T o[5];
    product(1, o);
    LdsPut<T, 5>(out + V5 * kPenLanes, o);
    __builtin_amdgcn_sched_barrier(0);
    halo = LdsPeek(&ln.haloReady);
    LdsGet<T, kLate<T>>(&sl.late[1][0][lane], late[1]);
    product(0, o);
    LdsPut<T, 5>(out, o);
    // this step's slot (read in the step before) and ring columns are free,
    // and its products are in LDS (a wave's LDS operations complete in order)
    LdsPost(&ln.xReady, st + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (more && __builtin_amdgcn_readfirstlane(halo) < st + 2) LdsWait<0>(&ln.haloReady, st + 2, err);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int ro = kPW * ((st + 1) % kHaloRing), po = kProdStep * (st & (kProdRing - 1));
    LdsGet<T, 5>(inB + (firstB ? ro : po), xB);
    LdsGet<T, 5>(inA + (firstA ? ro : po), xA);
    LdsGet<T, kLate<T>>(&sl.late[0][0][lane], late[0]);
    cur = &sl;
    const int kk = st - off;
    const bool act = col && kk >= 0 && kk < nc;
    if (act) {
      product(2, oC);
      if (store & 1) {
#pragma unroll
        for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = xn[e];
      }
    }
    if ((FWD || FULL) && (store & 2) && (WHOLE || act)) {
#pragma unroll
      for (int e = 0; e < 5; ++e) Xs[e * kPenLanes] = FULL ? S[e] : xn[e];
    }
    p += sC;
    if constexpr (WHOLE) Xs += (FWD ? 5 : -5) * kPenLanes;
    else Xs = PenStore<T, FWD, FULL>(b, pen, min(st + 1, ns - 1), recLane);
  }
}

// `store`: bit 0 du in the natural layout, bit 1 in sweep order (a one-sweep
// forward pass, whose backward pass reads it) or, of a full pass, the sums for
// the next (PenStore)
template <typename T, bool FWD, bool FULL>
__global__ void __launch_bounds__(kPenWaves * kPenLanes) KLusgsPencil(PencilGroup G, Params P, int store) {
  __shared__ PenShared<T, FULL> sh;
  const int tid = threadIdx.x, lane = tid % kPenLanes;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kPenLanes);
  if (tid == 0) {
    sh.link.ticket = PencilTicket(G);
    sh.link.haloReady = sh.link.xReady = sh.link.sentReady = 0;
  }
  if (tid < kPenSlots) sh.stageReady[tid] = 0;
  __syncthreads();
  const int t = __builtin_amdgcn_readfirstlane(sh.link.ticket);
  const int4 ent = G.entries[FWD ? t : G.nent - 1 - t];
  const DevBlock b = G.blocks[ent.z];
  const Pencil pen = MakePencil<FWD>(b, ent);
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(3);
    PencilAxis(b, pen, [&](auto c, auto whole) {
      PenCompute<T, FWD, FULL, c.value, whole.value>(b, P, pen, sh, lane, store, G.err);
    });
  } else if (wave == 1) {
    PenHalo<T, FWD>(G, b, pen, sh.link, lane, OpBuf<T>::Bt(b));
  } else if (wave == 2) {
    PenSend<T, FWD>(G, b, pen, sh.link, lane);
  } else {
    // stager j: steps j, j + kStagers, ...
    const int j = wave - 3, recLane = RecordLane(b, lane);
    for (int st = j; st < pen.ns; st += kStagers) {
      PenStage<T, FWD, FULL>(b, P, pen, sh.slot[j], lane, recLane, st, &sh.link.xReady, G.err);
      LdsPost(&sh.stageReady[j], st + 1);
    }
    PenEmpty<T, FWD>(G, b, pen, j * kPenLanes + lane, kStagers * kPenLanes);
  }
}

// ---------------------------------------------------------------------------
// Block LU-SGS pencil sweep (blusgs): the scheme of KLusgsPencil with 5x5
// blocks.  A cell's outgoing product across axis q is J_q du, J_q the block its
// neighbour has for it (NeighbourBlock: this cell's Rusanov Jacobian at the
// shared face with its thin-shear-layer Jacobian), and du = D^-1 (b + sum of
// the incoming products).  Four stager waves a step (one for each of the three
// blocks, one for D^-1, right-hand side or forward du, and the other-side sum
// of a full sweep) form the next step in LDS; the compute wave applies the four
// matrices, row by row in BlockMult's order, so the result is that of
// KLusgsForward / KLusgsBackward bit for bit.
//
// Bound by the step: one wave's 195 FP64 operations and 54 16-byte LDS reads,
// 1.09 us alone in FP64 (48^3 without viscous terms), and what it waits for.  On
// the eight blocks of the 1.03M-cell channel a step takes 1.87 us, 0.42 of them
// for its blocks (the stagers issue and wait for their loads, 184 pencils at
// once, for as long as they form) and 0.42 for the pencil upstream.  A pass there
// takes 354 us (FP32 319), of eight blocks of 59 x 39 x 19 and smaller 189 (170),
// of 24 x 16 x 8 and smaller 68 (58); the tile sweep with per-tile flags that was
// here before took 508 (494), 207 (317) and 83 (138), so it is gone.  FP32 waves
// of 168 registers hold two sets of stagers without scratch (one set: 343, 195,
// 73 us); FP64 waves of 168 spill (820 us), so one set with 256.
constexpr int kBlkSlots = 2;
template <typename T>
constexpr int kBlkSets = sizeof(T) == 4 ? 2 : 1;  // groups of four stager waves, each taking every kBlkSets-th step
template <typename T>
constexpr int kBlkWaves = 3 + 4 * kBlkSets<T>;
static_assert(kBlkSlots % kBlkSets<float> == 0 && kBlkSlots % kBlkSets<double> == 0, "a stager's slots");
template <bool FULL>
constexpr int kBlkR = FULL ? 10 : 5;  // right-hand side (forward du), other-side sum
template <typename T, bool FULL>
struct BlkSlot {
  LdsVec<T> J[3][Vecs<T>(25)][kPenLanes];
  LdsVec<T> D[kPenLanes * Vecs<T>(25)];  // the step's D^-1 as they are in memory, one cell behind the other
  LdsVec<T> r[Vecs<T>(kBlkR<FULL>)][kPenLanes];
};
constexpr int kBlkParts = 4;  // blocks of A, B, C; the rest
template <typename T, bool FULL>
struct BlkShared {
  BlkSlot<T, FULL> slot[kBlkSlots];
  PenLink<T> link;
  int ready[kBlkSlots];  // parts put into the slot so far: step st is there at kBlkParts (st / kBlkSlots + 1)
};

// one more part in a slot (the LDS writes before it are done, see LdsPost)
__device__ __forceinline__ void LdsAdd(int *p) {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  if (__lane_id() == 0) __hip_atomic_fetch_add(p, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// stager of the blocks of axis A + q: the cell's values and the face's
struct BlkRaw {
  double W[5], mu, kc, vg[9], a[4], dist;
};
template <bool FWD, bool VISC>
__device__ __forceinline__ void BlkLoad(const DevBlock &b, const Pencil &pen, int q, int recLane, int st, BlkRaw &r) {
  int rl;
  const long rec = StepAt(b, pen, FWD ? st : pen.ns - 1 - st, recLane, rl);
  constexpr int nF = kPenF + (VISC ? 3 : 0);
  const double *S = b.skS + rec * BlockRecord(VISC) * kPenLanes + rl;
  const double *F = b.skF + ((FWD ? pen.nrec : 0) + rec) * nF * kPenLanes + rl;
#pragma unroll
  for (int e = 0; e < 5; ++e) r.W[e] = S[e * kPenLanes];
#pragma unroll
  for (int e = 0; e < 4; ++e) r.a[e] = F[(4 * q + e) * kPenLanes];
  if constexpr (VISC) {
    r.mu = S[10 * kPenLanes];
    r.kc = S[11 * kPenLanes];
#pragma unroll
    for (int e = 0; e < 9; ++e) r.vg[e] = S[(12 + e) * kPenLanes];
    r.dist = F[(kPenF + q) * kPenLanes];
  }
}
// the block, formed in FP64 as NeighbourBlock forms it, in the operator's
// precision
template <typename T, bool FWD, bool VISC>
__device__ __forceinline__ void BlkForm(const Params &P, const BlkRaw &r, T out[25]) {
#pragma clang fp contract(off)
  const GasT<double> g = Cast<double>(P.gas);
  double J[25];
  RusanovJacobian<double>(g, r.W, r.a[0], r.a[1], r.a[2], r.a[3], FWD, J);
  if constexpr (VISC) {
    double V[25];
    TSLJacobian(g, P.visc, r.W, r.mu, r.kc, make_double4(r.a[0], r.a[1], r.a[2], r.a[3]), r.dist, FWD, r.vg, V);
#pragma unroll
    for (int q = 0; q < 25; ++q) J[q] = FWD ? J[q] - V[q] : J[q] + V[q];
  }
#pragma unroll
  for (int q = 0; q < 25; ++q) out[q] = T(J[q]);
}

template <typename T, bool FWD, bool FULL>
__device__ __forceinline__ void BlkStage(const DevBlock &b, const Params &P, const Pencil &pen,
                                         BlkShared<T, FULL> &sh, int lane, int set, int part, int *err) {
  const int *xReady = &sh.link.xReady;
  const int recLane = RecordLane(b, lane);
  if (part < 3) {
    // With and without the viscous terms in loops of their own.  The stagers of
    // a viscous block bound the pass (a step of one pencil alone: 3240 cycles, 760
    // of them the compute wave waiting for its blocks; without the viscous terms
    // 2820 and 2): a branch in the loop cost them 5 % of a pass.
    auto blocks = [&](auto visc) {
      constexpr bool kVisc = visc.value;
      BlkRaw r;
      auto load = [&](int st) { BlkLoad<FWD, kVisc>(b, pen, part, recLane, min(st, pen.ns - 1), r); };
      load(set);
      for (int st = set; st < pen.ns; st += kBlkSets<T>) {
        T J[25];
        BlkForm<T, FWD, kVisc>(P, r, J);
        // formed here, not behind the wait for the slot (where the compiler
        // would put it: FP32 pass 167 -> 255 us on 48^3 cells)
#pragma unroll
        for (int q = 0; q < 25; ++q) asm volatile("" : "+v"(J[q]));
        // the next step's loads are in flight while the slot is waited for
        load(st + kBlkSets<T>);
        const int slot = st % kBlkSlots;
        LdsWait<1>(xReady, st - kBlkSlots + 1, err);
        LdsPut<T, 25>(&sh.slot[slot].J[part][0][lane], J);
        LdsAdd(&sh.ready[slot]);
      }
    };
    if (P.visc.on) blocks(std::true_type{});
    else blocks(std::false_type{});
    return;
  }
  constexpr int V = Vecs<T>(25);
  T d[V * kVecN<T>], r[kBlkR<FULL>];
  auto load = [&](int st) {
    int rl;
    const long rec = StepAt(b, pen, FWD ? st : pen.ns - 1 - st, recLane, rl);
    // the step's cells, and what follows them in memory where they are fewer
    // than 64 (the array has that much more behind its last record)
    const LdsVec<T> *ai = (const LdsVec<T> *)OpBuf<T>::Abi(b) + (rec * kPenLanes + (rl - recLane)) * V + lane;
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const LdsVec<T> w = ai[q * kPenLanes];
#pragma unroll
      for (int e = 0; e < kVecN<T>; ++e) d[q * kVecN<T> + e] = w.v[e];
    }
    if (FWD || FULL) {
      const double *S = b.skS + (rec * BlockRecord(P.visc.on) + 5) * kPenLanes + rl;
#pragma unroll
      for (int e = 0; e < 5; ++e) r[e] = T(S[e * kPenLanes]);
    } else {
      const T *X = (const T *)b.skX + rec * 5 * kPenLanes + rl;
#pragma unroll
      for (int e = 0; e < 5; ++e) r[e] = X[e * kPenLanes];
    }
    if constexpr (FULL) {
      const T *o = (const T *)b.skO + rec * 5 * kPenLanes + rl;
#pragma unroll
      for (int e = 0; e < 5; ++e) r[5 + e] = o[e * kPenLanes];
    }
  };
  if (set < pen.ns) load(set);
  for (int st = set; st < pen.ns; st += kBlkSets<T>) {
    const int slot = st % kBlkSlots;
    LdsWait<1>(xReady, st - kBlkSlots + 1, err);
    LdsPut<T, V * kVecN<T>>(&sh.slot[slot].D[lane], d);
    LdsPut<T, kBlkR<FULL>>(&sh.slot[slot].r[0][lane], r);
    LdsAdd(&sh.ready[slot]);
    load(min(st + kBlkSets<T>, pen.ns - 1));
  }
}

template <typename T, bool FWD, bool FULL, int C, bool WHOLE>
__device__ __forceinline__ void BlkCompute(const DevBlock &b, const Pencil &pen, BlkShared<T, FULL> &sh, int lane,
                                           int store, const T *bt, int *err) {
  constexpr int sgn = FWD ? -1 : 1;  // direction of the dependency neighbours
  constexpr int V5 = Vecs<T>(5);
  PenLink<T> &ln = sh.link;
  const bool sends = pen.toA || pen.toB;
  const int ns = pen.ns, nc = pen.nc;
  const int la = lane % kPW, lb = lane / kPW;
  const bool col = la < pen.wa && lb < pen.wb;
  const int off = FWD ? la + lb : (pen.wa - 1 - la) + (pen.wb - 1 - lb);
  const bool firstA = FWD ? la == 0 : la == pen.wa - 1, firstB = FWD ? lb == 0 : lb == pen.wb - 1;
  const int nlA = min(max(lane + sgn, 0), kPenLanes - 1), nlB = min(max(lane + sgn * kPW, 0), kPenLanes - 1);
  const LdsVec<T> *const inA = firstA ? &ln.halo[0][0][lb] : &ln.prod[0][0][0][nlA];
  const LdsVec<T> *const inB = firstB ? &ln.halo[1][0][la] : &ln.prod[0][1][0][nlB];
  constexpr int kProdStep = 2 * V5 * kPenLanes;  // vectors of one step of the product ring
  T oC[5];
  PenFirst<T, FWD>(b, pen, lane, bt, oC);
  T *const x = OpBuf<T>::X(b);
  int i0, j0, k0;
  Map3(C, FWD ? -off : nc - 1 + off, pen.a * kPW + la, pen.b * kPW + lb, i0, j0, k0);
  const int sC = -sgn * (C == 0 ? 1 : (C == 1 ? b.ni : b.ni * b.nj));
  int p = i0 + j0 * b.ni + k0 * b.ni * b.nj;  // cell of step st (of the active steps)
  const int recLane = RecordLane(b, lane);
  T *Xs = PenStore<T, FWD, FULL>(b, pen, 0, recLane);  // (see PenCompute)
  T xA[5], xB[5], S[5], d[25], r[kBlkR<FULL>], JA[25], JB[25];
  LdsWait<0>(&sh.ready[0], kBlkParts, err);
  LdsGet<T, 25, 1>(&sh.slot[0].D[recLane * Vecs<T>(25)], d);
  LdsGet<T, kBlkR<FULL>>(&sh.slot[0].r[0][lane], r);
  LdsWait<0>(&ln.haloReady, 1, err);
  LdsGet<T, 5>(inA, xA);
  LdsGet<T, 5>(inB, xB);
  for (int st = 0; st < ns; ++st) {
    const bool more = st + 1 < ns;
    const int cur = st % kBlkSlots, next = (st + 1) % kBlkSlots;
    const BlkSlot<T, FULL> &sl = sh.slot[cur], &nx = sh.slot[next];
    // the dependency-side sum, i, j, k order from +0 (see PenCompute)
    T xn[5], v[5], o[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const T o0 = C == 2 ? xA[e] : (C == 0 ? oC[e] : xB[e]), o1 = C == 2 ? xB[e] : (C == 0 ? xA[e] : oC[e]),
              o2 = C == 2 ? oC[e] : (C == 0 ? xB[e] : xA[e]);
      const T D = ((T(0) + o0) + o1) + o2;
      S[e] = D;
      if constexpr (FULL) v[e] = FWD ? r[e] + (D - r[5 + e]) : (r[e] + r[5 + e]) - D;
      else v[e] = FWD ? r[e] + D : D;
    }
    BlockMult<T>(d, v, xn);
    if constexpr (!FULL && !FWD) {
#pragma unroll
      for (int e = 0; e < 5; ++e) xn[e] = r[e] - xn[e];
    }
    __builtin_amdgcn_sched_barrier(0);
    LdsGet<T, 25>(&sl.J[1][0][lane], JB);
    LdsGet<T, 25>(&sl.J[0][0][lane], JA);
    const int ready = LdsPeek(&sh.ready[next]), need = kBlkParts * ((st + 1) / kBlkSlots + 1);
    const int sent = LdsPeek(&ln.sentReady);
    BlockMult<T>(JB, xn, o);
    // the product ring's place is free once its products have been sent
    if (sends && __builtin_amdgcn_readfirstlane(sent) < st + 1 - kProdRing)
      LdsWait<0>(&ln.sentReady, st + 1 - kProdRing, err);
    LdsVec<T> *const out = &ln.prod[st & (kProdRing - 1)][0][0][lane];
    LdsPut<T, 5>(out + V5 * kPenLanes, o);
    __builtin_amdgcn_sched_barrier(0);
    LdsGet<T, 25>(&sl.J[2][0][lane], JB);
    const int halo = LdsPeek(&ln.haloReady);
    BlockMult<T>(JA, xn, o);
    LdsPut<T, 5>(out, o);
    // the slot has been read, its products are in LDS
    LdsPost(&ln.xReady, st + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (more && __builtin_amdgcn_readfirstlane(ready) < need) LdsWait<0>(&sh.ready[next], need, err);
    const int kk = st - off;
    const bool act = col && kk >= 0 && kk < nc;
    if constexpr (sizeof(T) == 8) {
      if (act) BlockMult<T>(JB, xn, oC);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    LdsGet<T, kBlkR<FULL>>(&nx.r[0][lane], r);
    LdsGet<T, 25, 1>(&nx.D[recLane * Vecs<T>(25)], d);
    if (more && __builtin_amdgcn_readfirstlane(halo) < st + 2) LdsWait<0>(&ln.haloReady, st + 2, err);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int ro = kPW * ((st + 1) % kHaloRing), po = kProdStep * (st & (kProdRing - 1));
    LdsGet<T, 5>(inB + (firstB ? ro : po), xB);
    LdsGet<T, 5>(inA + (firstA ? ro : po), xA);
    __builtin_amdgcn_sched_barrier(0);
    if (act) {
      if constexpr (sizeof(T) == 4) BlockMult<T>(JB, xn, oC);
      if (store & 1) {
#pragma unroll
        for (int e = 0; e < 5; ++e) x[e * b.ncell + p] = xn[e];
      }
    }
    if ((FWD || FULL) && (store & 2) && (WHOLE || act)) {
#pragma unroll
      for (int e = 0; e < 5; ++e) Xs[e * kPenLanes] = FULL ? S[e] : xn[e];
    }
    p += sC;
    if constexpr (WHOLE) Xs += (FWD ? 5 : -5) * kPenLanes;
    else Xs = PenStore<T, FWD, FULL>(b, pen, min(st + 1, ns - 1), recLane);
  }
}

// `store` as in KLusgsPencil.  The first forward pass starts from du = 0, so
// its connection terms are zero (J 0 sums to +0) and are not formed.
template <typename T, bool FWD, bool FULL>
__global__ void __launch_bounds__(kBlkWaves<T> * kPenLanes) KBlockPencil(PencilGroup G, Params P, int store) {
  __shared__ BlkShared<T, FULL> sh;
  const int tid = threadIdx.x, lane = tid % kPenLanes;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kPenLanes);
  if (tid == 0) {
    sh.link.ticket = PencilTicket(G);
    sh.link.haloReady = sh.link.xReady = sh.link.sentReady = 0;
  }
  if (tid < kBlkSlots) sh.ready[tid] = 0;
  __syncthreads();
  const int t = __builtin_amdgcn_readfirstlane(sh.link.ticket);
  const int4 ent = G.entries[FWD ? t : G.nent - 1 - t];
  const DevBlock b = G.blocks[ent.z];
  const Pencil pen = MakePencil<FWD>(b, ent);
  const T *bt = FWD && !FULL ? nullptr : OpBuf<T>::Bt(b);
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(3);
    PencilAxis(b, pen, [&](auto c, auto whole) {
      BlkCompute<T, FWD, FULL, c.value, whole.value>(b, pen, sh, lane, store, bt, G.err);
    });
  } else if (wave == 1) {
    PenHalo<T, FWD>(G, b, pen, sh.link, lane, bt);
  } else if (wave == 2) {
    PenSend<T, FWD>(G, b, pen, sh.link, lane);
  } else {
    // waves 4 and 8 share the compute wave's SIMD (waves are dealt to the four
    // SIMDs in turn): they take the light part
    constexpr int kSets = kBlkSets<T>;
    const int heavy = wave == 3 ? 0 : wave - 4 - (wave - 5) / 4;  // 3, 5, 6, 7, 9, 10
    const bool light = wave % 4 == 0;
    BlkStage<T, FWD, FULL>(b, P, pen, sh, lane, light ? wave / 4 - 1 : heavy % kSets, light ? 3 : heavy / kSets, G.err);
    PenEmpty<T, FWD>(G, b, pen, (wave - 3) * kPenLanes + lane, 4 * kBlkSets<T> * kPenLanes);
  }
}

}  // namespace ath
