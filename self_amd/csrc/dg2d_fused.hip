// Fused DGSEM tendency + low-storage RK3 stage kernels and the Model2D engine.
//
// One launch per RK stage does the whole of CalculateTendency_Model2D + UpdateGRK3
// (src/SELF_Model2D.f90:710-752, 816-859) for a block of elements:
//   phase 0  node work-items: load S (and G), physical flux -> contravariant flux (LDS),
//            nodal trace quantities q(S) (LDS)
//   phase 1  face work-items: own traces from LDS (bMatrix contraction), neighbour traces
//            from the previous launch's trace buffer (the only cross-element read),
//            boundary conditions, Riemann flux * nScale (LDS)
//   phase 2  node work-items: weak DG divergence (dgMatrix + bMatrix/qWeights), / J,
//            source, dSdt, G = a G + dSdt, S += (g dt) G; write S, G; q(S_new) -> LDS
//   phase 3  face work-items: traces of S_new -> the other trace buffer
// so per stage each element reads S, G, its static fields and its neighbours' traces and
// writes S, G and its own traces: the algorithmic minimum for a nodal DG stage with
// Gauss points (no collocated face nodes).  Trace buffers alternate between launches.
//
// Work mapping: blocks of 64, 128 or 256 work-items (the tile, autotuned per degree), EPB =
// THREADS/(N+1)^2 elements per block; at N = 7 one wave64 owns one element, lane = i + 8 j,
// so every variable is one 512-byte coalesced access and the per-element geometry record is
// wave-uniform.
//
// Geometry: the fast path takes affine elements (metric terms constant per element, true
// for the structured and block meshes); each element carries one 20-double record.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <mutex>
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "closure.hpp"
#include "mlp_rows.hpp"
#include "sw_adjoint.hpp"
#include "../../include/self_amd.h"

using namespace selfamd;

namespace {

constexpr int kThreads = 256;
constexpr int kNbrOrphan = -0x40000000;
// forward_step calls of at most this many steps with a step size other than the captured
// graphs' are launched stage by stage instead of recapturing
constexpr int kDirectSteps = 2;
// Calls of at least kResidentSteps steps take a resident launch where the mesh allows it, single
// steps from kResidentElements elements on: below, a cooperative launch of three stages costs what
// it saves (N = 7: 28.8 against 28.3 us per call at 10^2 elements before the gate, which adds 2 to 3;
// 34.6 against 36.2 at 40^2.  On 17 meshes of all physics from 1,024 to 14,400 elements no call of 1 to
// 8 steps is slower than by graphs).
constexpr int kResidentSteps = 2, kResidentElements = 1024;
// Instances whose registers spill pay for it once per call: from this many steps on (SW N = 3,
// 18,400 elements: 60 against 49 us for one step, 10.2 against 11.3 us per stage).
constexpr int kResidentSpillSteps = 5;
// Resident launches of one process run one after another, where step graphs of several streams
// overlap.  So while this many other models step at the same time (company_of), meshes of up to
// kCompanyWaves wavefronts per CU, a stage of which leaves most of the device idle, take graphs.  Steps
// of K models, all enqueued from one thread before any is waited for, by graphs and by resident launches:
//   SW 32^2 N = 3 (1 wavefront per CU), 100 steps   K = 2 1,340 and 1,140 us, K = 3 1,480 and 1,800, K = 8 3,220 and 4,690
//   Euler 16^2 N = 4 (1), 100 steps                 K = 2 2,130 and 1,540, K = 3 2,270 and 2,360, K = 8 4,740 and 6,200
//   linear SW 20^2 N = 7 (2), 200 steps             K = 2 2,920 and 2,070, K = 3 3,220 and 3,140, K = 8 7,130 and 8,320
//   Euler 60^2 N = 4 (7), 24 steps                  K = 2 1,020 and 630, K = 3 1,280 and 930, K = 8 3,750 and 2,500
//   SW 64^2 N = 7 (16), 24 steps                    K = 2 1,050 and 800, K = 3 1,420 and 1,240, K = 8 3,700 and 3,230
constexpr int kCompany = 2, kCompanyWaves = 4;  // the latter: leaves_room
// After a launch that found no place for all its blocks, this many calls take step graphs.
constexpr int kHeldOffCalls = 64;
// Longer calls are several resident launches, so that other streams get the device in between.  A mesh
// that leaves room for others' wavefronts beside its own does not keep them waiting (a step of a 256^2
// mesh takes 0.33 ms beside 10^2 elements), and its launches are long ones; a step beside SW 64^2
// N = 7, which holds every register, waits for the launch to end: 62 ms with 4,096 steps, 6.7 with 512,
// which cost 0.6 % of the call.
constexpr int kResidentLaunchSteps = 4096, kResidentFullSteps = 512;

// Williamson low-storage RK3 (src/SELF_Model.f90:25-27)
constexpr double kRk3A[3] = {0.0, -5.0 / 9.0, -153.0 / 128.0};
constexpr double kRk3G[3] = {1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0};

struct Params {
  double g, fCori, gamma, Rgas;
  double auxConst, stat2Const;  // value of the static fields when no array is given
};

struct FusedArgs {
  double *S, *G, *dSdt;
  const double *traceIn;
  double *traceOut;
  // SW lagged velocity traces, read from the previous stage's buffer and written to the other
  // one for the next stage.  Affine mode: u.n of each face node, own side only, (0:N,4,nEl);
  // the outer side's value is the neighbour's own, negated (the two sides' normals are
  // opposite).  Nodal mode: the vector (u, v) of each face node, (2,0:N,4,nEl), and both normal
  // velocities are formed with this side's normal, as the reference does, because on curved
  // elements interpolated below the mesh degree the two sides' normals differ.
  const double *unIn;
  double *unOut;
  const double *aux;        // SW topography / LSW bathymetry / Euler potential, or null
  const double *stat2;      // LSW Coriolis / Euler drag, or null
  const double *presTrace;  // Euler prescribed traces (0:N,9,4,nEl), or null
  const double *geom;       // per-element records (affine mode)
  const double *ndsdx, *nJ, *nnHat, *nnScale;  // per-node metrics (nodal mode), SEMQuad shapes
  const int32_t *nbr;       // per (side, element) neighbour code
  const double *mats;       // dgM(P*P) D(P*P) bM(2P) qW(P) 1/qW(P)
  int nEl;
  double rkA, rkGdt;        // stage coefficients a_m and g_m*dt
  double rkG;               // g_m alone: batched runs take dt from their element records
  int perElemDt;            // 1: g_m * dt_e with dt_e in the element record (batched runs)
  int writeG;               // 0 at the last RK3 stage: the next step's first stage (a_1 = 0) never reads G
  int reverse;              // 1: blocks take the elements in reverse order (alternate stages)
  const int32_t *elems;     // the launch's elements (a band), or null: elements 0 .. nEl-1
  const double *corr;       // learned tendency correction (interior layout), or null
  // global mean of the mass-variable correction: shiftScale times the sum of nShift doubles (the
  // row tiles' mass integrals; every wavefront adds them in the same order)
  const double *corrShift;
  int nShift;
  double shiftScale;
  // MODE 1 only, or null: the contravariant flux (2,0:N,0:N,nVar,nEl) and its weak divergence
  // divided by J (0:N,0:N,nVar,nEl), the flux and fluxDivergence registers of
  // CalculateTendency_Model2D (src/SELF_Model2D.f90:816-859)
  double *fluxOut, *fluxDivOut;
  int anyBoundary;          // 1 when some element side is a physical boundary (neighbour code < 0)
  Params p;
};

// ------------------------------------------------------------------------------
// Physics policies
// ------------------------------------------------------------------------------

// Nonlinear shallow water (src/models/SELF_ShallowWater.f90): state (Hu, Hv, H), traces
// are the state traces, aux = topography (gradient in the source, trace in radiation BC).
struct PhysSW {
  static constexpr int kKind = SELFAMD_MODEL_SW;
  static constexpr int NV = 3, NT = 3;
  static constexpr bool kAuxGrad = true, kAuxTrace = true, kLag = true;
  static constexpr bool kAuxTraceInFlux = false;  // the topography trace enters the radiation BC only
  __device__ static void volume(const double *s, double, const Params &p, double *fx, double *fy, double *q) {
    const double Hu = s[0], Hv = s[1], H = s[2];
    const double invH = 1.0 / H;
    const double u = Hu * invH, v = Hv * invH;  // PreTendency velocity (src/models/SELF_ShallowWater.f90:206-218)
    fx[0] = u * Hu + 0.5 * p.g * H * H;
    fy[0] = v * Hu;
    fx[1] = u * Hv;
    fy[1] = v * Hv + 0.5 * p.g * H * H;
    fx[2] = Hu;
    fy[2] = Hv;
    q[0] = Hu; q[1] = Hv; q[2] = H;
  }
  __device__ static void nodal(const double *s, double *q) { q[0] = s[0]; q[1] = s[1]; q[2] = s[2]; }
  __device__ static void source(const double *s, double gx, double gy, double, const Params &p, double *src) {
    src[0] = -p.fCori * s[1] + p.g * s[2] * gx;
    src[1] = p.fCori * s[0] + p.g * s[2] * gy;
    src[2] = 0.0;
  }
  // SetBoundaryCondition_ShallowWater (src/models/SELF_ShallowWater.f90:284-343)
  __device__ static void bc(const double *qL, double auxB, double nx, double ny, int bcid, const double *, bool, double *qR) {
    if (bcid == SELFAMD_BC_NONORMALFLOW) {
      qR[0] = (ny * ny - nx * nx) * qL[0] - 2.0 * nx * ny * qL[1];
      qR[1] = (nx * nx - ny * ny) * qL[1] - 2.0 * nx * ny * qL[0];
      qR[2] = qL[2];
    } else {
      qR[0] = 0.0; qR[1] = 0.0; qR[2] = auxB;
    }
  }
  // RiemannSolver_ShallowWater (src/models/SELF_ShallowWater.f90:451-529); unL/unR are the
  // lagged normal velocities.
  __device__ static void riemann(const double *qL, const double *qR, double nx, double ny, double nmag, double,
                                 double unL, double unR, const Params &p, double *f) {
    const double g = p.g;
    const double HuL = qL[0], HvL = qL[1], HL = qL[2], HuR = qR[0], HvR = qR[1], HR = qR[2];
    const double cL = sqrt(g * HL), cR = sqrt(g * HR);
    const double fL0 = HuL * unL + g * HL * HL * 0.5 * nx, fL1 = HvL * unL + g * HL * HL * 0.5 * ny;
    const double fL2 = HuL * nx + HvL * ny;
    const double fR0 = HuR * unR + g * HR * HR * 0.5 * nx, fR1 = HvR * unR + g * HR * HR * 0.5 * ny;
    const double fR2 = HuR * nx + HvR * ny;
    const double a = fmax(fmax(fabs(unL + cL), fabs(unR + cR)), fmax(fabs(unL - cL), fabs(unR - cR)));
    f[0] = 0.5 * (fL0 + fR0 + a * (HuL - HuR)) * nmag;
    f[1] = 0.5 * (fL1 + fR1 + a * (HvL - HvR)) * nmag;
    f[2] = 0.5 * (fL2 + fR2 + a * (HL - HR)) * nmag;
  }
};

// Linear shallow water (src/models/SELF_LinearShallowWater.f90): state (u, v, eta),
// aux = bathymetry H (flux and trace for c), stat2 = Coriolis f (source).
struct PhysLSW {
  static constexpr int kKind = SELFAMD_MODEL_LSW;
  static constexpr int NV = 3, NT = 3;
  static constexpr bool kAuxGrad = false, kAuxTrace = true, kLag = false;
  static constexpr bool kAuxTraceInFlux = true;  // the Riemann flux takes c = sqrt(g H) of the bathymetry trace
  __device__ static void volume(const double *s, double H, const Params &p, double *fx, double *fy, double *q) {
    fx[0] = p.g * s[2]; fy[0] = 0.0;
    fx[1] = 0.0;        fy[1] = p.g * s[2];
    fx[2] = H * s[0];   fy[2] = H * s[1];
    q[0] = s[0]; q[1] = s[1]; q[2] = s[2];
  }
  __device__ static void nodal(const double *s, double *q) { q[0] = s[0]; q[1] = s[1]; q[2] = s[2]; }
  __device__ static void source(const double *s, double, double, double f, const Params &, double *src) {
    src[0] = f * s[1];
    src[1] = -f * s[0];
    src[2] = 0.0;
  }
  __device__ static void bc(const double *qL, double, double nx, double ny, int bcid, const double *, bool, double *qR) {
    if (bcid == SELFAMD_BC_NONORMALFLOW) {
      qR[0] = (ny * ny - nx * nx) * qL[0] - 2.0 * nx * ny * qL[1];
      qR[1] = (nx * nx - ny * ny) * qL[1] - 2.0 * nx * ny * qL[0];
      qR[2] = qL[2];
    } else {
      qR[0] = 0.0; qR[1] = 0.0; qR[2] = 0.0;
    }
  }
  // characteristic upwind flux (src/models/SELF_LinearShallowWater.f90:500-557)
  __device__ static void riemann(const double *qL, const double *qR, double nx, double ny, double nmag, double Hb,
                                 double, double, const Params &p, double *f) {
    const double g = p.g;
    const double c = sqrt(g * Hb);
    const double unL = qL[0] * nx + qL[1] * ny, unR = qR[0] * nx + qR[1] * ny;
    const double wL = 0.5 * (unL / g + qL[2] / c), wR = 0.5 * (unR / g - qR[2] / c);
    f[0] = g * c * (wL - wR) * nx * nmag;
    f[1] = g * c * (wL - wR) * ny * nmag;
    f[2] = c * c * (wL + wR) * nmag;
  }
};

// Compressible ideal gas (src/models/SELF_CompressibleIdealGas2D.f90): state
// (rho u, rho v, rho, rho E); traces: state(4), primitive u, v, p, enthalpy rho E + p,
// sound speed c (each interpolated from its nodal values, as PreTendency does);
// aux = gravity potential (gradient in the source), stat2 = drag coefficient.
struct PhysEuler {
  static constexpr int kKind = SELFAMD_MODEL_EULER;
  static constexpr int NV = 4, NT = 9;
  static constexpr bool kAuxGrad = true, kAuxTrace = false, kLag = false;
  static constexpr bool kAuxTraceInFlux = false;
  __device__ static void nodal_p(const double *s, const Params &p, double &u, double &v, double &pr, double &ke,
                                 double &invRho) {
    invRho = 1.0 / s[2];
    u = s[0] * invRho;
    v = s[1] * invRho;
    ke = 0.5 * (s[0] * u + s[1] * v);
    pr = (p.gamma - 1.0) * (s[3] - ke);
  }
  __device__ static void nodal_q(const double *s, const Params &p, double *q) {
    double u, v, pr, ke, invRho;
    nodal_p(s, p, u, v, pr, ke, invRho);
    q[0] = s[0]; q[1] = s[1]; q[2] = s[2]; q[3] = s[3];
    q[4] = u; q[5] = v; q[6] = pr;
    q[7] = s[3] + pr;                        // diagnostics(2): enthalpy
    q[8] = sqrt(p.gamma * pr * invRho);      // diagnostics(3): sound speed
  }
  __device__ static void volume(const double *s, double, const Params &p, double *fx, double *fy, double *q) {
    nodal_q(s, p, q);
    const double u = q[4], v = q[5], pr = q[6], Hn = q[7];
    fx[0] = u * s[0] + pr; fy[0] = v * s[0];
    fx[1] = u * s[1];      fy[1] = v * s[1] + pr;
    fx[2] = s[0];          fy[2] = s[1];
    fx[3] = u * Hn;        fy[3] = v * Hn;
  }
  __device__ static void source(const double *s, double gx, double gy, double Cd, const Params &, double *src) {
    src[0] = -s[2] * gx - Cd * s[0];
    src[1] = -s[2] * gy - Cd * s[1];
    src[2] = 0.0;
    src[3] = -s[0] * gx - s[0] * gy;  // quirk: energy source uses rho*u twice
  }
  // SetBoundaryCondition_CompressibleIdealGas2D (src/models/SELF_CompressibleIdealGas2D.f90:1217-1323)
  __device__ static void bc(const double *qL, double, double nx, double ny, int bcid, const double *pres, bool hasPres,
                            double *qR) {
    if (bcid == SELFAMD_BC_NONORMALFLOW) {
      qR[0] = (ny * ny - nx * nx) * qL[0] - 2.0 * nx * ny * qL[1];
      qR[1] = (nx * nx - ny * ny) * qL[1] - 2.0 * nx * ny * qL[0];
      qR[2] = qL[2]; qR[3] = qL[3];
      qR[4] = (ny * ny - nx * nx) * qL[4] - 2.0 * nx * ny * qL[5];
      qR[5] = (nx * nx - ny * ny) * qL[5] - 2.0 * nx * ny * qL[4];
      qR[6] = qL[6]; qR[7] = qL[7]; qR[8] = qL[8];
    } else if ((bcid == SELFAMD_BC_PRESCRIBED || bcid == SELFAMD_BC_RADIATION) && hasPres) {
      for (int k = 0; k < 9; k++) qR[k] = pres[k];
    } else {
      for (int k = 0; k < 9; k++) qR[k] = 0.0;
    }
  }
  // NaiveLLF (src/models/SELF_CompressibleIdealGas2D.f90:1455-1542)
  __device__ static void riemann(const double *qL, const double *qR, double nx, double ny, double nmag, double,
                                 double, double, const Params &, double *f) {
    const double unL = qL[4] * nx + qL[5] * ny, unR = qR[4] * nx + qR[5] * ny;
    const double fL0 = unL * qL[0] + qL[6] * nx, fL1 = unL * qL[1] + qL[6] * ny;
    const double fL2 = qL[0] * nx + qL[1] * ny, fL3 = unL * qL[7];
    const double fR0 = unR * qR[0] + qR[6] * nx, fR1 = unR * qR[1] + qR[6] * ny;
    const double fR2 = qR[0] * nx + qR[1] * ny, fR3 = unR * qR[7];
    const double a = fmax(fabs(unL), fabs(unR)) + fmax(fabs(qL[8]), fabs(qR[8]));
    f[0] = 0.5 * (fL0 + fR0 + a * (qL[0] - qR[0])) * nmag;
    f[1] = 0.5 * (fL1 + fR1 + a * (qL[1] - qR[1])) * nmag;
    f[2] = 0.5 * (fL2 + fR2 + a * (qL[2] - qR[2])) * nmag;
    f[3] = 0.5 * (fL3 + fR3 + a * (qL[3] - qR[3])) * nmag;
  }
  __device__ static void nodal(const double *s, double *q) {}  // unused: nodal_q needs params
};

template <class Phys>
__device__ inline void phys_nodal(const double *s, const Params &p, double *q) {
  if constexpr (Phys::NT == 9) PhysEuler::nodal_q(s, p, q);
  else Phys::nodal(s, q);
}

// Sum of x over the lane pair l, l ^ 32 of a wavefront, returned to both lanes.  The
// exchange is v_permlane32_swap (gfx950), a VALU operation: it does not use the LDS pipe that
// a shuffle through ds_bpermute would occupy.  Both lanes get the same sum x_l + x_(l+32).
// Lagged SW normal velocities (the layouts are described with FusedArgs::unIn): the own side's
// and the outer side's u.n at face-node slot fb (the neighbour's slot for the outer side).
template <bool NODAL>
__device__ inline double lag_own(const double *un, size_t fb, double nx, double ny) {
  if constexpr (NODAL) return un[2 * fb] * nx + un[2 * fb + 1] * ny;
  return un[fb];
}
// The outer side's value is formed in two steps: lag_outer_raw at the load (affine: the stored
// value as it is, so that no arithmetic waits for the load there) and outer_un where it is used.
template <bool NODAL>
__device__ inline double lag_outer_raw(const double *un, size_t fbNeighbour, double nx, double ny) {
  if constexpr (NODAL) return un[2 * fbNeighbour] * nx + un[2 * fbNeighbour + 1] * ny;
  return un[fbNeighbour];
}
template <bool NODAL>
__device__ inline double outer_un(double raw) {
  if constexpr (NODAL) return raw;
  return -raw;
}

// Ordering point between kernel phases.  When every element's node lanes and face lanes lie in
// one wavefront (WAVE), a phase only reads LDS values its own wavefront wrote, and a wavefront's
// LDS accesses execute in program order: a code-motion barrier suffices.  A workgroup barrier
// would also make each wavefront wait for its outstanding global stores (the workgroup-scope
// release) and for the block's slowest wavefront.
template <bool WAVE>
__device__ inline void phase_sync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

__device__ inline double pair_sum32(double x) {
  const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  // a[0], b[0]: the value of lane l mod 32; a[1], b[1]: the value of lane l mod 32 + 32
  return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
}

// Sums of x over 16, 32 or all 64 lanes, in every lane of them, by VALU lane exchanges: lanes l ^ 32,
// l ^ 16, then rotations by 8, 4, 2 and 1 within each row of 16 lanes, which exchange what xors
// would (the partial sums repeat with that period).
__device__ inline double row_sum16(double x) {
  auto rotate = [](double v, auto n) {  // DPP row_ror:n
    constexpr int ctrl = 0x120 + decltype(n)::value;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
  };
  x += rotate(x, std::integral_constant<int, 8>{});
  x += rotate(x, std::integral_constant<int, 4>{});
  x += rotate(x, std::integral_constant<int, 2>{});
  x += rotate(x, std::integral_constant<int, 1>{});
  return x;
}
__device__ inline double half_sum32(double x) {
  const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return row_sum16(__hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]));
}
__device__ inline double wave_sum(double x) { return half_sum32(pair_sum32(x)); }

// ------------------------------------------------------------------------------
// The fused kernel
// ------------------------------------------------------------------------------
// MODE 0: RK stage (update S, G, write next traces); MODE 1: tendency only (write dSdt).
// NODAL: metric terms per node and per face node exactly as SEMQuad stores them (curved
// elements, and the reference's own per-node metric values); otherwise one affine record
// per element.  THREADS: block size (the tile shape); EPB = THREADS/(N+1)^2 elements per
// block.  With THREADS = 64 at N = 7 a block is one wavefront owning one element, so its
// barriers never wait on other waves.
//
// Every global load the stage needs is issued before any arithmetic: the element's state,
// RK register and static field on the node lanes, and (on the face lanes) the neighbour
// code, the neighbour's traces and the lagged normal velocities.  The gather of neighbour
// traces is the only dependent load and it overlaps the volume-flux work.
//
// Tile parameters: THREADS work-items per block (THREADS / (N+1)^2 elements), WPE the
// occupancy the register allocator must allow (waves per SIMD; 1 = unconstrained), XCD an
// element order in which the blocks one XCD receives cover a contiguous run of elements.
// With a.reverse the elements are visited last to first: successive stages alternate
// direction, so a stage starts on the elements whose data the previous stage touched last.
//
// LDS of one tile (block) of the stage kernel, in doubles: the node arrays sQ, sF1, sF2, the
// static field sAux, the nodal-mode metric products sGb, the face fluxes sBF and the matrices
// sM, each starting on a 16-byte boundary.
template <class Phys, int N, bool NODAL, int THREADS>
struct TileLds {
  static constexpr int NP = N + 1, NN = NP * NP, EPB = THREADS / NN, NF = 4 * NP;
  static constexpr int NV = Phys::NV, NT = Phys::NT;
  static constexpr bool USE_AUX = Phys::kAuxGrad || Phys::kAuxTrace;
  static constexpr bool GRADN = NODAL && Phys::kAuxGrad;
  // At N = 5 two pad doubles per element array (38 instead of 36) shift the elements of a
  // tile against each other in the banks: 70.0 against 71.1 us per SW launch at 256^2 (row
  // strides of 7 were slower, 72.3-72.7 us).  Matrices hold entry (c, r) at c + MRS r, with two
  // pad doubles per 8-double row (they are written once per tile).
  static constexpr int MRS = NP % 8 == 0 ? NP + 2 : NP, NNS = NP == 6 ? NN + 2 : NN;
  static constexpr int even(int n) { return (n + 1) & ~1; }
  static constexpr int Q = 0;
  static constexpr int F1 = Q + even(NT * EPB * NNS);
  static constexpr int F2 = F1 + even(NV * EPB * NNS);
  static constexpr int AUX = F2 + even(NV * EPB * NNS);
  static constexpr int GB = AUX + even(USE_AUX ? EPB * NNS : 1);
  static constexpr int BF = GB + even(GRADN ? 4 * EPB * NNS : 1);
  static constexpr int M = BF + even(NV * EPB * NF);
  static constexpr int SIZE = M + even(2 * NP * MRS + 4 * NP);
  // face-lane arrangement (see the stage kernel): every face node has its own lane; two lanes per
  // face node; N = 5 face lanes padded to 32 per element; every element's node and face lanes in
  // one wavefront
  static constexpr bool ONE_FACE_PASS = EPB * NF <= THREADS;
  static constexpr bool SPLIT = ONE_FACE_PASS && 2 * EPB * NF <= THREADS && NF <= 32;
  static constexpr bool FPAD = !SPLIT && NF == 24 && 32 * EPB <= THREADS;
  static constexpr bool WAVE = (NN == 64 && SPLIT) || (NN == 16 && NF == 16 && ONE_FACE_PASS && !SPLIT && !FPAD);
};

// The tile's interpolation and derivative matrices and quadrature weights into its LDS (dgM, D
// in rows of MRS, bM(2P), qW, 1/qW), from mats = [dgM, D, bM, qW, 1/qW] as SetupMatrices stores
// them.  Every work-item of the block takes part.
template <class Phys, int N, bool NODAL, int THREADS>
__device__ __forceinline__ int tile_matrix_slot(int k) {
  constexpr int NP = N + 1, NN = NP * NP, MRS = TileLds<Phys, N, NODAL, THREADS>::MRS;
  const int r = k % NN;
  return k < 2 * NN ? (k / NN) * NP * MRS + (r / NP) * MRS + r % NP : 2 * NP * MRS + k - 2 * NN;
}
template <class Phys, int N, bool NODAL, int THREADS>
__device__ __forceinline__ void load_tile_matrices(const double *mats, double *lds, int tid) {
  double *sM = lds + TileLds<Phys, N, NODAL, THREADS>::M;
  for (int k = tid; k < 2 * (N + 1) * (N + 1) + 4 * (N + 1); k += THREADS)
    sM[tile_matrix_slot<Phys, N, NODAL, THREADS>(k)] = mats[k];
}

// One tile of the stage kernel: tile blk of the launch's element list (after any reordering),
// with the tile's LDS at lds, run by work-item tid of the block.  The __global__ wrappers
// below map blocks to tiles.  PRELOADED: the block has already put the matrices into the LDS
// (load_tile_matrices) and made them visible, so the tile neither loads them nor needs a block
// barrier where the element's own wavefront suffices.
template <class Phys, int N, int MODE, bool NODAL, int THREADS, bool PRELOADED = false>
__device__ __forceinline__ void fused_tile(const FusedArgs &a, int blk, double *lds, const int tid) {
  using L = TileLds<Phys, N, NODAL, THREADS>;
  constexpr int NP = N + 1, NN = NP * NP, EPB = THREADS / NN, NF = 4 * NP;
  constexpr int NV = Phys::NV, NT = Phys::NT;
  constexpr bool USE_AUX = Phys::kAuxGrad || Phys::kAuxTrace;
  constexpr bool ONE_FACE_PASS = L::ONE_FACE_PASS;  // every face node has its own lane
  // two lanes per face node (lanes l and l ^ 32 of a wavefront): each interpolates half of
  // the face line, the halves are summed across the pair
  constexpr bool SPLIT = L::SPLIT;
  static_assert(EPB >= 1, "block too small for one element");
  // LDS layouts.  Node arrays hold node (i, j) at slot(i, j).  With 8 x 8 nodes a row is 64
  // bytes, and a column access (fixed i, one row per lane group) would find rows 0, 2, 4, 6 in
  // the same banks; permuting the columns of row j by i ^ (j & 6) spreads them over the banks,
  // keeps the pairs (2m, 2m + 1) adjacent for 16-byte reads and keeps every row in place, so
  // row-wise writes stay conflict-free.
  constexpr bool SWZ = NP == 8;
  constexpr int MRS = L::MRS, NNS = L::NNS;
  auto slot = [](int i_, int j_) { return SWZ ? NP * j_ + (i_ ^ (j_ & 6)) : i_ + NP * j_; };
  auto sQ = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::Q);
  auto sF1 = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::F1);
  auto sF2 = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::F2);
  auto sAux = reinterpret_cast<double (*)[USE_AUX ? NNS : 1]>(lds + L::AUX);
  // nodal mode: static field times the node's contravariant metric, for GradientSF
  constexpr bool GRADN = L::GRADN;
  auto sGb = reinterpret_cast<double (*)[GRADN ? EPB : 1][GRADN ? NNS : 1]>(lds + L::GB);
  auto sBF = reinterpret_cast<double (*)[EPB][NF]>(lds + L::BF);
  double *sM = lds + L::M;  // dgM, D (rows of MRS), bM(2P), qW, 1/qW

  const int el = tid / NN, node = tid % NN;
  const int i = node % NP, j = node / NP;
  const int nl = slot(i, j);  // the node's LDS slot
  const int pe = blk * EPB + el;  // position in the launch's element list
  bool nodeActive = el < EPB && pe < a.nEl;
  int e = a.elems ? (nodeActive ? a.elems[pe] : 0) : pe;
  // one element per wavefront: its index, whether it is active, and every address and record
  // value derived from it are uniform, so they live in scalar registers and the branches on
  // them are scalar
  if constexpr (NN == 64) {
    e = __builtin_amdgcn_readfirstlane(e);
    nodeActive = __builtin_amdgcn_readfirstlane((int)nodeActive) != 0;
  }
  // ---- face lanes ----
  // SPLIT: wavefront w covers the face nodes of element w (NF <= 32 slots), lanes l and l + 32
  // share face node l; otherwise face node = thread index
  // FPAD (N = 5, tiles of 128 or 256): each element's 24 face nodes take 32 lanes, south and
  // north faces in lanes 0-11 and east and west in lanes 16-27 of the group, so that a 16-lane
  // LDS group reads either columns or rows of the element, never both (no bank conflicts)
  constexpr bool FPAD = L::FPAD;
  const int fhalf = SPLIT ? (tid >> 5) & 1 : 0;
  const int fslot = SPLIT ? (tid & 31) : FPAD ? (tid & 15) : 0;
  const int fidx = SPLIT ? (tid >> 6) * NF + fslot : FPAD ? (tid >> 5) * NF + (fslot % 12) : tid;
  const int fel = fidx / NF, fslotN = fidx % NF;
  // SPLIT: slots take the sides in the order south, north, east, west, so that the lanes of a
  // 16-lane LDS group read opposite faces, whose face lines are the same nodes (no bank
  // conflicts between them)
  const int side = SPLIT  ? ((fslotN / NP) >> 1 | ((fslotN / NP) & 1) << 1)
                   : FPAD ? ((tid >> 4) & 1) + (fslot >= NP ? 2 : 0)
                          : fslotN / NP;
  const int fi = fslotN % NP, fnode = side * NP + fi;
  // element-to-wavefront locality of the node and face lanes (see phase_sync): at N = 7 a
  // wavefront owns one element (face lanes split in pairs); at N = 3 an element's 16 nodes and 16
  // face nodes share the same 16 lanes
  constexpr bool WAVE = L::WAVE;
  const int pf = blk * EPB + fel;
  const bool faceActive = ONE_FACE_PASS && (!SPLIT || fslot < NF) && (!FPAD || fslot < 2 * NP) && fel < EPB &&
                          pf < a.nEl;
  // one element per wavefront (N = 7, face lanes split in pairs): the face lanes' element is the
  // node lanes' one, already in a scalar register
  int fe;
  if constexpr (SPLIT && NF == 32 && NN == 64) fe = e;
  else fe = a.elems ? (faceActive ? a.elems[pf] : 0) : pf;
  // SPLIT: LDS slots of the half face line this lane interpolates (phases 1 and 3).  South and
  // north faces run along j through column fi, east and west along i through row fi.
  constexpr int FH0 = NP / 2, FHN = NP - FH0;
  int foff[SPLIT ? FHN : 1];
  if constexpr (SPLIT) {
    const bool alongJ = (side == 0 || side == 2);
    const int lo = fhalf ? FH0 : 0;
#pragma unroll
    for (int t = 0; t < FHN; t++) foff[t] = alongJ ? slot(fi, lo + t) : slot(lo + t, fi);
  }
  // ---- loads ----
  // The vector-memory counter completes in issue order, and a wait after a branch must cover
  // every path into it.  So every load is issued before any of them is waited for: the
  // neighbour codes (first, since the trace loads depend on them), the matrices (unless
  // preloaded), the node lanes' streams (on every path: inactive lanes and absent fields read
  // element 0 or the state, and the values are discarded), then the loads addressed through
  // the codes, which wait for the codes alone; the matrices go to LDS last.
  // one element per wavefront (N = 7, face lanes split in pairs): the element's four codes are
  // one scalar load further down; otherwise each face lane's code is the first vector load
  constexpr bool SCALAR_CODES = SPLIT && NF == 32 && NN == 64;
  int code = 0;
  if constexpr (!SCALAR_CODES) {
    const bool own = faceActive && fhalf == 0;
    const int c = a.nbr[4 * (size_t)(own ? fe : 0) + side];
    code = own ? c : 0;
  }
  constexpr int MCNT = 2 * NN + 4 * NP, MPL = PRELOADED ? 1 : (MCNT + THREADS - 1) / THREADS;
  double mreg[MPL];
  if constexpr (!PRELOADED) {
#pragma unroll
    for (int q = 0; q < MPL; q++) mreg[q] = a.mats[min(tid + q * THREADS, MCNT - 1)];
  }
  const size_t sBase = (size_t)e * NV * NN;  // S(0,0,0,e)
  const size_t nodeAt = nodeActive ? (size_t)e * NN + node : (size_t)node;  // inactive: element 0
  double s[NV], gReg[NV];
  double auxVal = a.p.auxConst, statVal = a.p.stat2Const;
  double dsdx[4] = {0, 0, 0, 0}, invJ = 1.0;
  {
    const size_t sAt = nodeActive ? sBase + node : (size_t)node;
    // state and RK register: non-temporal loads.  This stage overwrites both, so caching the
    // lines read here buys nothing; measured 5 % faster per launch than cached loads at N = 7
    // (non-temporal loads of the static field or of the neighbour traces, which later stages
    // or neighbours reuse, were slower).
#pragma unroll
    for (int v = 0; v < NV; v++) s[v] = __builtin_nontemporal_load(&a.S[sAt + (size_t)v * NN]);
    if constexpr (MODE == 0) {
      // the first stage (rkA = 0) reads element 0's, a few cached lines, and discards them
      const bool useG = a.rkA != 0.0;
      const size_t gAt = useG ? sAt : (size_t)node;
      double gl[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) gl[v] = __builtin_nontemporal_load(&a.G[gAt + (size_t)v * NN]);
#pragma unroll
      for (int v = 0; v < NV; v++) gReg[v] = useG ? gl[v] : 0.0;
    } else {
#pragma unroll
      for (int v = 0; v < NV; v++) gReg[v] = 0.0;
    }
    if constexpr (USE_AUX) {
      const double av = a.aux ? a.aux[nodeAt] : a.S[node];
      if (a.aux) auxVal = av;
    }
    const double sv = a.stat2 ? a.stat2[nodeAt] : a.S[node];
    if (a.stat2) statVal = sv;
    if constexpr (NODAL) {
      const double *gn = a.ndsdx + 4 * nodeAt;
      dsdx[0] = gn[0]; dsdx[1] = gn[1]; dsdx[2] = gn[2]; dsdx[3] = gn[3];
      invJ = 1.0 / a.nJ[nodeAt];
    } else {
      const double *gr = a.geom + (nodeActive ? (size_t)e : 0) * kGeomStride;
      dsdx[0] = gr[0]; dsdx[1] = gr[1]; dsdx[2] = gr[2]; dsdx[3] = gr[3];
      invJ = gr[6];  // 1/J, precomputed in the element record
    }
  }
  if constexpr (SCALAR_CODES) {
    // (a wavefront past the last element of a ragged last tile reads element 0's codes; the
    // wavefront's node and face lanes are the same element, so nodeActive, a scalar, decides)
    const int4 c4 = *reinterpret_cast<const int4 *>(a.nbr + 4 * (size_t)(nodeActive ? fe : 0));
    // all four in scalar registers at once (one load, one wait), then a per-lane select
    const int cx = __builtin_amdgcn_readfirstlane(c4.x), cy = __builtin_amdgcn_readfirstlane(c4.y);
    const int cz = __builtin_amdgcn_readfirstlane(c4.z), cw = __builtin_amdgcn_readfirstlane(c4.w);
    code = (side & 2) ? ((side & 1) ? cw : cz) : ((side & 1) ? cy : cx);
    if (!(faceActive && fhalf == 0)) code = 0;
  }

  double qR[NT], unL = 0.0, unR = 0.0, nx = 0.0, ny = 0.0, nmag = 0.0;
  if (faceActive && fhalf == 0) {
    // normals: first in nodal mode, where the lagged normal velocities need them; after the
    // neighbour loads in affine mode (measured slightly faster there)
    if constexpr (NODAL) {
      const size_t fb = (size_t)fi + NP * (side + 4 * (size_t)fe);
      nx = a.nnHat[2 * fb]; ny = a.nnHat[2 * fb + 1]; nmag = a.nnScale[fb];
    }
    if (code >= 0) {
      const int flip = code & 1, s2 = (code >> 1) & 3;
      const size_t e2 = (size_t)(code >> 3);
      const size_t nb = (size_t)(flip ? N - fi : fi) + NP * (s2 + 4 * e2);
      const double *tr = a.traceIn + (size_t)(flip ? N - fi : fi) + NP * (size_t)NT * (s2 + 4 * e2);
#pragma unroll
      for (int k = 0; k < NT; k++) qR[k] = tr[(size_t)k * NP];
      if (Phys::kLag) unR = lag_outer_raw<NODAL>(a.unIn, nb, nx, ny);
    }
    if (Phys::kLag) unL = lag_own<NODAL>(a.unIn, (size_t)fi + NP * (side + 4 * (size_t)fe), nx, ny);
    if constexpr (!NODAL) {
      const double *gr = a.geom + (size_t)fe * kGeomStride;
      nx = gr[8 + side]; ny = gr[12 + side]; nmag = gr[16 + side];
    }
  }

  // the matrices into LDS once every load is in flight
  if constexpr (!PRELOADED) {
#pragma unroll
    for (int q = 0; q < MPL; q++) {
      const int k = tid + q * THREADS;
      if (k < MCNT) sM[tile_matrix_slot<Phys, N, NODAL, THREADS>(k)] = mreg[q];
    }
  }
  // the closure's mean mass correction, in scalar registers: the loads overlap those above, and a
  // wavefront's sum of 256 doubles (64 x 64 elements) replaces a launch of one block between the
  // network and the stage: 4.5 us, against 0.5 us more here (6.2 against 5.7 us per launch)
  double shift = 0.0;
  const bool corrected = !PRELOADED && a.corr;  // batches, which preload, have no closure
  if (corrected) {
    double part = 0.0;
    for (int k = tid & 63; k < a.nShift; k += 256) {
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = a.corrShift[min(k + 64 * q, a.nShift - 1)];
#pragma unroll
      for (int q = 0; q < 4; q++) part += k + 64 * q < a.nShift ? v[q] : 0.0;
    }
    part = wave_sum(part);
    part *= a.shiftScale;
    shift = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(part)),
                             __builtin_amdgcn_readfirstlane(__double2loint(part)));
  }
  const double *dgM = sM, *Dm = sM + NP * MRS, *bM0 = sM + 2 * NP * MRS, *bM1 = bM0 + NP, *qW = bM1 + NP;

  // ---- phase 0: volume fluxes, nodal trace quantities ----
  if (nodeActive) {
    double fx[NV], fy[NV], q[NT];
    Phys::volume(s, auxVal, a.p, fx, fy, q);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      // ContravariantProjection (src/SELF_MappedData.f90:2220-2269)
      sF1[v][el][nl] = dsdx[0] * fx[v] + dsdx[1] * fy[v];
      sF2[v][el][nl] = dsdx[2] * fx[v] + dsdx[3] * fy[v];
      if (MODE == 1 && a.fluxOut) {
        double *fo = a.fluxOut + 2 * (sBase + (size_t)v * NN + node);
        fo[0] = sF1[v][el][nl];
        fo[1] = sF2[v][el][nl];
      }
    }
#pragma unroll
    for (int k = 0; k < NT; k++) sQ[k][el][nl] = q[k];
    if (USE_AUX) sAux[el][nl] = auxVal;
    if constexpr (GRADN) {
#pragma unroll
      for (int k = 0; k < 4; k++) sGb[k][el][nl] = auxVal * dsdx[k];
    }
  }
  // the matrices (written by the whole block) and the element's node values
  if constexpr (PRELOADED) phase_sync<WAVE>();
  else __syncthreads();

  // ---- phase 1: faces ----
  auto face = [&](int fel_, int side_, int fi_, int fe_, int fnode_, int code_, double *qR_, double unL_, double unR_,
                  double nx_, double ny_, double nmag_) {
    // own traces, ScalarBoundaryInterp_2D order (src/SELF_Lagrange.f90:2241-2270)
    const double *bm = (side_ == 1 || side_ == 2) ? bM1 : bM0;
    // nodes of the face line: column i = fi for south / north, row j = fi for east / west
    const bool alongJ = (side_ == 0 || side_ == 2);
    double qL[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) qL[k] = 0.0;
    // a static field's trace that enters only boundary conditions (SW topography) is skipped on
    // meshes without boundary sides (the condition is uniform over the launch, so the lane pairs
    // of SPLIT stay together)
    const bool auxTrace = Phys::kAuxTrace && a.aux && (Phys::kAuxTraceInFlux || a.anyBoundary);
    double auxB = a.p.auxConst;
    if (auxTrace) auxB = 0.0;
    if constexpr (SPLIT) {
      const int lo = fhalf ? FH0 : 0;
#pragma unroll
      for (int t = 0; t < FHN; t++) {
        const int ii = lo + t;
        if (fhalf == 0 && t >= FH0) break;
        const int nd = foff[t];
#pragma unroll
        for (int k = 0; k < NT; k++) qL[k] += bm[ii] * sQ[k][fel_][nd];
        if (auxTrace) auxB += bm[ii] * sAux[fel_][nd];
      }
#pragma unroll
      for (int k = 0; k < NT; k++) qL[k] = pair_sum32(qL[k]);
      if (auxTrace) auxB = pair_sum32(auxB);
      if (fhalf) return;  // the pair's first lane does the boundary and Riemann work
    } else {
#pragma unroll
      for (int ii = 0; ii < NP; ii++) {
        const int nd = alongJ ? slot(fi_, ii) : slot(ii, fi_);
#pragma unroll
        for (int k = 0; k < NT; k++) qL[k] += bm[ii] * sQ[k][fel_][nd];
        if (auxTrace) auxB += bm[ii] * sAux[fel_][nd];
      }
    }
    const bool interior = code_ >= 0;
    if (!interior) {
      if (code_ == kNbrOrphan) {
#pragma unroll
        for (int k = 0; k < NT; k++) qR_[k] = 0.0;
      } else {
        const double *pres =
            a.presTrace ? a.presTrace + (size_t)fi_ + NP * (size_t)NT * (side_ + 4 * (size_t)fe_) : nullptr;
        // the prescribed values go by value with a flag (a pointer that may be null would keep
        // the array in scratch memory)
        double pv[NT];
#pragma unroll
        for (int k = 0; k < NT; k++) pv[k] = pres ? pres[(size_t)k * NP] : 0.0;
        Phys::bc(qL, auxB, nx_, ny_, -code_ - 1, pv, pres != nullptr, qR_);
      }
    }
    if (Phys::kLag) {
      // velocity traces lag one stage (src/models/SELF_ShallowWater.f90:222-237): the stored
      // velocities are used now and this stage's are stored for the next one
      const double invH = 1.0 / qL[2];
      const size_t fb = (size_t)fi_ + NP * (side_ + 4 * (size_t)fe_);
      if constexpr (NODAL) {
        a.unOut[2 * fb] = qL[0] * invH;
        a.unOut[2 * fb + 1] = qL[1] * invH;
      } else {
        a.unOut[fb] = (qL[0] * invH) * nx_ + (qL[1] * invH) * ny_;
      }
    }
    double fstar[NV];
    Phys::riemann(qL, qR_, nx_, ny_, nmag_, auxB, unL_, outer_un<NODAL>(unR_), a.p, fstar);
#pragma unroll
    for (int v = 0; v < NV; v++) sBF[v][fel_][fnode_] = fstar[v];
  };
  if constexpr (ONE_FACE_PASS) {
    if (faceActive) face(fel, side, fi, fe, fnode, code, qR, unL, unR, nx, ny, nmag);
  } else {
    // N = 1, 2: more face nodes than lanes; load and compute face by face
    for (int ft = tid; ft < EPB * NF; ft += THREADS) {
      const int fel2 = ft / NF, fnode2 = ft % NF, side2 = fnode2 / NP, fi2 = fnode2 % NP;
      const int pf2 = blk * EPB + fel2;
      if (pf2 >= a.nEl) continue;
      const int fe2 = a.elems ? a.elems[pf2] : pf2;
      double qR2[NT], unL2 = 0.0, unR2 = 0.0, nx2, ny2, nmag2;
      const int code2 = a.nbr[4 * (size_t)fe2 + side2];
      if constexpr (NODAL) {
        const size_t fb = (size_t)fi2 + NP * (side2 + 4 * (size_t)fe2);
        nx2 = a.nnHat[2 * fb]; ny2 = a.nnHat[2 * fb + 1]; nmag2 = a.nnScale[fb];
      } else {
        const double *gr = a.geom + (size_t)fe2 * kGeomStride;
        nx2 = gr[8 + side2]; ny2 = gr[12 + side2]; nmag2 = gr[16 + side2];
      }
      if (code2 >= 0) {
        const int flip = code2 & 1, s2 = (code2 >> 1) & 3;
        const size_t e2 = (size_t)(code2 >> 3);
        const double *tr = a.traceIn + (size_t)(flip ? N - fi2 : fi2) + NP * (size_t)NT * (s2 + 4 * e2);
        for (int k = 0; k < NT; k++) qR2[k] = tr[(size_t)k * NP];
        if (Phys::kLag) unR2 = lag_outer_raw<NODAL>(a.unIn, (size_t)(flip ? N - fi2 : fi2) + NP * (s2 + 4 * e2), nx2, ny2);
      }
      if (Phys::kLag) unL2 = lag_own<NODAL>(a.unIn, (size_t)fi2 + NP * (side2 + 4 * (size_t)fe2), nx2, ny2);
      face(fel2, side2, fi2, fe2, fnode2, code2, qR2, unL2, unR2, nx2, ny2, nmag2);
    }
  }
  phase_sync<WAVE>();

  // ---- phase 2: divergence, source, update ----
  if (nodeActive) {
    // One pass over the line index ii for every sum of the phase: the volume terms of the weak
    // divergence of each variable (VectorDGDivergence_2D, src/SELF_Lagrange.f90:1589-1625; xi
    // and eta sums in separate FMA chains) and GradientSF of the static field
    // (src/SELF_MappedData.f90:1080-1149).  Each matrix entry is read from LDS once for all
    // variables; every sum keeps its own accumulation order.
    constexpr bool GRAD = Phys::kAuxGrad;
    const bool grad = GRAD && a.aux;
    double dxs[NV], des[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) { dxs[v] = 0.0; des[v] = 0.0; }
    double gx = 0.0, gy = 0.0, dxi = 0.0, deta = 0.0;
    // one step of the sums at line index ii: matrix entries and row-wise (xi) operands come in
    // as pairs (ii, ii + 1) when NP is even (16-byte LDS reads: the pairs are adjacent and
    // aligned in every node and matrix layout); the loop is not unrolled further, so the
    // compiler does not hoist every LDS read of the phase (that took 192 VGPRs)
    auto line = [&](int ii, double ai, double aj, const double *f1, double di, double dj, double bx) {
#pragma unroll
      for (int v = 0; v < NV; v++) {
        dxs[v] = dxs[v] + ai * f1[v];
        des[v] = des[v] + aj * sF2[v][el][slot(i, ii)];
      }
      if (GRAD && grad) {
        if constexpr (GRADN) {
          gx = gx + di * sGb[0][el][slot(ii, j)] + dj * sGb[2][el][slot(i, ii)];
          gy = gy + di * sGb[1][el][slot(ii, j)] + dj * sGb[3][el][slot(i, ii)];
        } else {
          dxi = dxi + di * bx;
          deta = deta + dj * sAux[el][slot(i, ii)];
        }
      }
    };
    if constexpr (NP % 2 == 0) {
#pragma unroll 1
      for (int ii = 0; ii < NP; ii += 2) {
        const double2 ai = *reinterpret_cast<const double2 *>(&dgM[ii + MRS * i]);
        const double2 aj = *reinterpret_cast<const double2 *>(&dgM[ii + MRS * j]);
        double2 di = {0.0, 0.0}, dj = {0.0, 0.0}, bx = {0.0, 0.0};
        if (GRAD && grad) {
          di = *reinterpret_cast<const double2 *>(&Dm[ii + MRS * i]);
          dj = *reinterpret_cast<const double2 *>(&Dm[ii + MRS * j]);
          if constexpr (!GRADN) bx = *reinterpret_cast<const double2 *>(&sAux[el][slot(ii, j)]);
        }
        double f1a[NV], f1b[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          const double2 f = *reinterpret_cast<const double2 *>(&sF1[v][el][slot(ii, j)]);
          f1a[v] = f.x;
          f1b[v] = f.y;
        }
        line(ii, ai.x, aj.x, f1a, di.x, dj.x, bx.x);
        line(ii + 1, ai.y, aj.y, f1b, di.y, dj.y, bx.y);
      }
    } else {
#pragma unroll 2
      for (int ii = 0; ii < NP; ii++) {
        double f1[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) f1[v] = sF1[v][el][slot(ii, j)];
        line(ii, dgM[ii + MRS * i], dgM[ii + MRS * j], f1, Dm[ii + MRS * i], Dm[ii + MRS * j],
             USE_AUX ? sAux[el][slot(ii, j)] : 0.0);
      }
    }
    if (GRAD && grad) {
      if constexpr (!GRADN) {
        // affine element: the metric terms are constant, so they factor out of the sums
        gx = dsdx[0] * dxi + dsdx[2] * deta;
        gy = dsdx[1] * dxi + dsdx[3] * deta;
      }
      gx = gx * invJ;
      gy = gy * invJ;
    }
    double src[NV];
    Phys::source(s, gx, gy, statVal, a.p, src);
    // per-run step size of a batched launch: the same IEEE product g_m*dt as a single run
    const double gdt = (MODE == 0 && a.perElemDt) ? a.rkG * a.geom[(size_t)e * kGeomStride + 5] : a.rkGdt;
    const double iwi = qW[NP + i], iwj = qW[NP + j];  // 1/w_i, 1/w_j
    const double bi1 = bM1[i], bi0 = bM0[i], bj1 = bM1[j], bj0 = bM0[j];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      // surface terms of the weak divergence, then JacobianWeight
      double d = dxs[v] + des[v];
      d = d + (bi1 * sBF[v][el][NP + j] + bi0 * sBF[v][el][3 * NP + j]) * iwi +
          (bj1 * sBF[v][el][2 * NP + i] + bj0 * sBF[v][el][i]) * iwj;
      d = d * invJ;
      if (MODE == 1 && a.fluxDivOut) a.fluxDivOut[sBase + (size_t)v * NN + node] = d;
      double dsdt = src[v] - d;
      if (corrected) {
        // closure: mass correction made mean-free over the mesh (variable 2 is H / eta / rho)
        double c = a.corr[sBase + (size_t)v * NN + node];
        if (v == 2) c -= shift;
        dsdt += c;
      }
      if (MODE == 1) {
        a.dSdt[sBase + (size_t)v * NN + node] = dsdt;
      } else {
        const double gn = a.rkA * gReg[v] + dsdt;
        s[v] = s[v] + gdt * gn;
        if (a.writeG) a.G[sBase + (size_t)v * NN + node] = gn;
        a.S[sBase + (size_t)v * NN + node] = s[v];
      }
    }
    if (MODE == 0) {
      double q[NT];
      phys_nodal<Phys>(s, a.p, q);
#pragma unroll
      for (int k = 0; k < NT; k++) sQ[k][el][nl] = q[k];
    }
  }
  if (MODE == 1) return;
  phase_sync<WAVE>();

  // ---- phase 3: traces of the updated state ----
  if constexpr (SPLIT) {
    if (faceActive) {
      const double *bm = (side == 1 || side == 2) ? bM1 : bM0;
      const int lo = fhalf ? FH0 : 0;
      double qn[NT];
#pragma unroll
      for (int k = 0; k < NT; k++) qn[k] = 0.0;
#pragma unroll
      for (int t = 0; t < FHN; t++) {
        const int ii = lo + t;
        if (fhalf == 0 && t >= FH0) break;
        const int nd = foff[t];
#pragma unroll
        for (int k = 0; k < NT; k++) qn[k] += bm[ii] * sQ[k][fel][nd];
      }
#pragma unroll
      for (int k = 0; k < NT; k++) qn[k] = pair_sum32(qn[k]);
      if (fhalf == 0) {
        double *tr = a.traceOut + (size_t)fi + NP * (size_t)NT * (side + 4 * (size_t)fe);
#pragma unroll
        for (int k = 0; k < NT; k++) tr[(size_t)k * NP] = qn[k];
      }
    }
    return;
  }
  if constexpr (FPAD) {
    // the face lanes of phase 1, in their padded order
    if (faceActive) {
      const double *bm = (side == 1 || side == 2) ? bM1 : bM0;
      const bool alongJ = (side == 0 || side == 2);
      double qn[NT];
#pragma unroll
      for (int k = 0; k < NT; k++) qn[k] = 0.0;
#pragma unroll
      for (int ii = 0; ii < NP; ii++) {
        const int nd = alongJ ? slot(fi, ii) : slot(ii, fi);
#pragma unroll
        for (int k = 0; k < NT; k++) qn[k] += bm[ii] * sQ[k][fel][nd];
      }
      double *tr = a.traceOut + (size_t)fi + NP * (size_t)NT * (side + 4 * (size_t)fe);
#pragma unroll
      for (int k = 0; k < NT; k++) tr[(size_t)k * NP] = qn[k];
    }
    return;
  }
  for (int ft = tid; ft < EPB * NF; ft += THREADS) {
    const int fel3 = ft / NF, fnode3 = ft % NF;
    const int side3 = fnode3 / NP, fi3 = fnode3 % NP;
    const int pf3 = blk * EPB + fel3;
    if (pf3 >= a.nEl) continue;
    const int fe3 = a.elems ? a.elems[pf3] : pf3;
    const double *bm = (side3 == 1 || side3 == 2) ? bM1 : bM0;
    const bool alongJ = (side3 == 0 || side3 == 2);
    double qn[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) qn[k] = 0.0;
#pragma unroll
    for (int ii = 0; ii < NP; ii++) {
      const int nd = alongJ ? slot(fi3, ii) : slot(ii, fi3);
#pragma unroll
      for (int k = 0; k < NT; k++) qn[k] += bm[ii] * sQ[k][fel3][nd];
    }
    double *tr = a.traceOut + (size_t)fi3 + NP * (size_t)NT * (side3 + 4 * (size_t)fe3);
#pragma unroll
    for (int k = 0; k < NT; k++) tr[(size_t)k * NP] = qn[k];
  }
}

// The stage kernel: one tile per block.  XCD orders the tiles so that the blocks one XCD
// receives (the dispatcher deals blocks to the 8 XCDs in turn) cover a contiguous run of
// elements, whose neighbours then share that XCD's L2; a.reverse visits the tiles last to
// first (successive stages alternate direction).
template <class Phys, int N, int MODE, bool NODAL, int THREADS, int WPE = 1, bool XCD = false>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPE, 8))) k_fused(const FusedArgs a) {
  __shared__ __align__(16) double lds[TileLds<Phys, N, NODAL, THREADS>::SIZE];
  int blk = blockIdx.x;
  if constexpr (XCD) {
    const int nb = gridDim.x, q = nb >> 3, rem = nb & 7, x = blk & 7, k = blk >> 3;
    blk = x < rem ? x * (q + 1) + k : rem * (q + 1) + (x - rem) * q + k;
  }
  if (a.reverse) blk = (int)gridDim.x - 1 - blk;
  fused_tile<Phys, N, MODE, NODAL, THREADS>(a, blk, lds, threadIdx.x);
}

// Batched runs of several degrees in ONE launch per RK stage: a persistent grid (as many blocks
// as the device holds at once) over the tile lists of the degree groups N = 3, 5, 7, in that
// order (a tile of 256 work-items: 16, 7 or 4 elements).  Blocks are dispatched to the eight
// XCDs in turn (block b to XCD b mod 8), so each group's tile list is cut into eight contiguous
// parts and the blocks of XCD x stride through part x: every block gets the same mix of
// degrees and all blocks sweep the groups together.  A block loads a group's matrices into its
// LDS once; where each element lives in one wavefront (N = 3 and 7) the tiles then need no
// block barrier at all.  Per tile the arithmetic is that of the degree's own stage kernel, so
// every run stays bit-identical to its separate solve; each group's element order alternates
// between stages.
constexpr int kPersistentDegrees[3] = {3, 5, 7};
struct PersistentArgs {
  FusedArgs g[3];  // the groups of degree 3, 5, 7 (nEl = 0 when a degree is absent)
};
static_assert(sizeof(PersistentArgs) <= 4096, "kernel arguments exceed the 4 KiB kernarg segment");

template <class Phys>
__global__ void __launch_bounds__(256) k_batch_persistent(const PersistentArgs b) {
  constexpr int S3 = TileLds<Phys, 3, false, 256>::SIZE, S5 = TileLds<Phys, 5, false, 256>::SIZE,
                S7 = TileLds<Phys, 7, false, 256>::SIZE;
  constexpr int SMAX = S3 > S5 ? (S3 > S7 ? S3 : S7) : (S5 > S7 ? S5 : S7);
  __shared__ __align__(16) double lds[SMAX];
  const int G = gridDim.x, x = blockIdx.x & 7, r = blockIdx.x >> 3;
  const int cx = (G >> 3) + (x < (G & 7) ? 1 : 0);  // blocks on this XCD
  // one loop per degree, so that what the compiler keeps in registers across one degree's
  // tiles is not live during another's
  auto group = [&](auto deg, int k) {
    constexpr int N = decltype(deg)::value;
    using L = TileLds<Phys, N, false, 256>;
    const FusedArgs &a = b.g[k];
    const int nt = (a.nEl + L::EPB - 1) / L::EPB;
    const int l0 = (int)(((long long)nt * x) >> 3) + r, hi = (int)(((long long)nt * (x + 1)) >> 3);
    if (l0 >= hi) return;  // uniform over the block
    // the previous group's tiles are done with the LDS
    __syncthreads();
    load_tile_matrices<Phys, N, false, 256>(a.mats, lds, threadIdx.x);
    __syncthreads();
#pragma unroll 1
    for (int l = l0; l < hi; l += cx) {
      const int blk = a.reverse ? nt - 1 - l : l;
      // the work-item index, opaque to the compiler in each iteration: the tile's lane-derived
      // offsets are then formed per tile as in the one-tile kernel, not hoisted out of the loop
      // and held in registers across it
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      __builtin_assume(tid >= 0 && tid < 256);
      fused_tile<Phys, N, 0, false, 256, true>(a, blk, lds, tid);
      // the next tile reuses the LDS: where each element lives in one wavefront, that
      // wavefront's own accesses are in program order
      phase_sync<L::WAVE>();
    }
  };
  group(std::integral_constant<int, 3>{}, 0);
  group(std::integral_constant<int, 5>{}, 1);
  group(std::integral_constant<int, 7>{}, 2);
}

// ------------------------------------------------------------------------------
// Resident stepping: all RK stages of a call in one launch, for meshes that fit the device
// ------------------------------------------------------------------------------
// What bounds a small mesh is not the arithmetic but what comes once per stage: the launch (1.3 us,
// with the write-back of the stage's dirty L2 lines up to 4 us), reloading state, metrics and
// matrices (0.8 to 2 us before the first instruction that needs them), and interpolating own traces
// that the previous stage had.  When every block can be resident at once, one cooperative launch
// keeps the state, RK register, metrics, normals and the constant source gradient in registers and
// exchanges only face traces:
//   per stage  node lanes: volume flux -> LDS; face lanes: the neighbours' traces, boundary
//              conditions, Riemann flux -> LDS; node lanes: divergence, update; face lanes: traces
//              of the new state -> registers and the exchange ring.
// The arithmetic and its order are the stage kernel's, so the results are the same bits.
// Measured per stage (200-, 40- and 20-step calls): linear SW 10^2 N = 7 4.0 -> 1.7 us, 45 x 37 N = 6
// 8.0 -> 2.8 us, Euler 93 x 61 N = 4 15.3 -> 7.3 us.  Instances: WPE = 1 leaves the registers to the
// compiler and unrolls the divergence; where the mesh needs more blocks than fit that way, 3, 4 or 5
// wavefronts per SIMD (twice the elements and more).
//
// Exchange: ring buffer m mod 3 takes stage m's traces (and lagged velocities).  Every value is its
// own flag: a slot holds kEmpty, a signalling NaN that no arithmetic produces, until its owner
// stores the value, with relaxed agent-scope atomics on both sides; the reader polls its own
// values.  Face nodes are paired one to one: this lane reads the slots of lane L', and L' reads
// this lane's.  At stage m, L' has stored its traces of stage m - 1, so it has read this lane's of
// stage m - 2, and this lane empties those slots; the stores are complete (vmcnt 0) before this
// lane stores its traces of stage m, which L' must have seen before it polls the emptied slots
// again (for stage m + 1).  A call has a multiple of three stages and the last one stores to the
// trace buffers instead, so the next call finds the slots of its stage -2 filled and empties them
// first, and all others empty.
//
// With a closure (NET) a block has 16 elements, a row tile of the network, and the stage starts with
// features -> network -> correction in LDS.  The network's weights stay in registers (at 128 hidden
// units 80 of them; 1 block per CU), so a stage reads nothing from memory but traces and the other
// blocks' mass integrals, which every block sends to all others right after the network and needs
// only at the update.  64 x 64 elements, N = 3, 51 -> 128 -> 128 -> 48, per stage: 16.2 us in two
// launches (network 8.1 us of them), 6.6 us here: network 3.9, face and volume work 2.5.  With the
// integrals in one copy that all blocks poll, sent after the face phase, the wait for them alone was
// 3.3 us (9.5 us per stage).  A call of one step takes 78 us with set and get, 110 in launches.
//
// All blocks must be on the device at once.  The launch is cooperative, which the runtime refuses if
// they cannot be, but the runtime counts on an empty device: blocks of other streams that are there
// when the first blocks arrive leave gaps between theirs, and where the launch needs every register
// (SW N = 7, 4,096 blocks: four wavefronts of 128 of a SIMD's 512 registers) the last ones then never
// fit, however long the others wait.  So the blocks first meet at a gate, before anything is stored:
// each counts itself in, the last one opens the gate, and a block that has looked gatePolls times
// (some ms) closes it for good.  Whichever comes first holds for all blocks: of a launch whose gate
// is closed every block ends at once, as do those of the launches after it, and the host takes their
// steps by step graphs.  Past the gate every wait is for a block that is running; they are bounded
// all the same: a lane that has found slots empty `polls` times in a launch waits no more and raises
// `timedOut`, which the next synchronising call reports.
constexpr unsigned long long kEmpty = 0x7FF0DEAD7FF0DEADull;
constexpr int kPolls = 1 << 26, kGatePolls = 1 << 12;

// What a model's resident launches tell the host, in host memory.
struct ResidentReport {
  int timedOut;      // a wait past the gate gave up
  unsigned started;  // the last launch whose gate has opened
  unsigned refused;  // the launch whose gate was closed, or 0
};

// The gate, in device memory.  Launch L finds the verdict at 2 (L - 1), and it ends at 2 L (open) or
// odd (closed, for this launch and all that follow).  A launch's blocks count themselves in by groups.
// What a launch needs only before and after its stages is here too and not in the kernel arguments,
// where it would be held in registers throughout.
constexpr int kGateGroups = 64;
struct ResidentGate {
  struct alignas(128) Word {
    unsigned long long value;
  };
  Word verdict, groupsIn, in[kGateGroups];
  ResidentReport *report;
  int polls;      // per launch and lane
  int gatePolls;  // 0: the gate never opens
};
struct ResidentArgs {
  unsigned long long *ring;  // 3 buffers (0:N, NX, 4, nEl)
  int stages;                // 3 per step
  double rkA[3], rkGdt[3];   // a_m, g_m dt
  ResidentGate *gate;
};
// With a closure attached (NET): the network and where the blocks exchange their mass integrals
struct ResidentNetArgs {
  MlpWeights w;
  const float *inMean, *inScale, *outMean, *outScale;
  double shiftScale;
  unsigned long long *mass;  // 3 buffers, used like the trace ring, of kMassCopies times massStride values
  int massStride;            // one value per block, rounded up to 4 KiB
};

// The blocks' integrals go to every block: in as many copies as there are XCDs, so that not all
// blocks read the same few lines.
constexpr int kMassCopies = 8;

template <class Phys, int N, bool NODAL, bool NET = false>
struct ResidentTile {
  static constexpr int NP = N + 1, NN = NP * NP, NF = 4 * NP;
  // one wavefront per block, so that no phase boundary is a block barrier, except at N = 5, where
  // a wavefront would hold a single element on 36 of its lanes, and with a closure, whose network
  // takes 16 elements through its layers with 8 wavefronts
  static constexpr int T = NET ? kRowThreads : N == 5 ? 128 : 64;
  static constexpr int EPB = NET ? kRowTile : T / NN < T / NF ? T / NN : T / NF;
  static constexpr int FACE0 = NET ? T - EPB * NF : 0;  // first face lane
  static constexpr bool WAVE = T == 64;
  static constexpr bool SPLIT = N >= 6;  // the face sums of the stage kernel's tiles
  static constexpr int NV = Phys::NV, NT = Phys::NT, NX = NT + (Phys::kLag ? (NODAL ? 2 : 1) : 0);
  static constexpr int MRS = NP % 8 == 0 ? NP + 2 : NP, NNS = NP == 6 ? NN + 2 : NN;
  static constexpr int even(int n) { return (n + 1) & ~1; }
  // LDS in doubles; the static field and its metric products (prologue only) lie over BF and F1, F2
  static constexpr int Q = 0, F1 = Q + even(NT * EPB * NNS), F2 = F1 + even(NV * EPB * NNS);
  static constexpr int BF = F2 + even(NV * EPB * NNS), M = BF + even(NV * EPB * NF);
  // affine metrics of the block's elements (scalar registers instead where a wavefront is one)
  static constexpr int REC = M + even(2 * NP * MRS + 4 * NP), RECS = NODAL || NN == 64 ? 0 : 6 * EPB;
  // The tile's packets, staged so that the ring is written in whole lines (at N = 7 every store is
  // one; in runs of 8 (N + 1) bytes Euler 60^2 N = 1 took 11.7 us per stage, 4 us in lines): over F1
  // and F2 where they fit and no other wavefront uses those
  static constexpr bool STAGED = NP != 8;
  static constexpr int PKS = STAGED ? EPB * NF * NX : 0, PKOVER = WAVE && PKS <= F2 + even(NV * EPB * NNS) - F1;
  static constexpr int PK = PKOVER ? F1 : REC + RECS;
  static constexpr int SIZE = REC + RECS + (PKOVER ? 0 : even(PKS));
  static_assert(NNS <= NV * NF && F2 + even(NV * EPB * NNS) - F1 >= 4 * EPB * NNS, "prologue arrays do not fit");
};

__device__ inline unsigned long long ring_load(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void ring_store(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline unsigned long long gate_count(ResidentGate::Word &word) {
  return __hip_atomic_fetch_add(&word.value, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Settles the verdict, which this launch found at `found`, unless it is settled.
__device__ inline void gate_decide(ResidentGate *gate, unsigned long long found, bool open) {
  if (found & 1) return;
  const unsigned launch = (unsigned)(found >> 1) + 1;
  unsigned long long expected = found;
  if (__hip_atomic_compare_exchange_strong(&gate->verdict.value, &expected, open ? found + 2 : found + 1, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
    __hip_atomic_store(open ? &gate->report->started : &gate->report->refused, launch, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);  // the host may be looking
  }
}
// One work-item of every block: counts the block in and waits for the verdict.  The block has not
// been counted when it reads the verdict first, so that is the one before this launch's, or closed.
__device__ inline bool gate_opens(ResidentGate *gate) {
  const unsigned groups = min((unsigned)kGateGroups, gridDim.x), group = blockIdx.x % groups;
  const unsigned members = gridDim.x / groups + (group < gridDim.x % groups ? 1 : 0);
  const int polls = gate->gatePolls;
  const unsigned long long found = ring_load(&gate->verdict.value);
  if (found & 1) return false;
  if (gate_count(gate->in[group]) == members - 1) {
    ring_store(&gate->in[group].value, 0);  // for the next launch
    if (gate_count(gate->groupsIn) == groups - 1) {
      ring_store(&gate->groupsIn.value, 0);
      gate_decide(gate, found, polls > 0);
    }
  }
  for (int k = polls;; k--) {
    const unsigned long long seen = ring_load(&gate->verdict.value);
    if (seen != found) return !(seen & 1);
    if (k <= 0) gate_decide(gate, found, false);
  }
}

// The closure's network in a resident block: wavefront w holds the weights of columns 16 w .. 16 w +
// 15 of all three layers in registers for the whole call, pieces of 64 reduction indices each.
constexpr int kResidentHidden = 128;  // one 16-column tile per wavefront
template <int NIN, int NO>
struct ResidentNet {
  static constexpr int PIECES = pad64(NIN) / 64;
  static constexpr int LDX = rows_ld(NIN), LDH = rows_ld(kResidentHidden), LDO = rows_ld(NO);
  static constexpr int FLOATS = kRowTile * (LDX + 2 * LDH + LDO) + 2 * NO;
  static_assert(NIN <= 128 && NO <= 128, "a wavefront holds one tile of the output layer");
  float w1[PIECES][16], w2[2][16], w3[2][16], b1, b2, b3;
  int nH, wave, lane;

  __device__ void load(const ResidentNetArgs &n, int tid) {
    nH = n.w.nH;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    const int col = 16 * wave + (lane & 15), g = lane >> 4;
    const RowsOperand o1{n.w.W1, nH, NIN, nH}, o2{n.w.W2, nH, nH, nH}, o3{n.w.W3, NO, nH, NO};
#pragma unroll
    for (int k = 0; k < PIECES; k++) rows_load<false, false>(o1, col, g, 64 * k, w1[k]);
#pragma unroll
    for (int k = 0; k < 2; k++) {
      rows_load<false, false>(o2, col, g, 64 * k, w2[k]);
      rows_load<false, false>(o3, col, g, 64 * k, w3[k]);
    }
    b1 = n.w.b1[min(col, nH - 1)];
    b2 = n.w.b2[min(col, nH - 1)];
    b3 = n.w.b3[min(col, NO - 1)];
  }
  // one layer of this wavefront's columns: out(rows, column) = act(in W + b), 0 past `width`
  template <bool GELU, int K>
  __device__ void layer(const float *in, int ldIn, const float (&w)[K][16], bool second, float bias, int width,
                        float *out, int ldOut) const {
    if (16 * wave >= pad16(width)) return;
    const float *rows = in + (lane & 15) * ldIn + 4 * (lane >> 4);
    f32x4 acc = rows_mul(rows, w[0], f32x4{0.f, 0.f, 0.f, 0.f});
    if (K > 1 && second) acc = rows_mul(rows + 64, w[K - 1], acc);
    const int col = 16 * wave + (lane & 15), g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float y = acc[i] + bias;
      if constexpr (GELU) y = gelu_f(y);
      out[(4 * g + i) * ldOut + col] = col < width ? y : 0.f;
    }
  }
  // the network from the features in sX to the outputs in sO (not ended by a barrier)
  __device__ void run(const float *sX, float *sH1, float *sH2, float *sO) const {
    const bool second = nH > 64;
    layer<true>(sX, LDX, w1, true, b1, nH, sH1, LDH);
    __syncthreads();
    layer<true>(sH1, LDH, w2, second, b2, nH, sH2, LDH);
    __syncthreads();
    layer<false>(sH2, LDH, w3, second, b3, NO, sO, LDO);
  }
};

__global__ void k_ring_fill(unsigned long long *ring, size_t n) {
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
    ring[t] = kEmpty;
}
// The gate before launch number launches + 1.
__global__ void k_gate_reset(ResidentGate *gate, unsigned launches, ResidentReport *report, int polls, int gatePolls) {
  gate->in[threadIdx.x].value = 0;
  if (threadIdx.x) return;
  gate->groupsIn.value = 0;
  gate->verdict.value = 2ull * launches;
  gate->report = report;
  gate->polls = polls;
  gate->gatePolls = gatePolls;
}

template <class Phys, int N, bool NODAL, int WPE, bool NET = false>
__global__ void __launch_bounds__((ResidentTile<Phys, N, NODAL, NET>::T)) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
k_resident(const FusedArgs a, const ResidentArgs ra, const ResidentNetArgs na) {
  using L = ResidentTile<Phys, N, NODAL, NET>;
  constexpr int NP = L::NP, NN = L::NN, NF = L::NF, T = L::T, EPB = L::EPB, NV = L::NV, NT = L::NT, NX = L::NX;
  constexpr int MRS = L::MRS, NNS = L::NNS;
  constexpr bool SPLIT = L::SPLIT, WAVE = L::WAVE, SWZ = NP == 8;
  constexpr bool USE_AUX = Phys::kAuxGrad || Phys::kAuxTrace, GRAD = Phys::kAuxGrad, GRADN = NODAL && GRAD;
  __shared__ __align__(16) double lds[L::SIZE];
  auto slot = [](int i_, int j_) { return SWZ ? NP * j_ + (i_ ^ (j_ & 6)) : i_ + NP * j_; };
  auto sQ = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::Q);
  auto sF1 = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::F1);
  auto sF2 = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::F2);
  auto sBF = reinterpret_cast<double (*)[EPB][NF]>(lds + L::BF);
  auto sAux = reinterpret_cast<double (*)[NNS]>(lds + L::BF);
  auto sGb = reinterpret_cast<double (*)[EPB][NNS]>(lds + L::F1);
  double *sM = lds + L::M;
  const double *dgM = sM, *Dm = sM + NP * MRS, *bM0 = sM + 2 * NP * MRS, *bM1 = bM0 + NP, *qW = bM1 + NP;
  const int tid = threadIdx.x;

  // ---- lanes: nodes, and face nodes as in the stage kernel ----
  const int el = tid / NN, node = tid % NN, i = node % NP, j = node / NP, nl = slot(i, j);
  int e = blockIdx.x * EPB + el;
  bool nodeActive = el < EPB && e < a.nEl;
  if constexpr (NN == 64) {
    e = __builtin_amdgcn_readfirstlane(e);
    nodeActive = __builtin_amdgcn_readfirstlane((int)nodeActive) != 0;
  }
  const int fhalf = SPLIT ? tid >> 5 : 0, fslot = SPLIT ? tid & 31 : max(tid - L::FACE0, 0);
  const int fel = fslot / NF, fslotN = fslot % NF;
  const int side = SPLIT ? ((fslotN / NP) >> 1 | ((fslotN / NP) & 1) << 1) : fslotN / NP;
  const int fi = fslotN % NP, fnode = side * NP + fi, fe = blockIdx.x * EPB + fel;
  const bool faceActive = tid >= L::FACE0 && fel < EPB && fe < a.nEl && (!SPLIT || fslot < NF);
  const bool faceOwner = faceActive && fhalf == 0;  // the lane of a pair that has the face node
  const bool alongJ = side == 0 || side == 2;
  constexpr int FH0 = NP / 2, FHN = NP - FH0;

  for (int k = tid; k < 2 * NN + 4 * NP; k += T) {
    const int r = k % NN;
    sM[k < 2 * NN ? (k / NN) * NP * MRS + (r / NP) * MRS + r % NP : 2 * NP * MRS + k - 2 * NN] = a.mats[k];
  }

  // ---- prologue: everything that stays in registers ----
  const size_t sBase = (size_t)e * NV * NN, nodeAt = nodeActive ? (size_t)e * NN + node : (size_t)node;
  double s[NV], g[NV], auxVal = a.p.auxConst, statVal = a.p.stat2Const, dsdx[4] = {0, 0, 0, 0}, invJ = 1.0;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    s[v] = a.S[(nodeActive ? sBase + node : (size_t)node) + (size_t)v * NN];
    g[v] = 0.0;
  }
  if (USE_AUX && a.aux) auxVal = a.aux[nodeAt];
  if (a.stat2) statVal = a.stat2[nodeAt];
  if constexpr (NODAL) {
    const double *gn = a.ndsdx + 4 * nodeAt;
    dsdx[0] = gn[0]; dsdx[1] = gn[1]; dsdx[2] = gn[2]; dsdx[3] = gn[3];
    invJ = 1.0 / a.nJ[nodeAt];
  } else {
    const double *gr = a.geom + (nodeActive ? (size_t)e : 0) * kGeomStride;
    dsdx[0] = gr[0]; dsdx[1] = gr[1]; dsdx[2] = gr[2]; dsdx[3] = gr[3];
    invJ = gr[6];
  }
  int code = kNbrOrphan;
  double nx = 0.0, ny = 0.0, nmag = 0.0, unL = 0.0, unR = 0.0, qL[NT], qR[NT];
  unsigned mine = 0, theirs = 0;  // slots of this lane and of the lane it reads, within a ring buffer
  const unsigned ringLen = NP * NX * 4 * (unsigned)a.nEl;  // resident meshes are small
  if (faceOwner) {
    code = a.nbr[4 * (size_t)fe + side];
    const size_t fb = (size_t)fi + NP * (side + 4 * (size_t)fe);
    if constexpr (NODAL) {
      nx = a.nnHat[2 * fb]; ny = a.nnHat[2 * fb + 1]; nmag = a.nnScale[fb];
    } else {
      const double *gr = a.geom + (size_t)fe * kGeomStride;
      nx = gr[8 + side]; ny = gr[12 + side]; nmag = gr[16 + side];
    }
    mine = fi + NP * NX * (side + 4 * (unsigned)fe);
    // stage 0 reads the previous launch's traces and lagged velocities
    if (code >= 0) {
      const int s2 = (code >> 1) & 3, fi2 = (code & 1) ? N - fi : fi;
      const size_t e2 = (size_t)(code >> 3), nb = (size_t)fi2 + NP * (s2 + 4 * e2);
      const double *tr = a.traceIn + (size_t)fi2 + NP * (size_t)NT * (s2 + 4 * e2);
#pragma unroll
      for (int k = 0; k < NT; k++) qR[k] = tr[(size_t)k * NP];
      if (Phys::kLag) unR = lag_outer_raw<NODAL>(a.unIn, nb, nx, ny);
      theirs = fi2 + NP * NX * (s2 + 4 * (unsigned)e2);
    }
    if (Phys::kLag) unL = lag_own<NODAL>(a.unIn, fb, nx, ny);
  }
  if (nodeActive) {
    double q[NT];
    phys_nodal<Phys>(s, a.p, q);
#pragma unroll
    for (int k = 0; k < NT; k++) sQ[k][el][nl] = q[k];
    if (USE_AUX) sAux[el][nl] = auxVal;
    if constexpr (GRADN) {
#pragma unroll
      for (int k = 0; k < 4; k++) sGb[k][el][nl] = auxVal * dsdx[k];
    }
  }
  __syncthreads();
  // GradientSF of the static field (constant over the call) and its trace
  double gx = 0.0, gy = 0.0;
  if (GRAD && a.aux && nodeActive) {
    double dxi = 0.0, deta = 0.0;
    for (int ii = 0; ii < NP; ii++) {
      const double di = Dm[ii + MRS * i], dj = Dm[ii + MRS * j];
      if constexpr (GRADN) {
        gx = gx + di * sGb[0][el][slot(ii, j)] + dj * sGb[2][el][slot(i, ii)];
        gy = gy + di * sGb[1][el][slot(ii, j)] + dj * sGb[3][el][slot(i, ii)];
      } else {
        dxi = dxi + di * sAux[el][slot(ii, j)];
        deta = deta + dj * sAux[el][slot(i, ii)];
      }
    }
    if constexpr (!GRADN) {
      gx = dsdx[0] * dxi + dsdx[2] * deta;
      gy = dsdx[1] * dxi + dsdx[3] * deta;
    }
    gx = gx * invJ;
    gy = gy * invJ;
  }
  // sums over this lane's face line (its half of it, added across the pair): out[k] += b(ii) at(k, node)
  auto face_line = [&](auto count, auto at, double *out) {
    constexpr int K = decltype(count)::value;
    const double *bm = (side == 1 || side == 2) ? bM1 : bM0;
#pragma unroll
    for (int k = 0; k < K; k++) out[k] = 0.0;
    if constexpr (SPLIT) {
      const int lo = fhalf ? FH0 : 0;
#pragma unroll
      for (int t = 0; t < FHN; t++) {
        const int ii = lo + t;
        if (fhalf == 0 && t >= FH0) break;
        const int nd = alongJ ? slot(fi, ii) : slot(ii, fi);
#pragma unroll
        for (int k = 0; k < K; k++) out[k] += bm[ii] * at(k, nd);
      }
#pragma unroll
      for (int k = 0; k < K; k++) out[k] = pair_sum32(out[k]);
    } else {
#pragma unroll
      for (int ii = 0; ii < NP; ii++) {
        const int nd = alongJ ? slot(fi, ii) : slot(ii, fi);
#pragma unroll
        for (int k = 0; k < K; k++) out[k] += bm[ii] * at(k, nd);
      }
    }
  };
  using CountT = std::integral_constant<int, NT>;
  using Count1 = std::integral_constant<int, 1>;
  double auxB = a.p.auxConst;
  if (faceActive) {
    if (Phys::kAuxTrace && a.aux && (Phys::kAuxTraceInFlux || a.anyBoundary))
      face_line(Count1{}, [&](int, int nd) { return sAux[fel][nd]; }, &auxB);
    face_line(CountT{}, [&](int k, int nd) { return sQ[k][fel][nd]; }, qL);
  }
  __syncthreads();  // the prologue's arrays are overwritten from here on
  // affine metrics come from LDS at each use rather than from 10 registers held throughout
  double *rec = lds + L::REC + 6 * (el < EPB ? el : 0);
  if constexpr (L::RECS > 0) {
    if (nodeActive && node == 0) {
#pragma unroll
      for (int k = 0; k < 4; k++) rec[k] = dsdx[k];
      rec[4] = invJ;
    }
    __syncthreads();
  }

  // the closure: network, features that stay (the element's metric terms), scales and weights
  constexpr int NO = NV * NN, NIN = NO + 3;
  using Net = ResidentNet<NET ? NIN : 1, NET ? NO : 1>;
  __shared__ __align__(16) float netLds[NET ? Net::FLOATS : 4];
  __shared__ double sWeight[NET ? NO : 1], sJ[NET ? EPB : 1], sRed[NET ? EPB : 1], sShift;
  float *sX = netLds, *sH1 = sX + kRowTile * Net::LDX, *sH2 = sH1 + kRowTile * Net::LDH, *sO = sH2 + kRowTile * Net::LDH;
  float *sScale = sO + kRowTile * Net::LDO, *sMean = sScale + NO;
  [[maybe_unused]] Net net;
  [[maybe_unused]] float inMean[NV], inScale[NV];
  if constexpr (NET) {
    net.load(na, tid);
    for (int k = tid; k < Net::FLOATS - 2 * NO; k += T) netLds[k] = 0.f;  // rows and columns that stay empty
    for (int k = tid; k < NO; k += T) {
      sScale[k] = na.outScale[k];
      sMean[k] = na.outMean[k];
      const int nd = k - 2 * NN;  // variable 2 is H / eta / rho
      sWeight[k] = nd >= 0 && nd < NN ? qW[nd % NP] * qW[nd / NP] : 0.0;
    }
    __syncthreads();
    for (int k = tid; k < 3 * EPB; k += T) {
      const int row = k / 3, c = k % 3;
      const size_t re = (size_t)blockIdx.x * EPB + row;
      if (re < (size_t)a.nEl) {
        const double *gr = a.geom + re * kGeomStride;
        const double raw = gr[c == 0 ? 4 : c == 1 ? 0 : 3];
        sX[row * Net::LDX + NO + c] = (float)((raw - (double)na.inMean[NO + c]) / (double)na.inScale[NO + c]);
        if (c == 0) sJ[row] = raw;
      } else if (c == 0) {
        sJ[row] = 0.0;
      }
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
      inMean[v] = na.inMean[v * NN + node];
      inScale[v] = na.inScale[v * NN + node];
    }
  }

  // ---- the gate, behind the prologue's loads: uniform ones are scalar loads only before a kernel's
  // first store (with the gate at the start SW N = 7 takes 132 registers against 126) ----
  bool open = false;
  if (tid == 0) open = gate_opens(ra.gate);
  if constexpr (WAVE) {
    open = __builtin_amdgcn_readfirstlane((int)open) != 0;
  } else {
    __shared__ int sOpen;
    if (tid == 0) sOpen = open;
    __syncthreads();
    open = sOpen != 0;
  }
  if (!open) return;

  // ---- stages ----
  const unsigned tileAt = blockIdx.x * (unsigned)(EPB * NF * NX);
  const int tileSlots = min(EPB, a.nEl - (int)blockIdx.x * EPB) * NF * NX;
  int budget = ra.gate->polls - 1, fill = 0;  // fill: m mod 3
#pragma unroll 1
  for (int m = 0; m < ra.stages; m++) {
    const bool last = m == ra.stages - 1;
    const int before = fill == 0 ? 2 : fill - 1, empty = fill == 2 ? 0 : fill + 1;  // (m - 1), (m - 2) mod 3
    if (nodeActive) {
      double fx[NV], fy[NV], q[NT];
      Phys::volume(s, auxVal, a.p, fx, fy, q);
      if constexpr (L::RECS > 0) {
#pragma unroll
        for (int k = 0; k < 4; k++) dsdx[k] = rec[k];
      }
#pragma unroll
      for (int v = 0; v < NV; v++) {
        sF1[v][el][nl] = dsdx[0] * fx[v] + dsdx[1] * fy[v];
        sF2[v][el][nl] = dsdx[2] * fx[v] + dsdx[3] * fy[v];
      }
      if constexpr (NET) {
#pragma unroll
        for (int v = 0; v < NV; v++)
          sX[el * Net::LDX + v * NN + node] = (float)((s[v] - (double)inMean[v]) / (double)inScale[v]);
      }
    }
    if constexpr (NET) {
      // every block has read this one's integral of stage m - 2: their integrals of stage m - 1 are here
      const size_t mine8 = (size_t)(net.lane & (kMassCopies - 1)) * na.massStride + blockIdx.x;
      const bool publisher = net.wave == T / 64 - 1 && net.lane < kMassCopies;
      if (publisher) ring_store(na.mass + (size_t)empty * kMassCopies * na.massStride + mine8, kEmpty);
      __syncthreads();
      net.run(sX, sH1, sH2, sO);
      __syncthreads();
      // integral of the mass variable's correction over each element: 32 work-items per element
      const int row = tid >> 5;
      double mass = 0.0;
      for (int k = tid & 31; k < NO; k += 32) {
        const double c = (double)sO[row * Net::LDO + k] * (double)sScale[k] + (double)sMean[k];
        mass += sWeight[k] * c;
      }
      mass = half_sum32(mass);
      if ((tid & 31) == 0) sRed[row] = sJ[row] * mass;
      __syncthreads();
      if (net.wave == T / 64 - 1) {  // as early as it can be: the face phase hides its way to the other blocks
        const double own = row_sum16(sRed[net.lane & 15]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the emptied slots first (see above)
        if (publisher)
          ring_store(na.mass + (size_t)fill * kMassCopies * na.massStride + mine8, (unsigned long long)__double_as_longlong(own));
      }
    }
    double lag0 = 0.0, lag1 = 0.0;  // this stage's own face velocity, for the next one
    if (faceOwner) {
      if (code >= 0 && m > 0) {
        const unsigned long long *p = ra.ring + (size_t)before * ringLen + theirs;
        unsigned long long x[NX];
        for (;;) {
          bool ok = true;
#pragma unroll
          for (int k = 0; k < NX; k++) x[k] = ring_load(p + k * NP);
#pragma unroll
          for (int k = 0; k < NX; k++) ok = ok && x[k] != kEmpty;
          if (ok || --budget < 0) break;
        }
#pragma unroll
        for (int k = 0; k < NT; k++) qR[k] = __longlong_as_double((long long)x[k]);
        if constexpr (Phys::kLag) {
          const double u = __longlong_as_double((long long)x[NT]);
          if constexpr (NODAL) unR = u * nx + __longlong_as_double((long long)x[NX - 1]) * ny;
          else unR = u;
        }
      } else if (code < 0) {
        if (code == kNbrOrphan) {
#pragma unroll
          for (int k = 0; k < NT; k++) qR[k] = 0.0;
        } else {
          const double *pres = a.presTrace ? a.presTrace + (size_t)fi + NP * (size_t)NT * (side + 4 * (size_t)fe) : nullptr;
          double pv[NT];
#pragma unroll
          for (int k = 0; k < NT; k++) pv[k] = pres ? pres[(size_t)k * NP] : 0.0;
          Phys::bc(qL, auxB, nx, ny, -code - 1, pv, pres != nullptr, qR);
        }
      }
      if (!L::STAGED && code >= 0) {
#pragma unroll
        for (int k = 0; k < NX; k++) ring_store(ra.ring + (size_t)empty * ringLen + mine + k * NP, kEmpty);
      }
      if constexpr (Phys::kLag) {
        const double invH = 1.0 / qL[2];
        if constexpr (NODAL) {
          lag0 = qL[0] * invH;
          lag1 = qL[1] * invH;
        } else {
          lag0 = (qL[0] * invH) * nx + (qL[1] * invH) * ny;
        }
      }
      double fstar[NV];
      Phys::riemann(qL, qR, nx, ny, nmag, auxB, unL, outer_un<NODAL>(unR), a.p, fstar);
#pragma unroll
      for (int v = 0; v < NV; v++) sBF[v][fel][fnode] = fstar[v];
    }
    phase_sync<WAVE>();
    if constexpr (L::STAGED)  // every lane of the tile has its neighbour's traces
      for (int k = tid; k < tileSlots; k += T) ring_store(ra.ring + (size_t)empty * ringLen + tileAt + k, kEmpty);

    auto divergence = [&](double *dxs, double *des) {
#pragma unroll
      for (int v = 0; v < NV; v++) { dxs[v] = 0.0; des[v] = 0.0; }
      auto line = [&](int ii) {
        const double ai = dgM[ii + MRS * i], aj = dgM[ii + MRS * j];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          dxs[v] = dxs[v] + ai * sF1[v][el][slot(ii, j)];
          des[v] = des[v] + aj * sF2[v][el][slot(i, ii)];
        }
      };
      if constexpr (WPE <= 2) {
#pragma unroll
        for (int ii = 0; ii < NP; ii++) line(ii);
      } else {
#pragma unroll 2
        for (int ii = 0; ii < NP; ii++) line(ii);
      }
    };
    auto update = [&](const double *dxs, const double *des, double shift) {
      double src[NV];
      Phys::source(s, gx, gy, statVal, a.p, src);
      const double rkA = ra.rkA[fill], gdt = ra.rkGdt[fill];
      const double iwi = qW[NP + i], iwj = qW[NP + j];
      const double bi1 = bM1[i], bi0 = bM0[i], bj1 = bM1[j], bj0 = bM0[j];
      if constexpr (L::RECS > 0) invJ = rec[4];
#pragma unroll
      for (int v = 0; v < NV; v++) {
        double d = dxs[v] + des[v];
        d = d + (bi1 * sBF[v][el][NP + j] + bi0 * sBF[v][el][3 * NP + j]) * iwi +
            (bj1 * sBF[v][el][2 * NP + i] + bj0 * sBF[v][el][i]) * iwj;
        d = d * invJ;
        double dsdt = src[v] - d;
        if constexpr (NET) {
          const int k = v * NN + node;
          double c = (double)sO[el * Net::LDO + k] * (double)sScale[k] + (double)sMean[k];
          if (v == 2) c -= shift;
          dsdt += c;
        }
        g[v] = rkA * (fill == 0 ? 0.0 : g[v]) + dsdt;
        s[v] = s[v] + gdt * g[v];
        // the RK register that the last step's second stage leaves behind
        if (m == ra.stages - 2) a.G[sBase + (size_t)v * NN + node] = g[v];
      }
      double q[NT];
      phys_nodal<Phys>(s, a.p, q);
#pragma unroll
      for (int k = 0; k < NT; k++) sQ[k][el][nl] = q[k];
    };
    if constexpr (NET) {
      // the last wavefront, which has no nodes, adds up all blocks' integrals meanwhile, in the
      // order of the stage kernel
      static_assert(EPB * NN <= T - 64, "the last wavefront has nodes");
      double dxs[NV], des[NV];
      if (nodeActive) divergence(dxs, des);
      if (net.wave == T / 64 - 1) {
        double part = 0.0;
        const unsigned long long *box =
            na.mass + (size_t)(fill * kMassCopies + (int)(blockIdx.x & (kMassCopies - 1))) * na.massStride;
        const int n = (int)gridDim.x;
        for (int k = net.lane; k < n; k += 256) {
          unsigned long long x[4];
          for (;;) {
            bool ok = true;
#pragma unroll
            for (int q = 0; q < 4; q++) x[q] = ring_load(box + min(k + 64 * q, n - 1));
#pragma unroll
            for (int q = 0; q < 4; q++) ok = ok && x[q] != kEmpty;
            if (ok || --budget < 0) break;
          }
#pragma unroll
          for (int q = 0; q < 4; q++) part += k + 64 * q < n ? __longlong_as_double((long long)x[q]) : 0.0;
        }
        part = wave_sum(part);
        part *= na.shiftScale;
        if (net.lane == 0) sShift = part;
      }
      __syncthreads();
      if (nodeActive) update(dxs, des, sShift);
    } else if (nodeActive) {
      double dxs[NV], des[NV];
      divergence(dxs, des);
      update(dxs, des, 0.0);
    }
    phase_sync<WAVE>();

    if (faceActive) {
      face_line(CountT{}, [&](int k, int nd) { return sQ[k][fel][nd]; }, qL);
      if (fhalf == 0) {
        if (!last) {
          if constexpr (L::STAGED) {
            double *p = lds + L::PK + fi + NP * NX * (side + 4 * fel);
#pragma unroll
            for (int k = 0; k < NT; k++) p[k * NP] = qL[k];
            if constexpr (Phys::kLag) p[NT * NP] = lag0;
            if constexpr (Phys::kLag && NODAL) p[(NX - 1) * NP] = lag1;
          } else if (code >= 0) {
            // the emptied slots before the new traces (see above)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            unsigned long long *p = ra.ring + (size_t)fill * ringLen + mine;
#pragma unroll
            for (int k = 0; k < NT; k++) ring_store(p + k * NP, (unsigned long long)__double_as_longlong(qL[k]));
            if constexpr (Phys::kLag) ring_store(p + NT * NP, (unsigned long long)__double_as_longlong(lag0));
            if constexpr (Phys::kLag && NODAL) ring_store(p + (NX - 1) * NP, (unsigned long long)__double_as_longlong(lag1));
          }
        } else {
          const size_t fb = (size_t)fi + NP * (side + 4 * (size_t)fe);
          double *tr = a.traceOut + (size_t)fi + NP * (size_t)NT * (side + 4 * (size_t)fe);
#pragma unroll
          for (int k = 0; k < NT; k++) tr[(size_t)k * NP] = qL[k];
          if constexpr (Phys::kLag && NODAL) { a.unOut[2 * fb] = lag0; a.unOut[2 * fb + 1] = lag1; }
          else if constexpr (Phys::kLag) a.unOut[fb] = lag0;
        }
        if constexpr (Phys::kLag) unL = NODAL ? lag0 * nx + lag1 * ny : lag0;
      }
    }
    if constexpr (L::STAGED)
      if (!last) {
        phase_sync<WAVE>();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the emptied slots before the new traces (see above)
        for (int k = tid; k < tileSlots; k += T)
          ring_store(ra.ring + (size_t)fill * ringLen + tileAt + k, (unsigned long long)__double_as_longlong(lds[L::PK + k]));
        if constexpr (WAVE) phase_sync<WAVE>();
      }
    fill = empty;
  }
  if (nodeActive) {
#pragma unroll
    for (int v = 0; v < NV; v++) a.S[sBase + (size_t)v * NN + node] = s[v];
  }
  if (budget < 0) ra.gate->report->timedOut = 1;
}

// ------------------------------------------------------------------------------
// Integrals of the state: CalculateEntropy and mass-type integrals
// ------------------------------------------------------------------------------
// One work-item per node forms w_i w_j J f(S) (the per-node J as SEMQuad stores it); blocks
// sum in a fixed tree order into partial sums, and one block adds those in a fixed order, so
// the result does not depend on scheduling.
constexpr int kIntBlock = 256;
enum IntegralKind { kIntSWEntropy = 0, kIntLSWEntropy = 1, kIntEulerEntropy = 2, kIntVariable = 3 };

__device__ inline void block_sum_store(double v, double *out) {
  __shared__ double red[kIntBlock];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int st = kIntBlock / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

template <int WHAT>
__global__ void __launch_bounds__(kIntBlock) k_integral_partial(const double *S, const double *aux, const double *J,
                                                                const double *qW, Params p, int N, int nVar, int var,
                                                                size_t nNodes, double *partial) {
  const size_t n = blockIdx.x * (size_t)kIntBlock + threadIdx.x;
  double v = 0.0;
  if (n < nNodes) {
    const int P = N + 1, PP = P * P;
    const size_t e = n / PP;
    const int node = (int)(n - e * PP), i = node % P, j = node / P;
    const double jac = J[n], wi = qW[i], wj = qW[j];
    const double *s = S + e * (size_t)nVar * PP + node;  // variable k at s[k * PP]
    if (WHAT == kIntSWEntropy) {
      // CalculateEntropy_ShallowWater (src/models/SELF_ShallowWater.f90:149-188)
      const double Hu = s[0], Hv = s[PP], H = s[2 * PP], b = aux ? aux[n] : p.auxConst;
      v = (0.5 * (Hu * Hu / H + Hv * Hv / H) + 0.5 * p.g * H * H - p.g * H * b) * jac * wi * wj;
    } else if (WHAT == kIntLSWEntropy) {
      // CalculateEntropy_LinearShallowWater (src/models/SELF_LinearShallowWater.f90:171-216)
      const double u = s[0], vv = s[PP], eta = s[2 * PP], H = aux ? aux[n] : p.auxConst;
      v = 0.5 * (H * (u * u + vv * vv) + p.g * eta * eta) * jac * wi * wj;
    } else if (WHAT == kIntEulerEntropy) {
      // CalculateEntropy_CompressibleIdealGas2D (src/models/SELF_CompressibleIdealGas2D.f90:782-823)
      // with the pressure of the current state (ConservativeToPrimitive, :1129-1170)
      const double rhoU = s[0], rhoV = s[PP], rho = s[2 * PP], rhoE = s[3 * PP];
      const double u = rhoU / rho, vv = rhoV / rho;
      const double pr = (p.gamma - 1.0) * (rhoE - 0.5 * (rhoU * u + rhoV * vv));
      v = rho * (log(pr) - p.gamma * log(rho)) / (p.gamma - 1.0) * wi * wj * jac;
    } else {
      v = s[(size_t)var * PP] * wi * wj * jac;
    }
  }
  block_sum_store(v, partial + blockIdx.x);
}

// one block: work-item t adds partial[t], partial[t + kIntBlock], ... in order, then the
// block sums the work-items' totals in a fixed tree order
__global__ void __launch_bounds__(kIntBlock) k_sum_partials(const double *partial, int n, double *out) {
  double v = 0.0;
  for (int k = threadIdx.x; k < n; k += kIntBlock) v += partial[k];
  block_sum_store(v, out);
}

// A state taken in (SetSolution) in one pass over it: copied to S, interpolated to the faces
// (BoundaryInterp), and from the same registers the SW lagged velocities of the first stage and
// the Euler prescribed traces.  What bounds it: memory on large meshes, the launch on small ones.
// As copy, trace, velocity and trace copy launches one after another, with the call's
// synchronisation: linear SW 10^2 N = 7 19.0 us, SW 256^2 N = 7 85, Euler 400^2 N = 7 432; in one
// pass 15.5, 61 and 189.
struct StateArgs {
  const double *src;
  double *S;      // or null: traces only
  double *trace;
  double *un;     // SW lagged velocities (nnHat: the nodal mode's vectors), or null
  double *pres;   // Euler prescribed traces, or null; only sides on the physical boundary are read
  const double *geom, *nnHat, *mats;
  const int32_t *nbr;
  Params p;
  int nEl;
};
template <class Phys, int N>
__global__ void __launch_bounds__(kThreads) k_state_in(const StateArgs a) {
  constexpr int NP = N + 1, NN = NP * NP, EPB = kThreads / NN, NF = 4 * NP;
  constexpr int NV = Phys::NV, NT = Phys::NT;
  __shared__ double sQ[NT][EPB][NN];
  const int tid = threadIdx.x;
  const int el = tid / NN, node = tid % NN;
  const int e = blockIdx.x * EPB + el;
  if (el < EPB && e < a.nEl) {
    const size_t at = (size_t)e * NV * NN + node;
    double s[NV], q[NT];
#pragma unroll
    for (int v = 0; v < NV; v++) s[v] = a.src[at + (size_t)v * NN];
    if (a.S) {
#pragma unroll
      for (int v = 0; v < NV; v++) a.S[at + (size_t)v * NN] = s[v];
    }
    phys_nodal<Phys>(s, a.p, q);
#pragma unroll
    for (int k = 0; k < NT; k++) sQ[k][el][node] = q[k];
  }
  __syncthreads();
  for (int ft = tid; ft < EPB * NF; ft += kThreads) {
    const int fel = ft / NF, fnode = ft % NF, side = fnode / NP, fi = fnode % NP;
    const int fe = blockIdx.x * EPB + fel;
    if (fe >= a.nEl) continue;
    const double *bm = a.mats + 2 * NN + ((side == 1 || side == 2) ? NP : 0);
    const bool alongJ = (side == 0 || side == 2);
    double qn[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) qn[k] = 0.0;
#pragma unroll
    for (int ii = 0; ii < NP; ii++) {
      const int nd = alongJ ? fi + NP * ii : ii + NP * fi;
#pragma unroll
      for (int k = 0; k < NT; k++) qn[k] += bm[ii] * sQ[k][fel][nd];
    }
    const size_t first = (size_t)fi + NP * (size_t)NT * (side + 4 * (size_t)fe);
#pragma unroll
    for (int k = 0; k < NT; k++) a.trace[first + (size_t)k * NP] = qn[k];
    if (a.pres && a.nbr[side + 4 * (size_t)fe] < 0) {
#pragma unroll
      for (int k = 0; k < NT; k++) a.pres[first + (size_t)k * NP] = qn[k];
    }
    if constexpr (Phys::kLag) {
      const size_t fb = (size_t)fi + NP * (side + 4 * (size_t)fe);
      if (a.un && a.nnHat) {
        a.un[2 * fb] = qn[0] / qn[2];
        a.un[2 * fb + 1] = qn[1] / qn[2];
      } else if (a.un) {
        const double *gr = a.geom + (size_t)fe * kGeomStride;
        const double nx = gr[8 + side], ny = gr[12 + side];
        a.un[fb] = (qn[0] / qn[2]) * nx + (qn[1] / qn[2]) * ny;
      }
    }
  }
}

// Initial SW lagged normal velocities (own side of each face node) from the current traces:
// at the first stage after SetSolution the reference's velocity traces come from
// SetSolution's BoundaryInterp.
template <int N>
__global__ void k_sw_un_init(const double *trace, double *un, const double *geom, const double *nnHat, int nEl) {
  constexpr int NP = N + 1;
  const size_t total = (size_t)NP * 4 * nEl;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    const int fi = t % NP, side = (t / NP) % 4;
    const size_t e = t / (4 * NP);
    double nx, ny;
    if (nnHat) {
      nx = nnHat[2 * t]; ny = nnHat[2 * t + 1];
    } else {
      const double *gr = geom + e * kGeomStride;
      nx = gr[8 + side]; ny = gr[12 + side];
    }
    const double *tl = trace + fi + NP * 3 * (side + 4 * e);
    if (nnHat) {
      un[2 * t] = tl[0] / tl[2 * NP];
      un[2 * t + 1] = tl[NP] / tl[2 * NP];
    } else {
      un[t] = (tl[0] / tl[2 * NP]) * nx + (tl[NP] / tl[2 * NP]) * ny;
    }
  }
}

// Block size (tile) per polynomial degree: one wavefront per element at N = 7, larger
// blocks where an element covers only part of a wavefront.  N = 5 with nodal metrics: 7 elements
// on 252 of 256 lanes against 3 on 108 of 128; per stage SW 121 x 87 20.2 against 21.2 us, 300 x
// 200 81.7 and 86.2, Euler 121 x 87 25.3 and 27.0, linear SW 17.0 and 18.1 (with affine metrics
// the tuned tiles' 128 lanes are the faster ones).
template <int N>
constexpr int tile_threads(bool nodal = false) {
  return N == 7 ? 64 : N == 6 ? 64 : N == 5 ? (nodal ? 256 : 128) : N == 4 ? 128 : 256;
}

// Tuned tiles: the stage kernel (affine metrics, RK update) of SW at N = 3, 5, 7 and of LSW
// and Euler at N = 7 comes in 18 variants.  v < 12: v = 4 t + 2 r + x with THREADS = 64 << t,
// element order alternating between stages when r = 1, XCD-contiguous element order when
// x = 1.  v = 12 + 2 t + w: THREADS = 64 << t, alternating order, and an occupancy target of
// 5 + w wavefronts per SIMD for the register allocator (a few registers spill to scratch).  The table below (per N; -1 =
// the default tile) is set by selfamd_tile_set, normally from the autotuner's measurements.
// Variants whose blocks leave room for two lanes per face node split the face-line sums
// between the pair (round-off level differences); otherwise the arithmetic is identical.
constexpr int kTileVariants = 18;
// g_tile[kind][N]: SW at N = 3, 5, 7; LSW and Euler at N = 7
int g_tile[4][8] = {{-1, -1, -1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1, -1, -1},
                    {-1, -1, -1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1, -1, -1}};
inline bool tunable(int kind, int N) {
  return (kind == SELFAMD_MODEL_SW && (N == 3 || N == 5 || N == 7)) ||
         ((kind == SELFAMD_MODEL_LSW || kind == SELFAMD_MODEL_EULER) && N == 7);
}
inline int tile_of(int kind, int N) { return tunable(kind, N) ? g_tile[kind][N] : -1; }
// Launches of at most kSmallLaunch elements (a few per CU) take small tiles in plain element
// order, whatever the table (tuned on 256^2 meshes) says.  Measured per launch: SW at N = 7,
// 64 wide, 4.75 against 5.54 us at 10^2 and 10.8 against 14.7 us at 64^2 (the tuned 256-wide
// alternating tile wins from 96^2 on); SW at N = 5, 128 wide in XCD order, 8.6 against 12.1 us
// at 64^2 (equal at 128^2); LSW and Euler at N = 7, 64 wide, 4.4 against 5.1 us (10^2) and
// 7.2 against 9.6 us (32^2).  The face sums split as the table's tile does (N = 5 keeps a
// table entry of 64 wide, which splits), so a run's results do not depend on launch sizes.
constexpr int kSmallLaunch = 8192;
inline int tile_for(int kind, int N, int nEl) {
  const int v = tile_of(kind, N);
  if (tunable(kind, N) && nEl <= kSmallLaunch) {
    if (N == 7) return 0;
    const bool split64 = v >= 0 && ((v < 12 && (v >> 2) == 0) || v == 12 || v == 13);
    if (N == 5 && !split64) return 5;
  }
  return v;
}
// element order alternates between stages (the default tiles alternate too)
inline bool tile_alternates(int kind, int N, int nEl) {
  const int v = tile_for(kind, N, nEl);
  return v < 0 || v >= 12 || (v & 2);
}
int g_tileEpoch = 0;
// whether tile variant v of N = 5 splits the face sums between lane pairs (the 64-wide ones)
inline bool tile_splits5(int v) { return v >= 0 && ((v < 12 && (v >> 2) == 0) || v == 12 || v == 13); }


template <class Phys, int N>
hipError_t launch_tile(int v, const FusedArgs &a, hipStream_t st) {
  constexpr int NN = (N + 1) * (N + 1);
  switch (v) {
#define V(IDX, T, W, X)                                                                        \
  case IDX: {                                                                                  \
    constexpr int EPB = T / NN;                                                                \
    hipLaunchKernelGGL((k_fused<Phys, N, 0, false, T, W, X>), dim3((a.nEl + EPB - 1) / EPB), T, 0, st, a); \
    return hipGetLastError();                                                                  \
  }
    V(0, 64, 1, false) V(1, 64, 1, true) V(2, 64, 1, false) V(3, 64, 1, true)
    V(4, 128, 1, false) V(5, 128, 1, true) V(6, 128, 1, false) V(7, 128, 1, true)
    V(8, 256, 1, false) V(9, 256, 1, true) V(10, 256, 1, false) V(11, 256, 1, true)
    V(12, 64, 5, false) V(13, 64, 6, false) V(14, 128, 5, false) V(15, 128, 6, false)
    V(16, 256, 5, false) V(17, 256, 6, false)
#undef V
    default: return hipErrorInvalidValue;
  }
}

template <class Phys>
struct Launcher {
  static hipError_t stage(int N, int mode, bool nodal, const FusedArgs &a, hipStream_t st) {
    const int v = (mode == 0 && !nodal) ? tile_for(Phys::kKind, N, a.nEl) : -1;
    if (v >= 0) {
      if constexpr (std::is_same<Phys, PhysSW>::value) {
        if (N == 3) return launch_tile<Phys, 3>(v, a, st);
        if (N == 5) return launch_tile<Phys, 5>(v, a, st);
      }
      if (N == 7) return launch_tile<Phys, 7>(v, a, st);
    }
    switch (N) {
#define CASE(NN_)                                                                                     \
  case NN_: {                                                                                         \
    constexpr int T = tile_threads<NN_>(), TNOD = tile_threads<NN_>(true);                            \
    const int EPB = (nodal ? TNOD : T) / ((NN_ + 1) * (NN_ + 1));                                     \
    dim3 grid((a.nEl + EPB - 1) / EPB);                                                               \
    if (nodal) {                                                                                      \
      if (mode == 0) hipLaunchKernelGGL((k_fused<Phys, NN_, 0, true, TNOD>), grid, TNOD, 0, st, a);   \
      else hipLaunchKernelGGL((k_fused<Phys, NN_, 1, true, TNOD>), grid, TNOD, 0, st, a);             \
    } else {                                                                                          \
      if (mode == 0) hipLaunchKernelGGL((k_fused<Phys, NN_, 0, false, T>), grid, T, 0, st, a);        \
      else hipLaunchKernelGGL((k_fused<Phys, NN_, 1, false, T>), grid, T, 0, st, a);                  \
    }                                                                                                 \
    return hipGetLastError();                                                                         \
  }
      CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
      default: return hipErrorInvalidValue;
    }
  }
  static hipError_t state_in(int N, const StateArgs &a, hipStream_t st) {
    switch (N) {
#define CASE(NN_)                                                                                   \
  case NN_: {                                                                                       \
    constexpr int EPB = kThreads / ((NN_ + 1) * (NN_ + 1));                                         \
    hipLaunchKernelGGL((k_state_in<Phys, NN_>), dim3((a.nEl + EPB - 1) / EPB), kThreads, 0, st, a); \
    return hipGetLastError();                                                                       \
  }
      CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
      default: return hipErrorInvalidValue;
    }
  }
};

hipError_t launch_un_init(int N, const double *tr, double *un, const double *geom, const double *nnHat, int nEl,
                          hipStream_t st) {
  const size_t n = (size_t)(N + 1) * 4 * nEl;
  const unsigned blocks = (unsigned)((n + 255) / 256);
  switch (N) {
#define CASE(NN_) \
  case NN_: hipLaunchKernelGGL((k_sw_un_init<NN_>), dim3(blocks), 256, 0, st, tr, un, geom, nnHat, nEl); return hipGetLastError();
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
    default: return hipErrorInvalidValue;
  }
}

struct ResidentKernel {
  const void *fn = nullptr;
  int threads = 0, elements = 0, values = 0;  // per block: work-items, elements; ring values per face node
};
// dense 1, 2, 3: instances held to the registers of 3, 4 and 5 wavefronts per SIMD, for more resident
// blocks.  Per stage of 20-step calls, stage launches against resident ones: 4 wavefronts, SW 64^2
// N = 7 9.7 and 6.0 us, N = 5 6,000 elements 11.1 and 5.9, linear SW 128^2 N = 3 12.2 and 8.2; 5
// wavefronts (4,096 to 5,120 blocks), SW N = 7 12.1 and 8.1, N = 3 11.3 and 10.2, linear SW N = 7 10.6
// and 5.9, N = 2 13.7 and 10.2.  SW with 5 wavefronts loses at N = 1 (12.6 and 15.6) and gains
// nothing at N = 2 on nodal metrics, linear SW at N = 1 neither; Euler needs more registers or LDS.
constexpr int kResidentDense = 4;
template <class Phys, int N, bool NODAL>
ResidentKernel resident_instance(int dense) {
  using L = ResidentTile<Phys, N, NODAL>;
  constexpr bool FIVE = Phys::NV == 3 && (N >= 3 || (N == 2 && !Phys::kLag));
  constexpr bool FOUR = Phys::NV == 3 || !(N == 2 || N == 3 || N == 5);  // LDS of these Euler tiles: 3 at most
  const void *fn = nullptr;
  switch (dense) {
    case 0: fn = reinterpret_cast<const void *>(&k_resident<Phys, N, NODAL, 1>); break;
    case 1: fn = reinterpret_cast<const void *>(&k_resident<Phys, N, NODAL, 3>); break;
    case 2:
      if constexpr (FOUR) fn = reinterpret_cast<const void *>(&k_resident<Phys, N, NODAL, 4>);
      break;
    case 3:
      if constexpr (FIVE) fn = reinterpret_cast<const void *>(&k_resident<Phys, N, NODAL, 5>);
  }
  return {fn, L::T, L::EPB, L::NX};
}
template <class Phys, bool NODAL>
ResidentKernel resident_of(int N, int dense) {
  switch (N) {
#define CASE(NN_) case NN_: return resident_instance<Phys, NN_, NODAL>(dense);
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
    default: return {};
  }
}
// with a closure attached (affine metrics): degrees whose nodes leave a wavefront of the block free
template <class Phys>
ResidentKernel resident_net_of(int N) {
  switch (N) {
#define CASE(NN_)                                                                                   \
  case NN_: {                                                                                       \
    using L = ResidentTile<Phys, NN_, false, true>;                                                 \
    return {reinterpret_cast<const void *>(&k_resident<Phys, NN_, false, 2, true>), L::T, L::EPB, L::NX}; \
  }
    CASE(1) CASE(2) CASE(3) CASE(4)
#undef CASE
    default: return {};
  }
}
ResidentKernel resident_net_kernel(int kind, int N) {
  switch (kind) {
    case SELFAMD_MODEL_SW: return resident_net_of<PhysSW>(N);
    case SELFAMD_MODEL_LSW: return resident_net_of<PhysLSW>(N);
    default: return resident_net_of<PhysEuler>(N);
  }
}
ResidentKernel resident_kernel(int kind, int N, bool nodal, int dense) {
  switch (kind) {
    case SELFAMD_MODEL_SW: return nodal ? resident_of<PhysSW, true>(N, dense) : resident_of<PhysSW, false>(N, dense);
    case SELFAMD_MODEL_LSW: return nodal ? resident_of<PhysLSW, true>(N, dense) : resident_of<PhysLSW, false>(N, dense);
    default: return nodal ? resident_of<PhysEuler, true>(N, dense) : resident_of<PhysEuler, false>(N, dense);
  }
}

}  // namespace

// ------------------------------------------------------------------------------
// Model2D engine
// ------------------------------------------------------------------------------
struct selfamd_model2d {
  int kind = 0, N = 0, nEl = 0, nVar = 0, nT = 0;
  int device = 0;  // the GPU the model's buffers live on (current device at creation)
  hipStream_t stream = nullptr;
  bool ownStream = false;
  double *S = nullptr, *G = nullptr, *trace[2] = {nullptr, nullptr}, *un[2] = {nullptr, nullptr};
  double *geom = nullptr, *mats = nullptr, *aux = nullptr, *stat2 = nullptr, *presTrace = nullptr;
  // per-node metrics (copied from SEMQuad at creation); used when `nodal` is set
  double *ndsdx = nullptr, *nJ = nullptr, *nnHat = nullptr, *nnScale = nullptr;
  bool affine = true, nodal = false;
  bool anyBoundary = false;  // some element side is a physical boundary (neighbour code < 0)
  int32_t *nbr = nullptr;
  int cur = 0;  // trace buffer holding the traces of the current S
  Params p{};
  double t = 0.0;
  // captured one-step graphs, one per starting trace buffer
  hipGraphExec_t graph[2] = {nullptr, nullptr};
  // graphs of 2^k steps (k = 1 .. top_level()), per starting trace buffer, captured (for both
  // buffers) when a call first needs them; 2^k steps flip the trace buffer an even number of
  // times, so the start parity is unchanged after each.  A call replays the largest as often as it fits, then each
  // smaller one at most once and, for an odd count, the one-step graph.  Between two replays
  // the GPU idles ~9 us, a tenth of a stage launch on small meshes.
  static constexpr int kGraphLevels = 7;        // up to 64 steps per graph
  static constexpr int kGraphLevelsBanded = 4;  // banded stepping: up to 8 (many more nodes per step)
  hipGraphExec_t graphP[kGraphLevels][2] = {};
  int top_level() const { return (nBands > 0 ? kGraphLevelsBanded : kGraphLevels) - 1; }
  double graphDt = -1.0;
  int graphEpoch = -1;  // tile table version the graphs were captured with
  ClosureBuffers *closure = nullptr;
  double *intScratch = nullptr;  // partial sums of the state integrals (allocated on first use)
  size_t intScratchLen = 0;
  double *adjTrace = nullptr, *adjChi = nullptr;  // tendency adjoint: traces of its state, neighbour-trace cotangents

  // Banded stepping: the elements split into bands of whole BFS levels of the element graph
  // (neighbours differ by at most one band); one RK3 step runs stage s of band b in round
  // b + s, rounds in order and, within a round, stages in order.  A band's data are then
  // touched three times within ~3 bands' worth of traffic, i.e. while they are still in the
  // Infinity Cache.  Dependencies (neighbour traces of the previous stage in the buffer of
  // that stage's parity, none overwritten before its last reader) hold by this order.
  int nBands = 0;
  int32_t *bandElems = nullptr;   // elements sorted by band
  std::vector<int> bandStart;     // nBands + 1 offsets into bandElems
  std::vector<int32_t> hnbr;      // host copy of the neighbour codes

  // resident stepping: the exchange ring (allocated on first use), the blocks that can be
  // resident at once (-1: not asked yet; 0: not available), the gate and what the launches report
  unsigned long long *ring = nullptr;
  size_t ringLen = 0;
  int ringValues = 0;  // values per face node of the slot layout the ring was emptied for
  int residentBlocks[2][kResidentDense] = {{-1, -1, -1, -1}, {-1, -1, -1, -1}};  // [nodal][dense]
  bool residentSpills[2][kResidentDense] = {};  // whether those instances' registers spill
  int residentNetBlocks = -1;                   // with a closure
  int residentCUs = 0;                          // of the device
  bool paired = false;  // every interior side's neighbour names that side as its own neighbour
  bool stageLaunches = false;  // asked for by the caller
  ResidentGate *gate = nullptr;
  ResidentReport *report = nullptr;
  int polls = kPolls, gatePolls = kGatePolls;
  bool gateReset = false;  // the gate is to be set up before the next launch
  unsigned launches = 0;  // resident launches so far: the last one's number
  int heldOff = 0;        // calls still to take step graphs after a refused launch
  // other models stepping at the same time (company_of)
  std::atomic<bool> unwaited{false};  // steps have been enqueued since the stream was last waited for
  unsigned long long lastCall = 0;
  int joined = 0;
  // Launches that may yet be refused: `count` alike from launch `first` on, which starts from trace
  // buffer `cur`.
  struct Pending {
    unsigned first, count;
    int nSteps, cur;
    double dt;
  };
  std::vector<Pending> pending;
  unsigned started() const { return __atomic_load_n(&report->started, __ATOMIC_RELAXED); }
  bool refused() const { return report && __atomic_load_n(&report->refused, __ATOMIC_RELAXED) != 0; }
  bool timed_out() const { return report && __atomic_load_n(&report->timedOut, __ATOMIC_RELAXED) != 0; }

  FusedArgs stage_args(int traceIn) const {
    FusedArgs a{};
    a.S = S; a.G = G;
    a.traceIn = trace[traceIn];
    a.traceOut = trace[traceIn ^ 1];
    a.unIn = un[traceIn]; a.unOut = un[traceIn ^ 1];
    a.aux = aux; a.stat2 = stat2; a.presTrace = presTrace;
    a.geom = geom; a.nbr = nbr; a.mats = mats; a.nEl = nEl;
    a.ndsdx = ndsdx; a.nJ = nJ; a.nnHat = nnHat; a.nnScale = nnScale;
    a.anyBoundary = anyBoundary;
    a.p = p;
    return a;
  }
  // Whether a call of nSteps steps runs as resident launches: the mesh's blocks are all resident
  // at once, and the stages saved pay for a cooperative launch.
  // Sets the kernel to launch.
  bool resident(int nSteps, ResidentKernel &k);
  bool leaves_room(const ResidentKernel &k) const {
    return (size_t)((nEl + k.elements - 1) / k.elements) * (k.threads / 64) <= (size_t)kCompanyWaves * residentCUs;
  }
  int mass_stride(const ResidentKernel &k) const { return ((nEl + k.elements - 1) / k.elements + 511) & ~511; }
  hipError_t launch_resident(const ResidentKernel &k, int nSteps, double dt);

  hipError_t launch_stage(int mode, int stage, double dt, int traceIn, double *dSdt, int band = -1,
                          double *fluxOut = nullptr, double *fluxDivOut = nullptr) {
    FusedArgs a = stage_args(traceIn);
    a.fluxOut = fluxOut;
    a.fluxDivOut = fluxDivOut;
    if (closure) {
      hipError_t e = closure_evaluate(*closure, S, geom, mats + 2 * (N + 1) * (N + 1) + 2 * (N + 1), N, nVar, 2, nEl,
                                      stream);
      if (e != hipSuccess) return e;
      a.corr = closure->corr;
      a.corrShift = closure->shiftParts;
      a.nShift = closure->nShift;
      a.shiftScale = closure->shiftScale;
    }
    a.dSdt = dSdt;
    if (band >= 0) {
      a.elems = bandElems + bandStart[band];
      a.nEl = bandStart[band + 1] - bandStart[band];
    }
    a.rkA = kRk3A[stage];
    a.rkGdt = kRk3G[stage] * dt;
    a.rkG = kRk3G[stage];
    a.writeG = stage != 2;
    // element order alternates with the trace buffer parity, i.e. from stage to stage
    a.reverse = tile_alternates(kind, N, a.nEl) ? traceIn : 0;
    a.perElemDt = 0;
    switch (kind) {
      case SELFAMD_MODEL_SW: return Launcher<PhysSW>::stage(N, mode, nodal, a, stream);
      case SELFAMD_MODEL_LSW: return Launcher<PhysLSW>::stage(N, mode, nodal, a, stream);
      default: return Launcher<PhysEuler>::stage(N, mode, nodal, a, stream);
    }
  }
  // the state at `src` (S itself: already there) becomes the current one
  hipError_t launch_state_in(const double *src) {
    StateArgs a{};
    a.src = src; a.S = src == S ? nullptr : S; a.trace = trace[cur]; a.un = un[cur]; a.pres = presTrace;
    a.geom = geom; a.nnHat = nodal ? nnHat : nullptr; a.mats = mats; a.nbr = nbr; a.p = p; a.nEl = nEl;
    switch (kind) {
      case SELFAMD_MODEL_SW: return Launcher<PhysSW>::state_in(N, a, stream);
      case SELFAMD_MODEL_LSW: return Launcher<PhysLSW>::state_in(N, a, stream);
      default: return Launcher<PhysEuler>::state_in(N, a, stream);
    }
  }
  void drop_graphs() {
    for (auto &g : graph)
      if (g) { (void)hipGraphExecDestroy(g); g = nullptr; }
    for (auto &lv : graphP)
      for (auto &g : lv)
        if (g) { (void)hipGraphExecDestroy(g); g = nullptr; }
    graphDt = -1.0;
  }
  // captures `steps` RK3 steps starting from trace buffer `start`
  hipError_t capture(int start, int steps, double dt, hipGraphExec_t *out) {
    hipGraph_t g;
    hipError_t e = hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return e;
    int tin = start;
    hipError_t le = hipSuccess;
    for (int n = 0; n < steps; n++) {
      if (nBands > 0) {
        for (int r = 0; r < nBands + 2 && le == hipSuccess; r++)
          for (int st = 0; st < 3 && le == hipSuccess; st++) {
            const int b = r - st;
            if (b >= 0 && b < nBands) le = launch_stage(0, st, dt, tin ^ (st & 1), nullptr, b);
          }
        tin ^= 1;  // three stages
      } else {
        for (int st = 0; st < 3 && le == hipSuccess; st++) {
          le = launch_stage(0, st, dt, tin, nullptr);
          tin ^= 1;
        }
      }
    }
    hipError_t ce = hipStreamEndCapture(stream, &g);
    if (le != hipSuccess) return le;
    if (ce != hipSuccess) return ce;
    hipError_t ie = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    // the graph's first replay would otherwise carry its upload to the device (~25 us at 8
    // steps), inside whatever timed region first needs it
    if (ie == hipSuccess) ie = hipGraphUpload(*out, stream);
    return ie;
  }
  // `steps` RK3 steps launched stage by stage on the stream, without a graph
  hipError_t launch_steps(int steps, double dt) {
    for (int n = 0; n < steps; n++) {
      if (nBands > 0) {
        for (int r = 0; r < nBands + 2; r++)
          for (int st = 0; st < 3; st++) {
            const int b = r - st;
            if (b >= 0 && b < nBands) {
              hipError_t e = launch_stage(0, st, dt, cur ^ (st & 1), nullptr, b);
              if (e != hipSuccess) return e;
            }
          }
        cur ^= 1;
      } else {
        for (int st = 0; st < 3; st++) {
          hipError_t e = launch_stage(0, st, dt, cur, nullptr);
          if (e != hipSuccess) return e;
          cur ^= 1;
        }
      }
      t += dt;
    }
    return hipSuccess;
  }
};

using Model = selfamd_model2d;

namespace {
// The models whose meshes fit the device, and their step calls so far, in one order.
struct SteppingModels {
  std::mutex mutex;
  std::vector<Model *> models;
  unsigned long long calls = 0;
};
SteppingModels &stepping_models() {
  static SteppingModels *const all = new SteppingModels();  // outlives every model
  return *all;
}
// With a step call on m: how many other models of its device step at the same time.  That is those
// with steps enqueued since m's last call and not yet waited for, or, where m comes first in a round of
// calls, those that were enqueued like that beside m's last one.
int company_of(Model *m) {
  SteppingModels &all = stepping_models();
  const std::lock_guard<std::mutex> lock(all.mutex);
  if (m->lastCall == 0) all.models.push_back(m);
  auto beside = [m](const Model *o) {
    return o != m && o->device == m->device && o->unwaited && o->lastCall > m->lastCall;
  };
  const int others = (int)std::count_if(all.models.begin(), all.models.end(), beside);
  for (Model *o : all.models)
    if (beside(o)) o->joined = std::max(o->joined, others);
  const int company = std::max(others, m->joined);
  m->joined = 0;
  m->unwaited = true;
  m->lastCall = ++all.calls;
  return company;
}
hipError_t drain(Model *m) {
  const hipError_t e = hipStreamSynchronize(m->stream);
  if (e == hipSuccess) m->unwaited = false;
  return e;
}
void leave_company(Model *m) {
  SteppingModels &all = stepping_models();
  const std::lock_guard<std::mutex> lock(all.mutex);
  all.models.erase(std::remove(all.models.begin(), all.models.end(), m), all.models.end());
}
}  // namespace

bool selfamd_model2d::resident(int nSteps, ResidentKernel &k) {
  if (nSteps < (nEl < kResidentElements ? kResidentSteps : 1) || nBands > 0 || !paired || stageLaunches || timed_out()) return false;
  if (heldOff > 0) {
    heldOff--;
    return false;
  }
  int current = -1;  // the ring is allocated on the current device
  if (hipGetDevice(&current) != hipSuccess || current != device) return false;
  // the 64-wide tile of nonlinear SW at N = 5 splits the face sums; the resident kernel does not
  if (kind == SELFAMD_MODEL_SW && N == 5 && tile_splits5(tile_of(kind, 5))) return false;
  // whether the device holds k's blocks at once; their number and whether k spills are asked once
  auto capacity = [&](int &blocks, bool &spills) {
    if (blocks < 0) {
      int cus = 0, perCU = 0, coop = 0;
      if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
          hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess ||
          hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, k.fn, k.threads, 0) != hipSuccess) {
        (void)hipGetLastError();
        perCU = 0;
      }
      hipFuncAttributes at{};
      if (hipFuncGetAttributes(&at, k.fn) != hipSuccess) {
        (void)hipGetLastError();
        perCU = 0;
      }
      residentCUs = cus;
      spills = at.localSizeBytes > 0;
      blocks = coop ? cus * perCU : 0;
      // Euler at N = 2 on a full device: 3,060 blocks 17.1 us per stage, in launches 15.9; 2,600 blocks
      // 10.2 and 14.1
      if (kind == SELFAMD_MODEL_EULER && N == 2) blocks -= blocks / 8;
    }
    if (spills && !closure && nSteps < kResidentSpillSteps) return false;  // a closure's launch pays from one step on
    return (nEl + k.elements - 1) / k.elements <= blocks;
  };
  bool fits = false;
  if (closure) {
    bool netSpills = false;
    k = resident_net_kernel(kind, N);
    const MlpWeights w = mlp_weights(closure->mlp);
    fits = k.fn && !nodal && w.rows && w.nH <= kResidentHidden && capacity(residentNetBlocks, netSpills);
  } else {
    for (int dense = 0; dense < kResidentDense && !fits; dense++) {
      k = resident_kernel(kind, N, nodal, dense);
      fits = k.fn && capacity(residentBlocks[nodal][dense], residentSpills[nodal][dense]);
    }
  }
  if (!fits) return false;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return false;
  }
  const size_t len = 3 * ((size_t)(N + 1) * k.values * 4 * nEl + (closure ? (size_t)kMassCopies * mass_stride(k) : 0));
  if (ringLen < len) {
    if (ring) (void)hipFree(ring);
    ring = nullptr;
    ringLen = 0;
    if (!report) {
      if (hipHostMalloc(&report, sizeof(ResidentReport), hipHostMallocDefault) != hipSuccess) {
        report = nullptr;
        (void)hipGetLastError();
        return false;
      }
      *report = {0, launches, 0};
    }
    if (!gate) {
      if (hipMalloc(&gate, sizeof(ResidentGate)) != hipSuccess) {
        gate = nullptr;
        (void)hipGetLastError();
        return false;
      }
      gateReset = true;
    }
    if (hipMalloc(&ring, sizeof(unsigned long long) * len) != hipSuccess) {
      ring = nullptr;
      (void)hipGetLastError();
      return false;
    }
    ringLen = len;
    ringValues = 0;
  }
  if (ringValues != k.values) {  // first use, or the metric mode (and with it the slot layout) changed
    hipLaunchKernelGGL(k_ring_fill, (unsigned)std::min<size_t>((ringLen + 255) / 256, 4096), 256, 0, stream, ring, ringLen);
    if (hipGetLastError() != hipSuccess) return false;
    ringValues = k.values;
  }
  if (gateReset) {
    hipLaunchKernelGGL(k_gate_reset, 1, kGateGroups, 0, stream, gate, launches, report, polls, gatePolls);
    if (hipGetLastError() != hipSuccess) return false;
    gateReset = false;
  }
  return true;
}

hipError_t selfamd_model2d::launch_resident(const ResidentKernel &k, int nSteps, double dt) {
  FusedArgs a = stage_args(cur);
  const int end = cur ^ (nSteps & 1);  // the trace buffer after 3 nSteps stages
  a.traceOut = trace[end];
  a.unOut = un[end];
  ResidentArgs ra{};
  ra.ring = ring;
  ra.stages = 3 * nSteps;
  for (int q = 0; q < 3; q++) {
    ra.rkA[q] = kRk3A[q];
    ra.rkGdt[q] = kRk3G[q] * dt;
  }
  ra.gate = gate;
  ResidentNetArgs na{};
  if (closure) {
    na.w = mlp_weights(closure->mlp);
    na.inMean = closure->inMean; na.inScale = closure->inScale;
    na.outMean = closure->outMean; na.outScale = closure->outScale;
    na.shiftScale = closure->invArea;
    na.mass = ring + 3 * (size_t)(N + 1) * k.values * 4 * nEl;
    na.massStride = mass_stride(k);
  }
  void *args[] = {&a, &ra, &na};
  const hipError_t e = hipLaunchCooperativeKernel(k.fn, dim3((nEl + k.elements - 1) / k.elements), dim3(k.threads), args, 0, stream);
  if (e != hipSuccess) return e;
  launches++;
  const unsigned in = started();
  pending.erase(pending.begin(), std::find_if(pending.begin(), pending.end(), [in](const Pending &p) {
    return (int)(in - (p.first + p.count - 1)) < 0;
  }));
  if (!pending.empty() && pending.back().nSteps == nSteps && pending.back().dt == dt) pending.back().count++;
  else pending.push_back({launches, 1, nSteps, cur, dt});
  cur = end;
  for (int q = 0; q < nSteps; q++) t += dt;
  return hipSuccess;
}

namespace {
void free_closure(ClosureBuffers *c) {
  if (!c) return;
  void *bufs[] = {c->X,    c->Y,     c->inMean, c->inScale, c->outMean,   c->outScale,
                  c->corr, c->elemMass, c->shift, c->dY,      c->dX,        c->vjpPartial};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  delete c;
}
}  // namespace

extern "C" {

int selfamd_model2d_nvar(int kind) { return kind == SELFAMD_MODEL_EULER ? 4 : 3; }

int selfamd_model2d_create(selfamd_model2d **out, int kind, int N, int nEl, const int32_t *sideInfo,
                           const double *dsdx, const double *J, const double *nHatb, const double *nScaleb,
                           void *stream) {
  SELFAMD_REQUIRE(out, "model2d_create: null output handle");
  *out = nullptr;
  SELFAMD_REQUIRE(kind == SELFAMD_MODEL_LSW || kind == SELFAMD_MODEL_SW || kind == SELFAMD_MODEL_EULER,
                  "model2d_create: unknown model kind %d", kind);
  SELFAMD_REQUIRE(N >= 1 && N <= 7, "model2d_create: fused kernels cover 1 <= N <= 7 (got %d)", N);
  SELFAMD_REQUIRE(nEl >= 1, "model2d_create: nEl=%d", nEl);
  SELFAMD_REQUIRE(sideInfo && dsdx && J && nHatb && nScaleb, "model2d_create: null geometry/connectivity");
  const int P = N + 1, PP = P * P;
  // neighbour codes from sideInfo (validated: bit-exact copy of the connectivity)
  std::vector<int32_t> nbr((size_t)4 * nEl);
  for (int e = 0; e < nEl; e++)
    for (int s = 0; s < 4; s++) {
      const int32_t *si = sideInfo + 5 * (s + 4 * (size_t)e);
      const int e2 = si[2], bcid = si[4];
      int code;
      if (bcid == 0) {
        const int s2 = si[3] / 10, flip = si[3] - 10 * s2;
        SELFAMD_REQUIRE(e2 >= 1 && e2 <= nEl && s2 >= 1 && s2 <= 4 && (flip == 0 || flip == 1),
                        "model2d_create: bad interior side (elem %d side %d): e2=%d s2=%d flip=%d", e + 1, s + 1,
                        e2, s2, flip);
        SELFAMD_REQUIRE(e2 - 1 < (1 << 27), "model2d_create: too many elements");
        code = ((e2 - 1) << 3) | ((s2 - 1) << 1) | flip;
      } else if (e2 == 0) {
        code = -bcid - 1;
      } else {
        code = kNbrOrphan;  // periodic-tagged HOPr side: never exchanged, ext state stays 0
      }
      nbr[4 * (size_t)e + s] = code;
    }
  // per-element affine geometry records
  const size_t nn = (size_t)PP * nEl, nb = (size_t)P * 4 * nEl;
  std::vector<double> hdsdx(4 * nn), hJ(nn), hn(2 * nb), hs(nb);
  SELFAMD_HIP(hipMemcpy(hdsdx.data(), dsdx, sizeof(double) * 4 * nn, hipMemcpyDeviceToHost));
  SELFAMD_HIP(hipMemcpy(hJ.data(), J, sizeof(double) * nn, hipMemcpyDeviceToHost));
  SELFAMD_HIP(hipMemcpy(hn.data(), nHatb, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost));
  SELFAMD_HIP(hipMemcpy(hs.data(), nScaleb, sizeof(double) * nb, hipMemcpyDeviceToHost));
  // Per-element affine records: metric terms constant over each element up to round-off use
  // one record; otherwise the nodal metrics are used.  The round-off of a derivative of
  // interpolated coordinates grows like (coordinate magnitude / element size) x eps: on the
  // unit square it is ~3e-12 relative at 64 x 64 elements, ~1e-11 at 256 x 256 and ~2e-11 at
  // 512 x 512, so the tolerance is 1e-10 (meshes up to ~2048 elements across).
  constexpr double kAffineTol = 1e-10;
  std::vector<double> rec((size_t)kGeomStride * nEl, 0.0);
  bool affine = true;
  for (int e = 0; e < nEl && affine; e++) {
    double *r = rec.data() + (size_t)kGeomStride * e;
    const double *d0 = hdsdx.data() + 4 * (size_t)PP * e;
    double scale = 0.0;
    for (int k = 0; k < 4; k++) { r[k] = d0[k]; scale = std::fmax(scale, std::fabs(d0[k])); }
    r[4] = hJ[(size_t)PP * e];
    r[6] = 1.0 / r[4];
    for (int n = 0; n < PP && affine; n++) {
      for (int k = 0; k < 4; k++)
        if (std::fabs(d0[4 * n + k] - r[k]) > kAffineTol * scale) affine = false;
      if (std::fabs(hJ[(size_t)PP * e + n] - r[4]) > kAffineTol * std::fabs(r[4])) affine = false;
    }
    for (int s = 0; s < 4 && affine; s++) {
      const size_t b0 = (size_t)P * (s + 4 * (size_t)e);
      r[8 + s] = hn[2 * b0];
      r[12 + s] = hn[2 * b0 + 1];
      r[16 + s] = hs[b0];
      for (int i = 1; i < P; i++)
        if (std::fabs(hn[2 * (b0 + i)] - r[8 + s]) > kAffineTol || std::fabs(hn[2 * (b0 + i) + 1] - r[12 + s]) > kAffineTol ||
            std::fabs(hs[b0 + i] - r[16 + s]) > kAffineTol * std::fabs(r[16 + s]))
          affine = false;
    }
  }
  // Lagrange matrices on Gauss points
  double cp[8], tp[8], bw[8], qw[8], iM[64], dM[64], dgM[64], bM[16];
  int rc = selfamd_lagrange_init(N, SELFAMD_GAUSS, N, SELFAMD_GAUSS, cp, tp, bw, qw, iM, dM, dgM, bM);
  if (rc) return rc;
  std::vector<double> mats(2 * PP + 4 * P);
  for (int k = 0; k < PP; k++) { mats[k] = dgM[k]; mats[PP + k] = dM[k]; }
  for (int k = 0; k < 2 * P; k++) mats[2 * PP + k] = bM[k];
  for (int k = 0; k < P; k++) mats[2 * PP + 2 * P + k] = qw[k];
  for (int k = 0; k < P; k++) mats[2 * PP + 3 * P + k] = 1.0 / qw[k];

  Model *m = new Model();
  m->kind = kind; m->N = N; m->nEl = nEl;
  m->hnbr = nbr;
  m->paired = nEl < (1 << 27);
  for (int e = 0; e < nEl && m->paired; e++)
    for (int sd = 0; sd < 4; sd++) {
      const int c = nbr[4 * (size_t)e + sd];
      if (c >= 0 && nbr[4 * (size_t)(c >> 3) + ((c >> 1) & 3)] != ((e << 3) | (sd << 1) | (c & 1))) m->paired = false;
    }
  m->anyBoundary = std::any_of(nbr.begin(), nbr.end(), [](int32_t c) { return c < 0; });
  m->affine = affine;
  m->nodal = !affine;
  m->nVar = selfamd_model2d_nvar(kind);
  m->nT = kind == SELFAMD_MODEL_EULER ? 9 : 3;
  m->p.g = 1.0; m->p.fCori = 0.0; m->p.gamma = 1.4; m->p.Rgas = 1.0;
  m->p.auxConst = 0.0;  // static fields default to zero until a Set* call provides them
  m->p.stat2Const = 0.0;
  auto fail = [&](int code) { selfamd_model2d_destroy(m); return code; };
  if (hipGetDevice(&m->device) != hipSuccess) {
    set_error("model2d_create: hipGetDevice failed");
    return fail(kHipError);
  }
  if (stream) {
    m->stream = reinterpret_cast<hipStream_t>(stream);
  } else {
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
      set_error("model2d_create: hipStreamCreate failed");
      return fail(kHipError);
    }
    m->ownStream = true;
  }
  const size_t nS = nn * m->nVar, nT = (size_t)P * m->nT * 4 * nEl;
  if (hipMalloc(&m->S, sizeof(double) * nS) != hipSuccess || hipMalloc(&m->G, sizeof(double) * nS) != hipSuccess ||
      hipMalloc(&m->trace[0], sizeof(double) * nT) != hipSuccess ||
      hipMalloc(&m->trace[1], sizeof(double) * nT) != hipSuccess ||
      hipMalloc(&m->geom, sizeof(double) * rec.size()) != hipSuccess ||
      hipMalloc(&m->mats, sizeof(double) * mats.size()) != hipSuccess ||
      hipMalloc(&m->nbr, sizeof(int32_t) * nbr.size()) != hipSuccess ||
      hipMalloc(&m->ndsdx, sizeof(double) * 4 * nn) != hipSuccess || hipMalloc(&m->nJ, sizeof(double) * nn) != hipSuccess ||
      hipMalloc(&m->nnHat, sizeof(double) * 2 * nb) != hipSuccess ||
      hipMalloc(&m->nnScale, sizeof(double) * nb) != hipSuccess) {
    set_error("model2d_create: device allocation failed (%zu doubles of state)", nS);
    return fail(kHipError);
  }
  // lagged velocities: room for the nodal mode's vectors (2 doubles per face node)
  if (kind == SELFAMD_MODEL_SW && (hipMalloc(&m->un[0], sizeof(double) * 2 * (size_t)P * 4 * nEl) != hipSuccess ||
                                   hipMalloc(&m->un[1], sizeof(double) * 2 * (size_t)P * 4 * nEl) != hipSuccess)) {
    set_error("model2d_create: device allocation failed (un)");
    return fail(kHipError);
  }
  if (hipMemcpy(m->geom, rec.data(), sizeof(double) * rec.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(m->mats, mats.data(), sizeof(double) * mats.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(m->nbr, nbr.data(), sizeof(int32_t) * nbr.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(m->ndsdx, dsdx, sizeof(double) * 4 * nn, hipMemcpyDeviceToDevice) != hipSuccess ||
      hipMemcpy(m->nJ, J, sizeof(double) * nn, hipMemcpyDeviceToDevice) != hipSuccess ||
      hipMemcpy(m->nnHat, nHatb, sizeof(double) * 2 * nb, hipMemcpyDeviceToDevice) != hipSuccess ||
      hipMemcpy(m->nnScale, nScaleb, sizeof(double) * nb, hipMemcpyDeviceToDevice) != hipSuccess ||
      hipMemsetAsync(m->S, 0, sizeof(double) * nS, m->stream) != hipSuccess ||
      hipMemsetAsync(m->G, 0, sizeof(double) * nS, m->stream) != hipSuccess ||
      hipMemsetAsync(m->trace[0], 0, sizeof(double) * nT, m->stream) != hipSuccess ||
      hipMemsetAsync(m->trace[1], 0, sizeof(double) * nT, m->stream) != hipSuccess ||
      (m->un[0] && hipMemsetAsync(m->un[0], 0, sizeof(double) * 2 * (size_t)P * 4 * nEl, m->stream) != hipSuccess) ||
      (m->un[1] && hipMemsetAsync(m->un[1], 0, sizeof(double) * 2 * (size_t)P * 4 * nEl, m->stream) != hipSuccess) ||
      hipStreamSynchronize(nullptr) != hipSuccess ||  // copies into device memory may still be under way
      hipStreamSynchronize(m->stream) != hipSuccess) {
    set_error("model2d_create: device initialisation failed");
    return fail(kHipError);
  }
  *out = m;
  return kOk;
}

int selfamd_model2d_destroy(selfamd_model2d *m) {
  if (!m) return kOk;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  m->drop_graphs();
  free_closure(m->closure);
  double *bufs[] = {m->S,    m->G,    m->trace[0], m->trace[1], m->un[0], m->un[1], m->geom,  m->mats,
                    m->aux,  m->stat2, m->presTrace, m->ndsdx, m->nJ,    m->nnHat, m->nnScale};
  if (m->bandElems) (void)hipFree(m->bandElems);
  if (m->ring) (void)hipFree(m->ring);
  leave_company(m);
  if (m->gate) (void)hipFree(m->gate);
  if (m->report) (void)hipHostFree(m->report);
  if (m->intScratch) (void)hipFree(m->intScratch);
  if (m->adjTrace) (void)hipFree(m->adjTrace);
  if (m->adjChi) (void)hipFree(m->adjChi);
  for (double *b : bufs)
    if (b) (void)hipFree(b);
  if (m->nbr) (void)hipFree(m->nbr);
  if (m->ownStream && m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return kOk;
}

namespace {
int step_graphs(selfamd_model2d *m, int nSteps, double dt);

// after the model's stream has been waited for
int resident_status(const selfamd_model2d *m) {
  SELFAMD_REQUIRE(!m->timed_out(),
                  "model2d: a resident launch gave up waiting for a neighbour's traces; the state is not valid");
  return kOk;
}

// With the model's stream waited for: the steps of a refused launch and of those after it, by step
// graphs.  Nothing of the model has changed since it was refused.
int take_refused_steps(selfamd_model2d *m) {
  std::vector<selfamd_model2d::Pending> todo;
  todo.swap(m->pending);
  if (!m->refused()) return kOk;
  const unsigned first = m->report->refused;
  m->report->refused = 0;
  m->gateReset = true;
  m->heldOff = kHeldOffCalls;
  const double t = m->t;  // has counted these steps
  bool taken = false;
  for (const auto &p : todo) {
    for (unsigned k = 0; k < p.count; k++) {
      if ((int)(p.first + k - first) < 0) continue;
      if (!taken) m->cur = p.cur ^ (p.nSteps & (int)k & 1);
      taken = true;
      if (const int status = step_graphs(m, p.nSteps, p.dt)) return status;
    }
  }
  m->t = t;
  SELFAMD_HIP(drain(m));
  return kOk;
}

// Waits for the model's stream; the steps that were asked for have been taken when it returns.
int wait_for(selfamd_model2d *m) {
  SELFAMD_HIP(drain(m));
  if (!m->pending.empty())
    if (const int status = take_refused_steps(m)) return status;
  return resident_status(m);
}

// Before other work on the state, and before anything that the steps depend on changes: every
// resident launch has been let in (which a launch on an idle device is some us after the call), or the
// steps have been taken.
int settle(selfamd_model2d *m) {
  if (m->pending.empty()) return kOk;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  SELFAMD_HIP(hipStreamIsCapturing(m->stream, &capturing));
  const bool captured = capturing != hipStreamCaptureStatusNone;  // since the launch: not to be waited for
  const auto until = std::chrono::steady_clock::now() +
                     (captured ? std::chrono::microseconds(60'000'000) : std::chrono::microseconds(200));
  while (m->started() != m->launches && !m->refused() && std::chrono::steady_clock::now() < until) {}
  if (m->started() == m->launches) {
    m->pending.clear();
    return kOk;
  }
  SELFAMD_REQUIRE(!captured, "model2d: steps before the capture have not been taken; wait for the model before its "
                             "stream is captured");
  SELFAMD_HIP(drain(m));
  return take_refused_steps(m);
}
#define SELFAMD_SETTLE(m)                              \
  do {                                                 \
    if (const int status_ = settle(m)) return status_; \
  } while (0)

// A valid state has been stored, after all pending steps, and the stream waited for.
void state_replaced(selfamd_model2d *m) {
  m->pending.clear();
  if (m->refused()) {
    m->report->refused = 0;
    m->gateReset = true;
  }
  if (m->timed_out()) {
    m->report->timedOut = 0;
    m->ringValues = 0;  // the exchange ring is emptied before its next use
  }
}
}  // namespace

int selfamd_model2d_set_param(selfamd_model2d *m, int which, double value) {
  SELFAMD_REQUIRE(m, "model2d_set_param: null model");
  SELFAMD_SETTLE(m);
  switch (which) {
    case SELFAMD_PARAM_G: m->p.g = value; break;
    case SELFAMD_PARAM_FCORI: m->p.fCori = value; break;
    case SELFAMD_PARAM_GAMMA: m->p.gamma = value; break;
    case SELFAMD_PARAM_RGAS: m->p.Rgas = value; break;
    case SELFAMD_PARAM_NODAL_METRICS:
      SELFAMD_REQUIRE(value != 0.0 || m->affine, "model2d_set_param: the mesh is not affine; nodal metrics required");
      if (m->nodal != (value != 0.0) && m->kind == SELFAMD_MODEL_SW) {
        // the two modes keep the SW velocity lag in different layouts: restart it from the
        // current traces, as SetSolution does
        m->nodal = value != 0.0;
        SELFAMD_HIP(launch_un_init(m->N, m->trace[m->cur], m->un[m->cur], m->geom, m->nodal ? m->nnHat : nullptr,
                                   m->nEl, m->stream));
        SELFAMD_HIP(drain(m));
      }
      m->nodal = value != 0.0;
      break;
    case SELFAMD_PARAM_POLLS:
    case SELFAMD_PARAM_GATE_POLLS:
      SELFAMD_REQUIRE(value >= 0.0 && value <= 2147483647.0, "model2d_set_param: %g polls", value);
      (which == SELFAMD_PARAM_POLLS ? m->polls : m->gatePolls) = (int)value;
      m->gateReset = m->gate != nullptr;
      return kOk;
    case SELFAMD_PARAM_STAGE_LAUNCHES: m->stageLaunches = value != 0.0; return kOk;
    default: SELFAMD_REQUIRE(false, "model2d_set_param: unknown parameter %d", which);
  }
  m->drop_graphs();
  return kOk;
}

int selfamd_model2d_set_field(selfamd_model2d *m, int which, const double *field) {
  SELFAMD_REQUIRE(m && field, "model2d_set_field: null argument");
  const size_t n = (size_t)(m->N + 1) * (m->N + 1) * m->nEl;
  double **slot = nullptr;
  if ((which == SELFAMD_FIELD_TOPOGRAPHY && m->kind == SELFAMD_MODEL_SW) ||
      (which == SELFAMD_FIELD_BATHYMETRY && m->kind == SELFAMD_MODEL_LSW) ||
      (which == SELFAMD_FIELD_POTENTIAL && m->kind == SELFAMD_MODEL_EULER))
    slot = &m->aux;
  else if ((which == SELFAMD_FIELD_CORIOLIS && m->kind == SELFAMD_MODEL_LSW) ||
           (which == SELFAMD_FIELD_DRAG && m->kind == SELFAMD_MODEL_EULER))
    slot = &m->stat2;
  SELFAMD_REQUIRE(slot, "model2d_set_field: field %d does not apply to model kind %d", which, m->kind);
  SELFAMD_SETTLE(m);
  if (!*slot) SELFAMD_HIP(hipMalloc(slot, sizeof(double) * n));
  SELFAMD_HIP(hipMemcpyAsync(*slot, field, sizeof(double) * n, hipMemcpyDeviceToDevice, m->stream));
  SELFAMD_HIP(drain(m));
  m->drop_graphs();
  return kOk;
}

int selfamd_model2d_set_solution(selfamd_model2d *m, const double *interior) {
  SELFAMD_REQUIRE(m && interior, "model2d_set_solution: null argument");
  const size_t n = (size_t)(m->N + 1) * (m->N + 1) * m->nVar * m->nEl;
  const Source from = source_of(interior, sizeof(double) * n, sizeof(double), m->device);
  SELFAMD_REQUIRE(from != Source::kShort, "model2d_set_solution: the array holds less than the state's %zu bytes",
                  sizeof(double) * n);
  if (m->kind == SELFAMD_MODEL_EULER && !m->presTrace) {
    // prescribed boundary state := traces of this state (SetPrescribedSolutionFromSolution)
    SELFAMD_HIP(hipMalloc(&m->presTrace, sizeof(double) * (size_t)(m->N + 1) * 9 * 4 * m->nEl));
    m->drop_graphs();  // captured without it
  }
  const bool direct = from == Source::kKernel;
  if (!direct) SELFAMD_HIP(hipMemcpyAsync(m->S, interior, sizeof(double) * n, hipMemcpyDeviceToDevice, m->stream));
  SELFAMD_HIP(m->launch_state_in(direct ? interior : m->S));
  SELFAMD_HIP(drain(m));
  state_replaced(m);
  return kOk;
}

int selfamd_model2d_get_solution(selfamd_model2d *m, double *interior) {
  SELFAMD_REQUIRE(m && interior, "model2d_get_solution: null argument");
  SELFAMD_SETTLE(m);
  const size_t n = (size_t)(m->N + 1) * (m->N + 1) * m->nVar * m->nEl;
  SELFAMD_HIP(hipMemcpyAsync(interior, m->S, sizeof(double) * n, hipMemcpyDeviceToDevice, m->stream));
  SELFAMD_HIP(drain(m));
  return resident_status(m);
}

// integral of the current state over the mesh (the integrand kind, and the variable for
// kIntVariable); synchronises the model's stream
static int model_integral(selfamd_model2d *m, int what, int var, double *value, const char *who) {
  SELFAMD_SETTLE(m);
  const size_t PP = (size_t)(m->N + 1) * (m->N + 1), nNodes = PP * m->nEl;
  const int nBlocks = (int)((nNodes + kIntBlock - 1) / kIntBlock);
  if (m->intScratchLen < (size_t)nBlocks + 1) {
    if (m->intScratch) SELFAMD_HIP(hipFree(m->intScratch));
    m->intScratch = nullptr;
    m->intScratchLen = 0;
    if (hipMalloc(&m->intScratch, sizeof(double) * (nBlocks + 1)) != hipSuccess) {
      set_error("%s: device allocation failed", who);
      return kHipError;
    }
    m->intScratchLen = (size_t)nBlocks + 1;
  }
  const double *qW = m->mats + 2 * PP + 2 * (m->N + 1);
  switch (what) {
#define INT_CASE(W)                                                                                        \
  case W:                                                                                                 \
    hipLaunchKernelGGL((k_integral_partial<W>), dim3(nBlocks), dim3(kIntBlock), 0, m->stream, m->S, m->aux, \
                       m->nJ, qW, m->p, m->N, m->nVar, var, nNodes, m->intScratch);                         \
    break;
    INT_CASE(kIntSWEntropy) INT_CASE(kIntLSWEntropy) INT_CASE(kIntEulerEntropy) INT_CASE(kIntVariable)
#undef INT_CASE
    default: set_error("%s: unknown integral", who); return kBadArgument;
  }
  SELFAMD_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kIntBlock), 0, m->stream, m->intScratch, nBlocks,
                     m->intScratch + nBlocks);
  SELFAMD_CHECK_LAUNCH();
  SELFAMD_HIP(hipMemcpyAsync(value, m->intScratch + nBlocks, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  SELFAMD_HIP(drain(m));
  return resident_status(m);
}

namespace {
// Partial sums of selfamd_model2d_integral_noalloc: one per block of kIntBlock nodes, then the
// total.  A file-scope device array, so that entry point allocates nothing; every GPU that runs
// it holds its own copy (512 KiB) until the process ends.  Host code must not pass `scratch`
// itself to a kernel (in host code the name is a host-side stand-in): it uses the device
// address that scratch_address() looks up once per device.
constexpr int kNoAllocPartials = 65536;  // meshes of up to 65536 * 256 = 16,777,216 nodes
__device__ __align__(256) double scratch[kNoAllocPartials + 1];
constexpr int kMaxDevices = 64;
double *g_scratchDev[kMaxDevices] = {};
std::mutex g_scratchMutex;

// device address of `scratch` on device `dev`, which must be the current device
hipError_t scratch_address(int dev, double **out) {
  std::lock_guard<std::mutex> lock(g_scratchMutex);
  if (!g_scratchDev[dev]) {
    void *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratchDev[dev] = static_cast<double *>(ptr);
  }
  *out = g_scratchDev[dev];
  return hipSuccess;
}
}  // namespace

int selfamd_model2d_integral_noalloc(selfamd_model2d *m, int var, double *value) {
  SELFAMD_REQUIRE(m && value, "model2d_integral_noalloc: null argument");
  SELFAMD_REQUIRE(var >= 0 && var < m->nVar, "model2d_integral_noalloc: variable %d out of range (nVar = %d)", var,
                  m->nVar);
  const size_t PP = (size_t)(m->N + 1) * (m->N + 1), nNodes = PP * m->nEl;
  const size_t nBlocks = (nNodes + kIntBlock - 1) / kIntBlock;
  SELFAMD_REQUIRE(nBlocks <= (size_t)kNoAllocPartials,
                  "model2d_integral_noalloc: the mesh has %zu nodes; this entry point takes at most %zu "
                  "(use selfamd_model2d_integral)", nNodes, (size_t)kNoAllocPartials * kIntBlock);
  int dev = -1;
  SELFAMD_HIP(hipGetDevice(&dev));
  SELFAMD_REQUIRE(dev == m->device, "model2d_integral_noalloc: the model lives on device %d, the current device is %d",
                  m->device, dev);
  SELFAMD_REQUIRE(dev >= 0 && dev < kMaxDevices, "model2d_integral_noalloc: device %d out of range", dev);
  SELFAMD_SETTLE(m);
  double *part = nullptr;
  SELFAMD_HIP(scratch_address(dev, &part));
  // every block writes its own partial sum, so nothing in the array needs clearing first
  const double *qW = m->mats + 2 * PP + 2 * (m->N + 1);
  hipLaunchKernelGGL((k_integral_partial<kIntVariable>), dim3((unsigned)nBlocks), dim3(kIntBlock), 0, m->stream, m->S,
                     m->aux, m->nJ, qW, m->p, m->N, m->nVar, var, nNodes, part);
  SELFAMD_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kIntBlock), 0, m->stream, part, (int)nBlocks, value);
  SELFAMD_CHECK_LAUNCH();
  return kOk;
}

int selfamd_model2d_entropy(selfamd_model2d *m, double *entropy) {
  SELFAMD_REQUIRE(m && entropy, "model2d_entropy: null argument");
  const int what = m->kind == SELFAMD_MODEL_SW ? kIntSWEntropy
                   : m->kind == SELFAMD_MODEL_LSW ? kIntLSWEntropy : kIntEulerEntropy;
  return model_integral(m, what, 0, entropy, "model2d_entropy");
}

int selfamd_model2d_integral(selfamd_model2d *m, int var, double *value) {
  SELFAMD_REQUIRE(m && value, "model2d_integral: null argument");
  SELFAMD_REQUIRE(var >= 0 && var < m->nVar, "model2d_integral: variable %d out of range (nVar = %d)", var, m->nVar);
  return model_integral(m, kIntVariable, var, value, "model2d_integral");
}

int selfamd_model2d_tendency(selfamd_model2d *m, double *dSdt) {
  SELFAMD_REQUIRE(m && dSdt, "model2d_tendency: null argument");
  SELFAMD_SETTLE(m);
  SELFAMD_HIP(m->launch_stage(1, 0, 0.0, m->cur, dSdt));
  if (m->un[0]) {
    // the evaluation's velocities become the lag state of the next stage
    SELFAMD_HIP(hipMemcpyAsync(m->un[m->cur], m->un[m->cur ^ 1],
                               sizeof(double) * (m->nodal ? 2 : 1) * (m->N + 1) * 4 * (size_t)m->nEl,
                               hipMemcpyDeviceToDevice, m->stream));
  }
  SELFAMD_HIP(drain(m));
  return resident_status(m);
}

int selfamd_model2d_flux_registers(selfamd_model2d *m, double *fluxDivergence, double *flux) {
  SELFAMD_REQUIRE(m && fluxDivergence && flux, "model2d_flux_registers: null argument");
  SELFAMD_SETTLE(m);
  // a tendency evaluation of the current state that keeps the lag state and writes no dSdt
  // register of the caller's (the model's own buffer takes it)
  double *scratch = nullptr;
  const size_t n = (size_t)(m->N + 1) * (m->N + 1) * m->nVar * m->nEl;
  SELFAMD_HIP(hipMalloc(&scratch, sizeof(double) * n));
  hipError_t e = m->launch_stage(1, 0, 0.0, m->cur, scratch, -1, flux, fluxDivergence);
  if (e == hipSuccess) e = drain(m);
  (void)hipFree(scratch);
  SELFAMD_HIP(e);
  return resident_status(m);
}

namespace {
// a few steps of another size than the captured graphs' (e.g. ForwardStep's shorter last step
// up to tn) are launched directly, so the graphs of the running step size survive
bool direct_steps(const selfamd_model2d *m, int nSteps, double dt) {
  return m->graphDt > 0.0 && m->graphDt != dt && m->graphEpoch == g_tileEpoch && nSteps <= kDirectSteps;
}
// captures the graphs that nSteps steps of size dt from the current trace buffer replay
hipError_t prepare_graphs(selfamd_model2d *m, int nSteps, double dt) {
  if (nSteps == 0 || direct_steps(m, nSteps, dt)) return hipSuccess;
  if (m->graphDt != dt || m->graphEpoch != g_tileEpoch) {
    m->drop_graphs();
    for (int start = 0; start < 2; start++) {
      hipError_t e = m->capture(start, 1, dt, &m->graph[start]);
      if (e != hipSuccess) return e;
    }
    m->graphDt = dt;
    m->graphEpoch = g_tileEpoch;
  }
  // the 2^k-step graphs of nSteps' decomposition (they keep the current buffer), for both
  // starting buffers, so that a later call of the same size finds them whichever is current
  const int top = m->top_level();
  int rem = nSteps;
  for (int k = top; k >= 1; k--) {
    const int s = 1 << k;
    if (rem < s) continue;
    for (int start = 0; start < 2; start++)
      if (!m->graphP[k][start]) {
        const hipError_t e = m->capture(start, s, dt, &m->graphP[k][start]);
        if (e != hipSuccess) return e;
      }
    rem = k == top ? rem % s : rem - s;
  }
  return hipSuccess;
}
}  // namespace

int selfamd_model2d_forward_step(selfamd_model2d *m, int nSteps, double dt) {
  SELFAMD_REQUIRE(m && nSteps >= 0 && dt > 0.0, "model2d_forward_step: bad arguments (nSteps=%d dt=%g)", nSteps, dt);
  if (nSteps == 0) return kOk;
  if (m->refused()) SELFAMD_SETTLE(m);
  ResidentKernel kernel;
  if (m->resident(nSteps, kernel) && (company_of(m) < kCompany || !m->leaves_room(kernel))) {
    hipError_t e = hipSuccess;
    while (e == hipSuccess && nSteps > 0) {
      const int n = std::min(nSteps, m->leaves_room(kernel) ? kResidentLaunchSteps : kResidentFullSteps);
      e = m->launch_resident(kernel, n, dt);
      if (e == hipSuccess) nSteps -= n;
    }
    if (nSteps == 0) {
      // The network may change next, in stream order: its steps are under way, or taken, first.
      if (m->closure) SELFAMD_SETTLE(m);
      return kOk;
    }
    // not accepted by the runtime: step graphs from here on
    (void)hipGetLastError();
    for (auto &blocks : m->residentBlocks)
      for (int &b : blocks) b = 0;
    m->residentNetBlocks = 0;
  }
  SELFAMD_SETTLE(m);
  return step_graphs(m, nSteps, dt);
}

namespace {
int step_graphs(selfamd_model2d *m, int nSteps, double dt) {
  if (direct_steps(m, nSteps, dt)) {
    SELFAMD_HIP(m->launch_steps(nSteps, dt));
    return kOk;
  }
  SELFAMD_HIP(prepare_graphs(m, nSteps, dt));
  const int top = m->top_level();
  int n = nSteps;
  for (int k = top; k >= 1; k--) {
    const int s = 1 << k;
    while (n >= s) {
      SELFAMD_HIP(hipGraphLaunch(m->graphP[k][m->cur], m->stream));  // 3s stage flips: parity unchanged
      for (int q = 0; q < s; q++) m->t += dt;
      n -= s;
      if (k != top) break;
    }
  }
  if (n == 1) {
    SELFAMD_HIP(hipGraphLaunch(m->graph[m->cur], m->stream));
    m->cur ^= 1;  // three stages flip the trace buffer three times
    m->t += dt;
  }
  return kOk;
}
}  // namespace

int selfamd_model2d_synchronize(selfamd_model2d *m) {
  SELFAMD_REQUIRE(m, "model2d_synchronize: null model");
  return wait_for(m);
}

int selfamd_model2d_stream(selfamd_model2d *m, void **stream) {
  SELFAMD_REQUIRE(m && stream, "model2d_stream: null argument");
  *stream = (void *)m->stream;
  return kOk;
}

int selfamd_model2d_time_steps(selfamd_model2d *m, int nSteps, double dt, double *elapsedMs) {
  SELFAMD_REQUIRE(m && elapsedMs && nSteps >= 0 && dt > 0.0, "model2d_time_steps: bad arguments");
  // graph capture is host work: done before the first event, so the GPU's idle time during it
  // is not timed
  SELFAMD_SETTLE(m);
  ResidentKernel kernel;
  if (!m->resident(nSteps, kernel)) SELFAMD_HIP(prepare_graphs(m, nSteps, dt));
  hipEvent_t e0, e1;
  SELFAMD_HIP(hipEventCreate(&e0));
  SELFAMD_HIP(hipEventCreate(&e1));
  SELFAMD_HIP(hipEventRecord(e0, m->stream));
  int rc = selfamd_model2d_forward_step(m, nSteps, dt);
  if (rc) return rc;
  SELFAMD_HIP(hipEventRecord(e1, m->stream));
  SELFAMD_HIP(hipEventSynchronize(e1));
  if (m->refused()) {  // the steps are taken now
    SELFAMD_HIP(hipEventRecord(e0, m->stream));
    if ((rc = wait_for(m))) return rc;
    SELFAMD_HIP(hipEventRecord(e1, m->stream));
    SELFAMD_HIP(hipEventSynchronize(e1));
  }
  float ms = 0.f;
  SELFAMD_HIP(hipEventElapsedTime(&ms, e0, e1));
  *elapsedMs = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return wait_for(m);
}

int selfamd_model2d_set_closure(selfamd_model2d *m, selfamd_mlp *mlp, const float *inMean, const float *inScale,
                                const float *outMean, const float *outScale) {
  SELFAMD_REQUIRE(m, "model2d_set_closure: null model");
  SELFAMD_SETTLE(m);
  SELFAMD_HIP(drain(m));
  m->drop_graphs();
  free_closure(m->closure);
  m->closure = nullptr;
  if (!mlp) return kOk;
  SELFAMD_REQUIRE(inMean && inScale && outMean && outScale, "model2d_set_closure: null normalisation array");
  SELFAMD_REQUIRE(m->affine, "model2d_set_closure: the closure reads the affine element records; mesh is not affine");
  SELFAMD_REQUIRE(m->nBands == 0, "model2d_set_closure: banded stepping is on (selfamd_model2d_set_bands(model, 0))");
  const int P = m->N + 1, NN = P * P;
  int nIn = 0, nOut = 0, maxB = 0;
  mlp_shape(mlp, &nIn, &nOut, &maxB);
  SELFAMD_REQUIRE(nIn == m->nVar * NN + 3 && nOut == m->nVar * NN,
                  "model2d_set_closure: network shape %d -> %d does not match %d nodal values + 3 metric scalars", nIn,
                  nOut, m->nVar * NN);
  SELFAMD_REQUIRE(maxB >= m->nEl, "model2d_set_closure: network batch %d < %d elements", maxB, m->nEl);
  // Sum of w_i w_j J over the mesh, for the mean-free mass correction
  std::vector<double> rec((size_t)kGeomStride * m->nEl), mats(2 * NN + 3 * P);
  SELFAMD_HIP(hipMemcpy(rec.data(), m->geom, sizeof(double) * rec.size(), hipMemcpyDeviceToHost));
  SELFAMD_HIP(hipMemcpy(mats.data(), m->mats, sizeof(double) * mats.size(), hipMemcpyDeviceToHost));
  double sw = 0.0, area = 0.0;
  for (int i = 0; i < P; i++) sw += mats[2 * NN + 2 * P + i];
  for (int e = 0; e < m->nEl; e++) area += rec[(size_t)kGeomStride * e + 4] * sw * sw;
  ClosureBuffers *c = new ClosureBuffers();
  c->mlp = mlp; c->nIn = nIn; c->nOut = nOut; c->invArea = 1.0 / area;
  const size_t nEl = m->nEl;
  const bool layers = !mlp_weights(mlp).rows;  // the row kernels keep outputs and input cotangents to themselves
  bool ok = hipMalloc(&c->X, 4 * nEl * nIn) == hipSuccess && (!layers || hipMalloc(&c->Y, 4 * nEl * nOut) == hipSuccess) &&
            hipMalloc(&c->inMean, 4 * nIn) == hipSuccess && hipMalloc(&c->inScale, 4 * nIn) == hipSuccess &&
            hipMalloc(&c->outMean, 4 * nOut) == hipSuccess && hipMalloc(&c->outScale, 4 * nOut) == hipSuccess &&
            hipMalloc(&c->corr, 8 * nEl * nOut) == hipSuccess && hipMalloc(&c->elemMass, 8 * nEl) == hipSuccess &&
            hipMalloc(&c->shift, 8) == hipSuccess && hipMalloc(&c->dY, 4 * nEl * nOut) == hipSuccess &&
            (!layers || hipMalloc(&c->dX, 4 * nEl * nIn) == hipSuccess) &&
            hipMalloc(&c->vjpPartial, 8 * closure_vjp_partials(m->N, m->nEl)) == hipSuccess;
  ok = ok && hipMemcpy(c->inMean, inMean, 4 * nIn, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(c->inScale, inScale, 4 * nIn, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(c->outMean, outMean, 4 * nOut, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(c->outScale, outScale, 4 * nOut, hipMemcpyHostToDevice) == hipSuccess &&
       hipStreamSynchronize(nullptr) == hipSuccess;
  if (!ok) {
    free_closure(c);
    set_error("model2d_set_closure: device allocation or copy failed");
    return kHipError;
  }
  m->closure = c;
  return kOk;
}

int selfamd_model2d_stage(selfamd_model2d *m, int stage, double dt, double *Ssave, double *unSave) {
  SELFAMD_REQUIRE(m && stage >= 0 && stage < 3 && dt > 0.0, "model2d_stage: bad arguments (stage=%d dt=%g)", stage, dt);
  SELFAMD_REQUIRE(m->nBands == 0, "model2d_stage: banded stepping is on");
  SELFAMD_SETTLE(m);
  const size_t nS = (size_t)(m->N + 1) * (m->N + 1) * m->nVar * m->nEl;
  if (Ssave) SELFAMD_HIP(hipMemcpyAsync(Ssave, m->S, sizeof(double) * nS, hipMemcpyDeviceToDevice, m->stream));
  if (unSave) {
    SELFAMD_REQUIRE(m->un[0], "model2d_stage: this model has no lagged velocities to save");
    const size_t nU = (size_t)(m->nodal ? 2 : 1) * (m->N + 1) * 4 * m->nEl;
    SELFAMD_HIP(hipMemcpyAsync(unSave, m->un[m->cur], sizeof(double) * nU, hipMemcpyDeviceToDevice, m->stream));
  }
  SELFAMD_HIP(m->launch_stage(0, stage, dt, m->cur, nullptr));
  m->cur ^= 1;
  if (stage == 2) m->t += dt;
  SELFAMD_HIP(drain(m));
  return resident_status(m);
}

int selfamd_model2d_tendency_vjp(selfamd_model2d *m, const double *S, const double *un, const double *lambda,
                                 double *mu, const double *Sprev, double *muPrev) {
  SELFAMD_REQUIRE(m && S && un && lambda && mu, "model2d_tendency_vjp: null argument");
  SELFAMD_REQUIRE(!Sprev == !muPrev, "model2d_tendency_vjp: Sprev and muPrev go together");
  SELFAMD_REQUIRE(m->kind == SELFAMD_MODEL_SW && !m->nodal && !m->anyBoundary,
                  "model2d_tendency_vjp: only nonlinear shallow water on affine meshes without boundary sides");
  const size_t nTr = (size_t)(m->N + 1) * 3 * 4 * m->nEl;
  // scratch: traces of S and of Sprev, neighbour-trace cotangents, lagged-velocity cotangents
  if (!m->adjTrace) SELFAMD_HIP(hipMalloc(&m->adjTrace, sizeof(double) * 2 * nTr));
  if (!m->adjChi) SELFAMD_HIP(hipMalloc(&m->adjChi, sizeof(double) * nTr * 5 / 3));
  StateArgs tr{};  // traces only
  tr.src = S; tr.trace = m->adjTrace; tr.mats = m->mats; tr.p = m->p; tr.nEl = m->nEl;
  SELFAMD_HIP(Launcher<PhysSW>::state_in(m->N, tr, m->stream));
  if (Sprev) {
    tr.src = Sprev; tr.trace = m->adjTrace + nTr;
    SELFAMD_HIP(Launcher<PhysSW>::state_in(m->N, tr, m->stream));
  }
  SELFAMD_HIP(sw_tendency_vjp(m->N, m->nEl, S, m->adjTrace, un, m->aux, m->geom, m->nbr, m->mats, m->p.g, m->p.fCori,
                              m->p.auxConst, lambda, mu, m->adjChi, m->adjTrace + nTr, muPrev, m->adjChi + nTr,
                              m->stream));
  SELFAMD_HIP(drain(m));
  return kOk;
}

int selfamd_model2d_closure_vjp(selfamd_model2d *m, const double *S, const double *lambda, double *mu) {
  SELFAMD_REQUIRE(m && S && lambda && mu, "model2d_closure_vjp: null argument");
  SELFAMD_REQUIRE(m->closure, "model2d_closure_vjp: no closure attached");
  const int P = m->N + 1;
  SELFAMD_HIP(closure_vjp(*m->closure, S, m->geom, m->mats + 2 * P * P + 2 * P, lambda, mu, m->N, m->nVar, 2, m->nEl,
                          m->stream));
  SELFAMD_HIP(drain(m));
  return kOk;
}

int selfamd_model2d_set_bands(selfamd_model2d *m, int nBands) {
  SELFAMD_REQUIRE(m && nBands >= 0, "model2d_set_bands: bad arguments");
  SELFAMD_REQUIRE(nBands == 0 || !m->closure, "model2d_set_bands: banded stepping does not take a closure");
  SELFAMD_SETTLE(m);
  SELFAMD_HIP(drain(m));
  m->drop_graphs();
  if (m->bandElems) (void)hipFree(m->bandElems);
  m->bandElems = nullptr;
  m->bandStart.clear();
  m->nBands = 0;
  if (nBands == 0) return kOk;
  const int nEl = m->nEl;
  SELFAMD_REQUIRE(nBands >= 2 && nBands <= nEl, "model2d_set_bands: need 2 <= nBands <= nEl (got %d)", nBands);
  // BFS levels of the element graph (interior neighbours), component after component
  std::vector<int> level(nEl, -1), queue;
  queue.reserve(nEl);
  int base = 0;
  for (int seed = 0; seed < nEl; seed++) {
    if (level[seed] >= 0) continue;
    size_t head = queue.size();
    level[seed] = base;
    queue.push_back(seed);
    int top = base;
    while (head < queue.size()) {
      const int e = queue[head++];
      for (int sd = 0; sd < 4; sd++) {
        const int c = m->hnbr[4 * (size_t)e + sd];
        if (c < 0) continue;
        const int e2 = c >> 3;
        if (level[e2] < 0) {
          level[e2] = level[e] + 1;
          top = std::max(top, level[e2]);
          queue.push_back(e2);
        }
      }
    }
    base = top + 1;
  }
  const int nLevels = base;
  std::vector<int> perLevel(nLevels, 0);
  for (int e = 0; e < nEl; e++) perLevel[level[e]]++;
  // consecutive whole levels per band, about nEl / nBands elements each
  std::vector<int> bandOf(nLevels, 0);
  int b = 0;
  long acc = 0;
  for (int l = 0; l < nLevels; l++) {
    bandOf[l] = b;
    acc += perLevel[l];
    if (b < nBands - 1 && acc >= (long)nEl * (b + 1) / nBands) b++;
  }
  const int used = bandOf[nLevels - 1] + 1;
  SELFAMD_REQUIRE(used >= 2, "model2d_set_bands: the element graph has too few BFS levels (%d) for %d bands",
                  nLevels, nBands);
  nBands = used;  // a band boundary can only fall between levels
  for (int e = 0; e < nEl; e++)
    for (int sd = 0; sd < 4; sd++) {
      const int c = m->hnbr[4 * (size_t)e + sd];
      if (c < 0) continue;
      const int d = bandOf[level[e]] - bandOf[level[c >> 3]];
      SELFAMD_REQUIRE(d >= -1 && d <= 1, "model2d_set_bands: neighbours %d and %d are more than one band apart", e,
                      c >> 3);
    }
  std::vector<int32_t> order;
  order.reserve(nEl);
  std::vector<int> start(nBands + 1, 0);
  for (int e = 0; e < nEl; e++) start[bandOf[level[e]] + 1]++;
  for (int k = 0; k < nBands; k++) start[k + 1] += start[k];
  order.assign(nEl, 0);
  std::vector<int> fill(start.begin(), start.end() - 1);
  for (int e = 0; e < nEl; e++) order[fill[bandOf[level[e]]]++] = e;  // by band, then element index
  SELFAMD_HIP(hipMalloc(&m->bandElems, sizeof(int32_t) * nEl));
  SELFAMD_HIP(hipMemcpy(m->bandElems, order.data(), sizeof(int32_t) * nEl, hipMemcpyHostToDevice));
  SELFAMD_HIP(hipStreamSynchronize(nullptr));
  m->bandStart = start;
  m->nBands = nBands;
  return kOk;
}

int selfamd_model2d_closure_features(selfamd_model2d *m, float *X) {
  SELFAMD_REQUIRE(m && X, "model2d_closure_features: null argument");
  SELFAMD_REQUIRE(m->closure, "model2d_closure_features: no closure attached");
  SELFAMD_SETTLE(m);
  SELFAMD_HIP(closure_features(m->S, m->geom, m->closure->inMean, m->closure->inScale, X, m->N, m->nVar, m->nEl,
                               m->stream));
  SELFAMD_HIP(drain(m));
  return resident_status(m);
}

int selfamd_tile_count(int kind, int N, int *count) {
  SELFAMD_REQUIRE(count, "tile_count: null argument");
  *count = tunable(kind, N) ? kTileVariants : 0;
  return kOk;
}

int selfamd_tile_info(int kind, int N, int variant, int *threads, int *alternate, int *xcdOrder, int *minWaves) {
  SELFAMD_REQUIRE(threads && alternate && xcdOrder && minWaves, "tile_info: null argument");
  SELFAMD_REQUIRE(tunable(kind, N) && variant >= 0 && variant < kTileVariants,
                  "tile_info: no variant %d for kind %d, N=%d", variant, kind, N);
  if (variant < 12) {
    *threads = 64 << (variant >> 2);
    *alternate = (variant >> 1) & 1;
    *xcdOrder = variant & 1;
    *minWaves = 1;
  } else {
    *threads = 64 << ((variant - 12) >> 1);
    *alternate = 1;
    *xcdOrder = 0;
    *minWaves = 5 + ((variant - 12) & 1);
  }
  return kOk;
}

int selfamd_tile_set(int kind, int N, int variant) {
  SELFAMD_REQUIRE(tunable(kind, N), "tile_set: kind %d, N=%d has no tile variants", kind, N);
  SELFAMD_REQUIRE(variant >= -1 && variant < kTileVariants, "tile_set: variant %d out of range", variant);
  g_tile[kind][N] = variant;
  g_tileEpoch++;
  return kOk;
}

int selfamd_tile_get(int kind, int N, int *variant) {
  SELFAMD_REQUIRE(variant, "tile_get: null argument");
  *variant = tile_of(kind, N);
  return kOk;
}

int selfamd_model2d_get_time(selfamd_model2d *m, double *t) {
  SELFAMD_REQUIRE(m && t, "model2d_get_time: null argument");
  *t = m->t;
  return kOk;
}
int selfamd_model2d_set_time(selfamd_model2d *m, double t) {
  SELFAMD_REQUIRE(m, "model2d_set_time: null model");
  m->t = t;
  return kOk;
}

}  // extern "C"

// ------------------------------------------------------------------------------
// Batched runs: many independent models advanced together
// ------------------------------------------------------------------------------
// Models of one polynomial degree are concatenated into one virtual mesh (state, traces,
// static fields, neighbour codes offset by each run's first element); each element record
// carries its run's dt.  One fused launch per degree group and RK stage advances every run
// of the group, and one hipGraph holds all groups' stages of one or more steps.  Per element the
// arithmetic is that of the single-run engine, so a batched run is bit-identical to the same
// run advanced alone.
namespace {
struct BatchGroup {
  int N = 0, nEl = 0;
  double *S = nullptr, *G = nullptr, *trace[2] = {nullptr, nullptr}, *un[2] = {nullptr, nullptr}, *geom = nullptr;
  double *mats = nullptr, *aux = nullptr, *stat2 = nullptr, *presTrace = nullptr;
  int32_t *nbr = nullptr;
  std::vector<int> runs;
  std::vector<size_t> first;  // first element of each run in the group
};
}  // namespace

namespace {
// Device-to-device copies of many arrays in one launch, the list in the kernel arguments: a copy
// call each costs 3 us whatever its size (48 runs of 8^2 to 64^2 elements, four arrays each: 567 us
// in 192 calls, 70 us in two launches).  blockIdx.y is the item, kCopyBlocks blocks stride through it;
// long arrays are several items of kCopyDoubles, so that the blocks grow with the data.
constexpr int kCopyItems = 160, kCopyBlocks = 48;
constexpr size_t kCopyDoubles = size_t(1) << 18;
struct CopyList {
  struct Item {
    const double *src;
    double *dst;
    size_t n;
  };
  Item item[kCopyItems];
  int count;
};
static_assert(sizeof(CopyList) <= 4096, "kernel arguments exceed the 4 KiB kernarg segment");
__global__ void __launch_bounds__(kThreads) k_copy_list(const CopyList list) {
  const CopyList::Item it = list.item[blockIdx.y];
  constexpr size_t STEP = (size_t)kCopyBlocks * kThreads;
  for (size_t k = blockIdx.x * (size_t)kThreads + threadIdx.x; k < it.n; k += 4 * STEP) {
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = it.src[min(k + q * STEP, it.n - 1)];
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (k + q * STEP < it.n) it.dst[k + q * STEP] = v[q];
  }
}
}  // namespace

struct selfamd_batch {
  int kind = 0;
  std::vector<Model *> models;
  std::vector<double> dt;
  std::vector<BatchGroup> groups;
  Params p{};
  bool anyBoundary = false;  // some run's mesh has a physical boundary side
  hipStream_t stream = nullptr;
  int cur = 0;
  hipGraphExec_t graph[2] = {nullptr, nullptr};  // one step, per starting trace buffer
  // graphs of 2^k steps (k = 1 .. kLevels - 1), per starting buffer, captured when a call first
  // needs them (2^k steps keep the starting buffer); a call replays the largest as often as it
  // fits and each smaller one at most once, as the single-run engine does
  static constexpr int kLevels = 5;  // up to 16 steps per graph
  hipGraphExec_t graphP[kLevels][2] = {};

  // SELFAMD_BATCH_PER_GROUP: one launch per degree group and stage; SELFAMD_BATCH_PERSISTENT:
  // one persistent launch per stage for all groups (SW, degrees 3, 5, 7)
  int mode = SELFAMD_BATCH_PER_GROUP;
  int persistentBlocks = 0;
  int device = 0;  // of the stream and the arrays

  FusedArgs group_args(const BatchGroup &g, int stage, int tin) const {
    FusedArgs a{};
    a.S = g.S; a.G = g.G; a.dSdt = nullptr;
    a.traceIn = g.trace[tin]; a.traceOut = g.trace[tin ^ 1];
    a.unIn = g.un[tin]; a.unOut = g.un[tin ^ 1];
    a.aux = g.aux; a.stat2 = g.stat2; a.presTrace = g.presTrace;
    a.geom = g.geom; a.nbr = g.nbr; a.mats = g.mats; a.nEl = g.nEl;
    a.rkA = kRk3A[stage]; a.rkG = kRk3G[stage]; a.rkGdt = 0.0; a.perElemDt = 1;
    a.writeG = stage != 2;
    a.reverse = tile_alternates(kind, g.N, g.nEl) ? tin : 0;
    a.anyBoundary = anyBoundary;
    a.p = p;
    return a;
  }
  hipError_t launch_group(const BatchGroup &g, int stage, int tin, hipStream_t st) {
    const FusedArgs a = group_args(g, stage, tin);
    switch (kind) {
      case SELFAMD_MODEL_SW: return Launcher<PhysSW>::stage(g.N, 0, false, a, st);
      case SELFAMD_MODEL_LSW: return Launcher<PhysLSW>::stage(g.N, 0, false, a, st);
      default: return Launcher<PhysEuler>::stage(g.N, 0, false, a, st);
    }
  }
  // whether the persistent kernel covers this batch: nonlinear SW, every degree 3, 5 or 7, and
  // the same face-sum split as the per-group tiles (its 256-wide tiles split at N = 7 and not
  // at N = 3 or 5; among the per-group tiles only the 64-wide ones at N = 5 split), so that
  // the results stay bit-identical to the separate solves
  bool persistent_ok() const {
    if (kind != SELFAMD_MODEL_SW) return false;
    for (const auto &g : groups) {
      if (g.N != 3 && g.N != 5 && g.N != 7) return false;
      if (g.N == 5) {
        const int v = tile_for(kind, 5, g.nEl);
        const int threads = v < 0 ? tile_threads<5>() : v < 12 ? 64 << (v >> 2) : 64 << ((v - 12) >> 1);
        if (threads == 64) return false;
      }
    }
    return true;
  }
  hipError_t launch_persistent(int stage, int tin) {
    PersistentArgs pa{};
    for (int k = 0; k < 3; k++)
      for (const auto &g : groups)
        if (g.N == kPersistentDegrees[k]) {
          pa.g[k] = group_args(g, stage, tin);
          pa.g[k].reverse = tin;  // per-element arithmetic does not depend on the order
        }
    hipLaunchKernelGGL(k_batch_persistent<PhysSW>, dim3(persistentBlocks), 256, 0, stream, pa);
    return hipGetLastError();
  }
  // Whether the groups of a graph of `steps` steps are branches of it: they are independent for the
  // whole call, and a stage launch then fills what another group's last wave leaves idle and starts
  // while that one ends.  10 steps of 48 shallow water runs of 8^2 to 64^2 elements (degrees 3, 5
  // and 7) take 1,650 us as branches and 1,950 in turn, 12 runs up to 32^2 335 and 500.  It costs a
  // fork and a join, 30 to 40 us per graph (one run each of degrees 3, 5 and 7, two steps: 304,000
  // nodes 118 and 128 us, 135,000 115 and 101; 10 steps of 8,000 nodes still 399 and 418, but with
  // two groups nothing).  And where the batch is larger than the Infinity Cache, a group's stages
  // find their data there only in turn (degrees 5 and 7, 10 steps: 192 MiB 1,835 and 1,963 us,
  // 264 MiB 2,567 and 2,544, 500 MiB 5,550 and 5,238).
  bool branches_pay(int steps) const {
    if (mode == SELFAMD_BATCH_PERSISTENT || groups.size() < 2) return false;
    size_t nodes = 0, bytes = 0;
    for (const auto &g : groups) {
      const size_t P = g.N + 1, n = P * P * g.nEl, faces = P * 4 * g.nEl;
      nodes += n;
      bytes += 8 * (n * (2 * models[0]->nVar + (g.aux != nullptr) + (g.stat2 != nullptr)) +
                    faces * (2 * models[0]->nT + (g.un[0] ? 2 : 0) + (g.presTrace ? models[0]->nT : 0)));
    }
    return bytes <= (size_t)256 << 20 && (nodes * steps >= (size_t)1 << 19 || (groups.size() > 2 && steps >= 8));
  }
  // Captures `steps` steps starting from trace buffer `start` (each step flips the buffer).
  hipError_t capture_steps(int start, int steps, hipGraphExec_t *out) {
    const DeviceScope scope(device);  // the branches' streams
    if (!scope.ok) return hipErrorInvalidDevice;
    const size_t branches = branches_pay(steps) ? groups.size() : 1;
    struct Branches {  // a stream and the event of its end for each branch but the first
      std::vector<hipStream_t> stream;
      std::vector<hipEvent_t> end;
      hipEvent_t fork = nullptr;
      hipError_t create(size_t n) {
        hipError_t e = n > 1 ? hipEventCreateWithFlags(&fork, hipEventDisableTiming) : hipSuccess;
        for (size_t k = 1; k < n && e == hipSuccess; k++) {
          hipStream_t s;
          hipEvent_t v;
          if ((e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking)) != hipSuccess) break;
          stream.push_back(s);
          if ((e = hipEventCreateWithFlags(&v, hipEventDisableTiming)) == hipSuccess) end.push_back(v);
        }
        return e;
      }
      ~Branches() {
        for (auto v : end) (void)hipEventDestroy(v);
        for (auto s : stream) (void)hipStreamDestroy(s);
        if (fork) (void)hipEventDestroy(fork);
      }
    } side;
    hipError_t e = side.create(branches);
    if (e != hipSuccess) return e;
    hipGraph_t gr;
    e = hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return e;
    hipError_t le = hipSuccess;
    // the stages of step n (each one flips the buffer)
    auto stages = [&](const BatchGroup &g, int n, hipStream_t st) {
      for (int k = 0; k < 3 && le == hipSuccess; k++) le = launch_group(g, k, start ^ ((n + k) & 1), st);
    };
    if (branches > 1) {
      le = hipEventRecord(side.fork, stream);
      for (size_t k = 0; k < branches && le == hipSuccess; k++) {
        const hipStream_t st = k ? side.stream[k - 1] : stream;
        if (k) le = hipStreamWaitEvent(st, side.fork, 0);
        for (int n = 0; n < steps; n++) stages(groups[k], n, st);
        if (k && le == hipSuccess) le = hipEventRecord(side.end[k - 1], st);
      }
      for (size_t k = 1; k < branches && le == hipSuccess; k++) le = hipStreamWaitEvent(stream, side.end[k - 1], 0);
    } else {
      for (int n = 0; n < steps && le == hipSuccess; n++) {
        const int tin = start ^ (n & 1), ng = (int)groups.size();
        if (mode == SELFAMD_BATCH_PERSISTENT) {
          for (int st = 0; st < 3 && le == hipSuccess; st++) le = launch_persistent(st, tin ^ (st & 1));
        } else {
          // Each group's three stages run back to back (a stage then starts on the data its
          // predecessor left in the Infinity Cache), and the group order reverses from step to
          // step (with the buffer parity), so that a group's last stage of one step is followed
          // by its first stage of the next.
          for (int k = 0; k < ng; k++) stages(groups[tin == 0 ? k : ng - 1 - k], n, stream);
        }
      }
    }
    hipError_t ce = hipStreamEndCapture(stream, &gr);
    if (le != hipSuccess) return le;
    if (ce != hipSuccess) return ce;
    hipError_t ie = hipGraphInstantiate(out, gr, nullptr, nullptr, 0);
    (void)hipGraphDestroy(gr);
    if (ie == hipSuccess) ie = hipGraphUpload(*out, stream);  // not on the first replay
    return ie;
  }
  void drop_graphs() {
    for (auto &gx : graph)
      if (gx) { (void)hipGraphExecDestroy(gx); gx = nullptr; }
    for (auto &lv : graphP)
      for (auto &gx : lv)
        if (gx) { (void)hipGraphExecDestroy(gx); gx = nullptr; }
  }
  // the one-step graphs of the current mode (the longer ones follow when first needed)
  hipError_t capture() {
    drop_graphs();
    for (int start = 0; start < 2; start++) {
      const hipError_t e = capture_steps(start, 1, &graph[start]);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  // the 2^k-step graphs of nSteps' decomposition, for both starting buffers
  hipError_t prepare(int nSteps) {
    const int top = kLevels - 1;
    int rem = nSteps;
    for (int k = top; k >= 1; k--) {
      const int s = 1 << k;
      if (rem < s) continue;
      for (int start = 0; start < 2; start++)
        if (!graphP[k][start]) {
          const hipError_t e = capture_steps(start, s, &graphP[k][start]);
          if (e != hipSuccess) return e;
        }
      rem = k == top ? rem % s : rem - s;
    }
    return hipSuccess;
  }
};

extern "C" {

int selfamd_batch_destroy(selfamd_batch *b) {
  if (!b) return kOk;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  b->drop_graphs();
  for (auto &g : b->groups) {
    double *bufs[] = {g.S, g.G, g.trace[0], g.trace[1], g.un[0], g.un[1], g.geom, g.mats, g.aux, g.stat2, g.presTrace};
    for (double *p : bufs)
      if (p) (void)hipFree(p);
    if (g.nbr) (void)hipFree(g.nbr);
  }
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return kOk;
}

int selfamd_batch_create(selfamd_batch **out, int nModels, selfamd_model2d *const *models, const double *dt) {
  SELFAMD_REQUIRE(out && models && dt && nModels >= 1, "batch_create: bad arguments");
  *out = nullptr;
  const Model *m0 = models[0];
  SELFAMD_REQUIRE(m0, "batch_create: null model");
  for (int r = 0; r < nModels; r++) {
    const Model *m = models[r];
    SELFAMD_REQUIRE(m && m->kind == m0->kind, "batch_create: run %d: all runs must be the same model kind", r);
    SELFAMD_REQUIRE(!m->nodal, "batch_create: run %d uses nodal metrics; batched runs take affine meshes", r);
    SELFAMD_REQUIRE(!m->closure, "batch_create: run %d has a closure attached; batched launches do not apply it", r);
    SELFAMD_REQUIRE(dt[r] > 0.0, "batch_create: run %d: dt must be positive", r);
    SELFAMD_REQUIRE(memcmp(&m->p, &m0->p, sizeof(Params)) == 0,
                    "batch_create: run %d: physical parameters differ from run 0", r);
    SELFAMD_REQUIRE((m->aux != nullptr) == (m0->aux != nullptr) && (m->stat2 != nullptr) == (m0->stat2 != nullptr) &&
                        (m->presTrace != nullptr) == (m0->presTrace != nullptr),
                    "batch_create: run %d: static fields must be set on all runs or on none", r);
    if (const int status = wait_for(models[r])) return status;
  }
  selfamd_batch *b = new selfamd_batch();
  b->kind = m0->kind;
  b->p = m0->p;
  for (int r = 0; r < nModels; r++) b->anyBoundary = b->anyBoundary || models[r]->anyBoundary;
  b->models.assign(models, models + nModels);
  b->dt.assign(dt, dt + nModels);
  auto fail = [&](const char *what, int code = kHipError) {
    set_error("batch_create: %s", what);
    selfamd_batch_destroy(b);
    return code;
  };
  if (hipGetDevice(&b->device) != hipSuccess) return fail("no device");
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) return fail("stream creation failed");
  for (int N = 1; N <= 7; N++) {
    BatchGroup g;
    g.N = N;
    size_t total = 0;
    for (int r = 0; r < nModels; r++)
      if (models[r]->N == N) { g.runs.push_back(r); g.first.push_back(total); total += models[r]->nEl; }
    if (g.runs.empty()) continue;
    if (total >= (size_t)1 << 27) return fail("a degree group has too many elements (at most 2^27)", kBadArgument);
    g.nEl = (int)total;
    const size_t P = N + 1, PP = P * P, nV = m0->nVar, nT = m0->nT;
    const size_t nS = total * PP * nV, nTr = total * P * nT * 4;
    if (hipMalloc(&g.S, 8 * nS) || hipMalloc(&g.G, 8 * nS) || hipMalloc(&g.trace[0], 8 * nTr) ||
        hipMalloc(&g.trace[1], 8 * nTr) || hipMalloc(&g.geom, 8 * kGeomStride * total) ||
        hipMalloc(&g.mats, 8 * (2 * PP + 4 * P)) || hipMalloc(&g.nbr, 4 * 4 * total) ||
        (m0->un[0] && (hipMalloc(&g.un[0], 8 * total * P * 4) || hipMalloc(&g.un[1], 8 * total * P * 4))) || (m0->aux && hipMalloc(&g.aux, 8 * total * PP)) ||
        (m0->stat2 && hipMalloc(&g.stat2, 8 * total * PP)) || (m0->presTrace && hipMalloc(&g.presTrace, 8 * nTr))) {
      b->groups.push_back(g);
      return fail("device allocation failed");
    }
    b->groups.push_back(g);
    BatchGroup &G = b->groups.back();
    if (hipMemcpy(G.mats, models[G.runs[0]]->mats, 8 * (2 * PP + 4 * P), hipMemcpyDeviceToDevice))
      return fail("copy failed");
    std::vector<double> rec;
    std::vector<int32_t> nb;
    for (size_t k = 0; k < G.runs.size(); k++) {
      const Model *m = models[G.runs[k]];
      const size_t off = G.first[k], ne = m->nEl;
      hipError_t e = hipSuccess;
      e = e ? e : hipMemcpy(G.S + off * PP * nV, m->S, 8 * ne * PP * nV, hipMemcpyDeviceToDevice);
      e = e ? e : hipMemcpy(G.G + off * PP * nV, m->G, 8 * ne * PP * nV, hipMemcpyDeviceToDevice);
      e = e ? e : hipMemcpy(G.trace[0] + off * P * nT * 4, m->trace[m->cur], 8 * ne * P * nT * 4, hipMemcpyDeviceToDevice);
      if (G.un[0]) e = e ? e : hipMemcpy(G.un[0] + off * P * 4, m->un[m->cur], 8 * ne * P * 4, hipMemcpyDeviceToDevice);
      if (G.aux) e = e ? e : hipMemcpy(G.aux + off * PP, m->aux, 8 * ne * PP, hipMemcpyDeviceToDevice);
      if (G.stat2) e = e ? e : hipMemcpy(G.stat2 + off * PP, m->stat2, 8 * ne * PP, hipMemcpyDeviceToDevice);
      if (G.presTrace)
        e = e ? e : hipMemcpy(G.presTrace + off * P * nT * 4, m->presTrace, 8 * ne * P * nT * 4, hipMemcpyDeviceToDevice);
      rec.resize(kGeomStride * ne);
      nb.resize(4 * ne);
      e = e ? e : hipMemcpy(rec.data(), m->geom, 8 * kGeomStride * ne, hipMemcpyDeviceToHost);
      e = e ? e : hipMemcpy(nb.data(), m->nbr, 4 * 4 * ne, hipMemcpyDeviceToHost);
      if (e) return fail("copy failed");
      for (size_t q = 0; q < ne; q++) rec[kGeomStride * q + 5] = b->dt[G.runs[k]];
      for (auto &c : nb)
        if (c >= 0) c += (int32_t)(off << 3);  // neighbour element index shifts by the run's offset
      e = hipMemcpy(G.geom + kGeomStride * off, rec.data(), 8 * kGeomStride * ne, hipMemcpyHostToDevice);
      e = e ? e : hipMemcpy(G.nbr + 4 * off, nb.data(), 4 * 4 * ne, hipMemcpyHostToDevice);
      if (e) return fail("copy failed");
    }
  }
  // copies into device memory may still be under way, and the batch's stream would not wait for them
  if (hipStreamSynchronize(nullptr) != hipSuccess) return fail("copy failed");
  if (b->capture() != hipSuccess) return fail("stage graph capture failed");
  *out = b;
  return kOk;
}

int selfamd_batch_set_mode(selfamd_batch *b, int mode) {
  SELFAMD_REQUIRE(b && (mode == SELFAMD_BATCH_PER_GROUP || mode == SELFAMD_BATCH_PERSISTENT),
                  "batch_set_mode: bad arguments (mode=%d)", mode);
  SELFAMD_REQUIRE(mode == SELFAMD_BATCH_PER_GROUP || b->persistent_ok(),
                  "batch_set_mode: the persistent launch takes nonlinear SW runs of degrees 3, 5 and 7 "
                  "whose per-group tile at N = 5 is not 64 wide (that tile splits the face sums)");
  SELFAMD_HIP(hipStreamSynchronize(b->stream));
  if (mode == SELFAMD_BATCH_PERSISTENT && b->persistentBlocks == 0) {
    int dev = 0, cus = 0, perCU = 0;
    SELFAMD_HIP(hipGetDevice(&dev));
    SELFAMD_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    SELFAMD_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, k_batch_persistent<PhysSW>, 256, 0));
    SELFAMD_REQUIRE(cus > 0 && perCU > 0, "batch_set_mode: no resident block for the persistent kernel");
    b->persistentBlocks = cus * perCU;
  }
  const int previous = b->mode;
  b->mode = mode;
  const hipError_t e = b->capture();
  if (e != hipSuccess) {
    // keep the batch usable: back to the previous mode's graphs
    b->mode = previous;
    const hipError_t e2 = b->capture();
    set_error("batch_set_mode: graph capture failed: %s%s", hipGetErrorString(e),
              e2 == hipSuccess ? "" : " (the previous mode's graphs could not be restored either)");
    return kHipError;
  }
  return kOk;
}

int selfamd_batch_forward_step(selfamd_batch *b, int nSteps) {
  SELFAMD_REQUIRE(b && nSteps >= 0, "batch_forward_step: bad arguments");
  SELFAMD_HIP(b->prepare(nSteps));
  const int top = selfamd_batch::kLevels - 1;
  int n = nSteps;
  for (int k = top; k >= 1; k--) {
    const int s = 1 << k;
    while (n >= s) {
      SELFAMD_HIP(hipGraphLaunch(b->graphP[k][b->cur], b->stream));  // an even step count: same buffer
      n -= s;
      if (k != top) break;
    }
  }
  if (n == 1) {
    SELFAMD_HIP(hipGraphLaunch(b->graph[b->cur], b->stream));
    b->cur ^= 1;
  }
  for (size_t r = 0; r < b->models.size(); r++) b->models[r]->t += nSteps * b->dt[r];
  return kOk;
}

int selfamd_batch_time_steps(selfamd_batch *b, int nSteps, double *elapsedMs) {
  SELFAMD_REQUIRE(b && elapsedMs && nSteps >= 0, "batch_time_steps: bad arguments");
  // graph capture is host work: done before the first event
  SELFAMD_HIP(b->prepare(nSteps));
  hipEvent_t e0, e1;
  SELFAMD_HIP(hipEventCreate(&e0));
  SELFAMD_HIP(hipEventCreate(&e1));
  SELFAMD_HIP(hipEventRecord(e0, b->stream));
  int rc = selfamd_batch_forward_step(b, nSteps);
  if (rc) return rc;
  SELFAMD_HIP(hipEventRecord(e1, b->stream));
  SELFAMD_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  SELFAMD_HIP(hipEventElapsedTime(&ms, e0, e1));
  *elapsedMs = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return kOk;
}

// Copies every run's state (solution, RK register, traces, lagged velocities) back into its
// model handle, which then continues on its own exactly where the batch left it.
int selfamd_batch_scatter(selfamd_batch *b) {
  SELFAMD_REQUIRE(b, "batch_scatter: null batch");
  SELFAMD_HIP(hipStreamSynchronize(b->stream));
  // on the default stream, behind any caller's work on a blocking stream of a model
  for (Model *m : b->models) SELFAMD_HIP(drain(m));
  const DeviceScope scope(b->device);
  SELFAMD_REQUIRE(scope.ok, "batch_scatter: the batch's device cannot be made current");
  CopyList list{};
  auto flush = [&]() -> hipError_t {
    if (list.count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy_list, dim3(kCopyBlocks, list.count), kThreads, 0, nullptr, list);
    list.count = 0;
    return hipGetLastError();
  };
  for (auto &G : b->groups) {
    const size_t P = G.N + 1, PP = P * P;
    for (size_t k = 0; k < G.runs.size(); k++) {
      Model *m = b->models[G.runs[k]];
      const size_t off = G.first[k], ne = m->nEl, nV = m->nVar, nT = m->nT;
      const CopyList::Item items[4] = {{G.S + off * PP * nV, m->S, ne * PP * nV},
                                       {G.G + off * PP * nV, m->G, ne * PP * nV},
                                       {G.trace[b->cur] + off * P * nT * 4, m->trace[m->cur], ne * P * nT * 4},
                                       {m->un[0] ? G.un[b->cur] + off * P * 4 : nullptr, m->un[m->cur], ne * P * 4}};
      for (const auto &it : items) {
        if (!it.src) continue;
        if (m->device != b->device) {  // a kernel may not reach it
          SELFAMD_HIP(hipMemcpy(it.dst, it.src, 8 * it.n, hipMemcpyDeviceToDevice));
          continue;
        }
        for (size_t at = 0; at < it.n; at += kCopyDoubles) {
          if (list.count == kCopyItems) SELFAMD_HIP(flush());
          list.item[list.count++] = {it.src + at, it.dst + at, std::min(kCopyDoubles, it.n - at)};
        }
      }
    }
  }
  SELFAMD_HIP(flush());
  SELFAMD_HIP(hipStreamSynchronize(nullptr));
  for (Model *m : b->models) state_replaced(m);
  return kOk;
}

int selfamd_batch_info(selfamd_batch *b, int *nGroups, double *totalDof) {
  SELFAMD_REQUIRE(b && nGroups && totalDof, "batch_info: null argument");
  *nGroups = (int)b->groups.size();
  double dof = 0.0;
  for (auto &g : b->groups) dof += (double)g.nEl * (g.N + 1) * (g.N + 1) * b->models[0]->nVar;
  *totalDof = dof;
  return kOk;
}

}  // extern "C"
