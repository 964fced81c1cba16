// Device kernels of the MI355X flow-solver hot path (gfx950, wave64).
//
// Layout (device numbering, nested Morton order, see solver.hip):
//   node state      u[c*n+i] (SoA, 6 comps), uprev, p, dt, dtt, mu, vort,
//                   divg, diss[5], src[6], tdiff
//   rec0[8*i]       AoS per node: rho, u, v, w, rhoE, p, nu~, mu  (gathers)
//   mom[4*i]        AoS per node: the state's momenta, pad (levels with JST or fluxType 1-3)
//   grec[GREC*i]    AoS per node (HLLC-2): grad 15 | 1/lo 5 | 1/hi 5 | pad
//                   (lo/hi = nodeHelpArray 16-25: min/max over sides - q)
//   edges           ea[e], eb[e] (ends in reference orientation), w[3*e] AoS
//   incidence       sliced ELL, one wavefront per slice of 64 nodes:
//                   slot (k, lane) at ell_ptr[s] + 64*k + lane holds
//                   ell_e = edge<<1 | role (role 1: node is eb), ell_nbr,
//                   and ellw[3][slot] = the side weights signed for the
//                   node (+w as ea, -w as eb)
//   boundary sides  ba, bb, bind, wb[3*s]; per node CSR bs_ptr/bs_list
//                   (side<<1 | end)
// Every edge loop of the reference (scatter to both ends) is evaluated here
// as a gather at each node over its incidence list in a fixed order, so
// results are deterministic and no atomics are used.  The HLLC flux is the
// exception: it is evaluated once per edge, in blocks of sides whose per-node
// sums the stage kernel adds, or, on small first-order levels, in the stage's
// own blocks of nodes (k_stage_blk).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/flite3d_amd.h"

namespace fk {

constexpr int SLICE = 64;
constexpr int GREC = 26;
// viscous record per node: a side's viscous and SA-diffusion fluxes are
// w.(node's own part + the other's), so the record holds those parts, all that
// a neighbour reads, in one 128-byte line: stress 6 | energy flux k grad T +
// tau.v 3 | diffusion flux (Re mu/rho + nu~) grad nu~ 3 | the SA time step's
// viscosity | nodal cb2 term | pad.  (Stress, velocity, grad nu~ and the
// diffusion coefficient's three factors took this line and the neighbour's
// gather record: the second pass, staged, took 838 us with the SA time steps
// and 767 without on 2.1M nodes; 601 and 441 with this record, 535 and 419
// since the staging's loads are in flight together.)
constexpr int VREC = 16;
constexpr int NTHR = 256;

struct DevParams {
  double gamma, mach, Re, Pr, Prt;
  double inflow[2][6];
  double inflow_temperature;
  int isentropic, sa, order, autoclip, nsig, bterm;
  double clip, max_inc, min_rho, max_turb, turb_k;
  double beta0;  // Davis wave-speed factor sqrt((gamma - 1) / (2 gamma))
  // interior flux (1 central, 2 LLF, 3 Roe, 4 HLLC) and the JST dissipation
  // of the first three: second-order factor, fourth-order factor on grid 1
  // and below it, matrix scaling and its entropy fix
  int ftype, matdiss;
  double k2, k4, k4c, hcf;
  // dual time stepping on a fixed mesh: unsteady (flowType != 0), time
  // differences added (addTimeStep), BDF2 on grid 1, physical time step
  int unsteady, add_time, bdf2;
  double dtp;
  double prolong_relax, turb_prolong_relax, mg_bc_relax;
  // batched conditions: per condition (Mach, inflowField(1:6,1), spare),
  // 8 doubles each; null for a single condition
  const double *cond;
  __device__ __forceinline__ void to_batch(int b) {
    if (!cond) return;
    const double *q = cond + 8 * (size_t)b;
    mach = q[0];
#pragma unroll
    for (int k = 0; k < 6; ++k) inflow[0][k] = q[1 + k];
  }
  // farfield state `row` (0: inflowField(:,1), 1: inflowField(:,2)) copied
  // out by value: selecting rows with constant indices keeps the parameter
  // block in registers (a run-time row index would force it into scratch)
  __device__ __forceinline__ void inflow_row(int row, double *o) const {
#pragma unroll
    for (int k = 0; k < 6; ++k) o[k] = row == 0 ? inflow[0][k] : inflow[1][k];
  }
};

// node boundary class from nodeIndicatorArray ranges; bit 4 marks host
// index < numberOfBoundaryNodes (boundary-first numbering)
enum : int { NC_NONE = 0, NC_WALL = 1, NC_SYM = 2, NC_FAR1 = 3, NC_FAR2 = 4, NC_INVWALL = 9 };
constexpr int NC_MASK = 15;
constexpr int NC_BFIRST = 16;

// node blocks of the one-launch stages: nodes, tasks (one a thread), staged
// nodes, incidences, lanes summing a node
constexpr int SB_NODES = 32, SB_TASKS = NTHR, SB_CAP = 224, SB_INC = 512, SB_SUB = NTHR / SB_NODES;

template <typename R>
struct LevelDev {
  int n, ne, nbs, gnum;
  const int *ea, *eb;
  const R *w;          // 3 per edge
  const int *ba, *bb, *bind;
  const R *wb;         // 3 per boundary side
  const int *ell_ptr, *ell_k;
  const int *ell_e, *ell_nbr;
  const R *ellw;       // signed side weights per ELL slot, SoA: [c * nslot + slot]
  long long nslot;
  const int *bs_ptr, *bs_list;
  // side blocks of k_flux_blk (one shape's tables): fb_head[4 k ..] = {first
  // side e0, first entry n0, first incidence ibase, 0} of block k (nfb + 1
  // headers, the last one closing the lists); block k serves sides e0 ..
  // next e0 - 1 and stages the nodes fb_node[FB_SHAPE_NODES[shape] k ..]
  // (n1 - n0 of them, the rest -1);
  // fb_loc[e] = both ends' positions in that list (first end in the low 16
  // bits)
  int nfb;
  const int *fb_head, *fb_node;
  const unsigned *fb_loc;
  // per-node partial sums of the side fluxes (k_flux_blk): entry q = n0 +
  // the node's position in its block; fb_inc[fb_iptr[q] ..] = the entry's
  // sides within its block (local side << 1 | 1 when the node is the side's
  // second end); node i's entries are pn_ent[pn_ptr[i] ..], in block order
  long long nent;
  const int *fb_iptr, *pn_ptr, *pn_ent;
  const unsigned short *fb_inc;
  R *pbuf;
  // node blocks of the LDS-staged gathers: block k serves nodes
  // gb_first[k] .. gb_first[k+1]-1 and stages their neighbours
  // gb_node[gb_nptr[k] ..]; ell_loc[slot] = the slot's neighbour in that list
  // (0xffff for an empty slot)
  int ngb;
  const int *gb_first, *gb_nptr, *gb_node;
  const unsigned short *ell_loc;
  // node blocks of the one-launch stages (k_stage_blk), block k's tables at
  // fixed places: sb_node[SB_CAP k ..] = the staged nodes, the block's own
  // (consecutive) first and then their other neighbours, -1 beyond;
  // sb_loc[SB_TASKS k + t] = task t: both ends' staged positions (12 bits
  // each) | kind << 24 (0: an interior side, k + 1: a boundary side of
  // indicator k (k <= 0 as 0: they are walls alike), seen from its first
  // listed end, 255: none), sb_w[3] (SoA, stride SB_TASKS nsb) its weight;
  // sb_inc[SB_INC k + ..] = the tasks of the block's nodes (task << 1 | 1
  // when the node is the side's second end), node m's from sb_iptr[(SB_NODES
  // + 1) k + m] (the block's nodes end where the list does)
  int nsb;
  const int *sb_node;
  const unsigned *sb_loc;
  const unsigned short *sb_inc, *sb_iptr;
  const R *sb_w;
  const R *vol, *xyz, *wd, *nrm;  // nrm: 3 per node AoS
  const int *ncls;
  R *u, *uprev, *rhs, *diss, *src, *p, *dt, *dtt, *mu, *vort, *divg, *tdiff;
  R *rec0, *grec, *tau, *dnu, *fbuf, *bbuf, *ws;  // tau, dnu = tau + 9: VREC-strided, one shared record
  R *rec1;  // the next state's gather records while a walking stage reads rec0 (null: no such stage)
  // the conserved momenta beside the records, for differences of neighbouring
  // states: rho (m / rho) is not m (null: no such terms), and those of rec1
  R *mom, *mom1;
  const R *wsum;  // 3 per node: sum w + 2 sum_b w over the node's sides (levels with gradients)
  R *jst;  // JST node record (8 per node): L(U) 5, pressure switch, side count, volume / time step
  R *uold, *uold2;  // solutions at the last two physical times (6 per node, unsteady only)
  // moving meshes (null on a fixed mesh): GCL weight per side and 2 per
  // boundary side, previous volumes and movement (3 per node AoS) on level 1
  const R *gcl, *bgcl, *volp, *volp2, *cmv;
  // batched conditions: nb copies of every state array, condition-major;
  // gstride = gradient-record elements per condition (0 if none)
  int nb;
  long long gstride;
  __device__ __forceinline__ void to_batch(int b) {
    if (b == 0) return;
    size_t bn = (size_t)b * (size_t)n;
    u += 6 * bn;
    uprev += 6 * bn;
    rhs += 6 * bn;
    diss += 5 * bn;
    src += 6 * bn;
    p += bn;
    dt += bn;
    dtt += bn;
    mu += bn;
    vort += bn;
    divg += bn;
    tdiff += bn;
    rec0 += 8 * bn;
    if (rec1) rec1 += 8 * bn;
    if (mom) mom += 4 * bn;
    if (mom1) mom1 += 4 * bn;
    grec += (size_t)b * (size_t)gstride;
    tau += VREC * bn;
    dnu += VREC * bn;
    fbuf += (size_t)b * 6 * (size_t)ne;
    pbuf += (size_t)b * 6 * (size_t)nent;
    bbuf += (size_t)b * 10 * (size_t)nbs;
    ws += 3 * bn;
    jst += 8 * bn;
    uold += 6 * bn;
    uold2 += 6 * bn;
  }
};

__device__ __forceinline__ int gtid() { return blockIdx.x * blockDim.x + threadIdx.x; }

// XCD-aware block order: the hardware hands workgroup b to XCD b % 8; this
// remaps so that each XCD walks one contiguous range of logical blocks and
// its L2 sees one compact window of nodes/sides instead of every 8th block.
constexpr int NXCD = 8;
__device__ __forceinline__ int xcd_block() {
  int b = blockIdx.x, nb = gridDim.x;
  if (nb < 2 * NXCD) return b;
  int x = b % NXCD, k = b / NXCD;
  int q = nb / NXCD, r = nb % NXCD;
  int start = x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q;
  return start + k;
}
__device__ __forceinline__ int gtid_x() { return xcd_block() * blockDim.x + threadIdx.x; }

// Batched conditions: logical workgroup lb serves condition b = lb % nb on
// block lb / nb of the nodes or sides, so consecutive workgroups gather the
// same mesh data for successive conditions and find it in L2.  nb = 1 is
// the plain index.
__device__ __forceinline__ int btid(int nb, int &b) {
  int lb = xcd_block();
  b = lb % nb;
  return (lb / nb) * blockDim.x + threadIdx.x;
}

template <typename R>
__device__ __forceinline__ R rmax(R a, R b) { return a > b ? a : b; }
template <typename R>
__device__ __forceinline__ R rmin(R a, R b) { return a < b ? a : b; }

// Forward-mode dual number: a value and one directional derivative.  The
// residual's side and boundary fluxes are templated on their arithmetic
// type; evaluated on Dual they give the exact derivative along the seeded
// direction (the tangent), and seeded along an input its row of the
// transposed Jacobian products (the metric and mesh adjoints; the state
// adjoint's side flux has a reverse sweep of its own).  Comparisons and
// selections act on the value, so the derivative is that of the branch the
// value takes.  Kept in its own namespace so that its sqrt/fabs/fmin/fmax
// are found by argument lookup only and never hide the double versions.
namespace ad {
struct Dual {
  double v, d;
  __host__ __device__ Dual() : v(0), d(0) {}
  __host__ __device__ Dual(double x) : v(x), d(0) {}
  __host__ __device__ Dual(double x, double y) : v(x), d(y) {}
};
__device__ __forceinline__ Dual operator+(Dual a, Dual b) { return Dual(a.v + b.v, a.d + b.d); }
__device__ __forceinline__ Dual operator-(Dual a, Dual b) { return Dual(a.v - b.v, a.d - b.d); }
__device__ __forceinline__ Dual operator-(Dual a) { return Dual(-a.v, -a.d); }
__device__ __forceinline__ Dual operator*(Dual a, Dual b) { return Dual(a.v * b.v, a.d * b.v + a.v * b.d); }
__device__ __forceinline__ Dual operator/(Dual a, Dual b) {
  double q = a.v / b.v;
  return Dual(q, (a.d - q * b.d) / b.v);
}
__device__ __forceinline__ Dual &operator+=(Dual &a, Dual b) { return a = a + b; }
__device__ __forceinline__ Dual &operator-=(Dual &a, Dual b) { return a = a - b; }
__device__ __forceinline__ Dual &operator*=(Dual &a, Dual b) { return a = a * b; }
__device__ __forceinline__ bool operator<(Dual a, Dual b) { return a.v < b.v; }
__device__ __forceinline__ bool operator>(Dual a, Dual b) { return a.v > b.v; }
__device__ __forceinline__ bool operator<=(Dual a, Dual b) { return a.v <= b.v; }
__device__ __forceinline__ bool operator>=(Dual a, Dual b) { return a.v >= b.v; }
__device__ __forceinline__ bool operator==(Dual a, Dual b) { return a.v == b.v; }
__device__ __forceinline__ bool operator!=(Dual a, Dual b) { return a.v != b.v; }
__device__ __forceinline__ Dual sqrt(Dual a) {
  double r = ::sqrt(a.v);
  return Dual(r, r > 0.0 ? a.d / (2.0 * r) : 0.0);
}
__device__ __forceinline__ Dual fabs(Dual a) { return a.v < 0.0 ? -a : a; }
__device__ __forceinline__ Dual exp(Dual a) {
  double e = ::exp(a.v);
  return Dual(e, e * a.d);
}
__device__ __forceinline__ Dual pow(Dual a, double p) {
  double r = ::pow(a.v, p);
  return Dual(r, a.v != 0.0 ? p * r / a.v * a.d : 0.0);
}
__device__ __forceinline__ Dual fmin(Dual a, Dual b) { return b.v < a.v ? b : a; }
__device__ __forceinline__ Dual fmax(Dual a, Dual b) { return b.v > a.v ? b : a; }
}  // namespace ad

// The incidence lists and slot weights are streamed once per gather launch:
// nontemporal loads keep them from evicting the node records that
// neighbouring nodes re-read from L2.
template <typename T>
__device__ __forceinline__ T ldnt(const T *p) { return __builtin_nontemporal_load(p); }

// N consecutive values of a gather record in 16-byte loads (8-byte loads for
// FP32 records whose stride is not a multiple of 16 bytes): fewer memory
// instructions per lane for the scattered record reads.  p must be aligned
// to 16 bytes (FP64, or FP32 with N % 4 == 0) or 8 bytes (other FP32).
template <int N, typename R>
__device__ __forceinline__ void ldrec(const R *p, R *o) {
  if constexpr (sizeof(R) == 8) {
    static_assert(N % 2 == 0, "FP64 records load in pairs");
    const double2 *q = reinterpret_cast<const double2 *>(p);
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      double2 v = q[k];
      o[2 * k] = v.x;
      o[2 * k + 1] = v.y;
    }
  } else if constexpr (N % 4 == 0) {
    const float4 *q = reinterpret_cast<const float4 *>(p);
#pragma unroll
    for (int k = 0; k < N / 4; ++k) {
      float4 v = q[k];
      o[4 * k] = v.x;
      o[4 * k + 1] = v.y;
      o[4 * k + 2] = v.z;
      o[4 * k + 3] = v.w;
    }
  } else {
    static_assert(N % 2 == 0, "FP32 records load in pairs");
    const float2 *q = reinterpret_cast<const float2 *>(p);
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      float2 v = q[k];
      o[2 * k] = v.x;
      o[2 * k + 1] = v.y;
    }
  }
}

// Lanes per node in the gather kernels.  SUB consecutive lanes of a
// wavefront share node i = t / SUB and split its incidence lists
// round-robin (lane `sub` takes slots sub, sub+SUB, ...); their partial
// results are combined by a fixed xor butterfly, so every lane of the group
// ends with the same bits whatever the scheduling.  SUB = 1 on large levels;
// on small coarse levels SUB > 1 puts more lanes on the chip and shortens
// each lane's chain of dependent gathers.
template <int SUB>
__device__ __forceinline__ void node_lanes(int nb, int &b, int &i, int &sub) {
  int t = btid(nb, b);
  i = t / SUB;
  sub = t % SUB;
}
template <int SUB, typename T>
__device__ __forceinline__ T lsum(T v) {
#pragma unroll
  for (int m = 1; m < SUB; m <<= 1) v += __shfl_xor(v, m, SUB);
  return v;
}
template <int SUB, typename T>
__device__ __forceinline__ T lmin(T v) {
#pragma unroll
  for (int m = 1; m < SUB; m <<= 1) {
    T o = __shfl_xor(v, m, SUB);
    v = o < v ? o : v;
  }
  return v;
}

// iterate this lane's share of the incidence of node i: f(edge, role)
template <int SUB, typename R, typename F>
__device__ __forceinline__ void for_edges(const LevelDev<R> &L, int i, int sub, F f) {
  int s = i / SLICE, lane = i % SLICE;
  int base = L.ell_ptr[s], K = L.ell_k[s];
  for (int k = sub; k < K; k += SUB) {
    int v = ldnt(L.ell_e + base + k * SLICE + lane);
    if (v < 0) continue;
    f(v >> 1, v & 1);
  }
}

// neighbours with the node-signed side weights (+w when the node is the
// side's first end, -w when it is the second): f(nbr, wx, wy, wz).  A
// reference scatter "+f to i1, -f to i2" with f linear in w becomes "+f(w_s)"
// here, with the same rounding since the sign flip is exact.
// for_slots also passes the slot, for the side and the node's role in it.
template <int SUB, typename R, typename F>
__device__ __forceinline__ void for_slots(const LevelDev<R> &L, int i, int sub, F f) {
  int s = i / SLICE, lane = i % SLICE;
  int base = L.ell_ptr[s], K = L.ell_k[s];
  const long long ns = L.nslot;
  for (int k = sub; k < K; k += SUB) {
    int slot = base + k * SLICE + lane;
    int j = ldnt(L.ell_nbr + slot);
    if (j < 0) continue;
    f(slot, j, ldnt(L.ellw + slot), ldnt(L.ellw + ns + slot), ldnt(L.ellw + 2 * ns + slot));
  }
}
template <int SUB, typename R, typename F>
__device__ __forceinline__ void for_edges_w(const LevelDev<R> &L, int i, int sub, F f) {
  for_slots<SUB>(L, i, sub, [&](int, int j, R wx, R wy, R wz) { f(j, wx, wy, wz); });
}

// ---------------------------------------------------------------------------
// LDS staging of node records for blocks of sides or nodes
// ---------------------------------------------------------------------------
template <typename R> struct Pair;
template <> struct Pair<double> { using type = double2; };
template <> struct Pair<float> { using type = float2; };

// Neighbour walks of node i: f(qj, tj, wx, wy, wz) per interior side with w
// the node-signed side weights and either qj the neighbour's gather record
// (AUXW = 0; MOM: with its momenta as tj) or tj the first AUXW words of its
// viscous record, in registers.  walk_global reads the neighbours' records
// from memory; walk_staged the viscous records from the LDS slots a node block
// staged.
template <int SUB, int AUXW = 0, bool MOM = false, typename R, typename F>
__device__ __forceinline__ void walk_global(const LevelDev<R> &L, int i, int sub, F f) {
  static_assert(!(MOM && AUXW > 0), "one of the two");
  for_edges_w<SUB>(L, i, sub, [&](int j, R wx, R wy, R wz) {
    if constexpr (MOM) {
      R qj[8], mj[4];
      ldrec<8>(L.rec0 + 8 * (size_t)j, qj);
      ldrec<4>(L.mom + 4 * (size_t)j, mj);
      f(qj, mj, wx, wy, wz);
    } else if constexpr (AUXW == 0) {
      R qj[8];
      ldrec<8>(L.rec0 + 8 * (size_t)j, qj);
      f(qj, (const R *)nullptr, wx, wy, wz);
    } else {
      R tj[AUXW];
      ldrec<AUXW>(L.tau + VREC * (size_t)j, tj);
      f((const R *)nullptr, tj, wx, wy, wz);
    }
  });
}
template <int SUB, int S, typename R, typename F>
__device__ __forceinline__ void walk_staged(const LevelDev<R> &L, const R *sn, int i, int sub, F f) {
  int s = i / SLICE, lane = i % SLICE;
  int base = L.ell_ptr[s], K = L.ell_k[s];
  const long long ns = L.nslot;
  for (int k = sub; k < K; k += SUB) {
    int slot = base + k * SLICE + lane;
    unsigned loc = ldnt(L.ell_loc + slot);
    if (loc == 0xffffu) continue;
    f((const R *)nullptr, sn + loc * S, ldnt(L.ellw + slot), ldnt(L.ellw + ns + slot), ldnt(L.ellw + 2 * ns + slot));
  }
}

// Node blocks with their neighbours' records staged in LDS.  A block serves
// up to GB_NODES consecutive nodes, GB_SUB lanes each, whose neighbours are
// at most GB_CAP distinct nodes (tables built at upload).  Its threads copy
// those records into LDS with loads in which consecutive lanes read
// consecutive words of one record, so a wavefront touches a few cache lines
// per load instead of one per lane; the walks then read the neighbours from
// LDS.  The arithmetic and its order are those of k_gather with SUB = GB_SUB.
constexpr int GB_SUB = 4;
constexpr int GB_NODES = NTHR / GB_SUB;
constexpr int GB_CAP = 288;

// ---------------------------------------------------------------------------
// node preparation: makePressureField (DEF:13612-13630) + gather records
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ R state_pressure(const DevParams &P, const R *q) {
#pragma clang fp contract(off)
  R pp = R(P.gamma - 1.0) * (q[4] - R(0.5) * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0]);
  return pp > R(0.1) ? pp : R(0.1);
}

template <typename R>
__device__ __forceinline__ void write_momenta(R *mom, int i, R m1, R m2, R m3) {
  if (!mom) return;
  R *m = mom + 4 * (size_t)i;
  m[0] = m1;
  m[1] = m2;
  m[2] = m3;
}

// pressure, gather record (into rec) and momenta (into mom) of node i for the
// state q[6]
template <typename R>
__device__ __forceinline__ void write_record(const LevelDev<R> &L, const DevParams &P, int i, const R *q, R mu,
                                             R *rec, R *mom) {
  R pp = state_pressure(P, q);
  L.p[i] = pp;
  write_momenta(mom, i, q[1], q[2], q[3]);
  R *g = rec + 8 * (size_t)i;
  g[0] = q[0];
  g[1] = q[1] / q[0];
  g[2] = q[2] / q[0];
  g[3] = q[3] / q[0];
  g[4] = q[4];
  g[5] = pp;
  g[6] = P.sa ? q[5] : R(0);
  g[7] = mu;
}

// What a smoothing step starts from: the pressure and gather record of the
// state q[6] and the state itself as the step's previous one (ncopy
// components), and with `zero` an empty dissipation.  Every kernel that
// leaves a level's state ready for its next smoothing step does this in the
// same launch (k_restrict_forcing, k_map_state, k_prolong).
template <typename R>
__device__ __forceinline__ void begin_step(const LevelDev<R> &L, const DevParams &P, int i, const R *q, R mu,
                                           int ncopy, int zero) {
  const size_t n = L.n;
  write_record(L, P, i, q, mu, L.rec0, L.mom);
  for (int c = 0; c < ncopy; ++c) L.uprev[c * n + i] = q[c];
  if (zero)
    for (int c = 0; c < 5; ++c) L.diss[c * n + i] = R(0);
}

// pressure and records of the current state; ncopy > 0 and zero as begin_step
template <typename R>
__global__ void k_prep(LevelDev<R> L, DevParams P, int ncopy, int zero) {
  int bb_;
  int i = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  const size_t n = L.n;
  R q[6];
  for (int c = 0; c < 6; ++c) q[c] = L.u[c * n + i];
  begin_step(L, P, i, q, L.mu[i], ncopy, zero);
}

// gather records from the current state without recomputing p (parity ops)
template <typename R>
__global__ void k_pack(LevelDev<R> L, DevParams P) {
  int bb_;
  int i = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  int n = L.n;
  R r = L.u[i];
  write_momenta(L.mom, i, L.u[n + i], L.u[2 * n + i], L.u[3 * n + i]);
  R *q = L.rec0 + 8 * (size_t)i;
  q[0] = r;
  q[1] = L.u[n + i] / r;
  q[2] = L.u[2 * n + i] / r;
  q[3] = L.u[3 * n + i] / r;
  q[4] = L.u[4 * n + i];
  q[5] = L.p[i];
  q[6] = P.sa ? L.u[5 * n + i] : R(0);
  q[7] = L.mu[i];
}

// ---------------------------------------------------------------------------
// computeGradient (DEF:2923-3245) + LocalMinMax (DEF:3248-3459), gathered
// ---------------------------------------------------------------------------
// In the form of a walk part (init / edge / bside / reduce / finish, like the
// gather parts below): Green-Gauss sums over the interior sides (q_i + q_j) w
// and the boundary sides (3 q_i + q_o) w, and the minimum and maximum of the
// neighbours' values.  GradViscPart carries it along the viscous pass 1 where
// both are due; elsewhere the gradient kernels walk it alone.
// The sums are taken as sum (q_j - q_i) w + sum_b (q_o - q_i) w + 2 q_i W with
// W = sum w + 2 sum_b w, the node's own weights summed without rounding at
// upload (wsum): the terms of q_i cancel over a node's sides, and summed
// with the rest they left a rounding of q_i, not of the differences, that
// depended on the lanes (tangent of RANS 64^3: 1.0e-13 with 4 lanes, 1.2e-13
// with 1; 1.0e-13 so with 1, 4 and 16, at the same time).
template <typename R>
struct GradPart {
  static constexpr int AUXW = 0;
  R q0[5], g[15], mn[5], mx[5];
  __device__ void init(const LevelDev<R> &, const DevParams &, int, const R *qi) {
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      q0[c] = qi[c];
      mn[c] = R(1e15);
      mx[c] = R(1e15);
    }
#pragma unroll
    for (int c = 0; c < 15; ++c) g[c] = 0;
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *, const R *qj, R wx, R wy, R wz) {
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      R d = qj[c] - q0[c];
      g[c] += d * wx;
      g[5 + c] += d * wy;
      g[10 + c] += d * wz;
      R lo = rmin(q0[c], qj[c]);
      R hi = rmin(-q0[c], -qj[c]);
      mn[c] = rmin(mn[c], lo);
      mx[c] = rmin(mx[c], hi);
    }
  }
  __device__ void bside(const LevelDev<R> &, const DevParams &, const R *, int, int, int, const R *qo, R wx, R wy,
                        R wz) {
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      R d = qo[c] - q0[c];
      g[c] += d * wx;
      g[5 + c] += d * wy;
      g[10 + c] += d * wz;
    }
  }
  template <int SUB>
  __device__ void reduce() {
#pragma unroll
    for (int c = 0; c < 15; ++c) g[c] = lsum<SUB>(g[c]);
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      mn[c] = lmin<SUB>(mn[c]);
      mx[c] = lmin<SUB>(mx[c]);
    }
  }
  // the node's own terms, then its record: gradient 15, reciprocal bounds 5 +
  // 5, pad
  __device__ void values(const LevelDev<R> &L, int i, R *out) {
    const R *W = L.wsum + 3 * (size_t)i;
    R wx = R(2) * W[0], wy = R(2) * W[1], wz = R(2) * W[2];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      g[c] += q0[c] * wx;
      g[5 + c] += q0[c] * wy;
      g[10 + c] += q0[c] * wz;
    }
    R vt = R(1) / L.vol[i];
#pragma unroll
    for (int c = 0; c < 15; ++c) out[c] = g[c] * vt;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      R lo = mn[c] - q0[c];
      R hi = -mx[c] - q0[c];
      out[15 + c] = lo < R(0) ? R(1) / lo : R(0);
      out[20 + c] = hi > R(0) ? R(1) / hi : R(0);
    }
    out[25] = 0;
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &, int i, const R *) {
    R v[GREC];
    values(L, i, v);
    R *out = L.grec + GREC * (size_t)i;
#pragma unroll
    for (int c = 0; c < GREC; ++c) out[c] = v[c];
  }
};

// the record of node i into out[26]; false on the lanes that do not own it
template <typename R, int SUB, typename Walk>
__device__ __forceinline__ bool grad_minmax_vals(LevelDev<R> &L, const DevParams &P, int i, int sub, Walk walk,
                                                 R *out) {
  const R *qi = L.rec0 + 8 * (size_t)i;
  GradPart<R> gp;
  gp.init(L, P, i, qi);
  walk([&](const R *qj, const R *tj, R wx, R wy, R wz) { gp.edge(L, P, qi, tj, qj, wx, wy, wz); });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    gp.bside(L, P, qi, s, o, 0, L.rec0 + 8 * (size_t)o, L.wb[3 * s], L.wb[3 * s + 1], L.wb[3 * s + 2]);
  }
  if (SUB > 1) {
    gp.template reduce<SUB>();
    if (sub) return false;
  }
  gp.values(L, i, out);
  return true;
}

template <typename R, int SUB, typename Walk>
__device__ __forceinline__ void grad_minmax_body(LevelDev<R> &L, const DevParams &P, int i, int sub, Walk walk) {
  R v[GREC];
  if (!grad_minmax_vals<R, SUB>(L, P, i, sub, walk, v)) return;
  R *out = L.grec + GREC * (size_t)i;
#pragma unroll
  for (int c = 0; c < GREC; ++c) out[c] = v[c];
}

// the block's records stored through LDS in two halves of 13 words (one node
// per thread): a thread's record lands in LDS at a 13-word stride
// (conflict-free for 64-bit words), then consecutive lanes store
// consecutive words of the block's contiguous record range, instead of
// every store instruction touching one cache line per lane
template <typename R>
__device__ __forceinline__ void store_grec(R *st, const R *v, bool ok, R *base, int cnt) {
  constexpr int HW = GREC / 2;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (ok) {
#pragma unroll
      for (int c = 0; c < HW; ++c) st[threadIdx.x * HW + c] = v[h * HW + c];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < HW; ++k) {
      int idx = k * NTHR + (int)threadIdx.x;
      int node = idx / HW, cc = idx - node * HW;
      if (node < cnt) base[GREC * (size_t)node + h * HW + cc] = st[idx];
    }
    __syncthreads();
  }
}

template <typename R>
__global__ void __launch_bounds__(NTHR) k_grad_minmax_st(LevelDev<R> L, DevParams P) {
  __shared__ R st[NTHR * (GREC / 2)];
  int bb_;
  int i = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  const int i0 = i - (int)threadIdx.x;
  R v[GREC];
  bool ok = i < L.n && grad_minmax_vals<R, 1>(L, P, i, 0, [&](auto f) { walk_global<1>(L, i, 0, f); }, v);
  store_grec(st, v, ok, L.grec + GREC * (size_t)i0, L.n - i0 < NTHR ? L.n - i0 : NTHR);
}

template <typename R, int SUB>
__global__ void k_grad_minmax(LevelDev<R> L, DevParams P) {
  int i, sub;
  int bb_;
  node_lanes<SUB>(L.nb, bb_, i, sub);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  grad_minmax_body<R, SUB>(L, P, i, sub, [&](auto f) { walk_global<SUB>(L, i, sub, f); });
}

// Reciprocal and reciprocal square root in the FP64 flux: the hardware
// estimates (v_rcp_f64, v_rsq_f64) refined by two Newton-Raphson steps,
// y <- y + y (1 - b y) and y <- y + y (1/2 - x y^2 / 2), as fused
// multiply-adds.  The results stay within a few ulp of the correctly rounded
// quotient and root at about half the instructions of the IEEE sequences.
// frcp needs a finite nonzero argument (every call site guarantees it);
// frsqrt maps +inf to 0 as 1/sqrt does.  Other arithmetic types (FP32
// levels, dual numbers) use the plain operations.
template <typename T>
__device__ __forceinline__ T frcp(T b) { return T(1) / b; }
template <>
__device__ __forceinline__ double frcp<double>(double b) {
  double y = __builtin_amdgcn_rcp(b);
  double e = fma(-b, y, 1.0);
  y = fma(y, e, y);
  e = fma(-b, y, 1.0);
  return fma(y, e, y);
}
template <typename T>
__device__ __forceinline__ T frsqrt(T x) { return T(1) / sqrt(x); }
template <>
__device__ __forceinline__ double frsqrt<double>(double x) {
  double y = __builtin_amdgcn_rsq(x);
  double h = 0.5 * x;
  double e = fma(-h * y, y, 0.5);
  y = fma(y, e, y);
  e = fma(-h * y, y, 0.5);
  y = fma(y, e, y);
  return x == __builtin_inf() ? 0.0 : y;
}

// LED local clipping (DEF:1852-1889) with precomputed reciprocal bounds.
// Branch-free: the bound is selected by the sign of a, so a wavefront
// evaluates the reciprocal root once whatever the signs of its lanes.
template <int NSIG, typename R>
__device__ __forceinline__ R led(R a, R ilo, R ihi) {
  R a1 = R(2) * a;
  R iv = a1 > R(0) ? ihi : ilo;
  R t = a1 * iv, t2 = t * t;
  R iden = NSIG == 4 ? frsqrt(sqrt(R(1) + t2 * t2)) : frsqrt(R(1) + t2);
  R r = a * iden;  // the reference's 0.5 * a1 * iden: 0.5 * (2 a) is a exactly
  r = iv == R(0) ? R(0) : r;
  return (a1 > R(0) || a1 < R(0)) ? r : a;  // a == 0 (or NaN) passes through
}

// HLLC interior flux of one side (makeRHS, DEF:1794-2100) from the two
// ends' gather records A, B (rho, u, v, w, rhoE, p, nu~, mu) and the side
// weights; writes o[0..5] (component 5: SA convection, DEF:6873-6880).
// Second order also reads both ends' gradient records G1, G2 (grad 15 |
// 1/lo 5 | 1/hi 5), of type TG (R, or dual numbers for the linearisation),
// and coordinates X1, X2; first order ignores them.
// T is the arithmetic type: the level's R for the residual, a dual number
// for its tangent and its mesh adjoint; with T a dual number the second-order branch
// takes the gradient records (TG) and the coordinates (TX) as dual numbers
// too when their derivatives are wanted.
// upwinded SA convection of one side (makeSARHS, DEF:6873-6880) from the
// ends' gather records
//
// Its linearisation takes the upwind term's sign from sa_upwind alone: x =
// w.(m_b - m_a) of m = nu~ v against nu~_a - nu~_b, 0 where either vanishes
// (fluid at rest at both ends, say), which counts as positive seen from the
// side's first end.  Without contraction x has the same bits from either end
// (differences and weights change sign together), so the tangent and both
// ends' shares of the adjoint take one branch.
__device__ __forceinline__ int sa_upwind(const double *ma, const double *mb, double ta, double tb, double wx, double wy,
                                         double wz) {
#pragma clang fp contract(off)
  const double x = wx * (mb[0] * tb - ma[0] * ta) + wy * (mb[1] * tb - ma[1] * ta) + wz * (mb[2] * tb - ma[2] * ta);
  const double dt = ta - tb;
  if (x == 0.0 || dt == 0.0) return 0;
  return (x < 0.0) == (dt < 0.0) ? 1 : -1;
}
template <typename T>
__device__ __forceinline__ T sa_side_convection(const T *A, const T *B, T wx, T wy, T wz) {
  T u1 = A[1], v1 = A[2], w1 = A[3], t1 = A[6];
  T u2 = B[1], v2 = B[2], w2 = B[3], t2 = B[6];
  T fsa = wx * (u1 * t1 + u2 * t2) + wy * (v1 * t1 + v2 * t2) + wz * (w1 * t1 + w2 * t2);
  T dtt = t1 - t2;
  if (fabs(dtt) > T(1e-20)) {
    T id = frcp(dtt);
    T ax = (u2 * t2 - u1 * t1) * id, ay = (v2 * t2 - v1 * t1) * id, az = (w2 * t2 - w1 * t1) * id;
    T y = wx * ax + wy * ay + wz * az;
    if constexpr (std::is_same_v<T, ad::Dual>) {
      const double ma[3] = {u1.v, v1.v, w1.v}, mb[3] = {u2.v, v2.v, w2.v};
      y = sa_upwind(ma, mb, t1.v, t2.v, wx.v, wy.v, wz.v) < 0 ? -y : y;
    } else {
      y = fabs(y);
    }
    fsa = fsa + y * dtt;
  }
  return fsa;
}

// MUSCL slope of component j (DEF:1840-1944): the two ends' projected
// gradients a, b (before limiting), the LED bounds of the first end (ilo1,
// ihi1) and of the second (ilo2, ihi2), the clip length hl
template <int NSIG, typename T>
__device__ __forceinline__ T muscl_slope(const DevParams &P, T a, T b, T ilo1, T ihi1, T ilo2, T ihi2, T hl) {
  if (P.autoclip == 1) {
    a = led<NSIG>(a, ilo1, ihi1);
    b = -led<NSIG>(-b, ilo2, ihi2);
  }
  T c;
  if (a * b <= T(0)) {
    c = 0;
  } else {
    c = fabs(a) <= fabs(b) ? a : b;
    if (fabs(c) > hl && hl > T(0)) c = c > T(0) ? hl : -hl;
  }
  return c;
}

// a node's gradient of component j projected on half the side vector
template <typename T, typename TG>
__device__ __forceinline__ T muscl_projection(const TG *G, T dx, T dy, T dz, int j) {
  return T(0.5) * (G[j] * dx + G[j + 5] * dy + G[j + 10] * dz);
}

// the side's half-length clip hl and projected gradients a[5], b[5]
template <typename T, typename TG, typename TX>
__device__ __forceinline__ T muscl_projections(const DevParams &P, const TG *G1, const TG *G2, const TX *X1,
                                               const TX *X2, T *a, T *b) {
  T dx = X2[0] - X1[0], dy = X2[1] - X1[1], dz = X2[2] - X1[2];
  T hl = T(0.5) * T(P.clip) * sqrt(dx * dx + dy * dy + dz * dz);
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    a[j] = muscl_projection<T>(G1, dx, dy, dz, j);
    b[j] = muscl_projection<T>(G2, dx, dy, dz, j);
  }
  return hl;
}

template <typename T, typename R, bool SA>
__device__ __forceinline__ void side_flux_d(const DevParams &P, const T *A, const T *B, const T *d, T wx, T wy, T wz,
                                            T *o, R wg);

template <typename T, typename R, int ORDER, bool SA, int NSIG, typename TG = R, typename TX = R>
__device__ __forceinline__ void side_flux(const DevParams &P, const TG *G1, const TG *G2, const TX *X1, const TX *X2,
                                          const T *A, const T *B, T wx, T wy, T wz, T *o, R wg = R(0)) {
  if constexpr (ORDER > 1) {
    T a[5], b[5], d[5];
    T hl = muscl_projections<T>(P, G1, G2, X1, X2, a, b);
#pragma unroll
    for (int j = 0; j < 5; ++j)
      d[j] = muscl_slope<NSIG, T>(P, a[j], b[j], T(G1[15 + j]), T(G1[20 + j]), T(G2[15 + j]), T(G2[20 + j]), hl);
    side_flux_d<T, R, SA>(P, A, B, d, wx, wy, wz, o, wg);
  } else {
    side_flux_d<T, R, SA>(P, A, B, (const T *)nullptr, wx, wy, wz, o, wg);
  }
}

// the HLLC flux of one side from the two ends' records and the MUSCL slopes
// d[5] of the primitive states (null: first order): the left state is A + d,
// the right B - d, with the reference's positivity guards
template <typename T, typename R, bool SA>
__device__ __forceinline__ void side_flux_d(const DevParams &P, const T *A, const T *B, const T *d, T wx, T wy, T wz,
                                            T *o, R wg) {
  T gam = T(P.gamma), gm1 = gam - T(1);
  T roe1 = A[0], u1 = A[1], v1 = A[2], w1 = A[3], re1 = A[4], pr1 = A[5];
  T roe2 = B[0], u2 = B[1], v2 = B[2], w2 = B[3], re2 = B[4], pr2 = B[5];
  T fsa = 0;
  if (SA) fsa = sa_side_convection(A, B, wx, wy, wz);
  T ru1 = roe1 * u1, rv1 = roe1 * v1, rw1 = roe1 * w1, rh1 = re1 + pr1;
  T ru2 = roe2 * u2, rv2 = roe2 * v2, rw2 = roe2 * w2, rh2 = re2 + pr2;
  T nx = T(2) * wx, ny = T(2) * wy, nz = T(2) * wz;
  T n2 = nx * nx + ny * ny + nz * nz;
  T inv = n2 > T(0) ? frsqrt(n2) : T(0);
  T rnorm1 = n2 * inv;  // |2w|
  T rnx = nx * inv, rny = ny * inv, rnz = nz * inv;
  if (d) {
    if (roe1 + d[0] > T(0.1)) roe1 = roe1 + d[0];
    u1 += d[1]; v1 += d[2]; w1 += d[3];
    if (re1 + d[4] > T(0.0001)) re1 = re1 + d[4];
    pr1 = gm1 * (re1 - T(0.5) * (u1 * u1 + v1 * v1 + w1 * w1) * roe1);
    pr1 = pr1 > T(0.1) ? pr1 : T(0.1);
    rh1 = re1 + pr1;
    ru1 = roe1 * u1; rv1 = roe1 * v1; rw1 = roe1 * w1;
    if (roe2 - d[0] > T(0.1)) roe2 = roe2 - d[0];
    u2 -= d[1]; v2 -= d[2]; w2 -= d[3];
    if (re2 - d[4] > T(0.0001)) re2 = re2 - d[4];
    pr2 = gm1 * (re2 - T(0.5) * (u2 * u2 + v2 * v2 + w2 * w2) * roe2);
    pr2 = pr2 > T(0.1) ? pr2 : T(0.1);
    rh2 = re2 + pr2;
    ru2 = roe2 * u2; rv2 = roe2 * v2; rw2 = roe2 * w2;
  }
  T rinv1 = frcp(roe1), rinv2 = frcp(roe2);
  T nv1 = u1 * rnx + v1 * rny + w1 * rnz;
  T nv2 = u2 * rnx + v2 * rny + w2 * rnz;
  T beta0 = T(P.beta0);
  T rroe = sqrt(roe2 * rinv1);
  T iro = frcp(T(1) + rroe);
  T ut = (u1 + u2 * rroe) * iro, vt = (v1 + v2 * rroe) * iro, wt = (w1 + w2 * rroe) * iro;
  T qt = ut * rnx + vt * rny + wt * rnz;
  T ht = (rh1 * rinv1 + rh2 * rinv2 * rroe) * iro;
  T ct = sqrt(fabs(gm1 * (ht - T(0.5) * (ut * ut + vt * vt + wt * wt))));
  T c1 = sqrt(gm1 * fabs(rh1 * rinv1 - T(0.5) * (u1 * u1 + v1 * v1 + w1 * w1)));
  T c2 = sqrt(gm1 * fabs(rh2 * rinv2 - T(0.5) * (u2 * u2 + v2 * v2 + w2 * w2)));
  T sl = fmin(fmin(nv1 - beta0 * c1, qt - ct), nv2 - beta0 * c2);
  T sr = fmax(fmax(nv2 + beta0 * c2, qt + ct), nv1 + beta0 * c1);
  T sm = roe2 * nv2 * (sr - nv2) - roe1 * nv1 * (sl - nv1) + pr1 - pr2;
  T fact = roe2 * (sr - nv2) - roe1 * (sl - nv1);
  if (fact != T(0)) fact = frcp(fact);
  sm = fact * sm;
  // upwind side K: left when sl > 0 or (sl <= 0 < sm), right when
  // sm <= 0 <= sr or sr < 0; neither only for NaN wave speeds, where the
  // central flux is kept.  Both sides share one code path (selected
  // operands), so a wavefront evaluates the star state once.
  bool lft = sl > T(0) || (sl <= T(0) && sm > T(0));
  bool rgt = (sm <= T(0) && sr >= T(0)) || sr < T(0);
  if (!lft && !rgt) {
    // the central part of the nodes' states (DEF:1798-1802), kept when no
    // HLLC branch is taken (NaN wave speeds)
    T a1 = A[0] * A[1], a2 = A[0] * A[2], a3 = A[0] * A[3], ah = A[4] + A[5];
    T b1 = B[0] * B[1], b2 = B[0] * B[2], b3 = B[0] * B[3], bh = B[4] + B[5];
    o[0] = wx * (a1 + b1) + wy * (a2 + b2) + wz * (a3 + b3);
    o[1] = wx * (a1 * A[1] + A[5] + b1 * B[1] + B[5]) + wy * (a1 * A[2] + b1 * B[2]) + wz * (a1 * A[3] + b1 * B[3]);
    o[2] = wx * (a2 * A[1] + b2 * B[1]) + wy * (a2 * A[2] + A[5] + b2 * B[2] + B[5]) + wz * (a2 * A[3] + b2 * B[3]);
    o[3] = wx * (a3 * A[1] + b3 * B[1]) + wy * (a3 * A[2] + b3 * B[2]) + wz * (a3 * A[3] + A[5] + b3 * B[3] + B[5]);
    o[4] = wx * (ah * A[1] + bh * B[1]) + wy * (ah * A[2] + bh * B[2]) + wz * (ah * A[3] + bh * B[3]);
    if (wg != R(0)) {  // moving mesh: the left state's GCL share (DEF:2081-2085)
      o[0] -= A[0] * wg;
      o[1] -= ru1 * wg;
      o[2] -= rv1 * wg;
      o[3] -= rw1 * wg;
      o[4] -= A[4] * wg;
    }
    o[5] = fsa;
    return;
  }
  T rk = lft ? roe1 : roe2, uk = lft ? u1 : u2, vk = lft ? v1 : v2, wk = lft ? w1 : w2;
  T ek = lft ? re1 : re2, pk = lft ? pr1 : pr2, nvk = lft ? nv1 : nv2;
  T ruk = lft ? ru1 : ru2, rvk = lft ? rv1 : rv2, rwk = lft ? rw1 : rw2, rhk = lft ? rh1 : rh2;
  T sk = lft ? sl : sr;
  bool star = lft ? !(sl > T(0)) : !(sr < T(0));
  T f[5];
  f[0] = rnx * ruk + rny * rvk + rnz * rwk;
  f[1] = rnx * (ruk * uk + pk) + rny * (ruk * vk) + rnz * (ruk * wk);
  f[2] = rnx * (rvk * uk) + rny * (rvk * vk + pk) + rnz * (rvk * wk);
  f[3] = rnx * (rwk * uk) + rny * (rwk * vk) + rnz * (rwk * wk + pk);
  f[4] = rnx * (rhk * uk) + rny * (rhk * vk) + rnz * (rhk * wk);
  T fk = sk - sm;
  // the state the flux is taken from (DEF:2081-2085 subtract it times the
  // side's GCL weight / dt on a moving mesh): the star state, or U_K with
  // the node's own density and energy and the reconstructed momentum (the
  // reference's r1, E1 are not reconstructed, its ru1..rw1 are)
  T q0 = lft ? A[0] : B[0], q1 = ruk, q2 = rvk, q3 = rwk, q4 = lft ? A[4] : B[4];
  if (star && fk == T(0)) {  // degenerate star state: U_K as reconstructed (DEF:1997-2003, 2012-2018)
    q0 = rk;
    q4 = ek;
  } else if (star) {
    fk = frcp(fk);
    T a = sk - nvk;
    T pks = rk * (nvk - sk) * (nvk - sm) + pk;
    T ps = pks - pk;
    T s0 = rk * a * fk, s1 = (a * rk * uk + ps * rnx) * fk;
    T s2 = (a * rk * vk + ps * rny) * fk, s3 = (a * rk * wk + ps * rnz) * fk;
    T s4 = (a * ek - pk * nvk + pks * sm) * fk;
    f[0] += sk * (s0 - rk);
    f[1] += sk * (s1 - ruk);
    f[2] += sk * (s2 - rvk);
    f[3] += sk * (s3 - rwk);
    f[4] += sk * (s4 - ek);
    q0 = s0;
    q1 = s1;
    q2 = s2;
    q3 = s3;
    q4 = s4;
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) o[c] = f[c] * rnorm1;
  if (wg != R(0)) {
    o[0] -= q0 * wg;
    o[1] -= q1 * wg;
    o[2] -= q2 * wg;
    o[3] -= q3 * wg;
    o[4] -= q4 * wg;
  }
  o[5] = fsa;
}

// HLLC interior flux (makeRHS, DEF:1794-2100), one evaluation per edge.
// fbuf[6*e + c]: flux leaving ea towards eb (+ to ea, - to eb).
template <typename R, int ORDER, bool SA, int NSIG>
__global__ void k_flux(LevelDev<R> L, DevParams P) {
  int bb_;
  int e = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (e >= L.ne) return;
  int ia = L.ea[e], ib = L.eb[e];
  R A[8], B[8];
  ldrec<8>(L.rec0 + 8 * (size_t)ia, A);
  ldrec<8>(L.rec0 + 8 * (size_t)ib, B);
  R wx = L.w[3 * e], wy = L.w[3 * e + 1], wz = L.w[3 * e + 2];
  const R *G1 = nullptr, *G2 = nullptr, *X1 = nullptr, *X2 = nullptr;
  if constexpr (ORDER > 1) {
    G1 = L.grec + GREC * (size_t)ia;
    G2 = L.grec + GREC * (size_t)ib;
    X1 = L.xyz + 3 * (size_t)ia;
    X2 = L.xyz + 3 * (size_t)ib;
  }
  R wg = L.gcl ? L.gcl[e] / R(P.dtp) : R(0);
  side_flux<R, R, ORDER, SA, NSIG>(P, G1, G2, X1, X2, A, B, wx, wy, wz, L.fbuf + 6 * (size_t)e, wg);
}

// physical flux of one state through unit normal
template <typename R>
__device__ __forceinline__ void phys_flux(const R *q, R rnx, R rny, R rnz, R *f) {
  R rho = q[0], u = q[1], v = q[2], w = q[3], pr = q[5], rh = q[4] + q[5];
  R nv = u * rnx + v * rny + w * rnz;
  f[0] = rho * nv;
  f[1] = pr * rnx + rho * u * nv;
  f[2] = pr * rny + rho * v * nv;
  f[3] = pr * rnz + rho * w * nv;
  f[4] = rh * nv;
}

// farfield Roe flux of one state against the inflow state (DEF:2258-2446)
template <typename R>
__device__ __forceinline__ void farfield_roe(const double *inf, const R *q, R gm1, R rnx, R rny, R rnz, R *f) {
  R ro = R(inf[0]), uo = R(inf[1]), vo = R(inf[2]), wo = R(inf[3]), eo = R(inf[4]), po = R(inf[5]);
  R rho = q[0], uu = q[1], vv = q[2], ww = q[3], eps = q[4], pr = q[5];
  R rh = eps + pr, h = rh / rho;
  R nv = uu * rnx + vv * rny + ww * rnz;
  R fl1 = rho * nv, fl2 = pr * rnx + rho * uu * nv, fl3 = pr * rny + rho * vv * nv;
  R fl4 = pr * rnz + rho * ww * nv, fl5 = rh * nv;
  R epsr = eo * ro, hr = eo + po / ro;
  R unr = uo * rnx + vo * rny + wo * rnz;
  R fr1 = ro * unr, fr2 = rnx * po + ro * uo * unr, fr3 = rny * po + ro * vo * unr;
  R fr4 = rnz * po + ro * wo * unr, fr5 = (epsr + po) * unr;
  R di = sqrt(ro / rho), d1 = R(1) / (di + R(1));
  R ui = (di * uo + uu) * d1, vi = (di * vo + vv) * d1, wi = (di * wo + ww) * d1, hi = (di * hr + h) * d1;
  R af = R(0.5) * (ui * ui + vi * vi + wi * wi);
  R ci2 = gm1 * (hi - af);
  ci2 = ci2 > R(1e-5) ? ci2 : R(1e-5);
  R ci = sqrt(ci2), ici = R(1) / ci;
  R ucp = ui * rnx + vi * rny + wi * rnz;
  R du1 = ro - rho, du2 = ro * uo - rho * uu, du3 = ro * vo - rho * vv;
  R du4 = ro * wo - rho * ww, du5 = epsr - eps;
  R rl1 = fabs(ucp + ci), rl2 = fabs(ucp - ci), rl3 = fabs(ucp);
  R s1 = R(0.5) * (rl1 + rl2), s2 = R(0.5) * (rl1 - rl2);
  R al1x = gm1 * (af * du1 - ui * du2 - vi * du3 - wi * du4 + du5);
  R al2x = -ucp * du1 + du2 * rnx + du3 * rny + du4 * rnz;
  R cc1 = ((s1 - rl3) * al1x / ci2) + (s2 * al2x * ici);
  R cc2 = (s2 * al1x * ici) + (s1 - rl3) * al2x;
  f[0] = R(0.5) * (fr1 + fl1) - R(0.5) * (rl3 * du1 + cc1);
  f[1] = R(0.5) * (fr2 + fl2) - R(0.5) * (rl3 * du2 + cc1 * ui + cc2 * rnx);
  f[2] = R(0.5) * (fr3 + fl3) - R(0.5) * (rl3 * du3 + cc1 * vi + cc2 * rny);
  f[3] = R(0.5) * (fr4 + fl4) - R(0.5) * (rl3 * du4 + cc1 * wi + cc2 * rnz);
  f[4] = R(0.5) * (fr5 + fl5) - R(0.5) * (rl3 * du5 + cc1 * hi + cc2 * ucp);
}

// the boundary flux of one end's state along the side's unit normal
template <typename R>
__device__ __forceinline__ void bside_state_flux(const DevParams &P, int ind, const R *q, R rnx, R rny, R rnz, R *f) {
  if (ind <= 2 || ind == 9) {
    phys_flux(q, rnx, rny, rnz, f);
  } else {
    double inf[6];
    P.inflow_row(ind - 3, inf);
    farfield_roe(inf, q, R(P.gamma - 1.0), rnx, rny, rnz, f);
  }
}

// boundary-side loop of makeRHS (DEF:2116-2446): contributions to both ends,
// bbuf[10*s + 5*end + c]
template <typename R>
__device__ __forceinline__ void bflux_side(const LevelDev<R> &L, const DevParams &P, int s) {
  int ia = L.ba[s], ib = L.bb[s], ind = L.bind[s];
  R wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
  R *o = L.bbuf + 10 * (size_t)s;
  // moving mesh: -(3 U_1 + U_2) g_1 / dt to the first end, -(U_1 + 3 U_2)
  // g_2 / dt to the second (boundaryTerm 1), -4 U_k g_k / dt otherwise, on
  // every boundary side (DEF:2124-2179)
  R gc[10];
#pragma unroll
  for (int c = 0; c < 10; ++c) gc[c] = 0;
  if (L.bgcl) {
    const size_t n = L.n;
    R g1 = L.bgcl[2 * (size_t)s] / R(P.dtp), g2 = L.bgcl[2 * (size_t)s + 1] / R(P.dtp);
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      R a = L.u[c * n + ia], b = L.u[c * n + ib];
      if (P.bterm == 1) {
        gc[c] = -(R(3) * a + b) * g1;
        gc[5 + c] = -(a + R(3) * b) * g2;
      } else {
        gc[c] = -a * (R(4) * g1);
        gc[5 + c] = -b * (R(4) * g2);
      }
    }
  }
  R rnorm = sqrt(wx * wx + wy * wy + wz * wz);
  if (!(rnorm > R(1e-10)) || !(ind <= 4 || ind == 9)) {
#pragma unroll
    for (int c = 0; c < 10; ++c) o[c] = gc[c];
    return;
  }
  R irn = R(1) / rnorm;
  R rnx = wx * irn, rny = wy * irn, rnz = wz * irn;
  const R *A = L.rec0 + 8 * (size_t)ia;
  const R *B = L.rec0 + 8 * (size_t)ib;
  R f1[5], f2[5];
  bside_state_flux(P, ind, A, rnx, rny, rnz, f1);
  bside_state_flux(P, ind, B, rnx, rny, rnz, f2);
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    if (P.bterm == 1) {
      o[c] = gc[c] + rnorm * (R(3) * f1[c] + f2[c]);
      o[5 + c] = gc[5 + c] + rnorm * (f1[c] + R(3) * f2[c]);
    } else {
      o[c] = gc[c] + rnorm * R(4) * f1[c];
      o[5 + c] = gc[5 + c] + rnorm * R(4) * f2[c];
    }
  }
}

template <typename R>
__global__ __launch_bounds__(NTHR) void k_bflux(LevelDev<R> L, DevParams P) {
  int bb_;
  int s = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (s >= L.nbs) return;
  bflux_side(L, P, s);
}

// The same flux with the two ends' records staged in LDS per block of
// sides, and the sides' fluxes summed per node inside the block.  A block
// serves up to FB_SIDES consecutive sides that touch at most FB_NODES
// distinct nodes (tables built at upload).  Its threads first copy the words
// of those nodes' records that the flux reads into LDS, with loads in which
// consecutive lanes read consecutive words of one record, so a wavefront
// touches a few cache lines per load instead of one line per lane; each
// thread then evaluates its side from LDS.  The block then sums, for each of
// its nodes, +f over the sides the node starts and -f over the sides it
// ends (two lanes per node, each over alternate sides of the node's list in
// side order, then the two sums added), and writes that partial sum to pbuf
// (one 6-word entry per block and node, in the order of the block's node
// list).  A node's
// residual is the sum of its entries in block order (k_stage), which
// replaces the gather of one flux record per incident side by a few partial
// sums per node.
// Every load of a block depends on its header or on nothing: the node list
// sits at a fixed place per block, so the records are two loads away from
// the start, and the sides' own words are requested before the staging.  The
// list goes through LDS, and all three records' loads are requested before
// the first is stored: reading the list beside every record load and waiting
// for each record in turn kept 24 reads in flight a CU and took 884 us on
// 14.8M sides (second order, SA), 656 now; 219 and 165 on 3.6M.
// BND: blocks spread evenly among the side blocks evaluate the boundary sides,
// one a thread, instead of a launch of their own (k_bflux).  That saves the
// launch where it is the cost: us merged / apart, first order 16 / 24 with 19k
// boundary sides and 72 / 71 with 89k; second order with SA 46 / 52 with 41k,
// 87 / 93 with 74k, 125 / 127 with 93k, 164 / 165 with 115k, but 343 / 341
// with 195k and 676 / 663 with 295k (the longer code takes registers from the
// sides).
// side-block shapes: FB_SHAPE_THR[k] sides per block (one thread each)
// touching at most FB_SHAPE_NODES[k] distinct nodes; the autotuner picks
// one per level (shape 0 unless it finds another faster)
constexpr int FB_NSHAPES = 2;
constexpr int FB_SHAPE_THR[FB_NSHAPES] = {256, 512};
constexpr int FB_SHAPE_NODES[FB_NSHAPES] = {128, 224};
static_assert(2 * FB_SHAPE_NODES[0] <= FB_SHAPE_THR[0] && 2 * FB_SHAPE_NODES[1] <= FB_SHAPE_THR[1],
              "two threads per staged node in the node sums");
constexpr int FB_REC = 7;  // gather-record words the flux reads (not mu)
constexpr int FB_SF = 7;   // LDS stride of a side flux (6 words, odd stride)
template <int ORDER>
constexpr int fb_stride() {  // LDS words per node: record 7 | grad + bounds 25 | coordinates 3
  return ORDER > 1 ? FB_REC + GREC - 1 + 3 : FB_REC;  // odd: lanes reading different nodes spread over banks
}
template <typename R, int ORDER, bool SA, int NSIG, int SHAPE, bool BND>
__global__ __launch_bounds__(FB_SHAPE_THR[SHAPE]) void k_flux_blk(LevelDev<R> L, DevParams P) {
  constexpr int FB_THR = FB_SHAPE_THR[SHAPE], FB_SIDES = FB_THR, FB_NODES = FB_SHAPE_NODES[SHAPE];
  constexpr int S = fb_stride<ORDER>();
  constexpr int SN = FB_NODES * S > FB_SIDES * FB_SF ? FB_NODES * S : FB_SIDES * FB_SF;
  __shared__ R sn[SN];
  __shared__ int sid[FB_NODES];
  __shared__ unsigned short sinc[2 * FB_SIDES];
  int lb = xcd_block();
  int bb_ = lb % L.nb, blk = lb / L.nb;
  L.to_batch(bb_);
  P.to_batch(bb_);
  if constexpr (BND) {
    const int nbb = (L.nbs + FB_THR - 1) / FB_THR, all = L.nfb + nbb;
    const int before = (int)((long long)blk * nbb / all);  // boundary blocks before this one
    if ((int)((long long)(blk + 1) * nbb / all) > before) {
      const int s = before * FB_THR + (int)threadIdx.x;
      if (s < L.nbs) bflux_side(L, P, s);
      return;
    }
    blk -= before;
  } else if (blk >= L.nfb) {
    return;
  }
  const int4 h0 = reinterpret_cast<const int4 *>(L.fb_head)[blk];
  const int4 h1 = reinterpret_cast<const int4 *>(L.fb_head)[blk + 1];
  const int n0 = h0.y, nn = h1.y - h0.y, ibase = h0.z;
  if (threadIdx.x < FB_NODES) sid[threadIdx.x] = L.fb_node[(size_t)blk * FB_NODES + threadIdx.x];
  // this thread's side: its words are requested before the staging
  const int e = h0.x + (int)threadIdx.x;
  const bool active = e < h1.x;
  unsigned loc = 0;
  R wx = 0, wy = 0, wz = 0, wg = 0;
  if (active) {
    loc = L.fb_loc[e];
    wx = L.w[3 * (size_t)e];
    wy = L.w[3 * (size_t)e + 1];
    wz = L.w[3 * (size_t)e + 2];
    if (L.gcl) wg = L.gcl[e] / R(P.dtp);
  }
  // this thread's node (two threads per node, `half` of its incidences
  // each) and the block's incidence lists
  int q0 = 0, q1 = 0;
  const int me = (int)threadIdx.x >> 1, half = (int)threadIdx.x & 1;
  if (me < nn) {
    q0 = L.fb_iptr[n0 + me] - ibase;
    q1 = L.fb_iptr[n0 + me + 1] - ibase;
  }
  {
    const int ni = h1.z - ibase;  // 2 x sides of the block
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      int t = threadIdx.x + q * FB_THR;
      if (t < ni) sinc[t] = L.fb_inc[ibase + t];
    }
  }
  // the nodes' records, all loads in flight before the first goes to LDS
  __syncthreads();
  {
    using P2 = typename Pair<R>::type;
    const int t = threadIdx.x;
    constexpr int U0 = 4, U1 = GREC / 2;  // two-word units of the two records
    constexpr int N0 = (FB_NODES * U0 + FB_THR - 1) / FB_THR;
    constexpr int N1 = ORDER > 1 ? (FB_NODES * U1 + FB_THR - 1) / FB_THR : 0;
    constexpr int N2 = ORDER > 1 ? (FB_NODES * 3 + FB_THR - 1) / FB_THR : 0;
    P2 v0[N0], v1[N1 ? N1 : 1];
    R v2[N2 ? N2 : 1];
#pragma unroll
    for (int q = 0; q < N0; ++q) {
      const int x = t + q * FB_THR, k = x / U0;
      if (k < nn) v0[q] = reinterpret_cast<const P2 *>(L.rec0 + 8 * (size_t)sid[k])[x - k * U0];
    }
#pragma unroll
    for (int q = 0; q < N1; ++q) {
      const int x = t + q * FB_THR, k = x / U1;
      if (k < nn) v1[q] = reinterpret_cast<const P2 *>(L.grec + GREC * (size_t)sid[k])[x - k * U1];
    }
#pragma unroll
    for (int q = 0; q < N2; ++q) {
      const int x = t + q * FB_THR, k = x / 3;
      if (k < nn) v2[q] = L.xyz[3 * (size_t)sid[k] + (x - 3 * k)];
    }
#pragma unroll
    for (int q = 0; q < N0; ++q) {
      const int x = t + q * FB_THR, k = x / U0, j = x - k * U0;
      if (k < nn) {
        sn[k * S + 2 * j] = v0[q].x;
        if (2 * j + 1 < FB_REC) sn[k * S + 2 * j + 1] = v0[q].y;
      }
    }
#pragma unroll
    for (int q = 0; q < N1; ++q) {
      const int x = t + q * FB_THR, k = x / U1, j = x - k * U1;
      if (k < nn) {
        sn[k * S + FB_REC + 2 * j] = v1[q].x;
        if (2 * j + 1 < GREC - 1) sn[k * S + FB_REC + 2 * j + 1] = v1[q].y;
      }
    }
#pragma unroll
    for (int q = 0; q < N2; ++q) {
      const int x = t + q * FB_THR, k = x / 3;
      if (k < nn) sn[k * S + FB_REC + GREC - 1 + (x - 3 * k)] = v2[q];
    }
  }
  __syncthreads();
  R fo[6];
  if (active) {
    const R *na = sn + (loc & 0xffffu) * S, *nb = sn + (loc >> 16) * S;
    const R *G1 = nullptr, *G2 = nullptr, *X1 = nullptr, *X2 = nullptr;
    if constexpr (ORDER > 1) {
      G1 = na + FB_REC;
      G2 = nb + FB_REC;
      X1 = na + FB_REC + GREC - 1;
      X2 = nb + FB_REC + GREC - 1;
    }
    side_flux<R, R, ORDER, SA, NSIG>(P, G1, G2, X1, X2, na, nb, wx, wy, wz, fo, wg);
  }
  __syncthreads();  // node records no longer needed: the side fluxes take their place
  R *sf = sn;
  if (active) {
#pragma unroll
    for (int c = 0; c < 6; ++c) sf[FB_SF * threadIdx.x + c] = fo[c];
  }
  __syncthreads();
  // node sums: the pair of lanes serving a node sums the even and the odd
  // positions of its incidence list, then adds the two sums (the same bits
  // on both lanes), and each lane stores three of the six words
  if (me < nn) {
    const int ent = n0 + me;
    R r[6] = {0, 0, 0, 0, 0, 0};
    for (int q = q0 + half; q < q1; q += 2) {
      unsigned v = sinc[q];
      const R *f = sf + FB_SF * (v >> 1);
      if (v & 1u) {
#pragma unroll
        for (int c = 0; c < 6; ++c) r[c] -= f[c];
      } else {
#pragma unroll
        for (int c = 0; c < 6; ++c) r[c] += f[c];
      }
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) r[c] += __shfl_xor(r[c], 1);
    R *o = L.pbuf + 6 * (size_t)ent + 3 * half;
    o[0] = half ? r[3] : r[0];
    o[1] = half ? r[4] : r[1];
    o[2] = half ? r[5] : r[2];
  }
}

// ---------------------------------------------------------------------------
// Interior fluxes 1-3 and their JST dissipation
// ---------------------------------------------------------------------------
// Interior side flux of fluxType 1 (central, DEF:1664-1669), 2 (local
// Lax-Friedrichs, DEF:1670-1724) or 3 (Roe, DEF:1725-1792) from the ends'
// conserved states and pressures, without reconstruction.  LLF and Roe are
// the textbook fluxes |w| (F_1 + F_2 + D) along w/|w|: the reference reads
// their densities (and Roe's enthalpies) before assigning them and subtracts
// the upwind term D, which reverses its sign; both are repaired here.
template <typename R>
__device__ __forceinline__ void simple_flux(const DevParams &P, int ft, const R *U1, R pr1, const R *U2, R pr2, R wx,
                                            R wy, R wz, R wg, R *f) {
  R r1 = U1[0], ru1 = U1[1], rv1 = U1[2], rw1 = U1[3], E1 = U1[4];
  R r2 = U2[0], ru2 = U2[1], rv2 = U2[2], rw2 = U2[3], E2 = U2[4];
  R rinv1 = R(1) / r1, rinv2 = R(1) / r2;
  R u1 = rinv1 * ru1, v1 = rinv1 * rv1, w1 = rinv1 * rw1, rh1 = E1 + pr1;
  R u2 = rinv2 * ru2, v2 = rinv2 * rv2, w2 = rinv2 * rw2, rh2 = E2 + pr2;
  const R us[5] = {r1 + r2, ru1 + ru2, rv1 + rv2, rw1 + rw2, E1 + E2};
  if (ft == 1) {
    f[0] = wx * (ru1 + ru2) + wy * (rv1 + rv2) + wz * (rw1 + rw2);
    f[1] = wx * (ru1 * u1 + pr1 + ru2 * u2 + pr2) + wy * (ru1 * v1 + ru2 * v2) + wz * (ru1 * w1 + ru2 * w2);
    f[2] = wx * (rv1 * u1 + rv2 * u2) + wy * (rv1 * v1 + pr1 + rv2 * v2 + pr2) + wz * (rv1 * w1 + rv2 * w2);
    f[3] = wx * (rw1 * u1 + rw2 * u2) + wy * (rw1 * v1 + rw2 * v2) + wz * (rw1 * w1 + pr1 + rw2 * w2 + pr2);
    f[4] = wx * (rh1 * u1 + rh2 * u2) + wy * (rh1 * v1 + rh2 * v2) + wz * (rh1 * w1 + rh2 * w2);
    if (wg != R(0))
#pragma unroll
      for (int c = 0; c < 5; ++c) f[c] -= us[c] * wg;
  } else {
#pragma unroll
    for (int c = 0; c < 5; ++c) f[c] = 0;
    R rnorm = sqrt(wx * wx + wy * wy + wz * wz);
    if (rnorm > R(1.0e-10)) {
      R rnx = wx / rnorm, rny = wy / rnorm, rnz = wz / rnorm;
      R nv1 = u1 * rnx + v1 * rny + w1 * rnz, nv2 = u2 * rnx + v2 * rny + w2 * rnz;
      R F1[5] = {r1 * nv1, pr1 * rnx + ru1 * nv1, pr1 * rny + rv1 * nv1, pr1 * rnz + rw1 * nv1, rh1 * nv1};
      R F2[5] = {r2 * nv2, pr2 * rnx + ru2 * nv2, pr2 * rny + rv2 * nv2, pr2 * rnz + rw2 * nv2, rh2 * nv2};
      R du[5] = {r1 - r2, ru1 - ru2, rv1 - rv2, rw1 - rw2, E1 - E2};
      R D[5];
      if (ft == 2) {
        R c1 = sqrt(R(P.gamma) * pr1 * rinv1), c2 = sqrt(R(P.gamma) * pr2 * rinv2);
        R l1 = fabs(nv1 + c1), l12 = fabs(nv2 + c2);
        if (l1 < l12) l1 = l12;
        R l2 = fabs(nv1 - c1), l22 = fabs(nv2 - c2);
        if (l2 < l22) l2 = l22;
        R lam = l1;
        if (lam < l2) lam = l2;
#pragma unroll
        for (int c = 0; c < 5; ++c) D[c] = lam * du[c];
      } else {
        R gam1 = R(P.gamma - 1.0);
        R h1 = rh1 * rinv1, h2 = rh2 * rinv2;
        R di = sqrt(r1 / r2), d1 = R(1) / (di + R(1));
        R ui = (di * u1 + u2) * d1, vi = (di * v1 + v2) * d1, wi = (di * w1 + w2) * d1;
        R hi = (di * h1 + h2) * d1;
        R ci2 = gam1 * (hi - R(0.5) * (ui * ui + vi * vi + wi * wi));
        ci2 = ci2 > R(1.0e-5) ? ci2 : R(1.0e-5);
        R ci = sqrt(ci2), af = R(0.5) * (ui * ui + vi * vi + wi * wi), ucp = ui * rnx + vi * rny + wi * rnz;
        R l1 = fabs(ucp + ci), l2 = fabs(ucp - ci), l3 = fabs(ucp);
        R s1 = R(0.5) * (l1 + l2), s2 = R(0.5) * (l1 - l2);
        R a1 = gam1 * (af * du[0] - ui * du[1] - vi * du[2] - wi * du[3] + du[4]);
        R a2 = -ucp * du[0] + du[1] * rnx + du[2] * rny + du[3] * rnz;
        R cc1 = ((s1 - l3) * a1 / ci2) + (s2 * a2 / ci);
        R cc2 = (s2 * a1 / ci) + (s1 - l3) * a2;
        D[0] = l3 * du[0] + cc1;
        D[1] = l3 * du[1] + cc1 * ui + cc2 * rnx;
        D[2] = l3 * du[2] + cc1 * vi + cc2 * rny;
        D[3] = l3 * du[3] + cc1 * wi + cc2 * rnz;
        D[4] = l3 * du[4] + cc1 * hi + cc2 * ucp;
      }
#pragma unroll
      for (int c = 0; c < 5; ++c) f[c] = rnorm * ((F1[c] + F2[c]) + D[c]);
      if (wg != R(0))
#pragma unroll
        for (int c = 0; c < 5; ++c) f[c] -= us[c] * wg;
    }
  }
}

// fbuf[6 e + c] as k_flux (component 5: SA convection from the records).
template <typename R, int FT, bool SA>
__global__ void k_flux_simple(LevelDev<R> L, DevParams P) {
  int bb_;
  int e = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (e >= L.ne) return;
  const size_t n = L.n;
  int ia = L.ea[e], ib = L.eb[e];
  R wx = L.w[3 * e], wy = L.w[3 * e + 1], wz = L.w[3 * e + 2];
  R ua[5], ub[5], f[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    ua[c] = L.u[c * n + ia];
    ub[c] = L.u[c * n + ib];
  }
  const R wg = L.gcl ? L.gcl[e] / R(P.dtp) : R(0);
  simple_flux(P, FT, ua, L.p[ia], ub, L.p[ib], wx, wy, wz, wg, f);
  R *o = L.fbuf + 6 * (size_t)e;
#pragma unroll
  for (int c = 0; c < 5; ++c) o[c] = f[c];
  if (SA) {
    R A[8], B[8];
    ldrec<8>(L.rec0 + 8 * (size_t)ia, A);
    ldrec<8>(L.rec0 + 8 * (size_t)ib, B);
    o[5] = sa_side_convection(A, B, wx, wy, wz);
  } else {
    o[5] = 0;
  }
}

// makeSASourceTerm (DEF:9285-9370) of one node on any arithmetic type: the
// density, nu~ (u(:,6)), the laminar viscosity (after the caller's guard),
// vorticity and divergence, wall distance and volume (TW: double, or dual
// numbers for the derivatives with respect to the mesh)
template <typename T, typename TW = double>
__device__ __forceinline__ T sa_source_t(const DevParams &P, T rho, T nu, T mu, T vort, T divg, TW wd, TW vt) {
  double Re = P.Re, ioRe = 1.0 / Re;
  double cb1 = 0.1355, cb2 = 0.622, k2 = 0.41 * 0.41, sigma = 2.0 / 3.0;
  double cw1 = cb1 / k2 + (1.0 + cb2) / sigma, cw2 = 0.3, cw36 = 64.0, cv13 = 7.1 * 7.1 * 7.1;
  double ct3 = 1.1, ct4 = 2.0;
  T mc = nu;
  mc = mc > T(0.0) ? mc : T(0.0);
  T ksi = rho * T(ioRe) * mc / mu;
  ksi = ksi > T(0.001) ? ksi : T(0.001);
  T ft2 = T(ct3) * exp(T(-ct4) * ksi * ksi);
  T k3 = ksi * ksi * ksi;
  T d = T(wd);
  d = d > T(1e-10) ? d : T(1e-10);
  T md = mc / d;
  T d2 = d * d;
  T fv1 = k3 / (k3 + T(cv13));
  T fv2 = T(1.0) - ksi / (T(1.0) + ksi * fv1);
  T Sc = vort + T(ioRe) * mc * fv2 / (T(k2) * d2);
  T r;
  if (fabs(Sc) > T(1e-10)) {
    r = T(ioRe) * mc / (Sc * T(k2) * d2);
    r = r < T(0.0) ? T(0.0) : (r > T(100.0) ? T(100.0) : r);
  } else {
    r = T(100.0);
  }
  T r2 = r * r, r6 = r2 * r2 * r2;
  T g = r + T(cw2) * (r6 - r);
  T g2 = g * g, g6 = g2 * g2 * g2;
  T rad = T(1.0 + cw36) / (g6 + T(cw36));
  T fw = rad > T(1e-10) ? g * pow(rad, 1.0 / 6.0) : T(::pow(1.0 + cw36, 1.0 / 6.0));
  return -T(vt) * T(cb1) * (T(1.0) - ft2) * Sc * mc + T(ioRe) * T(vt) * (T(cw1) * fw - T(cb1) * ft2 / T(k2)) * md * md -
         T(vt) * mc * divg;
}

// ---------------------------------------------------------------------------
// Tangent and adjoint of the level-1 convective residual R(U) (makeRHS,
// DEF:1525-2512: interior HLLC sides + boundary sides) for first-order
// HLLC without viscous or turbulence terms.  The side and boundary fluxes
// are re-evaluated from the conserved state (the tangent and the boundary
// adjoint on dual numbers, the side adjoint by a reverse sweep), so nothing
// per side is stored between the forward and the reverse sweeps.
// ---------------------------------------------------------------------------
// gather record of a conserved state exactly as k_prep forms it
template <typename T>
__device__ __forceinline__ void state_record(const T *U, double gamma, T *A) {
  T r = U[0], m1 = U[1], m2 = U[2], m3 = U[3], E = U[4];
  T pp = T(gamma - 1.0) * (E - T(0.5) * (m1 * m1 + m2 * m2 + m3 * m3) / r);
  pp = pp > T(0.1) ? pp : T(0.1);
  A[0] = r;
  A[1] = m1 / r;
  A[2] = m2 / r;
  A[3] = m3 / r;
  A[4] = E;
  A[5] = pp;
  A[6] = T(0);
  A[7] = T(0);
}

// boundary flux of one end (the per-end flux of k_bflux): F(U)·n̂
template <typename T, typename N>
__device__ __forceinline__ void bside_end_flux(const DevParams &P, int ind, const T *U, N rnx, N rny, N rnz, T *f) {
  T A[8];
  state_record(U, P.gamma, A);
  if (ind <= 2 || ind == 9) {
    phys_flux(A, T(rnx), T(rny), T(rnz), f);
  } else {
    double inf[6];
    P.inflow_row(ind - 3, inf);
    farfield_roe(inf, A, T(P.gamma - 1.0), T(rnx), T(rny), T(rnz), f);
  }
}

// (dA/dU)^T of the gather record's (rho, u, v, w, rhoE): shares b[5] on the
// record to shares on the conserved state
__device__ __forceinline__ void record_share(const double *A, const double *b, double *out) {
  const double ir = 1.0 / A[0];
  out[0] = b[0] - (b[1] * A[1] + b[2] * A[2] + b[3] * A[3]) * ir;
  out[1] = b[1] * ir;
  out[2] = b[2] * ir;
  out[3] = b[3] * ir;
  out[4] = b[4];
}
// the pressure's share bp of a record, on its primitive entries b[5]
// (p = (gamma - 1)(E - rho |v|^2 / 2), no share where it is clipped)
__device__ __forceinline__ void pressure_share(double gm1, double r, const double *v, double p_raw, double bp, double &br,
                                               double *bv, double &be) {
  if (!(p_raw > 0.1)) return;
  be += gm1 * bp;
  br -= 0.5 * gm1 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]) * bp;
#pragma unroll
  for (int k = 0; k < 3; ++k) bv[k] -= gm1 * r * v[k] * bp;
}

// Reverse sweep of side_flux_d (components 0..4): with multipliers dl on the
// flux, the shares sa, sb on the two ends' (rho, u, v, w, rhoE) and, second
// order (d non-null), sd on the slopes.  The pressures of the records are
// those of their states (state_record).  One forward and one backward pass
// over the branch the values take; seeding dual numbers on each of the 15
// inputs evaluated the whole flux 15 times at one wavefront a SIMD.
template <bool SECOND>
__device__ __forceinline__ void side_flux_reverse(const DevParams &P, const double *A, const double *B,
                                                  const double *d, double wx, double wy, double wz, const double *dl,
                                                  double *sa, double *sb, double *sd) {
  const double gm1 = P.gamma - 1.0, beta = P.beta0;
  const double nx = 2.0 * wx, ny = 2.0 * wy, nz = 2.0 * wz, n2 = nx * nx + ny * ny + nz * nz;
  const double inv = n2 > 0.0 ? 1.0 / ::sqrt(n2) : 0.0, size = n2 * inv;
  const double n[3] = {nx * inv, ny * inv, nz * inv};
  // forward: the two faces' states
  struct Face {
    double r, v[3], e, p, p_raw, rinv, h, nv, q, x, c;
    double br, bv[3], be, bp, bh, bnv, bc;
    bool fr, fe;
  } f[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    Face &F = f[k];
    const double *R = k ? B : A;
    const double sg = k ? -1.0 : 1.0;
    F.r = R[0];
    F.e = R[4];
    F.fr = F.fe = false;
#pragma unroll
    for (int q = 0; q < 3; ++q) F.v[q] = R[1 + q];
    if constexpr (SECOND) {
      F.fr = R[0] + sg * d[0] > 0.1;
      F.fe = R[4] + sg * d[4] > 0.0001;
      if (F.fr) F.r = R[0] + sg * d[0];
      if (F.fe) F.e = R[4] + sg * d[4];
#pragma unroll
      for (int q = 0; q < 3; ++q) F.v[q] = R[1 + q] + sg * d[1 + q];
    }
    F.q = F.v[0] * F.v[0] + F.v[1] * F.v[1] + F.v[2] * F.v[2];
    F.p_raw = gm1 * (F.e - 0.5 * F.q * F.r);
    F.p = F.p_raw > 0.1 ? F.p_raw : 0.1;
    F.rinv = 1.0 / F.r;
    F.h = (F.e + F.p) * F.rinv;
    F.nv = F.v[0] * n[0] + F.v[1] * n[1] + F.v[2] * n[2];
    F.x = F.h - 0.5 * F.q;
    F.c = ::sqrt(gm1 * ::fabs(F.x));
    F.br = F.be = F.bp = F.bh = F.bnv = F.bc = 0.0;
    F.bv[0] = F.bv[1] = F.bv[2] = 0.0;
  }
  const double rr = ::sqrt(f[1].r * f[0].rinv), iro = 1.0 / (1.0 + rr);
  double ut[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) ut[q] = (f[0].v[q] + f[1].v[q] * rr) * iro;
  const double ht = (f[0].h + f[1].h * rr) * iro, qt = ut[0] * n[0] + ut[1] * n[1] + ut[2] * n[2];
  const double y = gm1 * (ht - 0.5 * (ut[0] * ut[0] + ut[1] * ut[1] + ut[2] * ut[2])), ct = ::sqrt(::fabs(y));
  // the wave speeds and which of the three candidates each is
  int kl = 0, kr = 0;
  double sl = f[0].nv - beta * f[0].c, sr = f[1].nv + beta * f[1].c;
  if (qt - ct < sl) { sl = qt - ct; kl = 1; }
  if (f[1].nv - beta * f[1].c < sl) { sl = f[1].nv - beta * f[1].c; kl = 2; }
  if (qt + ct > sr) { sr = qt + ct; kr = 1; }
  if (f[0].nv + beta * f[0].c > sr) { sr = f[0].nv + beta * f[0].c; kr = 2; }
  const double num = f[1].r * f[1].nv * (sr - f[1].nv) - f[0].r * f[0].nv * (sl - f[0].nv) + f[0].p - f[1].p;
  const double den = f[1].r * (sr - f[1].nv) - f[0].r * (sl - f[0].nv), fact = den != 0.0 ? 1.0 / den : 0.0;
  const double sm = fact * num;
  const bool lft = sl > 0.0 || (sl <= 0.0 && sm > 0.0), rgt = (sm <= 0.0 && sr >= 0.0) || sr < 0.0;
  if (!lft && !rgt) {
    // the central flux of the nodes' states (NaN wave speeds)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double *R = k ? B : A;
      double *o = k ? sb : sa;
      const double wn = wx * R[1] + wy * R[2] + wz * R[3], ww[3] = {wx, wy, wz};
      const double m = dl[0] + dl[1] * R[1] + dl[2] * R[2] + dl[3] * R[3], h = R[4] + R[5];
      double bv[3];
      o[0] = wn * m;
#pragma unroll
      for (int q = 0; q < 3; ++q) bv[q] = R[0] * (ww[q] * m + wn * dl[1 + q]) + h * ww[q] * dl[4];
      o[4] = wn * dl[4];
      const double p_raw = gm1 * (R[4] - 0.5 * (R[1] * R[1] + R[2] * R[2] + R[3] * R[3]) * R[0]);
      pressure_share(gm1, R[0], R + 1, p_raw, dl[1] * wx + dl[2] * wy + dl[3] * wz + wn * dl[4], o[0], bv, o[4]);
#pragma unroll
      for (int q = 0; q < 3; ++q) o[1 + q] = bv[q];
    }
    if constexpr (SECOND)
#pragma unroll
      for (int c = 0; c < 5; ++c) sd[c] = 0.0;
    return;
  }
  // backward: the upwind side K, on selected copies
  double g[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) g[c] = dl[c] * size;
  const double r = lft ? f[0].r : f[1].r, e = lft ? f[0].e : f[1].e, p = lft ? f[0].p : f[1].p;
  const double nv = lft ? f[0].nv : f[1].nv, sk = lft ? sl : sr;
  double v[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) v[q] = lft ? f[0].v[q] : f[1].v[q];
  double br, bv[3], be, bp, bnv, bsk = 0.0, bsm = 0.0;
  {
    const double S = g[0] + g[1] * v[0] + g[2] * v[1] + g[3] * v[2];
    br = nv * S;
    bnv = r * S + (e + p) * g[4];
    be = nv * g[4];
    bp = g[1] * n[0] + g[2] * n[1] + g[3] * n[2] + nv * g[4];
#pragma unroll
    for (int q = 0; q < 3; ++q) bv[q] = r * nv * g[1 + q];
  }
  const bool star = lft ? !(sl > 0.0) : !(sr < 0.0);
  if (star && sk - sm != 0.0) {
    const double k = 1.0 / (sk - sm), a = sk - nv;
    const double pks = r * (nv - sk) * (nv - sm) + p, ps = pks - p;
    double s[5], b[5];
    s[0] = r * a * k;
#pragma unroll
    for (int q = 0; q < 3; ++q) s[1 + q] = (a * r * v[q] + ps * n[q]) * k;
    s[4] = (a * e - p * nv + pks * sm) * k;
    bsk += g[0] * (s[0] - r) + g[4] * (s[4] - e);
    br -= g[0] * sk;
    be -= g[4] * sk;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      bsk += g[1 + q] * (s[1 + q] - r * v[q]);
      br -= g[1 + q] * sk * v[q];
      bv[q] -= g[1 + q] * sk * r;
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) b[c] = g[c] * sk;
    const double bden = -k * (b[0] * s[0] + b[1] * s[1] + b[2] * s[2] + b[3] * s[3] + b[4] * s[4]);
    const double bw = b[0] + b[1] * v[0] + b[2] * v[1] + b[3] * v[2];
    const double ba = k * (r * bw + b[4] * e);
    const double bps = k * (b[1] * n[0] + b[2] * n[1] + b[3] * n[2]), bpks = k * sm * b[4] + bps;
    br += k * a * bw;
#pragma unroll
    for (int q = 0; q < 3; ++q) bv[q] += k * a * r * b[1 + q];
    be += k * a * b[4];
    bp += bpks - bps - k * nv * b[4];
    bnv -= k * p * b[4];
    bsm += k * pks * b[4];
    br += bpks * (nv - sk) * (nv - sm);
    bnv += bpks * r * ((nv - sm) + (nv - sk));
    bsk -= bpks * r * (nv - sm);
    bsm -= bpks * r * (nv - sk);
    bsk += ba + bden;
    bnv -= ba;
    bsm -= bden;
  }
  double bsl = lft ? bsk : 0.0, bsr = lft ? 0.0 : bsk;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const bool mine = lft == (k == 0);
    Face &F = f[k];
    F.br = mine ? br : 0.0;
    F.be = mine ? be : 0.0;
    F.bp = mine ? bp : 0.0;
    F.bnv = mine ? bnv : 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) F.bv[q] = mine ? bv[q] : 0.0;
  }
  {  // the contact speed
    const double bnum = bsm * fact, bden = -bsm * num * fact * fact;
    f[1].br += bnum * f[1].nv * (sr - f[1].nv) + bden * (sr - f[1].nv);
    f[1].bnv += bnum * f[1].r * (sr - 2.0 * f[1].nv) - bden * f[1].r;
    bsr += bnum * f[1].r * f[1].nv + bden * f[1].r;
    f[0].br -= bnum * f[0].nv * (sl - f[0].nv) + bden * (sl - f[0].nv);
    f[0].bnv += -bnum * f[0].r * (sl - 2.0 * f[0].nv) + bden * f[0].r;
    bsl -= bnum * f[0].r * f[0].nv + bden * f[0].r;
    f[0].bp += bnum;
    f[1].bp -= bnum;
  }
  // the outer wave speeds
  f[0].bnv += (kl == 0 ? bsl : 0.0) + (kr == 2 ? bsr : 0.0);
  f[0].bc = beta * ((kr == 2 ? bsr : 0.0) - (kl == 0 ? bsl : 0.0));
  f[1].bnv += (kl == 2 ? bsl : 0.0) + (kr == 0 ? bsr : 0.0);
  f[1].bc = beta * ((kr == 0 ? bsr : 0.0) - (kl == 2 ? bsl : 0.0));
  const double bqt = (kl == 1 ? bsl : 0.0) + (kr == 1 ? bsr : 0.0);
  const double bct = (kr == 1 ? bsr : 0.0) - (kl == 1 ? bsl : 0.0);
  const double by = ct > 0.0 ? bct * (y < 0.0 ? -0.5 : 0.5) / ct : 0.0, bht = gm1 * by;
  double brr = 0.0, biro = bht * (f[0].h + f[1].h * rr);
  f[0].bh += bht * iro;
  f[1].bh += bht * iro * rr;
  brr += bht * iro * f[1].h;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const double but = bqt * n[q] - gm1 * by * ut[q];
    f[0].bv[q] += but * iro;
    f[1].bv[q] += but * iro * rr;
    brr += but * iro * f[1].v[q];
    biro += but * (f[0].v[q] + f[1].v[q] * rr);
  }
  brr -= biro * iro * iro;
  const double brat = rr > 0.0 ? 0.5 * brr / rr : 0.0;
  f[1].br += brat * f[0].rinv;
  f[0].br -= brat * rr * rr * f[0].rinv;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    Face &F = f[k];
    const double bx = F.c > 0.0 ? F.bc * gm1 * (F.x < 0.0 ? -0.5 : 0.5) / F.c : 0.0;
    F.bh += bx;
    F.be += F.bh * F.rinv;
    F.bp += F.bh * F.rinv;
    F.br -= F.bh * F.h * F.rinv;
#pragma unroll
    for (int q = 0; q < 3; ++q) F.bv[q] += F.bnv * n[q] - bx * F.v[q];
    pressure_share(gm1, F.r, F.v, F.p_raw, F.bp, F.br, F.bv, F.be);
    double *o = k ? sb : sa;
    o[0] = F.br;
    o[1] = F.bv[0];
    o[2] = F.bv[1];
    o[3] = F.bv[2];
    o[4] = F.be;
  }
  if constexpr (SECOND) {
    sd[0] = (f[0].fr ? f[0].br : 0.0) - (f[1].fr ? f[1].br : 0.0);
    sd[4] = (f[0].fe ? f[0].be : 0.0) - (f[1].fe ? f[1].be : 0.0);
#pragma unroll
    for (int q = 0; q < 3; ++q) sd[1 + q] = f[0].bv[q] - f[1].bv[q];
  }
}

// tangent: fbuf/bbuf <- d(fluxes)/dU along du; the stage gather (MODE_RHS)
// then sums them into rhs = (dR/dU) du
template <bool SA>
__global__ __launch_bounds__(NTHR) void k_flux_tangent(LevelDev<double> L, DevParams P, const double *du) {
  using ad::Dual;
  int e = gtid_x();
  if (e >= L.ne) return;
  size_t n = L.n;
  int ia = L.ea[e], ib = L.eb[e];
  Dual Ua[5], Ub[5], A[8], B[8], o[6];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    Ua[c] = Dual(L.u[c * n + ia], du[c * n + ia]);
    Ub[c] = Dual(L.u[c * n + ib], du[c * n + ib]);
  }
  state_record(Ua, P.gamma, A);
  state_record(Ub, P.gamma, B);
  if (SA) {
    A[6] = Dual(L.u[5 * n + ia], du[5 * n + ia]);
    B[6] = Dual(L.u[5 * n + ib], du[5 * n + ib]);
  }
  side_flux<Dual, double, 1, SA, 2, double, double>(P, nullptr, nullptr, nullptr, nullptr, A, B, Dual(L.w[3 * e]),
                                                    Dual(L.w[3 * e + 1]), Dual(L.w[3 * e + 2]), o);
  double *f = L.fbuf + 6 * (size_t)e;
#pragma unroll
  for (int c = 0; c < 5; ++c) f[c] = o[c].d;
  f[5] = SA ? o[5].d : 0.0;
}

__global__ __launch_bounds__(NTHR) void k_bflux_tangent(LevelDev<double> L, DevParams P, const double *du) {
  using ad::Dual;
  int s = gtid_x();
  if (s >= L.nbs) return;
  size_t n = L.n;
  int ia = L.ba[s], ib = L.bb[s], ind = L.bind[s];
  double wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
  double *o = L.bbuf + 10 * (size_t)s;
  double rnorm = ::sqrt(wx * wx + wy * wy + wz * wz);
  if (!(rnorm > 1e-10) || !(ind <= 4 || ind == 9)) {
#pragma unroll
    for (int c = 0; c < 10; ++c) o[c] = 0;
    return;
  }
  double irn = 1.0 / rnorm;
  Dual Ua[5], Ub[5], f1[5], f2[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    Ua[c] = Dual(L.u[c * n + ia], du[c * n + ia]);
    Ub[c] = Dual(L.u[c * n + ib], du[c * n + ib]);
  }
  bside_end_flux(P, ind, Ua, wx * irn, wy * irn, wz * irn, f1);
  bside_end_flux(P, ind, Ub, wx * irn, wy * irn, wz * irn, f2);
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    if (P.bterm == 1) {
      o[c] = rnorm * (3.0 * f1[c].d + f2[c].d);
      o[5 + c] = rnorm * (f1[c].d + 3.0 * f2[c].d);
    } else {
      o[c] = rnorm * 4.0 * f1[c].d;
      o[5 + c] = rnorm * 4.0 * f2[c].d;
    }
  }
}

// adjoint, interior sides: side e adds +f to R(ea) and -f to R(eb), so its
// share of (dR/dU)^T lam is (df/dU_ea)^T d and (df/dU_eb)^T d with
// d = lam(ea) - lam(eb).  abuf[10*e + k]: k < 5 for U_ea, k >= 5 for U_eb.
__global__ __launch_bounds__(NTHR) void k_flux_adjoint(LevelDev<double> L, DevParams P, const double *lam, double *abuf) {
  int e = gtid_x();
  if (e >= L.ne) return;
  size_t n = L.n;
  int ia = L.ea[e], ib = L.eb[e];
  double ua[5], ub[5], d[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    ua[c] = L.u[c * n + ia];
    ub[c] = L.u[c * n + ib];
    d[c] = lam[c * n + ia] - lam[c * n + ib];
  }
  double A[8], B[8], sa[5], sb[5], sd[5];
  state_record(ua, P.gamma, A);
  state_record(ub, P.gamma, B);
  side_flux_reverse<false>(P, A, B, nullptr, L.w[3 * e], L.w[3 * e + 1], L.w[3 * e + 2], d, sa, sb, sd);
  double *o = abuf + 10 * (size_t)e;
  record_share(A, sa, o);
  record_share(B, sb, o + 5);
}

// adjoint, boundary sides: R(a) += |w|(3F_a + F_b), R(b) += |w|(F_a + 3F_b)
// (boundaryTerm 1; 4F_a and 4F_b for 2), so U_a receives
// |w| (dF_a/dU_a)^T (3 lam_a + lam_b), and alike for U_b.  bbuf layout as
// the residual's: [10*s + 5*end + k].
__global__ __launch_bounds__(NTHR) void k_bflux_adjoint(LevelDev<double> L, DevParams P, const double *lam) {
  using ad::Dual;
  int s = gtid_x();
  if (s >= L.nbs) return;
  size_t n = L.n;
  int ia = L.ba[s], ib = L.bb[s], ind = L.bind[s];
  double wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
  double *o = L.bbuf + 10 * (size_t)s;
  double rnorm = ::sqrt(wx * wx + wy * wy + wz * wz);
  if (!(rnorm > 1e-10) || !(ind <= 4 || ind == 9)) {
#pragma unroll
    for (int c = 0; c < 10; ++c) o[c] = 0;
    return;
  }
  double irn = 1.0 / rnorm;
#pragma unroll 1
  for (int end = 0; end < 2; ++end) {
    int me = end ? ib : ia;
    double wt[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      double la = lam[c * n + ia], lb = lam[c * n + ib];
      if (P.bterm == 1) wt[c] = rnorm * (end ? la + 3.0 * lb : 3.0 * la + lb);
      else wt[c] = rnorm * 4.0 * (end ? lb : la);
    }
#pragma unroll 1
    for (int k = 0; k < 5; ++k) {
      Dual U[5], f[5];
#pragma unroll
      for (int c = 0; c < 5; ++c) U[c] = Dual(L.u[c * n + me], k == c ? 1.0 : 0.0);
      bside_end_flux(P, ind, U, wx * irn, wy * irn, wz * irn, f);
      double acc = 0;
#pragma unroll
      for (int c = 0; c < 5; ++c) acc += wt[c] * f[c].d;
      o[5 * end + k] = acc;
    }
  }
}

// adjoint gather: out(i) = sum of node i's shares over its sides
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_adjoint_gather(LevelDev<double> L, const double *abuf, double *out) {
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (i >= L.n) return;
  double r[5] = {0, 0, 0, 0, 0};
  for_edges<SUB>(L, i, sub, [&](int e, int role) {
    const double *a = abuf + 10 * (size_t)e + 5 * role;
#pragma unroll
    for (int c = 0; c < 5; ++c) r[c] += a[c];
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k];
    const double *b = L.bbuf + 10 * (size_t)(v >> 1) + 5 * (v & 1);
#pragma unroll
    for (int c = 0; c < 5; ++c) r[c] += b[c];
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) r[c] = lsum<SUB>(r[c]);
  if (sub) return;
  size_t n = L.n;
#pragma unroll
  for (int c = 0; c < 5; ++c) out[c * n + i] = r[c];
  out[5 * n + i] = 0;
}

// adjoint of the SA convection (the side flux's component 6, makeSARHS
// DEF:6873-6880, first order at both orders: the node values of nu~ and
// the velocities): node i's share of sum over sides of (lam6_ea - lam6_eb) f6,
// added to out.  With m = nu~ v, X = w.(m_b - m_a) and s the sign of X / (nu~_a
// - nu~_b), f6 = w.(m_a + m_b) + s X, so with the node-signed weight node i's
// own m enters a side's term as (lam_i - lam_j)(1 - s) w.m_i from the first
// end and (1 + s) from the second: the walk sums that one vector, and its
// shares on v and nu~ follow at the end.  sa_upwind from the node has the sign
// of s at the first end and of -s at the second, so the role is read only
// where it is 0.  (Six dual passes of every side took 168 us at 275k nodes,
// 71 now.)
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_sa_conv_adjoint(LevelDev<double> L, DevParams P, const double *lam, double *out) {
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (i >= L.n) return;
  const size_t n = L.n;
  double qi[8], z[3] = {0, 0, 0};
  ldrec<8>(L.rec0 + 8 * (size_t)i, qi);
  const double li = lam[5 * n + i];
  for_slots<SUB>(L, i, sub, [&](int slot, int j, double wx, double wy, double wz) {
    double qj[8];
    ldrec<8>(L.rec0 + 8 * (size_t)j, qj);
    double c = li - lam[5 * n + j];
    if (::fabs(qi[6] - qj[6]) > 1e-20) {
      const int s = sa_upwind(qi + 1, qj + 1, qi[6], qj[6], wx, wy, wz);
      c *= s < 0 || (s == 0 && (L.ell_e[slot] & 1)) ? 2.0 : 0.0;
    }
    z[0] += c * wx;
    z[1] += c * wy;
    z[2] += c * wz;
  });
#pragma unroll
  for (int k = 0; k < 3; ++k) z[k] = lsum<SUB>(z[k]);
  if (sub) return;
  const double b[5] = {0.0, z[0] * qi[6], z[1] * qi[6], z[2] * qi[6], 0.0};
  double o[5];
  record_share(qi, b, o);
#pragma unroll
  for (int c = 0; c < 4; ++c) out[c * n + i] += o[c];
  out[5 * n + i] += z[0] * qi[1] + z[1] * qi[2] + z[2] * qi[3];
}

// Metric adjoint: the derivative of lam^T R with respect to the side
// weights at the current state, for the residual of the tangent and adjoint
// (first-order HLLC, inviscid).  The interior flux depends on w through
// n = 2w, |n| and n/|n|, the boundary flux through |w_b| and w_b/|w_b|;
// three dual passes per side, seeded on the weight components, give the
// three components of the derivative.  Side e adds +f to R(ea) and -f to
// R(eb), so its share is (lam_a - lam_b) . df/dw.
__global__ __launch_bounds__(NTHR) void k_flux_metric_adjoint(LevelDev<double> L, DevParams P, const double *lam, double *gw) {
  using ad::Dual;
  int e = gtid_x();
  if (e >= L.ne) return;
  size_t n = L.n;
  int ia = L.ea[e], ib = L.eb[e];
  Dual Ua[5], Ub[5], A[8], B[8];
  double d[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    Ua[c] = Dual(L.u[c * n + ia]);
    Ub[c] = Dual(L.u[c * n + ib]);
    d[c] = lam[c * n + ia] - lam[c * n + ib];
  }
  state_record(Ua, P.gamma, A);
  state_record(Ub, P.gamma, B);
  const double w0 = L.w[3 * e], w1 = L.w[3 * e + 1], w2 = L.w[3 * e + 2];
#pragma unroll 1
  for (int k = 0; k < 3; ++k) {
    Dual o[6];
    side_flux<Dual, double, 1, false, 2, double, double>(P, nullptr, nullptr, nullptr, nullptr, A, B, Dual(w0, k == 0 ? 1.0 : 0.0),
                                         Dual(w1, k == 1 ? 1.0 : 0.0), Dual(w2, k == 2 ? 1.0 : 0.0), o);
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 5; ++c) acc += d[c] * o[c].d;
    gw[3 * (size_t)e + k] = acc;
  }
}

// boundary sides: R(a) += |w|(3F_a + F_b), R(b) += |w|(F_a + 3F_b)
// (boundaryTerm 1; 4F_a and 4F_b for 2) with F evaluated along w/|w|
__global__ __launch_bounds__(NTHR) void k_bflux_metric_adjoint(LevelDev<double> L, DevParams P, const double *lam, double *gwb) {
  using ad::Dual;
  int s = gtid_x();
  if (s >= L.nbs) return;
  size_t n = L.n;
  int ia = L.ba[s], ib = L.bb[s], ind = L.bind[s];
  const double w0 = L.wb[3 * s], w1 = L.wb[3 * s + 1], w2 = L.wb[3 * s + 2];
  double *o = gwb + 3 * (size_t)s;
  double rn = ::sqrt(w0 * w0 + w1 * w1 + w2 * w2);
  if (!(rn > 1e-10) || !(ind <= 4 || ind == 9)) {
    o[0] = o[1] = o[2] = 0;
    return;
  }
  Dual Ua[5], Ub[5];
  double la[5], lb[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    Ua[c] = Dual(L.u[c * n + ia]);
    Ub[c] = Dual(L.u[c * n + ib]);
    la[c] = lam[c * n + ia];
    lb[c] = lam[c * n + ib];
  }
#pragma unroll 1
  for (int k = 0; k < 3; ++k) {
    Dual wx(w0, k == 0 ? 1.0 : 0.0), wy(w1, k == 1 ? 1.0 : 0.0), wz(w2, k == 2 ? 1.0 : 0.0);
    Dual rnorm = sqrt(wx * wx + wy * wy + wz * wz);
    Dual irn = Dual(1.0) / rnorm;
    Dual f1[5], f2[5];
    bside_end_flux(P, ind, Ua, wx * irn, wy * irn, wz * irn, f1);
    bside_end_flux(P, ind, Ub, wx * irn, wy * irn, wz * irn, f2);
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      Dual ra, rb;
      if (P.bterm == 1) {
        ra = rnorm * (Dual(3.0) * f1[c] + f2[c]);
        rb = rnorm * (f1[c] + Dual(3.0) * f2[c]);
      } else {
        ra = rnorm * Dual(4.0) * f1[c];
        rb = rnorm * Dual(4.0) * f2[c];
      }
      acc += la[c] * ra.d + lb[c] * rb.d;
    }
    o[k] = acc;
  }
}

// ---------------------------------------------------------------------------
// Tangent and adjoint of the second-order (MUSCL + LED) inviscid residual.
// Side (a, b)'s flux depends on both ends' gather records q, their
// Green-Gauss gradients G and reciprocal limiter bounds B (grad_minmax_body),
// and G and B on the neighbours' q.  The tangent forms dG and dB in plain sums
// and the slopes' tangents in closed form, and evaluates the HLLC flux on dual
// numbers.  The adjoint runs that flux's reverse sweep once a side, sums the
// shares per node, and transposes the gradient (a linear node gather) and the
// bounds (a
// bound 1/(q_k* - q_i) moves with the neighbour k* that attains the
// extremum and with the node itself).
// ---------------------------------------------------------------------------
constexpr int LIN_G = 25;                   // gradient 15 | 1/lo 5 | 1/hi 5
// adjoint shares per side: U_a 5 | slope projection 5, bound 5, side vector
// 3, code | U_b 5 (an end reads 19 consecutive words)
constexpr int LIN_SIDE = 24;

// tangent of the gather record (rho, u, v, w, rhoE, p) along du
// the gather record's tangent dq[DQ i ..] = (rho, u, v, w, E, p, nu~, T)
// along du (nu~ = u(:,6) with Spalart-Allmaras, else 0; T of the viscous
// record)
constexpr int DQ = 8;
__global__ __launch_bounds__(NTHR) void k_record_tangent(LevelDev<double> L, DevParams P, const double *du, double *dq) {
  using ad::Dual;
  int i = gtid_x();
  if (i >= L.n) return;
  size_t n = L.n;
  Dual U[5], A[8];
#pragma unroll
  for (int c = 0; c < 5; ++c) U[c] = Dual(L.u[c * n + i], du[c * n + i]);
  state_record(U, P.gamma, A);
  double *o = dq + DQ * (size_t)i;
#pragma unroll
  for (int c = 0; c < 6; ++c) o[c] = A[c].d;
  o[6] = P.sa ? du[5 * n + i] : 0.0;
  o[7] = (Dual(P.gamma / (P.gamma - 1.0)) * A[5] / A[0]).d;
}

// tangents of the gradient records along dq: gt[GREC i + k] (gradients 15,
// reciprocal bounds 10).  The bounds move with the extremal neighbours that
// k_minmax_arg names; B = 1 / (q_k - q_i), so dB = -B^2 (dq_k - dq_i).  The
// values are the level's own records, so that every branch of the side flux
// is taken as in the residual and the adjoint.  275k nodes: 253 us on dual
// records with the bounds compared in the walk; 198 with the named neighbours'
// ten words read behind a branch each and 216 following their indices in the
// walk; 174 with the records stored through LDS; 107 with the ten reads in
// flight together.
template <int SUB>
__device__ __forceinline__ bool grad_tangent_vals(const LevelDev<double> &L, int i, int sub, const double *dq, const int *amin,
                                                  double *out) {
  double q0[8], g[15];
  ldrec<8>(dq + DQ * (size_t)i, q0);
#pragma unroll
  for (int c = 0; c < 15; ++c) g[c] = 0.0;
  for_edges_w<SUB>(L, i, sub, [&](int j, double wx, double wy, double wz) {
    double qj[6];
    ldrec<6>(dq + DQ * (size_t)j, qj);
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      const double s = q0[c] + qj[c];
      g[c] += s * wx;
      g[5 + c] += s * wy;
      g[10 + c] += s * wz;
    }
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    const double wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      const double t = 3.0 * q0[c] + dq[DQ * (size_t)o + c];
      g[c] += t * wx;
      g[5 + c] += t * wy;
      g[10 + c] += t * wz;
    }
  }
#pragma unroll
  for (int c = 0; c < 15; ++c) g[c] = lsum<SUB>(g[c]);
  if (sub) return false;
  const double vt = 1.0 / L.vol[i];
  double B[12], dm[10];  // B: words 14 .. 25 of the record, in aligned pairs
  int km[10];
  const int2 *ap = reinterpret_cast<const int2 *>(amin + 10 * (size_t)i);
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    const int2 k2 = ap[c];
    km[2 * c] = k2.x;
    km[2 * c + 1] = k2.y;
  }
  ldrec<12>(L.grec + GREC * (size_t)i + 14, B);
  // the ten reads in flight together: no branch on the index
#pragma unroll
  for (int c = 0; c < 10; ++c) dm[c] = dq[DQ * (size_t)(km[c] < 0 ? i : km[c]) + (c < 5 ? c : c - 5)];
#pragma unroll
  for (int c = 0; c < 15; ++c) out[c] = g[c] * vt;
#pragma unroll
  for (int c = 0; c < 10; ++c) out[15 + c] = km[c] < 0 ? 0.0 : -B[1 + c] * B[1 + c] * (dm[c] - q0[c < 5 ? c : c - 5]);
  out[25] = 0.0;
  return true;
}

template <int SUB>
__global__ __launch_bounds__(NTHR) void k_grad_tangent(LevelDev<double> L, const double *dq, const int *amin, double *gt) {
  __shared__ double st[SUB == 1 ? NTHR * (GREC / 2) : 1];
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  double v[GREC];
  const bool ok = i < L.n && grad_tangent_vals<SUB>(L, i, sub, dq, amin, v);
  if (SUB == 1) {
    const int i0 = i - (int)threadIdx.x;
    store_grec(st, v, ok, gt + GREC * (size_t)i0, L.n - i0 < NTHR ? L.n - i0 : NTHR);
  } else if (ok) {
    double *out = gt + GREC * (size_t)i;
#pragma unroll
    for (int c = 0; c < GREC; ++c) out[c] = v[c];
  }
}

// node i's extremal neighbours: amin[10 i + c] = the node whose q_c sets
// the lower bound of component c (-1 if none: the bound is 0), amin[10 i +
// 5 + c] the upper one, with grad_minmax_body's comparisons in slot order
__global__ __launch_bounds__(NTHR) void k_minmax_arg(LevelDev<double> L, int *amin) {
  int i = gtid_x();
  if (i >= L.n) return;
  double q0[5], mn[5], mx[5];
  int kn[5], kx[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    q0[c] = L.rec0[8 * (size_t)i + c];
    mn[c] = 1e15;
    mx[c] = 1e15;
    kn[c] = kx[c] = -1;
  }
  for_edges_w<1>(L, i, 0, [&](int j, double, double, double) {
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      // rmin(a, b) = a < b ? a : b keeps b on ties, as grad_minmax_body does
      double qj = L.rec0[8 * (size_t)j + c];
      double lo = rmin(q0[c], qj);
      int klo = q0[c] < qj ? i : j;
      if (!(mn[c] < lo)) { mn[c] = lo; kn[c] = klo; }
      double hi = rmin(-q0[c], -qj);
      int khi = -q0[c] < -qj ? i : j;
      if (!(mx[c] < hi)) { mx[c] = hi; kx[c] = khi; }
    }
  });
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    amin[10 * (size_t)i + c] = (mn[c] - q0[c] < 0.0 && kn[c] != i) ? kn[c] : -1;
    amin[10 * (size_t)i + 5 + c] = (-mx[c] - q0[c] > 0.0 && kx[c] != i) ? kx[c] : -1;
  }
}

// LED-limited projection (led) with its derivatives: da along the projection,
// div along the reciprocal bound its sign selects
template <int NSIG>
__device__ __forceinline__ double led_slopes(double a, double ilo, double ihi, double &da, double &div, bool &hi) {
  hi = a > 0.0;
  const double iv = hi ? ihi : ilo;
  da = div = 0.0;
  if (!(a > 0.0 || a < 0.0)) {
    da = 1.0;
    return a;
  }
  if (iv == 0.0) return 0.0;
  const double t = 2.0 * a * iv, t2 = t * t;
  if (NSIG == 4) {
    const double den = 1.0 + t2 * t2, iden = 1.0 / ::sqrt(::sqrt(den));
    da = iden / den;
    div = -2.0 * a * a * t * t2 * da;
    return a * iden;
  }
  const double den = 1.0 + t2, iden = 1.0 / ::sqrt(den);
  da = iden / den;
  div = -2.0 * a * a * t * da;
  return a * iden;
}

// One end's projected gradients on half the side vector and the bounds their
// signs select (SG -1: the second end, whose slope is -led(-b)), values from
// the gradient record G and tangents from T, limited: v the limited
// projections, t their tangents
template <int NSIG>
__device__ __forceinline__ void limited_tangents(const DevParams &P, const double *G, const double *T, double dx, double dy,
                                                 double dz, double sg, double *v, double *t) {
  double g[GREC], r[GREC];
  ldrec<GREC>(G, g);
  ldrec<GREC>(T, r);
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const double a = 0.5 * (g[j] * dx + g[j + 5] * dy + g[j + 10] * dz);
    const double ta = 0.5 * (r[j] * dx + r[j + 5] * dy + r[j + 10] * dz);
    v[j] = a;
    t[j] = ta;
    if (P.autoclip == 1) {
      double da, div;
      bool hi;
      v[j] = sg * led_slopes<NSIG>(sg * a, g[15 + j], g[20 + j], da, div, hi);
      t[j] = da * ta + sg * div * (hi ? r[20 + j] : r[15 + j]);
    }
  }
}

// second-order side fluxes along (dq, dG, dB): fbuf[6 e + c] = d f_c
// (component 5: the SA convection along d nu~); the slopes' tangents in closed
// form, the HLLC flux of the states and slopes on dual numbers (275k nodes,
// 1.87M sides: 259 us with the limiter on dual numbers too, 235 now, bound by
// the two ends' records: 1.1 KB a side through L2)
template <int NSIG, bool SA>
__global__ __launch_bounds__(NTHR) void k_flux_tangent2(LevelDev<double> L, DevParams P, const double *dq, const double *gt) {
  using ad::Dual;
  int e = gtid_x();
  if (e >= L.ne) return;
  int ia = L.ea[e], ib = L.eb[e];
  const double *xa = L.xyz + 3 * (size_t)ia, *xb = L.xyz + 3 * (size_t)ib;
  const double dx = xb[0] - xa[0], dy = xb[1] - xa[1], dz = xb[2] - xa[2];
  const double hl = 0.5 * P.clip * ::sqrt(dx * dx + dy * dy + dz * dz);
  double va[5], ta[5], vb[5], tb[5];
  limited_tangents<NSIG>(P, L.grec + GREC * (size_t)ia, gt + GREC * (size_t)ia, dx, dy, dz, 1.0, va, ta);
  limited_tangents<NSIG>(P, L.grec + GREC * (size_t)ib, gt + GREC * (size_t)ib, dx, dy, dz, -1.0, vb, tb);
  Dual A[8], B[8], D[5], o[6];
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    double c = 0.0, t = 0.0;
    if (!(va[j] * vb[j] <= 0.0)) {
      const bool first = ::fabs(va[j]) <= ::fabs(vb[j]);
      c = first ? va[j] : vb[j];
      t = first ? ta[j] : tb[j];
      if (::fabs(c) > hl && hl > 0.0) {
        c = c > 0.0 ? hl : -hl;
        t = 0.0;
      }
    }
    D[j] = Dual(c, t);
  }
  {
    double v[8], t[8];
    ldrec<8>(L.rec0 + 8 * (size_t)ia, v);
    ldrec<8>(dq + DQ * (size_t)ia, t);
#pragma unroll
    for (int c = 0; c < 7; ++c) A[c] = Dual(v[c], t[c]);
    ldrec<8>(L.rec0 + 8 * (size_t)ib, v);
    ldrec<8>(dq + DQ * (size_t)ib, t);
#pragma unroll
    for (int c = 0; c < 7; ++c) B[c] = Dual(v[c], t[c]);
  }
  side_flux_d<Dual, double, SA>(P, A, B, D, Dual(L.w[3 * e]), Dual(L.w[3 * e + 1]), Dual(L.w[3 * e + 2]), o, 0.0);
  double *f = L.fbuf + 6 * (size_t)e;
#pragma unroll
  for (int c = 0; c < 5; ++c) f[c] = o[c].d;
  f[5] = SA ? o[5].d : 0.0;
}

// adjoint shares of side e: dl = lam_a - lam_b against df/d(U_a, U_b,
// G_a, B_a, G_b, B_b).  The gradients and bounds reach the flux only through
// the five MUSCL slopes d_j: the reverse sweep of the flux gives the shares
// on U_a, U_b and d, and a slope is one end's limited projection (minmod), so
// its share goes to one end's gradient (along half the side vector) and one
// of that end's bounds.  Per component: the share on the projection, on the
// bound, and 3 bits of the code: 1 (first end) or 2 (second) or 0 (none), + 4
// for the upper bound.  (15 dual passes of the flux and 60 stored words took
// 1.9 ms and the gather 0.57 ms at 64^3; 0.25 and 0.23 now, 0.33 of the first
// before the two gradient records were read as whole aligned pairs.)
template <int NSIG>
__global__ __launch_bounds__(NTHR) void k_flux_adjoint2(LevelDev<double> L, DevParams P, const double *lam,
                                                        double *abuf2) {
  int e = gtid_x();
  if (e >= L.ne) return;
  size_t n = L.n;
  int ia = L.ea[e], ib = L.eb[e];
  double A[8], B[8], dl[5], d[5], da[5], db[5], iva[5], ivb[5];
  ldrec<8>(L.rec0 + 8 * (size_t)ia, A);
  ldrec<8>(L.rec0 + 8 * (size_t)ib, B);
#pragma unroll
  for (int c = 0; c < 5; ++c) dl[c] = lam[c * n + ia] - lam[c * n + ib];
  double ga[GREC], gb[GREC];
  ldrec<GREC>(L.grec + GREC * (size_t)ia, ga);
  ldrec<GREC>(L.grec + GREC * (size_t)ib, gb);
  const double *xa = L.xyz + 3 * (size_t)ia, *xb = L.xyz + 3 * (size_t)ib;
  const double dx = xb[0] - xa[0], dy = xb[1] - xa[1], dz = xb[2] - xa[2];
  const double hl = 0.5 * P.clip * ::sqrt(dx * dx + dy * dy + dz * dz);
  int code = 0;
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    double a = muscl_projection<double>(ga, dx, dy, dz, j), b = muscl_projection<double>(gb, dx, dy, dz, j);
    bool ha = false, hb = false;
    da[j] = db[j] = 1.0;
    iva[j] = ivb[j] = 0.0;
    if (P.autoclip == 1) {
      a = led_slopes<NSIG>(a, ga[15 + j], ga[20 + j], da[j], iva[j], ha);
      b = -led_slopes<NSIG>(-b, gb[15 + j], gb[20 + j], db[j], ivb[j], hb);
      ivb[j] = -ivb[j];
    }
    double c = 0.0;
    int who = 0;
    if (!(a * b <= 0.0)) {
      const bool first = ::fabs(a) <= ::fabs(b);
      c = first ? a : b;
      who = first ? 1 : 2;
      if (::fabs(c) > hl && hl > 0.0) {
        c = c > 0.0 ? hl : -hl;
        who = 0;
      }
    }
    d[j] = c;
    // the chosen end's derivatives, in da and iva
    da[j] = who == 1 ? da[j] : who == 2 ? db[j] : 0.0;
    iva[j] = who == 1 ? iva[j] : who == 2 ? ivb[j] : 0.0;
    code |= (who | ((who == 1 ? ha : hb) ? 4 : 0)) << (3 * j);
  }
  double sa[5], sb[5], sd[5], o[5];
  side_flux_reverse<true>(P, A, B, d, L.w[3 * e], L.w[3 * e + 1], L.w[3 * e + 2], dl, sa, sb, sd);
  double2 *out = reinterpret_cast<double2 *>(abuf2 + LIN_SIDE * (size_t)e);
  double w[LIN_SIDE];
  record_share(A, sa, o);
#pragma unroll
  for (int c = 0; c < 5; ++c) w[c] = o[c];
  record_share(B, sb, o);
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    w[19 + c] = o[c];
    w[5 + c] = sd[c] * da[c];
    w[10 + c] = sd[c] * iva[c];
  }
  w[15] = dx;
  w[16] = dy;
  w[17] = dz;
  w[18] = double(code);
#pragma unroll
  for (int c = 0; c < LIN_SIDE / 2; ++c) out[c] = make_double2(w[2 * c], w[2 * c + 1]);
}

// per node: ub = its conserved-state shares (sides and boundary sides),
// gbn = its gradient and bound shares.  SCALED: the gradients' divided by the
// node's volume and the bounds' times their squares, GREC words a node, as
// k_grad_adjoint reads its neighbours'.
// A side's words are read as aligned pairs, whole, and masked afterwards (a
// load behind each mask waits for the one before), and the scaled records are
// stored through LDS: 360 -> 226 us on 275k nodes with 1.87M sides.
template <bool SCALED, int SUB>
__global__ __launch_bounds__(NTHR) void k_adjoint_gather2(LevelDev<double> L, const double *abuf2, double *ub, double *gbn) {
  constexpr bool STORE = SCALED && SUB == 1;
  __shared__ double st[STORE ? NTHR * (GREC / 2) : 1];
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (!STORE && i >= L.n) return;
  double r[5] = {0, 0, 0, 0, 0}, g[GREC];
#pragma unroll
  for (int c = 0; c < GREC; ++c) g[c] = 0;
  if (i < L.n) {
    for_edges<SUB>(L, i, sub, [&](int e, int role) {
      const double *a = abuf2 + LIN_SIDE * (size_t)e;
      double u[6], w[16];  // words 0 .. 5 or 18 .. 23, and 4 .. 19
      ldrec<6>(a + 18 * role, u);
      ldrec<16>(a + 4, w);
      const double hx = 0.5 * w[11], hy = 0.5 * w[12], hz = 0.5 * w[13];
      const int code = int(w[14]);
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        r[c] += role ? u[c + 1] : u[c];
        const int k = code >> (3 * c);
        const bool mine = (k & 3) == role + 1;
        const double v = mine ? w[1 + c] : 0.0, b = mine ? w[6 + c] : 0.0;
        g[c] += v * hx;
        g[5 + c] += v * hy;
        g[10 + c] += v * hz;
        g[15 + c] += k & 4 ? 0.0 : b;
        g[20 + c] += k & 4 ? b : 0.0;
      }
    });
    for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
      int v = L.bs_list[k];
      const double *b = L.bbuf + 10 * (size_t)(v >> 1) + 5 * (v & 1);
#pragma unroll
      for (int c = 0; c < 5; ++c) r[c] += b[c];
    }
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) r[c] = lsum<SUB>(r[c]);
#pragma unroll
  for (int c = 0; c < LIN_G; ++c) g[c] = lsum<SUB>(g[c]);
  const bool ok = i < L.n && !sub;
  if (ok) {
#pragma unroll
    for (int c = 0; c < 5; ++c) ub[5 * (size_t)i + c] = r[c];
    if constexpr (SCALED) {
      const double iv = 1.0 / L.vol[i];
      double B[12];  // words 14 .. 25 of the gradient record
      ldrec<12>(L.grec + GREC * (size_t)i + 14, B);
#pragma unroll
      for (int c = 0; c < 15; ++c) g[c] *= iv;
#pragma unroll
      for (int c = 15; c < LIN_G; ++c) g[c] = g[c] * B[c - 14] * B[c - 14];
    }
  }
  if constexpr (STORE) {
    const int i0 = i - (int)threadIdx.x;
    store_grec(st, g, ok, gbn + GREC * (size_t)i0, L.n - i0 < NTHR ? L.n - i0 : NTHR);
  } else if (ok) {
    constexpr int NW = SCALED ? GREC : LIN_G;
#pragma unroll
    for (int c = 0; c < NW; ++c) gbn[NW * (size_t)i + c] = g[c];
  }
}

// transpose of the gradient and bounds: qb[5 j + c] = sum over the G and B
// that q_j(c) enters of their shares times d(G, B)/dq_j(c); gbn as
// k_adjoint_gather2<true> scales it, so a neighbour costs its 15 gradient
// shares, its ten extremal-neighbour indices and a bound's share only where
// node j attains it (with the raw shares, the volumes and the bounds read per
// neighbour it took 462 us at 64^3, 161 now; with the bounds' shares always
// read, 270: the two more lines a neighbour cost more than the branches).
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_grad_adjoint(LevelDev<double> L, const double *gbn, const int *amin, double *qb) {
  int j, sub, bb_;
  node_lanes<SUB>(1, bb_, j, sub);
  if (j >= L.n) return;
  double r[5] = {0, 0, 0, 0, 0}, s[3] = {0, 0, 0};
  const double *gj = gbn + GREC * (size_t)j;
  // neighbours i: G_i holds (q_i + q_j) w_s(i -> j) / V_i with w_s(i -> j) = -w_s(j -> i)
  for_edges_w<SUB>(L, j, sub, [&](int i, double wx, double wy, double wz) {
    s[0] += wx;
    s[1] += wy;
    s[2] += wz;
    const double *gi = gbn + GREC * (size_t)i;
    double g[16];
    ldrec<16>(gi, g);
    const int2 *am = reinterpret_cast<const int2 *>(amin + 10 * (size_t)i);
    int k[10];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      int2 t = am[c];
      k[2 * c] = t.x;
      k[2 * c + 1] = t.y;
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      r[c] -= g[c] * wx + g[5 + c] * wy + g[10 + c] * wz;
      if (k[c] == j) r[c] -= gi[15 + c];
      if (k[5 + c] == j) r[c] -= gi[20 + c];
    }
  });
  // boundary sides: G_j holds (3 q_j + q_o) w_b / V_j and G_o (3 q_o + q_j) w_b / V_o
  for (int k = L.bs_ptr[j] + sub; k < L.bs_ptr[j + 1]; k += SUB) {
    int v = L.bs_list[k], b = v >> 1;
    int o = (v & 1) ? L.ba[b] : L.bb[b];
    double wx = L.wb[3 * b], wy = L.wb[3 * b + 1], wz = L.wb[3 * b + 2];
    s[0] += 3.0 * wx;
    s[1] += 3.0 * wy;
    s[2] += 3.0 * wz;
    const double *go = gbn + GREC * (size_t)o;
#pragma unroll
    for (int c = 0; c < 5; ++c) r[c] += go[c] * wx + go[5 + c] * wy + go[10 + c] * wz;
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) r[c] = lsum<SUB>(r[c]);
#pragma unroll
  for (int c = 0; c < 3; ++c) s[c] = lsum<SUB>(s[c]);
  if (sub) return;
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    r[c] += gj[c] * s[0] + gj[5 + c] * s[1] + gj[10 + c] * s[2];
    r[c] += gj[15 + c] + gj[20 + c];
    qb[5 * (size_t)j + c] = r[c];
  }
}

// out(i) = ub(i) + (dq/dU)^T qb(i): the record's dependence on the state
__global__ __launch_bounds__(NTHR) void k_record_adjoint(LevelDev<double> L, DevParams P, const double *ub, const double *qb, double *out) {
  using ad::Dual;
  int i = gtid_x();
  if (i >= L.n) return;
  size_t n = L.n;
  double u[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) u[c] = L.u[c * n + i];
#pragma unroll 1
  for (int k = 0; k < 5; ++k) {
    Dual U[5], A[8];
#pragma unroll
    for (int c = 0; c < 5; ++c) U[c] = Dual(u[c], k == c ? 1.0 : 0.0);
    state_record(U, P.gamma, A);
    double acc = ub[5 * (size_t)i + k];
#pragma unroll
    for (int c = 0; c < 5; ++c) acc += qb[5 * (size_t)i + c] * A[c].d;
    out[k * n + i] = acc;
  }
  out[5 * n + i] = 0;
}

// ---------------------------------------------------------------------------
// Mesh adjoint of the second-order residual: d(lam^T R) with respect to the
// side weights, boundary-side weights, dual volumes and coordinates.  The
// side flux reads w directly, the coordinates through dx = X_b - X_a (the
// reconstruction and its clip length), and the Green-Gauss gradients G,
// which hold (q_a + q_b) w_s / V (sides, node-signed w_s) and
// (3 q_i + q_o) w_b / V (boundary sides).  gbn = d(lam^T R)/d(G, B) per node
// from the state adjoint's side shares (k_flux_adjoint2, k_adjoint_gather2).
// ---------------------------------------------------------------------------
// per side: gw[3 e + k] (direct and through both ends' gradients) and
// gdx[3 e + k] = d(lam^T R)/d dx_k
template <int NSIG>
__global__ __launch_bounds__(NTHR) void k_flux_mesh_adjoint2(LevelDev<double> L, DevParams P, const double *lam, const double *gbn,
                                     double *gw, double *gdx) {
  using ad::Dual;
  int e = gtid_x();
  if (e >= L.ne) return;
  size_t n = L.n;
  int ia = L.ea[e], ib = L.eb[e];
  Dual Ua[5], Ub[5], A[8], B[8], GA[LIN_G], GB[LIN_G];
  double d[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    Ua[c] = Dual(L.u[c * n + ia]);
    Ub[c] = Dual(L.u[c * n + ib]);
    d[c] = lam[c * n + ia] - lam[c * n + ib];
  }
  state_record(Ua, P.gamma, A);
  state_record(Ub, P.gamma, B);
  const double *ga = L.grec + GREC * (size_t)ia, *gb = L.grec + GREC * (size_t)ib;
#pragma unroll
  for (int c = 0; c < LIN_G; ++c) {
    GA[c] = Dual(ga[c]);
    GB[c] = Dual(gb[c]);
  }
  const double w0 = L.w[3 * e], w1 = L.w[3 * e + 1], w2 = L.w[3 * e + 2];
  const double *xa = L.xyz + 3 * (size_t)ia, *xb = L.xyz + 3 * (size_t)ib;
#pragma unroll 1
  for (int k = 0; k < 6; ++k) {
    Dual XA[3] = {Dual(xa[0]), Dual(xa[1]), Dual(xa[2])};
    Dual XB[3] = {Dual(xb[0], k == 3 ? 1.0 : 0.0), Dual(xb[1], k == 4 ? 1.0 : 0.0), Dual(xb[2], k == 5 ? 1.0 : 0.0)};
    Dual o[6];
    side_flux<Dual, double, 2, false, NSIG, Dual, Dual>(P, GA, GB, XA, XB, A, B, Dual(w0, k == 0 ? 1.0 : 0.0),
                                                        Dual(w1, k == 1 ? 1.0 : 0.0), Dual(w2, k == 2 ? 1.0 : 0.0), o);
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 5; ++c) acc += d[c] * o[c].d;
    if (k < 3) {
      // the gradients: G_a holds (q_a + q_b) w / V_a, G_b holds -(q_a + q_b) w / V_b
      const double *qa = L.rec0 + 8 * (size_t)ia, *qb = L.rec0 + 8 * (size_t)ib;
      const double *sa = gbn + LIN_G * (size_t)ia + 5 * k, *sb = gbn + LIN_G * (size_t)ib + 5 * k;
      const double iva = 1.0 / L.vol[ia], ivb = 1.0 / L.vol[ib];
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        double s = qa[c] + qb[c];
        acc += sa[c] * s * iva - sb[c] * s * ivb;
      }
      gw[3 * (size_t)e + k] = acc;
    } else {
      gdx[3 * (size_t)e + k - 3] = acc;
    }
  }
}

// per boundary side: adds the gradients' share to gwb (the direct share of
// the first-order boundary flux is k_bflux_metric_adjoint's): G_a holds
// (3 q_a + q_b) w_b / V_a and G_b holds (3 q_b + q_a) w_b / V_b
__global__ __launch_bounds__(NTHR) void k_bgrad_mesh_adjoint(LevelDev<double> L, const double *gbn, double *gwb) {
  int s = gtid_x();
  if (s >= L.nbs) return;
  int ia = L.ba[s], ib = L.bb[s];
  const double *qa = L.rec0 + 8 * (size_t)ia, *qb = L.rec0 + 8 * (size_t)ib;
  const double iva = 1.0 / L.vol[ia], ivb = 1.0 / L.vol[ib];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double *sa = gbn + LIN_G * (size_t)ia + 5 * k, *sb = gbn + LIN_G * (size_t)ib + 5 * k;
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 5; ++c)
      acc += sa[c] * (3.0 * qa[c] + qb[c]) * iva + sb[c] * (3.0 * qb[c] + qa[c]) * ivb;
    gwb[3 * (size_t)s + k] += acc;
  }
}

// per node: d(lam^T R)/dV_i = -sum gbn_i . G_i / V_i (G is a sum over V)
__global__ __launch_bounds__(NTHR) void k_vol_mesh_adjoint(LevelDev<double> L, const double *gbn, double *gvol) {
  int i = gtid_x();
  if (i >= L.n) return;
  const double *g = L.grec + GREC * (size_t)i, *s = gbn + LIN_G * (size_t)i;
  double acc = 0;
#pragma unroll
  for (int c = 0; c < 15; ++c) acc += s[c] * g[c];
  gvol[i] = -acc / L.vol[i];
}

// ---------------------------------------------------------------------------
// Tangent and adjoint of the laminar viscous term (makeViscosityTerm,
// DEF:5198-5893; dissipation(:,2:5) = -A).  A node's record a = (u, v, w, T)
// with T = gamma/(gamma-1) p/rho; its Green-Gauss sums g = sum (a_i + a_j)
// w + sum_b (3 a_i + a_o) w_b; the stress and heat flux from g/V, the
// Sutherland viscosity of max(T, 0.001) and the adiabatic-wall projection;
// A = sum over sides of E(tau_i, tau_j, u_i, u_j; w) and over non-symmetry
// boundary sides of B(tau_i, tau_o, u_i, u_o; w_b).  The functions below
// form the terms of visc_node and ViscFluxPart on any arithmetic type, the
// energy flux from both ends' stresses and velocities instead of their sums.
// ---------------------------------------------------------------------------
constexpr int VLIN = 66;  // scratch doubles per node of the viscous linearisation

// Sutherland's laminar viscosity of max(T, 0.001) (ViscNodePart::finish)
template <typename T>
__device__ __forceinline__ T sutherland(const DevParams &P, T Traw) {
  T Tn = Traw;
  if (Tn <= T(0.001)) Tn = T(0.001);
  T tc = T((P.gamma - 1.0) * P.mach * P.mach), Tin = T(P.inflow_temperature);
  T tct = tc * Tn;
  return T(1.0 / P.Re) * ((tct * sqrt(tct)) * ((Tin + T(198.6)) / (tc * Tin * Tn + T(198.6))));
}

// vorticity magnitude and divergence from the Green-Gauss sums (ViscNodePart::finish)
template <typename T, typename TV = double>
__device__ __forceinline__ void visc_vort_divg(const T *g, TV vol, T &vort, T &divg) {
  T vt = T(1.0) / T(vol);
  T dudx = g[0] * vt, dvdx = g[1] * vt, dwdx = g[2] * vt;
  T dudy = g[4] * vt, dvdy = g[5] * vt, dwdy = g[6] * vt;
  T dudz = g[8] * vt, dvdz = g[9] * vt, dwdz = g[10] * vt;
  vort = sqrt((dudy - dvdx) * (dudy - dvdx) + (dvdz - dwdy) * (dvdz - dwdy) + (dwdx - dudz) * (dwdx - dudz));
  divg = dudx + dvdy + dwdz;
}

// viscosity and conductivity of the stress law, the eddy viscosity's shares
// included with Spalart-Allmaras
template <typename T>
__device__ __forceinline__ void visc_coef(const DevParams &P, T Traw, T rho, T nu, T &mu, T &k) {
  mu = sutherland(P, Traw);
  k = T(1.0 / P.Pr) * mu;
  if (P.sa) {
    T tvc = T(1.0 / P.Re) * rho * nu;
    T ksi = tvc / mu;
    T k3 = ksi * ksi * ksi;
    tvc = tvc * k3 / (k3 + T(357.9));
    mu = mu + tvc;
    k = k + tvc * T(1.0 / P.Prt);
  }
}

// stress and heat flux of a node; with Spalart-Allmaras the eddy viscosity
// of (rho, nu~) is added to both (DEF:5556-5566).  The volume and the wall
// normal are of type TV (double, or dual numbers for the mesh derivatives).
template <typename T, typename TV = double>
__device__ __forceinline__ void visc_tau(const DevParams &P, const T *g, TV vol, T Traw, bool wall, const TV *nrm,
                                         T *t, T rho = T(0.0), T nu = T(0.0)) {
  T vt = T(1.0) / T(vol);
  T dudx = g[0] * vt, dvdx = g[1] * vt, dwdx = g[2] * vt, dTdx = g[3] * vt;
  T dudy = g[4] * vt, dvdy = g[5] * vt, dwdy = g[6] * vt, dTdy = g[7] * vt;
  T dudz = g[8] * vt, dvdz = g[9] * vt, dwdz = g[10] * vt, dTdz = g[11] * vt;
  T mu, k;
  visc_coef(P, Traw, rho, nu, mu, k);
  T two3 = T(2.0 / 3.0), four3 = T(4.0 / 3.0);
  t[0] = mu * (four3 * dudx - two3 * (dvdy + dwdz));
  t[1] = mu * (dudy + dvdx);
  t[2] = mu * (dudz + dwdx);
  t[3] = mu * (four3 * dvdy - two3 * (dudx + dwdz));
  t[4] = mu * (dvdz + dwdy);
  t[5] = mu * (four3 * dwdz - two3 * (dudx + dvdy));
  t[6] = k * dTdx;
  t[7] = k * dTdy;
  t[8] = k * dTdz;
  if (wall) {
    T nx = T(nrm[0]), ny = T(nrm[1]), nz = T(nrm[2]);
    T nt = t[6] * nx + t[7] * ny + t[8] * nz;
    t[6] -= nt * nx;
    t[7] -= nt * ny;
    t[8] -= nt * nz;
  }
}

template <typename T, typename W>
__device__ __forceinline__ void visc_edge(const T *t1, const T *tj, const T *q1, const T *q2, W wx_, W wy_, W wz_,
                                          T *a) {
  T wx = T(wx_), wy = T(wy_), wz = T(wz_);
  T u1 = q1[0], v1 = q1[1], w1 = q1[2], u2 = q2[0], v2 = q2[1], w2 = q2[2];
  T d[9];
#pragma unroll
  for (int c = 0; c < 9; ++c) d[c] = t1[c] + tj[c];
  T dut1 = u1 * t1[0] + u2 * tj[0] + v1 * t1[1] + v2 * tj[1] + w1 * t1[2] + w2 * tj[2];
  T dut2 = u1 * t1[1] + u2 * tj[1] + v1 * t1[3] + v2 * tj[3] + w1 * t1[4] + w2 * tj[4];
  T dut3 = u1 * t1[2] + u2 * tj[2] + v1 * t1[4] + v2 * tj[4] + w1 * t1[5] + w2 * tj[5];
  a[0] += wx * d[0] + wy * d[1] + wz * d[2];
  a[1] += wx * d[1] + wy * d[3] + wz * d[4];
  a[2] += wx * d[2] + wy * d[4] + wz * d[5];
  a[3] += wx * (d[6] + dut1) + wy * (d[7] + dut2) + wz * (d[8] + dut3);
}

template <typename T, typename W>
__device__ __forceinline__ void visc_bside(const T *t1, const T *to, const T *q1, const T *qo, W wx_, W wy_, W wz_,
                                           T *a) {
  T wx = T(wx_), wy = T(wy_), wz = T(wz_);
  T u1 = q1[0], v1 = q1[1], w1 = q1[2], u2 = qo[0], v2 = qo[1], w2 = qo[2];
  T d[9];
#pragma unroll
  for (int c = 0; c < 9; ++c) d[c] = t1[c] + to[c];
  T du11 = u1 * t1[0] + v1 * t1[1] + w1 * t1[2], du12 = u2 * to[0] + v2 * to[1] + w2 * to[2];
  T du21 = u1 * t1[1] + v1 * t1[3] + w1 * t1[4], du22 = u2 * to[1] + v2 * to[3] + w2 * to[4];
  T du31 = u1 * t1[2] + v1 * t1[4] + w1 * t1[5], du32 = u2 * to[2] + v2 * to[4] + w2 * to[5];
  T dut1 = du11 + du12, dut2 = du21 + du22, dut3 = du31 + du32;
  a[0] += (wx * d[0] + wy * d[1] + wz * d[2]) + T(2) * (wx * t1[0] + wy * t1[1] + wz * t1[2]);
  a[1] += (wx * d[1] + wy * d[3] + wz * d[4]) + T(2) * (wx * t1[1] + wy * t1[3] + wz * t1[4]);
  a[2] += (wx * d[2] + wy * d[4] + wz * d[5]) + T(2) * (wx * t1[2] + wy * t1[4] + wz * t1[5]);
  a[3] += (wx * (d[6] + dut1) + wy * (d[7] + dut2) + wz * (d[8] + dut3)) +
          T(2) * (wx * (t1[6] + du11) + wy * (t1[7] + du21) + wz * (t1[8] + du31));
}

__device__ __forceinline__ bool visc_wall(const LevelDev<double> &L, int i) {
  return L.gnum == 1 && (L.ncls[i] & NC_MASK) == NC_WALL;
}

// Green-Gauss sums g[12] of the node records (values)
template <int SUB>
__device__ __forceinline__ void visc_sums(const LevelDev<double> &L, const DevParams &P, int i, int sub, double *g) {
  const double gog1 = P.gamma / (P.gamma - 1.0);
  double q[8];
  ldrec<8>(L.rec0 + 8 * (size_t)i, q);
  const double ai[4] = {q[1], q[2], q[3], gog1 * q[5] / q[0]};
#pragma unroll
  for (int c = 0; c < 12; ++c) g[c] = 0.0;
  for_edges_w<SUB>(L, i, sub, [&](int j, double wx, double wy, double wz) {
    double r[8];
    ldrec<8>(L.rec0 + 8 * (size_t)j, r);
    const double aj[4] = {r[1], r[2], r[3], gog1 * r[5] / r[0]}, ww[3] = {wx, wy, wz};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int c = 0; c < 4; ++c) g[4 * d + c] += (ai[c] + aj[c]) * ww[d];
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    double r[8];
    ldrec<8>(L.rec0 + 8 * (size_t)o, r);
    const double ao[4] = {r[1], r[2], r[3], gog1 * r[5] / r[0]};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int c = 0; c < 4; ++c) g[4 * d + c] += (2.0 * ai[c] + (ai[c] + ao[c])) * L.wb[3 * s + d];
  }
#pragma unroll
  for (int c = 0; c < 12; ++c) g[c] = lsum<SUB>(g[c]);
}

// the stress and heat-flux record of each node (values, for the adjoint and
// mesh kernels), taud[9 i + c]
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_visc_stress(LevelDev<double> L, DevParams P, ad::Dual *taud) {
  using ad::Dual;
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (i >= L.n) return;
  double g[12], t[9];
  visc_sums<SUB>(L, P, i, sub, g);
  if (sub) return;
  const double *q = L.rec0 + 8 * (size_t)i;
  visc_tau(P, g, L.vol[i], P.gamma / (P.gamma - 1.0) * q[5] / q[0], visc_wall(L, i), L.nrm + 3 * (size_t)i, t, q[0], q[6]);
#pragma unroll
  for (int c = 0; c < 9; ++c) taud[9 * (size_t)i + c] = Dual(t[c]);
}

// Tangent of the viscous term and, with Spalart-Allmaras, of its diffusion
// (makeSADiffusion, DEF:7436-7808) and source (makeSASourceTerm,
// DEF:9285-9370) along the record tangent dq.  Pass 1, one walk: the sums of
// (u, v, w, T) and nu~ and their tangents; from them on dual numbers the
// node's parts of the side fluxes, whose tangents vt[12 i ..] = stress 6 |
// energy flux 3 | diffusion flux 3 are all that pass 2 reads of a neighbour;
// dnode[i] = the tangent of the nodal cb2 term and the source.  (Two walks per
// pass, on dual records with both ends' factors, took 542 us at 275k nodes;
// 204 now, 131 + 73.)
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_visc_tangent1(LevelDev<double> L, DevParams P, const double *dq, double *vt,
                                                        double *dnode) {
  using ad::Dual;
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (i >= L.n) return;
  const double gog1 = P.gamma / (P.gamma - 1.0);
  double qi[8], di[8];
  ldrec<8>(L.rec0 + 8 * (size_t)i, qi);
  ldrec<8>(dq + DQ * (size_t)i, di);
  // (u, v, w, T, nu~) and tangents
  const double a0[5] = {qi[1], qi[2], qi[3], gog1 * qi[5] / qi[0], qi[6]}, t0[5] = {di[1], di[2], di[3], di[7], di[6]};
  double g[15], h[15];
#pragma unroll
  for (int c = 0; c < 15; ++c) g[c] = h[c] = 0.0;
  for_edges_w<SUB>(L, i, sub, [&](int j, double wx, double wy, double wz) {
    double q[8], d[8];
    ldrec<8>(L.rec0 + 8 * (size_t)j, q);
    ldrec<8>(dq + DQ * (size_t)j, d);
    const double aj[5] = {q[1], q[2], q[3], gog1 * q[5] / q[0], q[6]}, tj[5] = {d[1], d[2], d[3], d[7], d[6]};
    const double ww[3] = {wx, wy, wz};
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        g[5 * k + c] += (a0[c] + aj[c]) * ww[k];
        h[5 * k + c] += (t0[c] + tj[c]) * ww[k];
      }
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    double q[8], d[8];
    ldrec<8>(L.rec0 + 8 * (size_t)o, q);
    ldrec<8>(dq + DQ * (size_t)o, d);
    const double ao[5] = {q[1], q[2], q[3], gog1 * q[5] / q[0], q[6]}, to[5] = {d[1], d[2], d[3], d[7], d[6]};
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const double w = L.wb[3 * s + x];
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        const bool four = c == 4 && P.bterm != 1;  // nu~ with boundaryTerm 2
        g[5 * x + c] += (four ? 4.0 * a0[c] : 3.0 * a0[c] + ao[c]) * w;
        h[5 * x + c] += (four ? 4.0 * t0[c] : 3.0 * t0[c] + to[c]) * w;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 15; ++c) {
    g[c] = lsum<SUB>(g[c]);
    h[c] = lsum<SUB>(h[c]);
  }
  if (sub) return;
  Dual G[12], t[9];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int c = 0; c < 4; ++c) G[4 * k + c] = Dual(g[5 * k + c], h[5 * k + c]);
  const Dual u(a0[0], t0[0]), v(a0[1], t0[1]), w(a0[2], t0[2]), T(a0[3], t0[3]);
  const Dual rho(qi[0], di[0]), nu(qi[6], di[6]);
  const double V = L.vol[i];
  visc_tau(P, G, V, T, visc_wall(L, i), L.nrm + 3 * (size_t)i, t, rho, nu);
  double *out = vt + 12 * (size_t)i;
#pragma unroll
  for (int c = 0; c < 6; ++c) out[c] = t[c].d;
  out[6] = (t[6] + u * t[0] + v * t[1] + w * t[2]).d;
  out[7] = (t[7] + u * t[1] + v * t[3] + w * t[4]).d;
  out[8] = (t[8] + u * t[2] + v * t[4] + w * t[5]).d;
  if (!P.sa) {
    out[9] = out[10] = out[11] = 0.0;
    return;
  }
  Dual mu = sutherland(P, T);
  const Dual coef = Dual(P.Re) * mu / rho + nu;
  const double iv = 1.0 / V, f1 = 1.0 / P.Re * 0.622 / (2.0 / 3.0);
  double gg = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const Dual d(g[5 * k + 4] * iv, h[5 * k + 4] * iv);
    out[9 + k] = (coef * d).d;
    gg += 2.0 * g[5 * k + 4] * d.d;
  }
  Dual vort, divg;
  visc_vort_divg(G, V, vort, divg);
  if (mu < Dual(0.1 / P.Re)) mu = Dual(0.1 * P.Re);  // sa_source's guard
  dnode[i] = -f1 * gg + sa_source_t<Dual>(P, rho, nu, mu, vort, divg, L.wd[i], V).d;
}

// pass 2: the side fluxes' tangents from both ends' parts, added to out
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_visc_tangent2(LevelDev<double> L, DevParams P, const double *vt,
                                                        const double *dnode, double *out) {
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (i >= L.n) return;
  const size_t n = L.n;
  double ti[12], a[5] = {0, 0, 0, 0, 0};
  ldrec<12>(vt + 12 * (size_t)i, ti);
  auto add = [&](const double *d, double wx, double wy, double wz) {
    a[0] += wx * d[0] + wy * d[1] + wz * d[2];
    a[1] += wx * d[1] + wy * d[3] + wz * d[4];
    a[2] += wx * d[2] + wy * d[4] + wz * d[5];
    a[3] += wx * d[6] + wy * d[7] + wz * d[8];
  };
  for_edges_w<SUB>(L, i, sub, [&](int j, double wx, double wy, double wz) {
    double d[12];
    ldrec<12>(vt + 12 * (size_t)j, d);
#pragma unroll
    for (int c = 0; c < 12; ++c) d[c] += ti[c];
    add(d, wx, wy, wz);
    a[4] += wx * d[9] + wy * d[10] + wz * d[11];
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1, ind = L.bind[s];
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    const double wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
    double d[12], e[12];
    ldrec<12>(vt + 12 * (size_t)o, d);
#pragma unroll
    for (int c = 0; c < 12; ++c) e[c] = 3.0 * ti[c] + d[c];
    if (ind != 2 && ind != 9) add(e, wx, wy, wz);
    if (P.bterm == 1) a[4] += wx * e[9] + wy * e[10] + wz * e[11];
    else a[4] += 4.0 * (wx * ti[9] + wy * ti[10] + wz * ti[11]);
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) a[c] = lsum<SUB>(a[c]);
  if (sub) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) out[(c + 1) * n + i] -= a[c];
  if (P.sa) out[5 * n + i] += dnode[i] - 1.0 / P.Re / (2.0 / 3.0) * a[4];
}

// adjoint pass 1: shares of lam^T(-A) on node i's stress record (taub 9)
// and velocities through the energy flux (ub 3); tau values in taud (pass 1
// without tangents).  A side's flux is the sum of its ends' own parts, each
// linear in the weight, so node i's part meets -(lam_i - lam_j) w over its
// sides and -(3 lam_i + lam_o) w_b over its boundary sides: the walk sums
// those 4 x 3 numbers, and the shares follow from the node's own stress and
// velocity.  (Twelve dual passes of each side's flux at both ends took 489 us
// at 275k nodes, 73 now.)
template <int SUB>
__global__ __launch_bounds__(NTHR) void k_visc_adjoint_tau(LevelDev<double> L, DevParams P, const double *lam, const ad::Dual *taud,
                                   double *taub, double *ubv) {
  int i, sub, bb_;
  node_lanes<SUB>(1, bb_, i, sub);
  if (i >= L.n) return;
  const size_t n = L.n;
  double li[4], M[4][3];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    li[c] = lam[(c + 1) * n + i];
    M[c][0] = M[c][1] = M[c][2] = 0.0;
  }
  for_edges_w<SUB>(L, i, sub, [&](int j, double wx, double wy, double wz) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const double m = lam[(c + 1) * n + j] - li[c];
      M[c][0] += m * wx;
      M[c][1] += m * wy;
      M[c][2] += m * wz;
    }
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1;
    int ind = L.bind[s];
    if (ind == 2 || ind == 9) continue;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const double m = -(3.0 * li[c] + lam[(c + 1) * n + o]);
#pragma unroll
      for (int d = 0; d < 3; ++d) M[c][d] += m * L.wb[3 * s + d];
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int d = 0; d < 3; ++d) M[c][d] = lsum<SUB>(M[c][d]);
  if (sub) return;
  double t[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) t[c] = taud[9 * (size_t)i + c].v;
  const double *q = L.rec0 + 8 * (size_t)i;
  const double u = q[1], v = q[2], w = q[3];
  const double *E = M[3];  // the energy flux: k grad T + tau . v
  double *tb = taub + 9 * (size_t)i, *ub = ubv + 3 * (size_t)i;
  tb[0] = M[0][0] + u * E[0];
  tb[1] = M[0][1] + M[1][0] + v * E[0] + u * E[1];
  tb[2] = M[0][2] + M[2][0] + w * E[0] + u * E[2];
  tb[3] = M[1][1] + v * E[1];
  tb[4] = M[1][2] + M[2][1] + w * E[1] + v * E[2];
  tb[5] = M[2][2] + w * E[2];
  tb[6] = E[0];
  tb[7] = E[1];
  tb[8] = E[2];
  ub[0] = t[0] * E[0] + t[1] * E[1] + t[2] * E[2];
  ub[1] = t[1] * E[0] + t[3] * E[1] + t[4] * E[2];
  ub[2] = t[2] * E[0] + t[4] * E[1] + t[5] * E[2];
}

// adjoint pass 2: the stress law transposed at each node, gbar[12] on the
// Green-Gauss sums and tbar on T (through the viscosity).  With
// Spalart-Allmaras the stress reads the eddy viscosity of (rho, nu~) and
// the node's SA source (multiplier lam(6)) reads rho, nu~, the laminar
// viscosity of T and the vorticity and divergence of the same sums;
// rnbar[2 i ..] = the shares on (rho, nu~).  The shares on the sums are closed
// forms, the others a dual pass each (with a pass for each sum too: 213 us at
// 275k nodes, 103 now).  lam may be null (no
// source term: the drag's friction alone drives taub).  With mbar (5 per
// node) also the shares on the mesh quantities the node reads: its volume,
// its wall normal (wall nodes, the adiabatic projection) and, with
// Spalart-Allmaras, its wall distance (the source).
__global__ __launch_bounds__(NTHR) void k_visc_adjoint_node(LevelDev<double> L, DevParams P, const double *lam, const double *taub,
                                    double *gbar, double *tbar, double *rnbar, double *mbar) {
  using ad::Dual;
  int i = gtid_x();
  if (i >= L.n) return;
  double gv[12];
  visc_sums<1>(L, P, i, 0, gv);
  const double *qi = L.rec0 + 8 * (size_t)i;
  const double Tv = P.gamma / (P.gamma - 1.0) * qi[5] / qi[0];
  const double *tb = taub + 9 * (size_t)i;
  const bool wall = visc_wall(L, i);
  const double l6 = (P.sa && lam) ? lam[5 * (size_t)L.n + i] : 0.0;
  const double *nr = L.nrm + 3 * (size_t)i;
  double m[5] = {0, 0, 0, 0, 0};
  const double vt = 1.0 / L.vol[i];
  {
    // the sums: the stress and heat flux are linear in them, the source reads
    // the vorticity (one dual pass for its share) and the divergence
    double mu, k, gb[12];
    visc_coef(P, Tv, qi[0], qi[6], mu, k);
    mu *= vt;
    k *= vt;
    const double tr = 2.0 / 3.0 * (tb[0] + tb[3] + tb[5]);
    gb[0] = mu * (2.0 * tb[0] - tr);
    gb[5] = mu * (2.0 * tb[3] - tr);
    gb[10] = mu * (2.0 * tb[5] - tr);
    gb[1] = gb[4] = mu * tb[1];
    gb[2] = gb[8] = mu * tb[2];
    gb[6] = gb[9] = mu * tb[4];
    const double nt = wall ? tb[6] * nr[0] + tb[7] * nr[1] + tb[8] * nr[2] : 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) gb[4 * d + 3] = k * (wall ? tb[6 + d] - nt * nr[d] : tb[6 + d]);
    if (l6 != 0.0) {
      double vort, divg, ml = sutherland(P, Tv);
      visc_vort_divg(gv, L.vol[i], vort, divg);
      if (ml < 0.1 / P.Re) ml = 0.1 * P.Re;
      const Dual S = sa_source_t<Dual, Dual>(P, Dual(qi[0]), Dual(qi[6]), Dual(ml), Dual(vort, 1.0), Dual(divg),
                                             Dual(L.wd[i]), Dual(L.vol[i]));
      const double sv = vort > 0.0 ? l6 * S.d * vt * vt / vort : 0.0;
      const double sd = -l6 * (qi[6] > 0.0 ? qi[6] : 0.0);
      const double c1 = sv * (gv[4] - gv[1]), c2 = sv * (gv[9] - gv[6]), c3 = sv * (gv[2] - gv[8]);
      gb[4] += c1;
      gb[1] -= c1;
      gb[9] += c2;
      gb[6] -= c2;
      gb[2] += c3;
      gb[8] -= c3;
      gb[0] += sd;
      gb[5] += sd;
      gb[10] += sd;
    }
    double2 *o = reinterpret_cast<double2 *>(gbar + 12 * (size_t)i);
#pragma unroll
    for (int c = 0; c < 6; ++c) o[c] = make_double2(gb[2 * c], gb[2 * c + 1]);
  }
  // seeds: 12 T, 13 rho, 14 nu~, 15 V, 16-18 the normal, 19 the wall distance
  const int passes = mbar ? 20 : (P.sa ? 15 : 13);
#pragma unroll 1
  for (int k = 12; k < passes; ++k) {
    if ((k == 13 || k == 14 || k == 19) && !P.sa) continue;
    if (k >= 16 && k <= 18 && !wall) continue;
    Dual gs[12], t[9];
#pragma unroll
    for (int c = 0; c < 12; ++c) gs[c] = Dual(gv[c]);
    const Dual T(Tv, k == 12 ? 1.0 : 0.0), R(qi[0], k == 13 ? 1.0 : 0.0), N(qi[6], k == 14 ? 1.0 : 0.0);
    const Dual Vd(L.vol[i], k == 15 ? 1.0 : 0.0), Wd(L.wd[i], k == 19 ? 1.0 : 0.0);
    const Dual nd[3] = {Dual(nr[0], k == 16 ? 1.0 : 0.0), Dual(nr[1], k == 17 ? 1.0 : 0.0),
                        Dual(nr[2], k == 18 ? 1.0 : 0.0)};
    visc_tau<Dual, Dual>(P, gs, Vd, T, wall, nd, t, R, N);
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 9; ++c) acc += tb[c] * t[c].d;
    if (l6 != 0.0) {
      // the source with sa_source's laminar viscosity guard
      Dual mu = sutherland(P, T);
      if (mu < Dual(0.1 / P.Re)) mu = Dual(0.1 * P.Re);
      Dual vort, divg;
      visc_vort_divg(gs, Vd, vort, divg);
      acc += l6 * sa_source_t<Dual, Dual>(P, R, N, mu, vort, divg, Wd, Vd).d;
    }
    if (k == 12) tbar[i] = acc;
    else if (k < 15) rnbar[2 * (size_t)i + (k - 13)] = acc;
    else if (k == 15) m[0] = acc;
    else if (k == 16) m[1] = acc;
    else if (k == 17) m[2] = acc;
    else if (k == 18) m[3] = acc;
    else m[4] = acc;
  }
  if (mbar)
#pragma unroll
    for (int c = 0; c < 5; ++c) mbar[5 * (size_t)i + c] = m[c];
}

// adjoint pass 3: the Green-Gauss sums transposed, abar[4 j + q] on node j's
// record (u, v, w, T), plus its direct shares (T through the viscosity, the
// velocities through the energy flux)
__global__ __launch_bounds__(NTHR) void k_visc_adjoint_grad(LevelDev<double> L, const double *gbar, const double *tbar, const double *ubv,
                                    double *abar) {
  int j = gtid_x();
  if (j >= L.n) return;
  const double *gj = gbar + 12 * (size_t)j;
  double r[4] = {ubv[3 * (size_t)j], ubv[3 * (size_t)j + 1], ubv[3 * (size_t)j + 2], tbar[j]};
  double sw[3] = {0, 0, 0};
  for_edges_w<1>(L, j, 0, [&](int i, double wx, double wy, double wz) {
    sw[0] += wx;
    sw[1] += wy;
    sw[2] += wz;
    const double *gi = gbar + 12 * (size_t)i;
    const double ww[3] = {wx, wy, wz};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] -= gi[4 * d + q] * ww[d];
  });
  double sb[3] = {0, 0, 0};
  for (int k = L.bs_ptr[j]; k < L.bs_ptr[j + 1]; ++k) {
    int v = L.bs_list[k], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    const double ww[3] = {L.wb[3 * s], L.wb[3 * s + 1], L.wb[3 * s + 2]};
    const double *go = gbar + 12 * (size_t)o;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      sb[d] += ww[d];
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] += go[4 * d + q] * ww[d];
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double s = sw[d] + 3.0 * sb[d];
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] += gj[4 * d + q] * s;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) abar[4 * (size_t)j + q] = r[q];
}

// adjoint pass 4: out(c, i) += (da/dU)^T abar (the record's dependence on
// the conserved state)
__global__ __launch_bounds__(NTHR) void k_visc_adjoint_record(LevelDev<double> L, DevParams P, const double *abar, double *out) {
  using ad::Dual;
  int i = gtid_x();
  if (i >= L.n) return;
  const size_t n = L.n;
  double u[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) u[c] = L.u[c * n + i];
  const double *ab = abar + 4 * (size_t)i;
#pragma unroll 1
  for (int k = 0; k < 5; ++k) {
    Dual U[5], A[8];
#pragma unroll
    for (int c = 0; c < 5; ++c) U[c] = Dual(u[c], k == c ? 1.0 : 0.0);
    state_record(U, P.gamma, A);
    Dual T = Dual(P.gamma / (P.gamma - 1.0)) * A[5] / A[0];
    out[k * n + i] += ab[0] * A[1].d + ab[1] * A[2].d + ab[2] * A[3].d + ab[3] * T.d;
  }
}

// adjoint of the SA diffusion (SADiff1Part and SADiff2Part transposed),
// multipliers m = lam(6).  Forward, node k: g_k = sum_j
// (nu_k + nu_j) w_kj + boundary terms, d_k = g_k / V_k, the nodal term
// -f1 g_k.d_k, and the side terms -f2 (v_k w.d_k + v_j w.d_j) with
// v = Re mu_lam / rho + nu~.  Pass 1, node k: W_k = sum_j (m_k - m_j) w_kj
// (+ (3 m_k + m_o) w_b, or 4 m_k w_b), the share on d_k is -f2 v_k W_k and
// on v_k -f2 W_k.d_k; gnbar[3 k] = the share on g_k; v_k's share goes to
// rho and nu~ (rnbar) and to T through Sutherland's law (tbar).
// With mbar it also adds the share on node k's volume (through d_k and the
// nodal term) to mbar[5 k] and keeps (d_k, v_k) in sad[4 k ..] for the side
// weights' shares (k_visc_mesh_side / k_visc_mesh_bside).
__global__ __launch_bounds__(NTHR) void k_sa_diff_adjoint1(LevelDev<double> L, DevParams P, const double *lam, double *gnbar, double *tbar,
                                   double *rnbar, double *mbar, double *sad) {
  using ad::Dual;
  int k = gtid_x();
  if (k >= L.n) return;
  const size_t n = L.n;
  const double *qk = L.rec0 + 8 * (size_t)k;
  const double mk = lam[5 * n + k], nk = qk[6];
  double g[3] = {0, 0, 0}, W[3] = {0, 0, 0};
  for_edges_w<1>(L, k, 0, [&](int j, double wx, double wy, double wz) {
    const double s = nk + L.rec0[8 * (size_t)j + 6], dm = mk - lam[5 * n + j];
    g[0] += wx * s;
    g[1] += wy * s;
    g[2] += wz * s;
    W[0] += wx * dm;
    W[1] += wy * dm;
    W[2] += wz * dm;
  });
  for (int q = L.bs_ptr[k]; q < L.bs_ptr[k + 1]; ++q) {
    int v = L.bs_list[q], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    const double c = P.bterm == 1 ? 3.0 * nk + L.rec0[8 * (size_t)o + 6] : 4.0 * nk;
    const double cm = P.bterm == 1 ? 3.0 * mk + lam[5 * n + o] : 4.0 * mk;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      g[d] += c * L.wb[3 * s + d];
      W[d] += cm * L.wb[3 * s + d];
    }
  }
  const double vt = 1.0 / L.vol[k];
  const double f1 = 1.0 / P.Re * 0.622 / (2.0 / 3.0), f2 = 1.0 / P.Re / (2.0 / 3.0);
  const double rho = qk[0], T = P.gamma / (P.gamma - 1.0) * qk[5] / rho;
  const Dual mu = sutherland(P, Dual(T, 1.0));
  const double vk = P.Re * mu.v / rho + nk;
  const double vb = -f2 * (W[0] * g[0] + W[1] * g[1] + W[2] * g[2]) * vt;
#pragma unroll
  for (int d = 0; d < 3; ++d) gnbar[3 * (size_t)k + d] = vt * (-f2 * vk * W[d] - 2.0 * f1 * mk * g[d]);
  tbar[k] += vb * P.Re / rho * mu.d;
  rnbar[2 * (size_t)k] -= vb * P.Re * mu.v / (rho * rho);
  rnbar[2 * (size_t)k + 1] += vb;
  if (mbar) {
    // vt = 1 / V scales d_k = g_k vt and the nodal term -f1 vt g_k.g_k
    double dg = 0, gg = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      dg += -f2 * vk * W[d] * g[d];
      gg += g[d] * g[d];
    }
    mbar[5 * (size_t)k] += -vt * vt * (dg - f1 * mk * gg);
#pragma unroll
    for (int d = 0; d < 3; ++d) sad[4 * (size_t)k + d] = g[d] * vt;
    sad[4 * (size_t)k + 3] = vk;
  }
}

// pass 2, node m: the grad nu~ sums transposed (node m's nu~ enters its own
// g with sum_j w_mj + 3 (or 4) sum_b w_b, its neighbours' g with w_jm =
// -w_mj and, boundaryTerm 1, its boundary partners' g with w_b), plus the
// (rho, nu~) shares; added to out
__global__ __launch_bounds__(NTHR) void k_sa_diff_adjoint2(LevelDev<double> L, DevParams P, const double *gnbar, const double *rnbar,
                                   double *out) {
  int m = gtid_x();
  if (m >= L.n) return;
  const size_t n = L.n;
  const double *gm = gnbar + 3 * (size_t)m;
  double r = rnbar[2 * (size_t)m + 1];
  for_edges_w<1>(L, m, 0, [&](int j, double wx, double wy, double wz) {
    const double *gj = gnbar + 3 * (size_t)j;
    r += wx * (gm[0] - gj[0]) + wy * (gm[1] - gj[1]) + wz * (gm[2] - gj[2]);
  });
  for (int q = L.bs_ptr[m]; q < L.bs_ptr[m + 1]; ++q) {
    int v = L.bs_list[q], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    const double wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
    const double *go = gnbar + 3 * (size_t)o;
    const double self = wx * gm[0] + wy * gm[1] + wz * gm[2];
    r += P.bterm == 1 ? 3.0 * self + (wx * go[0] + wy * go[1] + wz * go[2]) : 4.0 * self;
  }
  out[m] += rnbar[2 * (size_t)m];
  out[5 * n + m] += r;
}

// (u, v, w, T) of node i's record
__device__ __forceinline__ void visc_rec_v(const LevelDev<double> &L, const DevParams &P, int i, double *a) {
  const double *q = L.rec0 + 8 * (size_t)i;
  a[0] = q[1];
  a[1] = q[2];
  a[2] = q[3];
  a[3] = P.gamma / (P.gamma - 1.0) * q[5] / q[0];
}

// Mesh adjoint of the viscous and SA terms, interior side e: the share on
// its weight w (3), added to dgw[3 e ..].  w enters the Green-Gauss sums of
// both ends (g_a += (a_a + a_b) w, g_b -= (a_a + a_b) w; the same for nu~),
// the viscous edge flux of both ends (linear in w; node b's weight is -w)
// and the SA diffusion's side terms -f2 (v_a d_a + v_b d_b).w of node a
// (node b: the negative).  gbar / gnbar are the shares on the sums; lam
// null: the sums of the viscous records only (the drag's friction).
__global__ __launch_bounds__(NTHR) void k_visc_mesh_side(LevelDev<double> L, DevParams P, const double *lam, const ad::Dual *taud,
                                 const double *gbar, const double *gnbar, const double *sad, double *dgw) {
  int e = gtid_x();
  if (e >= L.ne) return;
  const size_t n = L.n;
  const int ia = L.ea[e], ib = L.eb[e];
  double aa[4], ab[4], r[3];
  visc_rec_v(L, P, ia, aa);
  visc_rec_v(L, P, ib, ab);
  const double *ga = gbar + 12 * (size_t)ia, *gb = gbar + 12 * (size_t)ib;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    r[d] = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[d] += (ga[4 * d + q] - gb[4 * d + q]) * (aa[q] + ab[q]);
  }
  if (lam) {
    double ta[9], tb[9], ma[4], mb[4];
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      ta[c] = taud[9 * (size_t)ia + c].v;
      tb[c] = taud[9 * (size_t)ib + c].v;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      ma[c] = -lam[(c + 1) * n + ia];
      mb[c] = -lam[(c + 1) * n + ib];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double e1[4] = {0, 0, 0, 0}, e2[4] = {0, 0, 0, 0};
      visc_edge(ta, tb, aa, ab, d == 0 ? 1.0 : 0.0, d == 1 ? 1.0 : 0.0, d == 2 ? 1.0 : 0.0, e1);
      visc_edge(tb, ta, ab, aa, d == 0 ? 1.0 : 0.0, d == 1 ? 1.0 : 0.0, d == 2 ? 1.0 : 0.0, e2);
#pragma unroll
      for (int c = 0; c < 4; ++c) r[d] += ma[c] * e1[c] - mb[c] * e2[c];
    }
    if (P.sa) {
      const double *na = gnbar + 3 * (size_t)ia, *nb = gnbar + 3 * (size_t)ib;
      const double *sa_ = sad + 4 * (size_t)ia, *sb = sad + 4 * (size_t)ib;
      const double sn = L.rec0[8 * (size_t)ia + 6] + L.rec0[8 * (size_t)ib + 6];
      const double f2 = 1.0 / P.Re / (2.0 / 3.0), dl6 = lam[5 * n + ia] - lam[5 * n + ib];
#pragma unroll
      for (int d = 0; d < 3; ++d) r[d] += (na[d] - nb[d]) * sn - f2 * dl6 * (sa_[3] * sa_[d] + sb[3] * sb[d]);
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) dgw[3 * (size_t)e + d] += r[d];
}

// the same for boundary side s (ends a, b, weight w_b, the same for both
// ends): the sums (3 a_i + a_o) w_b at each end, the viscous boundary flux
// of each end (indicators other than 2 and 9) and the SA diffusion's
// boundary terms (boundaryTerm 1: -f2 (3 v_i d_i + v_o d_o).w_b, 2:
// -4 f2 v_i d_i.w_b); added to dgwb[3 s ..]
__global__ __launch_bounds__(NTHR) void k_visc_mesh_bside(LevelDev<double> L, DevParams P, const double *lam, const ad::Dual *taud,
                                  const double *gbar, const double *gnbar, const double *sad, double *dgwb) {
  int s = gtid_x();
  if (s >= L.nbs) return;
  const size_t n = L.n;
  const int ia = L.ba[s], ib = L.bb[s], ind = L.bind[s];
  double aa[4], ab[4], r[3];
  visc_rec_v(L, P, ia, aa);
  visc_rec_v(L, P, ib, ab);
  const double *ga = gbar + 12 * (size_t)ia, *gb = gbar + 12 * (size_t)ib;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    r[d] = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      r[d] += ga[4 * d + q] * (3.0 * aa[q] + ab[q]) + gb[4 * d + q] * (3.0 * ab[q] + aa[q]);
  }
  if (lam) {
    if (!(ind == 2 || ind == 9)) {
      double ta[9], tb[9], ma[4], mb[4];
#pragma unroll
      for (int c = 0; c < 9; ++c) {
        ta[c] = taud[9 * (size_t)ia + c].v;
        tb[c] = taud[9 * (size_t)ib + c].v;
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        ma[c] = -lam[(c + 1) * n + ia];
        mb[c] = -lam[(c + 1) * n + ib];
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double e1[4] = {0, 0, 0, 0}, e2[4] = {0, 0, 0, 0};
        visc_bside(ta, tb, aa, ab, d == 0 ? 1.0 : 0.0, d == 1 ? 1.0 : 0.0, d == 2 ? 1.0 : 0.0, e1);
        visc_bside(tb, ta, ab, aa, d == 0 ? 1.0 : 0.0, d == 1 ? 1.0 : 0.0, d == 2 ? 1.0 : 0.0, e2);
#pragma unroll
        for (int c = 0; c < 4; ++c) r[d] += ma[c] * e1[c] + mb[c] * e2[c];
      }
    }
    if (P.sa) {
      const double *na = gnbar + 3 * (size_t)ia, *nb = gnbar + 3 * (size_t)ib;
      const double *sa_ = sad + 4 * (size_t)ia, *sb = sad + 4 * (size_t)ib;
      const double va = L.rec0[8 * (size_t)ia + 6], vb = L.rec0[8 * (size_t)ib + 6];
      const double f2 = 1.0 / P.Re / (2.0 / 3.0), la = lam[5 * n + ia], lb = lam[5 * n + ib];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (P.bterm == 1)
          r[d] += na[d] * (3.0 * va + vb) + nb[d] * (3.0 * vb + va) -
                  f2 * (la * (3.0 * sa_[3] * sa_[d] + sb[3] * sb[d]) + lb * (3.0 * sb[3] * sb[d] + sa_[3] * sa_[d]));
        else
          r[d] += na[d] * 4.0 * va + nb[d] * 4.0 * vb - f2 * 4.0 * (la * sa_[3] * sa_[d] + lb * sb[3] * sb[d]);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) dgwb[3 * (size_t)s + d] += r[d];
}

// the friction term of the drag (calculateLiftAndDrag, DEF:14757-14803,
// with ReynoldsNumber > 0): fct A_i ws_i.t at each counted wall node, with
// ws_i = tau_i n_i (the symmetric stress times the unit normal).  Writes its
// shares on the stress record (taub[9 i ..], the heat-flux slots 0), on the
// wall area (gaf[i]) and on the normal (gnf[3 i ..]: fct A_i tau_i t); the
// caller clears the arrays elsewhere.
__global__ __launch_bounds__(NTHR) void k_friction_shares(LevelDev<double> L, const int *wall_nodes, int nw, const double *warea,
                                  double fct, double t0, double t1, double t2, double groundplane,
                                  const ad::Dual *taud, double *taub, double *gaf, double *gnf) {
  int k = gtid();
  if (k >= nw) return;
  const int ip = wall_nodes[k];
  const double z = L.xyz ? L.xyz[3 * (size_t)ip + 2] : 0.0;
  if (!(z > groundplane + 0.01)) return;
  const double nx = L.nrm[3 * (size_t)ip], ny = L.nrm[3 * (size_t)ip + 1], nz = L.nrm[3 * (size_t)ip + 2];
  const double fa = fct * warea[ip];
  double tau[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) tau[c] = taud[9 * (size_t)ip + c].v;
  double *tb = taub + 9 * (size_t)ip;
  tb[0] = fa * nx * t0;
  tb[1] = fa * (ny * t0 + nx * t1);
  tb[2] = fa * (nz * t0 + nx * t2);
  tb[3] = fa * ny * t1;
  tb[4] = fa * (nz * t1 + ny * t2);
  tb[5] = fa * nz * t2;
  tb[6] = tb[7] = tb[8] = 0.0;
  const double tt0 = tau[0] * t0 + tau[1] * t1 + tau[2] * t2;
  const double tt1 = tau[1] * t0 + tau[3] * t1 + tau[4] * t2;
  const double tt2 = tau[2] * t0 + tau[4] * t1 + tau[5] * t2;
  gaf[ip] = fct * (tt0 * nx + tt1 * ny + tt2 * nz);
  gnf[3 * (size_t)ip] = fa * tt0;
  gnf[3 * (size_t)ip + 1] = fa * tt1;
  gnf[3 * (size_t)ip + 2] = fa * tt2;
}

// mesh adjoint of the SA convection (first order at both HLLC orders):
// side e's share on its weight w, (lam6_a - lam6_b) df6/dw from three dual
// passes; added to dgw[3 e ..]
__global__ __launch_bounds__(NTHR) void k_sa_conv_mesh_adjoint(LevelDev<double> L, DevParams P, const double *lam, double *dgw) {
  using ad::Dual;
  int e = gtid_x();
  if (e >= L.ne) return;
  const size_t n = L.n;
  const int ia = L.ea[e], ib = L.eb[e];
  Dual Ua[5], Ub[5], A[8], B[8];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    Ua[c] = Dual(L.u[c * n + ia]);
    Ub[c] = Dual(L.u[c * n + ib]);
  }
  state_record(Ua, P.gamma, A);
  state_record(Ub, P.gamma, B);
  A[6] = Dual(L.u[5 * n + ia]);
  B[6] = Dual(L.u[5 * n + ib]);
  const double dl = lam[5 * n + ia] - lam[5 * n + ib];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const Dual wx(L.w[3 * e], d == 0 ? 1.0 : 0.0), wy(L.w[3 * e + 1], d == 1 ? 1.0 : 0.0),
        wz(L.w[3 * e + 2], d == 2 ? 1.0 : 0.0);
    dgw[3 * (size_t)e + d] += dl * sa_side_convection(A, B, wx, wy, wz).d;
  }
}

// vectors (nc, N) in device memory and host numbering <-> the level's src /
// rhs (device numbering; d2h = the level's device-to-host index)
__global__ void k_load_host_order(const double *in, const int *d2h, int n, int nc, double *src) {
  int d = gtid_x();
  if (d >= n) return;
  const int h = d2h[d];
  for (int k = 0; k < 6; ++k) src[(size_t)k * n + d] = k < nc ? in[(size_t)k * n + h] : 0.0;
}
__global__ void k_store_host_order(const double *rhs, const int *d2h, int n, int nc, double *out) {
  int d = gtid_x();
  if (d >= n) return;
  const int h = d2h[d];
  for (int k = 0; k < nc; ++k) out[(size_t)k * n + h] = rhs[(size_t)k * n + d];
}

// a level's field <-> nc columns of n doubles in host numbering: component k
// of device node d is at f[sk k + si d]; components from `inv` on are
// reciprocals (the limiter bounds, 0 stays 0).  The renumbering and the
// conversion of FP32 levels run here, one pass at memory speed, so that the
// host only copies: its own pass over the nodes took 33 of the 48 ms of
// reading six components of 2.1M nodes.
template <typename R>
__global__ void k_field_out(const R *f, long long sk, long long si, const int *d2h, int n, int nc, int inv,
                            double *out) {
  int d = gtid_x();
  if (d >= n) return;
  const int h = d2h[d];
  for (int k = 0; k < nc; ++k) {
    double v = double(f[sk * k + si * d]);
    if (k >= inv) v = v != 0.0 ? 1.0 / v : 0.0;
    out[(size_t)k * n + h] = v;
  }
}
template <typename R>
__global__ void k_field_in(const double *in, const int *d2h, int n, int nc, R *f) {
  int d = gtid_x();
  if (d >= n) return;
  const int h = d2h[d];
  for (int k = 0; k < nc; ++k) f[(size_t)k * n + d] = R(in[(size_t)k * n + h]);
}

// out(1) += rnbar(rho), out(6) += rnbar(nu~)
__global__ void k_add_rho_nu(const double *rnbar, int n, double *out) {
  int i = gtid_x();
  if (i >= n) return;
  out[i] += rnbar[2 * (size_t)i];
  out[5 * (size_t)n + i] += rnbar[2 * (size_t)i + 1];
}

// partial derivative of the pressure drag (calculateLiftAndDrag,
// DEF:14757-14803: drag = (2/S) sum_wall -A_i (p_i - p_inf) n_i.t) with
// respect to the conserved state of each node; zero off the wall
__global__ void k_drag_state_gradient(LevelDev<double> L, DevParams P, const int *wall_nodes, int nw,
                                      const double *warea, double fct, double t0, double t1, double t2,
                                      double groundplane, double *out) {
  int k = gtid();
  if (k >= nw) return;
  int ip = wall_nodes[k];
  double z = L.xyz ? L.xyz[3 * (size_t)ip + 2] : 0.0;
  if (!(z > groundplane + 0.01)) return;
  size_t n = L.n;
  double r = L.u[ip], m1 = L.u[n + ip], m2 = L.u[2 * n + ip], m3 = L.u[3 * n + ip], E = L.u[4 * n + ip];
  double g1 = P.gamma - 1.0;
  double pp = g1 * (E - 0.5 * (m1 * m1 + m2 * m2 + m3 * m3) / r);
  double nt = L.nrm[3 * (size_t)ip] * t0 + L.nrm[3 * (size_t)ip + 1] * t1 + L.nrm[3 * (size_t)ip + 2] * t2;
  double s = -fct * warea[ip] * nt;
  if (!(pp > 0.1)) s = 0.0;  // clamped pressure: no dependence
  double ir = 1.0 / r;
  out[ip] += s * g1 * 0.5 * (m1 * m1 + m2 * m2 + m3 * m3) * ir * ir;
  out[n + ip] += -s * g1 * m1 * ir;
  out[2 * n + ip] += -s * g1 * m2 * ir;
  out[3 * n + ip] += -s * g1 * m3 * ir;
  out[4 * n + ip] += s * g1;
}

// ---------------------------------------------------------------------------
// Node-gather "parts".  Each reference edge loop of the time-step, viscous
// and Spalart-Allmaras routines is a part with the same five hooks:
//   init(i)                    node-local set-up
//   edge(j, w)                 one interior side of node i (signed weights)
//   bside(s, o, ind, w)        one boundary side of node i (o: other end)
//   reduce<SUB>()              combine the lanes' partial sums
//   finish(i)                  node-local epilogue and stores
// k_gather runs up to three parts over ONE walk of the incidence lists, so
// loops that read the same neighbours share their gathers.  Every part
// accumulates in the same order whether it runs alone or fused.
// ---------------------------------------------------------------------------
template <typename R>
struct NoPart {
  static constexpr int AUXW = 0;  // words read of the neighbours' viscous records (0: reads the gather records)
  __device__ void init(const LevelDev<R> &, const DevParams &, int, const R *) {}
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *, const R *, R, R, R) {}
  __device__ void bside(const LevelDev<R> &, const DevParams &, const R *, int, int, int, const R *, R, R, R) {}
  template <int SUB>
  __device__ void reduce() {}
  __device__ void finish(const LevelDev<R> &, const DevParams &, int, const R *) {}
};

// makeTimeSteps (DEF:13335-13610)
template <typename R>
struct TimeStepPart {
  static constexpr int AUXW = 0;
  R lam, lamv, cc, am, gam;
  bool visc;
  // a state's convective speed through a face: |w.v| + |w| c
  static __device__ __forceinline__ R speed(const DevParams &P, const R *q, R wx, R wy, R wz, R al) {
    R c = R(P.gamma) * q[5] / q[0];
    c = c > R(0.001) ? c : R(0.001);
    return fabs(wx * q[1] + wy * q[2] + wz * q[3]) + sqrt(c * al);
  }
  __device__ void init(const LevelDev<R> &, const DevParams &P, int, const R *qi) {
    gam = R(P.gamma);
    cc = gam * qi[5] / qi[0];
    cc = cc > R(0.001) ? cc : R(0.001);
    lam = 0;
    lamv = 0;
    visc = P.Re > 0.0;
    am = visc ? R(1.0 / P.Re) : R(0);
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &P, const R *qi, const R *, const R *qj, R wx, R wy,
                       R wz) {
    R al = wx * wx + wy * wy + wz * wz;
    R vn = wx * qi[1] + wy * qi[2] + wz * qi[3];
    lam += fabs(vn) + sqrt(cc * al);
    if (visc) {  // neighbour's viscosity (DEF:13432-13433)
      R vis = P.sa ? qj[7] + qj[6] * am : qj[7];
      vis = am > vis ? am : vis;
      lamv += R(2) * vis * al / qj[0];
    }
  }
  __device__ void bside(const LevelDev<R> &, const DevParams &P, const R *qi, int, int, int, const R *qo, R wx, R wy,
                        R wz) {
    R al = wx * wx + wy * wy + wz * wz;
    R cco = gam * qo[5] / qo[0];
    cco = cco > R(0.001) ? cco : R(0.001);
    R vn1 = fabs(wx * qi[1] + wy * qi[2] + wz * qi[3]);
    R vn2 = fabs(wx * qo[1] + wy * qo[2] + wz * qo[3]);
    R c1 = sqrt(cc * al), c2 = sqrt(cco * al);
    lam += vn1 + (vn1 + vn2) + c1 + (c1 + c2);
    if (visc) {
      R vis1 = P.sa ? qi[7] + qi[6] * am : qi[7];
      R vis2 = P.sa ? qo[7] + qo[6] * am : qo[7];
      vis1 = am > vis1 ? am : vis1;
      vis2 = am > vis2 ? am : vis2;
      R dv1 = R(2) * vis1 * al / qi[0], dv2 = R(2) * vis2 * al / qo[0];
      lamv += dv1 + (dv1 + dv2);
    }
  }
  template <int SUB>
  __device__ void reduce() {
    lam = lsum<SUB>(lam);
    lamv = lsum<SUB>(lamv);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &, int i, const R *) {
    R V = L.vol[i];
    L.dt[i] = R(0.5) / (lam / V + lamv / (V * V));
  }
};

// the node loop of makeViscosityTerm from the Green-Gauss sums g[4 d + q] of
// (u, v, w, T) and the node's temperature T
template <typename R>
__device__ __forceinline__ void visc_node(const LevelDev<R> &L, const DevParams &P, int i, const R *qi, const R *g, R T) {
  R vt = R(1) / L.vol[i];
  R dudx = g[0] * vt, dvdx = g[1] * vt, dwdx = g[2] * vt, dTdx = g[3] * vt;
  R dudy = g[4] * vt, dvdy = g[5] * vt, dwdy = g[6] * vt, dTdy = g[7] * vt;
  R dudz = g[8] * vt, dvdz = g[9] * vt, dwdz = g[10] * vt, dTdz = g[11] * vt;
  if (T <= R(0.001)) T = R(0.001);
  R tc = R((P.gamma - 1.0) * P.mach * P.mach), Tin = R(P.inflow_temperature);
  R tct = tc * T;
  R mu = R(1.0 / P.Re) * ((tct * sqrt(tct)) * ((Tin + R(198.6)) / (tc * Tin * T + R(198.6))));
  R k = R(1.0 / P.Pr) * mu;
  L.mu[i] = mu;
  L.vort[i] = sqrt((dudy - dvdx) * (dudy - dvdx) + (dvdz - dwdy) * (dvdz - dwdy) + (dwdx - dudz) * (dwdx - dudz));
  L.divg[i] = dudx + dvdy + dwdz;
  if (P.sa) {
    double tvc = (1.0 / P.Re) * double(qi[0]) * double(qi[6]);
    double ksi = tvc / double(mu);
    double k3 = ksi * ksi * ksi;
    tvc = tvc * k3 / (k3 + 357.9);
    mu = mu + R(tvc);
    k = k + R(tvc * (1.0 / P.Prt));
  }
  R t[9];
  R two3 = R(2.0 / 3.0), four3 = R(4.0 / 3.0);
  t[0] = mu * (four3 * dudx - two3 * (dvdy + dwdz));
  t[1] = mu * (dudy + dvdx);
  t[2] = mu * (dudz + dwdx);
  t[3] = mu * (four3 * dvdy - two3 * (dudx + dwdz));
  t[4] = mu * (dvdz + dwdy);
  t[5] = mu * (four3 * dwdz - two3 * (dudx + dvdy));
  t[6] = k * dTdx;
  t[7] = k * dTdy;
  t[8] = k * dTdz;
  int cls = L.ncls[i] & NC_MASK;
  if (L.gnum == 1 && cls != NC_NONE) {
    R nx = L.nrm[3 * (size_t)i], ny = L.nrm[3 * (size_t)i + 1], nz = L.nrm[3 * (size_t)i + 2];
    if (cls == NC_WALL) {  // setTemperatureForAdiabaticWall (DEF:5170-5196)
      R nt = t[6] * nx + t[7] * ny + t[8] * nz;
      t[6] -= nt * nx;
      t[7] -= nt * ny;
      t[8] -= nt * nz;
    }
    L.ws[3 * (size_t)i] = t[0] * nx + t[1] * ny + t[2] * nz;
    L.ws[3 * (size_t)i + 1] = t[1] * nx + t[3] * ny + t[4] * nz;
    L.ws[3 * (size_t)i + 2] = t[2] * nx + t[4] * ny + t[5] * nz;
  }
  t[6] += qi[1] * t[0] + qi[2] * t[1] + qi[3] * t[2];
  t[7] += qi[1] * t[1] + qi[2] * t[3] + qi[3] * t[4];
  t[8] += qi[1] * t[2] + qi[2] * t[4] + qi[3] * t[5];
  R *o = L.tau + VREC * (size_t)i;
#pragma unroll
  for (int c = 0; c < 9; ++c) o[c] = t[c];
}

// makeViscosityTerm (DEF:5198-5893), pass 1: gradients of (u,v,w,T) and the
// node loop (Sutherland, SA eddy viscosity, stress, heat flux, vorticity,
// divergence, adiabatic wall, wall stress).  tau: stress 6 + energy flux 3.
// The gather records keep the previous laminar viscosity, which makeTimeSteps
// reads of the neighbours in the same walk.
template <typename R>
struct ViscNodePart {
  static constexpr int AUXW = 0;
  R gog1, ai[4], g[12];
  __device__ void init(const LevelDev<R> &, const DevParams &P, int, const R *qi) {
    gog1 = R(P.gamma / (P.gamma - 1.0));
    ai[0] = qi[1];
    ai[1] = qi[2];
    ai[2] = qi[3];
    ai[3] = gog1 * qi[5] / qi[0];
#pragma unroll
    for (int c = 0; c < 12; ++c) g[c] = 0;
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *, const R *qj, R wx, R wy, R wz) {
    R aj[4] = {qj[1], qj[2], qj[3], gog1 * qj[5] / qj[0]};
    R ww[3] = {wx, wy, wz};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q) g[4 * d + q] += (ai[q] + aj[q]) * ww[d];
  }
  __device__ void bside(const LevelDev<R> &, const DevParams &, const R *, int, int, int, const R *qo, R wx, R wy,
                        R wz) {
    R ao[4] = {qo[1], qo[2], qo[3], gog1 * qo[5] / qo[0]};
    R ww[3] = {wx, wy, wz};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q) g[4 * d + q] += (R(2) * ai[q] + (ai[q] + ao[q])) * ww[d];
  }
  template <int SUB>
  __device__ void reduce() {
#pragma unroll
    for (int c = 0; c < 12; ++c) g[c] = lsum<SUB>(g[c]);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &P, int i, const R *qi) { visc_node(L, P, i, qi, g, ai[3]); }
};

// The gradient records and pass 1 of the viscous term from one walk
// (GradPart, ViscNodePart): the sums of the velocities are the same in both,
// so the temperature's three are all that the second adds.  Kept apart, the
// two walks of level 1 take 434 and 514 us (614 with the time steps) on 2.1M
// nodes, 400 bytes a node of side weights in each; together 718 (796).
template <typename R>
struct GradViscPart {
  static constexpr int AUXW = 0;
  GradPart<R> gp;
  R gog1, T, gT[3];
  __device__ void init(const LevelDev<R> &L, const DevParams &P, int i, const R *qi) {
    gp.init(L, P, i, qi);
    gog1 = R(P.gamma / (P.gamma - 1.0));
    T = gog1 * qi[5] / qi[0];
    gT[0] = gT[1] = gT[2] = 0;
  }
  __device__ void edge(const LevelDev<R> &L, const DevParams &P, const R *qi, const R *tj, const R *qj, R wx, R wy,
                       R wz) {
    gp.edge(L, P, qi, tj, qj, wx, wy, wz);
    R s = T + gog1 * qj[5] / qj[0];
    gT[0] += s * wx;
    gT[1] += s * wy;
    gT[2] += s * wz;
  }
  __device__ void bside(const LevelDev<R> &L, const DevParams &P, const R *qi, int s, int o, int ind, const R *qo, R wx,
                        R wy, R wz) {
    gp.bside(L, P, qi, s, o, ind, qo, wx, wy, wz);
    R t = R(2) * T + (T + gog1 * qo[5] / qo[0]);
    gT[0] += t * wx;
    gT[1] += t * wy;
    gT[2] += t * wz;
  }
  template <int SUB>
  __device__ void reduce() {
    gp.template reduce<SUB>();
#pragma unroll
    for (int d = 0; d < 3; ++d) gT[d] = lsum<SUB>(gT[d]);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &P, int i, const R *qi) {
    gp.finish(L, P, i, qi);
    R g[12];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
#pragma unroll
      for (int q = 0; q < 3; ++q) g[4 * d + q] = gp.g[5 * d + 1 + q];
      g[4 * d + 3] = gT[d];
    }
    visc_node(L, P, i, qi, g, T);
  }
};

// makeViscosityTerm pass 2 (DEF:5640-5893): dissipation(:,2:5) = -sum
template <typename R>
struct ViscFluxPart {
  static constexpr int AUXW = 10;
  R t1[9], a[4];
  __device__ void init(const LevelDev<R> &L, const DevParams &, int i, const R *) {
    const R *ti = L.tau + VREC * (size_t)i;
#pragma unroll
    for (int c = 0; c < 9; ++c) t1[c] = ti[c];
#pragma unroll
    for (int c = 0; c < 4; ++c) a[c] = 0;
  }
  __device__ __forceinline__ void add(const R *d, R wx, R wy, R wz) {
    a[0] += wx * d[0] + wy * d[1] + wz * d[2];
    a[1] += wx * d[1] + wy * d[3] + wz * d[4];
    a[2] += wx * d[2] + wy * d[4] + wz * d[5];
    a[3] += wx * d[6] + wy * d[7] + wz * d[8];
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *tj, const R *, R wx, R wy, R wz) {
    R d[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) d[c] = t1[c] + tj[c];
    add(d, wx, wy, wz);
  }
  __device__ void bside(const LevelDev<R> &L, const DevParams &, const R *, int, int o, int ind, const R *, R wx, R wy,
                        R wz) {
    if (ind == 2 || ind == 9) return;  // symmetry / inviscid wall carry no viscous flux
    const R *to = L.tau + VREC * (size_t)o;
    R d[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) d[c] = (t1[c] + to[c]) + R(2) * t1[c];
    add(d, wx, wy, wz);
  }
  template <int SUB>
  __device__ void reduce() {
#pragma unroll
    for (int c = 0; c < 4; ++c) a[c] = lsum<SUB>(a[c]);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &, int i, const R *) {
    int n = L.n;
    L.diss[i] = 0;
    L.diss[n + i] = -a[0];
    L.diss[2 * n + i] = -a[1];
    L.diss[3 * n + i] = -a[2];
    L.diss[4 * n + i] = -a[3];
  }
};

// makeTurbulentTimeSteps (DEF:12878-13099)
// its viscosity 1.5 (mu + 3 cb2 nu~ / Re) comes from the viscous records
// (sa_step_viscosity, SADiff1Part)
template <typename R>
__device__ __forceinline__ R sa_step_viscosity(const DevParams &P, R mu, R nu) {
  return R(1.5) * (mu + R(3) * R(0.622) * nu * R(1.0 / P.Re));
}
template <typename R>
struct SATimeStepPart {
  static constexpr int AUXW = 14;
  R tk, lam, lamv, self;
  __device__ void init(const LevelDev<R> &L, const DevParams &P, int i, const R *) {
    tk = R(P.turb_k);
    self = L.tau[VREC * (size_t)i + 12];
    lam = 0;
    lamv = 0;
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *qi, const R *tj, const R *, R wx, R wy, R wz) {
    R al = wx * wx + wy * wy + wz * wz;
    R vn = wx * qi[1] + wy * qi[2] + wz * qi[3];
    lam += tk * sqrt(al) + fabs(vn);
    lamv += R(2) * tj[12] * al;
  }
  __device__ void bside(const LevelDev<R> &L, const DevParams &P, const R *qi, int, int o, int, const R *, R wx, R wy,
                        R wz) {
    const R *qo = L.rec0 + 8 * (size_t)o;
    R al = wx * wx + wy * wy + wz * wz;
    R vn1 = tk * sqrt(al) + fabs(wx * qi[1] + wy * qi[2] + wz * qi[3]);
    R vn2 = tk * sqrt(al) + fabs(wx * qo[1] + wy * qo[2] + wz * qo[3]);
    lam += vn1 + (vn1 + vn2);
    R dv1 = R(2) * self * al, dv2 = R(2) * L.tau[VREC * (size_t)o + 12] * al;
    lamv += dv1 + (dv1 + dv2);
  }
  template <int SUB>
  __device__ void reduce() {
    lam = lsum<SUB>(lam);
    lamv = lsum<SUB>(lamv);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &P, int i, const R *qi) {
    R V = L.vol[i];
    R dt = R(0.5) / (lam / V + lamv / (V * V));
    R wd = L.wd[i];
    R di = wd > R(1e-10) ? R(1) / wd : R(1e10);
    di = di * di;
    R ioRe = R(1.0 / P.Re), ik2 = R(1.0 / (0.41 * 0.41)), cb1 = R(0.1355), ct3 = R(1.1);
    R cw1 = cb1 * ik2 + (R(1) + R(0.622)) * R(1.5);
    R nu = qi[6];
    R S = fabs(L.divg[i]) + cb1 * (L.vort[i] + (R(1) + ct3) * nu * ik2 * di * ioRe) + cw1 * nu * di * ioRe;
    L.dtt[i] = dt / (R(1) + R(0.5) * S * dt);
  }
};

// the SA time step's viscosity alone into the viscous records (parity op)
template <typename R>
__global__ void k_sa_step_viscosity(LevelDev<R> L, DevParams P) {
  int bb_;
  int i = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  L.tau[VREC * (size_t)i + 12] = sa_step_viscosity(P, L.mu[i], L.rec0[8 * (size_t)i + 6]);
}

// makeSADiffusion (DEF:7436-7808), pass 1: grad nu~, into the viscous record
// as the node's part of the diffusion flux (with the laminar viscosity that
// pass 1 of the viscous term has just stored), the SA time step's viscosity
// and the nodal cb2 term.  nu~ = u(:,6) is read from the gather records.
template <typename R>
struct SADiff1Part {
  static constexpr int AUXW = 0;
  R ti, g[3];
  __device__ void init(const LevelDev<R> &, const DevParams &, int, const R *qi) {
    ti = qi[6];
    g[0] = g[1] = g[2] = 0;
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *, const R *qj, R wx, R wy, R wz) {
    R s = ti + qj[6];
    g[0] += wx * s;
    g[1] += wy * s;
    g[2] += wz * s;
  }
  __device__ void bside(const LevelDev<R> &, const DevParams &P, const R *, int, int, int, const R *qo, R wx, R wy,
                        R wz) {
    R to = qo[6];
    R c = P.bterm == 1 ? (R(3) * ti + to) : R(4) * ti;
    g[0] += c * wx;
    g[1] += c * wy;
    g[2] += c * wz;
  }
  template <int SUB>
  __device__ void reduce() {
#pragma unroll
    for (int c = 0; c < 3; ++c) g[c] = lsum<SUB>(g[c]);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &P, int i, const R *qi) {
    R vt = R(1) / L.vol[i];
    R dx = g[0] * vt, dy = g[1] * vt, dz = g[2] * vt;
    R fact = R(1.0 / P.Re * 0.622 / (2.0 / 3.0));
    R mu = L.mu[i], v = R(P.Re) * mu / qi[0] + ti;
    R *o = L.dnu + VREC * (size_t)i;
    o[0] = v * dx;
    o[1] = v * dy;
    o[2] = v * dz;
    o[3] = sa_step_viscosity(P, mu, ti);
    o[4] = -(fact * (g[0] * dx + g[1] * dy + g[2] * dz));
  }
};

// makeSADiffusion pass 2
template <typename R>
struct SADiff2Part {
  static constexpr int AUXW = 12;
  R fact, acc, d0, d1, d2, d3;
  __device__ void init(const LevelDev<R> &L, const DevParams &P, int i, const R *) {
    const R *di = L.dnu + VREC * (size_t)i;
    d0 = di[0];
    d1 = di[1];
    d2 = di[2];
    d3 = di[4];
    fact = R(1.0 / P.Re / (2.0 / 3.0));
    acc = 0;
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *tj, const R *, R wx, R wy, R wz) {
    acc += wx * (d0 + tj[9]) + wy * (d1 + tj[10]) + wz * (d2 + tj[11]);
  }
  __device__ void bside(const LevelDev<R> &L, const DevParams &P, const R *, int, int o, int, const R *, R wx, R wy,
                        R wz) {
    const R *dq = L.dnu + VREC * (size_t)o;
    R fd1 = wx * d0 + wy * d1 + wz * d2;
    R fd2 = wx * dq[0] + wy * dq[1] + wz * dq[2];
    acc += P.bterm == 1 ? R(3) * fd1 + fd2 : R(4) * fd1;
  }
  template <int SUB>
  __device__ void reduce() {
    acc = lsum<SUB>(acc);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &, int i, const R *) { L.tdiff[i] = d3 - fact * acc; }
};

// JST passes 1, 2 and the node step of makeArtificialDissipation2
// (DEF:11531-11563, 11659-11672, 11746-11751):
//   L_i = (1/conn_i) sum (U_j - U_i), energy on E + p;
//   nu_i = 12 |sum (p_j - p_i) / sum (p_i + p_j)|;  conn_i = sides at i,
// with the node's volume over its time step (the one in L.dt, or that of
// makeTimeSteps earlier in the same walk) for the scalar form's scale.
template <typename R>
struct JstSumsPart {
  static constexpr int AUXW = 0;
  R U[5], p, h[5], h7, h8, conn;
  // the conserved state from the gather record and the momenta
  static __device__ __forceinline__ void state(const R *q, const R *m, R *u) {
    u[0] = q[0];
    u[1] = m[0];
    u[2] = m[1];
    u[3] = m[2];
    u[4] = q[4];
  }
  __device__ void init(const LevelDev<R> &L, const DevParams &, int i, const R *qi) {
    state(qi, L.mom + 4 * (size_t)i, U);
    p = qi[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) h[c] = 0;
    h7 = h8 = conn = 0;
  }
  __device__ void edge(const LevelDev<R> &, const DevParams &, const R *, const R *mj, const R *qj, R, R, R) {
    R V[5];
    state(qj, mj, V);
#pragma unroll
    for (int c = 0; c < 4; ++c) h[c] += V[c] - U[c];
    h[4] += (V[4] - U[4]) + (qj[5] - p);
    h7 += qj[5] - p;
    h8 += p + qj[5];
    conn += R(1);
  }
  __device__ void bside(const LevelDev<R> &, const DevParams &, const R *, int, int, int, const R *, R, R, R) {}
  template <int SUB>
  __device__ void reduce() {
#pragma unroll
    for (int c = 0; c < 5; ++c) h[c] = lsum<SUB>(h[c]);
    h7 = lsum<SUB>(h7);
    h8 = lsum<SUB>(h8);
    conn = lsum<SUB>(conn);
  }
  __device__ void finish(const LevelDev<R> &L, const DevParams &, int i, const R *) {
    R fact = R(1) / conn;
    R *o = L.jst + 8 * (size_t)i;
#pragma unroll
    for (int c = 0; c < 5; ++c) o[c] = fact * h[c];
    o[5] = R(12) * fabs(h7 / h8);
    o[6] = conn;
    o[7] = L.vol[i] / L.dt[i];
  }
};

template <typename T>
constexpr bool reads_momenta = false;
template <typename R>
constexpr bool reads_momenta<JstSumsPart<R>> = true;

constexpr int max3(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }

// one walk of node i's interior and boundary sides feeding up to three parts
template <typename R, int SUB, typename A, typename B, typename C, typename Walk>
__device__ __forceinline__ void gather_body(LevelDev<R> &L, const DevParams &P, int i, int sub, Walk walk) {
  const R *qi = L.rec0 + 8 * (size_t)i;
  A a;
  B b;
  C c;
  a.init(L, P, i, qi);
  b.init(L, P, i, qi);
  c.init(L, P, i, qi);
  walk([&](const R *qj, const R *tj, R wx, R wy, R wz) {
    a.edge(L, P, qi, tj, qj, wx, wy, wz);
    b.edge(L, P, qi, tj, qj, wx, wy, wz);
    c.edge(L, P, qi, tj, qj, wx, wy, wz);
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k], s = v >> 1;
    int o = (v & 1) ? L.ba[s] : L.bb[s];
    int ind = L.bind[s];
    R qo[8];
    if constexpr (max3(A::AUXW, B::AUXW, C::AUXW) == 0) ldrec<8>(L.rec0 + 8 * (size_t)o, qo);
    R wx = L.wb[3 * s], wy = L.wb[3 * s + 1], wz = L.wb[3 * s + 2];
    a.bside(L, P, qi, s, o, ind, qo, wx, wy, wz);
    b.bside(L, P, qi, s, o, ind, qo, wx, wy, wz);
    c.bside(L, P, qi, s, o, ind, qo, wx, wy, wz);
  }
  if (SUB > 1) {
    a.template reduce<SUB>();
    b.template reduce<SUB>();
    c.template reduce<SUB>();
    if (sub) return;
  }
  a.finish(L, P, i, qi);
  b.finish(L, P, i, qi);
  c.finish(L, P, i, qi);
}

template <typename R, int SUB, typename A, typename B, typename C>
__global__ __launch_bounds__(NTHR) void k_gather(LevelDev<R> L, DevParams P) {
  constexpr int W = max3(A::AUXW, B::AUXW, C::AUXW);
  int i, sub;
  int bb_;
  node_lanes<SUB>(L.nb, bb_, i, sub);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  constexpr bool MOM = reads_momenta<A> || reads_momenta<B> || reads_momenta<C>;
  gather_body<R, SUB, A, B, C>(L, P, i, sub, [&](auto f) { walk_global<SUB, W, MOM>(L, i, sub, f); });
}

template <typename R, typename A, typename B, typename C>
__global__ __launch_bounds__(NTHR) void k_gather_blk(LevelDev<R> L, DevParams P) {
  constexpr int W = max3(A::AUXW, B::AUXW, C::AUXW);
  static_assert(W > 0, "only viscous records are staged");
  constexpr int NS = W == 12 ? 12 : W - 1, S = NS | 1;  // words used, an odd LDS stride
  __shared__ R sn[GB_CAP * S];
  int lb = xcd_block();
  int bb_ = lb % L.nb, blk = lb / L.nb;
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (blk >= L.ngb) return;
  __shared__ int sid[GB_CAP];
  const int n0 = L.gb_nptr[blk], nn = L.gb_nptr[blk + 1] - n0, t = threadIdx.x;
  for (int k = t; k < nn; k += NTHR) sid[k] = L.gb_node[n0 + k];
  __syncthreads();
  {
    using P2 = typename Pair<R>::type;
    constexpr int U = W / 2, PER = (GB_CAP * U + NTHR - 1) / NTHR;
    P2 v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int x = t + q * NTHR, k = x / U;
      if (k < nn) v[q] = reinterpret_cast<const P2 *>(L.tau + VREC * (size_t)sid[k])[x - k * U];
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int x = t + q * NTHR, k = x / U, j = x - k * U;
      if (k < nn) {
        sn[k * S + 2 * j] = v[q].x;
        if (2 * j + 1 < NS) sn[k * S + 2 * j + 1] = v[q].y;
      }
    }
  }
  __syncthreads();
  int i = L.gb_first[blk] + (int)threadIdx.x / GB_SUB, sub = (int)threadIdx.x % GB_SUB;
  if (i >= L.gb_first[blk + 1]) return;
  gather_body<R, GB_SUB, A, B, C>(L, P, i, sub, [&](auto f) { walk_staged<GB_SUB, S>(L, sn, i, sub, f); });
}

// JST pass 3 (DEF:11788-11939): per side (a, b) with dr4 = L_a - L_b and
// dr2 = U_a - U_b,
//   scalar: d0 = min(V_a/dt_a, V_b/dt_b) / (conn_a + conn_b),
//           d2 = d0 k2 max(nu_a, nu_b), d4 = dim(d0 k4, d2);
//   matrix: dr4, dr2 <- |w| |A| dr4, |w| |A| dr2 (Roe matrix along w in
//           Turkel's form, Harten's fix), d2 = k2 max(nu), d4 = dim(k4, d2).
// D_a += -dr4 d4 + dr2 d2 and D_b += dr4 d4 - dr2 d2: at either end the
// differences taken from the node itself enter with the same signs.  Walked
// per node into the dissipation array (`add`: on top of the viscous term
// there; k4: coarse-grid factor below grid 1); the Roe averages take the
// side's stored orientation, so both ends form the same matrix.
// Both passes read the 64-byte records of the neighbours with the level's
// lanes per node; with one lane per node and the conserved state's seven
// scattered words per neighbour they took 19 + 27 us on 9k nodes and 23 + 40
// us on 160, now 8.2 + 6.0 and 6.4 + 5.7 (the first with the time steps).
template <typename R, bool MATRIX, int SUB>
__global__ void k_jst_flux(LevelDev<R> L, DevParams P, int add) {
  int i, sub;
  int bb_;
  node_lanes<SUB>(L.nb, bb_, i, sub);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  const size_t n = L.n;
  const R k2 = R(P.k2), k4 = R(L.gnum == 1 ? P.k4 : P.k4c);
  R qi[8], mi[4], ji[8], Ui[5], acc[5] = {0, 0, 0, 0, 0};
  ldrec<8>(L.rec0 + 8 * (size_t)i, qi);
  ldrec<4>(L.mom + 4 * (size_t)i, mi);
  ldrec<8>(L.jst + 8 * (size_t)i, ji);
  JstSumsPart<R>::state(qi, mi, Ui);
  const int s = i / SLICE, lane = i % SLICE;
  const int base = L.ell_ptr[s], K = L.ell_k[s];
  const long long ns = L.nslot;
  for (int k = sub; k < K; k += SUB) {
    const int slot = base + k * SLICE + lane;
    const int e = L.ell_e[slot];
    if (e < 0) continue;
    const size_t j = L.ell_nbr[slot];
    R qj[8], mj[4], jj[8], Uj[5];
    ldrec<8>(L.rec0 + 8 * j, qj);
    ldrec<4>(L.mom + 4 * j, mj);
    ldrec<8>(L.jst + 8 * j, jj);
    JstSumsPart<R>::state(qj, mj, Uj);
    R d4v[5], d2v[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      d4v[c] = ji[c] - jj[c];
      d2v[c] = Ui[c] - Uj[c];
    }
    R nu = ji[5] > jj[5] ? ji[5] : jj[5];
    R d2, d4;
    if constexpr (!MATRIX) {
      R d0 = (ji[7] < jj[7] ? ji[7] : jj[7]) / (ji[6] + jj[6]);
      d2 = d0 * k2 * nu;
      d4 = d0 * k4;
    } else {
      const R hcf = R(P.hcf), gam1 = R(P.gamma - 1.0);
      const R eps1 = R(1) / (hcf > R(1.e-5) ? hcf : R(1.e-5));
      R rnx = L.ellw[slot], rny = L.ellw[ns + slot], rnz = L.ellw[2 * ns + slot];
      R al = sqrt(rnx * rnx + rny * rny + rnz * rnz), vmo1 = R(1) / al;
      rnx *= vmo1;
      rny *= vmo1;
      rnz *= vmo1;
      const bool second = e & 1;
      R A[6], B[6];  // first and second end: rho, u, v, w, rhoE, p
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        A[c] = second ? qj[c] : qi[c];
        B[c] = second ? qi[c] : qj[c];
      }
      R hl = (A[4] + A[5]) * (R(1) / A[0]), hr = (B[4] + B[5]) * (R(1) / B[0]);
      R di = sqrt(B[0] / A[0]), d1 = R(1) / (di + R(1));
      R ui = (di * B[1] + A[1]) * d1, vi = (di * B[2] + A[2]) * d1, wi = (di * B[3] + A[3]) * d1;
      R hi = (di * hr + hl) * d1;
      R ci2 = gam1 * (hi - R(0.5) * (ui * ui + vi * vi + wi * wi)), ci = sqrt(ci2);
      R af = R(0.5) * (ui * ui + vi * vi + wi * wi), ucp = ui * rnx + vi * rny + wi * rnz;
      R l1 = fabs(ucp + ci), l2 = fabs(ucp - ci), l3 = fabs(ucp);
      if (l1 < hcf) l1 = R(0.5) * (l1 * l1 * eps1 + hcf);
      if (l2 < hcf) l2 = R(0.5) * (l2 * l2 * eps1 + hcf);
      if (l3 < hcf) l3 = R(0.5) * (l3 * l3 * eps1 + hcf);
      R s1 = R(0.5) * (l1 + l2), s2 = R(0.5) * (l1 - l2);
#pragma unroll
      for (int k_ = 0; k_ < 2; ++k_) {
        R *q = k_ == 0 ? d4v : d2v;
        R a1 = gam1 * (af * q[0] - ui * q[1] - vi * q[2] - wi * q[3] + q[4]);
        R a2 = -ucp * q[0] + q[1] * rnx + q[2] * rny + q[3] * rnz;
        R cc1 = ((s1 - l3) * a1 / ci2) + (s2 * a2 / ci);
        R cc2 = (s2 * a1 / ci) + (s1 - l3) * a2;
        R t0 = al * (l3 * q[0] + cc1), t1 = al * (l3 * q[1] + cc1 * ui + cc2 * rnx);
        R t2 = al * (l3 * q[2] + cc1 * vi + cc2 * rny), t3 = al * (l3 * q[3] + cc1 * wi + cc2 * rnz);
        R t4 = al * (l3 * q[4] + cc1 * hi + cc2 * ucp);
        q[0] = t0;
        q[1] = t1;
        q[2] = t2;
        q[3] = t3;
        q[4] = t4;
      }
      d2 = k2 * nu;
      d4 = k4;
    }
    d4 = d4 > d2 ? d4 - d2 : R(0);
#pragma unroll
    for (int c = 0; c < 5; ++c) acc[c] = acc[c] - d4v[c] * d4 + d2v[c] * d2;
  }
  if (SUB > 1) {
#pragma unroll
    for (int c = 0; c < 5; ++c) acc[c] = lsum<SUB>(acc[c]);
    if (sub) return;
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) L.diss[c * n + i] = (add ? L.diss[c * n + i] : R(0)) + acc[c];
}

// ---------------------------------------------------------------------------
// node-local pieces shared by the stage kernels
// ---------------------------------------------------------------------------

// what the boundary conditions read of a node: its class and unit normal
template <typename R>
struct NodeBc {
  int cls;
  R n[3];
};
template <typename R>
__device__ __forceinline__ NodeBc<R> node_bc(const LevelDev<R> &L, int i) {
  NodeBc<R> b{L.ncls[i] & NC_MASK, {0, 0, 0}};
  if (b.cls != NC_NONE)
    for (int k = 0; k < 3; ++k) b.n[k] = L.nrm[3 * (size_t)i + k];
  return b;
}

// setBCsOnIncrementField (DEF:4978-5140) for node i on r[0..5]
template <typename R>
__device__ __forceinline__ void bc_increment(const DevParams &P, const NodeBc<R> &b, R *r) {
  const int cls = b.cls;
  if (cls == NC_NONE || cls == NC_FAR1 || cls == NC_FAR2) return;
  const R nx = b.n[0], ny = b.n[1], nz = b.n[2];
  if (cls == NC_WALL && P.Re > 0.0) {
    r[1] = r[2] = r[3] = 0;
    if (!P.isentropic) r[4] = 0;
    if (P.sa) r[5] = 0;
    return;
  }
  R ni = r[1] * nx + r[2] * ny + r[3] * nz;
  r[1] -= ni * nx;
  r[2] -= ni * ny;
  r[3] -= ni * nz;
  if (P.sa && cls != NC_SYM) r[5] = 0;
}

// setBCsOnSolutionField (DEF:4364-4976) for node i on q[0..5]; rho_g is
// the density of the level's own solution at the time of the call (grp%u,
// which the wall velocity of an Euler wall multiplies whichever array q is).
// Wall velocities come from the level-1 coordinate movement of a moving
// mesh; coarse levels carry none (the reference reads an array it never
// allocates there) and take zero.
template <typename R>
__device__ __forceinline__ void bc_solution(const LevelDev<R> &L, const DevParams &P, int i, const NodeBc<R> &b, R *q,
                                            R rho_g) {
  const int cls = b.cls;
  if (cls == NC_NONE || cls == NC_FAR1 || cls == NC_FAR2) return;
  const R nx = b.n[0], ny = b.n[1], nz = b.n[2];
  const bool moving = L.cmv && L.gnum == 1 && cls == NC_WALL;
  if (cls == NC_WALL && P.Re > 0.0) {
    if (moving) {  // u(2:4) = u(1) * coordinateMovement / dt (DEF:4408)
      R s = q[0] / R(P.dtp);
      q[1] = s * L.cmv[3 * (size_t)i];
      q[2] = s * L.cmv[3 * (size_t)i + 1];
      q[3] = s * L.cmv[3 * (size_t)i + 2];
    } else {
      q[1] = q[2] = q[3] = 0;
    }
    if (!P.isentropic) q[4] = q[0] * R(P.inflow_temperature / P.gamma);
    if (P.sa) q[5] = 0;
    return;
  }
  R nv = q[1] * nx + q[2] * ny + q[3] * nz;
  q[1] -= nv * nx;
  q[2] -= nv * ny;
  q[3] -= nv * nz;
  if (moving && P.add_time) {  // the wall's normal velocity (DEF:4433-4442)
    R dtp = R(P.dtp);
    R wn = (L.cmv[3 * (size_t)i] / dtp) * nx + (L.cmv[3 * (size_t)i + 1] / dtp) * ny +
           (L.cmv[3 * (size_t)i + 2] / dtp) * nz;
    R m = rho_g * wn;
    q[1] += m * nx;
    q[2] += m * ny;
    q[3] += m * nz;
  }
  if (cls == NC_INVWALL && !P.isentropic)
    q[4] = q[0] * R(P.inflow_temperature / P.gamma) + R(0.5) * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0];
  if (P.sa && cls != NC_SYM) q[5] = 0;
}

// setOuterBoundaryConditions (DEF:4018-4251) for node i
template <typename R>
__device__ __forceinline__ void outer_bc(const DevParams &P, const NodeBc<R> &b, R *q, R p) {
  const int cls = b.cls;
  if (cls != NC_FAR1 && cls != NC_FAR2) return;
  double inf[6];
  P.inflow_row(cls - NC_FAR1, inf);
  const R nx = b.n[0], ny = b.n[1], nz = b.n[2];
  R rho0 = R(inf[0]), U1 = R(inf[1]), U2 = R(inf[2]), U3 = R(inf[3]);
  R gm1 = R(P.gamma - 1.0);
  R nv = U1 * nx + U2 * ny + U3 * nz;
  if (nv > R(0)) {
    R rho = q[0];
    (void)rho;
    q[0] = rho0;
    q[1] = U1 * rho0;
    q[2] = U2 * rho0;
    q[3] = U3 * rho0;
    q[4] = P.mach > 1.0 ? R(inf[4]) * rho0 : p / gm1 + R(0.5) * (U1 * U1 + U2 * U2 + U3 * U3) * rho0;
  } else if (P.mach < 1.0) {
    q[4] = R(inf[5]) / gm1 + R(0.5) * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0];
  }
  if (P.sa) q[5] = R(0.1);
}

// gather of the convective residual of node i: interior fluxes from the
// node's partial sums (pbuf) or from one record per incident side (fbuf),
// then the boundary-side shares
template <typename R, bool SA, int SUB>
__device__ __forceinline__ void gather_rhs(const LevelDev<R> &L, int i, int sub, bool partials, R *r) {
  for (int c = 0; c < 6; ++c) r[c] = 0;
  if (partials) {
    for (int k = L.pn_ptr[i] + sub; k < L.pn_ptr[i + 1]; k += SUB) {
      R f[6];
      ldrec<6>(L.pbuf + 6 * (size_t)L.pn_ent[k], f);
#pragma unroll
      for (int c = 0; c < (SA ? 6 : 5); ++c) r[c] += f[c];
    }
  } else for_edges<SUB>(L, i, sub, [&](int e, int role) {
    R f[6];
    ldrec<6>(L.fbuf + 6 * (size_t)e, f);
    if (role) {
#pragma unroll
      for (int c = 0; c < (SA ? 6 : 5); ++c) r[c] -= f[c];
    } else {
#pragma unroll
      for (int c = 0; c < (SA ? 6 : 5); ++c) r[c] += f[c];
    }
  });
  for (int k = L.bs_ptr[i] + sub; k < L.bs_ptr[i + 1]; k += SUB) {
    int v = L.bs_list[k];
    const R *b = L.bbuf + 10 * (size_t)(v >> 1) + 5 * (v & 1);
#pragma unroll
    for (int c = 0; c < 5; ++c) r[c] += b[c];
  }
  if (SUB > 1) {
#pragma unroll
    for (int c = 0; c < 6; ++c) r[c] = lsum<SUB>(r[c]);
  }
}

enum { FLUX_SIDES = 0, FLUX_PARTIALS = 1, FLUX_BLOCK = 2 };  // where a stage takes the interior fluxes from

// Stage kernel modes
//   MODE_RHS      rhs = makeRHS (+ makeSARHS/Source if SA)                 (parity)
//   MODE_STAGE    singleIteration RK stage body (DEF:1074-1180)
//   MODE_COARSE   restrictGrid coarse part (DEF:12185-12234)
//   MODE_FINE     restrictGrid fine part (DEF:12236-12361), rhs := increment
enum { MODE_RHS = 0, MODE_STAGE = 1, MODE_COARSE = 2, MODE_FINE = 3 };

struct StageArgs {
  double dtj, dtj_t, alpha;  // CFL*alpha_k, turbCFL*alpha_k, alpha_k
  int calc_turb;             // SA terms active in this stage
  int fas;                   // subtract alpha*sourceTerm (coarse levels)
  int has_src;               // level has a sourceTerm (gridNumber > 1)
  int partials;              // interior fluxes are per-node partial sums (pbuf), else per-side records (fbuf)
  int next_record;           // MODE_STAGE: also form p and the gather record of the new
                             // state for the next stage (not after the last stage: the
                             // pressure field then stays that of its start, as the
                             // reference's makePressureField leaves it)
};

// what a stage reads of its own node, beside its convective residual
template <typename R>
struct NodeIn {
  R up[6], vol, dt, diss[5], p, u0, u5, src[6], mu, vort, divg, wd, dtt, tdiff;
  NodeBc<R> bc;
};
template <typename R, bool SA>
__device__ __forceinline__ NodeIn<R> node_in(const LevelDev<R> &L, const StageArgs &S, int i) {
  const size_t n = L.n;
  NodeIn<R> in;
  for (int c = 0; c < 6; ++c) in.up[c] = L.uprev[c * n + i];
  for (int c = 0; c < 5; ++c) in.diss[c] = L.diss[c * n + i];
  in.vol = L.vol[i];
  in.dt = L.dt[i];
  in.p = L.p[i];
  in.u0 = L.u[i];
  in.u5 = L.u[5 * n + i];
  if (S.fas || S.has_src)
    for (int c = 0; c < 6; ++c) in.src[c] = L.src[c * n + i];
  in.mu = L.mu[i];
  if constexpr (SA) {
    in.vort = L.vort[i];
    in.divg = L.divg[i];
    in.wd = L.wd[i];
    in.dtt = L.dtt[i];
    in.tdiff = L.tdiff[i];
  }
  in.bc = node_bc(L, i);
  return in;
}

// makeSASourceTerm (DEF:9285-9370) for node i: the rhs(:,6) increment
template <typename R>
__device__ __forceinline__ double sa_source(const LevelDev<R> &L, const DevParams &P, int i, NodeIn<R> &in) {
  double mu = in.mu;
  if (mu < 0.1 / P.Re) {
    mu = 0.1 * P.Re;
    L.mu[i] = in.mu = R(mu);
  }
  return sa_source_t<double>(P, double(in.u0), double(in.u5), mu, double(in.vort), double(in.divg), double(in.wd),
                             double(in.vol));
}

// the stage at node i from its convective residual r[6]; rec, mom: where the
// next state's gather record and momenta go
template <typename R, int MODE, bool SA>
__device__ __forceinline__ void stage_node(const LevelDev<R> &L, const DevParams &P, const StageArgs &S, int i,
                                           NodeIn<R> &in, R *r, R *rec, R *mom) {
  const int n = L.n;
  bool sa_on = SA && S.calc_turb;
  if (sa_on) r[5] += R(sa_source(L, P, i, in));
  if (MODE == MODE_RHS) {
    for (int c = 0; c < 6; ++c) L.rhs[(size_t)c * n + i] = r[c];
    return;
  }
  if (P.unsteady && P.add_time) {
    // addTimeDifferences (DEF:1184-1241): BDF2 on grid 1 with the volumes
    // of the last two physical times (equal to V on a fixed mesh), BDF1
    // elsewhere, over components 1:5 (1:6 with SA).  restrictGrid adds it
    // on both grids (DEF:12208 on the restricted state, DEF:12285)
    const R V = in.vol, dtp = R(P.dtp);
    const R VP = L.volp ? L.volp[i] : V, VP2 = L.volp2 ? L.volp2[i] : V;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      if (c == 5 && !SA) break;
      const size_t k = (size_t)c * n + i;
      if (L.gnum == 1 && P.bdf2)
        r[c] = r[c] + (R(1.5) * V * L.u[k] - R(2.0) * VP * L.uold[k] + R(0.5) * VP2 * L.uold2[k]) / dtp;
      else
        r[c] = r[c] + V * (L.u[k] - L.uold[k]) / dtp;
    }
  }
  for (int c = 0; c < 5; ++c) r[c] += in.diss[c];
  if (SA) r[5] += in.tdiff;
  if (!SA) r[5] = 0;
  // solveSystem (DEF:1407-1479); unsteady: dt / (1 + 1.5 dt / dtp) for the
  // mean flow (DEF:1427-1436)
  R V = in.vol, dt = in.dt;
  if (P.unsteady) dt = dt / (R(1.0) + R(1.5) * dt / R(P.dtp));
  for (int c = 0; c < 5; ++c) r[c] = dt * r[c] / V;
  if (SA) r[5] = in.dtt * r[5] / V;
  bc_increment(P, in.bc, r);
  // updateSolutionVector (DEF:1292-1405)
  R q[6];
  const R *up = in.up;
  R dtj = R(S.dtj);
  for (int c = 0; c < 5; ++c) r[c] = dtj * r[c];
  if (SA) r[5] = R(S.dtj_t) * r[5];
  R inc = r[0];
  if (fabs(inc / up[0]) < R(P.max_inc)) {
    q[0] = up[0] - inc;
  } else {
    R sg = inc / fabs(inc);
    q[0] = up[0] - sg * R(P.max_inc) * up[0];
  }
  for (int c = 1; c < 5; ++c) q[c] = up[c] - r[c];
  if (SA) {
    R t = up[5] - r[5];
    q[5] = t > R(0) ? t : R(0);
  } else {
    q[5] = in.u5;
  }
  // density check on the grid's own u (DEF:1398-1403)
  R ug0 = in.u0;
  if (MODE == MODE_FINE) {
    if (ug0 < R(P.min_rho)) L.u[i] = R(P.min_rho);
  } else if (q[0] < R(P.min_rho)) {
    q[0] = R(P.min_rho);
  }
  // restrictGrid applies the state conditions to the updated state it
  // holds in rhs (DEF:12333-12336) while grp%u keeps the grid's own state
  bc_solution(L, P, i, in.bc, q, MODE == MODE_FINE ? (ug0 < R(P.min_rho) ? R(P.min_rho) : ug0) : q[0]);
  if (MODE == MODE_STAGE) {
    if (S.fas) {
      R a = R(S.alpha);
      for (int c = 0; c < 5; ++c) q[c] -= a * in.src[c];
      if (sa_on) q[5] -= a * in.src[5];
    }
    q[0] = q[0] > R(P.min_rho) ? q[0] : R(P.min_rho);
    if (sa_on) {
      q[5] = q[5] > R(0) ? q[5] : R(0);
      if (q[5] > R(P.max_turb)) q[5] = R(P.max_turb);
    }
    outer_bc(P, in.bc, q, in.p);
    for (int c = 0; c < 6; ++c) L.u[(size_t)c * n + i] = q[c];
    if (!S.next_record) return;
    // pressure and gather record of the new state, as k_prep forms them, so
    // the next stage starts without a separate pass
    write_record(L, P, i, q, in.mu, rec, mom);
  } else if (MODE == MODE_COARSE) {
    outer_bc(P, in.bc, q, in.p);
    for (int c = 0; c < 6; ++c) {
      L.src[(size_t)c * n + i] = q[c] - up[c];
      L.u[(size_t)c * n + i] = up[c];
    }
  } else {  // MODE_FINE
    if (S.has_src) {
      for (int c = 0; c < 5; ++c) q[c] -= in.src[c];
      if (SA) q[5] -= in.src[5];
    }
    if (SA) {
      q[5] = q[5] > R(0) ? q[5] : R(0);
      if (in.u5 > R(P.max_turb)) L.u[5 * (size_t)n + i] = R(P.max_turb);
    }
    outer_bc(P, in.bc, q, in.p);
    for (int c = 0; c < 5; ++c) L.rhs[(size_t)c * n + i] = q[c] - up[c];
    L.rhs[5 * (size_t)n + i] = SA ? q[5] - up[5] : R(0);
  }
}

template <typename R, int MODE, bool SA, int SUB>
__global__ void k_stage(LevelDev<R> L, DevParams P, StageArgs S) {
  int i, sub;
  int bb_;
  node_lanes<SUB>(L.nb, bb_, i, sub);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  R r[6];
  gather_rhs<R, SA, SUB>(L, i, sub, S.partials, r);
  if (sub) return;
  NodeIn<R> in = node_in<R, SA>(L, S, i);
  stage_node<R, MODE, SA>(L, P, S, i, in, r, L.rec0, L.mom);
}

// One launch per stage: the residual of a block of consecutive nodes and
// their update.  The block stages the records of its nodes and of their
// neighbours in LDS, each thread evaluates one task from them (an interior
// side that touches the block, or a boundary side seen from one of the
// block's nodes), the fluxes take the records' place in LDS, and the threads
// of a node sum its tasks and advance it.  A side between two blocks is
// evaluated by both, in its stored orientation, so both ends still take the
// same bits with opposite signs; that is about 1.4 times the arithmetic of
// the sides, for two launches less (side fluxes, boundary fluxes) and no
// partial sums through memory.  The neighbours' records are read while other
// blocks write theirs, so the next state's go to rec1 and the host swaps the
// two.  Latency bounds it, so one task a thread and blocks as large as that
// allows, tables at fixed places (the chain is node ids, records, result),
// and what the update reads of the block's own nodes staged beside the
// records.  Per stage, FP64 without SA,
// against the three launches: 8.8 us for 18 on 1.3k nodes, 23.5 for 27 on
// 33k; with the central, LLF and Roe fluxes, whose records carry the momenta
// too, 8.7 on 1.3k and 10.6 on 9k.  (A walk of each node's own sides, every
// flux at both ends, measured 14 and 40 us.)  Second-order sides stay with k_flux_blk: their records are
// five times as long and their arithmetic twice, so the repeated sides cost
// more than the launches.
// STEP: the nodes' local time steps (makeTimeSteps, inviscid) from the same
// tasks.
constexpr int SB_S = 7;    // LDS stride of a record (not mu) and of a task's result, odd
constexpr int SB_SM = 11;  // of a record with the momenta (fluxType 1-3)

constexpr int SB_IN = 32;  // rows of the update's inputs

template <typename R, int MODE, bool SA, bool HLLC, bool STEP>
__global__ __launch_bounds__(NTHR) void k_stage_blk(LevelDev<R> L, DevParams P, StageArgs S) {
  static_assert(SB_CAP <= SB_TASKS && !(SA && STEP), "one LDS area serves the records and the results");
  constexpr int RS = HLLC ? SB_S : SB_SM;
  __shared__ R sn[SB_CAP * RS > SB_TASKS * SB_S ? SB_CAP * RS : SB_TASKS * SB_S];
  __shared__ R own[SB_IN * SB_NODES];
  __shared__ unsigned short sinc[SB_INC];
  const int lb = xcd_block(), bb_ = lb % L.nb, blk = lb / L.nb, t = threadIdx.x;
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (blk >= L.nsb) return;
  const int *nodes = L.sb_node + (size_t)SB_CAP * blk;
  const size_t task = (size_t)SB_TASKS * blk + t, nt = (size_t)SB_TASKS * L.nsb, n = L.n;
  // this thread's task, the node it sums for and the block's incidences
  const unsigned loc = L.sb_loc[task];
  const R wx = L.sb_w[task], wy = L.sb_w[nt + task], wz = L.sb_w[2 * nt + task];
  const int me = t / SB_SUB, sub = t % SB_SUB, i = nodes[0] + me;
  const unsigned short *ip = L.sb_iptr + (SB_NODES + 1) * (size_t)blk + me;
  const int q0 = ip[0], q1 = ip[1];
#pragma unroll
  for (int q = 0; q < SB_INC / NTHR; ++q) sinc[t + q * NTHR] = L.sb_inc[(size_t)SB_INC * blk + t + q * NTHR];
  // the nodes' records, two words a load
  {
    constexpr int U = HLLC ? 4 : 6;  // two-word units of a record, with the momenta's
    constexpr int PER = (SB_CAP * U + NTHR - 1) / NTHR;
    using P2 = typename Pair<R>::type;
    int g[PER];
    P2 v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int k = (t + q * NTHR) / U;
      g[q] = k < SB_CAP ? nodes[k] : -1;
    }
#pragma unroll
    for (int q = 0; q < PER; ++q)
      if (g[q] >= 0) {
        const int j = (t + q * NTHR) % U;
        const R *rec = j < 4 ? L.rec0 + 8 * (size_t)g[q] + 2 * j : L.mom + 4 * (size_t)g[q] + 2 * (j - 4);
        v[q] = *reinterpret_cast<const P2 *>(rec);
      }
    // and the own nodes' inputs of the update: row r of thread group r
    const int m = t % SB_NODES, r8 = t / SB_NODES, oi = nodes[0] + m < (int)n ? nodes[0] + m : (int)n - 1;
    R x0 = r8 < 6 ? L.uprev[r8 * n + oi] : r8 == 6 ? L.vol[oi] : L.dt[oi];
    R x1 = r8 < 5 ? L.diss[r8 * n + oi] : r8 == 5 ? L.p[oi] : L.u[(r8 == 6 ? 0 : 5) * n + oi];
    R x2 = r8 < 6 ? L.src[r8 * n + oi] : L.nrm[3 * (size_t)oi + r8 - 6];
    R x3 = r8 == 0 ? L.nrm[3 * (size_t)oi + 2] : r8 == 1 ? R(L.ncls[oi]) : r8 == 2 ? L.mu[oi] : r8 == 3 ? L.vort[oi]
           : r8 == 4 ? L.divg[oi] : r8 == 5 ? L.wd[oi] : r8 == 6 ? L.dtt[oi] : L.tdiff[oi];
#pragma unroll
    for (int q = 0; q < PER; ++q)
      if (g[q] >= 0) {
        const int k = (t + q * NTHR) / U, j = (t + q * NTHR) % U;
        R *o = sn + RS * k + (j < 4 ? 2 * j : 2 * j - 1);  // the momenta follow nu~
        o[0] = v[q].x;
        if (j != 3 && j != 5) o[1] = v[q].y;  // not mu, not the pad
      }
    own[t] = x0;
    own[NTHR + t] = x1;
    own[2 * NTHR + t] = x2;
    own[3 * NTHR + t] = x3;
  }
  __syncthreads();
  const int kind = loc >> 24;
  R f[7] = {0, 0, 0, 0, 0, 0, 0};
  if (kind != 255) {
    const R *A = sn + (loc & 0xfffu) * RS, *B = sn + ((loc >> 12) & 0xfffu) * RS;
    if (kind == 0) {
      if constexpr (HLLC) {
        side_flux<R, R, 1, SA, 2>(P, (const R *)nullptr, (const R *)nullptr, (const R *)nullptr, (const R *)nullptr, A,
                                  B, wx, wy, wz, f);
      } else {
        const R UA[5] = {A[0], A[7], A[8], A[9], A[4]}, UB[5] = {B[0], B[7], B[8], B[9], B[4]};
        simple_flux(P, P.ftype, UA, A[5], UB, B[5], wx, wy, wz, R(0), f);
        f[5] = SA ? sa_side_convection(A, B, wx, wy, wz) : R(0);
      }
      if constexpr (STEP) {  // each end's own speed through the side
        const R al = wx * wx + wy * wy + wz * wz;
        f[5] = TimeStepPart<R>::speed(P, A, wx, wy, wz, al);
        f[6] = TimeStepPart<R>::speed(P, B, wx, wy, wz, al);
      }
    } else {
      const int ind = kind - 1;
      const R al = wx * wx + wy * wy + wz * wz, rnorm = sqrt(al);
      if (rnorm > R(1e-10) && (ind <= 4 || ind == 9)) {
        const R irn = R(1) / rnorm;
        R f1[5], f2[5];
        bside_state_flux(P, ind, A, wx * irn, wy * irn, wz * irn, f1);
        bside_state_flux(P, ind, B, wx * irn, wy * irn, wz * irn, f2);
#pragma unroll
        for (int c = 0; c < 5; ++c)
          f[c] = P.bterm == 1 ? rnorm * (R(3) * f1[c] + f2[c]) : rnorm * R(4) * f1[c];
      }
      if constexpr (STEP)
        f[5] = R(2) * TimeStepPart<R>::speed(P, A, wx, wy, wz, al) + TimeStepPart<R>::speed(P, B, wx, wy, wz, al);
    }
  }
  __syncthreads();  // the records are no longer needed: the results take their place
  if (kind != 255) {
#pragma unroll
    for (int c = 0; c < SB_S; ++c) sn[SB_S * t + c] = f[c];
  }
  __syncthreads();
  if (q0 == q1) return;  // beyond the block's nodes (each has a side)
  R r[6] = {0, 0, 0, 0, 0, 0}, lam = 0;
  for (int q = q0 + sub; q < q1; q += SB_SUB) {
    const unsigned v = sinc[q];
    const R *o = sn + SB_S * (v >> 1);
    const bool second = v & 1u;
#pragma unroll
    for (int c = 0; c < (SA ? 6 : 5); ++c) r[c] += second ? -o[c] : o[c];
    if constexpr (STEP) lam += second ? o[6] : o[5];
  }
#pragma unroll
  for (int c = 0; c < (SA ? 6 : 5); ++c) r[c] = lsum<SB_SUB>(r[c]);
  if constexpr (STEP) lam = lsum<SB_SUB>(lam);
  if (sub) return;
  auto row = [&](int x) { return own[SB_NODES * x + me]; };
  NodeIn<R> in;
  for (int c = 0; c < 6; ++c) in.up[c] = row(c);
  in.vol = row(6);
  in.dt = row(7);
  for (int c = 0; c < 5; ++c) in.diss[c] = row(8 + c);
  in.p = row(13);
  in.u0 = row(14);
  in.u5 = row(15);
  for (int c = 0; c < 6; ++c) in.src[c] = row(16 + c);
  for (int c = 0; c < 3; ++c) in.bc.n[c] = row(22 + c);
  in.bc.cls = int(row(25)) & NC_MASK;
  in.mu = row(26);
  in.vort = row(27);
  in.divg = row(28);
  in.wd = row(29);
  in.dtt = row(30);
  in.tdiff = row(31);
  if constexpr (STEP) L.dt[i] = in.dt = R(0.5) / (lam / in.vol);
  stage_node<R, MODE, SA>(L, P, S, i, in, r, L.rec1, HLLC ? L.mom : L.mom1);
}

// ---------------------------------------------------------------------------
// simple node kernels
// ---------------------------------------------------------------------------
template <typename R>
__global__ void k_copy_state(R *dst, const R *src, int n, int ncomp, int nb) {
  int bb_;
  int i = btid(nb, bb_);
  if (i >= n) return;
  dst += (size_t)bb_ * 6 * (size_t)n;
  src += (size_t)bb_ * 6 * (size_t)n;
  for (int c = 0; c < ncomp; ++c) dst[(size_t)c * n + i] = src[(size_t)c * n + i];
}

template <typename R>
__global__ void k_fill(R *dst, R v, size_t cnt) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cnt) dst[i] = v;
}

// node boundary conditions on the level's state (setBCsOnSolutionField)
template <typename R>
__global__ void k_bc_state(LevelDev<R> L, DevParams P) {
  int bb_;
  int i = btid(L.nb, bb_);
  L.to_batch(bb_);
  P.to_batch(bb_);
  if (i >= L.n) return;
  const size_t n = L.n;
  R q[6];
  for (int c = 0; c < 6; ++c) q[c] = L.u[c * n + i];
  bc_solution(L, P, i, node_bc(L, i), q, q[0]);
  for (int c = 0; c < 6; ++c) L.u[c * n + i] = q[c];
}

// restriction (mapFineToCoarse, DEF:12572-12690) as a gather over the fine
// members of each coarse node: out[c*nc+k] = sum_i rw_i in[c*nf+i].  In the
// nested device order the members of coarse node k are the contiguous fine
// range [cptr[k], cptr[k+1]); SUB lanes per coarse node read it coalesced.
//
// The transfers are node-local once the members are summed, so each is one
// launch with all that follows it at the node: the boundary conditions, the
// pressure and records, the forcing, the correction of the fine members.  On
// the small levels a launch costs 4-5 us whatever it does; as separate
// kernels (restriction of u and mu, pressure, conditions, copy, pressure,
// zero dissipation | restriction, forcing | restriction, conditions,
// correction, prolongation) a restriction took 9 launches more and a
// prolongation 3.  Every lane of a group ends its sum with the same bits
// (lsum), so the correction is formed on all of them.
struct Transfer {
  const int *cptr;
  const double *rw;
  int nf;  // fine nodes
};

// sum over the members of coarse node k of NC components of `in`
template <int SUB, int NC, typename RF>
__device__ __forceinline__ void restrict_sum(const Transfer &T, const RF *in, int k, int sub, double *acc) {
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  for (int i = T.cptr[k] + sub; i < T.cptr[k + 1]; i += SUB) {
    double r = T.rw[i];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] += r * double(in[(size_t)c * T.nf + i]);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = lsum<SUB>(acc[c]);
}

// six components of a state array
template <typename RF, typename RC, int SUB>
__global__ void k_restrict(Transfer T, const RF *in, RC *out, int nc, int nb) {
  int k, sub, bb_;
  node_lanes<SUB>(nb, bb_, k, sub);
  if (k >= nc) return;
  double acc[6];
  restrict_sum<SUB, 6>(T, in + (size_t)bb_ * 6 * (size_t)T.nf, k, sub, acc);
  if (sub) return;
  out += (size_t)bb_ * 6 * (size_t)nc;
#pragma unroll
  for (int c = 0; c < 6; ++c) out[(size_t)c * nc + k] = RC(acc[c]);
}

// mapFineToCoarse of u, ready for the coarse level's smoothing step
template <typename RF, typename RC, int SUB>
__global__ void k_map_state(LevelDev<RC> K, DevParams P, Transfer T, const RF *fu, int ncopy) {
  int k, sub, bb_;
  node_lanes<SUB>(K.nb, bb_, k, sub);
  K.to_batch(bb_);
  P.to_batch(bb_);
  if (k >= K.n) return;
  double acc[6];
  restrict_sum<SUB, 6>(T, fu + (size_t)bb_ * 6 * (size_t)T.nf, k, sub, acc);
  if (sub) return;
  RC q[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    q[c] = RC(acc[c]);
    K.u[(size_t)c * K.n + k] = q[c];
  }
  begin_step(K, P, k, q, K.mu[k], ncopy, 0);
}

// start of restrictGrid (DEF:12158-12184): u and the laminar viscosity
// restricted, the boundary conditions on the restricted state (with its own
// pressure), which is also kept as the previous one; pressure and records
template <typename RF, typename RC, int SUB>
__global__ void k_restrict_state(LevelDev<RC> K, DevParams P, Transfer T, const RF *fu, const RF *fmu, int zero) {
  int k, sub, bb_;
  node_lanes<SUB>(K.nb, bb_, k, sub);
  K.to_batch(bb_);
  P.to_batch(bb_);
  if (k >= K.n) return;
  double acc[6], am[1];
  restrict_sum<SUB, 6>(T, fu + (size_t)bb_ * 6 * (size_t)T.nf, k, sub, acc);
  restrict_sum<SUB, 1>(T, fmu + (size_t)bb_ * (size_t)T.nf, k, sub, am);
  if (sub) return;
  RC q[6], mu = RC(am[0]);
#pragma unroll
  for (int c = 0; c < 6; ++c) q[c] = RC(acc[c]);
  K.mu[k] = mu;
  RC pp = state_pressure(P, q);
  const NodeBc<RC> b = node_bc(K, k);
  bc_solution(K, P, k, b, q, q[0]);
  outer_bc(P, b, q, pp);
#pragma unroll
  for (int c = 0; c < 6; ++c) K.u[(size_t)c * K.n + k] = q[c];
  begin_step(K, P, k, q, mu, 6, zero);
}

// end of restrictGrid (DEF:12362-12428): the fine increment restricted to
// rhs_H, BC'd as an increment, sourceTerm -= rhs_H, u_H += rhs_H; with
// `begin` also the start of the coarse level's smoothing step
template <typename RF, typename RC, int SUB>
__global__ void k_restrict_forcing(LevelDev<RC> K, DevParams P, Transfer T, const RF *frhs, int begin) {
  int k, sub, bb_;
  node_lanes<SUB>(K.nb, bb_, k, sub);
  K.to_batch(bb_);
  P.to_batch(bb_);
  if (k >= K.n) return;
  double acc[6];
  restrict_sum<SUB, 6>(T, frhs + (size_t)bb_ * 6 * (size_t)T.nf, k, sub, acc);
  if (sub) return;
  const size_t n = K.n;
  RC r[6], q[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) r[c] = RC(acc[c]);
  bc_increment(P, node_bc(K, k), r);
  const int nc = P.sa ? 6 : 5;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    K.rhs[c * n + k] = r[c];
    q[c] = K.u[c * n + k];
    if (c < nc) {
      K.src[c * n + k] -= r[c];
      q[c] += r[c];
      K.u[c * n + k] = q[c];
    }
  }
  if (begin) begin_step(K, P, k, q, K.mu[k], nc, 0);
}

// prolongateGrid (DEF:12432-12570): the coarse correction v_H = u_H -
// BC(R u_h), BC'd as an increment, then on the fine members: inject, relax,
// add, boundary conditions, clamps; with `begin` also the start of the fine
// level's smoothing step
template <typename RF, typename RC, int SUB>
__global__ void k_prolong(LevelDev<RF> F, LevelDev<RC> K, DevParams P, Transfer T, int ncomp_add, int begin, int zero) {
  int k, sub, bb_;
  node_lanes<SUB>(K.nb, bb_, k, sub);
  F.to_batch(bb_);
  K.to_batch(bb_);
  P.to_batch(bb_);
  if (k >= K.n) return;
  const size_t nc = K.n, n = F.n;
  double acc[6];
  restrict_sum<SUB, 6>(T, F.u, k, sub, acc);
  RC q[6], r[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) q[c] = RC(acc[c]);
  const NodeBc<RC> kb = node_bc(K, k);
  bc_solution(K, P, k, kb, q, K.u[k]);
  outer_bc(P, kb, q, K.p[k]);
#pragma unroll
  for (int c = 0; c < 6; ++c) r[c] = K.u[c * nc + k] - q[c];
  if (!P.sa) r[5] = 0;
  bc_increment(P, kb, r);
  if (sub == 0) {
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      K.uprev[c * nc + k] = q[c];
      K.rhs[c * nc + k] = r[c];
    }
  }
  for (int i = T.cptr[k] + sub; i < T.cptr[k + 1]; i += SUB) {
    RF d[6], v[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) d[c] = RF(r[c]);
#pragma unroll
    for (int c = 0; c < 5; ++c) d[c] = RF(P.prolong_relax) * d[c];
    d[5] = RF(P.turb_prolong_relax) * d[5];
    const NodeBc<RF> fb = node_bc(F, i);
    if (F.ncls[i] & NC_BFIRST)
#pragma unroll
      for (int c = 0; c < 5; ++c) d[c] = RF(P.mg_bc_relax) * d[c];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      F.rhs[c * n + i] = d[c];
      v[c] = F.u[c * n + i];
      if (c < ncomp_add) v[c] = v[c] + d[c];
    }
    bc_solution(F, P, i, fb, v, v[0]);
    outer_bc(P, fb, v, F.p[i]);
    if (P.sa) v[5] = v[5] > RF(0) ? v[5] : RF(0);
    v[0] = v[0] > RF(P.min_rho) ? v[0] : RF(P.min_rho);
#pragma unroll
    for (int c = 0; c < 6; ++c) F.u[c * n + i] = v[c];
    if (begin) begin_step(F, P, i, v, F.mu[i], P.sa ? 6 : 5, zero);
  }
}

// ---------------------------------------------------------------------------
// monitor reductions (writeResiduals MG:1302-1445, calculateLiftAndDrag
// DEF:14710-14806), all on the device: up to MON_BLOCKS blocks stride over
// the nodes and the wall nodes, each thread accumulating its share in stride
// order; wavefront butterflies and one LDS step reduce the block to a record
// of MON_REC doubles; k_monitor_final reduces the records.  The wall's terms
// are summed one after another in the register's order, a chunk of NTHR nodes
// a block, and without contraction: a wall of one chunk has the bits of the
// serial loop this stands for (the drag tests compare them with the oracle's),
// which a tree has for some states only.  The order of
// every sum is fixed, so the results are reproducible bit for bit.  Record:
// sum (u - uprev)^2 [7], max |u - uprev| [7], host index of that maximum [7]
// (smallest index on ties), force integrals [8] (lift, drag, latF,
// frictionDrag, latM, longM, pressureLift, pressureDrag, before the
// 2/referenceArea factor).
// ---------------------------------------------------------------------------
constexpr int MON_BLOCKS = 512;
constexpr int MON_REC = 29;

struct ForceFrame {
  double ft[3], fn1[3], fn2[3];  // flow tangent, lift and lateral normals
  double groundplane, datum[3];
};

// the integrand of calculateLiftAndDrag at wall node ip (DEF:14757-14803)
template <typename R>
__device__ __forceinline__ void force_terms(const LevelDev<R> &L, const DevParams &P, const ForceFrame &F, int ip,
                                            const R *warea, double *o) {
#pragma clang fp contract(off)
  for (int c = 0; c < 8; ++c) o[c] = 0;
  double z = L.xyz ? double(L.xyz[3 * (size_t)ip + 2]) : 0.0;
  if (!(z > F.groundplane + 0.01)) return;
  double x = L.xyz ? double(L.xyz[3 * (size_t)ip]) : 0.0;
  double y = L.xyz ? double(L.xyz[3 * (size_t)ip + 1]) : 0.0;
  double xc = x - F.datum[0], yc = y - F.datum[1], zc = z - F.datum[2];
  double nx = L.nrm[3 * (size_t)ip], ny = L.nrm[3 * (size_t)ip + 1], nz = L.nrm[3 * (size_t)ip + 2];
  double a = warea[ip];
  double pinf = 1.0 / (P.gamma * P.mach * P.mach);
  double dp = double(L.p[ip]) - pinf;
  double n1 = nx * F.fn1[0] + ny * F.fn1[1] + nz * F.fn1[2];
  double n2 = nx * F.fn2[0] + ny * F.fn2[1] + nz * F.fn2[2];
  double nt = nx * F.ft[0] + ny * F.ft[1] + nz * F.ft[2];
  double lift = -a * dp * n1, latF = -a * dp * n2, drag = -a * dp * nt;
  double latM = xc * a * dp * n2 - yc * a * dp * nt;
  double longM = xc * a * dp * n1 - zc * a * dp * nt;
  double fd = 0;
  if (P.Re > 0.0) {
    double w1 = L.ws[3 * (size_t)ip], w2 = L.ws[3 * (size_t)ip + 1], w3 = L.ws[3 * (size_t)ip + 2];
    double s1 = w1 * F.fn1[0] + w2 * F.fn1[1] + w3 * F.fn1[2];
    double s2 = w1 * F.fn2[0] + w2 * F.fn2[1] + w3 * F.fn2[2];
    double st = w1 * F.ft[0] + w2 * F.ft[1] + w3 * F.ft[2];
    lift += a * s1;
    latF += a * s2;
    drag += a * st;
    fd = a * st;
    latM += -xc * a * s2 + yc * a * st;
    longM += -xc * a * s1 + zc * a * st;
  }
  o[0] = lift;
  o[1] = drag;
  o[2] = latF;
  o[3] = fd;
  o[4] = latM;
  o[5] = longM;
  o[6] = -double(L.p[ip]) * (a - pinf) * n1;
  o[7] = -double(L.p[ip]) * (a - pinf) * nt;
}

// max |d| with the smallest index among equal values
__device__ __forceinline__ void maxloc(double &m, int &k, double m2, int k2) {
  if (m2 > m || (m2 == m && k2 < k)) {
    m = m2;
    k = k2;
  }
}

// one wavefront's sum and (max, smallest index) by xor butterflies: every
// lane ends with the same bits
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v += __shfl_xor(v, m, 64);
  return v;
}
__device__ __forceinline__ void wave_maxloc(double &m, int &k) {
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) maxloc(m, k, __shfl_xor(m, s, 64), __shfl_xor(k, s, 64));
}

// Every block reduces its share to a record (block b's quantity q at
// part[MON_BLOCKS q + b]); k_monitor_final reduces the records, each quantity
// by one wavefront, to MON_REC doubles in host memory the device can write.
// Launches this small are latency alone, so the quantities share one barrier.
// (One launch whose last block reduces the records needs a device-wide fence
// in every block, which writes back its XCD's L2: it took 18 us on 9k nodes
// and 57 on 275k, where the two launches take 16 and 27.)
template <typename R>
__global__ __launch_bounds__(NTHR) void k_monitor_reduce(LevelDev<R> L, DevParams P, ForceFrame F, int nres,
                                                         const int *host_index, const int *wall_nodes, int nw,
                                                         const R *warea, double *part, int bsel) {
  L.to_batch(bsel);
  P.to_batch(bsel);
  constexpr int NW = NTHR / 64, FIRST_FORCE = 21;
  __shared__ double lds[FIRST_FORCE][NW];
  __shared__ double terms[8][NTHR + 1];  // odd stride: the eight summing lanes read different banks
  const int n = L.n, stride = gridDim.x * NTHR;
  double sum[7], mx[7];
  int mi[7];
#pragma unroll
  for (int j = 0; j < 7; ++j) {
    sum[j] = 0;
    mx[j] = 0;
    mi[j] = 0x7fffffff;
  }
  for (int i = blockIdx.x * NTHR + threadIdx.x; i < n; i += stride) {
    const int hi = host_index[i];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      if (j >= nres) break;
      double d = double(L.u[(size_t)j * n + i]) - double(L.uprev[(size_t)j * n + i]);
      sum[j] += d * d;
      maxloc(mx[j], mi[j], fabs(d), hi);
    }
  }
  // force integrals: quantity q's sum on thread q
  const int q = threadIdx.x;
  const bool force = q >= FIRST_FORCE && q < MON_REC;
  double v = 0;
  for (int k0 = blockIdx.x * NTHR; k0 < nw; k0 += stride) {
    const int cnt = nw - k0 < NTHR ? nw - k0 : NTHR;
    if (q < cnt) {
      double o[8];
      force_terms(L, P, F, wall_nodes[k0 + q], warea, o);
#pragma unroll
      for (int c = 0; c < 8; ++c) terms[c][q] = o[c];
    }
    __syncthreads();
    if (force)
      for (int k = 0; k < cnt; ++k) v += terms[q - FIRST_FORCE][k];
    __syncthreads();
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < 7; ++j) {
    const double t = wave_sum(sum[j]);
    wave_maxloc(mx[j], mi[j]);
    if (lane == 0) {
      lds[j][wave] = t;
      lds[7 + j][wave] = mx[j];
      lds[14 + j][wave] = double(mi[j]);
    }
  }
  __syncthreads();
  if (q >= 7 && q < FIRST_FORCE) {  // the maxima, and the indices that go with them
    const int j = q < 14 ? q : q - 7;
    double m = lds[j][0];
    int k = (int)lds[j + 7][0];
    for (int w = 1; w < NW; ++w) maxloc(m, k, lds[j][w], (int)lds[j + 7][w]);
    v = q < 14 ? m : double(k);
  } else if (q < 7) {
    for (int w = 0; w < NW; ++w) v += lds[q][w];
  }
  if (q < MON_REC) part[(size_t)MON_BLOCKS * q + blockIdx.x] = v;
}

// wavefront w of one block takes quantities w, w + FIN_NW, ..; all of a
// stride's records are requested before the first is used
constexpr int FIN_THR = 512, FIN_NW = FIN_THR / 64;
__global__ __launch_bounds__(FIN_THR) void k_monitor_final(const double *part, int nrec, double *out) {
  constexpr int PER = (MON_REC + FIN_NW - 1) / FIN_NW;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double v[PER];
  int kx[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    v[p] = 0;
    kx[p] = 0x7fffffff;
  }
  for (int b = lane; b < nrec; b += 64) {
    double x[PER], y[PER];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int r = wave + p * FIN_NW;
      x[p] = r < MON_REC ? part[(size_t)MON_BLOCKS * r + b] : 0.0;
      y[p] = r >= 7 && r < 14 ? part[(size_t)MON_BLOCKS * (r + 7) + b] : 0.0;
    }
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int r = wave + p * FIN_NW;
      if (r >= 7 && r < 14) maxloc(v[p], kx[p], x[p], (int)y[p]);
      else v[p] += x[p];
    }
  }
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int r = wave + p * FIN_NW;
    if (r >= 7 && r < 14) wave_maxloc(v[p], kx[p]);
    else v[p] = wave_sum(v[p]);
    if (lane == 0 && r < MON_REC && !(r >= 14 && r < 21)) {
      out[r] = v[p];
      if (r >= 7 && r < 14) out[r + 7] = double(kx[p]);
    }
  }
}

}  // namespace fk
