// mose_kernels.hpp — device data structures and kernels of the explicit step (gfx950).
//
// Memory layout in HBM
//   * Cell pool: the padded cells (gc = 2 ghost layers) of every block concatenated,
//     i fastest.  Conserved state is SoA over the pool: U[v * npool + cell], v = rho, rho u,
//     rho v, rho w, rho E, FP64.  Three state buffers: U^n, and two stage buffers.
//   * Geometry of rectilinear blocks: per block and direction a line of `LineEnt`
//     (cell length dl as the reference computes it, node spacing, reconstruction spacings
//     of the face on the cell's low side).  Normals are the axis unit vectors.
//   * Geometry of curvilinear blocks (any block not rectilinear switches the context to it):
//     per pool cell, SoA over the pool, NGEO FP64 arrays: the unit normal and area of the
//     cell's low face in each direction, the cell lengths dl, the volume, the unit rows of
//     the inverse Jacobian (CFL time step) and the reciprocal distance to the low neighbour's
//     centre (reconstruction), all from the reference's metric definitions.
//   * Work: a list of tiles (block, i0, j0, k-range).  Each workgroup of TX x TY threads
//     owns a TX x TY column patch and marches along k; the current k-plane's primitive
//     state with a 2-cell i/j halo is staged in LDS, the k-direction stencil of each column
//     lives in registers.  Every face flux is evaluated once.
#pragma once
#include "mose_device.hpp"

namespace mose {


// Ghost-op kinds.
enum { G_COPY = 0, G_ZG = 1, G_EXTRAP = 2, G_SYM = 3 };
// Face BC kinds used inside the stage kernel (bctype of a block face).
enum { F_CONN = 0, F_NONE = 1, F_EXTRAP = 2, F_SYM = 3, F_INFLOW = 4, F_INLET = 5, F_OUTFLOW = 6 };
// Scalars kept on the device.
enum { S_DT = 0, S_TIME = 1, S_NORM = 2, S_COUNT = 8 };
// Curvilinear geometry arrays (index g: array g * npool + cell).
//   GN + 4d + {0,1,2}: unit normal of the low face in direction d, GN + 4d + 3: its area;
//   GDL + d: dl; GVOL: volume; GVS + 3d + {0,1,2}: M(d,:)/|M(d,:)|; GRLO + d: 2/(dl(c-e_d)+dl(c)).
enum { GN = 0, GDL = 12, GVOL = 15, GVS = 16, GRLO = 25, NGEO = 28 };

struct LineEnt {
  double dl;      // cell length along the line (Compute_Metric_Tensor dl)
  double delta;   // node spacing x_i - x_{i-1} (face areas / volume)
  double rl0, rl1, rl2, lm, lp;   // spacing of the face between cells i-1 and i
  double rdl;     // 1 / dl (the diagonal metric of the viscous terms)
};

// Read-only data through the constant address space: loads from a wave-uniform address
// become scalar loads (s_load, scalar data cache) instead of vector loads into VGPRs.  Only
// for arrays no kernel writes while the loading kernel runs.
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;

struct BlockDev {
  int64_t off;       // pool index of padded cell (-1,-1,-1)
  int64_t sz;        // plane stride (ni+4)(nj+4)
  int ni, nj, nk, sy;
  int line[3];       // LineEnt index of padded position 0 (cell -1) per direction
  int bct[6];        // F_* per face
  int bcd[6];        // index of the 8-double data record (inflow), or -1
  int bcs[6];        // first slot of the face in the boundary-flux buffer, or -1
  int bvs[6];        // first slot of a connection face in the viscous-flux buffer, or -1
  int visc, pad_;    // laminar viscous terms on
  double vis[5];     // mu_ref, T_ref, S (Sutherland), cp / Pr, vnn
};

// One boundary face cell of a block connection when viscous terms are on: the stencil of
// BC_Connection_Visc (boundary cell, its ghost, the tangential neighbours of both sides).
struct ViscFace {
  int64_t loc, gh;     // pool index of the boundary cell and of its first ghost cell
  int64_t tn[4];       // boundary cell's neighbours: 1st tangential -, +, 2nd tangential -, +
  int64_t dn[4];       // the donor cell's neighbours in the same order (Pg(:,3:6))
  int b, d, slot, modfm2;
  double area;
  double ml[3], mg[3]; // diagonal metric (1/dl) of the boundary and ghost cells
};

// One boundary face cell of a non-connection face (flux computed by k_bcface).
struct BcFace {
  int64_t cb, cn;    // pool index of the boundary cell and of its interior neighbour
  int b, f;          // block (0-based), face (0..5)
  int slot, pad;     // output slot in the boundary-flux buffer
  double bdl, idl;   // half lengths of the two cells along the face normal
  double n[3];       // unit normal of the boundary face (increasing-index orientation)
  double area;       // face area
  double t[3];       // unit face diagonal (t_Vec of Setup_Inflow_Geometry, subsonic inlets)
};

struct Tile {
  int b, i0, j0, k0, k1, pad0, pad1, pad2;
};

// Largest patch (TX x TY threads) of any tile shape.  Every kernel launched with one thread
// per patch column (the stage kernels and k_dt, k_sd, k_prim_resid, k_irs_jacobi,
// k_irs_update) declares a launch bound of at least this, and the host refuses a shape above
// it (a launch with more threads than a kernel's bound fails).
constexpr int kMaxTileThreads = 512;

struct GhostOp {
  int64_t b;         // boundary cell (pool index)
  int64_t s;         // inward pool stride
  int64_t src1, src2;
  int type, pad;
  double n[3];
  // Archive slots of the op's second and third reads (copy: src1 / src2; extrapolation:
  // b + s / b + 2s), or -1: a read of a ghost cell that a later record of the same fill
  // writes takes that cell's value from the previous fill, as the reference's serial fill
  // does (blocks one or two cells thick).
  int a1, a2;
};

struct StageArgs {
  const double* __restrict__ Uin;
  const double* __restrict__ Un;
  double* __restrict__ Uout;
  double* __restrict__ Rout;
  const Tile* __restrict__ tiles;
  const BlockDev* __restrict__ blocks;
  const LineEnt* __restrict__ lines;
  const double* __restrict__ facebc;
  const double* __restrict__ geo;      // curvilinear geometry arrays (NGEO x npool) or null
  const double* __restrict__ scal;
  const double* dtloc;          // local time stepping: dt of each cell (same array as dtnext)
  double* __restrict__ partials;
  double* __restrict__ bcbuf;
  double* __restrict__ vbuf;    // viscous flux of connection faces (per unit area), viscous path
  const double* __restrict__ beta;   // shock-detector weight per pool cell (HLLE++ / HLLC+ / MUSCL-SD)
  int* err;
  unsigned long long* dtmin;   // last stage: CFL time step of the next step (min as bits)
  double* dtnext;              // last stage, local time stepping: dtlocal of the next step
  const int* iter;
  int* tq;                     // tile queues of the persistent stage launch (kTileQueues claim
                               // counters and a finished-workgroup counter), zero between launches
  int64_t npool;
  int ntiles;
  int nq;                      // queues in use: kTileQueues with the XCD-aware tile order, else 1
  int local_dt;
  int ndir, rampa;
  int irs_scale;               // MODE 2: write R* = -R dt / vol (residual smoothing) instead of R
  double rkc, gam, R, cfl;
};

// Persistent stage launch: the grid is the number of workgroups resident on the device (never
// more than there are tiles) and each workgroup takes tiles until none is left.  Queue x (x < nq)
// holds the tile positions x, x + nq, x + 2 nq, ...: with the XCD-aware order those are the tiles
// of one contiguous range of blocks, and workgroup w (dispatched to XCD w mod 8) works on queue
// w mod nq, so neighbouring tiles share an L2.  Workgroup w's first tile is position w, without a
// claim; the counters hold what was claimed beyond those.  The next tile is claimed with one
// atomicAdd, and a workgroup whose queue is empty looks at all other counters at once, one lane each
// (claim_other): a workgroup that read them one after the other spent 5 us at the end of every
// launch (a 1000-cell stage 15.0 us, now 10.2 us).  A launch with a workgroup for every tile makes
// no claims at all.  Every claim is one atomicAdd, so each tile is taken exactly once; the last
// workgroup to finish sets the counters back to zero for the next launch.
constexpr int kTileQueues = 8;

// tiles of queue x, and those of them that are the first tiles of workgroups
__device__ __forceinline__ int queue_len(int x, int nq, int n) { return (n - x + nq - 1) / nq; }

// A tile of the workgroup's own queue (one thread), or -1 when it is empty.
__device__ __forceinline__ int claim_own(int* tq, int nq, int ntiles) {
  const int x = (int)(blockIdx.x % (unsigned)nq);
  const int at = atomicAdd(tq + x, 1) + queue_len(x, nq, (int)gridDim.x);
  return at < queue_len(x, nq, ntiles) ? x + at * nq : -1;
}
// A tile of another queue (called by one whole wave), or -1 when all are empty.
__device__ __forceinline__ int claim_other(int* tq, int nq, int ntiles) {
  const int lane = (int)(threadIdx.x & 63);
  const int x = (int)((blockIdx.x + (unsigned)lane) % (unsigned)nq);
  const int first = queue_len(x, nq, (int)gridDim.x), len = queue_len(x, nq, ntiles);
  for (;;) {
    bool some = false;
    if (lane > 0 && lane < nq)
      some = __hip_atomic_load(tq + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + first < len;
    const unsigned long long m = __ballot(some);
    if (m == 0) return -1;
    const int s = __ffsll((unsigned long long)m) - 1;
    int t = -1;
    if (lane == s) {
      const int at = atomicAdd(tq + x, 1) + first;
      if (at < len) t = x + at * nq;
    }
    t = __shfl(t, s, 64);
    if (t >= 0) return t;      // else that queue has just become empty: look again
  }
}

// End of a workgroup's persistent loop (thread 0): the last workgroup resets the queues.
__device__ __forceinline__ void finish_tiles(int* tq) {
  if (atomicAdd(tq + kTileQueues, 1) == (int)gridDim.x - 1) {
    for (int x = 0; x <= kTileQueues; ++x) atomicExch(tq + x, 0);
  }
}

// Workgroup barrier ordering LDS accesses only.  __syncthreads() also orders global memory,
// which makes every wave wait for all of its outstanding global loads before the barrier;
// kernels whose threads exchange data only through LDS use this one, so that loads issued
// ahead of time (the next plane's cells) stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// First error of a launch wins (code, block, i, j, k); later ones are dropped.
__device__ __forceinline__ void set_error(int* err, int code, int b, int i, int j, int k) {
  if (atomicCAS(err, 0, code) == 0) {
    err[1] = b; err[2] = i; err[3] = j; err[4] = k;
  }
}

// Ghost layers (Fill_Ghost_Cell, Lib_Ghost.f90:11-137) on the conserved SoA state.
// Copies (101/201 Ghost_Connection, zero-gradient) move conserved values, which equal the
// primitive copies of the reference exactly; extrapolation (Ghost_Extrapolate) and the
// symmetry mirror (Ghost_Symmetry) act on primitive variables as in the reference.
// The records of one phase are independent: a record that reads a ghost cell written by an
// earlier record is in a later phase, and one that reads a ghost cell written by a later record
// reads it from arc, the values at the end of the previous fill (narc cells).
//
// The device's record: pool cells as 32-bit indexes (npool is below 2^31 / 5) and the mirror
// normal in an array of its own, 32 bytes in place of 80 -- the fill reads a record for the ten to
// twenty values it moves (256^3 periodic block, 393,216 records: fills one after the other 29.8 us, now
// 26.3 us; between the stages of a march 38 us).
struct GhostRec {
  int b, s;            // boundary cell, inward stride
  int src1, src2;
  int type;
  int a1, a2;          // archive slots of the second and third reads (GhostOp), or -1
  int nrm;             // G_SYM: index of the mirror normal
};
static_assert(sizeof(GhostRec) == 32, "two 16-byte loads");

struct GhostArgs {
  const GhostRec* __restrict__ ops;
  const double* __restrict__ nrm;     // 3 per G_SYM record
  double* U;
  double* arc;
  const int* save;             // 2 per record: archive slots of the two ghost cells it writes (-1: none); null
                               // where the archive has a pass of its own, or there is none
  int64_t N, narc;
  double gam;
  int nops;
  int nblk;                    // workgroups that fill ghosts (k_bcface; the others solve boundary faces)
  // start of a step (null: none), taken by the first thread of its first launch
  unsigned long long* dtmin;
  int* iter;
  double* scal;
  int time_accurate;
};

// Start of a step: iter += 1, take the CFL time step computed from the current state (by
// the previous step's last stage or by k_dt), time += dt when time-accurate, and reset the
// accumulator (dtglobal = 1e5, Mod_Explicit.f90:36-49) for this step's last stage.
__device__ __forceinline__ void begin_step(const GhostArgs& g) {
  *g.iter += 1;
  const double dt = __longlong_as_double((long long)*g.dtmin);
  g.scal[S_DT] = dt;
  if (g.time_accurate) g.scal[S_TIME] += dt;
  *g.dtmin = (unsigned long long)__double_as_longlong(1e5);
}

// prim2cons with the contraction of the energy written out, so that every copy of the fill gives the
// same bits (FP32-flux layouts turn a ghost cell one FP64 ulp away into another FP32 value now and
// then, which marches on to 1e-6 of the state).
__device__ __forceinline__ void ghost_cons(const double* P, double rgm1, double* U) {
  U[0] = P[0]; U[1] = P[0] * P[1]; U[2] = P[0] * P[2]; U[3] = P[0] * P[3];
  U[4] = __builtin_fma(rgm1, P[4], 0.5 * P[0] * (P[1] * P[1] + P[2] * P[2] + P[3] * P[3]));
}

// The ops q0, q0 + step, ... of one phase.
__device__ __forceinline__ void ghost_ops(const GhostArgs& g, int q0, int step) {
  if (q0 == 0 && g.dtmin) begin_step(g);
  const double gm1 = g.gam - 1.0, rgm1 = 1.0 / gm1;
  double* const U = g.U;
  double* const arc = g.arc;
  const int64_t N = g.N, narc = g.narc;
  for (int q = q0; q < g.nops; q += step) {
    const GhostRec op = g.ops[q];
    const int64_t d1 = op.b - op.s, d2 = op.b - 2 * (int64_t)op.s;
    auto rd = [&](int v, int64_t cell, int slot) { return slot >= 0 ? arc[v * narc + slot] : U[v * N + cell]; };
    const int s1 = g.save ? g.save[2 * q] : -1, s2 = g.save ? g.save[2 * q + 1] : -1;
    auto w1 = [&](int v, double x) { U[v * N + d1] = x; if (s1 >= 0) arc[v * narc + s1] = x; };
    auto w2 = [&](int v, double x) { U[v * N + d2] = x; if (s2 >= 0) arc[v * narc + s2] = x; };
    if (op.type == G_COPY) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double a1 = rd(v, op.src1, op.a1), a2 = rd(v, op.src2, op.a2);
        w1(v, a1);
        w2(v, a2);
      }
    } else if (op.type == G_ZG) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double x = U[v * N + op.b];
        w1(v, x);
        w2(v, x);
      }
    } else if (op.type == G_EXTRAP) {
      double u[5], Pb[5], P1[5], P2[5], G1[5], G2[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) u[v] = U[v * N + op.b];
      cons2prim(u, gm1, Pb);
#pragma unroll
      for (int v = 0; v < 5; ++v) u[v] = rd(v, op.b + op.s, op.a1);
      cons2prim(u, gm1, P1);
#pragma unroll
      for (int v = 0; v < 5; ++v) u[v] = rd(v, op.b + 2 * (int64_t)op.s, op.a2);
      cons2prim(u, gm1, P2);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        G1[v] = 3.0 * Pb[v] - 3.0 * P1[v] + P2[v];
        G2[v] = 3.0 * G1[v] - 3.0 * Pb[v] + P1[v];
      }
      ghost_cons(G1, rgm1, u);
#pragma unroll
      for (int v = 0; v < 5; ++v) w1(v, u[v]);
      ghost_cons(G2, rgm1, u);
#pragma unroll
      for (int v = 0; v < 5; ++v) w2(v, u[v]);
    } else {   // G_SYM: first layer only
      double u[5], P[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) u[v] = U[v * N + op.b];
      cons2prim(u, gm1, P);
      const double* n = g.nrm + 3 * (int64_t)op.nrm;
      const double un = P[1] * n[0] + P[2] * n[1] + P[3] * n[2];
      P[1] -= 2.0 * un * n[0];
      P[2] -= 2.0 * un * n[1];
      P[3] -= 2.0 * un * n[2];
      ghost_cons(P, rgm1, u);
#pragma unroll
      for (int v = 0; v < 5; ++v) w1(v, u[v]);
    }
  }
}

}  // namespace mose
