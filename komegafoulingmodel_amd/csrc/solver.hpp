// solver.hpp -- the implicit solves of the step: right-preconditioned
// BiCGStab (van der Vorst 1992) on five-point systems with diagonal 1.
//
// The assembled rows of k and omega are not diagonally dominant next to curved
// walls, so a stationary iteration can diverge; the reference uses restarted
// GMRES (GMRESSolver.cpp:227-355) for them and BiCGStab for the temperature
// (BiCGStabSolver.cpp).  Every system is solved on its own here: k and omega
// are two systems of one launch (grid.y), the temperature one.
//
// An iteration is three streaming passes and nothing else:
//   PV  p' = r + beta (p - omega v),  v' = A M^-1 p'     sums (rh, v')
//   ST  s = r - alpha v',  t = A M^-1 s                   sums (t, s), (t, t)
//   XR  x += alpha M^-1 p' + omega M^-1 s,  r' = s - omega t   sums (rh, r'), (r', r')
// A pass begins by adding up the previous pass's per-block sums and forming
// the scalars from them, in every block (at most about 512 pairs, from L2); one
// block writes the new solver state for the next pass.  State and sums are
// double buffered by pass parity, so no pass reads what another block of it
// writes.  A separate one-block kernel for the scalars costs about 5 us in
// the chain, as much as a whole pass on lattices of a few hundred thousand nodes.
// (A reduction finished inside the pass would need agent-scope release
// fences, which write back the L2 and cost more than a launch.)
//
// Bytes: the passes are bound by HBM on large lattices.  rh and the first p
// are the first residual itself, so r is never overwritten in its first buffer
// (later residuals alternate between two others) and the first iteration,
// which is the only one for most steady steps, moves 6 + 7 + 6 planes instead
// of 10 + 8 + 7; s is recomputed in XR.
#pragma once
#include "kernels.hpp"

namespace kofm {
namespace dev {

// Solver state of one system between passes.
struct SolveState {
  double rho, rhoNew, alpha, omega, beta;
  double r0, rn;
  double best;     // smallest residual so far
  double bnorm;    // ||b|| (stopping rule 1)
  double prevRes;  // the previous iteration's residual (stopping rule 1)
  int done, iters, restart;
  int sinceBest;   // iterations since the residual last fell below 0.999 best
  int nan;
};

// A solve whose residual has not fallen below 0.999 of its best for this
// many iterations has reached the rounding floor of FP64 and stops: past
// that point the recursively updated residual no longer follows b - A x,
// and further iterations move x without improving it.
constexpr int kBicgStagnation = 50;

// How the blocks of a pass cover the lattice: strips of kStripX columns cut
// into chunks of `rows` rows.  A block walks its chunk upwards four rows at a
// time, so that the loads of four rows are in flight together, the values above
// and below a node stay in its own lane's registers, and only the two
// horizontal neighbours are exchanged (through LDS).  Chunks are as tall as
// leaves about 256 blocks per system (two systems then give each CU two blocks
// of five waves): twice as many cost 5 to 20 % on lattices of 0.1 to 0.4
// million nodes, where a block's fixed work (adding up all blocks' sums, the
// rows beside the chunk) counts, and are no faster on 2 million.  The rows
// beside a chunk are mostly L2 hits: neighbouring chunks run on one XCD.
constexpr int kStripBlocks = 256;
constexpr int kStripX = 256;
constexpr int kStripThreads = kStripX + 64;  // and a wave for the columns beside the strip
constexpr int kRows = 4;  // rows a pass takes at a time
struct Strips {
  int strips, chunks, rows, nblk, per;
};
inline Strips stripsFor(int nX, int nY) {
  Strips s;
  s.strips = (nX + kStripX - 1) / kStripX;
  const int want = (nY * s.strips + kStripBlocks - 1) / kStripBlocks;
  s.rows = (want + kRows - 1) / kRows * kRows;
  s.chunks = (nY + s.rows - 1) / s.rows;
  s.nblk = s.strips * s.chunks;
  s.per = (s.nblk + 7) / 8;
  return s;
}

// One system.  Vectors are FP64 for every storage form: the omega field spans
// about seven decades (wall rows near 1000, core values near 1e-4) and FP32
// Krylov vectors cannot resolve the core next to the wall.  The vectors read
// zero on solid nodes, which no pass writes.
struct SolveSys {
  const uint16_t* mask;
  double* x;        // the iterate, in place
  const double* A;  // 4 planes: E, W, N, S
  double* r[3];     // r[0]: the first residual (= rh and the first p); then r[1], r[2] in turn
  double* p[2];
  double* v[2];
  double* t;
  SolveState* st;   // [2]
  double2* partial;  // [2][2 * nblk]
  SolveState* out;  // the state the last finish kernel saw
  double rtol, atol;
  int maxit;
  int crit;         // stopping rule: 0 as GMRESSolver, 1 as BiCGStabSolver
  int nX, nY, XF;
  int64_t D;
  Strips s;
};
struct SolvePair {
  SolveSys sys[2];
};

// This block's chunk: columns [x0, x0 + w), rows [y0, y1); false past the end.
struct Chunk {
  int T, x0, w, y0, y1;
};
__device__ __forceinline__ bool chunkOf(const Strips& s, int nX, int nY, Chunk& c) {
  c.T = int(blockIdx.x & 7) * s.per + int(blockIdx.x >> 3);  // a run of chunks per XCD
  if (int(blockIdx.x >> 3) >= s.per || c.T >= s.nblk) return false;
  const int strip = c.T / s.chunks, chunk = c.T - strip * s.chunks;
  c.x0 = strip * kStripX;
  c.w = min(kStripX, nX - c.x0);
  c.y0 = chunk * s.rows;
  c.y1 = min(c.y0 + s.rows, nY);
  return true;
}

// A sum carried with its rounding error (Knuth's two-sum): the passes' dot
// products then do not depend on how the lattice is cut into blocks, which
// ill-conditioned rows (fouled walls) would otherwise feel from the third
// iteration on.  The passes wait for memory; the extra additions are free.
struct Sum {
  double hi, lo;
  __device__ __forceinline__ void add(double x) {
    const double s = hi + x, z = s - hi;
    lo += (hi - (s - z)) + (x - z);
    hi = s;
  }
  __device__ __forceinline__ void add(const Sum& o) {
    add(o.hi);
    lo += o.lo;
  }
  __device__ __forceinline__ double value() const { return hi + lo; }
};

// One step of a sum over the wave: adds the value DPP moves here (0 where it
// moves none).
template <int CTRL, int ROWS>
__device__ __forceinline__ void waveStep(Sum& a) {
  auto mv = [](double d) {
    const uint64_t u = __builtin_bit_cast(uint64_t, d);
    const uint32_t lo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(u)), CTRL, ROWS, 0xf, true));
    const uint32_t hi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(u >> 32)), CTRL, ROWS, 0xf, true));
    return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
  };
  const Sum o{mv(a.hi), mv(a.lo)};
  a.add(o);
}
// The wave's sum, in lane 63: running sums over each row of 16 lanes, then
// each row's last lane into the row above it, then the lower half's into the
// upper.  (DPP moves cost a few cycles where a shuffle through LDS costs 60.)
__device__ __forceinline__ void waveSum(Sum& a) {
  waveStep<0x111, 0xf>(a);  // row_shr 1, 2, 4, 8
  waveStep<0x112, 0xf>(a);
  waveStep<0x114, 0xf>(a);
  waveStep<0x118, 0xf>(a);
  waveStep<0x142, 0xa>(a);  // row_bcast 15
  waveStep<0x143, 0xc>(a);  // row_bcast 31
}

// a and b summed over the block (every lane gets them).
template <int THREADS>
__device__ __forceinline__ void blockSum2(Sum& a, Sum& b) {
  __shared__ Sum red[2][THREADS / 64];
  waveSum(a);
  waveSum(b);
  if ((threadIdx.x & 63) == 63) {
    red[0][threadIdx.x >> 6] = a;
    red[1][threadIdx.x >> 6] = b;
  }
  __syncthreads();
  a = red[0][0];
  b = red[1][0];
#pragma unroll
  for (int w = 1; w < THREADS / 64; w++) {
    a.add(red[0][w]);
    b.add(red[1][w]);
  }
  __syncthreads();
}

// A block's sums to (and all blocks' sums from) the partials of pass parity
// `slot`: {a.hi, a.lo}, {b.hi, b.lo} per block.
template <int THREADS>
__device__ __forceinline__ void writePartial(const SolveSys& y, int T, int slot, Sum a, Sum b) {
  blockSum2<THREADS>(a, b);
  if (threadIdx.x == 0) {
    double2* out = y.partial + size_t(slot) * 2 * y.s.nblk + 2 * T;
    out[0] = make_double2(a.hi, a.lo);
    out[1] = make_double2(b.hi, b.lo);
  }
}
// In two parts, so that a pass can issue its own first loads in between: a
// wave's loads return in order, and the sums must not wait behind the rows.
template <int THREADS>
struct Partials {
  static constexpr int kAhead = 1;
  double2 a[kAhead], b[kAhead];
  __device__ __forceinline__ void load(const SolveSys& y, int slot) {
    const double2* in = y.partial + size_t(slot) * 2 * y.s.nblk;
#pragma unroll
    for (int k = 0; k < kAhead; k++) {
      const int i = int(threadIdx.x) + k * THREADS;
      a[k] = b[k] = make_double2(0., 0.);
      if (i < y.s.nblk) {
        a[k] = in[2 * i];
        b[k] = in[2 * i + 1];
      }
    }
  }
  __device__ __forceinline__ void sums(const SolveSys& y, int slot, double& outA, double& outB) const {
    const double2* in = y.partial + size_t(slot) * 2 * y.s.nblk;
    Sum p{}, q{};
#pragma unroll
    for (int k = 0; k < kAhead; k++) {
      p.add(a[k].x);
      p.lo += a[k].y;
      q.add(b[k].x);
      q.lo += b[k].y;
    }
    for (int i = int(threadIdx.x) + kAhead * THREADS; i < y.s.nblk; i += THREADS) {
      const double2 u = in[2 * i], v = in[2 * i + 1];
      p.add(u.x);
      p.lo += u.y;
      q.add(v.x);
      q.lo += v.y;
    }
    blockSum2<THREADS>(p, q);
    outA = p.value();
    outB = q.value();
  }
};

// The state after the pass whose sums are a, b.  stage 0: the first residual,
// 1: PV, 2: ST, 3: XR.
__device__ __forceinline__ void advance(SolveState& s, int stage, double a, double b,
                                        const SolveSys& y) {
  if (stage == 0) {
    // a = (r, r), b = (b, b) (rule 1); the first PV takes p = rh = r
    s = SolveState{};
    const double r0 = sqrt(a);
    s.r0 = s.rn = s.best = s.prevRes = r0;
    s.rho = s.alpha = s.omega = 1.;
    s.rhoNew = s.beta = a;
    s.restart = 1;
    if (y.crit == 1) {
      // BiCGStabSolver::solve (BiCGStabSolver.cpp:648-658): ||b|| <= 1e-16
      // ends the solve (the kernel leaves x; the reference copies b, the
      // same zero field up to 1e-16)
      const double bn = sqrt(b);
      s.bnorm = bn;
      if (!isfinite(r0) || !isfinite(bn))
        s.nan = s.done = 1;
      else if (bn <= 1.0e-16 || r0 == 0. || r0 <= y.rtol * bn)
        s.done = 1;
    } else if (!isfinite(r0)) {
      s.nan = s.done = 1;
    } else if (r0 == 0. || r0 <= y.atol) {
      s.done = 1;
    }
  } else if (stage == 1) {
    // a = (rh, v); a restart requested by the last stage 3 has now been
    // consumed by PV
    s.restart = 0;
    if (a == 0. || !isfinite(a)) {
      s.alpha = 0.;
      s.restart = 1;
    } else {
      s.alpha = s.rhoNew / a;
    }
  } else if (stage == 2) {
    // a = (t, s), b = (t, t)
    s.omega = (b > 0. && isfinite(b)) ? a / b : 0.;
  } else {
    // a = (rh, r), b = (r, r)
    const double rn = sqrt(b);
    s.iters += 1;
    s.rn = rn;
    if (!isfinite(rn)) {
      s.nan = s.done = 1;
      return;
    }
    if (y.crit == 1) {
      // BiCGStabSolver::reduceAndCheckConvergence (BiCGStabSolver.cpp:509-545):
      // a residual above 10 times the last one after the first iteration
      // fails like a non-finite one (the caller halves the time step);
      // converged at ||r|| <= rtol ||b|| or ||r|| <= atol ||r0||
      if (s.iters > 1 && rn > 10. * s.prevRes) {
        s.nan = s.done = 1;
        return;
      }
      s.prevRes = rn;
      if (rn <= y.rtol * s.bnorm || rn <= y.atol * s.r0 || s.iters >= y.maxit) {
        s.done = 1;
        return;
      }
    } else if (rn <= y.rtol * s.r0 || rn <= y.atol || s.iters >= y.maxit) {
      s.done = 1;
      return;
    }
    if (rn < 0.999 * s.best) {
      s.best = rn;
      s.sinceBest = 0;
    } else if (++s.sinceBest >= kBicgStagnation) {
      s.done = 1;
      return;
    }
    s.rho = s.rhoNew;
    s.rhoNew = a;
    if (a == 0. || s.omega == 0. || s.restart) {
      // breakdown or stagnation: restart with rh = r, p = v = 0
      s.restart = 1;
      s.rho = s.alpha = s.omega = 1.;
      s.rhoNew = s.beta = b;
    } else {
      s.beta = (a / s.rho) * (s.alpha / s.omega);
    }
  }
}

// True for a system that finished in an earlier pass: its state is passed on
// (pass parity par: a pass reads slot par and writes slot par ^ 1).
__device__ __forceinline__ bool passedOn(const SolveSys& y, int stage, int par, bool lead) {
  if (stage == 0 || !y.st[par].done) return false;
  if (lead && threadIdx.x == 0) y.st[par ^ 1] = y.st[par];
  return true;
}

// Start of a pass: the state with the previous pass's sums taken in.  False
// when that finishes the system.
template <int THREADS>
__device__ __forceinline__ bool beginPass(const SolveSys& y, const Partials<THREADS>& in, int stage,
                                          int par, bool lead, SolveState& s) {
  __shared__ SolveState sh;
  double a, b;
  in.sums(y, par, a, b);
  if (threadIdx.x == 0) {
    SolveState n{};
    if (stage != 0) n = y.st[par];
    advance(n, stage, a, b, y);
    sh = n;
    if (lead) y.st[par ^ 1] = n;
  }
  __syncthreads();
  s = sh;
  return s.done == 0;
}

// (M^-1 u)_i for u given by a function of the node index: with partner q,
// (u_i - a_iq u_q) / (1 - a_iq a_qi), the couplings taken from the rows in
// A (for a transposed system A holds the transposed rows, so this is M^T).
__device__ __forceinline__ double pairHat(uint32_t m, const double* __restrict__ A, size_t i,
                                          int64_t D, int XF, double u, double uUp, double uDown) {
  if (!(m & (kPairUp | kPairDown))) return u;
  const bool up = (m & kPairUp) != 0;
  const size_t q = up ? i + size_t(XF) : i - size_t(XF);
  const double aiq = A[i + size_t(up ? 2 : 3) * D];
  const double aqi = A[q + size_t(up ? 3 : 2) * D];
  return (u - aiq * (up ? uUp : uDown)) / (1. - aiq * aqi);
}

enum PassKind { kPassFirstPV, kPassPV, kPassST };

// PV and ST: u from the vectors, w = A M^-1 u, over one chunk.  Per four rows
// j .. j + 3 a lane loads the rows j + 2 .. j + 5 of its column (u-hat of a node
// may need its partner two rows from the last output), forms u-hat of the rows
// j + 1 .. j + 4 and puts it in LDS, a ring of eight rows.  Loads do not wait
// for the node types (the vectors read zero on solid nodes), and those of the
// first rows are issued before the previous pass's sums are added up.
template <int KIND>
struct ApplyPass {
  struct Raw {
    double r[kRows], p[kRows], v[kRows];
    uint32_t m[kRows];
  };
  struct Coef {
    double a[kRows][4], rh[kRows];
  };

  const SolveSys& y;
  const Chunk& c;
  const double *r, *po, *vo, *A;
  double *rh, *pn, *out;
  int64_t XF, D;
  bool inner, on;
  int pos, x;

  __device__ __forceinline__ ApplyPass(const SolveSys& sys, const Chunk& chunk, int it)
      : y(sys), c(chunk) {
    const int t = int(threadIdx.x);
    inner = t < c.w;
    on = inner || t == kStripX || t == kStripX + 1;
    pos = inner ? t + 1 : (t == kStripX ? 0 : c.w + 1);
    x = c.x0 + pos - 1;
    x = x < 0 ? x + y.nX : (x >= y.nX ? x - y.nX : x);
    XF = y.XF;
    D = y.D;
    A = y.A;
    r = it == 0 ? y.r[0] : y.r[1 + ((it - 1) & 1)];
    po = it == 1 ? y.r[0] : y.p[(it & 1) ^ 1];
    vo = KIND == kPassST ? y.v[it & 1] : y.v[(it & 1) ^ 1];
    rh = y.r[0];
    pn = y.p[it & 1];
    out = KIND == kPassST ? y.t : y.v[it & 1];
  }

  // rows k .. k + 3 of this lane's column; rows outside the lattice are solid
  __device__ __forceinline__ void load(Raw& q, int k) const {
    if (!on) {
#pragma unroll
      for (int i = 0; i < kRows; i++) q.m[i] = kSolid;
      return;
    }
#pragma unroll
    for (int i = 0; i < kRows; i++) {
      const int row = min(max(k + i, 0), y.nY - 1);
      const size_t g = size_t(x + XF * row);
      q.m[i] = row == k + i ? uint32_t(y.mask[g]) : uint32_t(kSolid);
      q.r[i] = r[g];
      if (KIND == kPassPV) q.p[i] = po[g];
      if (KIND != kPassFirstPV) q.v[i] = vo[g];
    }
  }
  // the rows' coefficients (and rh)
  __device__ __forceinline__ void load(Coef& q, int k) const {
    if (!inner) return;
#pragma unroll
    for (int i = 0; i < kRows; i++) {
      const size_t g = size_t(x + XF * min(k + i, y.nY - 1));
#pragma unroll
      for (int d = 0; d < 4; d++) q.a[i][d] = A[g + size_t(d) * D];
      if (KIND == kPassPV) q.rh[i] = rh[g];
    }
  }

  __device__ __forceinline__ double u(const Raw& q, int i, const SolveState& s) const {
    if (q.m[i] & kSolid) return 0.;
    if (KIND == kPassFirstPV) return q.r[i];
    if (KIND == kPassST) return q.r[i] - s.alpha * q.v[i];
    return s.restart ? q.r[i] : q.r[i] + s.beta * (q.p[i] - s.omega * q.v[i]);
  }

  __device__ __forceinline__ void run(const SolveState& s, const Raw& head, Raw& body, Coef& co,
                                      Sum& acc0, Sum& acc1) const {
    __shared__ double row[2 * kRows][kStripX + 2];
    // u and node types of rows j .. j + 5, u-hat of rows j - 1 .. j + 4
    double U[kRows + 2], H[kRows + 2];
    uint32_t M[kRows + 2];
    {
      const double um2 = u(head, 0, s), um1 = u(head, 1, s);
      U[0] = u(head, 2, s);
      U[1] = u(head, 3, s);
      M[0] = head.m[2];
      M[1] = head.m[3];
      const size_t g = size_t(x + XF * c.y0);
      H[0] = pairHat(head.m[1], A, g - XF, D, y.XF, um1, U[0], um2);
      H[1] = pairHat(M[0], A, g, D, y.XF, U[0], U[1], um1);
      if (on) row[c.y0 & 7][pos] = H[1];
    }
    for (int j = c.y0; j < c.y1; j += kRows) {
      const size_t g = size_t(x + XF * j);
#pragma unroll
      for (int i = 0; i < kRows; i++) {
        U[i + 2] = u(body, i, s);
        M[i + 2] = body.m[i];
      }
#pragma unroll
      for (int i = 0; i < kRows; i++) {
        H[i + 2] = pairHat(M[i + 1], A, g + size_t(XF) * (i + 1), D, y.XF, U[i + 1], U[i + 2], U[i]);
        if (on) row[(j + 1 + i) & 7][pos] = H[i + 2];
      }
      __syncthreads();
      if (inner) {
#pragma unroll
        for (int i = 0; i < kRows; i++) {
          if ((M[i] & kSolid) || j + i >= c.y1) continue;
          const double* e = row[(j + i) & 7];
          const double w = H[i + 1] + (co.a[i][0] * e[pos + 1] + co.a[i][1] * e[pos - 1] +
                                       co.a[i][2] * H[i + 2] + co.a[i][3] * H[i]);
          const size_t o = g + size_t(XF) * i;
          out[o] = w;
          if (KIND == kPassST) {
            acc0.add(w * U[i]);
            acc1.add(w * w);
          } else if (KIND == kPassFirstPV) {
            acc0.add(U[i] * w);
          } else {
            pn[o] = U[i];
            if (s.restart) rh[o] = U[i];  // rh = r
            acc0.add((s.restart ? U[i] : co.rh[i]) * w);
          }
        }
      }
      if (j + kRows >= c.y1) break;
      load(body, j + kRows + 2);
      load(co, j + kRows);
      U[0] = U[kRows];
      U[1] = U[kRows + 1];
      M[0] = M[kRows];
      M[1] = M[kRows + 1];
      H[0] = H[kRows];
      H[1] = H[kRows + 1];
      __syncthreads();
    }
  }
};

// The passes: grid.x covers the chunks (8 * per blocks), grid.y the systems.
// it: the iteration, par: the pass parity.
template <int KIND>
__global__ __launch_bounds__(kStripThreads) void solveApply(SolvePair P, int it, int par) {
  const SolveSys& y = P.sys[blockIdx.y];
  Chunk c;
  if (!chunkOf(y.s, y.nX, y.nY, c)) return;
  constexpr int stage = KIND == kPassFirstPV ? 0 : (KIND == kPassPV ? 3 : 1);
  if (passedOn(y, stage, par, c.T == 0)) return;
  Partials<kStripThreads> in;
  in.load(y, par);
  const ApplyPass<KIND> pass(y, c, it);
  typename ApplyPass<KIND>::Raw head, body;
  typename ApplyPass<KIND>::Coef co;
  pass.load(head, c.y0 - 2);
  pass.load(body, c.y0 + 2);
  pass.load(co, c.y0);
  SolveState s;
  if (!beginPass<kStripThreads>(y, in, stage, par, c.T == 0, s)) return;
  Sum a{}, b{};
  pass.run(s, head, body, co, a, b);
  writePartial<kStripThreads>(y, c.T, par ^ 1, a, b);
}

// XR over one chunk, four rows at a time so that their loads overlap.
template <bool FIRST>
struct UpdatePass {
  struct Raw {
    double r[kRows], p[kRows], v[kRows], t[kRows], rh[kRows], x[kRows];
    uint32_t m[kRows];
  };
  const SolveSys& y;
  const Chunk& c;
  const double *r, *p, *rh, *v;
  double* rn;
  int64_t XF, D;

  __device__ __forceinline__ UpdatePass(const SolveSys& sys, const Chunk& chunk, int it)
      : y(sys), c(chunk) {
    XF = y.XF;
    D = y.D;
    r = FIRST ? y.r[0] : y.r[1 + ((it - 1) & 1)];
    p = FIRST ? y.r[0] : y.p[it & 1];
    rh = y.r[0];
    v = y.v[it & 1];
    rn = y.r[1 + (it & 1)];
  }
  __device__ __forceinline__ size_t at(int k) const { return size_t(c.x0 + int(threadIdx.x) + XF * k); }

  __device__ __forceinline__ void load(Raw& q, int k) const {
#pragma unroll
    for (int j = 0; j < kRows; j++) {
      const int row = min(k + j, c.y1 - 1);
      const size_t i = at(row);
      q.m[j] = row == k + j ? uint32_t(y.mask[i]) : uint32_t(kSolid);
      q.r[j] = r[i];
      q.v[j] = v[i];
      q.t[j] = y.t[i];
      q.x[j] = y.x[i];
      q.p[j] = FIRST ? q.r[j] : p[i];
      q.rh[j] = FIRST ? q.r[j] : rh[i];
    }
  }
  __device__ __forceinline__ void run(const SolveState& s, Raw& q, Sum& acc0, Sum& acc1) const {
    const double al = s.alpha, om = s.omega;
    for (int k = c.y0;;) {
#pragma unroll
      for (int j = 0; j < kRows; j++) {
        if (q.m[j] & kSolid) continue;
        const size_t i = at(k + j);
        const double sc = q.r[j] - al * q.v[j];
        double ph = q.p[j], sh = sc;
        if (q.m[j] & (kPairUp | kPairDown)) {
          const size_t n = (q.m[j] & kPairUp) ? i + size_t(XF) : i - size_t(XF);
          const double pq = p[n], sq = r[n] - al * v[n];
          ph = pairHat(q.m[j], y.A, i, D, y.XF, ph, pq, pq);
          sh = pairHat(q.m[j], y.A, i, D, y.XF, sh, sq, sq);
        }
        y.x[i] = q.x[j] + (al * ph + om * sh);
        const double res = sc - om * q.t[j];
        rn[i] = res;
        acc0.add(q.rh[j] * res);
        acc1.add(res * res);
      }
      k += kRows;
      if (k >= c.y1) break;
      load(q, k);
    }
  }
};

template <bool FIRST>
__global__ __launch_bounds__(kStripX) void solveUpdate(SolvePair P, int it, int par) {
  const SolveSys& y = P.sys[blockIdx.y];
  Chunk c;
  if (!chunkOf(y.s, y.nX, y.nY, c)) return;
  if (passedOn(y, 2, par, c.T == 0)) return;
  Partials<kStripX> in;
  in.load(y, par);
  const UpdatePass<FIRST> pass(y, c, it);
  typename UpdatePass<FIRST>::Raw q;
  const bool inner = int(threadIdx.x) < c.w;
  if (inner) pass.load(q, c.y0);
  SolveState s;
  if (!beginPass<kStripX>(y, in, 2, par, c.T == 0, s)) return;
  Sum a{}, b{};
  if (inner) pass.run(s, q, a, b);
  writePartial<kStripX>(y, c.T, par ^ 1, a, b);
}

// After the last XR launched (parity par): takes its sums in and leaves every
// system's state in `out`; with flags, flags[0] = 1 when all have finished,
// flags[1] = 1 when one met a non-finite residual, flags[2] = the iterations
// they took.  The pass state is left alone, so more iterations may follow.
// One block.
__global__ __launch_bounds__(kStripX) void solveFinish(SolvePair P, int n, int par,
                                                       int* __restrict__ flags) {
  int done = 1, nan = 0, iters = 0;
  for (int k = 0; k < n; k++) {
    const SolveSys& y = P.sys[k];
    double a, b;
    Partials<kStripX> in;
    in.load(y, par);
    in.sums(y, par, a, b);
    SolveState s = y.st[par];
    if (!s.done) advance(s, 3, a, b, y);
    if (threadIdx.x == 0) *y.out = s;
    done = done && s.done;
    nan = nan || s.nan;
    iters = max(iters, s.iters);
  }
  if (flags && threadIdx.x == 0) {
    flags[0] = done;
    flags[1] = nan;
    flags[2] = iters;
  }
}

// ---------------------------------------------------------------------------
// assembly: the rows and the first residual
// ---------------------------------------------------------------------------

// Calls f(x, y) for the nodes of this lane's column in the block's chunk.
template <class F>
__device__ __forceinline__ void forChunk(const Chunk& c, F&& f) {
  if (int(threadIdx.x) >= c.w) return;
  for (int k = c.y0; k < c.y1; k++) f(c.x0 + int(threadIdx.x), k);
}

// Update_kOmega_Coeffs_Implicit (kOmegaKernels.cl:187-480): the normalised
// rows of both systems, then the first residual r = b - A x from the current
// K and O (the solve's initial guess); sums (r, r).  With prev set, K and O
// are also kept there (the restart point of the step).
template <class M>
__global__ __launch_bounds__(kStripX) void koCoeffs(
    const double* __restrict__ Nut, const double* __restrict__ Dk, const double* __restrict__ Do,
    const double* __restrict__ F1a, const double* __restrict__ dkdo, const double* __restrict__ Sx,
    const M* __restrict__ rho, const M* __restrict__ uxa, const M* __restrict__ uya,
    const double* __restrict__ dX, const double* __restrict__ Wd, double* __restrict__ prevK,
    double* __restrict__ prevO, SolvePair P, KOParams p) {
  Chunk c;
  if (!chunkOf(P.sys[0].s, p.nX, p.nY, c)) return;
  Sum acc[2]{};
  forChunk(c, [&](int x, int y) {
    const size_t g = size_t(x) + size_t(p.XF) * y;
    const uint32_t m = P.sys[0].mask[g];
    if (m & kSolid) return;
    KORows o;
    koCoeffRow<M>(x, g, m, P.sys[0].x, P.sys[1].x, Nut, Dk, Do, F1a, dkdo, Sx, rho, uxa, uya, dX,
                  Wd, p, o);
    size_t nb[4];
    nbIndex(p, x, g, nb);
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const double* A = v == 0 ? o.Ak : o.Ao;
      const double* X = P.sys[v].x;
      double* prev = v == 0 ? prevK : prevO;
      if (prev) prev[g] = X[g];
      double* Av = const_cast<double*>(P.sys[v].A);
#pragma unroll
      for (int d = 0; d < 4; d++) Av[g + size_t(d) * p.D] = A[d];
      const double b = v == 0 ? o.bk : o.bo;
      const double ax = X[g] + (A[0] * X[nb[0]] + A[1] * X[nb[1]] + A[2] * X[nb[2]] +
                                A[3] * X[nb[3]]);
      const double r = b - ax;
      P.sys[v].r[0][g] = r;
      acc[v].add(r * r);
    }
  });
  writePartial<kStripX>(P.sys[0], c.T, 0, acc[0], Sum{});
  writePartial<kStripX>(P.sys[1], c.T, 0, acc[1], Sum{});
}

// ---------------------------------------------------------------------------
// temperature (clVariablesFD)
// ---------------------------------------------------------------------------

struct TParams {
  double alphaFluid, alphaFoul, prTurbInv, tIn;
};

// The three-point weights of Update_T_Coeffs_Implicit (tfdKernels.cl:154-181):
// spacings held at 0.1 or more; the first derivative falls back to the
// two-point central difference where |the tested weight| > 10 (the x row
// tests its centre weight, the y row its north weight, as the kernel does).
__device__ __forceinline__ void tWeights(double dp, double dm, bool testCentre, double (&d1)[3],
                                         double (&d2)[3]) {
  dp = fmax(dp, 0.1);
  dm = fmax(dm, 0.1);
  const double dc = fmax(dp + dm, 0.1);
  d1[0] = dm / (dp * dc);
  d1[1] = -dp / (dm * dc);
  d1[2] = (dp - dm) / (dp * dm);
  d2[0] = 2. / (dp * dc);
  d2[1] = 2. / (dm * dc);
  d2[2] = -2. / (dp * dm);
  if (fabs(testCentre ? d1[2] : d1[0]) > 10.) {
    d1[0] = 1. / dc;
    d1[1] = -1. / dc;
    d1[2] = 0.;
  }
}

// Update_T_Coeffs_Implicit (tfdKernels.cl:122-280) in the five-point row
// form of the k-omega systems (diagonal 1; planes E, W, N, S), then the first
// residual r = b - A T from the current T; sums (r, r) and (b, b).  Rows on the nodes of tmask that are not
// solid (solid in the clean geometry); a node solid in the LB mask (the
// fouling layer) takes alphaFoul.  nu_t / Pr_t adds to alpha and the x and y
// differences of nu_t to the advection (the kernel multiplies the centre
// term by 1 / Pr_t twice, which is kept).  The source is T clamped to
// [0, T_in]; the inlet column's W coefficient moves to the right-hand side
// with T_in and the outlet column's E coefficient into the diagonal.  When
// Tprev is set, T is also copied there (the restart point of the step).
template <class M>
__global__ __launch_bounds__(kStripX) void thermalCoeffs(
    const uint16_t* __restrict__ lbmask,
    const double* __restrict__ dX0, const double* __restrict__ Nut, const M* __restrict__ uxa,
    const M* __restrict__ uya, double* __restrict__ Tprev, SolvePair P, TParams tp, double dt,
    KOParams p) {
  const SolveSys& sy = P.sys[0];
  Chunk c;
  if (!chunkOf(sy.s, p.nX, p.nY, c)) return;
  Sum rr{}, bb{};
  forChunk(c, [&](int x, int y) {
    const size_t g = size_t(x) + size_t(p.XF) * y;
    if (sy.mask[g] & kSolid) return;
    const double* T = sy.x;
    double dx1[3], dx2[3], dy1[3], dy2[3];
    tWeights(dX0[g], dX0[g + p.D], true, dx1, dx2);
    tWeights(dX0[g + 2 * p.D], dX0[g + 3 * p.D], false, dy1, dy2);
    size_t nb[4];
    nbIndex(p, x, g, nb);
    double alpha = (lbmask[g] & kSolid) ? tp.alphaFoul : tp.alphaFluid;
    const double at = Nut[g] * tp.prTurbInv;
    const double Jx = double(uxa[g]) -
                      tp.prTurbInv * (dx1[0] * Nut[nb[0]] + dx1[1] * Nut[nb[1]] + dx1[2] * at);
    const double Jy = double(uya[g]) -
                      tp.prTurbInv * (dy1[0] * Nut[nb[2]] + dy1[1] * Nut[nb[3]] + dy1[2] * at);
    alpha += at;
    const double Tg = T[g];
    double src = fmin(fmax(0., Tg), tp.tIn);
    double C = 1. + dt * (Jx * dx1[2] + Jy * dy1[2] - alpha * (dx2[2] + dy2[2]));
    const double S = dt * (Jy * dy1[1] - alpha * dy2[1]);
    const double W = dt * (Jx * dx1[1] - alpha * dx2[1]);
    if (x == 0) src -= tp.tIn * W;
    const double E = dt * (Jx * dx1[0] - alpha * dx2[0]);
    if (x == p.nX - 1) C += E;
    const double N = dt * (Jy * dy1[0] - alpha * dy2[0]);
    const double inv = 1. / C;
    double A[4];
    A[0] = x < p.nX - 1 ? E * inv : 0.;
    A[1] = x > 0 ? W * inv : 0.;
    A[2] = N * inv;
    A[3] = S * inv;
    const double b = src * inv;
#pragma unroll
    for (int d = 0; d < 4; d++) const_cast<double*>(sy.A)[g + size_t(d) * p.D] = A[d];
    const double ax = Tg + (A[0] * T[nb[0]] + A[1] * T[nb[1]] + A[2] * T[nb[2]] + A[3] * T[nb[3]]);
    const double r = b - ax;
    sy.r[0][g] = r;
    if (Tprev) Tprev[g] = Tg;
    rr.add(r * r);
    bb.add(b * b);
  });
  writePartial<kStripX>(sy, c.T, 0, rr, bb);
}

}  // namespace dev
}  // namespace kofm
