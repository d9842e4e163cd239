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
// of 10 + 7 + 8; s is recomputed in XR.
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
  double2* partial;  // [2][2 * max(nblk, n0)]: sums by pass parity
  SolveState* out;  // the state the last finish kernel saw
  double rtol, atol;
  int maxit;
  int crit;         // stopping rule: 0 as GMRESSolver, 1 as BiCGStabSolver
  int nX, nY, XF;
  int64_t D;
  Strips s;
  int n0;           // blocks of the assembly, whose sums open the solve
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

// A sum carried with its rounding error (Knuth's two-sum): how the lattice is
// cut into blocks then changes the passes' dot products by little more than
// their last rounding (the errors themselves are added up plainly), which
// ill-conditioned rows (fouled walls) would otherwise feel from the third
// iteration on.  The passes wait for memory; plain sums measured 0.6 to 1 us
// less of a pass's 5 to 40.
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
__device__ __forceinline__ double2* partialSlot(const SolveSys& y, int slot) {
  return y.partial + size_t(slot) * 2 * max(y.s.nblk, y.n0);
}
template <int THREADS>
__device__ __forceinline__ void writePartial(const SolveSys& y, int T, int slot, Sum a, Sum b) {
  blockSum2<THREADS>(a, b);
  if (threadIdx.x == 0) {
    double2* out = partialSlot(y, slot) + 2 * T;
    out[0] = make_double2(a.hi, a.lo);
    out[1] = make_double2(b.hi, b.lo);
  }
}
// In two parts, so that a pass can issue its own first loads in between: a
// wave's loads return in order, and the sums must not wait behind the rows.
template <int THREADS>
struct Partials {
  double2 a, b;
  __device__ __forceinline__ void load(const SolveSys& y, int slot, int n) {
    const double2* in = partialSlot(y, slot);
    const int i = int(threadIdx.x);
    a = b = make_double2(0., 0.);
    if (i < n) {
      a = in[2 * i];
      b = in[2 * i + 1];
    }
  }
  __device__ __forceinline__ void sums(const SolveSys& y, int slot, int n, double& outA,
                                       double& outB) const {
    const double2* in = partialSlot(y, slot);
    Sum p{a.x, a.y}, q{b.x, b.y};
    for (int i = int(threadIdx.x) + THREADS; i < n; i += THREADS) {
      const double2 u = in[2 * i], v = in[2 * i + 1];
      p.add(Sum{u.x, u.y});
      q.add(Sum{v.x, v.y});
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
  in.sums(y, par, stage == 0 ? y.n0 : y.s.nblk, a, b);
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

template <int KIND>
__device__ __forceinline__ void applyBlock(const SolveSys& y, int it, int par) {
  Chunk c;
  if (!chunkOf(y.s, y.nX, y.nY, c)) return;
  constexpr int stage = KIND == kPassFirstPV ? 0 : (KIND == kPassPV ? 3 : 1);
  if (passedOn(y, stage, par, c.T == 0)) return;
  Partials<kStripThreads> in;
  in.load(y, par, stage == 0 ? y.n0 : y.s.nblk);
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

// The passes: grid.x covers the chunks (8 * per blocks), grid.y the systems,
// which are the launch's arguments or, for the members of an ensemble, a table
// (grid.x then covers the largest).  it: the iteration, par: the pass parity.
template <int KIND>
__global__ __launch_bounds__(kStripThreads) void solveApply(SolvePair P, int it, int par) {
  applyBlock<KIND>(P.sys[blockIdx.y], it, par);
}
template <int KIND>
__global__ __launch_bounds__(kStripThreads) void solveApplyTable(const SolveSys* __restrict__ tab,
                                                                 int it, int par) {
  applyBlock<KIND>(tab[blockIdx.y], it, par);
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
__device__ __forceinline__ void updateBlock(const SolveSys& y, int it, int par) {
  Chunk c;
  if (!chunkOf(y.s, y.nX, y.nY, c)) return;
  if (passedOn(y, 2, par, c.T == 0)) return;
  Partials<kStripX> in;
  in.load(y, par, y.s.nblk);
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
template <bool FIRST>
__global__ __launch_bounds__(kStripX) void solveUpdate(SolvePair P, int it, int par) {
  updateBlock<FIRST>(P.sys[blockIdx.y], it, par);
}
template <bool FIRST>
__global__ __launch_bounds__(kStripX) void solveUpdateTable(const SolveSys* __restrict__ tab, int it,
                                                            int par) {
  updateBlock<FIRST>(tab[blockIdx.y], it, par);
}

// After the last XR launched (parity par): takes its sums in and leaves every
// system's state in `out`; with flags, flags[0] = 1 when all have finished,
// flags[1] = 1 when one met a non-finite residual, flags[2] = the iterations
// they took.  The pass state is left alone, so more iterations may follow.
// One block per lattice.
__device__ __forceinline__ void finishBlock(const SolveSys* __restrict__ sys, int n, int par,
                                            int* __restrict__ flags) {
  int done = 1, nan = 0, iters = 0;
  for (int k = 0; k < n; k++) {
    const SolveSys& y = sys[k];
    double a, b;
    Partials<kStripX> in;
    in.load(y, par, y.s.nblk);
    in.sums(y, par, y.s.nblk, a, b);
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
__global__ __launch_bounds__(kStripX) void solveFinish(SolvePair P, int n, int par,
                                                       int* __restrict__ flags) {
  finishBlock(P.sys, n, par, flags);
}
// two systems and four flags per member
__global__ __launch_bounds__(kStripX) void solveFinishTable(const SolveSys* __restrict__ tab, int par,
                                                            int* __restrict__ flags) {
  finishBlock(tab + 2 * blockIdx.x, 2, par, flags + 4 * blockIdx.x);
}

// ---------------------------------------------------------------------------
// assembly: the rows and the first residual
// ---------------------------------------------------------------------------

// The assembly kernels take tiles of 64 x 8 nodes with 256 lanes (two nodes
// each), up to kTileBlocks blocks walking their XCD's run of tiles: the two per
// CU that the k-omega assembly's registers allow, and few enough that the first
// pass can add up their sums.
constexpr int kTileX = 64, kTileY = 8, kTileLanes = 256, kTileBlocks = 512;
constexpr int kTileStep = kTileLanes / kTileX;  // rows between a lane's two nodes
struct Tiles {
  int tilesX, nTiles, per, blocks;
};
inline Tiles tilesFor(int nX, int nY) {
  Tiles t;
  t.tilesX = (nX + kTileX - 1) / kTileX;
  t.nTiles = t.tilesX * ((nY + kTileY - 1) / kTileY);
  t.per = (t.nTiles + 7) / 8;
  t.blocks = 8 * t.per < kTileBlocks ? 8 * t.per : kTileBlocks;
  return t;
}

// Calls f(x0, y0) for the tiles of this block: the blocks of XCD k = blockIdx
// % 8 walk the k-th run of tiles.
template <class F>
__device__ __forceinline__ void forTiles(const Tiles& t, F&& f) {
  const int xcd = int(blockIdx.x & 7), stride = t.blocks >> 3;
  const int end = min((xcd + 1) * t.per, t.nTiles);
  for (int T = xcd * t.per + int(blockIdx.x >> 3); T < end; T += stride)
    f((T % t.tilesX) * kTileX, (T / t.tilesX) * kTileY);
}
// Calls f(x, y) for this lane's nodes of every tile.
template <class F>
__device__ __forceinline__ void forTileNodes(const Tiles& t, int nX, int nY, F&& f) {
  forTiles(t, [&](int x0, int y0) {
    const int x = x0 + int(threadIdx.x) % kTileX, y = y0 + int(threadIdx.x) / kTileX;
    if (x >= nX) return;
    if (y < nY) f(x, y);
    if (y + kTileStep < nY) f(x, y + kTileStep);
  });
}

// Difference weights of nodes whose four wall spacings are 1 (fdCoeffsT(1, 1)).
#define KOFM_UNIT_WEIGHTS {0.5, -0.5, 0., 1., 1., -2.}

// Marks the nodes whose four spacings are exactly 1: every fluid node that is
// not next to a wall.  The assembly then neither reads the spacings (4 of its
// planes) nor divides by them (24 divisions per node).
__global__ __launch_bounds__(kBlockX) void unitSpacing(uint16_t* __restrict__ mask,
                                                       const double* __restrict__ dX, int64_t D) {
  const int64_t i = int64_t(blockIdx.x) * kBlockX + threadIdx.x;
  if (i >= D) return;
  const bool unit = dX[i] == 1. && dX[i + D] == 1. && dX[i + 2 * D] == 1. && dX[i + 3 * D] == 1.;
  mask[i] = uint16_t((mask[i] & ~uint32_t(kUnitDx)) | (unit ? uint32_t(kUnitDx) : 0u));
}

// What the k-omega assembly reads and writes beside the systems.
struct KOAssembly {
  const double *nut, *S, *dX, *wd;
  const void *rho, *ux, *uy;  // arithmetic type
  double *Dk, *Do;            // diffusivities: read on solid nodes, written when keepD
  double *F1, *dkdo;          // written when set (the adjoint's tape)
  double *prevK, *prevO;      // when set, k and omega are kept there (restart point)
  int keepD;
  double nu, dt;
  Tiles tiles;
};

// Update_kOmega_Diffusivities and Update_kOmega_Coeffs_Implicit
// (kOmegaKernels.cl:7-95, 187-480): the diffusivities of a tile and the ring
// around it go to LDS, then the normalised rows of both systems and the first
// residual r = b - A x from the current k and omega (the solve's initial
// guess); sums (r, r).  The ring's 144 evaluations beside the tile's 512 spare
// the five diffusivity planes a write and a read.  A solid node keeps the
// diffusivity it last had as a fluid node (zero if it never was).
// Its registers leave two waves per SIMD, so a lane issues the loads of its
// nodes together before it evaluates the first; then 4096 x 512 takes 106 us and
// 2000 x 204 22 us, where separate diffusivity and row kernels took 166 and 30.
// (Measured slower: a lane per node with extra waves for the ring, 116 and 36;
// 16 x 16 tiles, 167 and 38; fewer registers by spilling, 206 and more.)
template <class M>
__device__ __forceinline__ void assembleBlock(const SolvePair& P, const KOAssembly& q) {
  if (int(blockIdx.x) >= q.tiles.blocks) return;
  constexpr int RX = kTileX + 2, RY = kTileY + 2;
  __shared__ double ldk[RX * RY], ldo[RX * RY];
  const SolveSys& sy = P.sys[0];
  const int nX = sy.nX, nY = sy.nY;
  const int64_t XF = sy.XF, D = sy.D;
  const uint16_t* __restrict__ mask = sy.mask;
  const double* __restrict__ K = P.sys[0].x;
  const double* __restrict__ O = P.sys[1].x;
  const M* __restrict__ rho = static_cast<const M*>(q.rho);
  const M* __restrict__ uxa = static_cast<const M*>(q.ux);
  const M* __restrict__ uya = static_cast<const M*>(q.uy);
  const double* __restrict__ dX = q.dX;
  Sum acc[2]{};

  // A node's diffusivity inputs; lanes without a node take node 0's values and
  // use none, rows past the lattice the node's own.
  struct Node {
    size_t g;
    uint32_t m;
    double k[5], o[5], nut, wd, rho;
  };
  auto load = [&](Node& n, int x, int y, bool on) {
    n.g = on ? size_t(x) + size_t(XF) * y : 0;
    const size_t g = n.g;
    const size_t nb[4] = {on ? (x < nX - 1 ? g + 1 : g - x) : g, on ? (x > 0 ? g - 1 : g + (nX - 1)) : g,
                          on && y < nY - 1 ? g + XF : g, on && y > 0 ? g - XF : g};
    n.m = mask[g];
    if (!on) n.m = kSolid;
    n.k[0] = K[g];
    n.o[0] = O[g];
#pragma unroll
    for (int d = 0; d < 4; d++) {
      n.k[1 + d] = K[nb[d]];
      n.o[1 + d] = O[nb[d]];
    }
    n.nut = q.nut[g];
    n.wd = q.wd[g];
    n.rho = double(rho[g]);
  };
  auto diff = [&](const Node& n, bool on, double (&d)[ko::kDiffOutputs]) {
    if (n.m & kSolid) {
      d[ko::kDiffDk] = on ? q.Dk[n.g] : 0.;
      d[ko::kDiffDo] = on ? q.Do[n.g] : 0.;
      return;
    }
    double in[ko::kDiffInputs] = {n.k[0], n.k[1], n.k[2], n.k[3], n.k[4], n.o[0],
                                  n.o[1], n.o[2], n.o[3], n.o[4], n.nut,  n.wd,
                                  n.rho,  1.,     1.,     1.,     1.};
    if (n.m & kUnitDx) {
      const double ax[6] = KOFM_UNIT_WEIGHTS, ay[6] = KOFM_UNIT_WEIGHTS;
      ko::koDiffCore<double, double>(in, ax, ay, q.nu, d);
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) in[ko::kDiffDx + c] = dX[n.g + size_t(c) * D];
      ko::koDiffT<double>(in, q.nu, d);
    }
  };

  const int t = int(threadIdx.x);
  const int ix = t % kTileX, iy = t / kTileX;
  // this lane's ring node: the rows below and above, then the columns beside
  // the tile (corners are not used); east of a tile that the lattice's edge
  // cuts it follows the last column
  const bool ring = t < 2 * kTileX + 2 * kTileY;
  const int ringRow = t < 2 * kTileX ? (t < kTileX ? 0 : kTileY + 1) : 1 + t % kTileY;
  const int ringCol = t < 2 * kTileX ? 1 + t % kTileX : (t < 2 * kTileX + kTileY ? 0 : -1);

  forTiles(q.tiles, [&](int x0, int y0) {
    const int w = min(kTileX, nX - x0);
    Node n[2], e;
    bool on[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int y = y0 + iy + kTileStep * i;
      on[i] = ix < w && y < nY;
      load(n[i], x0 + ix, y, on[i]);
    }
    const int ec = ringCol < 0 ? w + 1 : ringCol;
    int ex = x0 + ec - 1;
    ex = ex < 0 ? nX - 1 : (ex >= nX ? ex - nX : ex);
    const int ey = y0 + ringRow - 1;
    const bool eon = ring && (ec <= w || ringCol < 0) && ey >= 0 && ey < nY;
    if (ring) load(e, ex, ey, eon);
    double d[2][ko::kDiffOutputs];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      diff(n[i], on[i], d[i]);
      const int c = (ix + 1) + RX * (iy + kTileStep * i + 1);
      ldk[c] = d[i][ko::kDiffDk];
      ldo[c] = d[i][ko::kDiffDo];
      if (n[i].m & kSolid) continue;
      if (q.keepD) {
        q.Dk[n[i].g] = d[i][ko::kDiffDk];
        q.Do[n[i].g] = d[i][ko::kDiffDo];
      }
      if (q.F1) {
        q.F1[n[i].g] = d[i][ko::kDiffF1];
        q.dkdo[n[i].g] = d[i][ko::kDiffMx];
        q.dkdo[n[i].g + D] = d[i][ko::kDiffMy];
      }
    }
    // (a cut tile's ring column may lie on a cell that an idle lane of the
    // tile has just written)
    if (w < kTileX) __syncthreads();
    if (eon) {
      double de[ko::kDiffOutputs];
      diff(e, true, de);
      ldk[ec + RX * ringRow] = de[ko::kDiffDk];
      ldo[ec + RX * ringRow] = de[ko::kDiffDo];
    }
    double S[2][3], u[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
      for (int c = 0; c < 3; c++) S[i][c] = q.S[n[i].g + size_t(c) * D];
      u[i][0] = double(uxa[n[i].g]);
      u[i][1] = double(uya[n[i].g]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if (n[i].m & kSolid) continue;
      const size_t g = n[i].g;
      const int c = (ix + 1) + RX * (iy + kTileStep * i + 1);
      double in[ko::kRowInputs] = {
          d[i][ko::kDiffDk], ldk[c + 1], ldk[c - 1], ldk[c + RX], ldk[c - RX],
          d[i][ko::kDiffDo], ldo[c + 1], ldo[c - 1], ldo[c + RX], ldo[c - RX],
          d[i][ko::kDiffMx], d[i][ko::kDiffMy], u[i][0], u[i][1], n[i].rho, n[i].k[0], n[i].o[0],
          d[i][ko::kDiffF1], n[i].nut, S[i][0], S[i][1], S[i][2], n[i].wd, 1., 1., 1., 1.};
      double out[ko::kRowOutputs];
      const bool nesw = (n[i].m & kNesw) != 0;
      if (n[i].m & kUnitDx) {
        const double ax[6] = KOFM_UNIT_WEIGHTS, ay[6] = KOFM_UNIT_WEIGHTS;
        ko::koRowCore<double, double>(in, ax, ay, nesw, q.nu, q.dt, out);
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) in[ko::kRowDx + j] = dX[g + size_t(j) * D];
        ko::koRowT<double>(in, nesw, q.nu, q.dt, out);
      }
#pragma unroll
      for (int v = 0; v < 2; v++) {
        const double* A = out + (v == 0 ? ko::kRowAk : ko::kRowAo);
        const double* X = v == 0 ? n[i].k : n[i].o;
        double* prev = v == 0 ? q.prevK : q.prevO;
        if (prev) prev[g] = X[0];
        double* Av = const_cast<double*>(P.sys[v].A);
#pragma unroll
        for (int j = 0; j < 4; j++) Av[g + size_t(j) * D] = A[j];
        const double ax = X[0] + (A[0] * X[1] + A[1] * X[2] + A[2] * X[3] + A[3] * X[4]);
        const double r = out[v == 0 ? ko::kRowBk : ko::kRowBo] - ax;
        P.sys[v].r[0][g] = r;
        acc[v].add(r * r);
      }
    }
    __syncthreads();
  });
  writePartial<kTileLanes>(P.sys[0], int(blockIdx.x), 0, acc[0], Sum{});
  writePartial<kTileLanes>(P.sys[1], int(blockIdx.x), 0, acc[1], Sum{});
}
template <class M>
__global__ __launch_bounds__(kTileLanes) void koAssemble(SolvePair P, KOAssembly q) {
  assembleBlock<M>(P, q);
}
// member blockIdx.y of an ensemble
template <class M>
__global__ __launch_bounds__(kTileLanes) void koAssembleTable(const SolvePair* __restrict__ P,
                                                              const KOAssembly* __restrict__ q) {
  assembleBlock<M>(P[blockIdx.y], q[blockIdx.y]);
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
__global__ __launch_bounds__(kTileLanes) void thermalCoeffs(
    const uint16_t* __restrict__ lbmask,
    const double* __restrict__ dX0, const double* __restrict__ Nut, const M* __restrict__ uxa,
    const M* __restrict__ uya, double* __restrict__ Tprev, SolvePair P, TParams tp, double dt,
    KOParams p, Tiles tiles) {
  const SolveSys& sy = P.sys[0];
  Sum rr{}, bb{};
  forTileNodes(tiles, p.nX, p.nY, [&](int x, int y) {
    const size_t g = size_t(x) + size_t(p.XF) * y;
    const uint32_t m = sy.mask[g];
    if (m & kSolid) return;
    const double* T = sy.x;
    // spacings of 1: first differences (1/2, -1/2, 0), second (1, 1, -2)
    double dx1[3] = {0.5, -0.5, 0.}, dx2[3] = {1., 1., -2.}, dy1[3] = {0.5, -0.5, 0.},
           dy2[3] = {1., 1., -2.};
    if (!(m & kUnitDx)) {
      tWeights(dX0[g], dX0[g + p.D], true, dx1, dx2);
      tWeights(dX0[g + 2 * p.D], dX0[g + 3 * p.D], false, dy1, dy2);
    }
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
  writePartial<kTileLanes>(sy, int(blockIdx.x), 0, rr, bb);
}

}  // namespace dev
}  // namespace kofm
