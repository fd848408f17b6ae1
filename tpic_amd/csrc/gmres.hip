// Restarted GMRES(m) for A(E_theta) = rhs on the device, FP64 throughout
// (run_gmres_system solves A x = b for any device b and initial x, and with
// Context::transposed_operator the adjoint system A^T x = b).
//
// Algorithm of Gmres::host_blocking_solve
// (include/tpic/ecsim/gmres/gmres_device.hpp:355-454): x0 = E^n, r = b - A x,
// tolerance relative to |b| (scale 1 for b = 0); each restart starts from r;
// each Arnoldi step applies A, forms the projection dots against the basis in
// one batch, orthogonalises by one classical Gram-Schmidt pass fused with the
// squared norm, appends the column to the Hessenberg matrix and applies the
// Givens rotations (ArnoldiLeastSquaresUpdate, :65-98). After each restart the
// true residual |b - A x| decides convergence; the solution is committed only
// when converged. Vectors hold every interior node, periodic duplicates
// included (:133-137), so dots weight shared nodes as the reference's compact
// vectors do.
//
// A step is a chain of dependent passes over vectors that are small on all but
// the largest grids, so what counts is their number. Basis vector j is kept as
// the orthogonalised image w_j with its factor s_j = 1 / |w_j| beside it (the
// operator's image, the dots and the update take the factor), so no pass
// normalises. The dots are formed by the operator's kernel where it can
// (operator_tail_form: up to 2048 blocks of 256 nodes, or of 256 columns of a
// plane), else by k_dot_batch, and the last
// block of k_orthogonalize to finish adds the squared norm and runs the Givens
// update. A step is two launches up to 16384 nodes, three (four with walls) up
// to 524288 nodes and four above, where it was seven (16^3: the solve's 10 operator
// calls and 8 steps took 340 us of kernels, now 140).
//
// The reference's host reads two control scalars per step. Here the Givens
// update tests them (the estimate against the tolerance, the breakdown) and
// raises a stop word, and the tests of the first and of the true residual are
// kernels too: the host enqueues the first residual, the steps it expects,
// the update, the true residual and the commit, each guarded by those words, and
// reads the words once. The same steps run and stop where they would.
//
// Reductions are deterministic: fixed partials added in a fixed order.
#include "internal.hpp"
#include "arrival.hpp"

#include <cmath>

namespace tpic_mi {
namespace {

constexpr unsigned kThreads = 256;
constexpr unsigned kWaves = kThreads / 64;
constexpr unsigned kTile = 4;
constexpr unsigned kReduceBlocks = 1024;
static_assert(kReduceBlocks <= kMaxBlocks);
constexpr int kMaxColumns = 64;  // tpic_mi_config.gmres_restart's limit

__device__ inline double block_reduce(double v, double* lds) {
  v = wave_sum(v);
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  double sum = 0.0;
  if (threadIdx.x == 0)
    for (unsigned w = 0; w < kWaves; ++w) sum += lds[w];
  __syncthreads();
  return sum;  // valid in thread 0
}

__device__ __forceinline__ bool finite(double v) { return fabs(v) <= 1.7976931348623157e308; }

// The solver's words, doubles on the device read back in one copy.
enum Word : int {
  kEstimate,    // residual estimate of the last step
  kBreakdown,   // 1: its image lay in the basis
  kStop,        // 1: later steps do nothing
  kSteps,       // steps of this restart when the stop was raised
  kNonfinite,   // 1: a non-finite recurrence
  kGo,          // 1: the restart's tail (update, true residual) is to run
  kConverged,   // 1: the true residual met the tolerance
  kCommit,      // 1: it did so after a restart, whose x is the solution (a guess that met it stays)
  kTails,       // tails run
  kDone,        // steps of the last tail
  kDoneBreakdown,
  kInitial2,    // |b - A x0|^2
  kRhs2,        // |b|^2
  kResidual2,   // |b - A x|^2 of the last tail
  kAbsolute,    // the tolerance on the residual
  kWords
};

// Device state of a solve: Hessenberg columns, rotations, right-hand side of
// the least-squares problem, basis factors, words.
struct SolverState {
  double *h, *cosine, *sine, *g, *scale, *word;
  int leading;  // entries of a Hessenberg column
  double tolerance;
};

SolverState solver_state(const GmresWorkspace& w, int m, double tolerance) {
  SolverState s;
  s.leading = m + 1;
  s.h = w.state;
  s.cosine = s.h + size_t(m) * (m + 1);
  s.sine = s.cosine + m;
  s.g = s.sine + m;
  s.scale = s.g + (m + 1);
  s.word = s.scale + (m + 1);
  s.tolerance = tolerance;
  return s;
}

// Products of the image with the first `columns` basis vectors, kTile columns
// per row of blocks; the last block of a row adds its partials into dots.
__global__ __launch_bounds__(kThreads) void k_dot_batch(const double* __restrict__ basis,
                                                        const double* __restrict__ image, double* partials,
                                                        double* __restrict__ dots, unsigned* arrivals,
                                                        unsigned count, unsigned columns, Guard guard) {
  if (guard.skips()) return;
  __shared__ double lds[kWaves][kTile];
  __shared__ bool s_last;
  const unsigned first = blockIdx.y * kTile;
  double sum[kTile] = {0.0, 0.0, 0.0, 0.0};
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < count; n += gridDim.x * blockDim.x) {
    const double v = image[n];
#pragma unroll
    for (unsigned r = 0; r < kTile; ++r)
      if (first + r < columns) sum[r] += basis[size_t(first + r) * count + n] * v;
  }
  // The tile's sums with one barrier; lanes 0..3 of wave 0 store them.
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
  for (unsigned r = 0; r < kTile; ++r) {
    const double total = wave_sum(sum[r]);
    if (lane == 0) lds[wave][r] = total;
  }
  __syncthreads();
  if (threadIdx.x < kTile && first + threadIdx.x < columns) {
    double total = 0.0;
    for (unsigned w = 0; w < kWaves; ++w) total += lds[w][threadIdx.x];
    put_partial(partials + size_t(first + threadIdx.x) * gridDim.x + blockIdx.x, total);
  }
  if (!last_to_arrive(arrivals + blockIdx.y * kCounters, blockIdx.x, gridDim.x, &s_last)) return;
  const unsigned c = first + wave;  // a wave per column
  double v = 0.0;
  if (c < columns)
    for (unsigned i = lane; i < gridDim.x; i += 64) v += get_partial(partials + size_t(c) * gridDim.x + i);
  v = wave_sum(v);
  if (c < columns && lane == 0) dots[c] = v;
}

// r = b - image; partial sums of |r|^2 and |b|^2 (rows 0 and 1).
__global__ __launch_bounds__(kThreads) void k_residual(const double* __restrict__ b,
                                                       const double* __restrict__ image,
                                                       double* __restrict__ r, double* __restrict__ partials,
                                                       unsigned count, Guard guard) {
  if (guard.skips()) return;
  __shared__ double lds[kWaves];
  double s0 = 0.0, s1 = 0.0;
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < count; n += gridDim.x * blockDim.x) {
    const double bv = b[n];
    const double v = bv - image[n];
    r[n] = v;
    s0 += v * v;
    s1 += bv * bv;
  }
  const double t0 = block_reduce(s0, lds), t1 = block_reduce(s1, lds);
  if (threadIdx.x == 0) {
    partials[blockIdx.x] = t0;
    partials[gridDim.x + blockIdx.x] = t1;
  }
}

// One block: the residual's squared norm from its partials, the convergence
// test, and the start of the next restart (its first basis vector is the
// residual). `first` is the residual of the initial guess, whose right-hand
// side norm also sets the tolerance; else the residual after a restart.
__global__ __launch_bounds__(kThreads) void k_residual_test(const double* __restrict__ partials, unsigned blocks,
                                                            SolverState s, int first, Guard guard) {
  if (guard.skips()) return;
  __shared__ double lds[kWaves];
  double s0 = 0.0, s1 = 0.0;
  for (unsigned i = threadIdx.x; i < blocks; i += kThreads) {
    s0 += partials[i];
    s1 += partials[blocks + i];
  }
  const double r2 = block_reduce(s0, lds), b2 = block_reduce(s1, lds);
  if (threadIdx.x != 0) return;
  double* w = s.word;
  double absolute = w[kAbsolute];
  bool good = finite(r2);
  if (first) {
    absolute = (b2 == 0.0 ? 1.0 : sqrt(b2)) * s.tolerance;
    good = good && finite(b2);
    w[kInitial2] = r2;
    w[kRhs2] = b2;
    w[kAbsolute] = absolute;
    w[kNonfinite] = 0.0;
    w[kTails] = 0.0;
    w[kDone] = 0.0;
    w[kDoneBreakdown] = 0.0;
  } else {
    w[kTails] += 1.0;
    w[kDone] = w[kSteps];
    w[kDoneBreakdown] = w[kBreakdown];
  }
  const double r = sqrt(r2);
  const bool converged = good && r <= absolute;
  w[kResidual2] = r2;
  w[kConverged] = converged ? 1.0 : 0.0;
  w[kCommit] = converged && !first ? 1.0 : 0.0;
  w[kStop] = converged || !good || (!first && w[kBreakdown] != 0.0) ? 1.0 : 0.0;
  w[kGo] = 0.0;
  w[kSteps] = 0.0;
  w[kBreakdown] = 0.0;
  s.g[0] = r;
  s.scale[0] = r2 > 0.0 ? 1.0 / r : 0.0;
}

// The Givens update of column `step` with the squared norm of its
// orthogonalised image (ArnoldiLeastSquaresUpdate, gmres_device.hpp:65-98) and
// the host's test of the two controls (:431-441). `column` holds the column's
// dots, `cosine` and `sine` the earlier rotations, all in LDS; `upper` is the
// last entry of the rotated right-hand side so far.
__device__ void append_column(const SolverState& s, int step, bool last, double norm2, double upper, double absolute,
                              double* column, const double* cosine, const double* sine) {
  const double sub = sqrt(norm2);
  for (int row = 0; row < step; ++row) {
    const double above = column[row], below = column[row + 1];
    column[row] = cosine[row] * above + sine[row] * below;
    column[row + 1] = -sine[row] * above + cosine[row] * below;
  }
  const double diagonal = column[step];
  const double den = hypot(diagonal, sub);
  const double c = den != 0.0 ? diagonal / den : 1.0;
  const double sn = den != 0.0 ? sub / den : 0.0;
  s.cosine[step] = c;
  s.sine[step] = sn;
  column[step] = c * diagonal + sn * sub;
  s.g[step] = c * upper;
  s.g[step + 1] = -sn * upper;
  s.scale[step + 1] = sub > 0.0 ? 1.0 / sub : 0.0;
  const double estimate = fabs(sn * upper);
  const bool good = finite(estimate), breakdown = sub == 0.0;
  s.word[kEstimate] = estimate;
  if (!good || breakdown || estimate <= absolute || last) {
    s.word[kNonfinite] = good ? 0.0 : 1.0;
    s.word[kBreakdown] = breakdown ? 1.0 : 0.0;
    s.word[kSteps] = double(step + 1);
    s.word[kGo] = good ? 1.0 : 0.0;
    s.word[kStop] = 1.0;
  }
}

// Classical Gram-Schmidt of the image against the basis vectors 0 .. step:
// w_{step+1} = image - sum_c (s_c dot_c) s_c w_c, the dots added here from
// `rows` partials per column. The last block to arrive adds the blocks'
// squared norms and appends the column. The vectors' first values are
// requested before the dots.
__global__ __launch_bounds__(kThreads) void k_orthogonalize(const double* __restrict__ basis,
                                                            const double* __restrict__ image,
                                                            double* __restrict__ target,
                                                            const double* __restrict__ dots, unsigned rows,
                                                            double* norms, unsigned* arrivals, unsigned count,
                                                            int step, int last, SolverState s, Guard guard) {
  __shared__ double lds[kWaves];
  __shared__ double s_column[kMaxColumns + 1], s_weight[kMaxColumns], s_cosine[kMaxColumns], s_sine[kMaxColumns];
  __shared__ bool s_last;
  const int columns = step + 1;
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const unsigned n0 = blockIdx.x * blockDim.x + threadIdx.x;
  // What does not wait for the dots is requested first: the first values of
  // the image and of up to kAhead basis vectors, the factors, the tail's state.
  constexpr int kAhead = 8;
  double value = 0.0, ahead[kAhead];
#pragma unroll
  for (int c = 0; c < kAhead; ++c) ahead[c] = c < columns && n0 < count ? basis[size_t(c) * count + n0] : 0.0;
  if (n0 < count) value = image[n0];
  const double scale = int(lane) < columns ? s.scale[lane] : 0.0;
  const double upper = s.g[step], absolute = s.word[kAbsolute];
  const bool skip = guard.skips();
  double dot[kMaxColumns / kWaves];
#pragma unroll
  for (int t = 0; t < int(kMaxColumns / kWaves); ++t) {
    const int c = int(wave) + t * int(kWaves);
    dot[t] = 0.0;
    if (c < columns)
      for (unsigned i = lane; i < rows; i += 64) dot[t] += dots[size_t(c) * rows + i];
  }
  if (int(threadIdx.x) < step) {
    s_cosine[threadIdx.x] = s.cosine[threadIdx.x];
    s_sine[threadIdx.x] = s.sine[threadIdx.x];
  }
  if (skip) return;
#pragma unroll
  for (int t = 0; t < int(kMaxColumns / kWaves); ++t) {
    const int c = int(wave) + t * int(kWaves);
    if (c < columns) {
      const double v = rows > 1 ? wave_sum(dot[t]) : dot[t], by = __shfl(scale, c, 64);
      if (lane == 0) {
        s_column[c] = by * v;
        s_weight[c] = by * (by * v);
      }
    }
  }
  __syncthreads();
  double norm2 = 0.0;
  if (n0 < count) {
#pragma unroll
    for (int c = 0; c < kAhead; ++c)
      if (c < columns) value -= s_weight[c] * ahead[c];
    for (int c = kAhead; c < columns; ++c) value -= s_weight[c] * basis[size_t(c) * count + n0];
    target[n0] = value;
    norm2 = value * value;
  }
  for (unsigned n = n0 + gridDim.x * blockDim.x; n < count; n += gridDim.x * blockDim.x) {
    value = image[n];
#pragma unroll 4
    for (int c = 0; c < columns; ++c) value -= s_weight[c] * basis[size_t(c) * count + n];
    target[n] = value;
    norm2 += value * value;
  }
  const double total = block_reduce(norm2, lds);
  if (threadIdx.x == 0) put_partial(norms + blockIdx.x, total);
  if (!last_to_arrive(arrivals, blockIdx.x, gridDim.x, &s_last)) return;
  double v = 0.0;
  for (unsigned i = threadIdx.x; i < gridDim.x; i += kThreads) v += get_partial(norms + i);
  const double sum = block_reduce(v, lds);
  if (threadIdx.x == 0) append_column(s, step, last != 0, sum, upper, absolute, s_column, s_cosine, s_sine);
  __syncthreads();
  double* const column = s.h + size_t(step) * s.leading;
  if (int(threadIdx.x) <= step) column[threadIdx.x] = s_column[threadIdx.x];
}

// x_out = x_in + sum_c y_c s_c w_c with the least-squares solution y of the
// restart's steps, which every block solves for by itself: the triangle goes
// to LDS and a lane per row takes the back substitution.
__global__ __launch_bounds__(kThreads) void k_update(const double* __restrict__ basis, const double* x_in,
                                                     double* x_out, unsigned count, SolverState s, Guard guard) {
  if (guard.skips()) return;
  __shared__ double s_h[kMaxColumns * kMaxColumns];
  __shared__ double s_y[kMaxColumns];
  const int columns = int(s.word[kSteps]);
  for (int t = int(threadIdx.x); t < columns * columns; t += int(kThreads))
    s_h[t] = s.h[size_t(t / columns) * s.leading + t % columns];
  __syncthreads();
  if (threadIdx.x < 64) {
    const int row = int(threadIdx.x);
    double rhs = row < columns ? s.g[row] : 0.0;
    for (int col = columns - 1; col >= 0; --col) {
      const double d = s_h[col * columns + col];
      const double y = d != 0.0 ? __shfl(rhs, col, 64) / d : 0.0;
      if (row < col) rhs -= s_h[col * columns + row] * y;
      if (row == col) s_y[col] = y * s.scale[col];
    }
  }
  __syncthreads();
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < count; n += gridDim.x * blockDim.x) {
    double value = x_in[n];
#pragma unroll 4
    for (int c = 0; c < columns; ++c) value += s_y[c] * basis[size_t(c) * count + n];
    x_out[n] = value;
  }
}

__global__ __launch_bounds__(kThreads) void k_commit(const double* __restrict__ x, double* __restrict__ solution,
                                                     unsigned count, Guard guard) {
  if (guard.skips()) return;
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < count; n += gridDim.x * blockDim.x) solution[n] = x[n];
}

}  // namespace

// Words of GmresWorkspace::arrivals: the orthogonalisation's counters, then
// those of each row of k_dot_batch's blocks.
size_t gmres_arrival_words(int m) { return (1 + size_t(m + kTile - 1) / kTile) * kCounters; }
// Blocks of both: more than four per CU only lengthen the last block's sum.
unsigned gmres_blocks(unsigned count, int cus) {
  return std::max(1u, std::min({(count + kThreads - 1) / kThreads, unsigned(cus > 0 ? cus : 256) * 4, kReduceBlocks}));
}
// Doubles of GmresWorkspace::partials: dots per block, norms per block, dots.
size_t gmres_partial_words(int m, unsigned blocks, unsigned tail_blocks) {
  return size_t(std::max(m, 2)) * std::max(blocks, tail_blocks) + blocks + size_t(m);
}
// Doubles of GmresWorkspace::state.
size_t gmres_state_words(int m) { return size_t(m) * (m + 1) + 4 * size_t(m) + 2 + kWords; }

int run_gmres(Context& ctx, int* converged_out, int* iterations_out, double* initial_out, double* residual_out,
              double* rhs_norm_out, double* relative_out) {
  return run_gmres_system(ctx, ctx.rhs, ctx.etheta, converged_out, iterations_out, initial_out, residual_out,
                          rhs_norm_out, relative_out);
}

int run_gmres_system(Context& ctx, const double* rhs_in, double* solution, int* converged_out, int* iterations_out,
                     double* initial_out, double* residual_out, double* rhs_norm_out, double* relative_out) {
  GmresWorkspace& w = ctx.gmres;
  hipStream_t st = ctx.stream;
  const unsigned n = w.count;
  const int m = ctx.num.restart;
  const SolverState s = solver_state(w, m, ctx.num.gmres_tol);
  const OperatorTailForm form = operator_tail_form(ctx);
  const unsigned tail_blocks = form.blocks;
  const unsigned rows = tail_blocks ? tail_blocks : w.blocks;  // partials per dot or norm
  double* const basis = w.basis;
  double* const norms = w.partials + size_t(std::max(m, 2)) * rows;
  double* const dots = norms + w.blocks;
  int rc = 0;
#define TPIC_TRY(expr, what)             \
  do {                                  \
    rc = check_hip(ctx, (expr), what);  \
    if (rc) return rc;                  \
  } while (0)
  // The first basis vector and the test of the residual b - A x.
  auto residual = [&](const double* x, int first, Guard guard) -> int {
    OperatorCall call;
    call.guard = guard;
    if (tail_blocks) {
      call.epilogue = OperatorEpilogue::residual;
      call.tail.rhs = rhs_in;
      call.tail.partials = w.partials;
      if (int e = launch_operator(ctx, x, basis, call)) return e;
    } else {
      if (int e = launch_operator(ctx, x, w.image, call)) return e;
      k_residual<<<w.blocks, kThreads, 0, st>>>(rhs_in, w.image, basis, w.partials, n, guard);
      if (int e = check_hip(ctx, hipGetLastError(), "gmres residual")) return e;
    }
    k_residual_test<<<1, kThreads, 0, st>>>(w.partials, rows, s, first, guard);
    return check_hip(ctx, hipGetLastError(), "gmres residual test");
  };
  auto arnoldi = [&](int col, bool last) -> int {
    const Guard running{s.word + kStop, 1.0};
    OperatorCall call;
    call.scale = s.scale + col;
    call.guard = running;
    if (tail_blocks) {
      call.epilogue = OperatorEpilogue::dots;
      call.tail.basis = basis;
      call.tail.columns = unsigned(col + 1);
      call.tail.partials = w.partials;
      call.tail.dots = dots;
      call.tail.arrivals = w.arrivals + kCounters;
    }
    if (int e = launch_operator(ctx, basis + size_t(col) * n, w.image, call)) return e;
    if (!tail_blocks) {
      const dim3 dgrid(w.blocks, unsigned((col + 1 + kTile - 1) / kTile));
      k_dot_batch<<<dgrid, kThreads, 0, st>>>(basis, w.image, w.partials, dots, w.arrivals + kCounters, n, unsigned(col + 1),
                                              running);
      if (int e = check_hip(ctx, hipGetLastError(), "gmres dots")) return e;
    }
    k_orthogonalize<<<w.blocks, kThreads, 0, st>>>(basis, w.image, basis + size_t(col + 1) * n,
                                                   form.finishes_dots ? dots : w.partials,
                                                   form.finishes_dots ? 1u : rows, norms,
                                                   w.arrivals, n, col, last ? 1 : 0, s, running);
    return check_hip(ctx, hipGetLastError(), "gmres orthogonalize");
  };
  // A restart's end, done once its stop word is up: update, true residual
  // (into the next restart's first basis vector), commit.
  auto finish = [&](const double* x) -> int {
    const Guard going{s.word + kGo, 0.0};
    k_update<<<w.blocks, kThreads, 0, st>>>(basis, x, w.x, n, s, going);
    if (int e = check_hip(ctx, hipGetLastError(), "gmres update")) return e;
    if (int e = residual(w.x, 0, going)) return e;
    k_commit<<<w.blocks, kThreads, 0, st>>>(w.x, solution, n, Guard{s.word + kCommit, 0.0});
    return check_hip(ctx, hipGetLastError(), "gmres commit");
  };
  phase_begin(ctx, Phase::solve);
  if ((rc = residual(solution, 1, Guard{}))) return rc;
  // Steps enqueued before the next read of the words, after `done` of this
  // solve: up to those that the operator's last solve took, then half as many
  // again. A step past the stop costs its launches (3.6 us each at 16^3; with
  // ten smoothing passes 23 of them), a read the time to refill the queue, and
  // the solves of a run change their steps slowly. With eight steps to every
  // read, a solve of two steps with ten passes at 16^3 took 1014 us, now 500
  // (one step to a read: 600), and a guess that met the tolerance 128, now 27
  // (a read of its own: 70); without smoothing two steps took 118, now 78.
  // Solves of one and two steps in turn, each expecting the other's: 97 us (110
  // with eight to a read), with ten passes 475 (one to a read: 425 to 545).
  int& expected = w.expected[ctx.transposed_operator ? 1 : 0];
  const auto batch = [&](int done, bool first) {
    if (done < expected) return std::min(kStepsPerRead, expected - done);
    return first ? 0 : std::min(kStepsPerRead, std::max(ctx.num.smoothing ? 1 : 2, done / 2));
  };
  bool converged = false, first_read = true;
  int iterations = 0, enqueued = 0, tails = 0;
  double word[kWords];
  while (!converged && iterations < ctx.num.max_iterations) {
    const int columns = std::min(m, ctx.num.max_iterations - iterations);
    const int upto = std::min(columns, enqueued + batch(iterations + enqueued, first_read));
    for (int col = enqueued; col < upto; ++col)
      if ((rc = arnoldi(col, col + 1 == columns))) return rc;
    enqueued = upto;
    if (enqueued && (rc = finish(tails ? w.x : solution))) return rc;
    TPIC_TRY(hipMemcpyAsync(w.controls, s.word, kWords * sizeof(double), hipMemcpyDeviceToHost, st),
             "gmres readback");
    TPIC_TRY(hipStreamSynchronize(st), "gmres readback");
    for (int k = 0; k < kWords; ++k) word[k] = w.controls[k];
    if (first_read && (!std::isfinite(word[kInitial2]) || !std::isfinite(word[kRhs2])))
      return fail(ctx, -3, "GMRES: nonfinite initial residual");
    first_read = false;
    if (word[kNonfinite] != 0.0) return fail(ctx, -3, "GMRES: nonfinite Arnoldi recurrence");
    converged = word[kConverged] != 0.0;
    if (int(word[kTails]) == tails) continue;  // converged from the start, or the restart goes on
    tails = int(word[kTails]);
    iterations += int(word[kDone]);
    enqueued = 0;
    if (!std::isfinite(word[kResidual2])) return fail(ctx, -3, "GMRES: nonfinite residual");
    if (word[kDoneBreakdown] != 0.0) break;
  }
  phase_end(ctx, Phase::solve);
  expected = iterations;
  const double res = std::sqrt(word[kResidual2]), rhs_norm = std::sqrt(word[kRhs2]);
  *converged_out = converged ? 1 : 0;
  *iterations_out = iterations;
  *initial_out = std::sqrt(word[kInitial2]);
  *residual_out = res;
  *rhs_norm_out = rhs_norm;
  *relative_out = res / (rhs_norm == 0.0 ? 1.0 : rhs_norm);
  return 0;
#undef TPIC_TRY
}

}  // namespace tpic_mi
