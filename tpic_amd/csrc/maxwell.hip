// Implicit Maxwell operator, right-hand side and field advance on one GPU
// (compact node/cell vectors; periodic neighbours by index wrap, closed walls
// by signed ghost images, constrained rows and dual-volume row scales).
//
//   rhs  = 1*E + delta*curl_C2N(B) - k*J                 (maxwell_device.hpp:152-171)
//   A(v) = 1*v + delta^2*curl_C2N(curl_N2C v) + k*(1/V)*M v  (:353-433, mass apply
//          mass_matrix_stencil.hpp:120-149: centre, 13 forward and 13 backward
//          blocks, backward blocks not transposed)
//   E'   = (1/th) E_th + (-(1-th)/th) E;  B' = 1*B + (-c dt) curl_N2C(E_th)
//                                                        (field_update_device.hpp:25-78)
//   Bn   = cell_to_node_average(B)                      (cell_to_node.hpp:19-32)
// with delta = c*th*dt and k = 4*pi*th*dt. Curls average four edge differences
// with the factor 1/4 in the reference's order (node_cell_curl.hpp:60-119).
//
// The operator is two kernels: the node->cell curl (24 B per cell) and one
// fused node kernel doing the cell->node curl, the 27-block mass product from
// the entry-major matrix (coalesced: neighbouring nodes read neighbouring
// words) and the three-term combination. Bound: HBM, 1008 B of matrix per node.
#include "internal.hpp"
#include "arrival.hpp"
#include "../../include/tpic_mi.h"

namespace tpic_mi {
namespace {

constexpr unsigned kThreads = 256;

struct Samples {
  double base, x, y, z, xy, xz, yz, xyz;
};

// Node sources: difference = neighbour - anchor; cell sources: anchor - neighbour.
template <bool NodeSource>
__device__ __forceinline__ double diff(double anchor, double neighbour) {
  return NodeSource ? neighbour - anchor : anchor - neighbour;
}

template <bool NodeSource>
__device__ __forceinline__ double derivative(const Samples& s, int axis, double inverse) {
  double sum;
  if (axis == 0)
    sum = diff<NodeSource>(s.base, s.x) + diff<NodeSource>(s.z, s.xz) + diff<NodeSource>(s.y, s.xy) +
          diff<NodeSource>(s.yz, s.xyz);
  else if (axis == 1)
    sum = diff<NodeSource>(s.base, s.y) + diff<NodeSource>(s.z, s.yz) + diff<NodeSource>(s.x, s.xy) +
          diff<NodeSource>(s.xz, s.xyz);
  else
    sum = diff<NodeSource>(s.base, s.z) + diff<NodeSource>(s.x, s.xz) + diff<NodeSource>(s.y, s.yz) +
          diff<NodeSource>(s.xy, s.xyz);
  return 0.25 * inverse * sum;
}

template <bool NodeSource>
__device__ __forceinline__ void curl_of(const Samples* s, const Grid& g, double& x, double& y, double& z) {
  x = derivative<NodeSource>(s[2], 1, g.iy) - derivative<NodeSource>(s[1], 2, g.iz);
  y = derivative<NodeSource>(s[0], 2, g.iz) - derivative<NodeSource>(s[2], 0, g.ix);
  z = derivative<NodeSource>(s[1], 0, g.ix) - derivative<NodeSource>(s[0], 1, g.iy);
}

// The 8 nodes of cell (i,j,k), all interior (no wrap needed).
__device__ __forceinline__ void load_cell_nodes(const Grid& g, const double* __restrict__ v, int i, int j, int k,
                                                Samples (&s)[3]) {
  const unsigned nodes = g.nodes();
  const unsigned sy = unsigned(g.nx + 1), sz = sy * unsigned(g.ny + 1);
  const unsigned n0 = g.node(i, j, k);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double* f = v + size_t(c) * nodes;
    s[c].base = f[n0];
    s[c].x = f[n0 + 1];
    s[c].y = f[n0 + sy];
    s[c].z = f[n0 + sz];
    s[c].xy = f[n0 + sy + 1];
    s[c].xz = f[n0 + sz + 1];
    s[c].yz = f[n0 + sz + sy];
    s[c].xyz = f[n0 + sz + sy + 1];
  }
}

__device__ __forceinline__ void n2c_at(const Grid& g, const double* __restrict__ v, int i, int j, int k, double& x,
                                       double& y, double& z) {
  Samples s[3];
  load_cell_nodes(g, v, i, j, k, s);
  curl_of<true>(s, g, x, y, z);
}

// Node (i,j,k) from its 8 cells: periodic wrap, or with Walls the wall
// ghosts (the interior image times the B-like ghost sign of each crossed
// face, field_boundary_device.hpp:26-57).
template <bool Walls>
__device__ __forceinline__ void c2n_at(const Grid& g, const double* __restrict__ b, int i, int j, int k, double& x,
                                       double& y, double& z) {
  const unsigned cells = g.cells();
  Samples s[3];
  if constexpr (!Walls) {
    const int i0 = wrap_cell(i, g.nx), i1 = wrap_cell(i - 1, g.nx);
    const int j0 = wrap_cell(j, g.ny), j1 = wrap_cell(j - 1, g.ny);
    const int k0 = wrap_cell(k, g.nz), k1 = wrap_cell(k - 1, g.nz);
    const unsigned at[8] = {g.cell(i0, j0, k0), g.cell(i1, j0, k0), g.cell(i0, j1, k0), g.cell(i0, j0, k1),
                            g.cell(i1, j1, k0), g.cell(i1, j0, k1), g.cell(i0, j1, k1), g.cell(i1, j1, k1)};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double* f = b + size_t(c) * cells;
      s[c].base = f[at[0]];
      s[c].x = f[at[1]];
      s[c].y = f[at[2]];
      s[c].z = f[at[3]];
      s[c].xy = f[at[4]];
      s[c].xz = f[at[5]];
      s[c].yz = f[at[6]];
      s[c].xyz = f[at[7]];
    }
  } else {
    int fi0, fi1, fj0, fj1, fk0, fk1;
    const int i0 = cell_image(g, 0, i, g.nx, fi0), i1 = cell_image(g, 0, i - 1, g.nx, fi1);
    const int j0 = cell_image(g, 1, j, g.ny, fj0), j1 = cell_image(g, 1, j - 1, g.ny, fj1);
    const int k0 = cell_image(g, 2, k, g.nz, fk0), k1 = cell_image(g, 2, k - 1, g.nz, fk1);
    const unsigned at[8] = {g.cell(i0, j0, k0), g.cell(i1, j0, k0), g.cell(i0, j1, k0), g.cell(i0, j0, k1),
                            g.cell(i1, j1, k0), g.cell(i1, j0, k1), g.cell(i0, j1, k1), g.cell(i1, j1, k1)};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double* f = b + size_t(c) * cells;
      s[c].base = b_ghost_sign(g, c, fi0, fj0, fk0) * f[at[0]];
      s[c].x = b_ghost_sign(g, c, fi1, fj0, fk0) * f[at[1]];
      s[c].y = b_ghost_sign(g, c, fi0, fj1, fk0) * f[at[2]];
      s[c].z = b_ghost_sign(g, c, fi0, fj0, fk1) * f[at[3]];
      s[c].xy = b_ghost_sign(g, c, fi1, fj1, fk0) * f[at[4]];
      s[c].xz = b_ghost_sign(g, c, fi1, fj0, fk1) * f[at[5]];
      s[c].yz = b_ghost_sign(g, c, fi0, fj1, fk1) * f[at[6]];
      s[c].xyz = b_ghost_sign(g, c, fi1, fj1, fk1) * f[at[7]];
    }
  }
  curl_of<false>(s, g, x, y, z);
}

__global__ __launch_bounds__(kThreads) void k_curl_n2c(Grid g, const double* __restrict__ v,
                                                       double* __restrict__ out, Guard guard) {
  if (guard.skips()) return;
  const unsigned cells = g.cells();
  for (unsigned c = blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += gridDim.x * blockDim.x) {
    const int i = int(c % unsigned(g.nx)), j = int((c / unsigned(g.nx)) % unsigned(g.ny)),
              k = int(c / (unsigned(g.nx) * unsigned(g.ny)));
    double x, y, z;
    n2c_at(g, v, i, j, k, x, y, z);
    out[c] = x;
    out[cells + c] = y;
    out[2 * size_t(cells) + c] = z;
  }
}

// curl_C2N of a cell vector at every node (periodic wrap).
__global__ __launch_bounds__(kThreads) void k_curl_c2n(Grid g, const double* __restrict__ b,
                                                       double* __restrict__ out) {
  const unsigned nodes = g.nodes();
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1);
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < nodes; n += gridDim.x * blockDim.x) {
    const int i = int(n % sx), j = int((n / sx) % sy), k = int(n / (sx * sy));
    double x, y, z;
    c2n_at<false>(g, b, i, j, k, x, y, z);
    out[n] = x;
    out[nodes + n] = y;
    out[2 * size_t(nodes) + n] = z;
  }
}

template <bool Walls>
__global__ __launch_bounds__(kThreads) void k_cell_to_node(Grid g, const double* __restrict__ b,
                                                           double* __restrict__ out) {
  const unsigned nodes = g.nodes(), cells = g.cells();
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1);
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < nodes; n += gridDim.x * blockDim.x) {
    const int i = int(n % sx), j = int((n / sx) % sy), k = int(n / (sx * sy));
    if constexpr (!Walls) {
      const int i0 = wrap_cell(i - 1, g.nx), i1 = wrap_cell(i, g.nx);
      const int j0 = wrap_cell(j - 1, g.ny), j1 = wrap_cell(j, g.ny);
      const int k0 = wrap_cell(k - 1, g.nz), k1 = wrap_cell(k, g.nz);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double* f = b + size_t(c) * cells;
        out[size_t(c) * nodes + n] = (f[g.cell(i0, j0, k0)] + f[g.cell(i1, j0, k0)] + f[g.cell(i0, j1, k0)] +
                                      f[g.cell(i1, j1, k0)] + f[g.cell(i0, j0, k1)] + f[g.cell(i1, j0, k1)] +
                                      f[g.cell(i0, j1, k1)] + f[g.cell(i1, j1, k1)]) *
                                     0.125;
      }
    } else {
      int fi0, fi1, fj0, fj1, fk0, fk1;
      const int i0 = cell_image(g, 0, i - 1, g.nx, fi0), i1 = cell_image(g, 0, i, g.nx, fi1);
      const int j0 = cell_image(g, 1, j - 1, g.ny, fj0), j1 = cell_image(g, 1, j, g.ny, fj1);
      const int k0 = cell_image(g, 2, k - 1, g.nz, fk0), k1 = cell_image(g, 2, k, g.nz, fk1);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double* f = b + size_t(c) * cells;
        out[size_t(c) * nodes + n] =
            (b_ghost_sign(g, c, fi0, fj0, fk0) * f[g.cell(i0, j0, k0)] +
             b_ghost_sign(g, c, fi1, fj0, fk0) * f[g.cell(i1, j0, k0)] +
             b_ghost_sign(g, c, fi0, fj1, fk0) * f[g.cell(i0, j1, k0)] +
             b_ghost_sign(g, c, fi1, fj1, fk0) * f[g.cell(i1, j1, k0)] +
             b_ghost_sign(g, c, fi0, fj0, fk1) * f[g.cell(i0, j0, k1)] +
             b_ghost_sign(g, c, fi1, fj0, fk1) * f[g.cell(i1, j0, k1)] +
             b_ghost_sign(g, c, fi0, fj1, fk1) * f[g.cell(i0, j1, k1)] +
             b_ghost_sign(g, c, fi1, fj1, fk1) * f[g.cell(i1, j1, k1)]) *
            0.125;
      }
    }
  }
}

// Zero the constrained rows of a node vector (enqueue_constrained_rows
// without input, field_boundary_device.hpp:60-120).
__global__ __launch_bounds__(kThreads) void k_zero_constrained(Grid g, double* __restrict__ v) {
  const unsigned nodes = g.nodes();
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1);
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < nodes; n += gridDim.x * blockDim.x) {
    const int i = int(n % sx), j = int((n / sx) % sy), k = int(n / (sx * sy));
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (g.constrained_row(c, i, j, k)) v[size_t(c) * nodes + n] = 0.0;
  }
}

// ---- energy-conserving smoothing ------------------------------------------
// One pass of the node stencil (node_smoothing_value, include/tpic/ecsim/
// fields/node_smoothing.hpp:27-58; node_smoothing_kernel,
// node_smoothing_device.hpp:20-41) at every node, reading neighbours through
// E-like ghosts: the periodic image, or on a wall axis the reflection through
// the wall node, negated where the face constrains the component (an odd
// ghost, boundary_conditions.hpp:56-72; field_boundary_device.hpp:26-57). A
// corner ghost carries the product of its faces' signs. Sums run in the
// reference's order: the six faces, the twelve edges, the eight corners, each
// left to right.
// MaxwellOperator::complete_smoothing (maxwell_device.hpp:452-490) projects
// the source before the first pass (complete_electric_refresh, :114-121, or
// the input projection of begin_apply_input, :270-272) and every pass's
// result: each pass here reads the source with its constrained rows as zero
// and writes its result with them zeroed, so S = P (pass P)^n.
constexpr int kFace7 = TPIC_MI_SMOOTH_FACE7, kBinomial27 = TPIC_MI_SMOOTH_BINOMIAL27;

// The E-like images of the neighbours i - 1, i, i + 1 along one axis: the
// node index, and per component bit (1 << c) whether the image is negated
// (an odd ghost) or read as zero (a constrained row, the projected source).
struct AxisImages {
  int at[3];
  unsigned char negate[3], zero[3];
};

template <bool Walls>
__device__ __forceinline__ AxisImages axis_images(const Grid& g, int axis, int i, int n) {
  AxisImages r;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int x = i + d - 1;
    r.negate[d] = 0;
    r.zero[d] = 0;
    if (!Walls || !g.field_wall[axis]) {
      r.at[d] = wrap_node(x, n);
      continue;
    }
    int image = x;
    if (x < 0) {
      image = -x;
      r.negate[d] = g.constrained[2 * axis];
    } else if (x > n) {
      image = 2 * n - x;
      r.negate[d] = g.constrained[2 * axis + 1];
    }
    r.at[d] = image;
    r.zero[d] = image == 0 ? g.constrained[2 * axis] : (image == n ? g.constrained[2 * axis + 1] : 0);
  }
  return r;
}

template <int Op, bool Walls>
__global__ __launch_bounds__(kThreads) void k_smooth(Grid g, const double* __restrict__ src,
                                                     double* __restrict__ dst, double alpha, double beta,
                                                     unsigned* __restrict__ validation, Guard guard) {
  if (guard.skips()) return;
  const unsigned nodes = g.nodes();
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1);
  unsigned flags = 0;
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < nodes; n += gridDim.x * blockDim.x) {
    const int i = int(n % sx), j = int((n / sx) % sy), k = int(n / (sx * sy));
    // The images are computed once per node and shared by the components.
    const AxisImages ax = axis_images<Walls>(g, 0, i, g.nx), ay = axis_images<Walls>(g, 1, j, g.ny),
                     az = axis_images<Walls>(g, 2, k, g.nz);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double* f = src + size_t(c) * nodes;
      const unsigned bit = 1u << c;
      auto at = [&](int di, int dj, int dk) {
        const double v = f[unsigned(ax.at[di + 1]) + sx * (unsigned(ay.at[dj + 1]) + sy * unsigned(az.at[dk + 1]))];
        if (!Walls) return v;
        if ((ax.zero[di + 1] | ay.zero[dj + 1] | az.zero[dk + 1]) & bit) return 0.0;
        return ((ax.negate[di + 1] ^ ay.negate[dj + 1] ^ az.negate[dk + 1]) & bit) ? -v : v;
      };
      const double face = at(-1, 0, 0) + at(1, 0, 0) + at(0, -1, 0) + at(0, 1, 0) + at(0, 0, -1) + at(0, 0, 1);
      double value;
      if (Op == kFace7) {
        value = alpha * at(0, 0, 0) + beta * face;
      } else {
        const double edge = at(-1, -1, 0) + at(1, -1, 0) + at(-1, 1, 0) + at(1, 1, 0) + at(-1, 0, -1) +
                            at(1, 0, -1) + at(-1, 0, 1) + at(1, 0, 1) + at(0, -1, -1) + at(0, 1, -1) +
                            at(0, -1, 1) + at(0, 1, 1);
        const double corner = at(-1, -1, -1) + at(1, -1, -1) + at(-1, 1, -1) + at(1, 1, -1) + at(-1, -1, 1) +
                              at(1, -1, 1) + at(-1, 1, 1) + at(1, 1, 1);
        value = (8.0 * at(0, 0, 0) + 4.0 * face + 2.0 * edge + corner) * (1.0 / 64.0);
      }
      if (!finite_value(value)) flags |= kInvalidField;
      if (Walls && g.constrained_row(c, i, j, k)) value = 0.0;
      dst[size_t(c) * nodes + n] = value;
    }
  }
  if (flags) atomicOr(validation, flags);
}

// The right-hand side, and the solve's initial guess E^n with its constrained
// rows zeroed (enqueue_rhs_fields copies E into theta and projects it,
// maxwell_device.hpp:140-142): a field set with nonzero constrained rows
// still starts the solve in the constrained subspace.
template <bool Walls>
__global__ __launch_bounds__(kThreads) void k_rhs(Grid g, const double* __restrict__ e, const double* __restrict__ b,
                                                  const double* __restrict__ current, double delta,
                                                  double current_factor, double* __restrict__ rhs,
                                                  double* __restrict__ theta, unsigned* __restrict__ validation) {
  const unsigned nodes = g.nodes();
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1);
  unsigned flags = 0;
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < nodes; n += gridDim.x * blockDim.x) {
    const int i = int(n % sx), j = int((n / sx) % sy), k = int(n / (sx * sy));
    double cv[3];
    c2n_at<Walls>(g, b, i, j, k, cv[0], cv[1], cv[2]);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t at = size_t(c) * nodes + n;
      const double start = e[at];
      double value = 1.0 * start + delta * cv[c] + (-current_factor) * current[at];
      const bool held = Walls && g.constrained_row(c, i, j, k);
      if (held) value = 0.0;
      rhs[at] = value;
      theta[at] = held ? 0.0 : start;
      if (!finite_value(value)) flags |= kInvalidField;
    }
  }
  if (flags) atomicOr(validation, flags);
}

constexpr int c_offsets[kStencils][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {1, 1, 0},
                                         {1, -1, 0}, {1, 0, 1}, {1, 0, -1}, {0, 1, 1}, {0, 1, -1},
                                         {1, -1, 1}, {1, 1, -1}, {-1, 1, 1}, {1, 1, 1}};

// image = 1*v + d2*curl_C2N(curl_cells) + k*(1/V)*M v at every interior node.
// M is read in its storage type (double, or float for the mixed forms); the
// products and sums are FP64.
// Rows per traversal tile of the operator apply (measured at 128^3: 16 and
// 32 rows are 6% faster than plane order for the FP64 matrix, 4% for FP32).
constexpr unsigned kApplyTileRows = 16;

// Node images of the neighbours of a node along each axis (offsets -1, 0,
// +1): on a wall axis the reflection through the wall node, else the periodic
// image.
struct NodeImages {
  int x[3], y[3], z[3];
};

template <bool Walls>
__device__ __forceinline__ NodeImages node_images(const Grid& g, int i, int j, int k) {
  NodeImages m;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    m.x[d] = d == 1 ? i : (Walls ? node_image(g, 0, i + d - 1, g.nx) : wrap_node(i + d - 1, g.nx));
    m.y[d] = d == 1 ? j : (Walls ? node_image(g, 1, j + d - 1, g.ny) : wrap_node(j + d - 1, g.ny));
    m.z[d] = d == 1 ? k : (Walls ? node_image(g, 2, k + d - 1, g.nz) : wrap_node(k + d - 1, g.nz));
  }
  return m;
}

// The vertex of a node and the vertex strides of its axes. Along an axis of
// one cell all four stored vertices are images of vertex 0 (the assembly sums
// the same cells in the same order for each), so the axis is read at vertex 0
// alone: the matrix of a plane is one plane's records, not four (the apply of
// a 512 x 512 x 1 grid took 179 us through all the images).
struct VertexWalk {
  int v0, sx, sy, sz;
};

__device__ __forceinline__ VertexWalk vertex_walk(const Grid& g, int i, int j, int k) {
  VertexWalk w;
  w.sx = g.nx == 1 ? 0 : 1;
  w.sy = g.ny == 1 ? 0 : g.nx + 3;
  w.sz = g.nz == 1 ? 0 : (g.nx + 3) * (g.ny + 3);
  w.v0 = int(g.vertex(g.nx == 1 ? 0 : i, g.ny == 1 ? 0 : j, g.nz == 1 ? 0 : k));
  return w;
}

// Stencils First .. Last - 1 of M v at a node: per stencil the forward block
// times v(i + o) and the backward block of the neighbour vertex (not
// transposed) times v(i - o); stencil 0 is the centre block alone. FP64
// products and sums. With Transposed every 3 x 3 block enters transposed: the
// mass part of the adjoint operator (the backward blocks are the forward
// pair's, not transposed, so M^T needs the transpose of every block). The
// values are loaded in one go and multiplied in another.
template <class MassT, bool Transposed, int First, int Last>
struct MassStencils {
  static constexpr int kBlocks = 2 * (Last - First) - (First == 0 ? 1 : 0);
  double a[kBlocks][3];
  MassT b[kBlocks][9];

  __device__ __forceinline__ void load_block(int t, const Grid& g, const double* __restrict__ v,
                                             const MassT* __restrict__ at, unsigned node) {
    const unsigned nodes = g.nodes();
    const size_t vs = g.vstride;
#pragma unroll
    for (int e = 0; e < 9; ++e) b[t][e] = at[size_t(e) * vs];
#pragma unroll
    for (int c = 0; c < 3; ++c) a[t][c] = v[size_t(c) * nodes + node];
  }

  __device__ __forceinline__ void load(const Grid& g, const double* __restrict__ v, const MassT* __restrict__ mass,
                                       const NodeImages& im, const VertexWalk& w) {
    int t = 0;
#pragma unroll
    for (int s = First; s < Last; ++s) {
      const int ox = c_offsets[s][0], oy = c_offsets[s][1], oz = c_offsets[s][2];
      const MassT* rows = mass + size_t(s) * 9 * g.vstride + w.v0;
      load_block(t++, g, v, rows, g.node(im.x[1 + ox], im.y[1 + oy], im.z[1 + oz]));
      if (s != 0)
        load_block(t++, g, v, rows - (ox * w.sx + oy * w.sy + oz * w.sz),
                   g.node(im.x[1 - ox], im.y[1 - oy], im.z[1 - oz]));
    }
  }

  __device__ __forceinline__ void add(double (&m)[3]) const {
#pragma unroll
    for (int t = 0; t < kBlocks; ++t)
#pragma unroll
      for (int r = 0; r < 3; ++r)
        m[r] += a[t][0] * double(b[t][Transposed ? r : 3 * r]) +
                a[t][1] * double(b[t][Transposed ? 3 + r : 3 * r + 1]) +
                a[t][2] * double(b[t][Transposed ? 6 + r : 3 * r + 2]);
  }
};

// Stencils First and on, one after the other.
template <class MassT, bool Transposed, int First>
__device__ __forceinline__ void add_stencils(const Grid& g, const double* __restrict__ v,
                                             const MassT* __restrict__ mass, const NodeImages& im,
                                             const VertexWalk& w, double (&m)[3]) {
  MassStencils<MassT, Transposed, First, First + 1> one;
  one.load(g, v, mass, im, w);
  one.add(m);
  if constexpr (First + 1 < kStencils) add_stencils<MassT, Transposed, First + 1>(g, v, mass, im, w, m);
}

// (1/V) f_g (M v) at node (i, j, kk).
template <class MassT, bool Walls, bool Transposed = false>
__device__ __forceinline__ void mass_rows(const Grid& g, const double* __restrict__ v,
                                          const MassT* __restrict__ mass, double inverse_volume, int i, int j,
                                          int kk, double& mx, double& my, double& mz) {
  double m[3] = {0.0, 0.0, 0.0};
  add_stencils<MassT, Transposed, 0>(g, v, mass, node_images<Walls>(g, i, j, kk), vertex_walk(g, i, j, kk), m);
  // mass_matrix_apply_device.hpp:34-35: the row scale (1/V) f_g.
  const double row_scale = Walls ? inverse_volume * double(g.dual_factor(i, j, kk)) : inverse_volume;
  mx = m[0] * row_scale;
  my = m[1] * row_scale;
  mz = m[2] * row_scale;
}

// Stages of k_apply: the fused image; with smoothing, the mass response
// (1/V) f_g M v alone (enqueue_mass_response), then the combination with the
// smoothed response (combine_image, maxwell_device.hpp:419-433).
constexpr int kFused = 0, kMassResponse = 1, kCombine = 2;

// What a kernel does with the image in its registers (OperatorTail).
constexpr int kPlain = 0, kDots = 1, kResidual = 2;

// The end of an operator kernel whose threads hold the images of N nodes each:
// stores them, or what `Epilogue` makes of them. Every thread of the block
// comes along; one that is not `present` holds a copy of another's nodes.
template <int Epilogue, int N>
__device__ __forceinline__ void finish_image(const double (&image)[N][3], const unsigned (&at)[N], bool present,
                                             unsigned nodes, double* __restrict__ out, const OperatorTail& tail) {
  if constexpr (Epilogue == kResidual) {
    __shared__ double s_norm[kThreads / 64][2];
    double r2 = 0.0, b2 = 0.0;
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const size_t n = size_t(c) * nodes + at[t];
        const double b = tail.rhs[n], r = b - image[t][c];
        if (present) out[n] = r;
        r2 += r * r;
        b2 += b * b;
      }
    r2 = wave_sum(present ? r2 : 0.0);
    b2 = wave_sum(present ? b2 : 0.0);
    if ((threadIdx.x & 63u) == 0) {
      s_norm[threadIdx.x >> 6][0] = r2;
      s_norm[threadIdx.x >> 6][1] = b2;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      double total = 0.0;
      for (unsigned w = 0; w < kThreads / 64; ++w) total += s_norm[w][threadIdx.x];
      tail.partials[size_t(threadIdx.x) * gridDim.x + blockIdx.x] = total;
    }
  } else {
    if (present)
#pragma unroll
      for (int t = 0; t < N; ++t)
#pragma unroll
        for (int c = 0; c < 3; ++c) out[size_t(c) * nodes + at[t]] = image[t][c];
  }
  if constexpr (Epilogue == kDots) {
    __shared__ double s_dot[kThreads / 64][64];
    __shared__ bool s_last;
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (unsigned col = 0; col < tail.columns; ++col) {
      const double* w = tail.basis + 3 * size_t(col) * nodes;
      double v = 0.0;
#pragma unroll
      for (int t = 0; t < N; ++t)
#pragma unroll
        for (int c = 0; c < 3; ++c) v += w[size_t(c) * nodes + at[t]] * image[t][c];
      v = wave_sum(present ? v : 0.0);
      if (lane == 0) s_dot[wave][col] = v;
    }
    __syncthreads();
    // Wave 0 stores the block's partials (at most 64 columns).
    if (threadIdx.x < tail.columns) {
      double total = 0.0;
      for (unsigned w = 0; w < kThreads / 64; ++w) total += s_dot[w][threadIdx.x];
      put_partial(tail.partials + size_t(threadIdx.x) * gridDim.x + blockIdx.x, total);
    }
    if (!last_to_arrive(tail.arrivals, blockIdx.x, gridDim.x, &s_last)) return;
    for (unsigned col = wave; col < tail.columns; col += kThreads / 64) {
      double total = 0.0;
      for (unsigned b = lane; b < gridDim.x; b += 64) total += get_partial(tail.partials + size_t(col) * gridDim.x + b);
      total = wave_sum(total);
      if (lane == 0) tail.dots[col] = total;
    }
  }
}

// A node per thread. With an epilogue (grids of at most kMaxBlocks blocks) a
// block goes on to what the solver reads the image for: kDots forms its
// products with `columns` basis vectors, the last block to arrive adding the
// blocks' parts, and kResidual writes rhs - image instead of the image and the
// block's parts of its squared norm and of rhs's. As a launch of their own
// the dots took 12 us at 100,000 nodes, the residual 5.
template <class MassT, bool Walls, int Stage, bool Transposed, int Epilogue>
__global__ __launch_bounds__(kThreads) void k_apply(Grid g, const double* __restrict__ v,
                                                    const double* __restrict__ curl_cells,
                                                    const MassT* __restrict__ mass,
                                                    const double* __restrict__ response, double d2, double k,
                                                    double inverse_volume, double* __restrict__ out,
                                                    unsigned tile_rows, const double* __restrict__ scale,
                                                    OperatorTail tail, Guard guard) {
  // A launch of a GMRES step after the solver stopped does nothing.
  if (guard.skips()) return;
  const unsigned nodes = g.nodes();
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1), sz = unsigned(g.nz + 1);
  unsigned L = xcd_logical_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const bool present = L < nodes;
  if (!present) {
    if (Epilogue == kPlain) return;
    L = nodes - 1;  // the lane goes along to the block's sums
  }
  // Traversal: full x rows, grouped into tiles of tile_rows rows; a tile's
  // planes are visited in z order, so the blocks of the planes k - 1 and k of
  // a tile are close in time (within one XCD) and the backward reads of the
  // stencils with a z offset find the matrix lines in L2.
  const int i = int(L % sx);
  const unsigned row = L / sx;
  const unsigned full = sy / tile_rows, span = sz * tile_rows;
  int j, kk;
  if (row < full * span) {
    const unsigned t = row / span, rem = row % span;
    kk = int(rem / tile_rows);
    j = int(t * tile_rows + rem % tile_rows);
  } else {
    const unsigned last = sy - full * tile_rows, rem = row - full * span;
    kk = int(rem / last);
    j = int(full * tile_rows + rem % last);
  }
  const unsigned n = g.node(i, j, kk);
  const double* vx = v;
  const double* vy = v + nodes;
  const double* vz = v + 2 * size_t(nodes);
  double mx, my, mz;
  if (Stage == kCombine) {
    mx = response[n];
    my = response[nodes + n];
    mz = response[2 * size_t(nodes) + n];
  } else {
    mass_rows<MassT, Walls, Transposed>(g, v, mass, inverse_volume, i, j, kk, mx, my, mz);
  }
  double cx = 0, cy = 0, cz = 0;
  if (Stage != kMassResponse) c2n_at<Walls>(g, curl_cells, i, j, kk, cx, cy, cz);
  if (Stage == kMassResponse) {
    out[n] = mx;
    out[nodes + n] = my;
    out[2 * size_t(nodes) + n] = mz;
    return;
  }
  double ox = 1.0 * vx[n] + d2 * cx + k * mx;
  double oy = 1.0 * vy[n] + d2 * cy + k * my;
  double oz = 1.0 * vz[n] + d2 * cz + k * mz;
  if (Walls) {
    // Constrained image rows take the (projected) input rows.
    if (g.constrained_row(0, i, j, kk)) ox = vx[n];
    if (g.constrained_row(1, i, j, kk)) oy = vy[n];
    if (g.constrained_row(2, i, j, kk)) oz = vz[n];
  }
  if (scale) {
    const double by = *scale;
    ox *= by;
    oy *= by;
    oz *= by;
  }
  const double image[1][3] = {{ox, oy, oz}};
  const unsigned at[1] = {n};
  finish_image<Epilogue>(image, at, present, nodes, out, tail);
}

// The operator of a plane, one periodic cell deep (nz = 1, periodic fields): a
// thread takes both of a column's nodes. They read the same matrix blocks and
// the same four cells, and the same neighbours in the blocks with a z offset
// (-1 is node 0, +1 node 1 for both), so a pair costs little more than a
// node: 18 of the 27 products and the curl term are shared. 512 x 512 x 1 in
// FP64 reads 267 MB of blocks in 90 us where a thread per node took 126 (55 us
// at the rate of a copy).
template <class MassT, bool Transposed>
__device__ __forceinline__ void add_block(const MassT (&b)[9], const double (&a)[3], double (&m)[3]) {
#pragma unroll
  for (int r = 0; r < 3; ++r)
    m[r] += a[0] * double(b[Transposed ? r : 3 * r]) + a[1] * double(b[Transposed ? 3 + r : 3 * r + 1]) +
            a[2] * double(b[Transposed ? 6 + r : 3 * r + 2]);
}

// The stencil whose forward (ahead) or backward block couples a node to its
// neighbour at (x, y, z).
struct BlockOf {
  int stencil;
  bool ahead;
};
constexpr BlockOf block_of(int x, int y, int z) {
  for (int s = 0; s < kStencils; ++s) {
    if (c_offsets[s][0] == x && c_offsets[s][1] == y && c_offsets[s][2] == z) return {s, true};
    if (c_offsets[s][0] == -x && c_offsets[s][1] == -y && c_offsets[s][2] == -z) return {s, false};
  }
  return {0, true};
}

template <class MassT, int X, int Y, int Z>
__device__ __forceinline__ void load_plane_block(const Grid& g, const MassT* __restrict__ mass, const VertexWalk& w,
                                                 MassT (&b)[9]) {
  constexpr BlockOf of = block_of(X, Y, Z);
  const MassT* rows = mass + size_t(of.stencil) * 9 * g.vstride + (of.ahead ? w.v0 : w.v0 + X * w.sx + Y * w.sy);
#pragma unroll
  for (int e = 0; e < 9; ++e) b[e] = rows[size_t(e) * g.vstride];
}

// The three blocks of the neighbouring column at (X, Y), then the others of a
// 3 x 3 patch: the column's two values are loaded once for all three.
template <class MassT, bool Transposed, int Position>
__device__ __forceinline__ void plane_columns(const Grid& g, const double* __restrict__ v,
                                              const MassT* __restrict__ mass, const NodeImages& im,
                                              const VertexWalk& w, double (&shared)[3], double (&own)[2][3]) {
  constexpr int X = Position % 3 - 1, Y = Position / 3 - 1;
  const unsigned nodes = g.nodes(), upper = unsigned(g.nx + 1) * unsigned(g.ny + 1);
  const unsigned node = unsigned(im.x[1 + X]) + unsigned(g.nx + 1) * unsigned(im.y[1 + Y]);
  MassT below[9], level[9], above[9];
  load_plane_block<MassT, X, Y, -1>(g, mass, w, below);
  load_plane_block<MassT, X, Y, 0>(g, mass, w, level);
  load_plane_block<MassT, X, Y, 1>(g, mass, w, above);
  double a[2][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    a[0][c] = v[size_t(c) * nodes + node];
    a[1][c] = v[size_t(c) * nodes + node + upper];
  }
  add_block<MassT, Transposed>(below, a[0], shared);
  add_block<MassT, Transposed>(above, a[1], shared);
  add_block<MassT, Transposed>(level, a[0], own[0]);
  add_block<MassT, Transposed>(level, a[1], own[1]);
  // The sums are formed here: left to the compiler they sink past the next
  // columns' loads (256 registers and a wave per SIMD, here about 90 and five).
#pragma unroll
  for (int c = 0; c < 3; ++c) asm volatile("" : "+v"(shared[c]), "+v"(own[0][c]), "+v"(own[1][c]) : : "memory");
  if constexpr (Position < 8) plane_columns<MassT, Transposed, Position + 1>(g, v, mass, im, w, shared, own);
}

template <class MassT, bool Transposed, int Epilogue>
__global__ __launch_bounds__(kThreads) void k_apply_plane(Grid g, const double* __restrict__ v,
                                                          const double* __restrict__ curl_cells,
                                                          const MassT* __restrict__ mass, double d2, double k,
                                                          double inverse_volume, double* __restrict__ out,
                                                          const double* __restrict__ scale, OperatorTail tail,
                                                          Guard guard) {
  if (guard.skips()) return;
  const unsigned sx = unsigned(g.nx + 1), columns = sx * unsigned(g.ny + 1), nodes = g.nodes();
  unsigned n = xcd_logical_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const bool present = n < columns;
  if (!present) {
    if (Epilogue == kPlain) return;
    n = columns - 1;
  }
  const int i = int(n % sx), j = int(n / sx);
  const NodeImages im = node_images<false>(g, i, j, 0);
  double shared[3] = {0.0, 0.0, 0.0}, own[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
  plane_columns<MassT, Transposed, 0>(g, v, mass, im, vertex_walk(g, i, j, 0), shared, own);
  double cc[3];
  c2n_at<false>(g, curl_cells, i, j, 0, cc[0], cc[1], cc[2]);
  const double by = scale ? *scale : 1.0;
  const unsigned at[2] = {n, n + columns};
  double image[2][3];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      image[t][c] = (v[size_t(c) * nodes + at[t]] + d2 * cc[c] + k * (inverse_volume * (shared[c] + own[t][c]))) * by;
  finish_image<Epilogue>(image, at, present, nodes, out, tail);
}

// The operator on a grid too small to fill the chip with a thread per node:
// a block takes 64 nodes (a lane each) and its eight waves share the work of
// every node: two stencils of M and one of the eight cells around the node,
// whose curl is formed in place (no curl pass). Each wave loads all it needs
// (up to 36 matrix entries and 36 vector values a lane) before it multiplies,
// and the eight parts meet in LDS. At 16^3 a thread per node leaves 20 blocks,
// whose lanes wait for their 27 x 12 loads in many turns: 14.6 us, and 3.6 us
// for the curl pass before it.
constexpr unsigned kParts = 8;

// One cell's part of curl_C2N(curl_N2C v) at node (i, j, k): the cell at
// offset (-Ax, -Ay, -Az) from the node.
template <bool Walls, int Ax, int Ay, int Az>
struct CurlCell {
  Samples s[3];
  double sign[3];

  __device__ __forceinline__ void load(const Grid& g, const double* __restrict__ v, int i, int j, int k) {
    int ci, cj, ck;
    if constexpr (!Walls) {
      ci = wrap_cell(i - Ax, g.nx), cj = wrap_cell(j - Ay, g.ny), ck = wrap_cell(k - Az, g.nz);
    } else {
      int fx, fy, fz;
      ci = cell_image(g, 0, i - Ax, g.nx, fx), cj = cell_image(g, 1, j - Ay, g.ny, fy);
      ck = cell_image(g, 2, k - Az, g.nz, fz);
#pragma unroll
      for (int c = 0; c < 3; ++c) sign[c] = b_ghost_sign(g, c, fx, fy, fz);
    }
    load_cell_nodes(g, v, ci, cj, ck, s);
  }

  __device__ __forceinline__ void add(const Grid& g, double d2, double (&sum)[3]) const {
    constexpr double dx = Ax ? -0.25 : 0.25, dy = Ay ? -0.25 : 0.25, dz = Az ? -0.25 : 0.25;
    double b[3];
    curl_of<true>(s, g, b[0], b[1], b[2]);
    if constexpr (Walls)
#pragma unroll
      for (int c = 0; c < 3; ++c) b[c] *= sign[c];
    sum[0] += d2 * (dy * g.iy * b[2] - dz * g.iz * b[1]);
    sum[1] += d2 * (dz * g.iz * b[0] - dx * g.ix * b[2]);
    sum[2] += d2 * (dx * g.ix * b[1] - dy * g.iy * b[0]);
  }
};

// Wave `Part`'s share of the operator at a node: stencils 2 Part and
// 2 Part + 1 (the last two waves one each), weighted by `f`, and cell Part.
template <class MassT, bool Walls, int Stage, bool Transposed, int Part>
__device__ __forceinline__ void operator_share(const Grid& g, const double* __restrict__ v,
                                               const MassT* __restrict__ mass, double f, double d2, int i, int j,
                                               int k, double (&sum)[3]) {
  constexpr int kFirst = Part < 6 ? 2 * Part : Part + 6, kLast = Part < 6 ? kFirst + 2 : kFirst + 1;
  MassStencils<MassT, Transposed, kFirst, kLast> stencils;
  CurlCell<Walls, (Part & 1), ((Part >> 1) & 1), (Part >> 2)> cell;
  if constexpr (Stage != kCombine) stencils.load(g, v, mass, node_images<Walls>(g, i, j, k), vertex_walk(g, i, j, k));
  if constexpr (Stage != kMassResponse) cell.load(g, v, i, j, k);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (Stage != kCombine) {
    double m[3] = {0.0, 0.0, 0.0};
    stencils.add(m);
#pragma unroll
    for (int c = 0; c < 3; ++c) sum[c] = f * m[c];
  }
  if constexpr (Stage != kMassResponse) cell.add(g, d2, sum);
}

template <class MassT, bool Walls, int Stage, bool Transposed, int Epilogue>
__global__ __launch_bounds__(64 * kParts) __attribute__((amdgpu_waves_per_eu(2, 3))) void k_apply_split(Grid g, const double* __restrict__ v,
                                                             const MassT* __restrict__ mass,
                                                             const double* __restrict__ response, double d2, double k,
                                                             double inverse_volume, double* __restrict__ out,
                                                             const double* __restrict__ scale, OperatorTail tail,
                                                             Guard guard) {
  if (guard.skips()) return;
  __shared__ double s_part[kParts][3][64];
  const unsigned lane = threadIdx.x & 63u;
  const unsigned part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned nodes = g.nodes();
  const unsigned L = blockIdx.x * 64u + lane;
  const bool present = L < nodes;
  const unsigned n = present ? L : nodes - 1;
  const unsigned sx = unsigned(g.nx + 1), sy = unsigned(g.ny + 1);
  const int i = int(n % sx), j = int((n / sx) % sy), kk = int(n / (sx * sy));
  // The columns this wave multiplies, requested before the operator's loads.
  constexpr unsigned kAhead = 2;
  double ahead[kAhead][3];
  if constexpr (Epilogue == kDots) {
#pragma unroll
    for (unsigned t = 0; t < kAhead; ++t) {
      const unsigned col = part + t * kParts;
#pragma unroll
      for (int c = 0; c < 3; ++c)
        ahead[t][c] = col < tail.columns ? tail.basis[(3 * size_t(col) + c) * nodes + n] : 0.0;
    }
  }
  double f = inverse_volume;
  if (Walls) f *= double(g.dual_factor(i, j, kk));
  if (Stage == kFused) f *= k;
  double sum[3] = {0.0, 0.0, 0.0};
  switch (part) {
    case 0: operator_share<MassT, Walls, Stage, Transposed, 0>(g, v, mass, f, d2, i, j, kk, sum); break;
    case 1: operator_share<MassT, Walls, Stage, Transposed, 1>(g, v, mass, f, d2, i, j, kk, sum); break;
    case 2: operator_share<MassT, Walls, Stage, Transposed, 2>(g, v, mass, f, d2, i, j, kk, sum); break;
    case 3: operator_share<MassT, Walls, Stage, Transposed, 3>(g, v, mass, f, d2, i, j, kk, sum); break;
    case 4: operator_share<MassT, Walls, Stage, Transposed, 4>(g, v, mass, f, d2, i, j, kk, sum); break;
    case 5: operator_share<MassT, Walls, Stage, Transposed, 5>(g, v, mass, f, d2, i, j, kk, sum); break;
    case 6: operator_share<MassT, Walls, Stage, Transposed, 6>(g, v, mass, f, d2, i, j, kk, sum); break;
    default: operator_share<MassT, Walls, Stage, Transposed, 7>(g, v, mass, f, d2, i, j, kk, sum); break;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) s_part[part][c][lane] = sum[c];
  __syncthreads();
  double image[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    image[c] = ((s_part[0][c][lane] + s_part[1][c][lane]) + (s_part[2][c][lane] + s_part[3][c][lane])) +
               ((s_part[4][c][lane] + s_part[5][c][lane]) + (s_part[6][c][lane] + s_part[7][c][lane]));
  if constexpr (Stage != kMassResponse) {
    const double by = scale ? *scale : 1.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t at = size_t(c) * nodes + n;
      if (Stage == kCombine) image[c] += k * response[at];
      image[c] += v[at];
      // Constrained image rows take the (projected) input rows.
      if (Walls && g.constrained_row(c, i, j, kk)) image[c] = v[at];
      image[c] *= by;
    }
  }
  if constexpr (Epilogue == kResidual) {
    double r2 = 0.0, b2 = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double rhs = tail.rhs[size_t(c) * nodes + n];
      image[c] = rhs - image[c];
      r2 += image[c] * image[c];
      b2 += rhs * rhs;
    }
    const double total = wave_sum(present ? (part == 0 ? r2 : b2) : 0.0);
    if (part < 2 && lane == 0) tail.partials[size_t(part) * gridDim.x + blockIdx.x] = total;
  }
  if (part == 0 && present)
#pragma unroll
    for (int c = 0; c < 3; ++c) out[size_t(c) * nodes + n] = image[c];
  if constexpr (Epilogue == kDots) {
    auto dot = [&](unsigned col, const double (&w)[3]) {
      const double total = wave_sum(present ? w[0] * image[0] + w[1] * image[1] + w[2] * image[2] : 0.0);
      if (lane == 0) tail.partials[size_t(col) * gridDim.x + blockIdx.x] = total;
    };
#pragma unroll
    for (unsigned t = 0; t < kAhead; ++t)
      if (part + t * kParts < tail.columns) dot(part + t * kParts, ahead[t]);
    for (unsigned col = part + kAhead * kParts; col < tail.columns; col += kParts) {
      double w[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) w[c] = tail.basis[(3 * size_t(col) + c) * nodes + n];
      dot(col, w);
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_next_e(unsigned count, const double* __restrict__ etheta,
                                                     double* __restrict__ e, double c0, double c1, int copy,
                                                     unsigned* __restrict__ validation) {
  unsigned flags = 0;
  for (unsigned n = blockIdx.x * blockDim.x + threadIdx.x; n < count; n += gridDim.x * blockDim.x) {
    const double value = copy ? etheta[n] : c0 * etheta[n] + c1 * e[n];
    e[n] = value;
    if (!finite_value(value)) flags |= kInvalidField;
  }
  if (flags) atomicOr(validation, flags);
}

__global__ __launch_bounds__(kThreads) void k_faraday(Grid g, const double* __restrict__ etheta,
                                                      double* __restrict__ b, double faraday,
                                                      unsigned* __restrict__ validation) {
  const unsigned cells = g.cells();
  unsigned flags = 0;
  for (unsigned c = blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += gridDim.x * blockDim.x) {
    const int i = int(c % unsigned(g.nx)), j = int((c / unsigned(g.nx)) % unsigned(g.ny)),
              k = int(c / (unsigned(g.nx) * unsigned(g.ny)));
    double r[3];
    n2c_at(g, etheta, i, j, k, r[0], r[1], r[2]);
#pragma unroll
    for (int comp = 0; comp < 3; ++comp) {
      const size_t at = size_t(comp) * cells + c;
      const double value = 1.0 * b[at] + faraday * r[comp];
      b[at] = value;
      if (!finite_value(value)) flags |= kInvalidField;
    }
  }
  if (flags) atomicOr(validation, flags);
}

unsigned blocks_for(const Context& ctx, uint64_t work) {
  const uint64_t want = (work + kThreads - 1) / kThreads;
  const uint64_t cap = uint64_t(ctx.cus > 0 ? ctx.cus : 256) * 32;
  return unsigned(want < cap ? (want ? want : 1) : cap);
}

}  // namespace

int launch_cell_to_node(Context& ctx) {
  if (ctx.grid.walls)
    k_cell_to_node<true><<<blocks_for(ctx, ctx.grid.nodes()), kThreads, 0, ctx.stream>>>(ctx.grid, ctx.b, ctx.bn);
  else
    k_cell_to_node<false><<<blocks_for(ctx, ctx.grid.nodes()), kThreads, 0, ctx.stream>>>(ctx.grid, ctx.b, ctx.bn);
  return check_hip(ctx, hipGetLastError(), "cell to node");
}

int launch_zero_constrained(Context& ctx, double* v) {
  if (!ctx.grid.walls) return 0;
  k_zero_constrained<<<blocks_for(ctx, ctx.grid.nodes()), kThreads, 0, ctx.stream>>>(ctx.grid, v);
  return check_hip(ctx, hipGetLastError(), "constrained rows");
}

int launch_smooth(Context& ctx, const double* src, double* dst, const double** result, Guard guard) {
  const Grid& g = ctx.grid;
  const Numerics& k = ctx.num;
  if (!k.smoothing || !ctx.smooth_a || !ctx.smooth_b)
    return fail(ctx, TPIC_MI_INVALID_STATE, "smoothing is not active");
  double* buffers[2] = {ctx.smooth_a, ctx.smooth_b};
  int next = src == ctx.smooth_a ? 1 : 0;
  const double* from = src;
  const unsigned blocks = blocks_for(ctx, g.nodes());
  for (int pass = 0; pass < k.smooth_iterations; ++pass) {
    const bool last = pass + 1 == k.smooth_iterations;
    double* to = last && dst ? dst : buffers[next];
    if (k.smooth_operator == TPIC_MI_SMOOTH_FACE7 && g.walls)
      k_smooth<kFace7, true><<<blocks, kThreads, 0, ctx.stream>>>(g, from, to, k.smooth_alpha, k.smooth_beta,
                                                                 ctx.validation, guard);
    else if (k.smooth_operator == TPIC_MI_SMOOTH_FACE7)
      k_smooth<kFace7, false><<<blocks, kThreads, 0, ctx.stream>>>(g, from, to, k.smooth_alpha, k.smooth_beta,
                                                                  ctx.validation, guard);
    else if (g.walls)
      k_smooth<kBinomial27, true><<<blocks, kThreads, 0, ctx.stream>>>(
          g, from, to, k.smooth_alpha, k.smooth_beta, ctx.validation, guard);
    else
      k_smooth<kBinomial27, false><<<blocks, kThreads, 0, ctx.stream>>>(
          g, from, to, k.smooth_alpha, k.smooth_beta, ctx.validation, guard);
    if (int rc = check_hip(ctx, hipGetLastError(), "node smoothing")) return rc;
    from = to;
    next ^= 1;
  }
  *result = from;
  return 0;
}

int launch_rhs(Context& ctx) {
  // complete_rhs (maxwell_device.hpp:151-171): with smoothing the current
  // term is S(J).
  const double* current = ctx.current;
  if (ctx.num.smoothing)
    if (int rc = launch_smooth(ctx, ctx.current, nullptr, &current)) return rc;
  if (ctx.grid.walls)
    k_rhs<true><<<blocks_for(ctx, ctx.grid.nodes()), kThreads, 0, ctx.stream>>>(
        ctx.grid, ctx.e, ctx.b, current, ctx.delta, ctx.current_factor, ctx.rhs, ctx.etheta, ctx.validation);
  else
    k_rhs<false><<<blocks_for(ctx, ctx.grid.nodes()), kThreads, 0, ctx.stream>>>(
        ctx.grid, ctx.e, ctx.b, current, ctx.delta, ctx.current_factor, ctx.rhs, ctx.etheta, ctx.validation);
  return check_hip(ctx, hipGetLastError(), "rhs");
}

namespace {

// Grids up to this many nodes take k_apply_split, larger ones the curl pass
// and a thread per node, or per column of a plane.
constexpr unsigned kSplitNodes = 16384;

struct OperatorArgs {
  const Grid& g;
  hipStream_t stream;
  double d2, k, inverse_volume;
  const double* scale;
  Guard guard;
  OperatorTail tail;
};

template <class MassT, bool Walls, int Stage, bool Transposed, int Epilogue>
void split_kernel(const OperatorArgs& a, const double* in, const MassT* mass, const double* response, double* out) {
  k_apply_split<MassT, Walls, Stage, Transposed, Epilogue>
      <<<(a.g.nodes() + 63u) / 64u, 64 * kParts, 0, a.stream>>>(a.g, in, mass, response, a.d2, a.k, a.inverse_volume,
                                                                out, a.scale, a.tail, a.guard);
}

template <class MassT, bool Walls, int Stage, bool Transposed>
void split_stage(const OperatorArgs& a, int epilogue, const double* in, const MassT* mass, const double* response,
                 double* out) {
  if constexpr (Stage != kMassResponse) {  // whose image is not the operator's
    if (epilogue == kDots) return split_kernel<MassT, Walls, Stage, Transposed, kDots>(a, in, mass, response, out);
    if (epilogue == kResidual)
      return split_kernel<MassT, Walls, Stage, Transposed, kResidual>(a, in, mass, response, out);
  }
  split_kernel<MassT, Walls, Stage, Transposed, kPlain>(a, in, mass, response, out);
}

// Rows per traversal tile: kApplyTileRows, fewer where a row is so long that a
// tile's matrix records of one plane (16 rows at 128^3: 2.1 MB) would not
// stay in an XCD's L2 until the next plane reads them.
template <class MassT>
unsigned apply_tile_rows(const Grid& g) {
  const unsigned row_bytes = unsigned(g.nx + 3) * unsigned(kEntries * sizeof(MassT));
  const unsigned fit = std::max(1u, 2200000u / row_bytes);
  return std::min({kApplyTileRows, fit, unsigned(g.ny + 1)});
}

template <class MassT, bool Walls, int Stage, bool Transposed, int Epilogue>
void node_kernel(const OperatorArgs& a, const double* in, const double* curl, const MassT* mass,
                 const double* response, double* out) {
  const unsigned rows = apply_tile_rows<MassT>(a.g);
  k_apply<MassT, Walls, Stage, Transposed, Epilogue>
      <<<(a.g.nodes() + kThreads - 1) / kThreads, kThreads, 0, a.stream>>>(
          a.g, in, curl, mass, response, a.d2, a.k, a.inverse_volume, out, rows, a.scale, a.tail, a.guard);
}

// Grids whose thread takes a column's two nodes, where they are past
// k_apply_split: an operator call (curl included) at 92 x 92 x 1 takes 14 us and
// 16 with a thread per node, at 181 x 181 17 and 26, at 512 x 512 98 and 121 (in
// floats 12 and 12, 12 and 17, 57 and 74). Decks and tests lay a plane in x and
// y; one that is a cell deep in x or y has its columns' nodes apart and takes
// the general form, as do planes with walls, whose two nodes differ in images
// and signs (cycles of 256 x 256 cells with 64 a cell: 1.27 ms one cell deep in
// z, 1.39 in y, 1.95 in x).
bool plane_form(const Grid& g) { return g.nz == 1 && !g.walls; }

// Threads of the forms that take whole nodes or columns.
unsigned node_threads(const Grid& g, bool plane) {
  return plane ? unsigned(g.nx + 1) * unsigned(g.ny + 1) : g.nodes();
}

template <class MassT, bool Transposed, int Epilogue>
void plane_kernel(const OperatorArgs& a, const double* in, const double* curl, const MassT* mass, double* out) {
  k_apply_plane<MassT, Transposed, Epilogue>
      <<<(node_threads(a.g, true) + kThreads - 1) / kThreads, kThreads, 0, a.stream>>>(
          a.g, in, curl, mass, a.d2, a.k, a.inverse_volume, out, a.scale, a.tail, a.guard);
}

template <class MassT, bool Walls, int Stage, bool Transposed = false>
void node_stage(const OperatorArgs& a, int epilogue, const double* in, const double* curl, const MassT* mass,
                const double* response, double* out) {
  if constexpr (Stage == kFused && !Walls) {
    if (plane_form(a.g)) {
      if (epilogue == kDots) return plane_kernel<MassT, Transposed, kDots>(a, in, curl, mass, out);
      if (epilogue == kResidual) return plane_kernel<MassT, Transposed, kResidual>(a, in, curl, mass, out);
      return plane_kernel<MassT, Transposed, kPlain>(a, in, curl, mass, out);
    }
  }
  if constexpr (Stage != kMassResponse) {
    if (epilogue == kDots)
      return node_kernel<MassT, Walls, Stage, Transposed, kDots>(a, in, curl, mass, response, out);
    if (epilogue == kResidual)
      return node_kernel<MassT, Walls, Stage, Transposed, kResidual>(a, in, curl, mass, response, out);
  }
  node_kernel<MassT, Walls, Stage, Transposed, kPlain>(a, in, curl, mass, response, out);
}

// image = A in by either form. Walls and smoothing take the mass response by
// itself: smoothing between two passes of S (complete_apply_smoothed,
// maxwell_device.hpp:389-417: x = S(v), r = (1/V) f_g M x, y = S(r),
// image = 1*v + d2*curl_C2N(curl_cells) + k*y with the constrained rows of v);
// with walls a thread per node would hold the kernel that does both to one
// wave per SIMD (256 registers). The sums are those of the fused form.
template <class MassT, bool Walls>
int operator_image(Context& ctx, const OperatorArgs& a, bool split, int epilogue, const double* in, double* out) {
  const MassT* mass = static_cast<const MassT*>(ctx.mass);
  const double* const curl = ctx.gmres.curl_cells;
  const double* response = ctx.mass_response;
  if (ctx.num.smoothing) {
    const double* x = nullptr;
    if (int rc = launch_smooth(ctx, in, nullptr, &x, a.guard)) return rc;
    double* r = x == ctx.smooth_a ? ctx.smooth_b : ctx.smooth_a;
    OperatorArgs plain = a;
    plain.scale = nullptr;
    if (split)
      split_stage<MassT, Walls, kMassResponse, false>(plain, kPlain, x, mass, nullptr, r);
    else
      node_stage<MassT, Walls, kMassResponse>(plain, kPlain, x, nullptr, mass, nullptr, r);
    if (int rc = check_hip(ctx, hipGetLastError(), "mass response")) return rc;
    if (int rc = launch_smooth(ctx, r, nullptr, &response, a.guard)) return rc;
  } else if (Walls && !split) {
    if (!ctx.mass_response)
      return fail(ctx, TPIC_MI_INVALID_STATE, "walled operator without its mass response buffer");
    OperatorArgs plain = a;
    plain.scale = nullptr;
    node_stage<MassT, Walls, kMassResponse>(plain, kPlain, in, nullptr, mass, nullptr, ctx.mass_response);
    if (int rc = check_hip(ctx, hipGetLastError(), "walled mass response")) return rc;
  } else {
    if (split)
      split_stage<MassT, Walls, kFused, false>(a, epilogue, in, mass, nullptr, out);
    else if constexpr (!Walls)
      node_stage<MassT, Walls, kFused>(a, epilogue, in, curl, mass, nullptr, out);
    return check_hip(ctx, hipGetLastError(), "operator apply");
  }
  if (split)
    split_stage<double, Walls, kCombine, false>(a, epilogue, in, nullptr, response, out);
  else
    node_stage<double, Walls, kCombine>(a, epilogue, in, curl, nullptr, response, out);
  return check_hip(ctx, hipGetLastError(), "operator combination");
}

// The adjoint operator of a periodic box: curl-curl is symmetric over the
// unique nodes, the mass blocks enter transposed.
template <class MassT>
int transposed_image(Context& ctx, const OperatorArgs& a, bool split, int epilogue, const double* in, double* out) {
  const MassT* mass = static_cast<const MassT*>(ctx.mass);
  if (split)
    split_stage<MassT, false, kFused, true>(a, epilogue, in, mass, nullptr, out);
  else
    node_stage<MassT, false, kFused, true>(a, epilogue, in, ctx.gmres.curl_cells, mass, nullptr, out);
  return check_hip(ctx, hipGetLastError(), "transposed operator apply");
}

}  // namespace

OperatorTailForm operator_tail_form(const Context& ctx) {
  const Grid& g = ctx.grid;
  if (g.nodes() <= kSplitNodes) return {(g.nodes() + 63u) / 64u, false};
  const bool plane = plane_form(g) && !ctx.num.smoothing;
  const unsigned blocks = (node_threads(g, plane) + kThreads - 1) / kThreads;
  return blocks <= kMaxBlocks ? OperatorTailForm{blocks, true} : OperatorTailForm{0, true};
}

int launch_operator(Context& ctx, const double* in, double* out, const OperatorCall& call) {
  const Grid& g = ctx.grid;
  const bool split = g.nodes() <= kSplitNodes;
  const OperatorArgs a{g, ctx.stream, ctx.delta * ctx.delta, ctx.current_factor, ctx.inverse_volume, call.scale,
                       call.guard, call.tail};
  const int epilogue = int(call.epilogue);
  phase_begin(ctx, Phase::spmv);
  int rc = 0;
  if (!split) {
    k_curl_n2c<<<blocks_for(ctx, g.cells()), kThreads, 0, ctx.stream>>>(g, in, ctx.gmres.curl_cells, call.guard);
    rc = check_hip(ctx, hipGetLastError(), "operator curl");
  }
  if (rc) {
  } else if (ctx.transposed_operator && (g.walls || ctx.num.smoothing)) {
    rc = fail(ctx, TPIC_MI_INVALID_STATE, "the transposed operator is built for periodic fields without smoothing");
  } else if (ctx.transposed_operator) {
    rc = ctx.mass_single ? transposed_image<float>(ctx, a, split, epilogue, in, out)
                         : transposed_image<double>(ctx, a, split, epilogue, in, out);
  } else if (g.walls) {
    rc = ctx.mass_single ? operator_image<float, true>(ctx, a, split, epilogue, in, out)
                         : operator_image<double, true>(ctx, a, split, epilogue, in, out);
  } else {
    rc = ctx.mass_single ? operator_image<float, false>(ctx, a, split, epilogue, in, out)
                         : operator_image<double, false>(ctx, a, split, epilogue, in, out);
  }
  phase_end(ctx, Phase::spmv);
  return rc;
}

int launch_curl_c2n(Context& ctx, const double* cells_in, double* nodes_out) {
  if (ctx.grid.walls) return fail(ctx, TPIC_MI_INVALID_STATE, "the standalone node curl is built for periodic fields");
  k_curl_c2n<<<blocks_for(ctx, ctx.grid.nodes()), kThreads, 0, ctx.stream>>>(ctx.grid, cells_in, nodes_out);
  return check_hip(ctx, hipGetLastError(), "node curl");
}

int launch_curl_n2c(Context& ctx, const double* nodes_in, double* cells_out) {
  k_curl_n2c<<<blocks_for(ctx, ctx.grid.cells()), kThreads, 0, ctx.stream>>>(ctx.grid, nodes_in, cells_out,
                                                                              Guard{});
  return check_hip(ctx, hipGetLastError(), "cell curl");
}

int launch_next_fields(Context& ctx) {
  const Grid& g = ctx.grid;
  const double th = ctx.num.theta;
  const bool copy = std::abs(th - 1.0) < 1e-10;
  const double c0 = 1.0 / th, c1 = -(1.0 - th) / th;
  phase_begin(ctx, Phase::advance);
  k_next_e<<<blocks_for(ctx, 3ull * g.nodes()), kThreads, 0, ctx.stream>>>(3 * g.nodes(), ctx.etheta, ctx.e, c0,
                                                                           c1, copy ? 1 : 0, ctx.validation);
  int rc = check_hip(ctx, hipGetLastError(), "E update");
  if (rc) return rc;
  k_faraday<<<blocks_for(ctx, g.cells()), kThreads, 0, ctx.stream>>>(g, ctx.etheta, ctx.b, -ctx.num.c * ctx.num.dt,
                                                                     ctx.validation);
  if ((rc = check_hip(ctx, hipGetLastError(), "Faraday update"))) return rc;
  rc = launch_cell_to_node(ctx);
  phase_end(ctx, Phase::advance);
  return rc;
}

}  // namespace tpic_mi
