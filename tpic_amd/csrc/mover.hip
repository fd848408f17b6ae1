// ECSIM particle mover: one coalesced SoA pass over a species.
//
// Per particle (detail::push_and_classify_particle,
// include/tpic/ecsim/particles/particle_mover_device.hpp:35-122):
//   W = CIC weights of the stored fractions; B, E_theta gathered at the 8 cell
//   corners with W; alpha = response(B) (particle_response.hpp:17-34);
//   v_new = 2*(alpha v + beta alpha E_theta) - v; per axis the displacement
//   dt*v_new/dx is added to the fraction, the integer shift floor(moved) moves
//   the cell and an exact 1.0 carries; then the whole-domain periodic/mirror
//   fold of communication::classify_particle_point
//   (include/tpic/communication/particles/particle_boundaries.hpp:111-165).
// A rejected record keeps every attribute and raises the validation word.
//
// Two kernels share the push: the sorted kernel walks the sorted species in
// aligned 64-particle blocks, stages the 48 corner field values of the block's
// bins once in LDS and reads them back, so a particle costs only its own 60 B
// read and 52 B write; the unsorted kernel gathers the corners per particle
// (input that was never sorted).
//
// Contraction is off in this translation unit (-ffp-contract=off and the
// pragma below): every product and sum rounds on its own, in the reference's
// expression order, so the result is bit-identical to the CPU oracle.
// Bound: HBM, 112 B per particle.
#include "internal.hpp"

#pragma clang fp contract(off)

namespace tpic_mi {
namespace {

constexpr unsigned kThreads = 256;
constexpr unsigned kWaves = kThreads / 64;

struct MoverParams {
  double beta, beta_over_c, dt, inverse_spacing[3];
  double extent[3];  // cells per axis
};

// cell modulo extent in [0, extent) for whole numbers below 2^34: they and
// the products are exact, and a quotient rounds across a whole number only
// from nearer than its own last place, where cell / extent never lies (it is a
// multiple of 1 / extent). A 64-bit integer remainder here held 30 registers.
__device__ __forceinline__ double modulo(double cell, double extent) {
  return cell - extent * floor(cell / extent);
}

// The mirror fold of a cell index in [extent, 2 extent): the reflected box,
// fraction and velocity reversed, an exact 1.0 carried back into the box.
__device__ __forceinline__ void mirror(double extent, double& whole, double& frac, double& vel) {
  whole = 2.0 * extent - whole - 1.0;
  frac = 1.0 - frac;
  vel = -vel;
  if (frac == 1.0) {
    if (whole + 1.0 < extent) {
      whole += 1.0;
      frac = 0.0;
    } else {
      frac = 1.0 - 1.1102230246251565e-16;  // 1 - epsilon/2
    }
  }
}

// The record of one particle as the mover reads it (60 B).
struct Raw {
  double rx, ry, rz, u, v, w, q;
  int32_t key;
};

__device__ __forceinline__ void load_raw(const ParticleView& s, uint32_t index, Raw& r) {
  r.rx = s.rx[index];
  r.ry = s.ry[index];
  r.rz = s.rz[index];
  r.u = s.u[index];
  r.v = s.v[index];
  r.w = s.w[index];
  r.q = s.q[index];
  r.key = s.cell[index];
}

// The same of particle `lane` of an aligned 64-particle block: the block's
// base is wave-uniform, so every address is a scalar base plus the lane's
// 32-bit offset.
__device__ __forceinline__ ParticleView block_view(const ParticleView& s, uint32_t block) {
  const size_t at = size_t(block) * 64u;
  return ParticleView{s.rx + at, s.ry + at, s.rz + at, s.u + at, s.v + at, s.w + at, s.q + at, s.cell + at, s.id};
}

// The pushed state of one particle: new key, fractions and velocity.
struct Pushed {
  int32_t key;
  double r[3], v[3];
};

// Record checks and the 8 CIC weights of the stored fractions (corners
// x-fastest). Returns the validation flags of a rejection, or 0.
__device__ __forceinline__ unsigned particle_weights(const Raw& r, double (&w)[8]) {
  const double fx = r.rx, fy = r.ry, fz = r.rz;
  const bool inside = fx >= 0.0 && fx < 1.0 && fy >= 0.0 && fy < 1.0 && fz >= 0.0 && fz < 1.0;
  const unsigned bad = !finite_value(r.q) ? kInvalidNonfinite : (!inside ? kInvalidFraction : 0u);
  const double cx = 1.0 - fx, cy = 1.0 - fy, cz = 1.0 - fz;
  w[0] = cx * cy * cz;
  w[1] = fx * cy * cz;
  w[2] = cx * fy * cz;
  w[3] = fx * fy * cz;
  w[4] = cx * cy * fz;
  w[5] = fx * cy * fz;
  w[6] = cx * fy * fz;
  w[7] = fx * fy * fz;
  return bad;
}

// B and E_theta at the particle: component c (Bx, By, Bz, Ex, Ey, Ez) is the
// weighted sum of corner(c, a) over a = 0..7 in that order.
template <class Corner>
__device__ __forceinline__ void interpolate(const double (&w)[8], const Corner& corner, double (&f)[6]) {
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    double value = 0.0;
#pragma unroll
    for (int a = 0; a < 8; ++a) value += w[a] * corner(c, a);
    f[c] = value;
    // Two components' corner values in flight (all 48 would hold 96 registers).
    if (c & 1) __builtin_amdgcn_sched_barrier(0);
  }
}

// Corner values staged per cell: 8 consecutive values per component.
struct StagedCorners {
  const double* v;
  __device__ double operator()(int c, int a) const { return v[c * 8 + a]; }
};

// Corner values read from the node fields (a particle outside the staged cell).
struct NodeCorners {
  const double* bnode;
  const double* etheta;
  unsigned nodes;
  unsigned at[8];
  __device__ double operator()(int c, int a) const {
    return c < 3 ? bnode[size_t(c) * nodes + at[a]] : etheta[size_t(c - 3) * nodes + at[a]];
  }
};

__device__ __forceinline__ unsigned push_fields(const Grid& g, const MoverParams& p, const Raw& r, int ci, int cj,
                                                int ck, const double (&f)[6], Pushed& out);

// Push and fold one particle of the validated interior cell (ci, cj, ck).
// `corner` gives the cell's 8 corner values of Bx, By, Bz, Ex, Ey, Ez.
// Returns the validation flags of a rejection (the record must then stay
// unchanged); on acceptance `out` holds the new state.
template <class Corner>
__device__ __forceinline__ unsigned push_particle(const Grid& g, const MoverParams& p, const Raw& r, int ci, int cj,
                                                  int ck, const Corner& corner, Pushed& out) {
  double w[8];
  const unsigned bad = particle_weights(r, w);
  double f[6];
  interpolate(w, corner, f);
  const unsigned flags = push_fields(g, p, r, ci, cj, ck, f, out);
  return bad ? bad : flags;
}

// The push from the interpolated fields: response, velocity update,
// displacement with carry, then the whole-domain fold.
__device__ __forceinline__ unsigned push_fields(const Grid& g, const MoverParams& p, const Raw& r, int ci, int cj,
                                                int ck, const double (&f)[6], Pushed& out) {
  const double fx = r.rx, fy = r.ry, fz = r.rz;
  const double bx = f[0], by = f[1], bz = f[2], ex = f[3], ey = f[4], ez = f[5];
  // ParticleResponse(bx, by, bz, beta_over_c)
  const double x = p.beta_over_c * bx, y = p.beta_over_c * by, z = p.beta_over_c * bz;
  const double n2 = x * x + y * y + z * z;
  const double inverse = 1.0 / (1.0 + n2);
  const double a0 = (1.0 + x * x) * inverse, a4 = (1.0 + y * y) * inverse, a8 = (1.0 + z * z) * inverse;
  const double xy = x * y * inverse, xz = x * z * inverse, yz = y * z * inverse;
  const double sx = x * inverse, syy = y * inverse, szz = z * inverse;
  const double a1 = xy + szz, a2 = xz - syy, a3 = xy - szz, a5 = yz + sx, a6 = xz + syy, a7 = yz - sx;
  const double u = r.u, v = r.v, ww = r.w;
  const double hx = a0 * u + a1 * v + a2 * ww;
  const double hy = a3 * u + a4 * v + a5 * ww;
  const double hz = a6 * u + a7 * v + a8 * ww;
  const double aex = a0 * ex + a1 * ey + a2 * ez;
  const double aey = a3 * ex + a4 * ey + a5 * ez;
  const double aez = a6 * ex + a7 * ey + a8 * ez;
  const double px = hx + p.beta * aex, py = hy + p.beta * aey, pz = hz + p.beta * aez;
  const int cell[3] = {ci, cj, ck};
  int pc[3];
  double frac[3] = {fx, fy, fz};
  double vel[3] = {2.0 * px - u, 2.0 * py - v, 2.0 * pz - ww};
  // Straight-line, with the first failing axis's flag kept: early returns
  // held the new state across their joins, in scratch memory.
  unsigned flags = 0;
#pragma unroll
  for (int axis = 0; axis < 3; ++axis) {
    const double displacement = p.dt * vel[axis] * p.inverse_spacing[axis];
    const double moved = frac[axis] + displacement;
    const double shift = floor(moved);
    const bool flight = shift >= -2147483648.0 && shift <= 2147483647.0;
    if (flags == 0u) flags = !finite_value(vel[axis]) ? kInvalidNonfinite : (!flight ? kInvalidFlight : 0u);
    frac[axis] = moved - shift;
    double whole = double(cell[axis]) + (flight ? shift : 0.0);
    if (frac[axis] == 1.0) {
      whole += 1.0;
      frac[axis] = 0.0;
    }
    const double extent = p.extent[axis];
    if (!(whole >= 0.0 && whole < extent)) {
      if (g.particle_periodic[axis]) {
        whole = modulo(whole, extent);
      } else {
        whole = modulo(whole, 2.0 * extent);
        if (whole >= extent) mirror(extent, whole, frac[axis], vel[axis]);
      }
    }
    pc[axis] = int(whole);
  }
  out.key = g.encode(pc[0], pc[1], pc[2]);
  out.r[0] = frac[0];
  out.r[1] = frac[1];
  out.r[2] = frac[2];
  out.v[0] = vel[0];
  out.v[1] = vel[1];
  out.v[2] = vel[2];
  return flags;
}

// The accepted state overwrites the record in place (a rejected record keeps
// every attribute).
__device__ __forceinline__ void store_pushed(const ParticleView& s, uint32_t index, const Pushed& out) {
  s.cell[index] = out.key;
  s.rx[index] = out.r[0];
  s.ry[index] = out.r[1];
  s.rz[index] = out.r[2];
  s.u[index] = out.v[0];
  s.v[index] = out.v[1];
  s.w[index] = out.v[2];
}

__device__ __forceinline__ void corner_nodes(const Grid& g, int ci, int cj, int ck, unsigned at[8]) {
  const unsigned n0 = g.node(ci, cj, ck);
  const unsigned sy = unsigned(g.nx + 1), sz = unsigned(g.nx + 1) * unsigned(g.ny + 1);
  at[0] = n0;
  at[1] = n0 + 1;
  at[2] = n0 + sy;
  at[3] = n0 + sy + 1;
  at[4] = n0 + sz;
  at[5] = n0 + sz + 1;
  at[6] = n0 + sz + sy;
  at[7] = n0 + sz + sy + 1;
}

// The interpolation of the rare lanes past the staged bins, one component at
// a time (48 node values in flight would take the registers of a whole block).
__device__ __forceinline__ void interpolate_nodes(const Grid& g, const double (&w)[8], int ci, int cj, int ck,
                                                  const double* __restrict__ bnode,
                                                  const double* __restrict__ etheta, double (&f)[6]) {
  const unsigned n0 = g.node(ci, cj, ck), nodes = g.nodes();
  const unsigned sy = unsigned(g.nx + 1), sz = unsigned(g.nx + 1) * unsigned(g.ny + 1);
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    const double* v = (c < 3 ? bnode + size_t(c) * nodes : etheta + size_t(c - 3) * nodes) + n0;
    double value = 0.0;
#pragma unroll
    for (int a = 0; a < 8; ++a)
      value += w[a] * v[unsigned(a & 1) + unsigned((a >> 1) & 1) * sy + unsigned(a >> 2) * sz];
    f[c] = value;
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The sorted mover walks the species array in aligned blocks of 64
// particles, not cell by cell: every record line is read once and every
// block is one full pass of the wave (a cell walk reads the line a cell
// shares with the next one twice and spends a second, nearly empty pass on a
// cell holding more than 64 particles). The particles of a block lie in a few
// bins, in ascending order: the 48 corner field values of the first Slots
// distinct bins are staged in LDS, and a lane reads those of its bin's slot. A
// lane past them gathers its corners from the node fields, which costs the
// wave a second pass: the slots follow the species' particles per cell. Two
// slots for every species cost 228 us per 2.55M particles at 27 per cell,
// where a block spans three or four bins; four cost about 92 us.
// Slots lie kSlotStride doubles apart (100 words: up to ten slots at one value
// start in distinct LDS banks).
constexpr unsigned kSlotStride = 50;

// The bin whose range holds sorted position `index` (the last bin whose
// first index is at most `index`), or -1 when no bin's range holds it.
__device__ int32_t holding_bin(const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ counts,
                               uint32_t bins, uint32_t index) {
  if (bins == 0 || offsets[0] > index) return -1;
  uint32_t lo = 0, hi = bins;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (offsets[mid] <= index)
      lo = mid;
    else
      hi = mid;
  }
  return index - offsets[lo] < counts[lo] ? int32_t(lo) : -1;
}

// A record the block walk does not push is flagged when the cell walk of the
// bins would have visited it and found a key other than the bin: its position
// lies in an interior bin's range and the key differs. Records in halo bin
// ranges, or in no range (a failed sort leaves every range empty), are left
// as they are without a flag.
__device__ unsigned unpushed_flags(const Grid& g, const uint32_t* __restrict__ offsets,
                                   const uint32_t* __restrict__ counts, uint32_t index, int32_t key) {
  const int32_t hb = holding_bin(offsets, counts, g.bins(), index);
  if (hb < 0 || hb == key) return 0u;
  int i, j, k;
  g.decode(hb, i, j, k);
  return g.interior(i, j, k) ? unsigned(kInvalidKey) : 0u;
}

// Lanes that start a bin of the block: a key in range that differs from the
// lane's below.
__device__ __forceinline__ uint64_t head_lanes(bool candidate, int32_t key, unsigned lane) {
  const int32_t below = __shfl_up(key, 1u, 64);
  return __builtin_amdgcn_ballot_w64(candidate && (lane == 0 || below != key));
}

// The slot of a lane's bin: the heads at or below the lane, less one (a lane
// below the first head is no candidate).
__device__ __forceinline__ unsigned slot_of(uint64_t heads) {
  const unsigned lane = threadIdx.x & 63u;
  return __builtin_amdgcn_mbcnt_hi(unsigned(heads >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(heads), 0u)) +
         unsigned((heads >> lane) & 1u) - 1u;
}

// The cell of a key, given the decoded cell of another key of the block:
// most keys of a block lie in one row.
struct BlockCell {
  int32_t key;
  int i, j, k;
};

__device__ __forceinline__ BlockCell block_cell(const Grid& g, int32_t key) {
  BlockCell c{key, 0, 0, 0};
  g.decode(key, c.i, c.j, c.k);
  return c;
}

__device__ __forceinline__ void cell_near(const Grid& g, const BlockCell& first, int32_t key, int& i, int& j, int& k) {
  i = first.i + (key - first.key);
  j = first.j;
  k = first.k;
  if (key < first.key || i > g.nx + 1) g.decode(key, i, j, k);
}

// Lane values of a block's staged corners: value v = lane + 64 t is corner
// v % 8 of component (v % 48) / 8 of slot v / 48, whose bin is that of the
// block's head v / 48; loaded when the bin is an interior cell (a slot without
// one is never read).
template <unsigned Slots>
struct StagedSlots {
  static constexpr unsigned kValues = Slots * 48;
  static constexpr unsigned kLoads = (kValues + 63) / 64;
  double v[kLoads];

  // `first` is the cell of the first head.
  __device__ __forceinline__ void load(const Grid& g, uint64_t heads, const BlockCell& first, int32_t key,
                                       const double* __restrict__ bnode, const double* __restrict__ etheta,
                                       unsigned lane) {
    const unsigned nodes = g.nodes();
    const unsigned sy = unsigned(g.nx + 1), sz = unsigned(g.nx + 1) * unsigned(g.ny + 1);
    // Wave-uniform: the lower node of every slot's cell, or none.
    constexpr unsigned kNone = 0xffffffffu;
    unsigned at[Slots];
    uint64_t m = heads;
#pragma unroll
    for (unsigned s = 0; s < Slots; ++s) {
      at[s] = kNone;
      if (m) {
        const int32_t bin = __builtin_amdgcn_readlane(key, int(__builtin_ctzll(m)));
        m &= m - 1;
        int i, j, k;
        cell_near(g, first, bin, i, j, k);
        if (g.interior(i, j, k)) at[s] = g.node(i, j, k);
      }
    }
#pragma unroll
    for (unsigned t = 0; t < kLoads; ++t) {
      const unsigned x = lane + 64u * t;
      // Lanes of load t lie in at most three slots: first slot (64 t) / 48.
      constexpr unsigned kLast = Slots - 1;
      const unsigned s0 = (64u * t) / 48u;
      const unsigned s1 = s0 + 1 < Slots ? s0 + 1 : kLast, s2 = s0 + 2 < Slots ? s0 + 2 : kLast;
      const unsigned slot = x / 48u;
      const unsigned node = slot == s0 ? at[s0] : (slot == s0 + 1 ? at[s1] : at[s2]);
      v[t] = 0.0;
      if (x < kValues && node != kNone) {
        const unsigned jv = x % 48u, comp = jv >> 3, a = jv & 7u;
        const unsigned n = node + (a & 1u) + ((a >> 1) & 1u) * sy + ((a >> 2) & 1u) * sz;
        v[t] = comp < 3 ? bnode[size_t(comp) * nodes + n] : etheta[size_t(comp - 3) * nodes + n];
      }
    }
  }

  __device__ __forceinline__ void stage(double* corner, unsigned lane) const {
#pragma unroll
    for (unsigned t = 0; t < kLoads; ++t) {
      const unsigned x = lane + 64u * t;
      if (x < kValues) corner[(x / 48u) * kSlotStride + x % 48u] = v[t];
    }
  }
};

__device__ __forceinline__ bool key_in_range(int32_t key, uint32_t bins) { return key >= 0 && uint32_t(key) < bins; }

// Each wave owns a contiguous range of blocks (remapped so an XCD's waves own
// neighbouring blocks) and walks it with a two-stage pipeline: the keys of
// block b+2, and the records, key ranges and staged corner fields of
// block b+1, are in flight while block b is pushed; block b+1's corners are
// staged in the second LDS buffer once b is done.
struct MoveSpecies {
  MoverParams p;
  ParticleView s;
  uint32_t n;
  const uint32_t* counts;
  const uint32_t* offsets;
  uint64_t* cross;  // or null
};

// The species of a launch, blockIdx.y.
struct MoveBatch {
  MoveSpecies species[kMaxSpecies];
};

template <unsigned Slots>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(Slots > 4 ? 3 : 4))) void k_move_blocks(
    Grid g, MoveBatch batch, const double* __restrict__ etheta, const double* __restrict__ bnode,
    unsigned* __restrict__ validation) {
  const MoveSpecies& sp = batch.species[blockIdx.y];
  const MoverParams& p = sp.p;
  const ParticleView s = sp.s;
  const uint32_t n = sp.n;
  const uint32_t* __restrict__ counts = sp.counts;
  const uint32_t* __restrict__ offsets = sp.offsets;
  uint64_t* __restrict__ cross = sp.cross;
  __shared__ __align__(16) double s_corner[kWaves][2][Slots * kSlotStride];
  const unsigned lane = threadIdx.x & 63u;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t bins = g.bins();
  const uint32_t nblocks = (n + 63u) / 64u;
  const unsigned waves_total = gridDim.x * kWaves;
  const unsigned wid = xcd_logical_block(blockIdx.x, gridDim.x) * kWaves + wave;
  const uint32_t per = (nblocks + waves_total - 1) / waves_total;
  const uint32_t b_begin = wid * per;
  const uint32_t b_end = b_begin + per < nblocks ? b_begin + per : nblocks;
  if (b_begin >= b_end) return;
  unsigned flags = 0;
  unsigned buf = 0;
  // Block b_begin: records, whether each lane lies in its key's bin range,
  // heads and staged corners; block b_begin + 1: keys.
  Raw cur;
  cur.key = -1;
  bool cur_in_range = false;
  uint64_t heads = 0;
  BlockCell cell0{};
  {
    const uint32_t index = b_begin * 64u + lane;
    if (index < n) load_raw(block_view(s, b_begin), lane, cur);
    const bool ranged = index < n && key_in_range(cur.key, bins);
    if (ranged) cur_in_range = index - offsets[cur.key] < counts[cur.key];
    heads = head_lanes(ranged, cur.key, lane);
    if (heads) {
      cell0 = block_cell(g, __builtin_amdgcn_readlane(cur.key, int(__builtin_ctzll(heads))));
      StagedSlots<Slots> cv;
      cv.load(g, heads, cell0, cur.key, bnode, etheta, lane);
      cv.stage(s_corner[wave][buf], lane);
    }
  }
  int32_t key1 = -1;
  if (b_begin + 1 < b_end && (b_begin + 1) * 64u + lane < n) key1 = block_view(s, b_begin + 1).cell[lane];
  for (uint32_t b = b_begin; b < b_end; ++b) {
    // Block b + 1: records, key ranges and staged corners; block b + 2: keys.
    const bool more = b + 1 < b_end;
    const uint32_t index1 = (b + 1) * 64u + lane;
    Raw nxt;
    nxt.key = -1;
    uint32_t first1 = 0, count1 = 0;
    StagedSlots<Slots> cv_next;
    uint64_t heads1 = 0;
    BlockCell cell1{};
    if (more) {
      // The key-dependent requests first (their lane reads of key1 then wait
      // only for key1's own load, issued a block earlier), then the records:
      // all of them stay in flight while block b is pushed.
      const bool ranged = index1 < n && key_in_range(key1, bins);
      heads1 = head_lanes(ranged, key1, lane);
      if (ranged) {
        first1 = offsets[key1];
        count1 = counts[key1];
      }
      if (heads1) {
        cell1 = block_cell(g, __builtin_amdgcn_readlane(key1, int(__builtin_ctzll(heads1))));
        cv_next.load(g, heads1, cell1, key1, bnode, etheta, lane);
      }
      if (index1 < n) load_raw(block_view(s, b + 1), lane, nxt);
    }
    int32_t key2 = -1;
    if (b + 2 < b_end && (b + 2) * 64u + lane < n) key2 = block_view(s, b + 2).cell[lane];
    // Push block b: the lanes of the staged bins read the staged corners; any
    // other lane (a block spanning more bins) gathers its corners from the
    // node fields.
    const double* corner = s_corner[wave][buf];
    const uint32_t index = b * 64u + lane;
    const int32_t key = cur.key;
    const bool candidate = index < n && key_in_range(key, bins);
    bool unpushed = index < n;
    bool crossed = false;  // pushed into another cell
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    if (candidate && cur_in_range) {
      int ci, cj, ck;
      cell_near(g, cell0, key, ci, cj, ck);
      if (g.interior(ci, cj, ck)) {
        unpushed = false;
        double w[8], fields[6];
        const unsigned bad = particle_weights(cur, w);
        const unsigned slot = slot_of(heads);
        if (slot < Slots)
          interpolate(w, StagedCorners{corner + slot * kSlotStride}, fields);
        else
          interpolate_nodes(g, w, ci, cj, ck, bnode, etheta, fields);
        Pushed out;
        unsigned f = push_fields(g, p, cur, ci, cj, ck, fields, out);
        if (bad) f = bad;
        if (f == 0u) {
          store_pushed(block_view(s, b), lane, out);
          crossed = out.key != key;
        }
        flags |= f;
      }
    }
    if (cross) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(crossed);
      if (lane == 0) cross[b] = m;
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    if (unpushed) flags |= unpushed_flags(g, offsets, counts, index, key);
    // Block b + 1 becomes current: its corners go to the other buffer.
    if (heads1) cv_next.stage(s_corner[wave][buf ^ 1u], lane);
    cur = nxt;
    cur_in_range = index1 - first1 < count1;
    heads = heads1;
    cell0 = cell1;
    key1 = key2;
    buf ^= 1u;
  }
  if (flags) atomicOr(validation, flags);
}

// Grid-stride over particles in any order (gathers per particle).
__global__ __launch_bounds__(kThreads) void k_move(Grid g, MoverParams p, ParticleView s, uint32_t n,
                                                   const double* __restrict__ etheta,
                                                   const double* __restrict__ bnode,
                                                   unsigned* __restrict__ validation) {
  const unsigned nodes = g.nodes();
  const int32_t bins = int32_t(g.bins());
  unsigned flags = 0;
  for (uint32_t index = blockIdx.x * blockDim.x + threadIdx.x; index < n; index += gridDim.x * blockDim.x) {
    const int32_t key = s.cell[index];
    int ci, cj, ck;
    if (key < 0 || key >= bins) {
      flags |= kInvalidKey;
      continue;
    }
    g.decode(key, ci, cj, ck);
    if (!g.interior(ci, cj, ck)) {
      flags |= kInvalidKey;
      continue;
    }
    NodeCorners corner{bnode, etheta, nodes, {}};
    corner_nodes(g, ci, cj, ck, corner.at);
    Raw r;
    load_raw(s, index, r);
    Pushed out;
    const unsigned f = push_particle(g, p, r, ci, cj, ck, corner, out);
    flags |= f;
    if (f == 0u) store_pushed(s, index, out);
  }
  if (flags) atomicOr(validation, flags);
}

// prepare_particle_mover_parameters (particle_mover_parameters.hpp:23-53):
// beta = (q/m) dt / 2, beta / c and 1 / spacing formed in double.
MoverParams mover_params(const Context& ctx, const SpeciesState& sp) {
  MoverParams p;
  const double beta = sp.q_over_m * ctx.num.dt / 2;
  p.beta = beta;
  p.beta_over_c = beta / ctx.num.c;
  p.dt = ctx.num.dt;
  p.inverse_spacing[0] = 1.0 / ctx.grid.dx;
  p.inverse_spacing[1] = 1.0 / ctx.grid.dy;
  p.inverse_spacing[2] = 1.0 / ctx.grid.dz;
  p.extent[0] = ctx.grid.nx;
  p.extent[1] = ctx.grid.ny;
  p.extent[2] = ctx.grid.nz;
  return p;
}

// About 32 blocks of 4 waves per CU, each wave a contiguous range of
// 64-particle blocks.
unsigned block_walk_blocks(const Context& ctx, uint32_t n) {
  const uint64_t want = (uint64_t((n + 63u) / 64u) + kWaves - 1) / kWaves;
  const uint64_t cap = uint64_t(ctx.cus > 0 ? ctx.cus : 256) * 32;
  return unsigned(std::max<uint64_t>(1, want < cap ? want : cap));
}

// Slots by the mean count c of a cell: 64 particles span 64 / c + 1 bins and
// more where counts vary. From 48 on two bins hold nearly every block (four
// instead of two: 1.3% of the cycle slower at 64 per cell and 128^3, 3.8% at
// 100 per cell and 512^2); four bins hold three or four bins' blocks down to
// 20 (cycle at 61 x 47 x 33 with 27 per cell: 1.61 ms with two, 1.34 ms with
// four), ten those of 8 a cell.
unsigned slots_for(const Context& ctx, const SpeciesState& sp) {
  const uint64_t cells = ctx.grid.cells();
  return sp.count >= 48 * cells ? 2u : (sp.count >= 20 * cells ? 4u : 10u);
}

}  // namespace

int launch_move(Context& ctx, int s, bool record_crossers) { return launch_moves(ctx, s, s + 1, &record_crossers); }

int launch_moves(Context& ctx, int first, int last, const bool* record_crossers) {
  bool any = false;
  for (int s = first; s < last; ++s) any = any || ctx.species[size_t(s)].count != 0;
  if (!any) return 0;
  phase_begin(ctx, Phase::move);
  const double* e = ctx.particle_field();
  for (int s = first; s < last; ++s) {
    const SpeciesState& sp = ctx.species[size_t(s)];
    if (sp.count == 0 || sp.sorted) continue;
    const unsigned blocks = unsigned(std::min<uint64_t>((uint64_t(sp.count) + kThreads - 1) / kThreads,
                                                        uint64_t(ctx.cus > 0 ? ctx.cus : 256) * 32));
    k_move<<<blocks, kThreads, 0, ctx.stream>>>(ctx.grid, mover_params(ctx, sp), sp.view(), sp.count, e, ctx.bn,
                                                ctx.validation);
    if (int rc = check_hip(ctx, hipGetLastError(), "mover")) return rc;
  }
  // The sorted species, one launch per number of slots.
  for (unsigned slots : {2u, 4u, 10u}) {
    MoveBatch batch{};
    unsigned species = 0, blocks = 0;
    for (int s = first; s < last; ++s) {
      SpeciesState& sp = ctx.species[size_t(s)];
      if (sp.count == 0 || !sp.sorted || slots_for(ctx, sp) != slots) continue;
      batch.species[species++] = MoveSpecies{mover_params(ctx, sp), sp.view(), sp.count, sp.counts, sp.offsets,
                                             record_crossers[s - first] ? sp.cross : nullptr};
      blocks = std::max(blocks, block_walk_blocks(ctx, sp.count));
      sp.sorted = false;  // also where this launch or a later one fails
    }
    if (species == 0) continue;
    const dim3 grid(blocks, species);
    if (slots == 2)
      k_move_blocks<2><<<grid, kThreads, 0, ctx.stream>>>(ctx.grid, batch, e, ctx.bn, ctx.validation);
    else if (slots == 4)
      k_move_blocks<4><<<grid, kThreads, 0, ctx.stream>>>(ctx.grid, batch, e, ctx.bn, ctx.validation);
    else
      k_move_blocks<10><<<grid, kThreads, 0, ctx.stream>>>(ctx.grid, batch, e, ctx.bn, ctx.validation);
    if (int rc = check_hip(ctx, hipGetLastError(), "mover")) return rc;
  }
  phase_end(ctx, Phase::move);
  return 0;
}

}  // namespace tpic_mi
