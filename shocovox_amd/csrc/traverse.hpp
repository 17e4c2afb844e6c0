// Per-ray octree traversal over the device layout (layout.hpp).
//
// The control flow and every floating-point operation follow
// get_by_ray_at_lod with MIP maps disabled (raytracing_on_cpu.rs:325-565),
// probe_brick (:256-312) and traverse_brick (:156-252), so that one ray takes
// the same path through the tree, bit for bit, as the reference CPU code (the P2
// form for directions of unit length, see dda_step_far):
//   * a 4-entry ring stack whose push overwrites the oldest entry and whose
//     pop past the retained entries restarts from the root after a 0.1 nudge
//     along the ray (:19-82, :548-562);
//   * the bitmap position is clamped to [1e-5, 4-1e-5] once per stack-loop
//     iteration and then advanced by step*4/size without a clamp (:425-436,
//     :510) - both are kept;
//   * brick voxels are tested through the occupancy sidecar, which holds
//     !pix_points_to_empty() for every voxel (node.rs:405-427).
// Two guards exist that the reference lacks: an iteration bound (the
// reference loop has no termination proof) and a bitmap-index range check
// (the reference would index its LUT out of bounds and panic). Either sets a
// flag on the ray; on well-formed inputs both stay clear.
//
// What differs from the reference is only how the same operations are laid
// out for 64-lane waves: the restart loop and the stack loop are one loop;
// POP and ADVANCE lanes share their first DDA step; the ring stack is a
// shift register; a miss carries only its flags; cast_ray_ww regroups a
// wave's brick probes; and trees whose sizes are powers of two (all device
// trees) use the exact power-of-two forms of the size arithmetic (P2).
#pragma once

#include "layout.hpp"
#include "svo_math.hpp"

namespace svo {

constexpr uint32_t FLAG_ITERATION_GUARD = 1u;
constexpr uint32_t FLAG_BITMAP_RANGE = 2u;
constexpr uint32_t MAX_TRAVERSAL_STEPS = 1u << 22;
// largest occupancy allocation (bytes) of a device tree: its reads take
// 32-bit byte offsets
constexpr uint64_t OCC_RANGE_MAX = 0xFFFFFFFFull;

struct TreeView {
  const NodeRec* nodes;
  const uint32_t* brick_pix;
  const uint32_t* brick_occ;
  const uint32_t* colors;
  const uint64_t* ray_lut;  // RAY_TO_NODE_OCCUPANCY_BITMASK_LUT, [pos*8 + dir]
  float size;
  uint32_t dim;
  uint32_t occ_words;
  uint32_t color_count;
  float inv_dim;  // pow2_rcp(dim): exact since the brick dimension is a power of two
  uint32_t node_count;
  uint32_t max_steps;  // iteration bound of one ray (MAX_TRAVERSAL_STEPS unless lowered)
  uint32_t mips_enabled;  // MIPMapStrategy::enabled: LOD queries probe node MIPs
  // bytes of the device's brick_occ allocation (below 2^32): the range of
  // its 32-bit offset reads (occ_word); 0 on the host, where it is unused
  uint32_t occ_range;
};

// Occupancy word flat >> 5 of the brick whose words begin at byte offset
// brick_off of brick_occ, for a probe whose cell index may lie outside the
// brick (`in` false: the caller then ignores the word). On the device the
// read is a buffer load whose range is the whole occupancy allocation, so
// such an index reads some word of the allocation, or 0 past its end, and
// needs no clamp; on the host it reads the brick's first word instead.
SVO_HD inline uint32_t occ_word(const TreeView& t, uint32_t brick_off, uint32_t flat, bool in) {
#if defined(__HIP_DEVICE_COMPILE__)
  (void)in;
  // 0x00020000: 32-bit data format, the word-read descriptor of gfx9 parts
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(t.brick_occ), 0, static_cast<int>(t.occ_range), 0x00020000);
  // (the word index made opaque: the offset is then one shift-add of the
  // brick's word offset, where the compiler would otherwise form
  // (flat >> 3) & ~3 and add it separately)
  uint32_t w = flat >> 5;
  asm volatile("" : "+v"(w));
  return __builtin_amdgcn_raw_buffer_load_b32(rsrc, static_cast<int>(brick_off + (w << 2)), 0, 0);
#else
  return t.brick_occ[(brick_off >> 2) + (in ? (flat >> 5) : 0u)];
#endif
}

// Every bounds size a traversal meets is the tree size halved k times (PUSH)
// or doubled back (POP), never below the brick dimension, and a brick's
// voxel size is a bounds size over the brick dimension. When the tree size
// is a power of two no larger than 2^24 and the brick dimension a power of
// two, all of these are powers of two in [1, 2^24] and all bounds
// coordinates are integers below 2^24. Then x / s equals x * (1/s) exactly
// and the POP's a - fmodf(a, b) equals floor(a / b) * b exactly (see
// pow2_rcp and sub_fmod), so the traversal can be compiled with P2 = true,
// without the general division and fmodf fallbacks; it is the same
// arithmetic, bit for bit, but for the brick walk of rays whose directions are not
// of unit length (dda_step_far). (Octree::new checks both powers through f32
// logarithms, which can admit a non-power at large sizes; such trees take
// the P2 = false form; the device upload refuses them.)
SVO_HD inline bool exact_pow2_sizes(uint64_t size, uint64_t dim) {
  return size != 0 && (size & (size - 1)) == 0 && size <= (1ull << 24) && dim != 0 &&
         (dim & (dim - 1)) == 0 && dim <= size;
}

// 1 / s for a bounds size s (a power of two in [1, 2^24] when P2): the
// exponent is negated by one integer subtraction
template <bool P2>
SVO_HD inline float size_rcp(float s) {
  if constexpr (P2) {
    return __builtin_bit_cast(float, 0x7F000000u - __builtin_bit_cast(uint32_t, s));
  } else {
    return pow2_rcp(s);
  }
}
template <bool P2>
SVO_HD inline float div_size(float x, float s, float rcp) {
  if constexpr (P2) {
    return x * rcp;
  } else {
    return div_by(x, s, rcp);
  }
}
template <bool P2>
SVO_HD inline V3f div3_size(V3f v, float s, float rcp) {
  if constexpr (P2) {
    return V3f{v.x * rcp, v.y * rcp, v.z * rcp};
  } else {
    return div3_by(v, s, rcp);
  }
}
// (p - min) * 4 / size, the position of p in the 4x4x4 bitmap of the node
// with bounds b (raytracing_on_cpu.rs:425-427). With P2, 4 and 1 / size are
// powers of two, so one scaling by their product rounds the same real
// number once, as the two steps do.
template <bool P2>
SVO_HD inline V3f bitmap_pos(V3f p, Cube b, float rcp) {
  if constexpr (P2) {
    const float k = rcp * 4.0f;
    return V3f{(p.x - b.min.x) * k, (p.y - b.min.y) * k, (p.z - b.min.z) * k};
  } else {
    return div3_by((p - b.min) * 4.0f, b.size, rcp);
  }
}
// st * 4 / s, the move of a node's bitmap position for a DDA step st (per
// axis +0.0, +-1 or NaN). With P2, 4 / s is a power of two and both
// products are exact, so one multiplication gives the same value.
template <bool P2>
SVO_HD inline V3f bitmap_move(V3f st, float s, float rcp) {
  if constexpr (P2) {
    const float k = rcp * 4.0f;
    return V3f{st.x * k, st.y * k, st.z * k};
  } else {
    return div3_by(st * 4.0f, s, rcp);
  }
}
// The POP's octant of the node within its parent (raytracing_on_cpu.rs:
// 450-461): hash_region(center - parent min, size). With P2 every bounds
// coordinate is a multiple of its size below 2^24 and min - parent min is
// exactly 0 or the size per axis, so the test center - parent min >= size
// is min != parent min.
template <bool P2>
SVO_HD inline uint32_t pop_octant(Cube b, V3f pmin) {
  if constexpr (P2) {
    return static_cast<uint32_t>(b.min.x != pmin.x) + static_cast<uint32_t>(b.min.z != pmin.z) * 2u +
           static_cast<uint32_t>(b.min.y != pmin.y) * 4u;
  } else {
    return hash_region(b.min + v3u(b.size / 2.0f) - pmin, b.size);
  }
}
// a - fmodf(a, b) for a bounds coordinate a >= +0 and b twice a bounds size
template <bool P2>
SVO_HD inline float sub_fmod_size(float a, float b, float rcp_b) {
  if constexpr (P2) {
    return floorf(a * rcp_b) * b;
  } else {
    return sub_fmod(a, b, rcp_b);
  }
}

// A ray's result. The normal of a hit is a function of the hit cell and the
// impact point (hit_normal); it is derived only where a caller asks for it.
// For a miss only `hit` (0) and `flags` are defined; consumers write the
// miss values themselves (see miss_result for what a miss reports).
struct CastResult {
  uint32_t hit;
  uint32_t pix;
  uint32_t flags;
  V3f impact;
  Cube cell;  // the voxel cell (Parted) or brick (Solid) that was hit
};

// get_by_ray's normal (raytracing_on_cpu.rs:296-311): cube_impact_normal of
// the hit cell at the impact point; zero for a miss.
SVO_HD inline V3f hit_normal(const CastResult& r) {
  return r.hit ? cube_impact_normal(r.cell, r.impact) : V3f{0.0f, 0.0f, 0.0f};
}

// Rust f32::clamp(min, max): NaN passes through
SVO_HD inline float rclamp(float x, float lo, float hi) {
  if (x < lo) x = lo;
  if (x > hi) x = hi;
  return x;
}

// BITMAP_INDEX_LUT[floor(x) as usize][floor(y)][floor(z)] = x + 4y + 16z
// The reference converts with `as usize`; a saturating u32 conversion gives
// the same value for 0..3 and a value above 3 (flagged) for everything else,
// without the 64-bit conversion sequence. The conversion truncates, which
// saturates to the same value as floor would: equal for x >= 0, and 0 for
// negative x and NaN either way, so the floor is left out.
SVO_HD inline uint32_t bitmap_index(V3f bp, uint32_t* flags) {
  uint32_t x = f2u32(bp.x);
  uint32_t y = f2u32(bp.y);
  uint32_t z = f2u32(bp.z);
  *flags |= (x | y | z) > 3u ? FLAG_BITMAP_RANGE : 0u;
  x = x > 3 ? 3 : x;
  y = y > 3 ? 3 : y;
  z = z > 3 ? 3 : z;
  return x + 4u * y + 16u * z;
}

// A ray that hit nothing: the only defined fields are hit and flags.
// (Materialising the miss values here would make the compiler set them in
// every loop iteration, ahead of the loop's exits.)
SVO_HD inline CastResult miss_flags(uint32_t flags) {
  CastResult r;
  r.hit = 0;
  r.flags = flags;
  return r;
}

// A miss with the values get_by_ray's callers see: no palette value, impact
// and cell zero.
SVO_HD inline CastResult miss_result(uint32_t flags) {
  CastResult r;
  r.hit = 0;
  r.pix = EMPTY_MARKER;
  r.flags = flags;
  r.impact = V3f{0.0f, 0.0f, 0.0f};
  r.cell = Cube{V3f{0.0f, 0.0f, 0.0f}, 0.0f};
  return r;
}

// bitmap_index(rclamp(bp, 1e-5, 4 - 1e-5)) without forming the clamped
// position: per axis, a saturating conversion (truncation, NaN -> 0) and a
// clamp of the integer to 0..3 give the same cell as clamping first (below
// 1e-5 and above 4 - 1e-5 the integer is <= 0 and >= 3; NaN passes the float
// clamp and converts to 0 either way), and no range test is needed.
// Truncation and floor differ only below 0, where both clamp to 0.
SVO_HD inline uint32_t clamp03(int32_t v) { return static_cast<uint32_t>(v < 0 ? 0 : (v > 3 ? 3 : v)); }
SVO_HD inline uint32_t bitmap_cell(V3f bp) {
  return clamp03(f2i32(bp.x)) + 4u * clamp03(f2i32(bp.y)) + 16u * clamp03(f2i32(bp.z));
}

// traverse_brick (raytracing_on_cpu.rs:156-252) over the occupancy of Parted
// brick `word` with bounds bb: moves p to where the walk ends and returns
// whether that is in an occupied cell, whose flat index goes to *cell.
// With SLICE > 0 (P2 only) a call takes at most SLICE steps; a walk that has
// not ended by then leaves its cell in *cell and sets *more, and the next call
// goes on from there (a cell's far corner is the same value whether it is
// reached by steps or formed from the cell's index).
constexpr uint32_t NO_CELL = 0xFFFFFFFFu;
template <bool P2, int SLICE = 0>
SVO_HD __attribute__((always_inline)) inline bool walk_brick(const TreeView& t, uint32_t word,
                                                             Cube bb, V3f d, V3f sig, V3f scale,
                                                             V3f* p, uint32_t* cell,
                                                             uint32_t* flags,
                                                             bool* more = nullptr) {
  static_assert(P2 || SLICE == 0, "only the P2 form walks in slices");
  const int dim = static_cast<int>(t.dim);
  const float fdim = static_cast<float>(t.dim);
  const float rcp_size = size_rcp<P2>(bb.size);
  V3f pib;
  if constexpr (P2) {
    // (p - min) * dim / size: dim and 1 / size are powers of two, so scaling
    // by their product rounds the same real number once, as the two steps do
    const float k = fdim * rcp_size;
    pib = (*p - bb.min) * k;
  } else {
    pib = div3_size<P2>((*p - bb.min) * fdim, bb.size, rcp_size);
  }
  auto clampi = [dim](int v) {
    const int a = v > 0 ? v : 0;
    return a < dim - 1 ? a : dim - 1;
  };
  int ix = clampi(f2i32(pib.x));
  int iy = clampi(f2i32(pib.y));
  int iz = clampi(f2i32(pib.z));
  if (SLICE > 0 && *cell != NO_CELL) {
    const uint32_t k = static_cast<uint32_t>(__builtin_ctz(t.dim));
    ix = static_cast<int>(*cell & (t.dim - 1u));
    iy = static_cast<int>((*cell >> k) & (t.dim - 1u));
    iz = static_cast<int>(*cell >> (2u * k));
  }
  const float unit = div_size<P2>(bb.size, fdim, t.inv_dim);
  // A step moves the cell by signum(direction) on the axes that stepped and
  // leaves the others (their step component is +0.0, and cell corners are
  // never -0.0): the per-axis moves are fixed for the whole probe.
  const V3f umove{sig.x * unit, sig.y * unit, sig.z * unit};
  const uint32_t shift = static_cast<uint32_t>(__builtin_ctz(t.dim));
  // ix + iy dim + iz dim^2 (P2: the factors as shifts)
  auto flat_of = [&](int x, int y, int z) -> uint32_t {
    if constexpr (P2) {
      return static_cast<uint32_t>(x) | (static_cast<uint32_t>(y) << shift) |
             (static_cast<uint32_t>(z) << (2u * shift));
    } else {
      return static_cast<uint32_t>(x + y * dim + z * dim * dim);
    }
  };
  // After the loop `occupied` says whether the ray stands in an occupied cell,
  // `in` (when not) whether it stopped inside the brick: on a NaN step or,
  // without P2, at the step bound.
  bool in, occupied;
  if constexpr (P2) {
    // Cell coordinates mirrored on the axes whose signum is -1: a = ix
    // (signum +1) or dim-1-ix = ix ^ (dim-1) (signum -1), so that every move
    // is +1 and an axis leaves the brick at a = dim; the cell's flat index is
    // the mirrored one xor the mirror mask.
    const uint32_t dm1 = t.dim - 1u;
    const uint32_t nx = sig.x < 0.0f ? dm1 : 0u;
    const uint32_t ny = sig.y < 0.0f ? dm1 : 0u;
    const uint32_t nz = sig.z < 0.0f ? dm1 : 0u;
    const uint32_t mirror = nx | (ny << shift) | (nz << (2u * shift));
    uint32_t ax = static_cast<uint32_t>(ix) ^ nx;
    uint32_t ay = static_cast<uint32_t>(iy) ^ ny;
    uint32_t az = static_cast<uint32_t>(iz) ^ nz;
    // occupancy words per brick: dim^3 / 32 rounded up, a power of two
    const uint32_t occ_off = (word << static_cast<uint32_t>(__builtin_ctz(t.occ_words))) * 4u;
    // cmin holds the cell's far corner (the corner the direction points to):
    // min + (i + 1) unit on an axis whose signum is +1, min + i unit on the
    // others. Every term is a multiple of unit (a power of two) no larger
    // than the tree size (at most 2^24), so each is exact in f32: the fused
    // form gives the same value as the reference's min + i unit, then + unit.
    V3f cmin{fmaf(static_cast<float>(static_cast<uint32_t>(ix) + (sig.x < 0.0f ? 0u : 1u)), unit,
                  bb.min.x),
             fmaf(static_cast<float>(static_cast<uint32_t>(iy) + (sig.y < 0.0f ? 0u : 1u)), unit,
                  bb.min.y),
             fmaf(static_cast<float>(static_cast<uint32_t>(iz) + (sig.z < 0.0f ? 0u : 1u)), unit,
                  bb.min.z)};
    // Each iteration takes the step out of the current cell while the cell's
    // word is still in flight, requests the next cell's word, and only then
    // keeps the step or, when the cell was occupied, drops it (by selects on
    // p and the index; the other state is not used after the loop). So a step
    // waits for its load only as long as its own arithmetic does not cover
    // it, and the loop has one exit and no masks to carry: a lone ray's step
    // 450 -> 275 cycles (the loop is 41 VALU + 8 SALU, where testing the cell
    // before stepping was 31 VALU + 27 SALU), 8 1080p frames in one batched
    // run 1.09 -> 0.97 ms.
    uint32_t flat = (ax | (ay << shift) | (az << (2u * shift))) ^ mirror;
    uint32_t bits = occ_word(t, occ_off, flat, true);
    uint32_t bit, stop;
    float m;
    for (int left = SLICE;;) {
      bool sx, sy, sz;
      V3f q = *p;
      m = dda_step_far(d, &q, cmin, scale, &sx, &sy, &sz);
      cmin = V3f{sx ? cmin.x + umove.x : cmin.x, sy ? cmin.y + umove.y : cmin.y,
                 sz ? cmin.z + umove.z : cmin.z};
      ax += static_cast<uint32_t>(sx);
      ay += static_cast<uint32_t>(sy);
      az += static_cast<uint32_t>(sz);
#if defined(__HIP_DEVICE_COMPILE__)
      // (the word is read from here on, behind the step's arithmetic)
      asm volatile("" : "+v"(bits) : "v"(ax), "v"(ay), "v"(az));
#endif
      bit = bit_of(bits, flat);
      const bool keep = bit == 0u;
      const uint32_t next = (ax | (ay << shift) | (az << (2u * shift))) ^ mirror;
      const uint32_t axes = ax | ay | az;
      bits = occ_word(t, occ_off, next, axes < t.dim);
      *p = V3f{keep ? q.x : p->x, keep ? q.y : p->y, keep ? q.z : p->z};
      flat = keep ? next : flat;
      // Leaves at an occupied cell, or outside the brick (an axis at dim: with
      // dim a power of two, a bit of `axes` above dim - 1). A step of length m
      // (not NaN) moves at least one axis, each axis only in its direction's
      // sign (signum is +-1 there: a NaN direction makes every distance NaN),
      // so the cell leaves the brick within 3 dim steps. A NaN step moves
      // nothing (p becomes NaN and stays so), so the loop would repeat that
      // state: it ends here.
      stop = bit | (axes & ~dm1);
      if ((stop != 0u) | !(m == m)) break;
      if (SLICE > 0 && --left == 0) break;
    }
#if defined(__HIP_DEVICE_COMPILE__)
    // (opaque here, so that the tests below are made after the loop and not
    // carried through it as masks)
    asm volatile("" : "+v"(bit), "+v"(m), "+v"(stop));
#endif
    occupied = bit != 0u;
    in = !(m == m);
    if (SLICE > 0) {
      *more = (stop == 0u) & (m == m);
      *cell = flat;
      if (in && !occupied) *flags |= FLAG_ITERATION_GUARD;
      return occupied;
    }
    ix = static_cast<int>(flat & dm1);
    iy = static_cast<int>((flat >> shift) & dm1);
    iz = static_cast<int>(flat >> (2u * shift));
  } else {
    V3f cmin = bb.min + V3f{static_cast<float>(ix), static_cast<float>(iy),
                            static_cast<float>(iz)} *
                            unit;
    const uint32_t* occ = t.brick_occ + static_cast<uint64_t>(word) * t.occ_words;
    const int mx = step_int(sig.x), my = step_int(sig.y), mz = step_int(sig.z);
    for (int left = 4 * dim + 16;;) {
      in = ix >= 0 && ix < dim && iy >= 0 && iy < dim && iz >= 0 && iz < dim;
      const uint32_t flat = in ? flat_of(ix, iy, iz) : 0u;
      const uint32_t bits = occ[flat >> 5];
      occupied = in & (bit_of(bits, flat) != 0u);
      if (!in | occupied) break;
      bool sx, sy, sz;
      dda_step_axes(d, sig, p, cmin, unit, scale, &sx, &sy, &sz);
      cmin = V3f{sx ? cmin.x + umove.x : cmin.x, sy ? cmin.y + umove.y : cmin.y,
                 sz ? cmin.z + umove.z : cmin.z};
      ix += sx ? mx : 0;
      iy += sy ? my : 0;
      iz += sz ? mz : 0;
      if (--left == 0) break;
    }
  }
  if (occupied) {
    *cell = flat_of(ix, iy, iz);
    return true;
  }
  if (in) *flags |= FLAG_ITERATION_GUARD;
  return false;
}

// The hit of a Solid brick, or of Parted brick `word` in flat cell `cell`, at p
// (raytracing_on_cpu.rs:256-295).
template <bool P2>
SVO_HD __attribute__((always_inline)) inline void brick_hit(const TreeView& t, uint32_t form,
                                                            uint32_t word, Cube bb,
                                                            uint32_t cell, V3f p, CastResult* r) {
  r->hit = 1;
  r->impact = p;
  if (form == FORM_SOLID) {
    r->pix = word;
    r->cell = bb;
    return;
  }
  const float fdim = static_cast<float>(t.dim);
  uint32_t ix, iy, iz;
  if constexpr (P2) {
    const uint32_t shift = static_cast<uint32_t>(__builtin_ctz(t.dim));
    ix = cell & (t.dim - 1u);
    iy = (cell >> shift) & (t.dim - 1u);
    iz = cell >> (2u * shift);
  } else {
    ix = cell % t.dim;
    iy = cell / t.dim % t.dim;
    iz = cell / (t.dim * t.dim);
  }
  const uint64_t n3 = static_cast<uint64_t>(t.dim) * t.dim * t.dim;
  r->pix = t.brick_pix[static_cast<uint64_t>(word) * n3 + cell];
  // (below the brick dimension: exact as signed or unsigned)
  const V3f scaled = V3f{static_cast<float>(static_cast<int>(ix)),
                         static_cast<float>(static_cast<int>(iy)),
                         static_cast<float>(static_cast<int>(iz))} *
                     bb.size;
  r->cell = Cube{bb.min + div3_size<P2>(scaled, fdim, t.inv_dim),
                 div_size<P2>(bb.size, fdim, t.inv_dim)};
}

// probe_brick (raytracing_on_cpu.rs:256-312)
template <bool P2>
SVO_HD __attribute__((always_inline)) inline bool probe_brick(const TreeView& t, uint32_t form,
                                                              uint32_t word, Cube bb, V3f d,
                                                              V3f sig, V3f scale, V3f* p,
                                                              CastResult* r) {
  uint32_t cell = 0u;
  if (form == FORM_EMPTY) return false;
  if (form != FORM_SOLID &&
      !walk_brick<P2>(t, word, bb, d, sig, scale, p, &cell, &r->flags))
    return false;
  brick_hit<P2>(t, form, word, bb, cell, *p, r);
  return true;
}

// The rest of a ray whose POP of the root empties the stack because the
// root has no occupied bitmap cell ahead of the ray (occupancy & LUT == 0).
// The reference then restarts from the root at p + 0.1 d, fails the same
// test, and so on until p leaves the tree: the LUT box of a cell holds the
// boxes of every cell further along the ray (each coordinate moves towards
// the box's far corner or stays), so no later position passes the test and
// the ray ends as a miss. Only the nudges and the iteration count remain,
// replayed here exactly (the restart's interior test, then one counted
// iteration per restart), and only when the count can decide anything: the
// ray ends as a miss either way, so the nudges matter only if they could
// exceed the iteration bound before p leaves the tree. A nudge moves p by
// fl(p + s) - p with s = fl(0.1 d); for a result inside the tree the rounding
// is at most size * 2^-25, so with m = max |s| >= size * 2^-20 every counted
// nudge moves p by at least 31/32 m along that axis, always the same way, and
// at most 1.04 size / m + 1 of them end inside the tree. When that is within
// the iterations left (tested with a factor of two to spare) the result is
// known at once. (A NaN component of s makes p leave at the first nudge.)
// The replay is one chain of adds and compares per ray, thousands long in a
// large tree: without it a 4K frame of a 1024^3 heightfield took 0.80 ms
// instead of 2.80 ms, 24 views of 12 small trees in one batched run 0.72 ms
// instead of 1.17 ms, and a 720p LOD frame of a 256^3 heightfield 0.25 ms
// instead of 2.69 ms.
// Not for a leaf root (its brick probe runs on every iteration), nor for
// MIP-enabled LOD rays unless mip_test_over holds.
SVO_HD inline CastResult crawl_out_of_root(const TreeView& t, V3f p, V3f d, uint32_t steps,
                                           uint32_t flags) {
  const V3f s = d * 0.1f;
  const float m = fmaxf(fmaxf(fabsf(s.x), fabsf(s.y)), fabsf(s.z));
  const uint32_t left = t.max_steps - steps;  // (no ray gets here past its bound)
  if (left >= 16u && m >= t.size * 0x1p-20f && m * static_cast<float>(left) >= 2.0f * t.size)
    return miss_flags(flags);
  for (;;) {
    p = p + s;
    if (!((p.x < t.size) & (p.y < t.size) & (p.z < t.size) & (p.x > 0.0f) & (p.y > 0.0f) &
          (p.z > 0.0f)))
      return miss_flags(flags);
    if (++steps > t.max_steps) return miss_flags(flags | FLAG_ITERATION_GUARD);
  }
}

// The MIP test of a stack-loop iteration (raytracing_on_cpu.rs:368-372): level
// below |o - snapped| / viewing distance, snapped being p rounded to a grid of
// 2 level. Its four correctly rounded divisions and square root are about 120
// instructions, and it mostly fails by far: snapped lies within
// level + size 2^-24 (the quotient's rounding) of p per axis, so
// |o - snapped| <= |o - p| + 1.7321 (level + size 2^-24), and with
// a = level (viewing distance - 1.75) - size 2^-23 > 0 the test fails whenever
// a^2 >= 1.002 |o - p|^2 (0.2% covers the other roundings; nothing is concluded
// from a huge, infinite or NaN |o - p|^2). 1080p LOD frame 143 -> 132 us,
// 500k LOD rays 209 -> 184 us.
SVO_HD inline bool mip_test(const TreeView& t, V3f o, V3f p, float mip_level,
                            float viewing_distance) {
  const V3f v = o - p;
  const float d2 = (v.x * v.x + v.y * v.y) + v.z * v.z;
  const float a = mip_level * (viewing_distance - 1.75f) - t.size * 0x1p-23f;
  if (a > 0.0f && mip_level > 0.0f && a * a >= 1.002f * d2 && d2 < 1e30f) return false;
  const float grid = mip_level * 2.0f;
  const V3f snapped{roundf(p.x / grid) * grid, roundf(p.y / grid) * grid,
                    roundf(p.z / grid) * grid};
  return mip_level < length(o - snapped) / viewing_distance;
}

// Whether the MIP test at the root (level < |o - snapped| / viewing distance,
// snapped being p rounded to a grid of 2 level) fails now and in every later
// restart of a ray that crawls out of the root. The level rises by one per
// restart and never falls; snapped lies within level of p per axis, so
// |o - snapped| <= far + 1.7321 level, far being the distance from o to the
// tree's farthest corner (0.1% covers the roundings of both sides). Once
// level * (viewing distance - 1.75) >= 1.001 far holds it holds from then on
// (for a viewing distance above 1.75).
SVO_HD inline bool mip_test_over(const TreeView& t, V3f o, float mip_level,
                                 float viewing_distance) {
  const V3f far{fmaxf(fabsf(o.x), fabsf(o.x - t.size)), fmaxf(fabsf(o.y), fabsf(o.y - t.size)),
                fmaxf(fabsf(o.z), fabsf(o.z - t.size))};
  const float f = 1.001f * length(far);  // (infinite: |o - snapped| may be, too)
  return viewing_distance > 1.75f && f < __builtin_inff() &&
         mip_level * (viewing_distance - 1.75f) >= f;
}

// The reference's NodeStack<u32, 4> (raytracing_on_cpu.rs:19-82): a ring of
// four whose push overwrites the oldest entry once full and whose count
// says how many entries are retained. Kept here as a shift register, s0 the
// top: a push shifts down (dropping the oldest), a pop shifts up, so the top
// is read without selecting among the four registers. Entries beyond
// `count` are never read, which makes the two forms equivalent.
struct RingStack {
  uint32_t s0, s1, s2, s3;
  uint32_t count;
  SVO_HD void push(uint32_t v) {
    s3 = s2;
    s2 = s1;
    s1 = s0;
    s0 = v;
    count = count < 4u ? count + 1u : 4u;
  }
  SVO_HD void pop() {
    s0 = s1;
    s1 = s2;
    s2 = s3;
    count -= 1u;
  }
};

// lut[i] by a 32-bit byte offset, which the load adds to the base itself (a
// 64-bit index is added by the vector unit first: 1080p frame 165 -> 163 us,
// 4K 499 -> 492).
template <class LutT>
SVO_HD inline uint64_t lut_word(const LutT* lut, uint32_t i) {
  return *reinterpret_cast<const LutT*>(reinterpret_cast<const char*>(lut) + (i << 3));
}

// get_by_ray_at_lod (raytracing_on_cpu.rs:325-565). Without LOD it is
// get_by_ray (viewing distance f32::MAX, under which the MIP test never
// passes). `lut` is the RAY_TO_NODE_OCCUPANCY_BITMASK_LUT, wherever the
// caller staged it. `top` optionally holds a copy of the first `ntop` node
// records (the top levels, as records are numbered breadth-first), e.g.
// staged in LDS; those records are read from it instead of t.nodes. P2
// requires exact_pow2_sizes(t.size, t.dim).
//
// With LOD and the tree's MIPs enabled, every stack-loop iteration first
// tests the node's level against the distance travelled (:368-386): the
// level starts at log2(size / dim), falls by one per PUSH, rises by one per
// POP and is not reset by a restart from the root; when the level is below
// |origin - round(p / (2 level)) * 2 level| / viewing_distance, the node's
// MIP brick is probed over the node's bounds like a uniform leaf's brick.
//
// How a wave runs it. A ray's time is the latency of its iterations, and a
// wave's the instructions of all paths its lanes take, so
//   * the loop has one exit, on a status each lane keeps in a register;
//     leaving from several places would carry a mask per place through every
//     iteration (scalar instructions were a third of the loop's);
//   * a hit lane leaves p, bounds, target and the stack as they are, and its
//     palette value and cell are worked out after the loop, once per wave
//     rather than in every iteration in which some lane hits (and the loop
//     holds none of the result's registers: 63 VGPRs, where it held 77);
//   * the LUT word of p's cell is requested beside the node record, not after
//     the record has shown that it is needed; a probe that moved p requests
//     it again;
//   * a step is kept as octant bits (step_octant_moved).
// Together a lone ray's iteration takes 0.56 us instead of 0.78, 8 1080p
// frames in one batched run 0.90 ms instead of 0.96, one of them 0.185 ms
// instead of 0.208.
struct RayWalk {
  V3f d, scale, p;
  Cube bounds;
  uint32_t target;
  RingStack stk;
  uint32_t dir_idx;  // hash_direction(d)
  uint32_t neg;      // octant bits of the axes the ray runs backwards along
  uint32_t steps, flags;
  uint32_t cell;     // flat cell of a hit, or of a sliced walk that goes on (else NO_CELL)
  uint32_t end;      // WALK_*
  uint32_t brick;    // deferred walks: BRICK_*, of the iteration under way
  float mip_level;   // LOD
};
enum : uint32_t { BRICK_NONE = 0, BRICK_DUE = 1, BRICK_DONE = 2 };
enum : uint32_t {
  WALK_RUNS = 0,
  WALK_HIT = 1,
  WALK_HIT_MIP = 2,
  WALK_MISS = 3,
  WALK_GUARD = 4,
  WALK_CRAWL = 5
};

template <bool LOD>
SVO_HD __attribute__((always_inline)) inline void walk_begin(const TreeView& t, V3f o, V3f d,
                                                            RayWalk& w) {
  w.d = d;
  w.dir_idx = hash_direction(d);
  // (for a NaN component every scale factor is NaN and no step moves any axis)
  w.neg = octant_of(__builtin_signbit(d.x), __builtin_signbit(d.y), __builtin_signbit(d.z));
  w.bounds = Cube{v3u(0.0f), t.size};
  w.stk = RingStack{0u, 0u, 0u, 0u, 1u};  // the root pushed
  float tt = 0.0f;
  const int ir = ray_setup(w.bounds, o, d, &tt, &w.scale);
  w.p = ir != 0 ? o + d * (ir == 2 ? tt : 0.0f) : o;
  w.target = hash_region(w.p - w.bounds.min, w.bounds.size / 2.0f);
  w.steps = 0;
  w.flags = 0;
  w.cell = NO_CELL;
  w.brick = BRICK_NONE;
  w.end = ir != 0 ? WALK_RUNS : WALK_MISS;
  // log2(size / dim) of two powers of two, exactly
  w.mip_level =
      LOD ? static_cast<float>(__builtin_ctz(static_cast<uint32_t>(t.size) / t.dim)) : 0.0f;
}

// One iteration of the reference's stack loop and, when the stack has
// emptied, its restart from the root (which ends the ray when the nudged point
// leaves the tree). With DEFER an iteration that meets a Parted brick of a
// leaf only marks it due; walk_slice walks it, and the next call goes on with
// the iteration from there.
template <bool LOD, bool P2, bool DEFER, class LutT>
SVO_HD __attribute__((always_inline)) inline void walk_iterate(
    const TreeView& t, const LutT* __restrict__ lut, V3f o, const NodeRec* top, uint32_t ntop,
    float viewing_distance, RayWalk& w) {
  const float lo = 0.00001f;
  const float hi = 4.0f - 0.00001f;
  V3f& d = w.d;
  V3f& p = w.p;
  const V3f scale = w.scale;
  const uint32_t dir_idx = w.dir_idx, neg = w.neg;
  Cube& bounds = w.bounds;
  uint32_t& target = w.target;
  RingStack& stk = w.stk;
  uint32_t& steps = w.steps;
  uint32_t& end = w.end;
  // signum(d) per axis, formed again in every iteration from d's sign bits
  // (one instruction each) rather than kept in three registers: the empty
  // asm makes d opaque here, so the compiler cannot hoist these (or other
  // values derived from d) out of the loop. For a NaN component the
  // reference's signum is NaN and this one +-1; then every scale factor is
  // NaN (each involves all three components), every DDA distance is NaN
  // and no step selects a signum, so the difference is never observed.
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(d.x), "+v"(d.y), "+v"(d.z));
#endif
  V3f sig{sign_one(d.x), sign_one(d.y), sign_one(d.z)};
  const bool fresh = !DEFER || w.brick == BRICK_NONE;
  if (fresh) ++steps;  // (against the bound at the iteration's end)
  const uint32_t key = stk.s0;
  const NodeRec& n = (key < ntop ? top : t.nodes)[key];
  const uint64_t occ = n.occ;
  const uint32_t meta = n.meta;
  // the child word of the current target, read together with the header
  // (same record, one round trip); with target OOB_OCTANT it is child[0]
  // and unused
  const uint32_t tword = n.child[target & 7u];
  // the position in the node's 4x4x4 bitmap; the clamp to [lo, hi]
  // (:425-436) is applied to the float position only where ADVANCE
  // continues from it, the cell index comes from bitmap_cell
  const float rcp_size = size_rcp<P2>(bounds.size);
  V3f bp = bitmap_pos<P2>(p, bounds, rcp_size);
  uint64_t ahead = lut_word(lut, bitmap_cell(bp) * 8u + dir_idx);
  auto moved_by_probe = [&]() {
    bp = bitmap_pos<P2>(p, bounds, rcp_size);
    ahead = lut_word(lut, bitmap_cell(bp) * 8u + dir_idx);
#if defined(__HIP_DEVICE_COMPILE__)
    // (used here, so that the two requests are not merged into one after
    // the probe)
    asm volatile("" : "+v"(ahead));
#endif
  };
  const uint32_t kind = node_kind(meta);
  const bool uniform = kind == KIND_UNIFORM_LEAF;  // backtracks after its probe
  if (LOD && t.mips_enabled && fresh) {
    if (mip_test(t, o, p, w.mip_level, viewing_distance)) {
      if (n.mip == FORM_SOLID) end = WALK_HIT_MIP;
      if (n.mip == FORM_PARTED) {
        if (walk_brick<P2>(t, n.mip_word, bounds, d, sig, scale, &p, &w.cell, &w.flags))
          end = WALK_HIT_MIP;
        moved_by_probe();
      }
    }
  }
  if ((!LOD || end == WALK_RUNS) && fresh && target != OOB_OCTANT &&
      (kind == KIND_UNIFORM_LEAF || kind == KIND_LEAF)) {
    const uint32_t slot = uniform ? 0u : target;
    const uint32_t form = brick_form(meta, slot);
    if (form == FORM_SOLID) end = WALK_HIT;
    if (form == FORM_PARTED) {
      if constexpr (DEFER) {
        w.brick = BRICK_DUE;
      } else {
        if (walk_brick<P2>(t, slot == target ? tword : n.child[0],
                           uniform ? bounds : child_bounds_for(bounds, target), d, sig, scale,
                           &p, &w.cell, &w.flags))
          end = WALK_HIT;
        moved_by_probe();
      }
    }
  }
  // signum(d) formed again past the probe, so that the values formed
  // before it are dead inside the probe's DDA loop (whose registers then
  // hold the per-axis cell moves rather than recomputing them each step)
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(d.x), "+v"(d.y), "+v"(d.z), "+v"(end));
#endif
  if ((!DEFER || w.brick != BRICK_DUE) && end == WALK_RUNS) {
    if constexpr (DEFER) w.brick = BRICK_NONE;
    sig = V3f{sign_one(d.x), sign_one(d.y), sign_one(d.z)};
    // (an empty bitmap has nothing ahead)
    const bool pop = uniform | (target == OOB_OCTANT) | ((occ & ahead) == 0ull);
    Cube tb = child_bounds_for(bounds, target);
    const bool push = !pop & (kind == KIND_INTERNAL) &
                      ((occ & octant_bitmap_mask(target)) != 0ull) & (tword != INVALID_INDEX);
    const bool emptied = pop & (stk.count == 1u);
    // PUSH, POP and ADVANCE leave the next bounds and target here, and the
    // stack moves once after them, by selects: the loop's state stays in
    // the same registers on every path.
    Cube next_bounds = bounds;
    uint32_t next_target = target;
    if (push) {
      // PUSH (:484-492)
      next_bounds = tb;
      next_target = hash_region(p - tb.min, tb.size / 2.0f);
    } else {
      // POP (:445-475) and ADVANCE (:497-544) both begin with one DDA step,
      // out of the node (POP, unless the stack empties) or out of the
      // target child (ADVANCE); it is issued once for the lanes of both.
      // (The POP's other values depend on the bounds only, so taking the
      // step before them changes nothing; nor does a step taken by an
      // ADVANCE that then meets the iteration bound, which ends the ray as
      // a miss.)
      bool sx = false, sy = false, sz = false;
      if (!emptied)
        dda_step_axes(d, sig, &p, (pop ? bounds : tb).min, (pop ? bounds : tb).size, scale, &sx,
                      &sy, &sz);
      const uint32_t moved = octant_of(sx, sy, sz);
      if (pop) {
        if (emptied) {
          if (key == 0u && !uniform && target != OOB_OCTANT && kind != KIND_LEAF &&
              (!LOD || !t.mips_enabled || n.mip == FORM_EMPTY ||
               mip_test_over(t, o, w.mip_level, viewing_distance))) {
            end = WALK_CRAWL;
          } else {
            // the reference's restart from the root (:551-562), which ends
            // the ray once the nudged point has left the tree (taken here,
            // not at the next iteration's start: nothing happens in
            // between)
            p = p + d * 0.1f;
            const bool inside = (p.x < t.size) & (p.y < t.size) & (p.z < t.size) &
                                (p.x > 0.0f) & (p.y > 0.0f) & (p.z > 0.0f);
            next_target = hash_region(p, t.size / 2.0f);
            next_bounds = Cube{v3u(0.0f), t.size};
            end = inside ? WALK_RUNS : WALK_MISS;
          }
        } else {
          // the parent's bounds and the sibling the step leads to
          const float s2 = bounds.size * 2.0f;
          const float rcp_s2 = size_rcp<P2>(s2);
          const V3f pmin{sub_fmod_size<P2>(bounds.min.x, s2, rcp_s2),
                         sub_fmod_size<P2>(bounds.min.y, s2, rcp_s2),
                         sub_fmod_size<P2>(bounds.min.z, s2, rcp_s2)};
          next_target = step_octant_moved(pop_octant<P2>(bounds, pmin), moved, neg);
          next_bounds = Cube{pmin, s2};
        }
      } else {
        // the rest of ADVANCE
        next_target = step_octant_moved(target, moved, neg);
        if (++steps > t.max_steps) end = WALK_GUARD;
        bp = V3f{rclamp(bp.x, lo, hi), rclamp(bp.y, lo, hi), rclamp(bp.z, lo, hi)};
        V3f move = bitmap_move<P2>(
            V3f{sx ? sig.x : 0.0f, sy ? sig.y : 0.0f, sz ? sig.z : 0.0f}, bounds.size,
            rcp_size);
        bool on = (next_target != OOB_OCTANT) & (end == WALK_RUNS);
        while (on) {
          tb = child_bounds_for(bounds, next_target);
          bp = bp + move;
          // stop at a reachable occupied child or a non-empty leaf brick;
          // both words are requested together, whichever the test needs
          const uint64_t there = lut_word(lut, bitmap_index(bp, &w.flags) * 8u + dir_idx);
          const uint32_t word = n.child[next_target];
          const bool child = (kind == KIND_INTERNAL) &
                             ((occ & octant_bitmap_mask(next_target)) != 0ull) &
                             ((there & occ) != 0ull) & (word != INVALID_INDEX);
          const bool brick =
              (kind == KIND_LEAF) & (brick_form(meta, next_target) != FORM_EMPTY);
          on = false;
          if (!(child | brick)) {
            if (++steps > t.max_steps) end = WALK_GUARD;
            dda_step_axes(d, sig, &p, tb.min, tb.size, scale, &sx, &sy, &sz);
            move = bitmap_move<P2>(
                V3f{sx ? sig.x : 0.0f, sy ? sig.y : 0.0f, sz ? sig.z : 0.0f}, bounds.size,
                rcp_size);
            next_target = step_octant_moved(next_target, octant_of(sx, sy, sz), neg);
            on = (next_target != OOB_OCTANT) & (end == WALK_RUNS);
          }
        }
      }
    }
    // PUSH shifts the stack down (its oldest entry drops out once four are
    // held), POP shifts it up, and a POP that empties it is followed by the
    // restart's push of the root; ADVANCE leaves it
    const uint32_t s0 = stk.s0, s1 = stk.s1, s2 = stk.s2, s3 = stk.s3;
    stk.s0 = push ? tword : (pop ? (emptied ? 0u : s1) : s0);
    stk.s1 = push ? s0 : (pop ? s2 : s1);
    stk.s2 = push ? s1 : (pop ? s3 : s2);
    stk.s3 = push ? s2 : s3;
    stk.count = push ? (stk.count < 4u ? stk.count + 1u : 4u)
                     : (pop ? (emptied ? 1u : stk.count - 1u) : stk.count);
    if (LOD) w.mip_level += push ? -1.0f : (pop ? 1.0f : 0.0f);
    bounds = next_bounds;
    target = next_target;
    // the next iteration would be one too many
    if (end == WALK_RUNS && steps >= t.max_steps) end = WALK_GUARD;
  }
}

// At most SLICE steps through the brick that walk_iterate marked due.
template <bool P2, int SLICE>
SVO_HD __attribute__((always_inline)) inline void walk_slice(const TreeView& t, const NodeRec* top,
                                                            uint32_t ntop, RayWalk& w) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(w.d.x), "+v"(w.d.y), "+v"(w.d.z));
#endif
  const V3f sig{sign_one(w.d.x), sign_one(w.d.y), sign_one(w.d.z)};
  const NodeRec& n = (w.stk.s0 < ntop ? top : t.nodes)[w.stk.s0];
  const bool uniform = node_kind(n.meta) == KIND_UNIFORM_LEAF;
  const Cube tb = child_bounds_for(w.bounds, w.target);
  const Cube bb{V3f{uniform ? w.bounds.min.x : tb.min.x, uniform ? w.bounds.min.y : tb.min.y,
                    uniform ? w.bounds.min.z : tb.min.z},
                uniform ? w.bounds.size : tb.size};
  bool more = false;
  if (walk_brick<P2, SLICE>(t, n.child[uniform ? 0u : w.target & 7u], bb, w.d, sig, w.scale, &w.p,
                            &w.cell, &w.flags, &more)) {
    w.end = WALK_HIT;
  } else if (!more) {
    w.cell = NO_CELL;
    w.brick = BRICK_DONE;
  }
}

// The result of a ray whose walk has ended.
template <bool LOD, bool P2>
SVO_HD __attribute__((always_inline)) inline CastResult walk_result(const TreeView& t,
                                                                   const NodeRec* top,
                                                                   uint32_t ntop, RayWalk& w) {
  CastResult r;
  r.hit = 0;
  r.flags = w.flags;
  uint32_t end = w.end;
#if defined(__HIP_DEVICE_COMPILE__)
  // (opaque here, so that the tests below are not carried through the loop)
  asm volatile("" : "+v"(end));
#endif
  if (end == WALK_CRAWL) return crawl_out_of_root(t, w.p, w.d, w.steps, r.flags);
  if (end == WALK_GUARD) r.flags |= FLAG_ITERATION_GUARD;
  const bool mip = LOD && end == WALK_HIT_MIP;
  if (end == WALK_HIT || mip) {
    // the brick that was hit, from the state the hit left as it was
    const NodeRec& n = (w.stk.s0 < ntop ? top : t.nodes)[w.stk.s0];
    const uint32_t meta = n.meta;
    const bool uniform = node_kind(meta) == KIND_UNIFORM_LEAF;
    const bool whole = uniform || mip;
    const uint32_t slot = uniform ? 0u : w.target & 7u;  // (unused by a MIP hit)
    const Cube tb = child_bounds_for(w.bounds, w.target);
    const Cube bb{V3f{whole ? w.bounds.min.x : tb.min.x, whole ? w.bounds.min.y : tb.min.y,
                      whole ? w.bounds.min.z : tb.min.z},
                  whole ? w.bounds.size : tb.size};
    brick_hit<P2>(t, mip ? n.mip : brick_form(meta, slot), mip ? n.mip_word : n.child[slot], bb,
                  w.cell, w.p, &r);
  }
  return r;
}

template <bool LOD, bool P2, class LutT>
SVO_HD __attribute__((always_inline)) inline CastResult cast_ray_impl(
    const TreeView& t, const LutT* __restrict__ lut, V3f o, V3f d, const NodeRec* top,
    uint32_t ntop, float viewing_distance) {
  RayWalk w;
  walk_begin<LOD>(t, o, d, w);
  if (w.end != WALK_RUNS) return miss_flags(0u);
  do {
    walk_iterate<LOD, P2, false>(t, lut, o, top, ntop, viewing_distance, w);
  } while (w.end == WALK_RUNS);
  return walk_result<LOD, P2>(t, top, ntop, w);
}

// The same traversal as cast_ray_impl<false, P2> with the work of a wave
// regrouped (the "while-while" arrangement of GPU ray traversal): each lane
// runs stack-loop iterations until its next iteration starts with a brick
// probe, or its ray ends; the wave then probes the due bricks of all such
// lanes together, and the rounds repeat. Every lane performs the same
// operations in the same order as in cast_ray_impl (an iteration interrupted
// for its probe resumes after it, re-reading its node record and without
// counting a second step), so results are identical bit for bit; only the
// interleaving across lanes differs, which keeps more lanes active in the
// brick DDA loop. (Ending a round's first phase early, once a quorum of
// the wave's lanes wait for their probes, measured slower.)
//
// CRAWL = false leaves out the crawl_out_of_root shortcut (the restarts are
// then run one by one, with the same result; the host tests run both forms).
template <bool P2, class LutT, bool CRAWL = true>
SVO_HD __attribute__((always_inline)) inline CastResult cast_ray_ww(
    const TreeView& t, const LutT* __restrict__ lut, V3f o, V3f d, const NodeRec* top,
    uint32_t ntop) {
  // (here, unlike in cast_ray_impl, zeroing the hit fields up front gives
  // the smaller register allocation, and measured 4% faster)
  CastResult r = miss_result(0u);

  const V3f scale = dda_scale_factors(d);
  const uint32_t dir_idx = hash_direction(d);
  const Cube root{v3u(0.0f), t.size};
  const float lo = 0.00001f;
  const float hi = 4.0f - 0.00001f;

  RingStack stk{0u, 0u, 0u, 0u, 1u};  // the root pushed
  Cube bounds = root;
  V3f p;
  uint32_t target;
  {
    float tt = 0.0f;
    const int ir = intersect_ray(root, o, d, &tt);
    if (ir != 0) {
      p = o + d * (ir == 2 ? tt : 0.0f);
      target = hash_region(p - root.min, root.size / 2.0f);
    } else {
      p = o;
      target = OOB_OCTANT;
    }
  }
  bool finished = target == OOB_OCTANT;
  bool probed = false;  // the current iteration's probe has run
  bool crawl = false;   // the ray ends in crawl_out_of_root, after the loop
  uint32_t steps = 0;
  for (;;) {
    // phase 1: stack-loop iterations up to the next due probe
    bool due = false;
    while (!finished) {
      // signum(d), formed in each iteration as in cast_ray_impl
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(d.x), "+v"(d.y), "+v"(d.z));
#endif
      const V3f sig{sign_one(d.x), sign_one(d.y), sign_one(d.z)};
      if (stk.count == 0u) {
        // restart from the root (:551-562)
        p = p + d * 0.1f;
        target = ((p.x < t.size) & (p.y < t.size) & (p.z < t.size) & (p.x > 0.0f) & (p.y > 0.0f) &
                   (p.z > 0.0f))
                     ? hash_region(p, t.size / 2.0f)
                     : OOB_OCTANT;
        if (target == OOB_OCTANT) {
          finished = true;
          break;
        }
        bounds = root;
        stk.push(0u);
      }
      if (!probed && ++steps > t.max_steps) {
        r.flags |= FLAG_ITERATION_GUARD;
        finished = true;
        break;
      }
      const uint32_t key = stk.s0;
      const NodeRec& n = (key < ntop ? top : t.nodes)[key];
      const uint64_t occ = n.occ;
      const uint32_t meta = n.meta;
      const uint32_t tword = n.child[target & 7u];
      const uint32_t kind = node_kind(meta);
      if (!probed && target != OOB_OCTANT && (kind == KIND_UNIFORM_LEAF || kind == KIND_LEAF)) {
        due = true;
        break;
      }
      probed = false;
      const bool backtrack = kind == KIND_UNIFORM_LEAF;
      const float rcp_size = size_rcp<P2>(bounds.size);
      V3f bp = bitmap_pos<P2>(p, bounds, rcp_size);
      uint32_t flat = bitmap_cell(bp);  // cell of the clamped position
      if (backtrack || target == OOB_OCTANT || occ == 0ull ||
          (occ & lut[flat * 8u + dir_idx]) == 0ull) {
        // POP (:445-475); a root with nothing ahead of the ray ends the
        // ray as crawl_out_of_root does, which runs after the loop (where
        // the loop's state is no longer live)
        if (CRAWL && stk.count == 1u && key == 0u && !backtrack && target != OOB_OCTANT &&
            kind != KIND_LEAF) {
          crawl = true;
          finished = true;
          break;
        }
        stk.pop();
        if (stk.count != 0u) {
          const float s2 = bounds.size * 2.0f;
          const float rcp_s2 = size_rcp<P2>(s2);
          const V3f pmin{sub_fmod_size<P2>(bounds.min.x, s2, rcp_s2),
                         sub_fmod_size<P2>(bounds.min.y, s2, rcp_s2),
                         sub_fmod_size<P2>(bounds.min.z, s2, rcp_s2)};
          const uint32_t from = pop_octant<P2>(bounds, pmin);
          const V3f st = dda_step(d, sig, &p, bounds, scale);
          target = step_octant(from, st);
          bounds.size *= 2.0f;
          bounds.min = pmin;
        }
        continue;
      }
      Cube tb = child_bounds_for(bounds, target);
      uint32_t tck = INVALID_INDEX;
      if (kind == KIND_INTERNAL && (occ & octant_bitmap_mask(target)) != 0ull) tck = tword;
      if (tck != INVALID_INDEX) {
        // PUSH (:484-492)
        bounds = tb;
        target = hash_region(p - tb.min, tb.size / 2.0f);
        stk.push(tck);
      } else {
        // ADVANCE (:497-544), from the clamped position
        bp = V3f{rclamp(bp.x, lo, hi), rclamp(bp.y, lo, hi), rclamp(bp.z, lo, hi)};
        for (;;) {
          if (++steps > t.max_steps) {
            r.flags |= FLAG_ITERATION_GUARD;
            finished = true;
            break;
          }
          const V3f st = dda_step(d, sig, &p, tb, scale);
          target = step_octant(target, st);
          if (target == OOB_OCTANT) break;
          tb = child_bounds_for(bounds, target);
          bp = bp + bitmap_move<P2>(st, bounds.size, rcp_size);
          flat = bitmap_index(bp, &r.flags);
          if (kind == KIND_LEAF && brick_form(meta, target) != FORM_EMPTY) break;
          if (kind == KIND_INTERNAL && (occ & octant_bitmap_mask(target)) != 0ull &&
              (lut[flat * 8u + dir_idx] & occ) != 0ull && n.child[target] != INVALID_INDEX)
            break;
        }
      }
    }
    if (finished) break;
    if (!due) continue;
    // phase 2: the due probe of the iteration, lanes of the wave together
    {
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(d.x), "+v"(d.y), "+v"(d.z));
#endif
      const V3f sig{sign_one(d.x), sign_one(d.y), sign_one(d.z)};
      const NodeRec& n = (stk.s0 < ntop ? top : t.nodes)[stk.s0];
      const uint32_t meta = n.meta;
      const bool uniform = node_kind(meta) == KIND_UNIFORM_LEAF;
      const uint32_t slot = uniform ? 0u : target;
      if (probe_brick<P2>(t, brick_form(meta, slot), n.child[slot],
                          uniform ? bounds : child_bounds_for(bounds, target), d, sig, scale,
                          &p, &r)) {
        r.hit = 1;
        return r;
      }
      probed = true;
    }
  }
  if (crawl) r.flags = crawl_out_of_root(t, p, d, steps, r.flags).flags;
  return r;
}

template <bool P2 = false, class LutT>
SVO_HD __attribute__((always_inline)) inline CastResult cast_ray(const TreeView& t,
                                                                const LutT* __restrict__ lut,
                                                                V3f o, V3f d,
                                                                const NodeRec* top = nullptr,
                                                                uint32_t ntop = 0u) {
  return cast_ray_impl<false, P2>(t, lut, o, d, top, ntop, 0.0f);
}

template <bool P2 = false, class LutT>
SVO_HD __attribute__((always_inline)) inline CastResult cast_ray_lod(
    const TreeView& t, const LutT* __restrict__ lut, V3f o, V3f d, float viewing_distance) {
  return cast_ray_impl<true, P2>(t, lut, o, d, nullptr, 0u, viewing_distance);
}

template <bool P2 = false>
SVO_HD __attribute__((always_inline)) inline CastResult cast_ray(const TreeView& t, V3f o,
                                                                V3f d) {
  return cast_ray<P2>(t, t.ray_lut, o, d);
}

// The same traversal as cast_ray in resumable form: ray_begin sets a ray up,
// each ray_step runs one iteration of the stack loop (and the restart from
// the root when the stack empties). A kernel can then hand a finished lane a
// new ray while the other lanes of its wave keep stepping. The operation
// sequence per ray is identical to cast_ray's. Only the traversal state and
// the flags live across steps; the result is written when the ray finishes.
struct RayState {
  V3f d, scale, p;
  Cube bounds;
  uint32_t head, count, target, steps, flags;
  // the ring stack's four slots as separate scalars: a dynamically indexed
  // array inside the state would be kept in scratch memory
  uint32_t stk0, stk1, stk2, stk3;
  SVO_HD uint32_t stk_get(uint32_t i) const {
    return i == 0u ? stk0 : (i == 1u ? stk1 : (i == 2u ? stk2 : stk3));
  }
  SVO_HD void stk_set(uint32_t i, uint32_t v) {
    stk0 = i == 0u ? v : stk0;
    stk1 = i == 1u ? v : stk1;
    stk2 = i == 2u ? v : stk2;
    stk3 = i == 3u ? v : stk3;
  }
};

// false when the ray misses the tree outright (its result is miss_result(0))
SVO_HD __attribute__((always_inline)) inline bool ray_begin(const TreeView& t, V3f o, V3f d,
                                                           RayState& s) {
  s.d = d;
  s.scale = dda_scale_factors(d);
  const Cube root{v3u(0.0f), t.size};
  float tt = 0.0f;
  const int ir = intersect_ray(root, o, d, &tt);
  if (ir == 0) return false;
  s.p = o + d * (ir == 2 ? tt : 0.0f);
  s.target = hash_region(s.p - root.min, root.size / 2.0f);
  if (s.target == OOB_OCTANT) return false;
  s.bounds = root;
  s.stk0 = 0u;
  s.stk1 = 0u;
  s.stk2 = 0u;
  s.stk3 = 0u;
  s.head = 1u;
  s.count = 1u;
  s.steps = 0u;
  s.flags = 0u;
  return true;
}

// true when the ray is finished; r then holds its result
template <class LutT>
SVO_HD __attribute__((always_inline)) inline bool ray_step(const TreeView& t,
                                                          const LutT* __restrict__ lut,
                                                          RayState& s, CastResult& r) {
  const float lo = 0.00001f;
  const float hi = 4.0f - 0.00001f;
  if (++s.steps > t.max_steps) {
    r = miss_result(s.flags | FLAG_ITERATION_GUARD);
    return true;
  }
  // cheap functions of the direction, recomputed rather than kept per lane
  const V3f sig{rsignum(s.d.x), rsignum(s.d.y), rsignum(s.d.z)};
  const uint32_t dir_idx = hash_direction(s.d);
  const NodeRec& n = t.nodes[s.stk_get(s.head)];
  const uint64_t occ = n.occ;
  const uint32_t meta = n.meta;
  const uint32_t kind = node_kind(meta);
  bool backtrack = kind == KIND_UNIFORM_LEAF;
  if (s.target != OOB_OCTANT && kind != KIND_INTERNAL && kind != KIND_NOTHING) {
    const bool uniform = kind == KIND_UNIFORM_LEAF;
    const uint32_t slot = uniform ? 0u : s.target;
    CastResult hr = miss_result(0u);
    if (probe_brick<false>(t, brick_form(meta, slot), n.child[slot],
                           uniform ? s.bounds : child_bounds_for(s.bounds, s.target), s.d, sig,
                           s.scale, &s.p, &hr)) {
      r = hr;
      r.hit = 1;
      r.flags = s.flags | hr.flags;
      return true;
    }
    s.flags |= hr.flags;
  }
  const float rcp_size = pow2_rcp(s.bounds.size);
  const V3f rel = (s.p - s.bounds.min) * 4.0f;
  V3f bp = div3_by(rel, s.bounds.size, rcp_size);
  bp = V3f{rclamp(bp.x, lo, hi), rclamp(bp.y, lo, hi), rclamp(bp.z, lo, hi)};
  uint32_t flat = bitmap_index(bp, &s.flags);
  if (backtrack || s.target == OOB_OCTANT || occ == 0ull ||
      (occ & lut[flat * 8u + dir_idx]) == 0ull) {
    // POP
    s.head = (s.head + 3u) & 3u;
    s.count -= 1u;
    if (s.count != 0u) {
      const V3f center = s.bounds.min + v3u(s.bounds.size / 2.0f);
      const float s2 = s.bounds.size * 2.0f;
      const float rcp_s2 = pow2_rcp(s2);
      const V3f pmin{sub_fmod(s.bounds.min.x, s2, rcp_s2), sub_fmod(s.bounds.min.y, s2, rcp_s2),
                     sub_fmod(s.bounds.min.z, s2, rcp_s2)};
      const uint32_t from = hash_region(center - pmin, s.bounds.size);
      const V3f st = dda_step(s.d, sig, &s.p, s.bounds, s.scale);
      s.target = step_octant(from, st);
      s.bounds.size *= 2.0f;
      s.bounds.min = pmin;
    }
  } else {
    Cube tb = child_bounds_for(s.bounds, s.target);
    uint32_t tck = INVALID_INDEX;
    if (kind == KIND_INTERNAL && (occ & octant_bitmap_mask(s.target)) != 0ull)
      tck = n.child[s.target];
    if (tck != INVALID_INDEX) {
      // PUSH
      s.bounds = tb;
      s.target = hash_region(s.p - tb.min, tb.size / 2.0f);
      s.head = (s.head + 1u) & 3u;
      s.count = s.count < 4u ? s.count + 1u : 4u;
      s.stk_set(s.head, tck);
    } else {
      // ADVANCE
      for (;;) {
        if (++s.steps > t.max_steps) {
          r = miss_result(s.flags | FLAG_ITERATION_GUARD);
          return true;
        }
        const V3f st = dda_step(s.d, sig, &s.p, tb, s.scale);
        s.target = step_octant(s.target, st);
        if (s.target == OOB_OCTANT) break;
        tb = child_bounds_for(s.bounds, s.target);
        const V3f sd = st * 4.0f;
        bp = bp + div3_by(sd, s.bounds.size, rcp_size);
        flat = bitmap_index(bp, &s.flags);
        if (kind == KIND_LEAF && brick_form(meta, s.target) != FORM_EMPTY) break;
        if (kind == KIND_INTERNAL && (occ & octant_bitmap_mask(s.target)) != 0ull &&
            (lut[flat * 8u + dir_idx] & occ) != 0ull && n.child[s.target] != INVALID_INDEX)
          break;
      }
    }
  }
  if (s.count == 0u) {
    // restart from the root
    s.p = s.p + s.d * 0.1f;
    s.target = (s.p.x < t.size && s.p.y < t.size && s.p.z < t.size && s.p.x > 0.0f &&
                s.p.y > 0.0f && s.p.z > 0.0f)
                   ? hash_region(s.p, t.size / 2.0f)
                   : OOB_OCTANT;
    if (s.target == OOB_OCTANT) {
      r = miss_result(s.flags);
      return true;
    }
    s.bounds = Cube{v3u(0.0f), t.size};
    s.head = (s.head + 1u) & 3u;
    s.count = 1u;
    s.stk_set(s.head, 0u);
  }
  return false;
}

// Voxel coordinate of a hit: floor(impact) clamped into the hit cell.
SVO_HD inline uint32_t hit_voxel_axis(float p, float cmin, float csize) {
  float f = floorf(p);
  const float hi = cmin + csize - 1.0f;
  f = f < cmin ? cmin : (f > hi ? hi : f);
  return f2u32(f);
}

// Ray of pixel (x, y) of a pinhole viewport (y = 0 is the bottom row), as the
// reference's CPU harness builds it (examples/cpu_render.rs:104-114) with the
// ray through the pixel centre.
struct Camera {
  V3f origin;
  V3f bottom_left;
  V3f right;
  V3f up;
  float pixel_w;
  float pixel_h;
};

// Camera of a Viewport{origin, direction, frustum, fov} (bevy/types.rs:55-71)
// as the reference's CPU harness derives it (examples/cpu_render.rs:78-94):
// up = +y, right = normalize(up x direction), glass `fov` in front of the eye.
SVO_HD inline Camera make_camera(V3f origin, V3f dir, float glass_w, float glass_h, float fov,
                                 uint32_t w, uint32_t h) {
  const V3f up{0.0f, 1.0f, 0.0f};
  Camera cam;
  cam.origin = origin;
  cam.up = up;
  cam.right = normalized(cross(up, dir));
  cam.pixel_w = glass_w / static_cast<float>(w);
  cam.pixel_h = glass_h / static_cast<float>(h);
  cam.bottom_left = ((origin + dir * fov) - up * (glass_h / 2.0f)) - cam.right * (glass_w / 2.0f);
  return cam;
}

SVO_HD inline V3f camera_ray_dir(const Camera& c, uint32_t x, uint32_t y) {
  const float fx = static_cast<float>(x) + 0.5f;
  const float fy = static_cast<float>(y) + 0.5f;
  const V3f glass = (c.bottom_left + (c.right * fx) * c.pixel_w) + (c.up * fy) * c.pixel_h;
  return normalized(glass - c.origin);
}

// Whether the camera looks down (or level): its image's top rows then hold the
// rays nearest to the horizon, which graze the most content. A launch ends
// with its slowest tiles, so the kernels that hand out an image's tiles in
// order begin with those rows (row 0 is the bottom): 1080p caves frame 184 ->
// 169 us, 4K heightfield frame 526 -> 503 us, eight 1080p frames in one run
// 738 -> 714 us; 720p over spheres 145 -> 149 us. (An image drawn top row
// first, begun at the bottom instead: 123 -> 125 us.)
SVO_HD inline bool looks_down(const Camera& c, uint32_t w, uint32_t h) {
  const float x = 0.5f * static_cast<float>(w) * c.pixel_w;
  const float y = 0.5f * static_cast<float>(h) * c.pixel_h;
  return !(c.bottom_left.y + c.right.y * x + c.up.y * y - c.origin.y > 0.0f);
}

}  // namespace svo
