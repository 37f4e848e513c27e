// ft_cells.h — spatial cells: per cell of a uniform grid over the scene, what can decide the
// scene distance at any point of the cell.  Built once per scene on the GPU (the kernels at
// the end), read by every distance evaluation.
//
// Leaf lists (scenes of many accel leaves).  The distance over a spine of hard unions is the
// least leaf distance.  Every primitive's distance changes by at most the distance moved, so
// with R the cell's half diagonal a leaf whose distance at the cell's centre exceeds the
// least one there by more than 2R is not the nearest anywhere in the cell, and the cell keeps
// the others.
//
// Cell programs (scenes of one accel leaf, a tree of blends).  Per cell the node program
// without the subtrees that cannot show through: an interval of every node's distance over
// the cell decides at each join whether one operand dominates it everywhere in the cell.
//
// In both a lane walks the entries of its own cell, so lanes whose rays have parted cost no
// more than lanes that march side by side.  Before, a wave evaluated the union of what its
// lanes needed in step: every node of a tree, or the BVH nodes and leaves of all its points.
// Measured, before and after: 1920x1080 Whitted frame of 4097 leaves 204 -> 17 ms, preview of 1501
// leaves at 1001x563 18.0 -> 0.88 ms, a batch of 12 scenes (8 to 2048 primitives) x 4 views at
// 256x256 777 -> 7.2 ms, of 5 scenes x 3 views at 61x37 15.0 -> 0.72 ms.  What bounds them now is
// VALU issue and the return path of the gathers together.
#pragma once

namespace ftd {

// Per-lane loads through a wave-uniform base pointer as global (not flat) accesses.
#if defined(__HIP_DEVICE_COMPILE__)
#define FT_GLOBAL_AS __attribute__((address_space(1)))
#else
#define FT_GLOBAL_AS
#endif
__device__ __forceinline__ float4 global_load4(const float4* base, unsigned i) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  const v4 v = ((const FT_GLOBAL_AS v4*)(unsigned long long)base)[i];
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ int4 global_load4(const int4* base, unsigned i) {
  typedef int v4 __attribute__((ext_vector_type(4)));
  const v4 v = ((const FT_GLOBAL_AS v4*)(unsigned long long)base)[i];
  return make_int4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 global_load2(const unsigned* base, unsigned i) {
  typedef unsigned v2 __attribute__((ext_vector_type(2)));
  const v2 v = *(const FT_GLOBAL_AS v2*)((const FT_GLOBAL_AS unsigned*)(unsigned long long)base + i);
  return make_uint2(v.x, v.y);
}
__device__ __forceinline__ unsigned global_load(const unsigned* base, unsigned i) {
  return ((const FT_GLOBAL_AS unsigned*)(unsigned long long)base)[i];
}

// ------------------------------------------------------------------ leaf lists
// One primitive of a leaf list.  The kinds share one formula, v = (max(ax, lo), ...),
// d = |v| + inside - off, whose terms are those of sdf_sphere / sdf_box / sdf_cylinder /
// sdf_torus (q = p - c, radial = sqrt(qx^2 + qz^2)):
//   sphere    a = |q|                          lo = -inf  off = radius
//   box       a = |q| - half                   lo = 0     off = rounding  inside = min(max a, 0)
//   cylinder  a = (radial - r, |qy| - h, -inf) lo = 0     off = rounding  inside = min(max a, 0)
//   torus     a = (radial - R, |qy|, 0)        lo = -inf  off = r
// so lanes with primitives of different kinds run the same instructions.
__device__ __forceinline__ float common_distance(float3 q, float ex, float ey, float ez, float off, bool radial,
                                                 bool clamped) {
  const float lo = clamped ? 0.0f : -__builtin_huge_valf();
  const float ax = (radial ? fsqrt(q.x * q.x + q.z * q.z) : fabsf(q.x)) - ex;
  const float ay = fabsf(q.y) - ey;
  const float az = radial ? (clamped ? -__builtin_huge_valf() : 0.0f) : fabsf(q.z) - ez;
  const float outside = len(mk(fmaxf(ax, lo), fmaxf(ay, lo), fmaxf(az, lo)));
  const float inside = clamped ? fminf(fmaxf(fmaxf(ax, ay), az), 0.0f) : 0.0f;
  return outside + inside - off;
}
__device__ __forceinline__ float leaf_prim_distance(const float4 A, const float4 B, float3 p) {
  const int flags = __float_as_int(A.w);
  return common_distance(mk(p.x - A.x, p.y - A.y, p.z - A.z), B.x, B.y, B.z, B.w, (flags & kLeafRadial) != 0,
                         (flags & kLeafClamped) != 0);
}

// The grid cell of p, -1 outside (NaN included).
__device__ __forceinline__ int cell_of(const DevScene& S, float3 p) {
  const float x = (p.x - S.cell_org[0]) * S.cell_inv, y = (p.y - S.cell_org[1]) * S.cell_inv,
              z = (p.z - S.cell_org[2]) * S.cell_inv;
  const bool in = x >= 0.0f && y >= 0.0f && z >= 0.0f && x < (float)S.cell_dims[0] && y < (float)S.cell_dims[1] &&
                  z < (float)S.cell_dims[2];
  return in ? ((int)z * S.cell_dims[1] + (int)y) * S.cell_dims[0] + (int)x : -1;
}

// bvh_distance_body's answer from the leaf list of p's cell.  The primitives of a list are in
// ascending rank (the order that decides between leaves of negative distance: the first such
// leaf is the answer), the leaves that need a program or a function come last and are
// evaluated where the reference's pruning test leaves them open.
template <bool kInfo>
__device__ __forceinline__ Info list_distance(const DevScene& S, int slot, int cell, float3 p) {
  const int4 r = global_load4(S.cell_lists, (unsigned)cell);
  const unsigned first = (unsigned)r.x;
  const int n = r.y & 0xffff, n_generic = r.y >> 16;
  float best = __builtin_huge_valf();
  int bj = -1;
  for (int k = 0; k < n; k += 2) {  // lists are padded to pairs with a primitive at infinity
    const uint2 it = global_load2(S.cell_items, first + (unsigned)k);
    const float4 A0 = global_load4(S.leaf_prims, 2 * it.x), B0 = global_load4(S.leaf_prims, 2 * it.x + 1);
    const float4 A1 = global_load4(S.leaf_prims, 2 * it.y), B1 = global_load4(S.leaf_prims, 2 * it.y + 1);
    const float d0 = leaf_prim_distance(A0, B0, p), d1 = leaf_prim_distance(A1, B1, p);
    if (d0 < best && best >= 0.0f) { best = d0; bj = (int)it.x; }
    if (d1 < best && best >= 0.0f) { best = d1; bj = (int)it.y; }
  }
  Info out;
  out.d = best;
  out.lb = best;
  out.obj = 0u;
  out.mat = 0u;
  out.leaf = -1;
  if (bj >= 0) out.leaf = __float_as_int(global_load4(S.leaf_boxes, 2u * (unsigned)bj).w);
  int rank = bj >= 0 ? __float_as_int(global_load4(S.leaf_boxes, 2u * (unsigned)bj + 1u).w) : 0x7fffffff;
  bool prim = bj >= 0;
  for (int k = 0; __builtin_amdgcn_ballot_w64(k < n_generic) != 0ull; ++k) {
    int li = -1, lr = 0;
    if (k < n_generic) {
      const unsigned j = global_load(S.cell_items, first + (unsigned)(((n + 1) & ~1) + k));
      const float4 lo = global_load4(S.leaf_boxes, 2 * j), hi = global_load4(S.leaf_boxes, 2 * j + 1);
      const float lb = aabb_lb_lit(p, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z);
      lr = __float_as_int(hi.w);
      if (!(lb > best) || (best < 0.0f && lb == 0.0f && lr < rank)) li = __float_as_int(lo.w);
    }
    if (li >= 0) {
      Info info;
      for_each_uniform(li, [&](int lead) { info = leaf_info_uniform<kInfo>(S, slot, lead, p); });
      const bool take = best < 0.0f ? (info.d < 0.0f && lr < rank) : info.d < best;
      if (take) {
        best = info.d;
        rank = lr;
        out = info;
        prim = false;
      }
    }
  }
  if (kInfo && prim) {
    const DNode& w = S.nodes[S.leaves[out.leaf].node];
    out.obj = w.obj;
    out.mat = w.mat;
  }
  if (S.flops) {
    float cost = 0.0f;
    for (int k = 0; k < n; ++k) {
      const int li = __float_as_int(global_load4(S.leaf_boxes, 2 * global_load(S.cell_items, first + (unsigned)(k))).w);
      if (li >= 0) cost += S.nodes[S.leaves[li].node].cost;
    }
    atomicAdd(S.flops, (unsigned long long)cost);
  }
  return out;
}

// bvh_walk_leaf's answer from the leaf list of p's cell.
__device__ __noinline__ int list_walk_leaf(int slot, int cell, float3 p) {
  const DevScene& S = scene_of(slot);
  const int4 r = global_load4(S.cell_lists, (unsigned)cell);
  const unsigned first = (unsigned)r.x;
  const int n = r.y & 0xffff, n_generic = r.y >> 16;
  float best = __builtin_huge_valf();
  int leaf = -1;
  for (int k = 0; k < n; ++k) {
    const unsigned j = global_load(S.cell_items, first + (unsigned)(k));
    const float d = leaf_prim_distance(global_load4(S.leaf_prims, 2 * j), global_load4(S.leaf_prims, 2 * j + 1), p);
    const int li = __float_as_int(global_load4(S.leaf_boxes, 2 * j).w);
    if (li >= 0 && (leaf < 0 || d < best || (d == best && li < leaf))) {
      best = d;
      leaf = li;
    }
  }
  for (int k = 0; __builtin_amdgcn_ballot_w64(k < n_generic) != 0ull; ++k) {
    int li = -1;
    if (k < n_generic) {
      const unsigned j = global_load(S.cell_items, first + (unsigned)(((n + 1) & ~1) + k));
      const float4 lo = global_load4(S.leaf_boxes, 2 * j), hi = global_load4(S.leaf_boxes, 2 * j + 1);
      if (aabb_lb_lit(p, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z) <= fmaxf(best, 0.0f)) li = __float_as_int(lo.w);
    }
    if (li >= 0) {
      float d = 0.0f;
      for_each_uniform(li, [&](int lead) { d = leaf_info_uniform(S, slot, lead, p, false).d; });
      if (leaf < 0 || d < best || (d == best && li < leaf)) {
        best = d;
        leaf = li;
      }
    }
  }
  return leaf;
}

// bvh_lower_bound's answer from the box list of p's cell: the least AABB bound, or some value
// at or below `stop`.
__device__ __forceinline__ float list_lower_bound(const DevScene& S, int cell, float3 p, float stop) {
  const int4 r = global_load4(S.cell_lists, (unsigned)cell);
  const unsigned first = (unsigned)r.z;
  float best = __builtin_huge_valf();
  for (int k = 0; k < r.w && best > stop; ++k) {
    const unsigned j = global_load(S.cell_items, first + (unsigned)(k));
    const float4 lo = global_load4(S.leaf_boxes, 2 * j), hi = global_load4(S.leaf_boxes, 2 * j + 1);
    best = fminf(best, aabb_lb_lit(p, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z));
  }
  return best;
}

// ------------------------------------------------------------------ cell programs
// What remains at a join: both operands, or the only one left.  The distance of what remains is
// the full program's bit for bit: a join keeps one operand only where its formula gives the
// same value for every larger (in a mirrored join, smaller) value of the other, which is
// then replaced by infinity.
constexpr int kOneBoth = 0, kOneLeft = 1, kOneRight = 2;

// Distance words, 8 bytes each: a primitive, the join that follows it, or both.
//   x: place of the primitive in the scene program (or of the join, where there is none) and
//      its form; what the join is: which operands remain and its formula on operands brought
//      to a union's (a blended intersection of a and b is -union(-a, -b), a difference
//      -union(-a, b), negations that are exact)
//   y: the join's radius; of stairs, whose count is needed too, the join's place
// Shading words, 4 bytes each: the x word of every node that remains, a word of its own for
// each, joins that leave their operand as it is included (their blend still normalises).
// The words carry the flags and the radius so that a word costs 8 + 16 + 12 bytes of gathers (with
// separate join records 56): the return path of the vector loads, not the arithmetic, is what
// the walk fills first (TD busy 84% of the 1080p frame's cycles at 56 bytes).
constexpr unsigned kWordNode = 0xfffffu;  // programs of up to 2^20 words
constexpr unsigned kWordRadial = 1u << 20, kWordClamped = 1u << 21, kWordExtended = 1u << 22;
constexpr int kWordOneShift = 23, kWordTypeShift = 25;
constexpr unsigned kWordFlipA = 1u << 28, kWordFlipB = 1u << 29, kWordJoin = 1u << 30, kWordPrim = 1u << 31;
enum { kJoinHard = 0, kJoinRound = 1, kJoinChamfer = 2, kJoinStairs = 3, kJoinSoft = 4 };

__device__ __forceinline__ bool is_diff(int kind) {
  return kind == FT_NODE_SUBTRACT || kind == FT_NODE_DIFF_ROUND || kind == FT_NODE_DIFF_CHAMFER ||
         kind == FT_NODE_DIFF_STAIRS;
}
__host__ __device__ __forceinline__ unsigned prim_word(const DOp& o, int k) {
  const int kind = o.code & kOpKindMask;
  const float shell = kind == FT_NODE_SPHERE ? o.p[1] : (kind == FT_NODE_BOX ? o.p[4] : (kind == FT_NODE_CYLINDER ? o.p[3] : 0.0f));
  unsigned w = kWordPrim | (unsigned)k;
  if (kind == FT_NODE_CYLINDER || kind == FT_NODE_TORUS) w |= kWordRadial;
  if (kind == FT_NODE_BOX || kind == FT_NODE_CYLINDER) w |= kWordClamped;
  if ((o.code & kOpRotated) || shell > 0.0f) w |= kWordExtended;
  return w;
}
__host__ __device__ __forceinline__ unsigned join_word(int kind, int one) {
  const unsigned w = kWordJoin | ((unsigned)one << kWordOneShift);
  const unsigned both = kWordFlipA | kWordFlipB, round = kJoinRound << kWordTypeShift,
                 chamfer = kJoinChamfer << kWordTypeShift, stairs = kJoinStairs << kWordTypeShift;
  switch (kind) {
    case FT_NODE_UNION_ROUND: return w | round;
    case FT_NODE_UNION_CHAMFER: return w | chamfer;
    case FT_NODE_UNION_STAIRS: return w | stairs;
    case FT_NODE_UNION_SOFT: return w | (kJoinSoft << kWordTypeShift);
    case FT_NODE_INTERSECT: return w | both;
    case FT_NODE_INTERSECT_ROUND: return w | round | both;
    case FT_NODE_INTERSECT_CHAMFER: return w | chamfer | both;
    case FT_NODE_INTERSECT_STAIRS: return w | stairs | both;
    case FT_NODE_SUBTRACT: return w | kWordFlipA;
    case FT_NODE_DIFF_ROUND: return w | round | kWordFlipA;
    case FT_NODE_DIFF_CHAMFER: return w | chamfer | kWordFlipA;
    default: return w | stairs | kWordFlipA;  // DIFF_STAIRS
  }
}
// a join's y word
__host__ __device__ __forceinline__ unsigned join_value(const DOp& o, int k) {
  const int kind = o.code & kOpKindMask;
  if (kind == FT_NODE_UNION_STAIRS || kind == FT_NODE_INTERSECT_STAIRS || kind == FT_NODE_DIFF_STAIRS) return (unsigned)k;
  const bool raw = kind == FT_NODE_UNION_CHAMFER || kind == FT_NODE_INTERSECT_CHAMFER || kind == FT_NODE_DIFF_CHAMFER;
  union {
    float f;
    unsigned u;
  } v;
  v.f = raw ? o.p[0] : fmaxf(fabsf(o.p[0]), 1.0e-6f);
  return v.u;
}
__device__ __forceinline__ float flip_sign(float x, unsigned bit31) {
  return __uint_as_float(__float_as_uint(x) ^ (bit31 & 0x80000000u));
}

// The value of a join whose other operand is out of reach (x: the operand that remains).
__device__ __forceinline__ float join_one(int kind, float x, bool right, float rr) {
  if (right && is_diff(kind)) x = -x;
  if (kind == FT_NODE_UNION_ROUND) return op_union_round(x, __builtin_huge_valf(), rr);
  if (kind == FT_NODE_DIFF_ROUND) return op_intersect_round(x, -__builtin_huge_valf(), rr);
  return x;
}

// What the evaluation of cell programs reads of the scene, and the lane's column of the LDS
// value stack: loaded once per march and kept in registers, since reading them again through
// the descriptor (and the block size) at each step put several dependent loads in front of
// every distance.
struct ProgramView {
  float ox, oy, oz, inv, fx, fy, fz;
  int nx, nxy, outside;
  const int4* cells;
  const unsigned* words;
  const float4* ops;
  const float4* ext;
  float* stack;  // this lane's entry 0 of the value plane
  int step;      // floats between entries
  int id_plane;  // floats from the value plane to the id plane
  __device__ __forceinline__ explicit ProgramView(const DevScene& S) {
    ox = S.cell_org[0];
    oy = S.cell_org[1];
    oz = S.cell_org[2];
    inv = S.cell_inv;
    fx = (float)S.cell_dims[0];
    fy = (float)S.cell_dims[1];
    fz = (float)S.cell_dims[2];
    nx = S.cell_dims[0];
    nxy = nx * S.cell_dims[1];
    outside = nxy * S.cell_dims[2];
    cells = S.cell_progs;
    words = S.cell_words;
    ops = S.cell_ops;
    ext = S.cell_ext;
    step = blockDim.x * blockDim.y;
    stack = ft_lds + threadIdx.y * blockDim.x + threadIdx.x;
    id_plane = 2 * S.stack_depth * step;
  }
  // the cell of p; the entry after the last cell is the whole program, for the points outside
  __device__ __forceinline__ unsigned cell(float3 p) const {
    const float x = (p.x - ox) * inv, y = (p.y - oy) * inv, z = (p.z - oz) * inv;
    const bool in = x >= 0.0f && y >= 0.0f && z >= 0.0f && x < fx && y < fy && z < fz;
    return (unsigned)(in ? (int)z * nxy + (int)y * nx + (int)x : outside);
  }
};

// A primitive of the cell programs: record A = centre, off, E = the extents; with a rotation
// and a shell where it names an extension (two float4: the three sin / cos pairs, the shell).
__device__ __forceinline__ float cell_prim_distance(const ProgramView& V, unsigned w, const float4 A, const float3 E,
                                                    float3 p) {
  float3 q = mk(p.x - A.x, p.y - A.y, p.z - A.z);
  float shell = 0.0f;
  if (w & kWordExtended) {
    const unsigned e = __float_as_uint(global_load4(V.ops, 2u * (w & kWordNode) + 1u).w) & kExtIndex;
    const float4 r0 = global_load4(V.ext, 2u * e), r1 = global_load4(V.ext, 2u * e + 1u);
    if (r1.w != 0.0f) {
      q = rot_z(q, r0.x, r0.y);
      q = rot_y(q, r0.z, r0.w);
      q = rot_x(q, r1.x, r1.y);
    }
    shell = r1.z;
  }
  const float d = common_distance(q, E.x, E.y, E.z, A.w, (w & kWordRadial) != 0u, (w & kWordClamped) != 0u);
  return (w & kWordExtended) ? shell_op(d, shell) : d;
}
__device__ __forceinline__ float3 global_load3(const float4* base, unsigned i) {
  typedef float v3 __attribute__((ext_vector_type(3)));
  struct __attribute__((packed, aligned(4))) P { float x, y, z; };
  const FT_GLOBAL_AS P* q = (const FT_GLOBAL_AS P*)((const FT_GLOBAL_AS char*)(unsigned long long)base + (size_t)16u * i);
  return mk(q->x, q->y, q->z);
}

// The union a join's formula is on operands brought to it; stairs ask for their record.
template <class F>
__device__ __forceinline__ float join_union(int type, float x, float y, float rr, F&& stairs) {
  const float m = fminf(x, y);
  if (type == kJoinRound) {
    const float ux = fmaxf(rr - x, 0.0f), uy = fmaxf(rr - y, 0.0f);
    return fmaxf(rr, m) - fsqrt(ux * ux + uy * uy);
  }
  if (type == kJoinChamfer) return fminf(m, (x - rr + y) * kInvSqrt2);
  if (type == kJoinStairs) {
    // beyond the steps the step term is at least m (cell_program)
    const float4 J = stairs();
    return y >= fmaxf(x, 0.0f) + J.x || x >= fmaxf(y, 0.0f) + J.x ? m : op_union_stairs(x, y, J.x, J.y);
  }
  return type == kJoinSoft ? op_union_soft(x, y, rr) : m;
}

// The scene distance (info) from the program of p's cell.  Each lane walks its own cell's
// words: rays of one wave lie in many cells (a 61x37 view puts up to 64 under one wave), and
// running the cells' programs one after the other for the lanes of each took 62 ms for the
// depth pass of 48 views at 256x256 and 6.2 ms for 15 views at 61x37.  The values below the
// top of the stack are in LDS, one column per lane; a primitive followed by its join needs
// none of it.  The cell's record holds its first word; the records of a word are requested
// while the word before it is evaluated, and the word after it at the same time.
template <bool kInfo>
__device__ __forceinline__ Info program_info(const DevScene& S, const ProgramView& V, float3 p) {
  const int4 r = global_load4(V.cells, V.cell(p));
  uint2 w = make_uint2((unsigned)r.x, (unsigned)r.y);
  const unsigned first = (unsigned)r.z;  // of the words after the first
  const int count = r.w;
  float4 A = global_load4(V.ops, 2u * (w.x & kWordNode));
  float3 E = global_load3(V.ops, 2u * (w.x & kWordNode) + 1u);
  uint2 next = global_load2(V.words, first);
  float top = 0.0f;
  int id = 0;
  float* st = V.stack;  // the entry after the last one below the top
  for (int k = 0; k < count; ++k) {
    // the next word's record, then the word after it, requested ahead of this word's work
    const float4 An = global_load4(V.ops, 2u * (next.x & kWordNode));
    const float3 En = global_load3(V.ops, 2u * (next.x & kWordNode) + 1u);
    const uint2 after = global_load2(V.words, first + 2u * (unsigned)k + 2u);
    const bool prim = (w.x & kWordPrim) != 0u, join = (w.x & kWordJoin) != 0u;
    const int one = (int)(w.x >> kWordOneShift) & 3;
    const bool both = join && one == kOneBoth;
    float a = top;
    int ida = id;
    if (prim) {
      if (!both) {
        *st = top;
        if (kInfo) reinterpret_cast<int*>(st)[V.id_plane] = id;
        st += V.step;
      }
      top = cell_prim_distance(V, w.x, A, E, p);
      if (kInfo) id = (int)(w.x & kWordNode);
    } else if (both) {
      st -= V.step;
      a = *st;
      if (kInfo) ida = reinterpret_cast<int*>(st)[V.id_plane];
    }
    if (join) {
      const unsigned fa = w.x << 3, fb = w.x << 2;
      const float x = both ? flip_sign(a, fa) : flip_sign(top, one == kOneLeft ? fa : fb);
      const float y = both ? flip_sign(top, fb) : __builtin_huge_valf();
      const int type = (int)(w.x >> kWordTypeShift) & 7;
      const float v = join_union(type, x, y, __uint_as_float(w.y), [&] { return global_load4(V.ops, 2u * w.y); });
      if (kInfo && both && x <= y) id = ida;
      top = flip_sign(v, fa);
    }
    w = next;
    next = after;
    A = An;
    E = En;
  }
  if (S.flops) {
    float cost = 0.0f;
    for (int k = -1; k < count - 1; ++k) {
      const unsigned v = k < 0 ? (unsigned)r.x : global_load(V.words, first + 2u * (unsigned)k);
      if (v & kWordPrim) cost += S.nodes[S.prog[v & kWordNode]].cost;
      if (v & kWordJoin) cost += 13.0f;
    }
    atomicAdd(S.flops, (unsigned long long)cost);
  }
  Info out;
  out.d = top;
  out.lb = top;
  out.obj = 0u;
  out.mat = 0u;
  out.leaf = -1;
  if (kInfo) {
    const DNode& n = S.nodes[S.prog[id]];
    out.obj = n.obj;
    out.mat = n.mat;
    out.leaf = n.leaf;
  }
  return out;
}
// The cell whose program answers at p (shading words).
__device__ __forceinline__ int program_of(const DevScene& S, float3 p) {
  const int c = cell_of(S, p);
  return c >= 0 ? c : S.cell_dims[0] * S.cell_dims[1] * S.cell_dims[2];
}

// ------------------------------------------------------------------ construction
// The cells are the children, 4 x 4 x 4, of a grid of parent cells.  A build looks at the whole
// scene once per parent and at the parent's result once per child, one wave per parent with
// a lane for each child (262 144 cells of a scene of 2048 primitives from scratch would be
// 64 times the work).
constexpr int kCellChildren = kCellChildrenSide;
struct CellGrid {
  float ox, oy, oz, cell;  // origin and side of the cubic cells (the children)
  int px, py, pz;          // parents along each axis
  float margin;            // bounds the rounding of a distance anywhere in the grid
};

// Cell (x, y, z) of a grid of cells of side `side`: its centre, and what its half diagonal can
// change a distance by.
__device__ __forceinline__ float3 cell_centre(const CellGrid& g, float side, int x, int y, int z) {
  return mk(g.ox + ((float)x + 0.5f) * side, g.oy + ((float)y + 0.5f) * side, g.oz + ((float)z + 0.5f) * side);
}
__device__ __forceinline__ float cell_radius(const CellGrid& g, float side) { return 0.8660255f * side * 1.00001f + g.margin; }
__device__ __forceinline__ float3 parent_centre(const CellGrid& g, int i) {
  return cell_centre(g, g.cell * kCellChildren, i % g.px, (i / g.px) % g.py, i / (g.px * g.py));
}
// The child of parent `i` that a lane stands for, and its index.
__device__ __forceinline__ float3 child_centre(const CellGrid& g, int i, int lane, int& index) {
  const int x = i % g.px * kCellChildren + (lane & 3), y = i / g.px % g.py * kCellChildren + ((lane >> 2) & 3),
            z = i / (g.px * g.py) * kCellChildren + (lane >> 4);
  index = (z * g.py * kCellChildren + y) * g.px * kCellChildren + x;
  return cell_centre(g, g.cell, x, y, z);
}

// The counters of a build, [0] words and the others what the host decides by beside them.  They hold
// more than 32 bits: whether a build's words fit is decided from their whole count.
typedef unsigned long long CellTotal;
constexpr int kCellTotals = 4;
// A leaf list has at most this many entries of a kind, since its two counts share a word; scenes
// with longer ones keep the BVH walk.
constexpr int kLongestList = 0x7fff;

// Room for `n` words from a counter, one atomic per wave.
__device__ __forceinline__ unsigned take_room(CellTotal* cursor, unsigned n) {
  unsigned incl = n;
  const int lane = (int)(threadIdx.x & 63u);
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const unsigned v = __shfl_up(incl, m, 64);
    if (lane >= m) incl += v;
  }
  unsigned base = 0u;
  if (lane == 63) base = (unsigned)atomicAdd(cursor, (CellTotal)incl);
  return __shfl(base, 63, 64) + incl - n;
}

// The leaf lists of one cell with centre c and radius R.  The candidates are `source` (null: all
// sorted leaves, [0, n_prims) primitives, [n_prims, n) known by their bounds only) for the
// distances and `source_box` for the bounds, read in step by the whole wave.  kWrite = false
// counts, the longer of the first two lists in `longest`; kWrite = true writes to the room taken in `r`.
struct LeafSource {
  const unsigned* items;  // null: leaf k is k
  int n_prims, n_others, n_boxes;
  unsigned prims, others, boxes;
};
template <bool kWrite>
__device__ __forceinline__ void leaf_lists_cell(const LeafSource& s, const float4* __restrict__ prims,
                                                const float4* __restrict__ boxes, unsigned none, float3 c, float R, bool mine,
                                                int4& r, int& longest, unsigned* __restrict__ items) {
  const auto P = uniform_ptr(prims);
  const auto X = uniform_ptr(boxes);
  const auto I = uniform_ptr(s.items);
  auto leaf = [&](unsigned first, int k) { return s.items ? I[first + (unsigned)k] : first + (unsigned)k; };
  auto prim = [&](unsigned j) {
    const float4 a = load_uniform(P + 2 * j), b = load_uniform(P + 2 * j + 1);
    return leaf_prim_distance(a, b, c);
  };
  auto box = [&](unsigned j) {
    const float4 a = load_uniform(X + 2 * j), b = load_uniform(X + 2 * j + 1);
    return aabb_lb_lit(c, a.x, a.y, a.z, b.x, b.y, b.z);
  };
  float near = __builtin_huge_valf(), near_box = __builtin_huge_valf();
  for (int k = 0; k < s.n_prims; ++k) near = fminf(near, prim(leaf(s.prims, k)));
  for (int k = 0; k < s.n_boxes; ++k) near_box = fminf(near_box, box(leaf(s.boxes, k)));
  const float keep = fmaxf(near + R, 0.0f) + R, keep_box = near_box + 2.0f * R;
  const int want_p = r.y & 0xffff, want_o = r.y >> 16, want_b = r.w, pad = (want_p + 1) & ~1;
  int np = 0, no = 0, nb = 0;
  for (int k = 0; k < s.n_prims; ++k) {
    const unsigned j = leaf(s.prims, k);
    if (!(prim(j) <= keep) || !mine) continue;
    if (kWrite && np < want_p) items[r.x + np] = j;
    ++np;
  }
  for (int k = 0; k < s.n_others; ++k) {
    const unsigned j = leaf(s.others, k);
    if (!(box(j) <= keep) || !mine) continue;
    if (kWrite && no < want_o) items[r.x + pad + no] = j;
    ++no;
  }
  for (int k = 0; k < s.n_boxes; ++k) {
    const unsigned j = leaf(s.boxes, k);
    if (!(box(j) <= keep_box) || !mine) continue;
    if (kWrite && nb < want_b) items[r.z + nb] = j;
    ++nb;
  }
  if (kWrite && mine) {
    if (pad != want_p) items[r.x + want_p] = none;  // pairs: the primitive at infinity
    // both passes keep the same leaves; an entry left over would name the one at infinity
    for (; np < want_p; ++np) items[r.x + np] = none;
    for (; no < want_o; ++no) items[r.x + pad + no] = none;
    for (; nb < want_b; ++nb) items[r.z + nb] = none;
  }
  if (!kWrite) {
    longest = max(np, no);
    r = make_int4(0, min(np, kLongestList) | (min(no, kLongestList) << 16), 0, nb);
  }
}

// Parents (kChild = false: 64 of them per wave, from all leaves) or their children (a wave per
// parent, from its lists `from` / `from_items`).  Counting adds the words needed to totals[0]
// and the longest list of either kind to totals[1]; writing takes room at totals[0].
template <bool kWrite, bool kChild>
__device__ __forceinline__ void leaf_lists_body(CellGrid g, const float4* __restrict__ prims,
                                                const float4* __restrict__ boxes, int n_prims, int n,
                                                const int4* __restrict__ from, const unsigned* __restrict__ from_items,
                                                int4* __restrict__ lists, unsigned* __restrict__ items,
                                                CellTotal* __restrict__ totals) {
  const int lane = (int)threadIdx.x, n_parents = g.px * g.py * g.pz;
  LeafSource s{nullptr, n_prims, n - n_prims, n, 0u, (unsigned)n_prims, 0u};
  int index;
  float3 c;
  float R;
  bool mine = true;
  if (kChild) {
    const int p = __builtin_amdgcn_readfirstlane((int)blockIdx.x);
    c = child_centre(g, p, lane, index);
    R = cell_radius(g, g.cell);
    const int4 f = load_uniform(uniform_ptr(from) + p);
    s = LeafSource{from_items, f.y & 0xffff, f.y >> 16, f.w, (unsigned)f.x, (unsigned)(f.x + (((f.y & 0xffff) + 1) & ~1)),
                   (unsigned)f.z};
  } else {
    index = (int)blockIdx.x * 64 + lane;
    mine = index < n_parents;
    index = min(index, n_parents - 1);
    c = parent_centre(g, index);
    R = cell_radius(g, g.cell * kCellChildren);
  }
  int4 r = kWrite ? lists[index] : make_int4(0, 0, 0, 0);
  auto words = [](const int4& v) { return (unsigned)((((((v.y & 0xffff) + 1) & ~1) + (v.y >> 16) + v.w) + 1) & ~1); };
  if (kWrite) {
    r.x = (int)take_room(&totals[0], mine ? words(r) : 0u);
    r.z = r.x + (((r.y & 0xffff) + 1) & ~1) + (r.y >> 16);
  }
  int longest = 0;
  leaf_lists_cell<kWrite>(s, prims, boxes, (unsigned)n, c, R, mine, r, longest, items);
  if (mine) lists[index] = r;
  if (!kWrite && mine) {
    atomicAdd(&totals[0], (CellTotal)words(r));
    atomicMax(&totals[1], (CellTotal)longest);
  }
}

// The program of one cell: the wave walks a program (the scene's, or the parent cell's shading
// words) in step, each lane for its own cell.  First the nodes in post order with the interval
// of each node's distance over the cell: a primitive's is its distance at the centre -+ R, a join's follows from its formula,
// which rises with the left operand and rises (differences: falls) with the right one.  Where
// one operand lies beyond the other by the blend radius k it cannot show:
//   unions       b >= max(a, 0) + k for all a, b of the cell: the value is a function of a alone
//                (round: b >= r gives uy = 0; chamfer: (a + b - r) / sqrt(2) >= a; stairs: the
//                step term is at least (a + b - r) / 2 >= a; soft: |a - b| >= r), and the blend
//                weight of the shading walk, smoothstep(0.5 + 0.5 (a - b) / k), is exactly 0
//   differences  the same on (-a, b), mirrored; hard ones with k = 0
//   blended intersections keep both (their shading walk blends toward the farther operand)
// `marks` keeps four bits per node and cell: the operand left over and whether its join then
// passes the value through unchanged.  Then the nodes that remain, from the root down: their
// counts, and on the second call (kWrite) their words.
constexpr int kMarkIdentity = 4;

__device__ __forceinline__ float3 join_interval(int kind, const DOp& o, float alo, float ahi, float blo, float bhi,
                                                float margin) {
  bool keep;
  const bool diff = is_diff(kind);
  const float l = diff ? bhi : blo, h = diff ? blo : bhi;  // the right operand at the low / high end
  float lo, hi;
  if (kind == FT_NODE_INTERSECT) {
    lo = fmaxf(alo, l);
    hi = fmaxf(ahi, h);
  } else if (kind == FT_NODE_SUBTRACT) {
    lo = fmaxf(alo, -l);
    hi = fmaxf(ahi, -h);
  } else {
    lo = smooth_op(kind, alo, l, o.p[0], o.p[1], keep);
    hi = smooth_op(kind, ahi, h, o.p[0], o.p[1], keep);
  }
  int mark = kOneBoth;
  const float k = kind == FT_NODE_INTERSECT || kind == FT_NODE_SUBTRACT ? 0.0f : fmaxf(fabsf(o.p[0]), 1.0e-6f);
  if (kind == FT_NODE_INTERSECT) {
    if (bhi + margin <= alo) mark = kOneLeft | kMarkIdentity;
    else if (ahi + margin <= blo) mark = kOneRight | kMarkIdentity;
  } else if (diff) {
    if (blo >= fmaxf(-alo, 0.0f) + k + margin)
      mark = kOneLeft | (kind != FT_NODE_DIFF_ROUND || ahi + margin <= -k ? kMarkIdentity : 0);
    else if (-ahi >= fmaxf(bhi, 0.0f) + k + margin)
      mark = kOneRight;
  } else if (kind == FT_NODE_UNION_ROUND || kind == FT_NODE_UNION_CHAMFER || kind == FT_NODE_UNION_STAIRS ||
             kind == FT_NODE_UNION_SOFT) {
    if (blo >= fmaxf(ahi, 0.0f) + k + margin)
      mark = kOneLeft | (kind != FT_NODE_UNION_ROUND || alo >= k + margin ? kMarkIdentity : 0);
    else if (alo >= fmaxf(bhi, 0.0f) + k + margin)
      mark = kOneRight | (kind != FT_NODE_UNION_ROUND || blo >= k + margin ? kMarkIdentity : 0);
  }
  return mk(lo - margin, hi + margin, __int_as_float(mark));
}

// The same for a join that has one operand left already: x = its interval.
__device__ __forceinline__ float3 join_one_interval(int kind, const DOp& o, bool right, float xlo, float xhi, float margin) {
  const bool mirror = right && is_diff(kind);
  const float lo = join_one(kind, mirror ? xhi : xlo, right, o.p[0]), hi = join_one(kind, mirror ? xlo : xhi, right, o.p[0]);
  const float k = fmaxf(fabsf(o.p[0]), 1.0e-6f);
  const bool round = kind == FT_NODE_UNION_ROUND || kind == FT_NODE_DIFF_ROUND;
  const bool same = !mirror && (!round || (kind == FT_NODE_UNION_ROUND ? xlo >= k + margin : xhi + margin <= -k));
  return mk(lo - margin, hi + margin, __int_as_float((right ? kOneRight : kOneLeft) | (same ? kMarkIdentity : 0)));
}

// `words`: null for the scene program (n words), else its shading words.  `marks`: this lane's
// first mark word, `stride` words apart.  Counting (kWrite = false) sets r.w and sh.y; writing
// takes the room given in r.z and sh.x (kShades only: shading words alone).  `surface`, of counting:
// the cell may hold some of the surface.
template <bool kWrite, bool kShadesOnly>
__device__ __forceinline__ void cell_program(const DOp* __restrict__ ops_, const unsigned* __restrict__ words_, int n,
                                             float3 c, float R, float margin, bool mine, unsigned* __restrict__ marks,
                                             int stride, int4& r, int2& sh, unsigned* __restrict__ out, bool& surface) {
  const auto ops = uniform_ptr(ops_);
  const auto words = uniform_ptr(words_);
  auto word = [&](int k) { return words_ ? words[k] : (unsigned)k; };
  if (!kWrite) {
    float lo[kRegStack], hi[kRegStack];
    for (int j = 0; j < kRegStack; ++j) lo[j] = hi[j] = 0.0f;
    int sp = 0;
    unsigned bits = 0u;
    for (int k = 0; k < n; ++k) {
      const unsigned w = word(k);
      const DOp o = load_uniform(ops + (w & kWordNode));
      const int kind = o.code & kOpKindMask, one = (int)(w >> kWordOneShift) & 3;
      sp = __builtin_amdgcn_readfirstlane(sp);
      const int i1 = (sp - 1) & (kRegStack - 1), i0 = (sp - 2) & (kRegStack - 1);
      const float blo = lo[i1], bhi = hi[i1], alo = lo[i0], ahi = hi[i0];
      int wt;
      float3 v;
      if (is_prim(kind)) {
        const float d = op_prim_distance(o, kind, c);
        wt = sp++ & (kRegStack - 1);
        v = mk(d - R, d + R, 0.0f);
      } else if (one != kOneBoth) {
        wt = i1;
        v = join_one_interval(kind, o, one == kOneRight, blo, bhi, margin);
      } else {
        wt = i0;
        --sp;
        v = join_interval(kind, o, alo, ahi, blo, bhi, margin);
      }
      lo[wt] = v.x;
      hi[wt] = v.y;
      bits |= (__float_as_uint(v.z) & 15u) << (4 * (k & 7));
      if ((k & 7) == 7 || k == n - 1) {
        if (mine) marks[(size_t)(k >> 3) * stride] = bits;
        bits = 0u;
      }
    }
    surface = lo[0] <= 0.0f && hi[0] >= 0.0f;  // the root's interval
    __threadfence_block();
  }
  // from the root down (reverse post order): a bit per pending subtree, set where it remains;
  // a join waits for the node before it, whose word it joins if that is a primitive
  const int want = r.w, want_shades = sh.y;
  int nv = 0, ns = 0, sp = 1;
  unsigned live = 1u, bits = 0u, waiting = 0u, value = 0u;
  auto put = [&](unsigned x, unsigned y) {
    const int at = want - 1 - nv;
    if (kWrite && !kShadesOnly && at > 0) {
      out[r.z + 2 * (at - 1)] = x;
      out[r.z + 2 * (at - 1) + 1] = y;
    } else if (kWrite && !kShadesOnly && at == 0) {
      r.x = (int)x;
      r.y = (int)y;
    }
    ++nv;
  };
  for (int k = n - 1; k >= 0; --k) {
    if ((k & 7) == 7 || k == n - 1) bits = mine ? marks[(size_t)(k >> 3) * stride] : 0u;
    const unsigned w = word(k);
    const int j = (int)(w & kWordNode), one = (int)(w >> kWordOneShift) & 3;
    const DOp o = load_uniform(ops + j);
    const int kind = o.code & kOpKindMask;
    --sp;
    const bool here = (live >> sp) & 1u;
    live &= ~(1u << sp);
    int mark = 0;
    if (!is_prim(kind)) {
      mark = (int)(bits >> (4 * (k & 7))) & 15;
      if (one != kOneBoth) {
        live |= (here ? 1u : 0u) << sp;
        ++sp;
      } else {
        live |= (here && (mark & 3) != kOneRight ? 1u : 0u) << sp;
        live |= (here && (mark & 3) != kOneLeft ? 1u : 0u) << (sp + 1);
        sp += 2;
      }
    }
    if (!here || !mine) continue;
    if (is_prim(kind)) {
      put(waiting | prim_word(o, j), value);
      waiting = 0u;
    } else if (!(mark & kMarkIdentity)) {
      if (waiting) put(waiting, value);
      waiting = join_word(kind, mark & 3);
      value = join_value(o, j);
    }
    if (kWrite && ns < want_shades)
      out[sh.x + want_shades - 1 - ns] = is_prim(kind) ? prim_word(o, j) : join_word(kind, mark & 3) | (unsigned)j;
    ++ns;
  }
  if (!kWrite) {
    r = make_int4(0, 0, 0, nv);
    sh = make_int2(0, ns);
  }
}

// Parents (64 per wave, from the scene program): shading words alone, which are the program
// their children start from, each parent's room a multiple of 8 words (its children's marks
// hold 8 words in one and are placed by it).  totals[0]: words.
template <bool kWrite>
__device__ __forceinline__ void cell_parents_body(CellGrid g, const DOp* __restrict__ ops, int n_prog,
                                                  unsigned* __restrict__ marks, int2* __restrict__ parents,
                                                  unsigned* __restrict__ words, CellTotal* __restrict__ totals) {
  const int n_parents = g.px * g.py * g.pz;
  const int i = (int)blockIdx.x * 64 + (int)threadIdx.x;
  const bool mine = i < n_parents;
  const int m = min(i, n_parents - 1);
  int4 r = make_int4(0, 0, 0, 0);
  int2 sh = kWrite ? parents[m] : make_int2(0, 0);
  bool surface = false;
  if (kWrite) sh.x = (int)take_room(&totals[0], mine ? (unsigned)(sh.y + 7) & ~7u : 0u);
  cell_program<kWrite, true>(ops, nullptr, n_prog, parent_centre(g, m), cell_radius(g, g.cell * kCellChildren),
                             0.25f * g.margin, mine, marks + m, n_parents, r, sh, words, surface);
  if (mine) parents[m] = sh;
  if (!kWrite && mine) atomicAdd(&totals[0], (CellTotal)((unsigned)(sh.y + 7) & ~7u));
}
// Children (a wave per parent).  totals[0]: words, [1]: distance words alone, [2]: those of the cells on
// the surface, [3]: these cells.
template <bool kWrite>
__device__ __forceinline__ void cell_children_body(CellGrid g, const DOp* __restrict__ ops, const int2* __restrict__ parents,
                                                   const unsigned* __restrict__ parent_words, unsigned* __restrict__ marks,
                                                   int4* __restrict__ progs, int2* __restrict__ shades,
                                                   unsigned* __restrict__ words, CellTotal* __restrict__ totals) {
  const int p = __builtin_amdgcn_readfirstlane((int)blockIdx.x);
  int index;
  const float3 c = child_centre(g, p, (int)threadIdx.x, index);
  const int2 from = load_uniform(uniform_ptr(parents) + p);
  int4 r = kWrite ? progs[index] : make_int4(0, 0, 0, 0);  // first word, where the others start, count
  int2 sh = kWrite ? shades[index] : make_int2(0, 0);
  if (kWrite) {
    r.z = (int)take_room(&totals[0], (unsigned)(2 * (r.w - 1) + ((sh.y + 1) & ~1)));
    sh.x = r.z + 2 * (r.w - 1);
  }
  bool surface = false;
  // the parent's marks: 64 lanes of ceil(n / 8) words, placed by its first word
  unsigned* const m = marks + (size_t)(from.x / 8) * 64 + threadIdx.x;
  cell_program<kWrite, false>(ops, parent_words + from.x, from.y, c, cell_radius(g, g.cell), 0.25f * g.margin, true, m, 64,
                              r, sh, words, surface);
  progs[index] = r;
  shades[index] = sh;
  if (!kWrite) {
    atomicAdd(&totals[0], (CellTotal)(2 * (r.w - 1) + ((sh.y + 1) & ~1)));
    atomicAdd(&totals[1], (CellTotal)r.w);
    if (surface) {
      atomicAdd(&totals[2], (CellTotal)r.w);
      atomicAdd(&totals[3], (CellTotal)1);
    }
  }
}

}  // namespace ftd
