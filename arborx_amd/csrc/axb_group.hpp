// axb_group.hpp -- the wavefront-wide search of a point tree ("group walk").
//
// 64 predicates that lie close together (consecutive in Hilbert or tree
// order) look at nearly the same leaves.  Instead of 64 walks, each with its
// own gathered record, decode and test per step, the wavefront searches
// once for all of them:
//   1. leaf blocks: 64 consecutive leaves each, with their boxes, and boxes
//      over 64 boxes each above them (a 64-wide implicit tree over the
//      sorted leaves, built with the tree).  One step tests the 64 boxes
//      below a node, one per lane, against the box around the wavefront's
//      predicates: the blocks within reach, in leaf order;
//   2. the leaves of those blocks, one block per step and one leaf per lane
//      (a coalesced load of 1 KiB), against the same box: the candidates,
//      gathered in LDS in leaf order;
//   3. every candidate against every predicate: a matrix product.  With
//      coordinates relative to the middle of the predicates,
//      |p - q|^2 - T = |p|^2 + (-2 q) . p + (|q|^2 - T) is one 8-term dot
//      product, so two 32x32x8 half-precision MFMAs test 32 candidates
//      against 64 predicates.  T is enlarged so that no rounding can lose a
//      hit (group_columns below); the sign bits become one bit mask of 32
//      candidates per lane;
//   4. each lane tests the candidates in its mask with the exact float
//      distance, in leaf order: results and their order are the rope walk's.
// A wavefront whose predicates are not close together (or not finite) finds
// too many blocks, or more candidates than pay (group_pays), and is sent back
// to walk the tree lane by lane.
#pragma once

#include "axb_internal.hpp"

namespace axb
{

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int GROUP_BLOCKS = 256; // leaf blocks a group may look at
constexpr int GROUP_NODES = 64;   // boxes of an upper level a group may open
constexpr int GROUP_WORDS = 5;    // candidates tested together: 32 per word
constexpr int GROUP_CAND = GROUP_WORDS * 32;
constexpr float GROUP_EXTENT = 30.f; // the group's half extent, in half-precision units
// Both coordinates of a pair are rounded to half precision with an error of
// at most 2^-7 per axis below 32, so a distance is off by at most
// 2 sqrt(3) 2^-7 = 0.0271; the float subtraction and scaling before it add
// less than 1e-4.
constexpr float GROUP_ROUNDING = 0.0275f;
// |p|^2 and |q|^2 - T (below 3000 each) enter as two halves (22 bits, less
// than 1e-3 off each); the product's single-precision sums of at most 8
// terms below 6000 are off by less than 8 * 6000 * 2^-23 = 0.006.
constexpr float GROUP_SUMS = 0.05f;

// LDS of one wavefront.
struct GroupLds
{
  uint4 leaf[GROUP_CAND + 96];      // candidates {x y z ~index} (up to 31 + 64 beyond a window)
  uint32_t mask[GROUP_WORDS][64];   // each lane's candidates, 32 per word
  uint64_t blocks[GROUP_NODES];     // leaf blocks within reach below each node of level 1
  uint32_t node[2][GROUP_NODES];
};

// Orders the wavefront's LDS accesses before and after this point (LDS
// operations of one wavefront complete in issue order).
AXB_D void wave_lds_order()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

AXB_D float wave_min(float v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
AXB_D float wave_max(float v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
AXB_D float wave_sum(float v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    v += __shfl_xor(v, o, 64);
  return v;
}
AXB_D float wave_uniform(float v)
{
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
AXB_D uint32_t lanes_below(uint64_t m)
{
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// What the lanes of a group search for: the box around their centres, the
// largest radius and its squared threshold, and the frame of the half
// coordinates.  (Uniform over the wavefront.)
struct GroupReach
{
  float lo[3], hi[3], mid[3];
  float r, thr, scale;
  float tiny; // far below any extent that matters
};

// A candidate's terms of the matrix product: {x y z |p|^2 high} in lanes
// 0-31, {|p|^2 low 1 1 0} in lanes 32-63.
AXB_D half4_t group_row(const GroupReach &g, uint4 s)
{
  const _Float16 hx = (_Float16)((bits_f(s.x) - g.mid[0]) * g.scale);
  const _Float16 hy = (_Float16)((bits_f(s.y) - g.mid[1]) * g.scale);
  const _Float16 hz = (_Float16)((bits_f(s.z) - g.mid[2]) * g.scale);
  const float fx = (float)hx, fy = (float)hy, fz = (float)hz;
  const float p2 = fx * fx + fy * fy + fz * fz;
  const _Float16 ph = (_Float16)p2;
  const _Float16 pl = (_Float16)(p2 - (float)ph);
  const bool low = (threadIdx.x & 63) < 32;
  return (half4_t){low ? hx : pl, low ? hy : (_Float16)1.f, low ? hz : (_Float16)1.f,
                   low ? ph : (_Float16)0.f};
}

// Squared distance of a point to the box around the group's centres, in the
// operation order of dist2_pp.  Subtraction, product and sum round
// monotonically, so a leaf within a lane's threshold passes.
AXB_D float group_point_d2(const GroupReach &g, float x, float y, float z)
{
  return dist2_pp(clamp_box(x, g.lo[0], g.hi[0]), clamp_box(y, g.lo[1], g.hi[1]),
                  clamp_box(z, g.lo[2], g.hi[2]), x, y, z);
}
// The same for a box (gaps per axis).
AXB_D float group_box_d2(const GroupReach &g, float4 a, float4 b)
{
  const float gx = fmaxf(fmaxf(a.x - g.hi[0], g.lo[0] - a.w), 0.f);
  const float gy = fmaxf(fmaxf(a.y - g.hi[1], g.lo[1] - b.x), 0.f);
  const float gz = fmaxf(fmaxf(a.z - g.hi[2], g.lo[2] - b.y), 0.f);
  float s = gx * gx;
  s = s + gy * gy;
  s = s + gz * gz;
  return s;
}

// The group's reach.  active: the lane has a finite centre and a radius
// r >= 0 (thr = sqrt_threshold(r)); other lanes have no hits (thr is finite
// or NaN: group_walk leaves infinite ones to the lanes' own walks).  False when
// the group cannot be searched this way (an infinite radius, or extents at
// which the halves' error bounds do not hold): every lane then walks alone.
AXB_D bool group_reach(float x, float y, float z, float r, float thr, bool active,
                       GroupReach &g)
{
  float h = 0.f;
  const float c[3] = {x, y, z};
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    g.lo[d] = wave_uniform(wave_min(active ? c[d] : FLT_MAX));
    g.hi[d] = wave_uniform(wave_max(active ? c[d] : -FLT_MAX));
    g.mid[d] = 0.5f * g.lo[d] + 0.5f * g.hi[d];
    h = fmaxf(h, fmaxf(g.hi[d] - g.mid[d], g.mid[d] - g.lo[d]));
  }
  const float rm = wave_uniform(wave_max(active ? r : 0.f));
  g.thr = wave_uniform(wave_max(active ? thr : 0.f));
  h = h + rm;
  g.r = rm;
  g.tiny = 1e-6f * h;
  g.scale = GROUP_EXTENT / h;
  // below 1e-12 squared distances may be denormal, above 1e15 overflow
  return h > 1e-12f && h < 1e15f;
}

// Leaf blocks within reach: L.blocks[j] has bit b set for block 64 node[j] +
// b, nodes in leaf order (node = L.node[the returned buffer]).  Returns the
// number of nodes, or -1 when more blocks or nodes are within reach than a
// group may look at.  see(m, a, b): the mask of the blocks within reach below
// a node, lane l with the box of block l.
template <class See>
AXB_D int group_blocks(const TreeView &tv, const GroupReach &g, GroupLds &L, int &buffer,
                       uint32_t &tested, See &&see)
{
  const int lane = threadIdx.x & 63;
  int cnt = 1, cur = 0;
  if (lane == 0)
    L.node[0][0] = 0u;
  for (int lev = tv.blk_levels - 1; lev >= 0; --lev)
  {
    wave_lds_order();
    const uint32_t total = tv.blk_count[lev];
    const float4 *boxes = tv.blk + 2 * (size_t)tv.blk_at[lev];
    int got = 0;
    for (int j = 0; j < cnt; ++j)
    {
      const uint32_t id = (uint32_t)__builtin_amdgcn_readfirstlane((int)L.node[cur][j]) * 64u +
                          (uint32_t)lane;
      bool in = false;
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
      if (id < total)
      {
        a = boxes[2 * (size_t)id], b = boxes[2 * (size_t)id + 1];
        in = group_box_d2(g, a, b) <= g.thr;
      }
      ++tested;
      const uint64_t m = __ballot(in);
      const int more = __popcll(m);
      if (got + more > (lev == 0 ? GROUP_BLOCKS : GROUP_NODES))
        return -1;
      if (lev == 0)
      {
        if (lane == 0)
          L.blocks[j] = m;
        see(m, a, b);
      }
      else if (in)
        L.node[cur ^ 1][got + (int)lanes_below(m)] = id;
      got += more;
    }
    if (lev > 0)
      cnt = got, cur ^= 1;
  }
  wave_lds_order();
  buffer = cur;
  return cnt;
}

// The part of a block's box, and so about of its leaves, within the box of
// the group's reach.
AXB_D float group_part(const GroupReach &g, float4 a, float4 b)
{
  const float bl[3] = {a.x, a.y, a.z}, bh[3] = {a.w, b.x, b.y};
  float part = 1.f;
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    const float cut = fminf(bh[d], g.hi[d] + g.r) - fmaxf(bl[d], g.lo[d] - g.r);
    part *= fmaxf(cut, g.tiny) * __builtin_amdgcn_rcpf(fmaxf(bh[d] - bl[d], g.tiny));
  }
  return part;
}

// Whether a group's search is less work than the walks of its 64 lanes, by the
// number of candidates.  A candidate costs 2.2 vector instructions per
// wavefront for its leaf and mask bit, and up to 15 in the exact loop, which
// runs as often as the busiest lane has candidates in a window: a lane's hits
// lie together, so about hits / GROUP_CAND of the time.
AXB_D float group_cost(float leaves, float hits)
{
  return leaves * (2.2f + 0.094f * fminf(hits, (float)GROUP_CAND));
}
// Walks that take about base + per_hit * hits instructions (base FLT_MAX: no
// limit).  known: hits of a lane as far as the caller knows them (else 0).
struct WalkCost
{
  float base, per_hit, known;
  float share; // of the reach's box in a lane's sphere, on average
  AXB_D void meet(const GroupReach &g, float r, bool active)
  {
    if (base == FLT_MAX)
      return;
    float box = (float)__popcll(__ballot(active)); // volumes in the group's own unit
#pragma unroll
    for (int d = 0; d < 3; ++d)
      box *= fmaxf(g.hi[d] - g.lo[d] + 2.f * g.r, g.tiny) * g.scale;
    const float u = active ? r * g.scale : 0.f;
    share = wave_uniform(wave_sum(4.18879f * u * u * u)) * __builtin_amdgcn_rcpf(box);
  }
  AXB_D bool pays(float leaves) const
  {
    const float hits = fmaxf(known, leaves * share);
    return group_cost(leaves, hits) <= base + per_hit * hits;
  }
};
// At most so many candidates.
struct LeafLimit
{
  float most;
  AXB_D void meet(const GroupReach &, float, bool) {}
  AXB_D bool pays(float leaves) const { return leaves <= most; }
};
struct NoLimit
{
  AXB_D void meet(const GroupReach &, float, bool) {}
  AXB_D bool pays(float) const { return true; }
};

// Whether searching the blocks that group_blocks found pays.
template <class Limit>
AXB_D bool group_pays(const TreeView &tv, const GroupReach &g, const GroupLds &L, int nodes,
                      int buffer, const Limit &limit)
{
  // most groups pay even if every leaf of their blocks is a candidate
  int blocks = 0;
  for (int j = 0; j < nodes; ++j)
    blocks += __popcll(L.blocks[j]);
  if (limit.pays(64.f * (float)__builtin_amdgcn_readfirstlane(blocks)))
    return true;
  const int lane = threadIdx.x & 63;
  const float4 *boxes = tv.blk + 2 * (size_t)tv.blk_at[0];
  float part = 0.f;
  for (int j = 0; j < nodes; ++j)
    if ((L.blocks[j] >> lane) & 1u)
    {
      const size_t id = (size_t)L.node[buffer][j] * 64u + (size_t)lane;
      part += group_part(g, boxes[2 * id], boxes[2 * id + 1]);
    }
  return limit.pays(64.f * wave_uniform(wave_sum(part)));
}

// The lane's predicate as the two matrix operands (columns 0-31 and 32-63
// of the group's 64 predicates; lanes 0-31 hold terms 0-3, the others 4-7).
AXB_D void group_columns(const GroupReach &g, float x, float y, float z, float r, bool active,
                         half4_t (&col)[2])
{
  const _Float16 hx = (_Float16)(active ? (x - g.mid[0]) * g.scale : 0.f);
  const _Float16 hy = (_Float16)(active ? (y - g.mid[1]) * g.scale : 0.f);
  const _Float16 hz = (_Float16)(active ? (z - g.mid[2]) * g.scale : 0.f);
  const float fx = (float)hx, fy = (float)hy, fz = (float)hz;
  const float reach = r * g.scale * 1.000001f + GROUP_ROUNDING;
  const float c = active ? fx * fx + fy * fy + fz * fz - (reach * reach + GROUP_SUMS) : 60000.f;
  const _Float16 ch = (_Float16)c;
  const _Float16 cl = (_Float16)(c - (float)ch);
  const half4_t a = {(_Float16)(-2.f * fx), (_Float16)(-2.f * fy), (_Float16)(-2.f * fz),
                     (_Float16)1.f};
  const half4_t b = {(_Float16)1.f, ch, cl, (_Float16)0.f};
  union
  {
    half4_t h;
    int w[2];
  } ua, ub, o;
  ua.h = a, ub.h = b;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < 2; ++j)
  {
    const int from = 32 * j + (lane & 31);
#pragma unroll
    for (int w = 0; w < 2; ++w)
    {
      const int va = __shfl(ua.w[w], from, 64), vb = __shfl(ub.w[w], from, 64);
      o.w[w] = lane < 32 ? va : vb;
    }
    col[j] = o.h;
  }
}

// Bit c of the lane's mask: candidate at + c may be within the lane's reach.
AXB_D uint32_t group_mask(const GroupLds &L, const GroupReach &g, int at,
                          const half4_t (&col)[2])
{
  // row m of the product holds the candidate whose sign lands at bit c of
  // the lane's mask: result register i of half h is row 8 (i / 4) + 4 h +
  // i % 4, and bit c = 16 h + i
  const int m = threadIdx.x & 31;
  const int c = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
  const half4_t row = group_row(g, L.leaf[at + c]);
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                         0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const f32x16_t d0 = __builtin_amdgcn_mfma_f32_32x32x8f16(row, col[0], zero, 0, 0, 0);
  const f32x16_t d1 = __builtin_amdgcn_mfma_f32_32x32x8f16(row, col[1], zero, 0, 0, 0);
  uint32_t bits[2] = {0u, 0u};
#pragma unroll
  for (int i = 15; i >= 0; --i)
    bits[0] = __builtin_amdgcn_alignbit(bits[0], __float_as_uint(d0[i]), 31);
#pragma unroll
  for (int i = 15; i >= 0; --i)
    bits[1] = __builtin_amdgcn_alignbit(bits[1], __float_as_uint(d1[i]), 31);
  // lane l < 32 holds half 0 of column l (and of column 32 + l), lane l + 32
  // half 1 of the same columns; afterwards every lane holds its own column
  const auto s = __builtin_amdgcn_permlane32_swap(bits[0], bits[1], false, false);
  return (uint32_t)s[0] | ((uint32_t)s[1] << 16);
}

// Every lane's exact tests of the candidates in its masks, in leaf order.
// words: bit w set when the lane's word w is not empty.  A window of many
// candidates per call keeps the lanes together: the loop runs as often as
// the busiest lane has candidates in the window.
template <bool SKIP, class Sink>
AXB_D void group_exact(const GroupLds &L, uint32_t words, float x, float y, float z, float thr,
                       int32_t skip, Sink &sink)
{
  const int lane = threadIdx.x & 63;
  if constexpr (Sink::COUNTS_ON)
    if (sink.full())
    {
      // too many already: a lane that only counts takes its candidates as
      // they are
      for (; words; words &= words - 1u)
        sink.cnt += __popc(L.mask[__builtin_ctz(words)][lane]);
    }
  uint32_t mask = 0;
  const uint4 *word = L.leaf;
  while (mask | words)
  {
    if (mask == 0)
    {
      const int w = __builtin_ctz(words);
      words &= words - 1u;
      mask = L.mask[w][lane];
      word = L.leaf + 32 * w;
    }
    const uint4 s = word[__builtin_ctz(mask)];
    mask &= mask - 1u;
    const float d2 = dist2_pp(x, y, z, bits_f(s.x), bits_f(s.y), bits_f(s.z));
    if (d2 <= thr)
      if (!SKIP || (int32_t)s.w != ~skip)
        sink.hit(~(int32_t)s.w, d2);
  }
}

// Calls fn(block, leaf) for every leaf of the blocks that group_blocks found
// (nodes of them, in L.blocks / L.node[buffer]), a block at a time and in
// leaf order, lane l with the block's leaf l (a copy of the last leaf past
// the end); the next block's leaves are in flight meanwhile.
template <class Fn>
AXB_D void group_leaves(const TreeView &tv, const GroupLds &L, int nodes, int buffer, Fn &&fn)
{
  const uint32_t n = (uint32_t)tv.n, lane = threadIdx.x & 63u;
  // node `at`, its remaining blocks in `rest`
  int at = -1;
  uint32_t base = 0;
  uint64_t rest = 0;
  auto next_block = [&](uint32_t &b) {
    while (rest == 0)
    {
      if (++at >= nodes)
        return false;
      const uint64_t m = L.blocks[at];
      rest = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)m) |
             ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(m >> 32)) << 32);
      base = (uint32_t)__builtin_amdgcn_readfirstlane((int)L.node[buffer][at]) * 64u;
    }
    b = base + (uint32_t)__builtin_ctzll(rest);
    rest &= rest - 1ull;
    return true;
  };
  auto load = [&](uint32_t b) {
    const uint32_t i = b * 64u + lane;
    return tv.leaves[i < n ? i : n - 1];
  };
  uint32_t blk = 0, blk_next = 0;
  uint4 s = make_uint4(0u, 0u, 0u, 0u);
  bool more = next_block(blk);
  if (more)
    s = load(blk);
  while (more)
  {
    const bool more_next = next_block(blk_next);
    uint4 s_next = s;
    if (more_next)
      s_next = load(blk_next);
    fn(blk, s);
    s = s_next;
    blk = blk_next;
    more = more_next;
  }
}

// All hits of the wavefront's predicates, each lane's in leaf order.  Every
// lane of the wavefront calls it (inactive ones too).  False: not searched
// (limit: WalkCost, LeafLimit or NoLimit), the lanes have to walk the tree
// themselves.  SKIP: the value `skip` is not
// reported.
template <bool SKIP, class Limit, class Sink>
AXB_D bool group_walk(const TreeView &tv, GroupLds &L, float x, float y, float z, float r,
                      float thr, bool active, int32_t skip, Limit limit, Sink &sink,
                      uint32_t &v_int, uint32_t &v_leaf)
{
  // an infinite radius reaches everything, from an infinite (inactive) centre
  // too
  if (__ballot(thr == INFINITY || (active && !(thr < INFINITY))))
    return false;
  if (__ballot(active) == 0)
    return true;
  GroupReach g;
  if (!group_reach(x, y, z, r, thr, active, g))
    return false;
  int buffer = 0;
  const int nodes =
      group_blocks(tv, g, L, buffer, v_int, [](uint64_t, const float4 &, const float4 &) {});
  if (nodes < 0)
    return false;
  limit.meet(g, r, active);
  if (!group_pays(tv, g, L, nodes, buffer, limit))
    return false;
  half4_t col[2];
  group_columns(g, x, y, z, r, active, col);
  const int lane = threadIdx.x & 63;
  const uint32_t n = (uint32_t)tv.n;
  int cnt = 0, done = 0; // candidates in LDS, and those whose masks are made
  uint32_t words = 0;
  group_leaves(tv, L, nodes, buffer, [&](uint32_t blk, uint4 s) {
    ++v_leaf;
    const bool in = blk * 64u + (uint32_t)lane < n &&
                    group_point_d2(g, bits_f(s.x), bits_f(s.y), bits_f(s.z)) <= g.thr;
    const uint64_t m = __ballot(in);
    if (in)
      L.leaf[cnt + (int)lanes_below(m)] = s; // below GROUP_CAND + 31 + 64
    cnt += __popcll(m);
    wave_lds_order();
    while (cnt - done >= 32)
    {
      const uint32_t w = group_mask(L, g, done, col);
      L.mask[done >> 5][lane] = w;
      words |= (w != 0 ? 1u : 0u) << (done >> 5);
      done += 32;
      if (done == GROUP_CAND)
      {
        group_exact<SKIP>(L, words, x, y, z, thr, skip, sink);
        words = 0;
        done = 0;
        cnt -= GROUP_CAND; // below 96
        uint4 a = s, b = s;
        if (lane < cnt)
          a = L.leaf[GROUP_CAND + lane];
        if (lane + 64 < cnt)
          b = L.leaf[GROUP_CAND + 64 + lane];
        wave_lds_order();
        if (lane < cnt)
          L.leaf[lane] = a;
        if (lane + 64 < cnt)
          L.leaf[64 + lane] = b;
        wave_lds_order();
      }
    }
  });
  if (cnt > done)
  {
    // the last, partial word: its bits past the candidates are dropped
    const uint32_t w = group_mask(L, g, done, col) & ((1u << (cnt - done)) - 1u);
    L.mask[done >> 5][lane] = w;
    words |= (w != 0 ? 1u : 0u) << (done >> 5);
  }
  group_exact<SKIP>(L, words, x, y, z, thr, skip, sink);
  return true;
}

// ------------------------------------------------------------ nearest
AXB_D float approx_cbrt(float v) // exp2(log2 / 3): for guesses only
{
  return __builtin_amdgcn_exp2f((1.f / 3.f) * __builtin_amdgcn_logf(v));
}

// The radius within which a lane should find about `want` leaves, from the
// leaves in and just around the group's box: their number over the volume
// they were counted in gives the density, and a ball that reaches beyond the
// scene box is enlarged for the part outside.  A guess: the caller counts
// what it finds.  spacing: about the distance between leaves.  False when
// the box holds too many blocks or there is nothing to go by.
AXB_D bool group_guess_radius(const TreeView &tv, GroupLds &L, float x, float y, float z,
                              bool active, float want, float spacing, float &r, uint32_t &v_int,
                              uint32_t &v_leaf)
{
  GroupReach g;
  if (!group_reach(x, y, z, 0.f, 0.f, active, g))
    return false; // all centres in one place
  const float ex = g.hi[0] - g.lo[0], ey = g.hi[1] - g.lo[1], ez = g.hi[2] - g.lo[2];
  float grow = 0.1f * fmaxf(fmaxf(ex, ey), ez);
  const uint32_t n = (uint32_t)tv.n, lane = threadIdx.x & 63u;
  int found = 0;
  for (int t = 0;; ++t)
  {
    g.thr = grow * grow;
    int buffer = 0;
    const int nodes =
      group_blocks(tv, g, L, buffer, v_int, [](uint64_t, const float4 &, const float4 &) {});
    if (nodes < 0)
      return false;
    found = 0;
    group_leaves(tv, L, nodes, buffer, [&](uint32_t blk, uint4 s) {
      ++v_leaf;
      found += __popcll(__ballot(
          blk * 64u + lane < n &&
          group_point_d2(g, bits_f(s.x), bits_f(s.y), bits_f(s.z)) <= g.thr));
    });
    wave_lds_order();
    if (found >= 24 || t == 5)
      break;
    grow = fmaxf(2.f * grow, 0.5f * spacing);
  }
  const float vol = ex * ey * ez + 2.f * grow * (ex * ey + ey * ez + ez * ex) +
                    3.14159265f * grow * grow * (ex + ey + ez) + 4.18879f * grow * grow * grow;
  const float r0 = approx_cbrt(0.238732f * want * vol / (float)(found > 0 ? found : 1));
  float in = 1.f;
  const float c[3] = {x, y, z};
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    const float gap = fmaxf(fminf(c[d] - tv.scene.lo[d], tv.scene.hi[d] - c[d]), 0.f);
    const float u = fminf(gap / r0, 1.f); // part of the ball's axis inside
    in *= 0.5f + 0.5f * u * (1.5f - 0.5f * u * u);
  }
  r = r0 / approx_cbrt(in);
  return wave_uniform(r0) > 0.f && r0 < 1e15f;
}

// The same from the lane's own density: every leaf block spreads its 64
// leaves over its box, and what falls into a cube around the lane's centre
// counts (the boxes of Morton blocks overlap, but each spreads its own leaves
// only).  Follows a density that differs between the lanes of a group, and
// reads no leaves, but is less exact where it does not.  per_query: leaves
// per predicate, which sets the cube's size.
AXB_D float lane_value(float v, int lane)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
AXB_D bool group_guess_own_radius(const TreeView &tv, GroupLds &L, float x, float y, float z,
                                  bool active, float want, float per_query, float &r,
                                  uint32_t &v_int)
{
  GroupReach g;
  if (!group_reach(x, y, z, 0.f, 0.f, active, g))
    return false;
  const float e[3] = {g.hi[0] - g.lo[0], g.hi[1] - g.lo[1], g.hi[2] - g.lo[2]};
  const float least = 0.2f * fmaxf(fmaxf(e[0], e[1]), e[2]);
  const float vol = fmaxf(e[0], least) * fmaxf(e[1], least) * fmaxf(e[2], least);
  // half the side of a cube of about want / 2 leaves, if the group's box
  // holds per_query for each of its predicates
  const float h = 0.5f * approx_cbrt(0.5f * want * vol /
                                     ((float)__popcll(__ballot(active)) * per_query));
  g.thr = h * h;
  const float lo[3] = {x - h, y - h, z - h}, hi[3] = {x + h, y + h, z + h};
  float mass = 0.f;
  int buffer = 0;
  const int nodes = group_blocks(
      tv, g, L, buffer, v_int, [&](uint64_t m, const float4 &a, const float4 &b) {
        // per axis: 1 / extent, 0 for a flat box
        const float ix = a.w > a.x ? __builtin_amdgcn_rcpf(a.w - a.x) : 0.f;
        const float iy = b.x > a.y ? __builtin_amdgcn_rcpf(b.x - a.y) : 0.f;
        const float iz = b.y > a.z ? __builtin_amdgcn_rcpf(b.y - a.z) : 0.f;
        for (uint64_t rest = m; rest; rest &= rest - 1ull)
        {
          const int l = __builtin_ctzll(rest);
          const float bl[3] = {lane_value(a.x, l), lane_value(a.y, l), lane_value(a.z, l)};
          const float bh[3] = {lane_value(a.w, l), lane_value(b.x, l), lane_value(b.y, l)};
          const float bi[3] = {lane_value(ix, l), lane_value(iy, l), lane_value(iz, l)};
          float part = 1.f;
#pragma unroll
          for (int d = 0; d < 3; ++d)
          {
            const float cut = fminf(hi[d], bh[d]) - fmaxf(lo[d], bl[d]);
            part *= bi[d] > 0.f ? fmaxf(cut, 0.f) * bi[d] : (cut >= 0.f ? 1.f : 0.f);
          }
          mass += part;
        }
      });
  wave_lds_order();
  if (nodes < 0)
    return false;
  // 64 mass leaves in the cube of volume 8 h^3
  r = h * approx_cbrt(want * 1.909859f / fmaxf(64.f * mass, 0.05f * want));
  return wave_uniform(h) > 0.f && h < 1e15f;
}

} // namespace axb
