// pd_parts.hpp — the coloured sweep loops over a spatial partition of the bodies (gfx950, FP64).
//
// The velocity stage (src/solver_velocity.hpp:498-904) and the position loop
// (src/solver_position.hpp:248-331) are chains of colour passes: ~25 x 8 and ~12 x 10 of them per
// substep, each over rows that touch distinct bodies.  One launch per pass costs 5-9 us of launch,
// dependent loads and cache writeback whatever its size, so below a few hundred thousand rows the
// chain, not the memory, is the time.  Here a whole loop is one launch:
//
//   * the bodies are split into parts that are compact in space, one part per workgroup, and a
//     part's body states live in its workgroup's LDS for the whole loop;
//   * a row belongs to the part of its bodies; a row between two parts is evaluated by both, each
//     updating its own body.  For that the two workgroups exchange the row's two body states: a
//     workgroup sends a body's state as soon as the body's previous row is done, usually some
//     colours before the other needs it, and there is no barrier over the grid;
//   * two lanes evaluate a row, one for each of its bodies, exchanging what the row's impulses need
//     of both: a colour pass of a part is a few waves' dependent FP64 arithmetic, and this shortens
//     it;
//   * a workgroup's rows lie in colour order in chunks of one wave, and a wave loads its next chunk
//     as soon as it has finished one, so that the latency passes during the colours in between (a
//     wave with one chunk never loads it again).
//
// Every body sees the same rows in the same order with the same operands as in the per-colour
// launches, so the result is the same bit for bit.
//
// Exchange.  A state is sent as one 16-byte line per double, (low word, seq, high word, seq) with
// seq the number of the pass it is for, by device-scope stores; the receiver polls the lines with
// device-scope loads until every seq is the pass's.  Each 8-byte half validates itself, so neither
// fences nor acknowledgements are waited for.  Lines alternate between two buffers by the parity
// of seq.  A part sends a row's line of pass p + 2 after it has evaluated the row in pass p + 1,
// for which it received the partner's line of that pass, which the partner sent after it had
// evaluated the row in pass p, that is, had read the line that is now overwritten.
//
// Waiting needs all workgroups to be running.  They first check in; if they are not all running
// within a bounded time (other work holds the compute units) they agree, through one compare-and-
// swap, to leave.  Workgroup 0 then runs a small loop alone from global memory; of a larger one the
// host waits for the outcome of the check-in, and takes the launches per colour.  They leave as well
// where one part holds most of the rows or more bodies than LDS slots.  Once all have checked in
// every wait ends, since a workgroup never leaves before the loop does; the waits are bounded all
// the same, in polls and not by a clock (a process may be suspended for any time, and its polls
// with it), and a wait that runs out raises an error on the host.
// Bound: below ~50k rows by a colour pass's chain, the loads of a row's bodies, its dependent FP64
// arithmetic and for a row between parts the hop: 4,099 resting spheres 631 us for ~175 velocity
// passes and 203 us for 108 position passes (kernel trace, 3.6 and 1.9 us each).  Above by the rows'
// constants, gathered anew in every pass: 100,003 spheres 3.5 and 4.0 TB/s, 1M poured 5.0 and 5.2.
// Substeps of resting beds, MI355X, launches per colour or one workgroup (before) -> this: 4,099
// spheres 2.31 -> 0.90 ms, 9,001 4.03 -> 0.99 ms, 100,003 3.14 -> 2.12 ms; 60,013 raining 2.67 ->
// 1.41 ms.
#pragma once

#include "pd_kernels.hpp"

namespace pd {

typedef unsigned pu4 __attribute__((ext_vector_type(4)));

constexpr int PT_V_THREADS = 512;   // (a velocity row's ~215 VGPRs allow two waves per SIMD)
constexpr int PT_P_THREADS = 1024;  // (a position row's ~85 four)
constexpr int PT_CHUNK = 32;  // rows of a chunk: two lanes each
constexpr int PT_MAX_PARTS = 256;
constexpr int PT_COLORS = 62;  // the last class (62) may hold rows sharing a body: not taken here
constexpr int PT_MAX_CELLS = 32768;
// LDS slot codes of a row's bodies in an entry (16 bits each)
constexpr int PT_REMOTE = 0xFFFD;  // another part's body: received
constexpr int PT_GLOBAL = 0xFFFE;  // this part's body without an LDS slot: in global memory
constexpr int PT_NONE = 0xFFFF;    // no body (plane or wall)
// LDS bodies per part: the states fill at most 150 KB of the 160 KB
constexpr int PT_LDS_BYTES = 158 * 1024;
constexpr int PT_VBODIES = 3200;  // 48 B each
constexpr int PT_PBODIES = 6400;  // 24 B each
// dynamic LDS of a loop: bodies, then 16 bytes per class
inline int partLdsBytes(int cap, int classes, int nd) { return ((cap * nd * 8 + 15) & ~15) + 16 * classes; }

// cells of the partition: a box halved PT levels times, always across its longest edge; the
// cell index is the path of halves, so consecutive cells are close in space
struct PartGrid {
  d3 lo, inv;            // cell coordinate = (x - lo) * inv
  int dim[3];            // powers of two
  int levels;
  unsigned long long axes;  // axis of level l in bits [2l, 2l + 2)
};
// the arrays of one partition
struct PartList {
  int numParts, numColors, cap;
  PartGrid* grid;
  unsigned long long* mask;  // [ids] colours of each id's rows
  int* listStart;  // [ids] where each id's rows start in list
  int* list;       // [2 x rows] each id's rows in colour order: 2 x row + side, sign bit: between
  int* listCnt;    // places of list given out
  int* skew;       // set when one part holds far more rows than the others
  int* hist;       // [cells] weight
  int* cellStart;  // [cells + 1] its scan
  int* partOf;     // [ids] part << 20 | place in the part
  int* partCnt;    // [parts] bodies
  int* partIds;    // [parts x cap] the bodies with an LDS slot
  int* bktCnt;     // [parts x colours x 2] entries: between parts, inside
  int4* bkt;       // [parts x colours] (first entry, entries between parts, entries, 0)
  int2* rank;      // [rows] a row's place among its bucket's (x: part of A, y: part of B)
  int4* ent;       // entries: (row, loc A | loc B << 16, id A, id B)
  // what follows each of the entry's two bodies' row: (line the body's next row is sent in + 1, or
  // 0 when that row lies inside the part) << 2 | 2: in the next pass | 1: this row is its first
  int2* nxt;
  double* lam2;    // impulses of the rows between parts as the part of body B holds them
  double4* lamT2;
  unsigned char* flag2;
};
// exchange areas of one partition
struct PartSync {
  void* lines;       // [2][2 x rows] state lines
  unsigned lineBytes;  // size of the area
  unsigned half;     // bytes of one parity
  pu4* red;          // [2][PT_MAX_PARTS] maxima
  unsigned* arrive;  // [PT_MAX_PARTS]
  unsigned* decision;
  unsigned seq0;     // passes of this launch are numbered seq0 + 1, ...
  unsigned epoch;
  int* busy;         // set when one workgroup ran the loop alone: no more check-ins this substep
  int* over;         // gets overBit when a part had more bodies than LDS slots
  int overBit;       // (1: velocity rows, 2: position rows)
  int* fail;         // set when a wait ran out
  // where the outcome of the check-in goes in host memory, epoch << 1 | 1 for all running: then
  // nobody runs the loop alone (null: workgroup 0 does)
  unsigned long long* outcome;
  int refuse;        // 1: leave at the check-in (tests)
  // tests: 1: the last workgroup never checks in; 2: it leaves after the check-in
  int absent;
  int waitPolls;     // polls after which a wait has run out
};
constexpr long PT_CHECKIN_TICKS = 200000;  // 2 ms of the 100 MHz clock
constexpr int PT_WAIT_POLLS = 1 << 22;     // (a poll takes 0.5-1 us)

// device-scope accesses
template <class T>
__device__ __forceinline__ T ldDevice(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void stDevice(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- building a partition ------------------------------------------------------------------
__device__ __forceinline__ int partCoord(double f, int dim) {
  if (f >= (double)(dim - 1)) return dim - 1;
  return f >= 0.0 ? (int)f : 0;  // (NaN: 0)
}
__device__ __forceinline__ int partCell(const PartGrid& g, double4 p) {
  const int cx = partCoord((p.x - g.lo.x) * g.inv.x, g.dim[0]);
  const int cy = partCoord((p.y - g.lo.y) * g.inv.y, g.dim[1]);
  const int cz = partCoord((p.z - g.lo.z) * g.inv.z, g.dim[2]);
  int tx = g.dim[0], ty = g.dim[1], tz = g.dim[2];
  int code = 0;
  unsigned long long a = g.axes;
  for (int l = 0; l < g.levels; ++l, a >>= 2) {
    const int d = (int)(a & 3);
    bool upper;
    if (d == 0) {
      tx >>= 1;
      upper = cx & tx;
    } else if (d == 1) {
      ty >>= 1;
      upper = cy & ty;
    } else {
      tz >>= 1;
      upper = cz & tz;
    }
    code = code * 2 + (upper ? 1 : 0);
  }
  return code;
}
// The extent of the rows' bodies, from 16 x 16 rows spread evenly, one per thread: the medians of
// the 16 groups' smallest and largest coordinates, about the 4 % and 96 % quantiles.  A few bodies
// far away (one that left its container) do not move them.  What is no number is left as it was.
__device__ __forceinline__ void partExtent(const double (&x)[3], double* lo, double* hi) {
  __shared__ double sh[6][16];
  double a[3], b[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    a[d] = b[d] = x[d];
    for (int off = 1; off < 16; off <<= 1) {
      a[d] = fmin(a[d], __shfl_xor(a[d], off, 64));
      b[d] = fmax(b[d], __shfl_xor(b[d], off, 64));
    }
    if ((threadIdx.x & 15) == 0) {
      sh[d][threadIdx.x >> 4] = a[d];
      sh[3 + d][threadIdx.x >> 4] = b[d];
    }
  }
  __syncthreads();
  if (threadIdx.x < 96) {
    const int q = (int)threadIdx.x >> 4, me = (int)threadIdx.x & 15;
    const double own = sh[q][me];
    int rank = 0;
    for (int j = 0; j < 16; ++j) {
      const double v = sh[q][j];
      rank += v < own || (v == own && j < me) ? 1 : 0;
    }
    if (q < 3 && rank == 7) lo[q] = own;
    if (q >= 3 && rank == 8) hi[q - 3] = own;
  }
  __syncthreads();
}
__global__ __launch_bounds__(TPB) void k_part_begin(PartList Q, int ids, int cells) {
  const int i = gtid();
  if (i < ids) Q.mask[i] = 0ull;
  if (i == 0) *Q.listCnt = 0;
  if (i < cells) Q.hist[i] = 0;
  if (i < Q.numParts) Q.partCnt[i] = 0;
  if (i < Q.numParts * Q.numColors * 2) Q.bktCnt[i] = 0;
}
// One workgroup lays the cells: over the quantiles above and 0.15 of their distance on either side,
// within the broadphase grid's box.  Bodies outside fall into the outermost cells.  (The halvings
// are few and would be spent on the way to one distant body: with 9,001 spheres, one of them a
// thousand bed widths away, the velocity loops took 1.26 ms over the whole box and take 0.36 over
// the quantiles.)
__device__ __forceinline__ void partLayCells(const PartList& Q, const Grid* box, const int2* ends,
                                             const double4* pos, int rows, int levels) {
  static_assert(TPB == 256, "16 groups of 16 samples");
  const int i = (int)threadIdx.x;
  __shared__ double lo[3], hi[3];
  const Grid b = *box;
  const double e[3] = {b.h * b.dim[0], b.h * b.dim[1], b.h * b.dim[2]};
  const double boxLo[3] = {b.lo.x, b.lo.y, b.lo.z};
  if (i < 3) {
    lo[i] = boxLo[i];
    hi[i] = boxLo[i] + e[i];
  }
  const int sample = ((int)threadIdx.x & 15) * 16 + ((int)threadIdx.x >> 4);
  const double4 p = pos[ends[(int)((long)sample * rows / TPB)].x];
  const double xyz[3] = {p.x, p.y, p.z};
  partExtent(xyz, lo, hi);
  if (i == 0) {
    PartGrid g;
    double l[3], w[3];
    for (int d = 0; d < 3; ++d) {
      const double m = 0.15 * (hi[d] - lo[d]);
      l[d] = fmax(lo[d] - m, boxLo[d]);
      w[d] = fmin(hi[d] + m, boxLo[d] + e[d]) - l[d];
      if (!(w[d] > 0.0)) {
        l[d] = boxLo[d];
        w[d] = e[d];
      }
    }
    double ex = w[0], ey = w[1], ez = w[2];
    int dx = 1, dy = 1, dz = 1;
    g.lo = d3{l[0], l[1], l[2]};
    g.levels = levels;
    g.axes = 0;
    for (int l = 0; l < levels; ++l) {
      int d;
      if (ez > ex && ez > ey) {
        d = 2;
        ez *= 0.5;
        dz *= 2;
      } else if (ey > ex) {
        d = 1;
        ey *= 0.5;
        dy *= 2;
      } else {
        d = 0;
        ex *= 0.5;
        dx *= 2;
      }
      g.axes |= (unsigned long long)d << (2 * l);
    }
    g.dim[0] = dx;
    g.dim[1] = dy;
    g.dim[2] = dz;
    g.inv = d3{1.0 / ex, 1.0 / ey, 1.0 / ez};
    *Q.grid = g;
  }
}
__device__ __forceinline__ int classOf(const ClassStarts& cs, int numColors, int k) {
  int lo = 0, hi = numColors - 1;
  while (lo < hi) {  // the last class starting at or before k
    const int m = (lo + hi + 1) >> 1;
    if (cs.s[m] <= k) lo = m;
    else hi = m - 1;
  }
  return lo;
}
// the colours of each body's rows; the first workgroup lays the cells meanwhile
__global__ __launch_bounds__(TPB) void k_part_colours(PartList Q, const int2* ends, ClassStarts cs,
                                                      int rows, const Grid* box, const double4* pos,
                                                      int levels) {
  if (blockIdx.x == 0) {
    partLayCells(Q, box, ends, pos, rows, levels);
    return;
  }
  const int k = gtid() - TPB;
  if (k >= rows) return;
  const int2 ab = ends[k];
  const unsigned long long bit = 1ull << classOf(cs, Q.numColors, k);
  atomicOr(&Q.mask[ab.x], bit);
  if (ab.y >= 0) atomicOr(&Q.mask[ab.y], bit);
}
// a body weighs its rows and a little more, so that a part of few rows does not take all bodies
__global__ __launch_bounds__(TPB) void k_part_hist(PartList Q, const double4* pos, int ids) {
  const int i = gtid();
  if (i >= ids) return;
  const int deg = __popcll(Q.mask[i]);
  if (deg) atomicAdd(&Q.hist[partCell(*Q.grid, pos[i])], deg + 2);
}
// part and place of every body with rows, and the place of its list of rows: one atomic per
// workgroup and part, and one per workgroup
__global__ __launch_bounds__(1024) void k_part_assign(PartList Q, const double4* pos, int ids,
                                                      int cells) {
  __shared__ int cnt[PT_MAX_PARTS], base[PT_MAX_PARTS], waveTot[16], listBase;
  for (int p = threadIdx.x; p < Q.numParts; p += blockDim.x) cnt[p] = 0;
  __syncthreads();
  const int i = gtid();
  const int deg = i < ids ? __popcll(Q.mask[i]) : 0;
  int part = -1, local = 0;
  if (deg > 0) {
    const long total = Q.cellStart[cells];
    const int at = Q.cellStart[partCell(*Q.grid, pos[i])];
    part = (int)((long)at * Q.numParts / (total > 0 ? total : 1));
    if (part >= Q.numParts) part = Q.numParts - 1;
    local = atomicAdd(&cnt[part], 1);
  }
  int inc = deg;
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  for (int off = 1; off < 64; off <<= 1) {
    const int x = __shfl_up(inc, off, 64);
    if (lane >= off) inc += x;
  }
  if (lane == 63) waveTot[wave] = inc;
  __syncthreads();
  for (int p = threadIdx.x; p < Q.numParts; p += blockDim.x)
    base[p] = cnt[p] ? atomicAdd(&Q.partCnt[p], cnt[p]) : 0;
  int before = inc - deg, all = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wave) before += waveTot[w];
    all += waveTot[w];
  }
  if (threadIdx.x == 0) listBase = all ? atomicAdd(Q.listCnt, all) : 0;
  __syncthreads();
  if (part < 0) return;
  const int loc = base[part] + local;
  Q.partOf[i] = part << 20 | min(loc, 0xFFFFF);  // (a place past cap only says that it is)
  Q.listStart[i] = listBase + before;
  if (loc < Q.cap) Q.partIds[part * Q.cap + loc] = i;
}
// a row's place among its body's rows in colour order (a body's rows have distinct colours)
__device__ __forceinline__ int colourRank(unsigned long long mask, int c) {
  return __popcll(mask & ((1ull << c) - 1ull));
}
// a row's place in its buckets.  The rows of a workgroup follow one another in their class, so most
// share a colour and few parts: those count in LDS, with one global atomic per workgroup and bucket.
__global__ __launch_bounds__(1024) void k_part_count(PartList Q, const int2* ends, ClassStarts cs,
                                                     int rows) {
  __shared__ int cnt[2 * PT_MAX_PARTS], base[2 * PT_MAX_PARTS];
  for (int p = threadIdx.x; p < 2 * Q.numParts; p += blockDim.x) cnt[p] = 0;
  const int k0 = (int)(blockIdx.x * blockDim.x);
  const int c0 = classOf(cs, Q.numColors, k0);
  __syncthreads();
  const int k = k0 + (int)threadIdx.x;
  int c = -1, ia = 0, ib = -1;  // LDS buckets: part x 2 + (1: inside)
  int2 r = make_int2(0, -1);
  if (k < rows) {
    const int2 ab = ends[k];
    c = classOf(cs, Q.numColors, k);
    const int pa = Q.partOf[ab.x] >> 20;
    const int pb = ab.y >= 0 ? Q.partOf[ab.y] >> 20 : pa;
    ia = 2 * pa + (pa == pb ? 1 : 0);
    if (pa != pb) ib = 2 * pb;
    const int sign = pa != pb ? (int)0x80000000 : 0;
    Q.list[Q.listStart[ab.x] + colourRank(Q.mask[ab.x], c)] = 2 * k | sign;
    if (ab.y >= 0) Q.list[Q.listStart[ab.y] + colourRank(Q.mask[ab.y], c)] = (2 * k + 1) | sign;
    if (c == c0) {
      r.x = atomicAdd(&cnt[ia], 1);
      if (ib >= 0) r.y = atomicAdd(&cnt[ib], 1);
    } else {
      r.x = atomicAdd(&Q.bktCnt[((ia >> 1) * Q.numColors + c) * 2 + (ia & 1)], 1);
      if (ib >= 0) r.y = atomicAdd(&Q.bktCnt[((ib >> 1) * Q.numColors + c) * 2], 1);
    }
  }
  __syncthreads();
  for (int p = threadIdx.x; p < 2 * Q.numParts; p += blockDim.x)
    base[p] = cnt[p] ? atomicAdd(&Q.bktCnt[((p >> 1) * Q.numColors + c0) * 2 + (p & 1)], cnt[p]) : 0;
  __syncthreads();
  if (k >= rows) return;
  if (c == c0) {
    r.x += base[ia];
    if (ib >= 0) r.y += base[ib];
  }
  Q.rank[k] = r;
}
// entry ranges: every (part, colour) starts a new chunk.  One workgroup.  A part that holds
// several times the average and more than its workgroup takes at once (`wide` rows of every colour)
// keeps all others waiting: bodies in places far apart, which the cells did not separate.
__global__ __launch_bounds__(1024) void k_part_ranges(PartList Q, int wide) {
  __shared__ int waveTot[16], first[PT_MAX_PARTS + 1];
  const int n = Q.numParts * Q.numColors;
  const int per = (n + 1023) / 1024;
  const int b0 = (int)threadIdx.x * per, e0 = min(b0 + per, n);
  int own = 0;
  for (int i = b0; i < e0; ++i) own += (Q.bktCnt[2 * i] + Q.bktCnt[2 * i + 1] + PT_CHUNK - 1) & ~(PT_CHUNK - 1);
  int inc = own;
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  for (int off = 1; off < 64; off <<= 1) {
    const int x = __shfl_up(inc, off, 64);
    if (lane >= off) inc += x;
  }
  if (lane == 63) waveTot[wave] = inc;
  __syncthreads();
  int at = inc - own;
  for (int w = 0; w < wave; ++w) at += waveTot[w];
  for (int i = b0; i < e0; ++i) {
    const int nb = Q.bktCnt[2 * i], ni = Q.bktCnt[2 * i + 1];
    if (i % Q.numColors == 0) first[i / Q.numColors] = at;
    Q.bkt[i] = make_int4(at, nb, nb + ni, 0);
    at += (nb + ni + PT_CHUNK - 1) & ~(PT_CHUNK - 1);
    if (i == n - 1) first[Q.numParts] = at;
  }
  __syncthreads();
  bool uneven = false;
  if ((int)threadIdx.x < Q.numParts) {
    const long own = first[threadIdx.x + 1] - first[threadIdx.x];
    uneven = own * Q.numParts > 4L * first[Q.numParts] && own > (long)wide * Q.numColors;
  }
  const int any = __syncthreads_or(uneven ? 1 : 0);
  if (threadIdx.x == 0) *Q.skew = any;
}
// VEL: also the second copies of the impulses and flags of the rows between parts
template <bool VEL>
__global__ __launch_bounds__(TPB) void k_part_fill(const Dev* __restrict__ Dp, PartList Q,
                                                   const int2* ends, ClassStarts cs, int rows) {
  const Dev& D = *Dp;
  const int k = gtid();
  if (k >= rows) return;
  const int2 ab = ends[k];
  const int c = classOf(cs, Q.numColors, k);
  const int la = Q.partOf[ab.x], lb = ab.y >= 0 ? Q.partOf[ab.y] : -1;
  const int pa = la >> 20, pb = lb >= 0 ? lb >> 20 : pa;
  auto code = [&](int l) {
    const int s = l & 0xFFFFF;
    return s < Q.cap ? s : PT_GLOBAL;
  };
  auto next = [&](int id) {
    const unsigned long long mask = Q.mask[id];
    const int rank = colourRank(mask, c), deg = __popcll(mask);
    const int wrap = rank + 1 == deg ? 1 : 0;
    const int to = Q.list[Q.listStart[id] + (wrap ? 0 : rank + 1)];
    return (to < 0 ? (to & 0x7FFFFFFF) + 1 : 0) << 2 | wrap << 1 | (rank == 0 ? 1 : 0);
  };
  const int2 r = Q.rank[k];
  const int4 ra = Q.bkt[pa * Q.numColors + c];
  const int2 nx = make_int2(next(ab.x), lb >= 0 ? next(ab.y) : 0);
  if (pa == pb) {
    const int e = ra.x + ra.y + r.x;
    Q.ent[e] = make_int4(k, code(la) | (lb >= 0 ? code(lb) : PT_NONE) << 16, ab.x, ab.y);
    Q.nxt[e] = nx;
    return;
  }
  const int4 rb = Q.bkt[pb * Q.numColors + c];
  Q.ent[ra.x + r.x] = make_int4(k, code(la) | PT_REMOTE << 16, ab.x, ab.y);
  Q.nxt[ra.x + r.x] = nx;
  Q.ent[rb.x + r.y] = make_int4(k, PT_REMOTE | code(lb) << 16, ab.x, ab.y);
  Q.nxt[rb.x + r.y] = nx;
  if (VEL) {
    Q.lam2[k] = D.vLam[k];
    Q.lamT2[k] = D.vLamT[k];
    Q.flag2[k] = D.vFlag[k];
  }
}

// ---- exchange ------------------------------------------------------------------------------
// cache policy of the line accesses: device scope (sc1), volatile for the compiler
constexpr int PT_AUX = (int)(0x80000000u | 16u);
__device__ __forceinline__ __amdgpu_buffer_rsrc_t lineRsrc(void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ void lineSend(__amdgpu_buffer_rsrc_t r, unsigned off, double x,
                                         unsigned seq) {
  const unsigned long long b = dbits(x);
  const pu4 w = {(unsigned)b, seq, (unsigned)(b >> 32), seq};
  __builtin_amdgcn_raw_buffer_store_b128(w, r, off, 0, PT_AUX);
}
__device__ __forceinline__ double lineValue(pu4 w) {
  return bitsd((unsigned long long)w.z << 32 | w.x);
}
// the error check of a wait, every 128 polls; true: give up
__device__ __forceinline__ bool waitOver(int polls, int most, int* fail) {
  if ((polls & 127) != 127) return false;
  if (ldDevice(fail)) return true;
  if (polls < most) return false;
  stDevice(fail, 1);
  return true;
}
// ND doubles sent with `seq`, by the lanes with `need`; every lane of the wave calls it
template <int ND>
__device__ __forceinline__ void lineRecv(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned seq,
                                         bool need, double* x, int most, int* fail) {
  bool wait = need;
  for (int n = 0;; ++n) {
    if (wait) {
      pu4 w[ND];
#pragma unroll
      for (int q = 0; q < ND; ++q) w[q] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16 * q, 0, PT_AUX);
      wait = false;
#pragma unroll
      for (int q = 0; q < ND; ++q) {
        wait = wait || w[q].y != seq || w[q].w != seq;
        x[q] = lineValue(w[q]);
      }
    }
    if (!__any(wait) || waitOver(n, most, fail)) break;
  }
}
__device__ __forceinline__ void partOutcome(const PartSync& Y, unsigned go) {
  if (Y.outcome)
    __hip_atomic_store(Y.outcome, (unsigned long long)Y.epoch << 1 | go, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}
// every workgroup is running, and `fits` in all of them: true in all of them, or false in all
__device__ __forceinline__ bool partCheckIn(const PartSync& Y, int me, int parts, bool fits,
                                            int* shGo) {
  const int tid = threadIdx.x;
  if (parts == 1) return fits && !Y.refuse;
  if (Y.absent == 1 && me == parts - 1) return false;
  if (tid == 0) stDevice(&Y.arrive[me], Y.epoch);
  // (busy is read here, beside the loads of the check-in: read before it, the loop that follows
  // was compiled 1.5 % slower, 100,003 spheres 748 against 735 us)
  bool ok = fits && !Y.refuse && ldDevice(Y.busy) == 0;
  if (ok && tid < parts) {
    const long t0 = (long)wall_clock64();
    for (int n = 1; ldDevice(&Y.arrive[tid]) != Y.epoch; ++n) {
      if ((n & 15) != 0) continue;
      if (ldDevice(Y.decision) >> 1 == Y.epoch) break;  // already decided
      if ((long)wall_clock64() - t0 > PT_CHECKIN_TICKS) {
        ok = false;
        break;
      }
    }
  }
  ok = __syncthreads_and(ok ? 1 : 0) != 0;
  if (tid == 0) {
    unsigned d = ldDevice(Y.decision);
    while (d >> 1 != Y.epoch) {
      const unsigned want = Y.epoch << 1 | (ok ? 1u : 0u);
      const unsigned was = atomicCAS(Y.decision, d, want);
      d = was == d ? want : was;
    }
    *shGo = (int)(d & 1u);
    if (me == 0) partOutcome(Y, d & 1u);
  }
  __syncthreads();
  return *shGo != 0;
}
// the maximum of m over every thread of every workgroup, in every thread
__device__ __forceinline__ unsigned long long partMax(unsigned long long m, const PartSync& Y,
                                                      int me, int parts, unsigned seq,
                                                      unsigned long long* sh) {
  const unsigned long long M = blockMaxAll(m, sh);
  if (parts == 1) return M;
  pu4* const area = Y.red + (seq & 1u) * PT_MAX_PARTS;
  const __amdgpu_buffer_rsrc_t r = lineRsrc(area, PT_MAX_PARTS * 16);
  if (threadIdx.x == 0) lineSend(r, me * 16, bitsd(M), seq);
  double x = 0.0;
  const bool need = (int)threadIdx.x < parts;
  lineRecv<1>(r, threadIdx.x * 16, seq, need, &x, Y.waitPolls, Y.fail);
  return blockMaxAll(need ? dbits(x) : 0ull, sh);
}

// ---- the pass over a part's rows -----------------------------------------------------------
// A part's chunks in class order: class c has table[c] = (first entry, entries between parts,
// entries, base), and its chunk j belongs to wave (base + j) mod WAVES.
template <int WAVES>
__device__ __forceinline__ void tableLoad(const PartList& Q, int me, int4* table) {
  if (Q.numParts > 1) {
    for (int c = threadIdx.x; c < Q.numColors; c += blockDim.x) table[c] = Q.bkt[me * Q.numColors + c];
    __syncthreads();
  }
  if (threadIdx.x < 64) {
    int at = 0;
    for (int c0 = 0; c0 < Q.numColors; c0 += 64) {
      const int c = c0 + (int)threadIdx.x;
      const int n = c < Q.numColors ? (table[c].z + PT_CHUNK - 1) / PT_CHUNK : 0;
      int inc = n;
      for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(inc, off, 64);
        if ((int)threadIdx.x >= off) inc += x;
      }
      if (c < Q.numColors) table[c].w = (at + inc - n) % WAVES;
      at += __shfl(inc, 63, 64);
    }
  }
  __syncthreads();
}
// Workgroup barrier that orders LDS only.  __syncthreads also waits for every global access in
// flight: the acknowledgements of the impulse stores and the loads issued ahead.
__device__ __forceinline__ void ldsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// the other lane's value of a row's pair of lanes (both lanes active)
__device__ __forceinline__ double pairOther(double x) {
  const unsigned long long b = dbits(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0xB1, 0xF, 0xF, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0xB1, 0xF, 0xF, true);
  return bitsd((unsigned long long)hi << 32 | lo);
}
__device__ __forceinline__ d3 pairOther3(d3 a) {
  return d3{pairOther(a.x), pairOther(a.y), pairOther(a.z)};
}
// x or -x
__device__ __forceinline__ double signed1(double x, unsigned long long sign) {
  return bitsd(dbits(x) ^ sign);
}
__device__ __forceinline__ d3 signed3(d3 a, unsigned long long sign) {
  return d3{signed1(a.x, sign), signed1(a.y, sign), signed1(a.z, sign)};
}

constexpr int DIRTY_BODY = 1, DIRTY_LAM = 2, DIRTY_LT = 4;

// Body states in LDS or global memory and on the wire.  VelPart / PosPart give the row type, its
// loading, the body state (ND doubles) and the row update; PartRun drives them.  Lanes 2i and
// 2i + 1 hold the same row, the even one its body A and the odd one its body B.
//
// A wave that has finished a chunk issues the loads of its next one into the same registers, and
// of the entry of the one after that, in the first colour in which it has nothing to do.  What
// a row needs evaluated before its bodies' states is evaluated in a later such colour, when there
// is one.  GLOB: a part may have more bodies than LDS slots.
struct ChunkAt {
  int c, j;
};
template <class R, bool GLOB>
struct PartRun {
  static constexpr int ND = R::ND, WAVES = R::THREADS / 64;
  // (by value: references to kernel arguments kept in an object would place the arguments in
  // scratch memory)
  const R rows;
  const int numColors;
  const int4* const ent;
  const int* const nxt;  // [entries][2]
  int* const fail;
  const int waitPolls;
  const unsigned half;
  const int4* const table;  // LDS [numColors]
  double* const body;       // LDS [cap][ND]
  const __amdgpu_buffer_rsrc_t lines;
  unsigned pass;  // number of the current pass
  int wave, sub;
  bool isB;
  ChunkAt at0, at1;    // the chunk in registers and the one after it (c = -1: none)
  int ek, el, ea, eb, en;  // its entry: row, slot codes, ids, and what follows this lane's body
  int nk, nl, na, nb, nn;  // the entry after it
  bool finished;       // the row in registers is evaluated
  bool pending;        // ... is done with: the next one is to be loaded
  typename R::Row cur;

  __device__ __forceinline__ PartRun(const R& r, const PartList& q, const PartSync& y,
                                     const int4* t, double* b)
      : rows(r), numColors(q.numColors), ent(q.ent), nxt((const int*)q.nxt), fail(y.fail),
        waitPolls(y.waitPolls), half(y.half), table(t), body(b),
        lines(lineRsrc(y.lines, y.lineBytes)), pass(y.seq0) {
    wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    sub = (int)(threadIdx.x & 63) >> 1;
    isB = threadIdx.x & 1;
    start();
  }
  // the wave's first chunk of a class
  __device__ __forceinline__ int firstChunk(int base) const {
    const int j = wave - base;
    return j < 0 ? j + WAVES : j;
  }
  // the wave's chunk at or after a in the cycle of classes (c = -1: the wave has none)
  __device__ __forceinline__ ChunkAt chunkAt(ChunkAt a) const {
    int4 t = table[a.c];
    for (int n = 0; n <= numColors; ++n) {
      if (a.j * PT_CHUNK < t.z) return a;
      a.c = a.c + 1 == numColors ? 0 : a.c + 1;
      t = table[a.c];
      a.j = firstChunk(t.w);
    }
    a.c = -1;
    return a;
  }
  __device__ __forceinline__ ChunkAt after(ChunkAt a) const {
    a.j += WAVES;
    return chunkAt(a);
  }
  // Loads ahead have no condition (a lane past the chunk's end takes the last entry): a value that
  // may or may not be loaded is settled, and waited for, where the condition ends.
  __device__ __forceinline__ void entry(ChunkAt a, int& k, int& l, int& ia, int& ib, int& n) const {
    const int4 t = table[a.c];
    const int at = t.x + min(a.j * PT_CHUNK + sub, t.z - 1);
    const int4 e = ent[at];
    n = nxt[2 * at + (isB ? 1 : 0)];
    k = e.x;
    l = e.y;
    ia = e.z;
    ib = e.w;
  }
  // load the wave's first chunk (again, when the rows' flags changed)
  __device__ __forceinline__ void start() {
    at0 = ChunkAt{-1, 0};
    finished = true;
    pending = false;
    if (numColors == 0) return;
    at0 = chunkAt(ChunkAt{0, firstChunk(table[0].w)});
    if (at0.c < 0) return;
    at1 = after(at0);
    entry(at0, ek, el, ea, eb, en);
    entry(at1, nk, nl, na, nb, nn);
    finished = false;
    rows.load(isB, ek, el, ea, eb, cur);
  }
  // take the next chunk; a wave with one chunk keeps it
  __device__ __forceinline__ void advance() {
    pending = false;
    if (at1.c == at0.c && at1.j == at0.j) return;
    at0 = at1;
    at1 = after(at1);
    ek = nk; el = nl; ea = na; eb = nb; en = nn;
    // (opaque: a test of an entry's word moved to where the word is loaded would wait for it there)
    asm volatile("" : "+v"(ek), "+v"(el), "+v"(ea), "+v"(eb), "+v"(en));
    finished = false;
    rows.load(isB, ek, el, ea, eb, cur);
    entry(at1, nk, nl, na, nb, nn);
  }
  __device__ __forceinline__ void finish() {
    if (finished) return;
    finished = true;
    rows.finish(isB, ek, eb >= 0, cur);
  }
  // this lane's slot code and body, and the other lane's slot code
  __device__ __forceinline__ int own(int l) const { return isB ? (int)((unsigned)l >> 16) : l & 0xFFFF; }
  __device__ __forceinline__ int other(int l) const { return isB ? l & 0xFFFF : (int)((unsigned)l >> 16); }
  __device__ __forceinline__ void bodyLoad(int loc, int id, double* x) const {
    if (GLOB && loc == PT_GLOBAL) {
      rows.globalLoad(id, x);
    } else {
#pragma unroll
      for (int q = 0; q < ND; ++q) x[q] = body[loc * ND + q];
    }
  }
  __device__ __forceinline__ void bodyStore(int loc, int id, const double* x) const {
    if (GLOB && loc == PT_GLOBAL) {
      rows.globalStore(id, x);
    } else {
#pragma unroll
      for (int q = 0; q < ND; ++q) body[loc * ND + q] = x[q];
    }
  }
  // byte offset of line 2 x row + side in pass `seq`
  __device__ __forceinline__ unsigned lineAt(unsigned line, unsigned seq) const {
    return (seq & 1u ? half : 0u) + line * (16u * ND);
  }
  __device__ __forceinline__ void send(unsigned line, unsigned seq, const double* x) const {
    const unsigned off = lineAt(line, seq);
#pragma unroll
    for (int q = 0; q < ND; ++q) lineSend(lines, off + 16 * q, x[q], seq);
  }
  // this lane's body, received when it is another part's
  __device__ __forceinline__ void state(bool live, int k, int l, int id, double* x) const {
    const int loc = own(l);
    const bool remote = live && loc == PT_REMOTE;
    if (live && !remote && loc != PT_NONE) bodyLoad(loc, id, x);
    if (__any(remote))
      lineRecv<ND>(lines, remote ? lineAt(2 * k + (isB ? 1 : 0), pass) : 0u, pass, remote, x, waitPolls, fail);
  }
  // send, for pass `seq`, the states of this wave's rows between parts: all of them, or of those
  // that are their body's first row in a pass (what the rows before do not send)
  __device__ __forceinline__ void sendRows(unsigned seq, bool all) const {
    for (int c = 0; c < numColors; ++c) {
      const int4 t = table[c];
      for (int j = firstChunk(t.w); j * PT_CHUNK < t.y; j += WAVES) {
        const int at = j * PT_CHUNK + sub;
        if (at >= t.y) continue;
        const int4 o = ent[t.x + at];
        const int loc = own(o.y), first = nxt[2 * (t.x + at) + (isB ? 1 : 0)] & 1;
        if (loc == PT_REMOTE || !(all || first)) continue;
        double x[ND];
        bodyLoad(loc, isB ? o.w : o.z, x);
        send(2 * o.x + (isB ? 1 : 0), seq, x);
      }
    }
  }
  // both lanes of a row of a body and its own image take what the row leaves in the body
  __device__ __forceinline__ void selfRow(bool changed, double* x) const {
    const int b = __builtin_amdgcn_update_dpp(0, changed ? 1 : 0, 0xB1, 0xF, 0xF, true);
    const bool fromB = isB ? changed : b != 0;
#pragma unroll
    for (int q = 0; q < ND; ++q) {
      const double o = pairOther(x[q]);
      if (fromB != isB) x[q] = o;
    }
  }
  // one pass over the colours; returns this thread's largest residual
  template <int MODE>
  __device__ __forceinline__ unsigned long long sweep(double thr) {
    ++pass;
    unsigned long long m = 0;
    int4 tn = numColors > 0 ? table[0] : make_int4(0, 0, 0, 0);
    for (int c = 0; c < numColors; ++c) {
      const int4 t = tn;
      tn = table[c + 1 < numColors ? c + 1 : 0];
      const int n = t.z;
      if (n == 0) continue;
      // the earlier colours' states are in LDS (or in global memory)
      if (GLOB) __syncthreads();
      else ldsBarrier();
      int j = firstChunk(t.w);
      if (j * PT_CHUNK >= n) {  // nothing to do in this colour: get ready for the next one
        if (pending) advance();
        else finish();
        continue;
      }
      if (pending) advance();
      for (;;) {
        // (the chunk in registers is this one)
        finish();
        double x[ND];
#pragma unroll
        for (int q = 0; q < ND; ++q) x[q] = 0.0;
        const bool live = j * PT_CHUNK + sub < n;
        const int id = isB ? eb : ea;
        state(live, ek, el, id, x);
        double amax = 0.0;
        const int dirty = rows.template apply<MODE>(isB, ek, cur, thr, x, amax);
        if (live) {
          const int loc = own(el);
          rows.save(isB, ek, el, cur, dirty);
          // (a body in contact with its own image: the row's body B is stored last)
          if (ea == eb) selfRow(dirty & DIRTY_BODY, x);
          if (((dirty & DIRTY_BODY) || ea == eb) && loc != PT_REMOTE) bodyStore(loc, id, x);
          if ((en >> 2) != 0 && loc != PT_REMOTE) send((en >> 2) - 1, pass + ((en >> 1) & 1), x);
          const unsigned long long a = dbits(amax);
          m = a > m ? a : m;
        }
        j += WAVES;
        if (j * PT_CHUNK >= n) break;
        advance();
      }
      pending = true;
    }
    return m;
  }
};

// Velocity rows (pgsRowB, gsRowB and warmApplyRowB with the two bodies in two lanes): the state is
// (v, w).  The odd lane works with the normal, the friction impulse and every relative quantity
// negated, which changes no rounding: what it adds to body B is what the row adds to it.
struct VelPart {
  static constexpr int ND = 6, THREADS = PT_V_THREADS;
  struct Row {
    d3 N, r, Tau;  // normal sum and this lane's arm and angular row
    double rest, mu, sgn, vn0, lenN, invLenN;
    double wn, wOther, growth, align;  // normal effective inverse masses; growth rate term
    double m, mSum;
    q4 q;
    d3 iI;
    double lam, pimp;
    d3 lt;
    double w4;     // as loaded: mu (even lane) or the sign (odd lane)
    double lam0;   // impulses as loaded; lam, lt, pimp have those being updated (one variable for
    double4 lt0;   // both would be settled, and its load waited for, where a chunk is kept)
    unsigned char fl;
    bool hasB;
  };
  const Dev& D;
  const double growthRate, restT;
  const PD_G Body64* const vw;
  const PD_G BodyC* const bc;
  const PD_G double4* const vN;
  const PD_G double4* const vRA;
  const PD_G double4* const vRB;
  const PD_G double4* const vWV;
  const PD_G double* const vVn0;
  PD_G double* const vLam;
  PD_G double4* const vLamT;
  PD_G unsigned char* const vFlag;
  PD_G double* const lam2;
  PD_G double4* const lamT2;
  PD_G unsigned char* const flag2;
  __device__ __forceinline__ VelPart(const Dev& d, const Params& P, const PartList& Q)
      : D(d), growthRate(P.growthRate), restT(P.restT), vw(d.vw), bc(d.bc), vN(d.vN), vRA(d.vRA),
        vRB(d.vRB), vWV(d.vWV), vVn0(d.vVn0), vLam(d.vLam), vLamT(d.vLamT), vFlag(d.vFlag),
        lam2((PD_G double*)Q.lam2), lamT2((PD_G double4*)Q.lamT2),
        flag2((PD_G unsigned char*)Q.flag2) {}
  // the part of body B keeps its own copy of a shared row's impulses and flags
  __device__ __forceinline__ static bool second(int l) { return (l & 0xFFFF) == PT_REMOTE; }
  __device__ __forceinline__ void load(bool isB, int k, int l, int ia, int ib, Row& w) const {
    const bool s2 = second(l);
    const int id = isB && ib >= 0 ? ib : ia;
    // (a boundary row's odd lane takes the wall's velocity in place of an orientation)
    const PD_G double4* const q = isB && ib < 0 ? vWV + k : &bc[id].q;
    const double4 q4v = *q, iim = bc[id].iim, n4 = vN[k];
    const double4 r4 = *(isB ? vRB + k : vRA + k);
    w.q = toq(q4v);
    w.iI = xyz(iim);
    w.m = iim.w;
    w.N = xyz(n4);
    w.rest = n4.w;
    w.r = xyz(r4);
    w.w4 = r4.w;
    w.vn0 = vVn0[k];
    w.lam0 = *(s2 ? lam2 + k : vLam + k);
    w.lt0 = *(s2 ? lamT2 + k : vLamT + k);
    w.fl = *(s2 ? flag2 + k : vFlag + k);
  }
  __device__ __forceinline__ void finish(bool isB, int k, bool hasB, Row& w) const {
    const unsigned long long sign = isB ? 1ull << 63 : 0ull;
    w.hasB = hasB;
    w.lam = w.lam0;
    w.lt = signed3(xyz(w.lt0), sign);
    w.pimp = w.lt0.w;
    w.N = signed3(w.N, sign);
    const double o4 = pairOther(w.w4);
    w.mu = isB ? o4 : w.w4;
    w.sgn = isB ? w.w4 : o4;
    double invN = 1.0;
    if (w.fl & F_ONE) {
      // one-point row: the one-term sums (rowTaus)
      w.Tau = add3(d3{0.0, 0.0, 0.0}, cross3(w.r, w.N));
    } else {
      const double4 t4 = *(isB ? D.vTB + k : D.vTA + k);
      w.Tau = xyz(t4);
      if (isB) invN = t4.w;
    }
    if (isB && !hasB) {
      const d3 v = scale3(d3{w.q.x, w.q.y, w.q.z}, invN);  // wallBody
      w.q = q4{v.x, v.y, v.z, 0.0};
      w.m = 0.0;
      w.iI = d3{0.0, 0.0, 0.0};
    }
    w.lenN = rowLenN(w.N);
    w.wn = dot3(w.N, w.N) * w.m + genInvMass(w.Tau, w.iI, w.q);
    w.wOther = pairOther(w.wn);
    w.mSum = w.m + pairOther(w.m);
    const d3 ro = pairOther3(w.r);
    // rA - rB (odd lane: negated); rA alone for a boundary row
    d3 diff = sub3(w.r, ro);
    if (!hasB) diff = isB ? neg3(ro) : w.r;
    w.growth = dot3(scale3(diff, growthRate), w.N);
    w.align = dot3(w.N, diff);
    w.invLenN = w.lenN > 0.0 ? 1.0 / w.lenN : 0.0;
  }
  __device__ __forceinline__ void globalLoad(int id, double* x) const {
    const Body64 b = vw[id];
    x[0] = b.v.x; x[1] = b.v.y; x[2] = b.v.z;
    x[3] = b.w.x; x[4] = b.w.y; x[5] = b.w.z;
  }
  __device__ __forceinline__ void globalStore(int id, const double* x) const {
    PD_G Body64* g = (PD_G Body64*)vw + id;
    g->v.x = x[0]; g->v.y = x[1]; g->v.z = x[2];
    g->w.x = x[3]; g->w.y = x[4]; g->w.z = x[5];
  }
  __device__ __forceinline__ static void push(const Row& w, d3 J, d3 torque, double* x) {
    x[0] += J.x * w.m;
    x[1] += J.y * w.m;
    x[2] += J.z * w.m;
    const d3 dw = angDelta(w.q, torque, w.iI);
    x[3] += dw.x;
    x[4] += dw.y;
    x[5] += dw.z;
  }
  // vA . N + wA . TauA - vB . N + wB . TauB, in that order in both lanes
  __device__ __forceinline__ static double normalVel(bool isB, const Row& w, d3 v, d3 om) {
    const double p1 = dot3(v, w.N), p2 = dot3(om, w.Tau);
    const double o1 = pairOther(p1), o2 = pairOther(p2);
    const double a1 = isB ? o1 : p1, a2 = isB ? o2 : p2, b1 = isB ? p1 : o1, b2 = isB ? p2 : o2;
    return a1 + a2 + b1 + b2;
  }
  // MODE 0 warm start, 1 PGS, 2 one-shot GS: returns what changed
  template <int MODE>
  __device__ __forceinline__ int apply(bool isB, int k, Row& w, double thr, double* x,
                                       double& amax) const {
    if (isB && !w.hasB) {
      x[0] = w.q.x;
      x[1] = w.q.y;
      x[2] = w.q.z;
    }
    const bool mine = !isB || w.hasB;
    if (MODE == 0) {
      // warmApplyRowB
      if (w.lam == 0.0 && !nonzero3(w.lt)) return 0;
      const double lambda = -w.sgn * w.lam;
      push(w, scale3(w.N, lambda), scale3(w.Tau, lambda), x);
      if (!nonzero3(w.lt)) return mine ? DIRTY_BODY : 0;
      if (w.lenN > 1e-9) {
        const d3 nhat = scale3(w.N, 1.0 / w.lenN);
        w.lt = sub3(w.lt, scale3(nhat, dot3(w.lt, nhat)));
      }
      push(w, w.lt, cross3(w.r, w.lt), x);
      return mine ? DIRTY_BODY | DIRTY_LT : DIRTY_LT;
    }
    if (w.lenN < 1e-9) return 0;
    double restitution = w.rest;
    const double vn = normalVel(isB, w, d3{x[0], x[1], x[2]}, d3{x[3], x[4], x[5]}) + w.growth;
    if (MODE == 2) {
      // gsRowB
      if (w.align > 0.0) {
        if (vn < 0.0) return 0;
      } else {
        if (vn > 0.0) return 0;
      }
      const double wTotal = w.wn + w.wOther;
      if (wTotal <= 0.0) return 0;
      amax = fabs(vn) / w.lenN;
      if (fabs(vn) < thr * w.lenN) restitution = 0.0;
      const double lambda = (-restitution * vn - vn) / wTotal;
      push(w, scale3(w.N, lambda), scale3(w.Tau, lambda), x);
      return mine ? DIRTY_BODY : 0;
    }
    // pgsRowB
    const int sf = (w.fl & F_SIDE1) ? 1 : ((w.fl & F_SIDE2) ? 2 : 0);
    const bool held = sf == (isB ? 1 : 2);  // the row leaves this lane's body as it is
    if (sf != 0) restitution = 0.0;
    const double wTotal = (held ? 0.0 : w.wn) + (sf != 0 && !held ? 0.0 : w.wOther);
    if (wTotal <= 0.0) return 0;
    int dirty = 0;
    const double v0til = w.sgn * w.vn0;
    const bool slow = fabs(w.vn0) < thr * w.lenN;
    if (slow) restitution = 0.0;
    const double target = (v0til > 0.0) ? -restitution * v0til : 0.0;
    const double vtil = w.sgn * vn;
    const double dp = (vtil - target) / wTotal;
    const double pOld = w.lam;
    double pNew = pOld + dp;
    if (pNew < 0.0) pNew = 0.0;
    const double dApplied = pNew - pOld;
    const double lamNow = dApplied != 0.0 ? pNew : pOld;
    if (dApplied != 0.0) {
      w.lam = pNew;
      dirty |= DIRTY_LAM;
      amax = fabs(dApplied) * wTotal / w.lenN;
      const double lambda = -w.sgn * dApplied;
      if (!held) {
        push(w, scale3(w.N, lambda), scale3(w.Tau, lambda), x);
        if (mine) dirty |= DIRTY_BODY;
      }
    }
    // friction cone
    const d3 ltOld = w.lt;
    if (w.mu > 0.0 || nonzero3(ltOld)) {
      const d3 nhat = scale3(w.N, w.invLenN);
      const d3 vp = add3(d3{x[0], x[1], x[2]}, cross3(d3{x[3], x[4], x[5]}, w.r));
      const d3 vrel = sub3(vp, pairOther3(vp));
      const d3 vt = sub3(vrel, scale3(nhat, dot3(vrel, nhat)));
      double beta = restT;
      if (beta != 0.0 && (sf != 0 || slow)) beta = 0.0;
      d3 vtErr = vt;
      if (beta != 0.0) {
        d3 v0 = signed3(xyz(D.vVt0[k]), isB ? 1ull << 63 : 0ull);
        v0 = sub3(v0, scale3(nhat, dot3(v0, nhat)));
        vtErr = add3(vt, scale3(v0, beta));
      }
      const double vtLen = sqrt(dot3(vtErr, vtErr));
      d3 ltNew = ltOld;
      double wT = w.mSum;
      if (vtLen > 1e-9) {
        const d3 that = scale3(vtErr, 1.0 / vtLen);
        const double wt =
            (held || !mine) ? 0.0 : w.m + genInvMass(cross3(w.r, that), w.iI, w.q);
        wT = wt + pairOther(wt);
        if (wT > 1e-9) ltNew = add3(ltOld, scale3(that, -vtLen / wT));
      }
      ltNew = sub3(ltNew, scale3(nhat, dot3(ltNew, nhat)));
      double nTot = fmax(lamNow, 0.0) * w.lenN;
      if (slow) nTot += fmax(w.pimp, 0.0);
      const double bound = w.mu * nTot;
      const double ltLen = sqrt(dot3(ltNew, ltNew));
      if (ltLen > bound) ltNew = (bound > 0.0) ? scale3(ltNew, bound / ltLen) : d3{0.0, 0.0, 0.0};
      const d3 dApp = sub3(ltNew, ltOld);
      if (nonzero3(dApp)) {
        w.lt = ltNew;
        dirty |= DIRTY_LT;
        const double dLen = sqrt(dot3(dApp, dApp));
        if (wT > 1e-9 && dLen * wT > amax) amax = dLen * wT;
        if (!held) {
          push(w, dApp, cross3(w.r, dApp), x);
          if (mine) dirty |= DIRTY_BODY;
        }
      }
    }
    return dirty;
  }
  __device__ __forceinline__ void save(bool isB, int k, int l, const Row& w, int dirty) const {
    if (isB) return;
    const bool s2 = second(l);
    if (dirty & DIRTY_LAM) *(s2 ? lam2 + k : vLam + k) = w.lam;
    if (dirty & DIRTY_LT) *(s2 ? lamT2 + k : vLamT + k) = tod4(w.lt, w.pimp);
  }
};

// The velocity stage one launch runs: optionally the warm-start pass, the sweep loop, and
// optionally the stabilization gate (src/sim.hpp:279-283) followed, for stabilization mode 1, by
// the side flags and the stabilization loop.
struct VStage {
  int warm;  // 1: warm-start pass first
  int iters;
  double thr, stopThr;
  int *stop, *count;
  int gate;      // 1: stabilization gate after the loop (writes stabRun and stabStop)
  int stabMode;  // the gate's mode; mode 1 also runs the side flags and the loop
  int stabIters;
  double stabThr;
  int *stabRun, *stabStop, *stabCount;
  d3 gHat;
  double riseThr, approachThr;
};
// The whole partition of a loop that one workgroup runs, built by that workgroup: a body's first
// row gives it its place, and the entries are the classes' rows as they lie.  table: LDS, one int4
// per class.
__device__ __forceinline__ void partSingle(const PartList& Q, const PD_G int2* ends,
                                           const ClassStarts& cs, int4* table) {
  __shared__ int bodies;
  const int r0 = cs.s[0], r1 = cs.s[Q.numColors];
  if (threadIdx.x == 0) bodies = 0;
  if (threadIdx.x < 64) {
    int at = 0;
    for (int c0 = 0; c0 < Q.numColors; c0 += 64) {
      const int c = c0 + (int)threadIdx.x;
      const int n = c < Q.numColors ? cs.s[c + 1] - cs.s[c] : 0;
      const int padded = (n + PT_CHUNK - 1) & ~(PT_CHUNK - 1);
      int inc = padded;
      for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(inc, off, 64);
        if ((int)threadIdx.x >= off) inc += x;
      }
      if (c < Q.numColors) table[c] = make_int4(at + inc - padded, 0, n, 0);
      at += __shfl(inc, 63, 64);
    }
  }
  for (int k = r0 + (int)threadIdx.x; k < r1; k += blockDim.x) {
    const int2 ab = ends[k];
    stDevice(&Q.partOf[ab.x], -1);
    if (ab.y >= 0) stDevice(&Q.partOf[ab.y], -1);
  }
  __syncthreads();
  auto place = [&](int id) {
    if (ldDevice(&Q.partOf[id]) != -1 || atomicCAS(&Q.partOf[id], -1, -2) != -1) return;
    const int loc = atomicAdd(&bodies, 1);
    stDevice(&Q.partOf[id], min(loc, 0xFFFFF));
    if (loc < Q.cap) Q.partIds[loc] = id;
  };
  for (int k = r0 + (int)threadIdx.x; k < r1; k += blockDim.x) {
    const int2 ab = ends[k];
    place(ab.x);
    if (ab.y >= 0) place(ab.y);
  }
  __syncthreads();
  auto code = [&](int id) {
    const int loc = ldDevice(&Q.partOf[id]);
    return loc < Q.cap ? loc : PT_GLOBAL;
  };
  for (int k = r0 + (int)threadIdx.x; k < r1; k += blockDim.x) {
    const int2 ab = ends[k];
    const int c = classOf(cs, Q.numColors, k);
    const int e = table[c].x + k - cs.s[c];
    Q.ent[e] = make_int4(k, code(ab.x) | (ab.y >= 0 ? code(ab.y) : PT_NONE) << 16, ab.x, ab.y);
    Q.nxt[e] = make_int2(0, 0);
  }
  if (threadIdx.x == 0) Q.partCnt[0] = bodies;
  __syncthreads();
}

// the stage by one workgroup, bodies in global memory
template <int MODE>
__device__ __forceinline__ void vStageAlone(const Dev& D, const Params& P, const ClassStarts& cs,
                                            int numColors, const VStage& S,
                                            unsigned long long* sh) {
  if (S.warm) vWarmPass(D, cs, numColors);
  vSweepLoop<MODE>(D, P, cs, numColors, S.iters, S.thr, S.stopThr, S.stop, S.count, sh);
  if (!S.gate) return;
  __syncthreads();  // the loop's last residual is in *D.maxApproachBits
  const int run = (S.stabMode != 0 && bitsd(*D.maxApproachBits) > S.stabThr) ? 1 : 0;
  __syncthreads();
  if (threadIdx.x == 0) {
    *S.stabRun = run;
    *S.stabStop = run ? 0 : 1;
  }
  if (!run || S.stabMode != 1) return;
  for (int k = cs.s[0] + (int)threadIdx.x; k < cs.s[numColors]; k += blockDim.x)
    sideFlagsRow(D, k, S.gHat, S.riseThr, S.approachThr, GBodies{D.vw});
  __syncthreads();
  vSweepLoop<1>(D, P, cs, numColors, S.stabIters, S.stabThr, S.stabThr, S.stabStop, S.stabCount, sh);
}
template <int MODE, bool GLOB>
__global__ __launch_bounds__(PT_V_THREADS) void k_vsolve_lds(const Dev* __restrict__ Dp, Params P,
                                                             ClassStarts cs, VStage S, PartList Q,
                                                             PartSync Y) {
  const Dev& D = *Dp;
  extern __shared__ double2 ptBody[];
  __shared__ unsigned long long sh[PT_V_THREADS / 64];
  __shared__ int go;
  const int me = blockIdx.x, parts = Q.numParts, tid = threadIdx.x;
  double* const body = reinterpret_cast<double*>(ptBody);
  int4* const table = reinterpret_cast<int4*>(ptBody + (Q.cap * 6 + 1) / 2);
  if (parts == 1) partSingle(Q, D.vAB, cs, table);
  const bool even = parts == 1 || *Q.skew == 0;
  const bool fits = !even || GLOB || Q.partCnt[me] <= Q.cap;
  if (!partCheckIn(Y, me, parts, even && fits, &go)) {
    if (tid == 0 && !fits) atomicOr(Y.over, Y.overBit);
    if (me != 0 || Y.outcome) return;
    if (tid == 0) *Y.busy = 1;
    vStageAlone<MODE>(D, P, cs, Q.numColors, S, sh);
    return;
  }
  if (Y.absent == 2 && me != 0 && me == parts - 1) return;
  const int nb = min(Q.partCnt[me], Q.cap);
  const VelPart rows(D, P, Q);
  for (int s = tid; s < nb; s += blockDim.x)
    rows.globalLoad(Q.partIds[me * Q.cap + s], body + 6 * s);
  tableLoad<PT_V_THREADS / 64>(Q, me, table);
  PartRun<VelPart, GLOB> run(rows, Q, Y, table, body);
  run.sendRows(run.pass + 1, false);
  unsigned red = Y.seq0;
  if (S.warm) (void)run.template sweep<0>(0.0);
  // phase 0: the sweep loop; phase 1: the stabilization loop
  for (int phase = 0;; ++phase) {
    const int iters = phase ? S.stabIters : S.iters;
    const double thr = phase ? S.stabThr : S.thr, stopThr = phase ? S.stabThr : S.stopThr;
    unsigned long long M = 0;
    int n = 0;
    bool done = false;
    while (n < iters && !done) {
      const unsigned long long m = run.template sweep<MODE>(thr);
      M = partMax(m, Y, me, parts, ++red, sh);
      ++n;
      done = bitsd(M) <= stopThr;
    }
    if (me == 0 && tid == 0 && n > 0) {
      *D.maxApproachBits = M;
      *(phase ? S.stabCount : S.count) += n;
      if (done) *(phase ? S.stabStop : S.stop) = 1;
    }
    if (phase || !S.gate) break;
    const bool runS = S.stabMode != 0 && bitsd(M) > S.stabThr;
    if (me == 0 && tid == 0) {
      *S.stabRun = runS ? 1 : 0;
      *S.stabStop = runS ? 0 : 1;
    }
    if (!runS || S.stabMode != 1) break;
    // side flags: every row needs both its bodies' velocities, so one exchange of all rows
    ++run.pass;
    __syncthreads();
    run.sendRows(run.pass, true);
    for (int c = 0; c < Q.numColors; ++c) {
      const int4 t = table[c];
      for (int j = run.firstChunk(t.w); j * PT_CHUNK < t.z; j += PT_V_THREADS / 64) {
        const int at = j * PT_CHUNK + run.sub;
        const bool live = at < t.z;
        const int4 en = Q.ent[t.x + min(at, t.z - 1)];
        double x[6] = {0, 0, 0, 0, 0, 0};
        run.state(live, en.x, en.y, run.isB ? en.w : en.z, x);
        const d3 v{x[0], x[1], x[2]};
        const d3 vo = pairOther3(v);
        if (!live || run.isB) continue;
        const bool s2 = VelPart::second(en.y);
        unsigned char* const fl = s2 ? Q.flag2 + en.x : (unsigned char*)D.vFlag + en.x;
        *fl = sideFlags(D, make_int2(en.z, en.w), *fl, D.vVn0[en.x], v, vo, S.gHat, S.riseThr,
                        S.approachThr);
      }
    }
    __syncthreads();  // (both lanes of a row read the flags next)
    run.start();  // (the rows have new flags)
    run.sendRows(run.pass + 1, false);
  }
  __syncthreads();
  for (int s = tid; s < nb; s += blockDim.x)
    rows.globalStore(Q.partIds[me * Q.cap + s], body + 6 * s);
}

// Position rows (posRow with the two bodies in two lanes, the odd one's normal negated): the state
// is the predicted position.
struct PosPart {
  static constexpr int ND = 3, THREADS = PT_P_THREADS;
  struct Row {
    d3 n, r;
    double wTotal, m, lam, lam0;  // (lam0: as loaded, see VelPart)
    bool hasB;
  };
  PD_G double4* const posPred;
  const PD_G double4* const pN;
  const PD_G double4* const pRA;
  const PD_G double4* const pRB;
  PD_G double* const pLam;
  __device__ __forceinline__ PosPart(const Dev& d)
      : posPred(d.posPred), pN(d.pN), pRA(d.pRA), pRB(d.pRB), pLam(d.pLam) {}
  __device__ __forceinline__ void load(bool isB, int k, int, int, int, Row& w) const {
    const double4 n4 = pN[k];
    const double4 r4 = *(isB ? pRB + k : pRA + k);
    w.n = xyz(n4);
    w.wTotal = n4.w;
    w.r = xyz(r4);
    w.m = r4.w;
    w.lam0 = pLam[k];  // (only the part of body A saves it)
  }
  __device__ __forceinline__ void finish(bool isB, int, bool hasB, Row& w) const {
    w.hasB = hasB;
    w.n = signed3(w.n, isB ? 1ull << 63 : 0ull);
    w.lam = w.lam0;
  }
  __device__ __forceinline__ void globalLoad(int id, double* x) const {
    const double4 p = posPred[id];
    x[0] = p.x; x[1] = p.y; x[2] = p.z;
  }
  __device__ __forceinline__ void globalStore(int id, const double* x) const {
    PD_G double4* p = posPred + id;
    p->x = x[0]; p->y = x[1]; p->z = x[2];
  }
  template <int MODE>
  __device__ __forceinline__ int apply(bool isB, int, Row& w, double, double* x,
                                       double& amax) const {
    const bool mine = !isB || w.hasB;
    // (a boundary row's second point is rB itself)
    d3 p = add3(d3{x[0], x[1], x[2]}, w.r);
    if (!mine) p = w.r;
    const double C = dot3(sub3(p, pairOther3(p)), w.n);
    if (C >= 0.0) return 0;
    if (w.wTotal < 1e-6) return 0;
    const double dLambda = -C / w.wTotal;
    w.lam += dLambda;
    x[0] = x[0] + w.n.x * dLambda * w.m;
    x[1] = x[1] + w.n.y * dLambda * w.m;
    x[2] = x[2] + w.n.z * dLambda * w.m;
    amax = -C;
    return mine ? DIRTY_BODY | DIRTY_LAM : DIRTY_LAM;
  }
  __device__ __forceinline__ void save(bool isB, int k, int l, const Row& w, int dirty) const {
    if (!isB && (dirty & DIRTY_LAM) && (l & 0xFFFF) != PT_REMOTE) pLam[k] = w.lam;
  }
};
// the position loop (strict stop: residual < tol); `gate` (optional): a flag that makes it return at
// once
template <bool GLOB>
__global__ __launch_bounds__(PT_P_THREADS) void k_psolve_lds(const Dev* __restrict__ Dp,
                                                             ClassStarts cs, int iters, double tol,
                                                             int* stop, int* count, PartList Q,
                                                             PartSync Y, const int* gate) {
  const Dev& D = *Dp;
  extern __shared__ double2 ptBody[];
  if (gate && *gate) {
    if (blockIdx.x == 0 && threadIdx.x == 0) partOutcome(Y, 1u);
    return;
  }
  __shared__ unsigned long long sh[PT_P_THREADS / 64];
  __shared__ int go;
  const int me = blockIdx.x, parts = Q.numParts, tid = threadIdx.x;
  double* const body = reinterpret_cast<double*>(ptBody);
  int4* const table = reinterpret_cast<int4*>(ptBody + (Q.cap * 3 + 1) / 2);
  if (parts == 1) partSingle(Q, D.pAB, cs, table);
  const bool even = parts == 1 || *Q.skew == 0;
  const bool fits = !even || GLOB || Q.partCnt[me] <= Q.cap;
  if (!partCheckIn(Y, me, parts, even && fits, &go)) {
    if (tid == 0 && !fits) atomicOr(Y.over, Y.overBit);
    if (me != 0 || Y.outcome) return;
    if (tid == 0) *Y.busy = 1;
    pSweepLoop(D, cs, Q.numColors, iters, tol, stop, count, sh);
    return;
  }
  if (Y.absent == 2 && me != 0 && me == parts - 1) return;
  const int nb = min(Q.partCnt[me], Q.cap);
  const PosPart rows(D);
  for (int s = tid; s < nb; s += blockDim.x)
    rows.globalLoad(Q.partIds[me * Q.cap + s], body + 3 * s);
  tableLoad<PT_P_THREADS / 64>(Q, me, table);
  PartRun<PosPart, GLOB> run(rows, Q, Y, table, body);
  run.sendRows(run.pass + 1, false);
  unsigned long long M = 0;
  int n = 0;
  bool done = false;
  while (n < iters && !done) {
    const unsigned long long m = run.template sweep<0>(0.0);
    M = partMax(m, Y, me, parts, Y.seq0 + n + 1, sh);
    ++n;
    done = bitsd(M) < tol;
  }
  if (me == 0 && tid == 0 && n > 0) {
    *D.maxOverlapBits = M;
    *count += n;
    if (done) *stop = 1;
  }
  __syncthreads();
  for (int s = tid; s < nb; s += blockDim.x)
    rows.globalStore(Q.partIds[me * Q.cap + s], body + 3 * s);
}

// ---- contact class 62 as a chain ------------------------------------------------------------
// The rows of one body follow one another in row order in this class, so it is a chain of waves of
// body-disjoint rows, for shell shapes (the many contacts of one pair) hundreds of them with a few
// dozen rows each.  With every slot's position in LDS one wavefront walks the chain, a row per lane:
// its LDS accesses are ordered without a barrier.  The rows of the next CHAIN_AHEAD steps are in
// registers or in flight and the entries of as many after them: a step's dependent arithmetic is
// ~450 clocks, a load ~1300.
constexpr int CHAIN_AHEAD = 4;
constexpr int CHAIN_THREADS = 256;  // (all of them move the positions)
constexpr int CHAIN_SLOTS = 6400;
inline int chainLdsBytes(int slots, int steps) { return slots * 24 + steps * 8; }
// entries in wave order: (row, slot A, slot B or -1, 0)
__global__ __launch_bounds__(TPB) void k_chain_entries(const Dev* __restrict__ Dp, const int* perm,
                                                       int count, int4* ent) {
  const Dev& D = *Dp;
  const int i = gtid();
  if (i >= count) return;
  const int k = perm[i];
  const int2 ab = D.pAB[k];
  ent[i] = make_int4(k, ab.x, ab.y, 0);
}
struct ChainRow {
  double4 n, rA, rB;
  double lam;
  int k, a, b;
};
__device__ __forceinline__ void chainLoad(const Dev& D, int4 e, ChainRow& w) {
  w.k = e.x;
  w.a = e.y;
  w.b = e.z;
  w.n = D.pN[e.x];
  w.rA = D.pRA[e.x];
  w.rB = D.pRB[e.x];
  w.lam = D.pLam[e.x];
}
// posRow on positions in LDS
__device__ __forceinline__ double chainRow(const Dev& D, const ChainRow& w, double* body) {
  const bool hasB = w.b >= 0;
  double* const a = body + 3 * w.a;
  double* const b = body + 3 * (hasB ? w.b : w.a);
  const d3 pA{a[0], a[1], a[2]}, pB{b[0], b[1], b[2]};
  const d3 n = xyz(w.n);
  d3 q = add3(pB, xyz(w.rB));
  if (!hasB) q = xyz(w.rB);
  const double C = dot3(sub3(add3(pA, xyz(w.rA)), q), n);
  if (C >= 0.0) return 0.0;
  if (w.n.w < 1e-6) return 0.0;
  const double dLambda = -C / w.n.w;
  D.pLam[w.k] = w.lam + dLambda;
  a[0] = pA.x + n.x * dLambda * w.rA.w;
  a[1] = pA.y + n.y * dLambda * w.rA.w;
  a[2] = pA.z + n.z * dLambda * w.rA.w;
  if (hasB) {
    b[0] = pB.x + -n.x * dLambda * w.rB.w;
    b[1] = pB.y + -n.y * dLambda * w.rB.w;
    b[2] = pB.z + -n.z * dLambda * w.rB.w;
  }
  return -C;
}
// steps: (first entry, rows), at most 64 rows of one wave each
__global__ __launch_bounds__(CHAIN_THREADS) void k_psweep_chain(const Dev* __restrict__ Dp,
                                                                const int4* ent, const int2* steps,
                                                                int numSteps, int numSlots,
                                                                const int* stop) {
  const Dev& D = *Dp;
  extern __shared__ double2 ptBody[];
  if (*stop) return;
  double* const body = reinterpret_cast<double*>(ptBody);
  int2* const st = reinterpret_cast<int2*>(body + 3 * numSlots);
  for (int i = threadIdx.x; i < numSlots; i += CHAIN_THREADS) {
    const double4 p = D.posPred[i];
    body[3 * i] = p.x;
    body[3 * i + 1] = p.y;
    body[3 * i + 2] = p.z;
  }
  for (int i = threadIdx.x; i < numSteps; i += CHAIN_THREADS) st[i] = steps[i];
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = (int)threadIdx.x;
    auto entry = [&](int s) {
      const int2 t = st[min(s, numSteps - 1)];
      return ent[t.x + min(lane, t.y - 1)];
    };
    ChainRow w[CHAIN_AHEAD];
    int4 e[CHAIN_AHEAD];
    unsigned long long m = 0;
#pragma unroll
    for (int q = 0; q < CHAIN_AHEAD; ++q) chainLoad(D, entry(q), w[q]);
#pragma unroll
    for (int q = 0; q < CHAIN_AHEAD; ++q) e[q] = entry(CHAIN_AHEAD + q);
    for (int s = 0; s < numSteps; s += CHAIN_AHEAD) {
#pragma unroll
      for (int q = 0; q < CHAIN_AHEAD; ++q) {
        if (s + q < numSteps && lane < st[s + q].y) {
          const unsigned long long a = dbits(chainRow(D, w[q], body));
          m = a > m ? a : m;
        }
        __builtin_amdgcn_wave_barrier();
        chainLoad(D, e[q], w[q]);
        e[q] = entry(s + q + 2 * CHAIN_AHEAD);
      }
    }
    m = waveMaxU64(m);
    if (lane == 0 && m) atomicMax((unsigned long long*)D.maxOverlapBits, m);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < numSlots; i += CHAIN_THREADS) {
    PD_G double4* const p = D.posPred + i;
    p->x = body[3 * i];
    p->y = body[3 * i + 1];
    p->z = body[3 * i + 2];
  }
}

}  // namespace pd
