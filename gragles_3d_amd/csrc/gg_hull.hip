// Level-set stage: grain existence, volume and surface area from the marching-
// cubes hull of the compared distance field, deletion of vanished grains and
// the box resize (grainhdl::level_set, src/grainhdl.cpp:669-684 ->
// LSbox::extractContour, src/box.cpp:1144-1161).
//
// The hull kernels walk the cells of a grain's input box as
// MarchingCubesAlgorithm::generateHull (src/marchingCubes.cpp:364-478): case
// index from the eight corners (inside = phi >= 0), VertexInterp
// (:484-499) on the cut edges, triangles from the case table, then the
// signed-tetrahedron volume term (src/grainHull.cpp:40-56, including its
// float(1/6) factor) and the triangle area (:120-131).  A grain exists iff
// some cell is cut.  Neumaier-compensated FP64 sums go to fixed slots of the
// grain's layers, and k_finalize adds them in layer order, so the result does
// not depend on scheduling.
#include <algorithm>

#include "gg_internal.h"

namespace gg {
namespace {
constexpr int kGridPerCU = 64;  // most workgroups per CU of a hull launch (each loads the triangle table once)
#include "mc_cases.inc"

// Triangle table row of each case: edge indices in nibbles, first triangle in
// the low nibbles, 0xF after the last entry.
__constant__ uint64_t c_tri[256];

// Cube corner q -> (dx,dy,dz) (src/marchingCubes.cpp:378-386) as bit masks
// over q: {0,0,1} {1,0,1} {1,0,0} {0,0,0} {0,1,1} {1,1,1} {1,1,0} {0,1,0}.
constexpr unsigned kCornerX = 0x66u, kCornerY = 0xF0u, kCornerZ = 0x33u;
// Edge e -> corner pair (src/marchingCubes.cpp:393-464) in nibbles:
// {0,1} {1,2} {2,3} {3,0} {4,5} {5,6} {6,7} {7,4} {0,4} {1,5} {2,6} {3,7}.
constexpr uint64_t kEdgeA = 0x321076543210ull, kEdgeB = 0x765447650321ull;

struct Acc {
  double s, c;
  __device__ void add(double x) {
    double t = s + x;
    if (fabs(s) >= fabs(x)) c += (s - t) + x;
    else c += (x - t) + s;
    s = t;
  }
  __device__ void merge(double s2, double c2) {
    double t = s + s2;
    double bp = t - s;
    double e = (s - (t - bp)) + (s2 - bp);
    s = t;
    c = c + c2 + e;
  }
};

constexpr int kTopoCapBits = 6;
static_assert((1 << kTopoCapBits) == kTopoCap, "grain topology table size");
static_assert(kTopoCap <= 64, "a junction list is a 64-bit mask over the grain table's slots");
constexpr int kJuncCapBits = 9;
static_assert((1 << kJuncCapBits) == kJuncCap, "grain junction table size");

// Cells are found from sign bits.  A wavefront loads a run of layers (one
// contiguous stretch of the box) in pieces of 64 voxels and keeps the ballot of
// phi >= 0 of each as one 64-bit word in LDS; a lane takes a row of cells (rows
// of more than 63 in two parts), shifts out the bits of its four corner rows and
// gets the row's cut cells (some corners inside, some outside) as one mask.  Most
// rows have none, and no corner value is read for a cell that is not cut.  Cut
// cells are queued and worked on 64 at a time, their corner values read again
// from the layers (cached).
constexpr int kHullAhead = 8;  // loads in flight

// An entry of a cell queue: x | y << 7 | layer << 14 (| case << 21).
__device__ inline uint32_t cell_entry(int x, int y, int k) {
  return (uint32_t)x | (uint32_t)y << 7 | (uint32_t)k << 14;
}

// The sign words of count voxels from src on; returns whether any is inside.
template <class T>
__device__ inline bool load_words(unsigned long long* w, const T* __restrict__ src, int count, int lane) {
  const int nw = (count + 63) >> 6;
  unsigned long long any = 0ull;
  for (int k0 = 0; k0 < nw; k0 += kHullAhead) {
    T v[kHullAhead];
#pragma unroll
    for (int u = 0; u < kHullAhead; ++u) {
      const int c = (k0 + u) * 64 + lane;
      v[u] = c < count ? src[c] : T(-1);
    }
    unsigned lo = 0, hi = 0;  // lane u: word k0 + u
#pragma unroll
    for (int u = 0; u < kHullAhead; ++u) {
      const unsigned long long m = __ballot(v[u] >= T(0));
      any |= m;
      lo = lane == u ? (unsigned)m : lo;
      hi = lane == u ? (unsigned)(m >> 32) : hi;
    }
    if (lane < kHullAhead && k0 + lane <= nw) w[k0 + lane] = (unsigned long long)hi << 32 | lo;
  }
  if (lane == 0 && (nw & (kHullAhead - 1)) == 0) w[nw] = 0ull;  // read past the end by word_bits
  return any != 0ull;
}

// 64 bits of the words from bit o on.
__device__ inline unsigned long long word_bits(const unsigned long long* w, int o) {
  const int i = o >> 6, sh = o & 63;
  const unsigned long long lo = w[i] >> sh;
  return sh ? lo | w[i + 1] << (64 - sh) : lo;
}

// LDS writes of a wavefront are seen by its later reads in order; this keeps
// the compiler from moving one past the other.
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Queues the cut cells of layers k0 .. k0 + nl - 1 (words of layers k0 .. k0 +
// nl in w), one per row and round.  push(entry, has) is called by the whole
// wavefront; CASE: entries with the cell's case index.
template <bool CASE, class F>
__device__ inline void cut_cells(const unsigned long long* w, int n, int k0, int nl, int lane, F push) {
  const int m1 = n - 1;
  const bool split = m1 > 63;  // rows of more than 63 cells in two parts
  const int rows = nl * m1, items = split ? 2 * rows : rows;
  const uint32_t inv = ((1u << 24) + (uint32_t)m1 - 1u) / (uint32_t)m1;  // r / m1 = r * inv >> 24 for r < 96^2
  for (int i0 = 0; i0 < items; i0 += 64) {
    const int it = i0 + lane;
    const bool live = it < items;
    const int r = live ? (split ? it >> 1 : it) : 0, xs = split && (it & 1) ? 63 : 0;
    const int kl = (int)(((uint64_t)(uint32_t)r * inv) >> 24), y = r - kl * m1;
    const int o = (kl * n + y) * n + xs;
    const unsigned long long m00 = word_bits(w, o), m10 = word_bits(w, o + n), m01 = word_bits(w, o + n * n),
                             m11 = word_bits(w, o + n * n + n);
    const unsigned long long any = m00 | m10 | m01 | m11, all = m00 & m10 & m01 & m11;
    const int width = min(63, m1 - xs);
    unsigned long long cut = live ? ((any | any >> 1) & ~(all & all >> 1)) & ((1ull << width) - 1ull) : 0ull;
    const uint32_t base = cell_entry(xs, y, k0 + kl);
    while (__ballot(cut != 0ull)) {
      const bool has = cut != 0ull;
      const int x = has ? (int)__builtin_ctzll(cut) : 0;
      cut &= cut - 1ull;
      uint32_t e = base + (uint32_t)x;
      if constexpr (CASE) {
        const unsigned a = (unsigned)(m01 >> x) & 3u, b = (unsigned)(m00 >> x) & 3u, c = (unsigned)(m11 >> x) & 3u,
                       d = (unsigned)(m10 >> x) & 3u;
        e |= (a | b >> 1 << 2 | (b & 1u) << 3 | c << 4 | d >> 1 << 6 | (d & 1u) << 7) << 21;
      }
      push(e, has);
    }
  }
}

// Corner values of the lane's cell into cv[corner * 64 + lane]; returns its case
// index (inside: phi >= 0).
template <class T>
__device__ inline unsigned stage_corners(T* cv, const T* __restrict__ p, int n, int nn2, int lane) {
  const T* q = p + nn2;
  const T v[8] = {q[0], q[1], p[1], p[0], q[n], q[n + 1], p[n + 1], p[n]};
  unsigned ci = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    cv[c * 64 + lane] = v[c];
    ci |= v[c] >= T(0) ? 1u << c : 0u;
  }
  return ci;
}

// Cube edge e as a word: corner a, corner b << 3, the offset of a (x, y, z bits
// 6..8), the edge's axis as bits 9..11 and bit 12 if b lies below a on it.
constexpr uint32_t edge_word(int e) {
  const unsigned a = (unsigned)(kEdgeA >> (4 * e)) & 15u, b = (unsigned)(kEdgeB >> (4 * e)) & 15u;
  const unsigned ax = (kCornerX >> a) & 1u, ay = (kCornerY >> a) & 1u, az = (kCornerZ >> a) & 1u;
  const unsigned bx = (kCornerX >> b) & 1u, by = (kCornerY >> b) & 1u, bz = (kCornerZ >> b) & 1u;
  const unsigned down = (ax & ~bx & 1u) | (ay & ~by & 1u) | (az & ~bz & 1u);
  return a | b << 3 | ax << 6 | ay << 7 | az << 8 | (ax ^ bx) << 9 | (ay ^ by) << 10 | (az ^ bz) << 11 | down << 12;
}

// VertexInterp (src/marchingCubes.cpp:484-499) at iso level 0 on the edge of
// word ew, in the cell with lower corner (x,y,z); the corner values from
// stage_corners.  An edge runs along one axis, so the vertex is the edge's first
// corner plus t along it: 0 where the first value is below 1e-5, +-1 where the
// second is, else +-mu.  (The reference also takes the first corner where the
// values are within 1e-5 of each other: one is inside and the other outside, so
// then one of them is below 1e-5.)
template <class T>
__device__ inline void edge_vertex(uint32_t ew, const T* cv, int slot, int x, int y, int z, double& px, double& py,
                                   double& pz) {
  const T v1 = cv[(ew & 7u) * 64 + slot], v2 = cv[((ew >> 3) & 7u) * 64 + slot];
  double t;
  if constexpr (sizeof(T) == 4) {
    // mu in FP32 (reciprocal, ~2 ulp): the values it interpolates are FP32
    // already.  |v| <= 1e-5f is |v| < 1e-5 (the float lies just below it).
    float mu = v1 * __builtin_amdgcn_rcpf(v1 - v2);
    mu = fabsf(v2) <= 1e-5f ? 1.0f : mu;
    mu = fabsf(v1) <= 1e-5f ? 0.0f : mu;
    t = (double)((ew >> 12) & 1u ? -mu : mu);
  } else {
    double mu = v1 / (v1 - v2);
    mu = fabs(v2) < 0.00001 ? 1.0 : mu;
    mu = fabs(v1) < 0.00001 ? 0.0 : mu;
    t = (ew >> 12) & 1u ? -mu : mu;
  }
  px = (double)(x + (int)((ew >> 6) & 1u)) + ((ew >> 9) & 1u ? t : 0.0);
  py = (double)(y + (int)((ew >> 7) & 1u)) + ((ew >> 10) & 1u ? t : 0.0);
  pz = (double)(z + (int)((ew >> 8) & 1u)) + ((ew >> 11) & 1u ? t : 0.0);
}

struct Tri {
  double p0x, p0y, p0z, p1x, p1y, p1z, p2x, p2y, p2z;
  __device__ double volume() const {  // src/grainHull.cpp:40-56
    const double v321 = p2x * p1y * p0z;
    const double v231 = p1x * p2y * p0z;
    const double v312 = p2x * p0y * p1z;
    const double v132 = p0x * p2y * p1z;
    const double v213 = p1x * p0y * p2z;
    const double v123 = p0x * p1y * p2z;
    return (double)(1.0f / 6.0f) * (-v321 + v231 + v312 - v132 - v213 + v123);
  }
  __device__ double area() const {  // src/grainHull.cpp:120-131, src/InterfacialElement.cpp:81-92
    const double abx = p0x - p1x, aby = p0y - p1y, abz = p0z - p1z;
    const double acx = p0x - p2x, acy = p0y - p2y, acz = p0z - p2z;
    const double cx = aby * acz - abz * acy;
    const double cy = abz * acx - abx * acz;
    const double cz = abx * acy - aby * acx;
    return sqrt(cx * cx + cy * cy + cz * cz) / 2.0;
  }
};
// The triangle of the table row's low three nibbles in the cell at (x, y, z).
template <class T>
__device__ inline Tri cell_triangle(uint32_t row, const uint32_t* s_edge, const T* cv, int slot, int x, int y, int z) {
  Tri t;
  edge_vertex<T>(s_edge[row & 15u], cv, slot, x, y, z, t.p0x, t.p0y, t.p0z);
  edge_vertex<T>(s_edge[(row >> 4) & 15u], cv, slot, x, y, z, t.p1x, t.p1y, t.p1z);
  edge_vertex<T>(s_edge[(row >> 8) & 15u], cv, slot, x, y, z, t.p2x, t.p2y, t.p2z);
  return t;
}

struct TriTable {
  uint64_t row[256];
  uint8_t count[256];  // triangles of each case
  uint32_t edge[16];
};
__device__ inline void load_tri_table(TriTable& s) {
  for (int i = threadIdx.x; i < 256; i += blockDim.x) {
    uint64_t row = c_tri[i];
    s.row[i] = row;
    int cnt = 0;
    for (; (row & 15u) != 15u; row >>= 12) ++cnt;
    s.count[i] = (uint8_t)cnt;
    if (i < 16) s.edge[i] = i < 12 ? edge_word(i) : 0u;
  }
}

// Compensated sums over the wavefront, the same on every run.
__device__ inline void wave_reduce(Acc& vol, Acc& area) {
  for (int off = 32; off > 0; off >>= 1) {
    const double s2 = __shfl_down(vol.s, off), c2 = __shfl_down(vol.c, off);
    const double a2 = __shfl_down(area.s, off), d2 = __shfl_down(area.c, off);
    vol.merge(s2, c2);
    area.merge(a2, d2);
  }
}

constexpr int kHullWords = 304;  // sign words in LDS: two layers of the largest box, or more of smaller ones
template <class T>
struct HullWave {
  unsigned long long w[kHullWords];
  uint32_t cells[128];
  uint16_t tq[5 * 64];  // triangles of the 64 cells at work: lane | triangle << 6
  uint8_t ci[64];       // their cases
  T cv[8 * 64];
};

// Existence, volume and area without topology: a wavefront takes kHullRun
// consecutive layer tiles of the plan (all classes, so the pieces of a run
// belong to one or two grains), carries a grain's pending cells and sums over
// its layers, and reuses the upper layer's words as the next lower ones.  Each
// lane of a batch of 64 cells then works on one triangle at a time.  A piece's
// sums go to the slot of its first layer, zeros to the others.
//
// What bounds it: latency (loads of a run, then the corner gathers and the
// chain of triangle arithmetic of a batch) at the six (FP32) and four (FP64)
// wavefronts per SIMD its registers allow; of the vector instructions about half
// are triangle arithmetic.  Before, two layers of values were staged in LDS per
// workgroup, every lane read eight corners of four cells to classify them, and
// each class had a launch whose XCDs took contiguous ranges, so that the
// largest boxes all went to one XCD.  Hull of one step, alone: 8000 grains FP32
// 1.46 -> 0.94 ms, FP64 2.35 -> 1.21; 20000 bimodal grains FP32 2.16 -> 1.12.  With
// contiguous ranges over all classes the last would be 2.25, with 16 loads in
// flight 2.31, at five wavefronts 2.37; runs of 8 layers leave 512 grains 60 %
// slower.
constexpr int kHullRun = 4;
template <class T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_hull(PlanDev P, DescDev din,
                                                                                      int32_t* exflag,
                                                                                      double* partials) {
  __shared__ HullWave<T> s_wave[4];
  __shared__ TriTable s_tri;
  load_tri_table(s_tri);
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  HullWave<T>& s = s_wave[wv];
  const unsigned long long below = (1ull << lane) - 1ull;
  // The classes with the largest boxes first (the longest pieces of work), each
  // class spread over the XCDs; workgroups take 4 consecutive runs.
  int skip = 0;  // workgroups of this XCD served by the classes before
  for (int cls = kClasses - 1; cls >= 0; --cls) {
    const int total = P.totals[kQLayers * kClasses + cls];
    const uint32_t* __restrict__ tmap = P.tmap[kQLayers] + P.tile_base[kQLayers * kClasses + cls];
    const int64_t slots = P.layer_base[cls];
    const TileRange tr = xcd_tiles((total + 4 * kHullRun - 1) / (4 * kHullRun), skip);
    skip = tr.skip;
    for (int bt = tr.first; bt < tr.end; bt += tr.step) {
      const int t1 = min(total, (bt * 4 + wv + 1) * kHullRun);
      for (int t = (bt * 4 + wv) * kHullRun; t < t1;) {  // pieces of one grain
        const uint32_t tile = tmap[t];
        const int g = (int)(tile >> 8), ka = (int)(tile & 0xFFu);
        const int32_t* b = din.bounds + 6 * g;
        const int x0 = b[0], y0 = b[1], z0 = b[2], n = b[3] - b[0], nn2 = n * n;
        const int kb = min(n, ka + t1 - t);  // its layers in this run: [ka, kb)
        const T* __restrict__ box = (const T*)din.arena + din.off[g];
        Acc vol{0.0, 0.0}, area{0.0, 0.0};
        int pend = 0;
        bool cut = false;
        auto batch = [&](int base, int cnt) {  // cells base .. base + cnt - 1 of the queue
          const uint32_t e = s.cells[base + min(lane, cnt - 1)];
          const int xl = e & 127u, yl = (e >> 7) & 127u, kl = (e >> 14) & 127u;
          const unsigned ci = stage_corners<T>(s.cv, box + ((int64_t)kl * n + yl) * n + xl, n, nn2, lane);
          s.ci[lane] = (uint8_t)ci;
          const int nt = lane < cnt ? s_tri.count[ci] : 0;
          int incl = nt;
  #pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(incl, o);
            if (lane >= o) incl += u;
          }
          const int nq = __builtin_amdgcn_readlane(incl, 63);
          for (int j = 0; j < nt; ++j) s.tq[incl - nt + j] = (uint16_t)(lane | j << 6);
          wave_fence();
          for (int q = lane; q < nq; q += 64) {
            const int v = s.tq[q], slot = v & 63;
            const uint32_t ce = s.cells[base + slot];
            const Tri tri = cell_triangle<T>((uint32_t)(s_tri.row[s.ci[slot]] >> (12 * (v >> 6))), s_tri.edge, s.cv, slot,
                                             x0 + (int)(ce & 127u), y0 + (int)((ce >> 7) & 127u),
                                             z0 + (int)((ce >> 14) & 127u));
            vol.add(tri.volume());
            area.add(tri.area());
          }
          wave_fence();  // the queue and the corners are refilled
        };
        for (int k = ka; k < min(kb, n - 1);) {
          // as many layers as the words hold
          const int nl = min(min(kb, n - 1) - k, (kHullWords * 64 - 64) / nn2 - 1);
          if (load_words<T>(s.w, box + (int64_t)k * nn2, (nl + 1) * nn2, lane)) {
            wave_fence();
            cut_cells<false>(s.w, n, k, nl, lane, [&](uint32_t e, bool has) {
              const unsigned long long m = __ballot(has);
              if (has) s.cells[pend + __popcll(m & below)] = e;
              pend += __popcll(m);
              cut = true;
              if (pend >= 64) {
                wave_fence();
                pend -= 64;
                batch(pend, 64);
              }
            });
            wave_fence();
          }
          k += nl;
        }
        if (pend > 0) batch(0, pend);
        wave_reduce(vol, area);
        if (lane == 0) {
          double* pp = partials + 4 * (slots + t);
          pp[0] = vol.s;
          pp[1] = vol.c;
          pp[2] = area.s;
          pp[3] = area.c;
          if (cut) atomicOr(&exflag[g], 1);
        }
        if (lane < 4)
          for (int u = 1; u < kb - ka; ++u) partials[4 * (slots + t + u) + lane] = 0.0;
        t += kb - ka;
      }
    }
  }
}

// A cell's barycenter sum (non-negative grid coordinates) in fixed point:
// integer adds make a list's position sum independent of the order in which
// cells add to it (exact to 2^-33 grid units per cell).
__device__ inline unsigned long long fixpos(double v) {
  return (unsigned long long)__double2ll_rn(v * kPosScale);
}

template <class T, int NMAX>
struct TopoWave {
  static constexpr int kWords = NMAX <= 48 ? 192 : 304;  // at least two layers
  static constexpr int kCells = 384;
  unsigned long long w[kWords];
  uint32_t cells[kCells + 64];
  T cv[8 * 64];
};
// The grain's tables while its hull is walked (layout of TopoDev's rows).
struct TopoLds {
  int key[kTopoCap], ord[kTopoCap];
  unsigned long long jm[kJuncCap], jp[3 * kJuncCap];
  double ja[kJuncCap];
  int jc[kJuncCap], jo[kJuncCap];
};

// The hull with topology: one workgroup per grain, so the grain's tables live in
// LDS and go out once, each wavefront with a share of the layers.  First every
// wavefront queues its cut cells and counts their triangles, and the grain's
// triangle records are reserved with one add; then the cells are worked on 64 at
// a time, one per lane: the ids at its corners (the grain itself inside, the
// IDLocal id outside, none outside the IDLocal box) into the id table with
// their first appearance, the mask of their slots into the junction table, and
// then its triangles, each made once for the volume, the area, the element sums
// and the record.  A wavefront whose queue fills up works it off at once and
// reserves those records by itself.
//
// What bounds it: latency, as without topology, and per cell the id and list
// look-ups and the chain of one cell's triangles (one lane per cell, because
// an element's sums add a cell's triangles in order).  128 registers (FP32; 26
// spilled outside the loops) let two workgroups share a CU: 6.3 ms per step at
// 20000 grains with records, against 10.4 at 185 registers.  A workgroup per
// (grain, layer) with tables in LDS merged into global ones, and each triangle
// made three times (volume, sums, record), took 26.5 ms; 2000 grains without
// records 1.7 -> 0.55 ms.
constexpr int kTopoWaves = 8;
template <class T, int NMAX>
__global__ __launch_bounds__(64 * kTopoWaves) __attribute__((amdgpu_waves_per_eu(4))) void k_hull_topo(PlanDev P, int c0, int c1, DescDev din, int32_t* exflag,
                                                               double* partials, IdlDev il, TopoDev topo,
                                                               int32_t* err) {
  __shared__ TopoWave<T, NMAX> s_wave[kTopoWaves];
  __shared__ TopoLds s_t;
  __shared__ TriTable s_tri;
  __shared__ int s_cnt[kTopoWaves];
  __shared__ unsigned long long s_raw;
  __shared__ double s_red[kTopoWaves][4];
  __shared__ int s_cut;
  load_tri_table(s_tri);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  TopoWave<T, NMAX>& s = s_wave[wv];
  const unsigned long long below = (1ull << lane) - 1ull;
  int ng = 0;  // grains of the classes (none of a plan that did not fit its arena)
  for (int c = c0; c < c1; ++c) ng += P.cls_count[c];
  for (int i = blockIdx.x; i < ng; i += gridDim.x) {
    const int p = P.cls_start[c0] + ng - 1 - i;  // the class with the larger boxes first
    const int g = P.grains[p];
    const int32_t* b = din.bounds + 6 * g;
    const int x0 = b[0], y0 = b[1], z0 = b[2], n = b[3] - b[0], m1 = n - 1, nn2 = n * n;
    const T* __restrict__ box = (const T*)din.arena + din.off[g];
    const int32_t* ib = il.bounds + 6 * g;
    const int ix0 = ib[0], iy0 = ib[1], iz0 = ib[2], inx = ib[3] - ib[0], iny = ib[4] - ib[1], inz = ib[5] - ib[2];
    const bool same = ix0 == x0 && iy0 == y0 && iz0 == z0 && inx == n && iny == n && inz == n;
    const uint32_t* __restrict__ idl = il.arena + il.off[g];
    for (int i = tid; i < kJuncCap; i += 64 * kTopoWaves) {
      s_t.jm[i] = 0ull;
      s_t.jp[3 * i] = s_t.jp[3 * i + 1] = s_t.jp[3 * i + 2] = 0ull;
      s_t.ja[i] = 0.0;
      s_t.jc[i] = 0;
      s_t.jo[i] = INT_MAX;
    }
    if (tid < kTopoCap) {
      s_t.key[tid] = -1;
      s_t.ord[tid] = INT_MAX;
    }
    if (tid == 0) s_cut = 0;
    __syncthreads();
    Acc vol{0.0, 0.0}, area{0.0, 0.0};
    // cells base .. base + cnt - 1 of the queue; their records go from raw[rec] on
    auto batch = [&](int base, int cnt, int64_t rec, bool records) -> int {
      const bool act = lane < cnt;
      const uint32_t e = s.cells[base + min(lane, cnt - 1)];
      const int xl = e & 127u, yl = (e >> 7) & 127u, kl = (e >> 14) & 127u;
      const int64_t at = ((int64_t)kl * n + yl) * n + xl;
      const unsigned ci = stage_corners<T>(s.cv, box + at, n, nn2, lane);
      uint32_t ids[8];
      if (same) {
        const uint32_t* i0 = idl + at;
        const uint32_t* i1 = i0 + nn2;
        ids[3] = i0[0];
        ids[2] = i0[1];
        ids[7] = i0[n];
        ids[6] = i0[n + 1];
        ids[0] = i1[0];
        ids[1] = i1[1];
        ids[4] = i1[n];
        ids[5] = i1[n + 1];
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int cx = x0 + xl + (int)((kCornerX >> q) & 1u) - ix0;
          const int cy = y0 + yl + (int)((kCornerY >> q) & 1u) - iy0;
          const int cz = z0 + kl + (int)((kCornerZ >> q) & 1u) - iz0;
          ids[q] = ((unsigned)cx < (unsigned)inx && (unsigned)cy < (unsigned)iny && (unsigned)cz < (unsigned)inz)
                       ? idl[((int64_t)cz * iny + cy) * inx + cx]
                       : 0xFFFFFFFFu;
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if ((ci >> q) & 1u) ids[q] = (uint32_t)g;
      const int cell = (kl * m1 + yl) * m1 + xl;
      // 1. grains: each distinct id with its first-appearance key (cell in the
      //    (z, y, x) loop * 8 + rank among the cell's ascending ids); the slots
      //    of the cell's ids make its list's mask
      uint64_t mask = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        bool first = act && ids[q] != 0xFFFFFFFFu;
        int rank = 0;
#pragma unroll
        for (int q2 = 0; q2 < q; ++q2) first &= ids[q2] != ids[q];
        if (!first) continue;
#pragma unroll
        for (int q2 = 0; q2 < 8; ++q2) {
          bool lower = ids[q2] < ids[q];
#pragma unroll
          for (int q3 = 0; q3 < q2; ++q3) lower &= ids[q3] != ids[q2];
          rank += lower ? 1 : 0;
        }
        const int key = (int)ids[q], o = cell * 8 + rank;
        uint32_t hsl = ((uint32_t)key * 2654435761u) >> (32 - kTopoCapBits);
        bool done = false;
        for (int pr = 0; pr < kTopoCap && !done; ++pr) {
          int old = s_t.key[hsl];
          if (old == -1) old = atomicCAS(&s_t.key[hsl], -1, key);
          if (old == -1 || old == key) {
            if (o < s_t.ord[hsl]) atomicMin(&s_t.ord[hsl], o);
            mask |= 1ull << hsl;
            done = true;
          }
          hsl = (hsl + 1) & (kTopoCap - 1);
        }
        if (!done) atomicOr(err, kErrTopo);
      }
      // 2. junctions: the cell's list as a mask over the grain's table slots
      int js = -1;
      if (mask != 0) {
        uint32_t hsl = (uint32_t)((mask * 0x9E3779B97F4A7C15ull) >> (64 - kJuncCapBits));
        for (int pr = 0; pr < kJuncCap && js < 0; ++pr) {
          unsigned long long old = s_t.jm[hsl];
          if (old == 0ull) old = atomicCAS(&s_t.jm[hsl], 0ull, (unsigned long long)mask);
          if (old == 0ull || old == mask) js = (int)hsl;
          hsl = (hsl + 1) & (kJuncCap - 1);
        }
        if (js < 0) atomicOr(err, kErrTopo);
        else if (cell < s_t.jo[js]) atomicMin(&s_t.jo[js], cell);
      }
      // 3. the triangles: volume, area, the element's barycenter and area sums
      //    (src/grainHull.cpp:227-270, src/triangle.h:12-18), the record
      const int nt = act ? s_tri.count[ci] : 0;
      int incl = nt;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
      }
      const int ntri = __builtin_amdgcn_readlane(incl, 63);
      wave_fence();
      uint64_t row = s_tri.row[ci];
      double sx = 0.0, sy = 0.0, sz = 0.0, sa = 0.0;
      TriRec* out = records ? topo.raw + rec + (incl - nt) : nullptr;
      for (int j = 0; j < nt; ++j, row >>= 12) {
        const Tri t = cell_triangle<T>((uint32_t)row, s_tri.edge, s.cv, lane, x0 + xl, y0 + yl, z0 + kl);
        vol.add(t.volume());
        const double ar = t.area();
        area.add(ar);
        sa += ar;
        TriRec r;
        r.x = (t.p0x + t.p1x + t.p2x) / 3;
        r.y = (t.p0y + t.p1y + t.p2y) / 3;
        r.z = (t.p0z + t.p1z + t.p2z) / 3;
        sx += r.x;
        sy += r.y;
        sz += r.z;
        if (records) {
          r.g = js >= 0 ? g : 0;  // grain 0 has no elements: the record is passed over
          r.slot = js >= 0 ? js : 0;
          out[j] = r;
        }
      }
      if (js >= 0) {
        atomicAdd(&s_t.jp[3 * js], fixpos(sx));
        atomicAdd(&s_t.jp[3 * js + 1], fixpos(sy));
        atomicAdd(&s_t.jp[3 * js + 2], fixpos(sz));
        atomicAdd(&s_t.ja[js], sa);
        atomicAdd(&s_t.jc[js], nt);
      }
      wave_fence();  // the queue and the corners are refilled
      return ntri;
    };
    // room for cnt records, or none (the device error is set): -1
    auto reserve = [&](int cnt) -> int64_t {
      const unsigned long long rb = atomicAdd(topo.raw_n, (unsigned long long)cnt);
      if (rb + (unsigned long long)cnt <= (unsigned long long)topo.raw_cap) return (int64_t)rb;
      atomicOr(err, kErrTri);
      for (unsigned long long r = rb; r < (unsigned long long)topo.raw_cap && r < rb + (unsigned long long)cnt; ++r)
        topo.raw[r].g = topo.raw[r].slot = 0;
      return -1;
    };
    auto triangles = [&](int base, int cnt) {  // of the queue's cells
      int c = 0;
      for (int i = lane; i < cnt; i += 64) c += s_tri.count[s.cells[base + i] >> 21];
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) c += __shfl_xor(c, o);
      return c;
    };
    // this wavefront's cut cells
    int pend = 0;
    bool cut = false;
    {
      const int k0 = m1 * wv / kTopoWaves, k1 = m1 * (wv + 1) / kTopoWaves;
      for (int k = k0; k < k1;) {
        const int nl = min(k1 - k, (TopoWave<T, NMAX>::kWords * 64 - 64) / nn2 - 1);
        if (load_words<T>(s.w, box + (int64_t)k * nn2, (nl + 1) * nn2, lane)) {
          wave_fence();
          cut_cells<true>(s.w, n, k, nl, lane, [&](uint32_t e, bool has) {
            const unsigned long long m = __ballot(has);
            if (has) s.cells[pend + __popcll(m & below)] = e;
            pend += __popcll(m);
            cut = true;
            if (pend > TopoWave<T, NMAX>::kCells) {
              wave_fence();
              pend -= 64;
              int64_t rec = -1;
              if (topo.corr) {
                const int c = triangles(pend, 64);
                if (lane == 0) rec = reserve(c);
                rec = __shfl(rec, 0);
              }
              batch(pend, 64, rec, rec >= 0);
            }
          });
          wave_fence();
        }
        k += nl;
      }
    }
    int64_t rec = -1;
    if (topo.corr) {
      const int c = triangles(0, pend);
      if (lane == 0) s_cnt[wv] = c;
      __syncthreads();
      if (tid == 0) {
        int tot = 0;
        for (int w = 0; w < kTopoWaves; ++w) tot += s_cnt[w];
        s_raw = tot ? (unsigned long long)reserve(tot) : 0ull;
      }
      __syncthreads();
      rec = (int64_t)s_raw;
      for (int w = 0; w < wv; ++w)
        if (rec >= 0) rec += s_cnt[w];
    }
    for (int base = 0; base < pend; base += 64) {
      const int c = batch(base, min(64, pend - base), rec, rec >= 0);
      if (rec >= 0) rec += c;
    }
    wave_reduce(vol, area);
    if (lane == 0) {
      s_red[wv][0] = vol.s;
      s_red[wv][1] = vol.c;
      s_red[wv][2] = area.s;
      s_red[wv][3] = area.c;
      if (cut) s_cut = 1;
    }
    __syncthreads();
    const int cls = size_class(n);
    const int64_t slot = P.layer_base[cls] + P.pre[kQLayers][p + cls];  // the grain's first layer (class c's prefixes start at cls_start[c] + c)
    if (tid == 0) {
      Acc va{s_red[0][0], s_red[0][1]}, aa{s_red[0][2], s_red[0][3]};
      for (int w = 1; w < kTopoWaves; ++w) {
        va.merge(s_red[w][0], s_red[w][1]);
        aa.merge(s_red[w][2], s_red[w][3]);
      }
      double* pp = partials + 4 * slot;
      pp[0] = va.s;
      pp[1] = va.c;
      pp[2] = aa.s;
      pp[3] = aa.c;
      if (s_cut) atomicOr(&exflag[g], 1);
    }
    for (int i = 4 + tid; i < 4 * n; i += 64 * kTopoWaves) partials[4 * slot + i] = 0.0;
    if (tid < kTopoCap) {
      topo.key[(int64_t)g * kTopoCap + tid] = s_t.key[tid];
      topo.ord[(int64_t)g * kTopoCap + tid] = s_t.ord[tid];
    }
    const int64_t jb = (int64_t)g * kJuncCap;
    for (int i = tid; i < kJuncCap; i += 64 * kTopoWaves) {
      topo.jkey[jb + i] = s_t.jm[i];
      topo.jcnt[jb + i] = s_t.jc[i];
      topo.jarea[jb + i] = s_t.ja[i];
      if (topo.corr) topo.jord[jb + i] = s_t.jo[i];
    }
    for (int i = tid; i < 3 * kJuncCap; i += 64 * kTopoWaves) topo.jpos[3 * jb + i] = s_t.jp[i];
    __syncthreads();  // the tables are refilled for the next grain
  }
}

// Per grain: vanished -> deleted; alive -> take the comparison list as the new
// neighbour list, decide existence, finish volume/area, resize the output box
// to the set-comparison bounds (+-grid_blowup, clamped, src/box.cpp:857-877)
// made cubic.  mode selects the parts:
//   kFinBounds  the output box of every alive grain (it follows from the
//               set-comparison bounds alone, so it can precede the hull)
//   kFinState   deletion, list flip, existence, volume and area (after the hull)
//   kFinCoarsen extractContour as a grid coarsening calls it
//               (src/grainhdl.cpp:1481-1490) rather than level_set: no
//               deletion, the neighbour lists stay, and newb holds resizeGrid's
//               bounds, taken as they are
// With kFinState the output box is written for grains that keep existing only.
__global__ void k_finalize(SimParams sp, PlanDev P, DescDev din, int32_t* state, ListDev ld, int32_t* exflag,
                           const double* __restrict__ partials, const int32_t* __restrict__ newb, DescDev dout,
                           double* volume, double* area, int mode) {
  const bool coarsen = mode & kFinCoarsen, do_state = mode & kFinState, do_bounds = mode & kFinBounds;
  for (int g = 1 + blockIdx.x * blockDim.x + threadIdx.x; g <= sp.N; g += gridDim.x * blockDim.x) {
    const int s = state[g];
    if (s == kVanished) {
      if (do_state && !coarsen) state[g] = kDeleted;
      continue;
    }
    if (s == kDoomed) {
      if (do_state) {
        ld.sel[g] ^= 1;
        exflag[g] = 0;
        state[g] = kVanished;
      }
      continue;
    }
    if (s != kAlive) continue;
    if (do_state) {
      if (!coarsen) ld.sel[g] ^= 1;
      const int ex = exflag[g];
      exflag[g] = 0;
      if (!ex) {
        state[g] = kVanished;
        continue;
      }
      const int pos = P.grain_pos[g];
      int c = 0;
      while (c + 1 < kClasses && pos >= P.cls_start[c + 1]) ++c;
      const int idx = pos - P.cls_start[c];
      const int first = P.pre[kQLayers][P.cls_start[c] + c + idx];
      const int n = box_n(din.bounds, g);
      const double* pp = partials + 4 * (P.layer_base[c] + first);
      Acc va{pp[0], pp[1]}, aa{pp[2], pp[3]};
      for (int l = 1; l < n; ++l) {
        va.merge(pp[4 * l], pp[4 * l + 1]);
        aa.merge(pp[4 * l + 2], pp[4 * l + 3]);
      }
      const double h = sp.h;
      volume[g] = fabs(va.s + va.c) * h * h * h;
      area[g] = (aa.s + aa.c) * h * h;
    }
    if (!do_bounds) continue;
    const int32_t* nb = newb + 6 * g;
    // Before the hull: a grain without a voxel >= 0 (empty set-comparison
    // bounds) has no hull and vanishes; it is left out of the output plan.
    if (!do_state && (nb[0] > nb[3] || nb[1] > nb[4] || nb[2] > nb[5])) {
      state[g] = kDoomed;
      continue;
    }
    int bb[6] = {nb[0] - sp.gb, nb[1] - sp.gb, nb[2] - sp.gb, nb[3] + sp.gb, nb[4] + sp.gb, nb[5] + sp.gb};
    if (coarsen) {
      for (int a = 0; a < 6; ++a) bb[a] = nb[a];
    } else {
      for (int a = 0; a < 3; ++a) {
        if (bb[a] < 0) bb[a] = 0;
        if (bb[a + 3] >= sp.ngp) bb[a + 3] = sp.ngp - 1;
      }
    }
    cube_bounds(bb, sp.ngp);
    for (int a = 0; a < 6; ++a) dout.bounds[6 * g + a] = bb[a];
  }
}

}  // namespace

void upload_mc_tables() {
  uint64_t tri[256];
  for (int c = 0; c < 256; ++c) {
    uint64_t row = ~0ull;
    const char* t = kTriCases[c];
    for (int i = 0; t[i]; ++i) {
      const char ch = t[i];
      const uint64_t e = (uint64_t)((ch >= '0' && ch <= '9') ? ch - '0' : ch - 'a' + 10);
      row = (row & ~(15ull << (4 * i))) | e << (4 * i);
    }
    tri[c] = row;
  }
  (void)hipMemcpyToSymbol(HIP_SYMBOL(c_tri), tri, sizeof(tri));
}

// Clears the topology tables of the grains the hull does not walk (it writes
// whole tables), and the triangle records, before a hull with topology on.
__global__ __launch_bounds__(256) void k_topo_clear(SimParams sp, PlanDev P, TopoDev topo) {
  if (topo.corr && blockIdx.x == 0 && threadIdx.x == 0) *topo.raw_n = 0ull;
  for (int g = blockIdx.x; g <= sp.N; g += gridDim.x) {
    if (g > 0 && P.grain_pos[g] >= 0) continue;
    const int64_t b = (int64_t)g * kTopoCap, jb = (int64_t)g * kJuncCap;
    for (int i = threadIdx.x; i < kTopoCap; i += 256) {
      topo.key[b + i] = -1;
      topo.ord[b + i] = INT_MAX;
    }
    for (int i = threadIdx.x; i < kJuncCap; i += 256) {
      topo.jkey[jb + i] = 0ull;
      topo.jcnt[jb + i] = 0;
      if (topo.corr) topo.jord[jb + i] = INT_MAX;
      topo.jpos[3 * (jb + i)] = 0ull;
      topo.jpos[3 * (jb + i) + 1] = 0ull;
      topo.jpos[3 * (jb + i) + 2] = 0ull;
      topo.jarea[jb + i] = 0.0;
    }
  }
}

void launch_topo_clear(const Launch& L, const SimParams& sp, const PlanDev& P, const TopoDev& topo) {
  hipLaunchKernelGGL(k_topo_clear, dim3(std::min(sp.N + 1, L.grid)), dim3(256), 0, L.stream, sp, P, topo);
}

template <class T>
void hull_all(const Launch& L, const SimParams& sp, const PlanDev& P, const DescDev& din, int32_t* exflag,
              double* partials, const IdlDev& il, const TopoDev& topo, int32_t* err) {
  if (!topo.on) {
    const int64_t need = ((int64_t)sp.N * kMaxN / (4 * kHullRun) + kXcds) / kXcds * kXcds;
    const int grid = (int)std::min<int64_t>((int64_t)L.cus * kGridPerCU, need);
    hipLaunchKernelGGL(k_hull<T>, dim3(grid), dim3(256), 0, L.stream, P, din, exflag, partials);
    return;
  }
  const int grid = std::min(sp.N, L.cus * kGridPerCU);
  hipLaunchKernelGGL((k_hull_topo<T, 48>), dim3(grid), dim3(64 * kTopoWaves), 0, L.stream, P, 0, 2, din, exflag,
                     partials, il, topo, err);
  hipLaunchKernelGGL((k_hull_topo<T, 96>), dim3(grid), dim3(64 * kTopoWaves), 0, L.stream, P, 2, 4, din, exflag,
                     partials, il, topo, err);
}

void launch_hull(const Launch& L, const SimParams& sp, const PlanDev& P, const DescDev& din, int32_t* exflag,
                 double* partials, const IdlDev& il, const TopoDev& topo, int32_t* err, bool fp32) {
  if (fp32) hull_all<float>(L, sp, P, din, exflag, partials, il, topo, err);
  else hull_all<double>(L, sp, P, din, exflag, partials, il, topo, err);
}

void launch_finalize(const Launch& L, const SimParams& sp, const PlanDev& P, int32_t* state, const ListDev& ld,
                     int32_t* exflag, const double* partials, const int32_t* newb, const DescDev& din,
                     const DescDev& dout, double* volume, double* area, int mode) {
  int blocks = (sp.N + 255) / 256;
  hipLaunchKernelGGL(k_finalize, dim3(blocks), dim3(256), 0, L.stream, sp, P, din, state, ld, exflag, partials,
                     newb, dout, volume, area, mode);
}

}  // namespace gg
