// Convolution correction: the correction branch of LSbox::executeConvolution
// (src/box.cpp:428-536) on the interfacial elements of every grain's last hull
// (GrainHull::computeGrainBoundaryElements / subDivideTrianglesToInterfacialElements
// / computeJunctionPosition with mergeJunction, src/grainHull.cpp:187-274,
// 483-531; element constructors src/InterfacialElement.cpp:52-404) found with
// GrainHull::projectPointToGrainBoundary (src/grainHull.cpp:570-660).
//
// After each hull that ran with the correction on (level set, grid coarsening):
//   k_elements     one workgroup per grain: the hull's distinct cut-cell id
//                  lists (the grain's junction table, with each list's first
//                  appearance) in first-appearance order become elements by
//                  size (2 grains: boundary, 3: triple line, 4: quadruple
//                  junction, else high-order junction) with their energy and
//                  mobility; quadruple junctions closer than 2 voxels merge as
//                  mergeJunction merges them; elements are laid out in the order
//                  the projection visits them (high-order junctions, quadruple
//                  junctions, triple lines, boundaries) with the start of each
//                  element's barycenters, and the grain reserves its range of
//                  the barycenter array.
//   k_tri_scatter  every triangle record of the hull goes to its element's
//                  range (the order inside an element does not matter: all its
//                  barycenters carry the element's weights).
//   k_slots        one workgroup per grain: per slot of the grain's hull-id table,
//                  the barycenters that can be nearest to some voxel of the new
//                  output box, as rows of the search's matrix product.
// After each convolution:
//   k_correct      one workgroup per (grain, run of z-layers) of the output box:
//                  the band voxels (|phi_in| < delta) are queued with the slot of
//                  their IDLocal id in the grain's hull-id table and grouped by
//                  slot (counting sort in LDS); a wavefront takes up to 128 of
//                  one slot and finds, for each, the element of the first nearest
//                  barycenter in projection order (squared distance, strict '<')
//                  among the elements that border its
//                  id; then phi_out = phi_in +
//                  (phi_out - phi_in) * w_energy * w_mobility and, with stored
//                  energies on, minus (SEE_self - SEE_id) * w_mobility * dt /
//                  TimeSlope^2.  The weights are GBInfo's as get_GBInfo hands
//                  them over: w_energy = the element's mobility, w_mobility =
//                  its energy (src/InterfacialElement.h:22-31, 70-72).
//
// FP64 arithmetic in the reference's operation order; only which barycenters need
// comparing in FP64 is found by a BF16-piece product with an error bound (below),
// so every result is FP64's.  The junction positions (used only for the merge test) are the hull's barycenter sums
// (fixed point, summed in any order to the same value) over their count.
#include "gg_internal.h"
#include "gg_runs.h"

namespace gg {
namespace {

constexpr int kEW = 256;                           // threads of an element-build workgroup
constexpr int kRec = kJuncCap + kJuncCap / 2;      // lists + high-order junctions made by merging
constexpr int kTopoCapBitsC = 6;
static_assert((1 << kTopoCapBitsC) == kTopoCap, "grain topology table size");
// most workgroups per CU of a correction launch: 16 times what is resident, for
// balance; each costs its start (correction per step at 20000 grains with 24:
// 16.1, 32: 16.3, 64: 15.8, 128: 15.9, 256: 16.1 ms)
constexpr int kCorrGridPerCU = 64;

enum { kClsGB = 0, kClsTL = 1, kClsQJ = 2, kClsHJ = 3 };

__device__ inline double pair_gam(const CorrDev& cd, int N, unsigned a, unsigned b) {
  return cd.aniso ? cd.gam[(int64_t)a * (N + 1) + b] : 1.0;
}
__device__ inline double pair_mob(const CorrDev& cd, int N, unsigned a, unsigned b) {
  return cd.aniso ? cd.mob[(int64_t)a * (N + 1) + b] : 1.0;
}

// TripleLine::computeMobility / computeEnergy (src/InterfacialElement.cpp:118-164)
__device__ inline void triple_line(const CorrDev& cd, int N, unsigned me, unsigned n0, unsigned n1, double& energy,
                                   double& mobility) {
  double avg = 0;
  avg += pair_mob(cd, N, me, n0);
  avg += pair_mob(cd, N, n0, n1);
  avg += pair_mob(cd, N, me, n1);
  avg /= 3;
  mobility = 1. / (cd.tl_inv + 1. / avg);
  const double g0 = pair_gam(cd, N, me, n0), g1 = pair_gam(cd, N, n0, n1), g2 = pair_gam(cd, N, me, n1);
  double sigma = g0 - g1 + g2;
  if (sigma < 0.01) sigma = 0.01;
  if (sigma > 1.0) sigma = 1.0;
  energy = sigma;
}

__global__ __launch_bounds__(kEW) void k_elements(SimParams sp, const int32_t* __restrict__ state, TopoDev topo,
                                                  CorrDev cd, int32_t* err) {
  __shared__ int s_key[kTopoCap];
  __shared__ int s_nl, s_self, s_E;
  __shared__ short s_ls[kJuncCap];      // junction-table slot of each list (compacted)
  __shared__ int s_lo[kJuncCap];        // its first appearance
  __shared__ short s_sorted[kJuncCap];  // compacted index of the r-th list in first-appearance order
  // records: the lists in first-appearance order (index r < nl), then the
  // high-order junctions made by merging
  __shared__ unsigned long long s_em[kRec];  // neighbour set (slots of the grain's hull-id table)
  __shared__ double s_en[kRec], s_mo[kRec];
  __shared__ double s_sx[kRec], s_sy[kRec], s_sz[kRec];  // barycenter sums (junctions)
  __shared__ int s_cnt[kRec];
  __shared__ signed char s_cls[kRec];
  __shared__ short s_red[kRec];   // record it was merged into (-1: none)
  __shared__ short s_elem[kRec];  // element index of a record that is an element
  __shared__ short s_hj[kRec], s_qj[kJuncCap];
  __shared__ short s_ord[kJuncCap];  // element -> record
  const int N = sp.N;
  const int tid = threadIdx.x;
  if (blockIdx.x == 0 && tid == 0) *cd.ready = 1;
  for (int g = 1 + blockIdx.x; g <= N; g += gridDim.x) {
    if (state[g] != kAlive) {
      if (tid == 0) cd.ecount[g] = 0;
      continue;
    }
    const int64_t jb = (int64_t)g * kJuncCap;
    if (tid < kTopoCap) s_key[tid] = topo.key[(int64_t)g * kTopoCap + tid];
    if (tid == 0) {
      s_nl = 0;
      s_self = -1;
    }
    __syncthreads();
    if (tid < kTopoCap && s_key[tid] == g) s_self = tid;
    for (int i = tid; i < kJuncCap; i += kEW) {
      if (topo.jkey[jb + i] != 0ull) {
        const int q = atomicAdd(&s_nl, 1);
        s_ls[q] = (short)i;
        s_lo[q] = topo.jord[jb + i];
      }
    }
    __syncthreads();
    const int nl = s_nl;
    for (int q = tid; q < nl; q += kEW) {
      const int o = s_lo[q];
      int r = 0;
      for (int j = 0; j < nl; ++j) r += (s_lo[j] < o) | ((s_lo[j] == o) & (j < q));
      s_sorted[r] = (short)q;
    }
    __syncthreads();
    // each list as an element: class by its number of grains, neighbour ids
    // ascending, energy and mobility (src/InterfacialElement.cpp:52-404)
    const unsigned me = (unsigned)g;
    for (int r = tid; r < nl; r += kEW) {
      const int slot = s_ls[s_sorted[r]];
      const unsigned long long m = topo.jkey[jb + slot];
      const int self = s_self;
      const unsigned long long nbm = self >= 0 ? m & ~(1ull << self) : m;
      const int size = __popcll(m);
      unsigned o[3] = {0u, 0u, 0u};
      int no = 0;
      if (size >= 2 && size <= 4) {
        for (unsigned long long t = nbm; t && no < 3; t &= t - 1) {
          unsigned v = (unsigned)s_key[__builtin_ctzll(t)];
          int p = no++;
          while (p > 0 && o[p - 1] > v) {
            o[p] = o[p - 1];
            --p;
          }
          o[p] = v;
        }
      }
      int cls;
      double en = 1.0, mo = 1.0;
      if (size == 2 && no == 1) {  // GrainBoundary
        cls = kClsGB;
        mo = pair_mob(cd, N, me, o[0]);
        en = pair_gam(cd, N, me, o[0]);
      } else if (size == 3 && no == 2) {  // TripleLine
        cls = kClsTL;
        triple_line(cd, N, me, o[0], o[1], en, mo);
      } else if (size == 4 && no == 3) {  // QuadrupleJunction: means over its triple lines
        cls = kClsQJ;
        double e1, m1, e2, m2, e3, m3;
        triple_line(cd, N, me, o[0], o[1], e1, m1);
        triple_line(cd, N, me, o[1], o[2], e2, m2);
        triple_line(cd, N, me, o[0], o[2], e3, m3);
        mo = (m1 + m2 + m3) / 3.0;
        en = (e1 + e2 + e3) / 3.0;
      } else {  // HighOrderJunction (other sizes)
        cls = kClsHJ;
      }
      s_em[r] = nbm;
      s_cls[r] = (signed char)cls;
      s_en[r] = en;
      s_mo[r] = mo;
      s_cnt[r] = topo.jcnt[jb + slot];
      s_sx[r] = (double)(long long)topo.jpos[3 * (jb + slot)] / kPosScale;
      s_sy[r] = (double)(long long)topo.jpos[3 * (jb + slot) + 1] / kPosScale;
      s_sz[r] = (double)(long long)topo.jpos[3 * (jb + slot) + 2] / kPosScale;
      s_red[r] = -1;
    }
    __syncthreads();
    // the merges and the order, by the first wavefront: every scan of a list for
    // the first near junction takes 64 of its entries at a time (one lane
    // testing one pair after the other: k_elements took 5.8 ms per step at 20000
    // grains, 82 % of it waiting; 1.0 ms this way); a merged entry is marked, not closed up
    if (tid < 64) {
      const int lane = tid;
      const unsigned long long below = (1ull << lane) - 1ull;
      auto settle = [] {  // what one lane wrote, before any lane reads it
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      };
      int nh = 0, nq = 0, nrec = nl;
      for (int r0 = 0; r0 < nl; r0 += 64) {
        const int c = r0 + lane < nl ? (int)s_cls[r0 + lane] : -1;
        const unsigned long long mh = __ballot(c == kClsHJ), mq = __ballot(c == kClsQJ);
        if (c == kClsHJ) s_hj[nh + __popcll(mh & below)] = (short)(r0 + lane);
        if (c == kClsQJ) s_qj[nq + __popcll(mq & below)] = (short)(r0 + lane);
        nh += __popcll(mh);
        nq += __popcll(mq);
      }
      settle();
      // first entry of list[lo, n) whose junction lies within 2 of record a's
      // (position = mean barycenter, computePosition), -1: none
      auto first_near = [&](int a, const short* list, int lo, int n) {
        const double na = (double)s_cnt[a];
        const double ax = s_sx[a] / na, ay = s_sy[a] / na, az = s_sz[a] / na;
        for (int j0 = lo; j0 < n; j0 += 64) {
          const int b = j0 + lane < n ? (int)list[j0 + lane] : -1;
          bool hit = false;
          if (b >= 0) {
            const double nb = (double)s_cnt[b];
            const double dx = ax - s_sx[b] / nb, dy = ay - s_sy[b] / nb, dz = az - s_sz[b] / nb;
            hit = sqrt(dx * dx + dy * dy + dz * dz) < 2;
          }
          const unsigned long long m = __ballot(hit);
          if (m) return j0 + (int)__builtin_ctzll(m);
        }
        return -1;
      };
      auto absorb = [&](int h, short* list, int at) {  // mergeWith: the entry's barycenters and ids join h
        if (lane == 0) {
          const int b = list[at];
          s_cnt[h] += s_cnt[b];
          s_sx[h] += s_sx[b];
          s_sy[h] += s_sy[b];
          s_sz[h] += s_sz[b];
          s_em[h] |= s_em[b];
          s_en[h] = s_mo[h] = 1.0;
          s_red[b] = (short)h;
          list[at] = -1;
        }
        settle();
      };
      // mergeJunction (src/grainHull.cpp:483-531)
      for (int i = 0; i < nq; ++i) {
        const int A = s_qj[i];
        if (A < 0) continue;
        const int j = first_near(A, s_qj, i + 1, nq);
        if (j < 0) continue;
        // HighOrderJunction(A, B): A's ids (B adds only ids A has), A's then B's
        // barycenters
        const int h = nrec++;
        if (lane == 0) {
          const int B = s_qj[j];
          s_em[h] = s_em[A];
          s_cnt[h] = s_cnt[A] + s_cnt[B];
          s_sx[h] = s_sx[A] + s_sx[B];
          s_sy[h] = s_sy[A] + s_sy[B];
          s_sz[h] = s_sz[A] + s_sz[B];
          s_en[h] = s_mo[h] = 1.0;
          s_cls[h] = kClsHJ;
          s_red[h] = -1;
          s_red[A] = s_red[B] = (short)h;
          s_qj[i] = s_qj[j] = -1;
          s_hj[nh] = (short)h;
        }
        ++nh;
        settle();
      }
      for (int k = 0; k < nh; ++k) {
        const int h = s_hj[k];
        for (int i = 0; (i = first_near(h, s_qj, i, nq)) >= 0; ++i) absorb(h, s_qj, i);
      }
      for (int i = 0; i < nh; ++i) {
        const int h = s_hj[i];
        if (h < 0) continue;
        for (int k = i + 1; (k = first_near(h, s_hj, k, nh)) >= 0; ++k) absorb(h, s_hj, k);
      }
      // projection order: high-order junctions, quadruple junctions, triple
      // lines, boundaries
      int E = 0;
      auto append = [&](bool take, int rec) {
        const unsigned long long m = __ballot(take);
        if (take) s_ord[E + __popcll(m & below)] = (short)rec;
        E += __popcll(m);
      };
      auto append_list = [&](const short* list, int n) {
        for (int t0 = 0; t0 < n; t0 += 64) {
          const int rec = t0 + lane < n ? (int)list[t0 + lane] : -1;
          append(rec >= 0, rec);
        }
      };
      auto append_class = [&](int cls) {
        for (int r0 = 0; r0 < nl; r0 += 64) append(r0 + lane < nl && s_cls[min(r0 + lane, nl - 1)] == cls, r0 + lane);
      };
      append_list(s_hj, nh);
      const int eh = E;
      append_list(s_qj, nq);
      const int eq = E;
      append_class(kClsTL);
      const int et = E;
      append_class(kClsGB);
      settle();
      long long acc = 0;
      int32_t* ef = cd.efirst + (int64_t)g * (kElemCap + 1);
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        const int rec = e < E ? (int)s_ord[e] : 0;
        const long long c = e < E ? (long long)s_cnt[rec] : 0ll;
        long long incl = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const long long u = __shfl_up(incl, d, 64);
          if (lane >= d) incl += u;
        }
        if (e < E) {
          s_elem[rec] = (short)e;
          ef[e] = (int32_t)(acc + incl - c);
        }
        acc += __shfl(incl, 63, 64);
      }
      if (lane == 0) {
        ef[E] = (int32_t)acc;
        const unsigned long long tb = atomicAdd(cd.tri_n, (unsigned long long)acc);
        if (tb + (unsigned long long)acc > (unsigned long long)cd.tri_cap) atomicOr(err, kErrTri);
        cd.tbase[g] = (int64_t)tb;
        cd.ecount[g] = E;
        cd.eclass[4 * g] = eh;
        cd.eclass[4 * g + 1] = eq - eh;
        cd.eclass[4 * g + 2] = et - eq;
        s_E = E;
      }
    }
    __syncthreads();
    const int E = s_E;
    const int64_t eb = (int64_t)g * kElemCap;
    for (int e = tid; e < E; e += kEW) {
      const int rec = s_ord[e];
      cd.emask[eb + e] = s_em[rec];
      cd.energy[eb + e] = s_en[rec];
      cd.mobility[eb + e] = s_mo[rec];
      cd.ecur[eb + e] = 0;
      const double n = (double)s_cnt[rec];
      const bool junction = s_cls[rec] >= kClsQJ;
      cd.epos[3 * (eb + e)] = junction ? s_sx[rec] / n : 0.0;
      cd.epos[3 * (eb + e) + 1] = junction ? s_sy[rec] / n : 0.0;
      cd.epos[3 * (eb + e) + 2] = junction ? s_sz[rec] / n : 0.0;
    }
    for (int r = tid; r < nl; r += kEW) {
      int rec = r;
      while (s_red[rec] >= 0) rec = s_red[rec];
      cd.slot_elem[jb + s_ls[s_sorted[r]]] = s_elem[rec];
    }
    __syncthreads();  // the LDS tables are refilled for the next grain
  }
}

// The pools' fill counters (a kernel, so that a captured step graph
// holds no memset node).
__global__ void k_clear_counters(unsigned long long* tri_n, int* row_n) {
  if (threadIdx.x == 0) *tri_n = 0ull;
  if (threadIdx.x == 1) *row_n = 0;
}

// Every triangle record of the last hull into its element's barycenter range.
// A grain's records are consecutive in the pool, one wavefront of its hull
// workgroup after the other (those a full cell queue forced out lie apart), so a
// wavefront's 64 records here name few elements: it reserves one run per (grain,
// element) among them.
__global__ __launch_bounds__(256) void k_tri_scatter(TopoDev topo, CorrDev cd) {
  unsigned long long n = *topo.raw_n;
  if (n > (unsigned long long)topo.raw_cap) n = (unsigned long long)topo.raw_cap;
  const int lane = threadIdx.x & 63;
  for (unsigned long long base = blockIdx.x * 256ull; base < n; base += (unsigned long long)gridDim.x * 256ull) {
    const unsigned long long r = base + threadIdx.x;
    bool valid = r < n;
    TriRec t{};
    int e = -1;
    unsigned key = 0u;
    if (valid) {
      t = topo.raw[r];
      e = cd.slot_elem[(int64_t)t.g * kJuncCap + t.slot];
      valid = (unsigned)e < (unsigned)cd.ecount[t.g];  // false only after a table overflow (device error set)
      key = (unsigned)t.g * (unsigned)kElemCap + (unsigned)e;
    }
    // one round per distinct (grain, element) among the wavefront's records;
    // then every leader reserves its run in the same instruction (1.5 ms per
    // step at 20000 grains; an add in every round, one after the other: 1.75)
    int lead = lane, at = 0, run = 0;
    bool done = !valid;
    for (;;) {
      const unsigned long long pend = __ballot(!done);
      if (pend == 0ull) break;
      const int leader = __ffsll((long long)pend) - 1;
      const unsigned k0 = __shfl(key, leader);
      const bool mine = !done && key == k0;
      const unsigned long long m = __ballot(mine);
      if (mine) {
        lead = leader;
        at = __popcll(m & ((1ull << lane) - 1ull));
        run = __popcll(m);
        done = true;
      }
    }
    int b0 = 0;
    if (valid && lane == lead) b0 = atomicAdd(&cd.ecur[key], run);
    const int64_t pos = __shfl(b0, lead) + at;
    if (valid) {
      const int64_t q = cd.tbase[t.g] + cd.efirst[(int64_t)t.g * (kElemCap + 1) + e] + pos;
      if (q < cd.tri_cap) {
        cd.tri[3 * q] = t.x;
        cd.tri[3 * q + 1] = t.y;
        cd.tri[3 * q + 2] = t.z;
      }
    }
  }
}

// Nearest element of a band voxel p among the elements that border its id, as a
// filter on the matrix cores with an FP64 decision.
//
// With q' = q - org, p' = p - (org.y, org.x, org.z) and D = org - (org.y,
// org.x, org.z) (the point's row and column stand for x and y, as in the
// reference), |q - p|^2 is W = R - 2 p'.q' plus terms that do not depend on q,
// where R = |q'|^2 + 2 q'.D.  W of 32 barycenters against 32 voxels is one
// v_mfma_f32_32x32x16_bf16: p' is a small integer (exact in BF16) and -2q' and
// R are three BF16 pieces each (store_row), so a product of a piece and p' is
// exact and the filter's error is the FP32 accumulation's.  The filter keeps,
// per voxel, the smallest W, its element, and the smallest W of any other
// element.  Where the two are closer than the error bound, and only there, the
// wavefront searches the bordering elements' barycenters in FP64 for the first
// nearest one in projection order, so the chosen element is always the
// reference's.
//
// Bound: with rho >= |q'| over the grain's rows, the terms of W sum to at most
// S = rho^2 + 2 rho (|D| + |p'|) in magnitude, their pieces to 1.01 S.  Of the
// instruction's adder nothing is assumed but that each rounding is within one
// unit of the last place, 2^-23 of a value that the pieces' sum bounds, so
// truncation is allowed and any order of the adds.  12 products are added: 12
// roundings, 24 x 2^-24 of 1.01 S, and the pieces' remainders are 2^-26 of a
// term: 24.5 x 2^-24, and kFilterEps is 26 x 2^-24 (measured on random rows and
// columns of every box size: at most 2.2 x 2^-24 S).  FP64 rounds a squared distance below 1e7 to 6e-9, so a gap also has to
// pass kDecided: the reference's rounded comparison then agrees with the exact
// one.  (Correction per step with 16, enough for an adder that rounds to nearest,
// 25 and 32 x 2^-24: 1000 grains 1.07, 1.09, 1.12 ms; 20000 15.5, 15.7, 15.8.)
//
// What bounds it: at 20000 grains (5.8e8 band voxels per step) the searches hold
// 14 groups of 8 rows on average (75 before k_slots leaves out the ones that
// cannot be nearest).  The FP64 search over boxed chunks that this replaced took
// 146 ms per step (and its chunk boxes 3.4); k_correct took 24.5 in this form,
// with fewer workgroups and runs of 8 layers instead of 4 for n <= 32 (fuller
// searches) 17.9, and with the runs dealt to the XCDs (below) 15.5; k_slots takes
// 2.5.
// Of the 15.5 ms (15.8 when this was taken), queueing and output are 8.1, the products and the minima behind
// them (vector) 6.2, the FP64 decisions 1.5 (4000 grains: 0.6, 0.8, 0.5 of 1.9;
// 343 in FP64: 0.08, 0.18, 0.15 of 0.42), at four wavefronts per SIMD (128
// registers; three, when it took 24.5: 28.9).  128 voxels per search read each
// row once for four products; 64 took 4 % longer.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr float kFilterEps = 26.0f / 16777216.0f;
constexpr float kDecided = 1e-6f;                 // a gap that FP64 rounding cannot turn round
constexpr float kNone = 3e38f;                    // above every filter value
// Voxels of 64 to decide from which on each lane searches for its own.  Correction
// per step at 4000 grains, 20000, 343 in FP64: with 12 2.00, 15.9, 0.47 ms; 20
// 1.94, 15.7, 0.43; 32 1.98, 15.8, 0.40; 4 2.23, 16.4, 0.60.
constexpr int kManyExact = 24;
constexpr int kTake = 128;  // voxels of a wavefront's search: each row is read once for four products

// A barycenter as a row of the filter: -2q' (three BF16 pieces per axis) and R
// (three pieces), 16 values with 4 spare; the columns repeat p' and 1 to match.
// Each piece is the nearest BF16 of what the pieces before it leave, so three
// of them hold 24 bits.
__device__ inline void store_row(uint16_t* __restrict__ row, double qx, double qy, double qz, double r) {
  const double v[4] = {-2.0 * qx, -2.0 * qy, -2.0 * qz, r};
  alignas(16) uint16_t w[kRowLen] = {};
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    double rest = v[a];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const __bf16 piece = (__bf16)(float)rest;
      rest -= (double)(float)piece;
      w[3 * a + k] = __builtin_bit_cast(uint16_t, piece);
    }
  }
  const uint4* s = (const uint4*)w;
  ((uint4*)row)[0] = s[0];
  ((uint4*)row)[1] = s[1];
}

// The filter's rows of every alive grain: per hull-id slot, element by element,
// the barycenters that can be nearest to some voxel of the grain's output box
// (the box the next convolution corrects).  Against the slot's nearest one to
// the box centre, q0, a barycenter q is left out when W(q) - W(q0) =
// R - R0 - 2 p'.(q' - q0') is positive for every p' of the box, |p'_a| <= half:
// because the point's row and column are swapped, most grains see their
// barycenters from far off the domain's diagonal plane x = y, and few remain.
// One workgroup per grain, one wavefront per slot.
__global__ __launch_bounds__(256) void k_slots(SimParams sp, const int32_t* __restrict__ state, DescDev dout,
                                               TopoDev topo, CorrDev cd) {
  __shared__ int s_key[kTopoCap];
  __shared__ unsigned long long s_em[kElemCap];
  __shared__ int s_ef[kElemCap + 1];
  __shared__ int s_rho;
  __shared__ double s_q0[kTopoCap][4];  // per slot: its nearest barycenter to the box centre, and R
  __shared__ int s_groups[kTopoCap], s_first[kTopoCap];
  static_assert(kTopoCap == 64, "one lane per slot");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int g = 1 + blockIdx.x; g <= sp.N; g += gridDim.x) {
    if (state[g] != kAlive) continue;
    const int64_t tb = cd.tbase[g];
    int E = cd.ecount[g];
    if (tb + cd.efirst[(int64_t)g * (kElemCap + 1) + E] > cd.tri_cap) E = 0;  // (the device error is set)
    for (int i = tid; i < kTopoCap; i += 256) s_key[i] = topo.key[(int64_t)g * kTopoCap + i];
    for (int e = tid; e < E; e += 256) s_em[e] = cd.emask[(int64_t)g * kElemCap + e];
    for (int e = tid; e <= E; e += 256) s_ef[e] = cd.efirst[(int64_t)g * (kElemCap + 1) + e];
    if (tid == 0) s_rho = 0;
    __syncthreads();
    const int32_t* b = dout.bounds + 6 * g;
    const int n = b[3] - b[0];
    const int ox = b[0] + n / 2, oy = b[1] + n / 2, oz = b[2] + n / 2;
    const double dd2 = 2.0 * (double)(ox - oy), half2 = 2.0 * (double)(n / 2);
    const double* __restrict__ tri = cd.tri + 3 * tb;
    float rho2 = 0.f;
    // f(r, valid): 64 barycenters (r relative to the grain's first) of the
    // slot's elements per call, element by element; after(e): past the
    // element's last call
    auto over = [&](int slot, auto f, auto after) {
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int el = e0 + lane;
        unsigned long long m = __ballot(el < E && ((s_em[el < E ? el : 0] >> slot) & 1ull));
        for (; m; m &= m - 1) {
          const int e = e0 + (int)__builtin_ctzll(m);
          const int r0 = s_ef[e], r1 = s_ef[e + 1];
          for (int r = r0; r < r1; r += 64) f(r + lane, r + lane < r1);
          after(e);
        }
      }
    };
    auto load = [&](int r, double& qx, double& qy, double& qz) {
      const double* q = tri + 3 * (int64_t)r;
      qx = q[0] - ox;
      qy = q[1] - oy;
      qz = q[2] - oz;
      return qx * qx + qy * qy + qz * qz + dd2 * (qx - qy);
    };
    // 1e-3: far above the rounding of either side (and of the FP64 search)
    auto keep = [&](const double* q0, double R, double qx, double qy, double qz) {
      return (R - q0[3]) - half2 * (fabs(qx - q0[0]) + fabs(qy - q0[1]) + fabs(qz - q0[2])) <= 1e-3;
    };
    for (int slot = wv; slot < kTopoCap; slot += 4) {
      if (s_key[slot] == -1 || s_key[slot] == g) {
        if (lane == 0) s_groups[slot] = 0;
        continue;
      }
      double R0 = 1e300, x0 = 0, y0 = 0, z0 = 0;
      over(
          slot,
          [&](int r, bool valid) {
            if (!valid) return;
            double qx, qy, qz;
            const double R = load(r, qx, qy, qz);
            if (R < R0) {
              R0 = R;
              x0 = qx;
              y0 = qy;
              z0 = qz;
            }
          },
          [](int) {});
      double best = R0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) best = fmin(best, __shfl_xor(best, o));
      const int src = (int)__builtin_ctzll(__ballot(R0 == best));
      const double q0[4] = {__shfl(x0, src), __shfl(y0, src), __shfl(z0, src), best};
      if (lane < 4) s_q0[slot][lane] = lane == 0 ? q0[0] : lane == 1 ? q0[1] : lane == 2 ? q0[2] : q0[3];
      int groups = 0, cnt = 0;
      over(
          slot,
          [&](int r, bool valid) {
            double qx, qy, qz;
            const double R = load(valid ? r : 0, qx, qy, qz);
            cnt += __popcll(__ballot(valid && keep(q0, R, qx, qy, qz)));
          },
          [&](int) {
            groups += (cnt + kChunk - 1) / kChunk;
            cnt = 0;
          });
      if (lane == 0) s_groups[slot] = groups;
    }
    __syncthreads();
    // the grain's groups are reserved with one add (2.5 ms per step at 20000
    // grains; one per slot, 2.8e5 on one counter: 3.7)
    if (wv == 0) {
      const int groups = s_groups[lane];
      int incl = groups;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d, 64);
        if (lane >= d) incl += u;
      }
      const int all = __builtin_amdgcn_readlane(incl, 63);
      int first = 0;
      if (lane == 0 && all > 0) first = atomicAdd(cd.row_n, all);
      first = __builtin_amdgcn_readfirstlane(first) + incl - groups;
      // no room: the slot is searched without a list
      const int2 sl = groups == 0 ? make_int2(0, 0)
                      : first > cd.row_groups - groups ? make_int2(0, -1) : make_int2(first, groups);
      cd.slist[(int64_t)g * kTopoCap + lane] = sl;
      s_first[lane] = sl.y > 0 ? sl.x : -1;
    }
    __syncthreads();
    for (int slot = wv; slot < kTopoCap; slot += 4) {
      int cur = s_first[slot], cnt = 0;
      if (cur < 0) continue;
      const double q0[4] = {s_q0[slot][0], s_q0[slot][1], s_q0[slot][2], s_q0[slot][3]};
      over(
          slot,
          [&](int r, bool valid) {
            double qx, qy, qz;
            const double R = load(valid ? r : 0, qx, qy, qz);
            const bool k = valid && keep(q0, R, qx, qy, qz);
            const unsigned long long m = __ballot(k);
            if (k) {
              const int pos = cnt + __popcll(m & ((1ull << lane) - 1ull));
              const int64_t row = (int64_t)cur * kChunk + pos;
              store_row(cd.rows + kRowLen * row, qx, qy, qz, R);
              cd.rsrc[row] = r;
              rho2 = fmaxf(rho2, (float)(qx * qx + qy * qy + qz * qz));
            }
            cnt += __popcll(m);
          },
          [&](int e) {
            const int ng = (cnt + kChunk - 1) / kChunk;
            if (cnt + lane < ng * kChunk) {
              const int64_t row = (int64_t)cur * kChunk + cnt + lane;
              store_row(cd.rows + kRowLen * row, 0.0, 0.0, 0.0, kFarPoint);
              cd.rsrc[row] = -1;
            }
            for (int t = lane; t < ng; t += 64) cd.tags[cur + t] = (uint16_t)(e | (t == ng - 1 ? kTagEnd : 0));
            cur += ng;
            cnt = 0;
          });
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) rho2 = fmaxf(rho2, __shfl_xor(rho2, o));
    if (lane == 0) atomicMax(&s_rho, __float_as_int(1.0001f * sqrtf(rho2)));  // non-negative: ordered as integers
    __syncthreads();
    if (tid == 0) {
      cd.org[g] = make_int4(ox, oy, oz, s_rho);
      cd.sbox[g] = make_int4(b[0], b[1], b[2], n);
    }
    __syncthreads();  // the tables are refilled for the next grain
  }
}

// The filter's values are finite, so its minima need no handling of NaN (which
// would be an extra instruction per operand).
#pragma float_control(precise, off, push)
__device__ inline float min4(const v16f& d, int u, float run) {
  return fminf(fminf(fminf(fminf(run, d[4 * u]), d[4 * u + 1]), d[4 * u + 2]), d[4 * u + 3]);
}
__device__ inline float min16(const v16f& d, float run) {
  float m = run;
#pragma unroll
  for (int i = 0; i < 16; i += 2) m = fminf(fminf(m, d[i]), d[i + 1]);
  return m;
}

// Two smallest filter values over different elements: m1 of element e1, m2 of
// any other.
struct Near {
  float m1, m2;
  int e1;
  __device__ void add(float m, int e) {  // element e's smallest value; elements come one by one
    m2 = fminf(m2, fmaxf(m1, m));
    e1 = m < m1 ? e : e1;
    m1 = fminf(m1, m);
  }
  __device__ void merge_halves() {  // the lane pair (l, l ^ 32) holds one voxel's two halves of the rows
    const float o1 = __shfl_xor(m1, 32), o2 = __shfl_xor(m2, 32);
    const int oe = __shfl_xor(e1, 32);
    const float other = fminf(m2, o2);
    m2 = oe == e1 ? other : fminf(other, fmaxf(m1, o1));
    e1 = o1 < m1 ? oe : e1;
    m1 = fminf(m1, o1);
  }
};
#pragma float_control(pop)

// One workgroup per (grain, run of ZT z-layers) of the output box: its band
// voxels are queued in LDS grouped by the slot of their IDLocal id in the
// grain's hull-id table, and a wavefront takes up to kTake of one slot at a
// time, whichever are left.
template <class T, int NMAX, int ZT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_correct(SimParams sp, PlanDev P, int cls, const int32_t* __restrict__ state,
                                                 DescDev din, DescDev dout, IdlDev il, TopoDev topo, CorrDev cd) {
  if (*cd.ready == 0) return;  // no hull yet (run_sim's first step)
  constexpr int kBuckets = kTopoCap + 1;  // a slot, or the last bucket: an id the hull does not name
  constexpr int kRow = run_chunk(NMAX, ZT);
  static_assert(kTopoCap == 64, "one lane per slot");
  constexpr int VPT = (ZT * NMAX * NMAX + 255) / 256;  // voxels per thread
  static_assert(ZT * NMAX * NMAX <= 0xFFFF, "cell indexes are 16-bit");
  __shared__ int s_key[kTopoCap];
  __shared__ uint16_t s_q[ZT * NMAX * NMAX];  // band voxels grouped by slot
  __shared__ int s_cnt[kBuckets];
  __shared__ int s_next;
  __shared__ int s_at[4][2];
  const int tid = threadIdx.x, lane = tid & 63;
  const T* __restrict__ ain = (const T*)din.arena;
  T* __restrict__ aout = (T*)dout.arena;
  const double delta = sp.delta;
  // The plan's tiles are single layers: a window of ZT consecutive ones holds the
  // first layers of the runs a workgroup takes next (about one), found with one
  // load.  A search's length depends on how far its grain is from the plane x =
  // y, so one range of tiles per XCD is uneven work; about a box's windows at a
  // time go to each XCD in turn (run_window), so a grain's runs still share an
  // L2.  Correction per step at 20000 grains, 4000, 1000: one range per XCD 24.6
  // ms at 20000; single windows in turn 15.7, 1.92, 1.10; a box's at a time 15.5,
  // 1.85, 1.08.  Single tiles in turn, each first layer taking its run, gave 16.3,
  // 1.97, 1.05, but boxes of equal sides have their first layers on one or two
  // XCDs: 3375 cubes of side 24, 7.2 ms against 1.8; 1331 of 32, 10.4 and 2.5; 1000 of
  // 48 and more, 14.0 and 7.0.
  int* at = s_at[tid >> 6];  // the loop's state during a run, off the registers
  for (int u = blockIdx.x, starts = 0;; u += starts ? 0 : gridDim.x) {
    const int total = P.totals[kQLayers * kClasses + cls];
    const int windows = ((total + ZT - 1) / ZT + kXcds * kRow - 1) / (kXcds * kRow) * (kXcds * kRow);
    // a grid with room for it takes the windows twice, the second time for what
    // begins in them after their first run: two runs of a window one after the
    // other are twice the latency of a small launch
    const bool twice = 2 * windows <= (int)gridDim.x, again = twice && u >= windows;
    if (u >= (twice ? 2 * windows : windows)) return;
    const int t = run_window(again ? u - windows : u, kRow) * ZT + lane;
    const bool mine = lane < ZT && t < total;
    const uint32_t v = P.tmap[kQLayers][P.tile_base[kQLayers * kClasses + cls] + (mine ? t : 0)];
    if (starts == 0) {
      starts = (int)__ballot(mine && (v & 0xFFu) % ZT == 0);
      if (twice) starts = again ? starts & (starts - 1) : starts & -starts;
      if (starts == 0) continue;
    }
    const uint32_t tile = (uint32_t)__builtin_amdgcn_readlane((int)v, __builtin_ctz(starts));
    const int g = (int)(tile >> 8), kl = (int)(tile & 0xFFu);
    at[0] = u;
    at[1] = starts & (starts - 1);
    const int32_t* b = dout.bounds + 6 * g;
    const int x0 = b[0], y0 = b[1], z0 = b[2], n = b[3] - b[0], nn2 = n * n;
    const int nv = min(ZT, n - kl) * nn2;  // voxels of the run
    // a grain whose barycenters did not fit the pool (the device error is set)
    // is corrected with the default weights
    const int64_t tb = cd.tbase[g];
    int E = cd.ecount[g];
    if (tb + cd.efirst[(int64_t)g * (kElemCap + 1) + E] > cd.tri_cap) E = 0;
    const int4 sb = cd.sbox[g];
    const bool lists = sb.x == x0 && sb.y == y0 && sb.z == z0 && sb.w == n;  // they hold for this box
    for (int i = tid; i < kTopoCap; i += 256) s_key[i] = topo.key[(int64_t)g * kTopoCap + i];
    if (tid < kBuckets) s_cnt[tid] = 0;
    if (tid == 0) s_next = 0;
    __syncthreads();
    // IDLocal as the resize to the output bounds leaves it: the old content at
    // the same linear index, 0 past its old size
    const int32_t* ob = il.bounds + 6 * g;
    const int64_t oldsize = (int64_t)(ob[3] - ob[0]) * (ob[4] - ob[1]) * (ob[5] - ob[2]);
    const int64_t lbase = (int64_t)kl * nn2;
    const uint32_t* __restrict__ idl = il.arena + il.off[g] + lbase;
    const int oldn = (int)min((int64_t)nv, oldsize - lbase);  // cells below it have an old id
    const T* __restrict__ in = ain + din.off[g] + lbase;
    T* __restrict__ out = aout + dout.off[g] + lbase;
    // counting sort of the band voxels by slot: each lane keeps its voxels'
    // bucket and rank in registers, so one LDS queue is enough
    int pk[VPT];  // bucket << 16 | rank in the bucket, -1: not in the band
#pragma unroll
    for (int u0 = 0; u0 < VPT; u0 += 4) {
      T v[4];
      uint32_t id[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = (u0 + u) * 256 + tid;
        if (u0 + u < VPT && c < nv) v[u] = in[c];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = (u0 + u) * 256 + tid;
        const bool band = u0 + u < VPT && c < nv && fabs((double)v[u]) < delta;
        if (u0 + u < VPT) pk[u0 + u] = band ? 0 : -1;
        id[u] = band && c < oldn ? idl[c] : 0u;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (u0 + u < VPT && pk[u0 + u] == 0) {
          int bucket = kTopoCap;
          uint32_t hsl = (id[u] * 2654435761u) >> (32 - kTopoCapBitsC);
          for (int pr = 0; pr < kTopoCap; ++pr) {
            const int k = s_key[hsl];
            if (k == (int)id[u]) {
              bucket = (int)hsl;
              break;
            }
            if (k == -1) break;
            hsl = (hsl + 1) & (kTopoCap - 1);
          }
          pk[u0 + u] = bucket << 16 | atomicAdd(&s_cnt[bucket], 1);
        }
      }
    }
    __syncthreads();
    // lane s: slot s's count, first queue entry and first chunk of kTake entries
    const int cnt = s_cnt[lane], cnt_none = s_cnt[kTopoCap];
    const int both = cnt | ((cnt + kTake - 1) / kTake) << 16;
    int incl = both;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(incl, d, 64);
      if (lane >= d) incl += u;
    }
    const int start = (incl - both) & 0xFFFF, chunk0 = (incl - both) >> 16;
    const int all = __builtin_amdgcn_readlane(incl, 63);
    const int named = all & 0xFFFF, nch = all >> 16;  // entries with a slot, and their chunks
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int bucket = pk[u] >> 16;
      const int at = __shfl(start, bucket & 63, 64);
      if (pk[u] >= 0) s_q[(bucket < kTopoCap ? at : named) + (pk[u] & 0xFFFF)] = (uint16_t)(u * 256 + tid);
    }
    __syncthreads();
    const double* __restrict__ tri = cd.tri + 3 * tb;
    const int4 o4 = cd.org[g];
    const double see_g = cd.see_on ? cd.see[g] : 0.0;
    const float fn = 1.0f / (float)n, fnn = 1.0f / (float)nn2;
    // coordinates of cell c of the run: its layer, row and column
    auto cell_at = [&](int c, int& zl, int& yl, int& xl) {
      zl = (int)((float)c * fnn);
      int r = c - zl * nn2;
      if (r < 0) { --zl; r += nn2; }
      if (r >= nn2) { ++zl; r -= nn2; }
      yl = (int)((float)r * fn);
      xl = r - yl * n;
      if (xl < 0) { --yl; xl += n; }
      if (xl >= n) { ++yl; xl -= n; }
    };
    const int nchunks = nch + (cnt_none + kTake - 1) / kTake;
    for (;;) {
      int j = 0;
      if (lane == 0) j = atomicAdd(&s_next, 1);
      j = __builtin_amdgcn_readfirstlane(j);
      if (j >= nchunks) break;
      int slot = -1, base, count;
      if (j < nch) {
        slot = 63 - (int)__builtin_clzll(__ballot(chunk0 <= j));
        const int off = (j - __builtin_amdgcn_readlane(chunk0, slot)) * kTake;
        base = __builtin_amdgcn_readlane(start, slot) + off;
        count = min(kTake, __builtin_amdgcn_readlane(cnt, slot) - off);
      } else {
        const int off = (j - nch) * kTake;
        base = named + off;
        count = min(kTake, cnt_none - off);
      }
      Near nr[4] = {{kNone, kNone, -1}, {kNone, kNone, -1}, {kNone, kNone, -1}, {kNone, kNone, -1}};
      bool listed = false;
      int first = 0, npos = 0;
      if (slot >= 0 && E > 0) {
        const int2 sl = cd.slist[(int64_t)g * kTopoCap + slot];
        first = __builtin_amdgcn_readfirstlane(sl.x);
        npos = __builtin_amdgcn_readfirstlane(sl.y);
        listed = lists && npos >= 0;
        if (listed && npos > 0) {
          // the voxels of queue entries base + 32 f + lane % 32 as columns
          v8bf col[4];
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            const int fc = s_q[base + min(f * 32 + (lane & 31), count - 1)];
            int fz, fy, fx;
            cell_at(fc, fz, fy, fx);
            const __bf16 bx = (__bf16)(float)(y0 + fy - o4.y), by = (__bf16)(float)(x0 + fx - o4.x),
                         bz = (__bf16)(float)(z0 + kl + fz - o4.z), one = (__bf16)1.0f, nul = (__bf16)0.0f;
            if (lane < 32) col[f] = v8bf{bx, bx, bx, by, by, by, bz, bz};
            else col[f] = v8bf{bz, one, one, one, nul, nul, nul, nul};
          }
          float run[4] = {kNone, kNone, kNone, kNone};  // the running minimum of the current element
          // lane's row of the four groups of a product, and its half of the row
          const uint16_t* __restrict__ mine =
              cd.rows + (int64_t)first * (kChunk * kRowLen) + (lane & 31) * kRowLen + (lane >> 5) * 8;
          for (int t0 = 0; t0 < npos; t0 += 64) {
            const int np = min(64, npos - t0);
            const int tag = lane < np ? (int)cd.tags[first + t0 + lane] : 0;  // lane t: group t0 + t's
            const unsigned long long ends = __ballot(tag & kTagEnd);
            auto fetch = [&](int i) {  // groups t0 + i .. + 3 (up to kRowSpare past the list: not used)
              return *(const v8bf*)(mine + (int64_t)(t0 + i) * (kChunk * kRowLen));
            };
            auto product = [&](const v8bf& a, int i) {
              const int nib = (int)(ends >> i) & 15;
              const bool whole = (nib & 7) == 0 && i + 4 <= np;  // the four groups are one element's
#pragma unroll
              for (int f = 0; f < 4; f += 2) {
                if (f * 32 >= count) break;
                const v16f d0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, col[f], v16f{}, 0, 0, 0);
                const v16f d1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, col[f + 1], v16f{}, 0, 0, 0);
                if (whole) {
                  run[f] = min16(d0, run[f]);
                  run[f + 1] = min16(d1, run[f + 1]);
                  if (nib) {
                    const int e = __builtin_amdgcn_readlane(tag, i + 3) & (kTagEnd - 1);
                    nr[f].add(run[f], e);
                    nr[f + 1].add(run[f + 1], e);
                    run[f] = run[f + 1] = kNone;
                  }
                } else {
#pragma unroll
                  for (int u = 0; u < 4; ++u) {
                    if (i + u < np) {
                      run[f] = min4(d0, u, run[f]);
                      run[f + 1] = min4(d1, u, run[f + 1]);
                      if ((nib >> u) & 1) {
                        const int e = __builtin_amdgcn_readlane(tag, i + u) & (kTagEnd - 1);
                        nr[f].add(run[f], e);
                        nr[f + 1].add(run[f + 1], e);
                        run[f] = run[f + 1] = kNone;
                      }
                    }
                  }
                }
              }
            };
            v8bf a0 = fetch(0), a1 = fetch(4);
            for (int i = 0; i < np; i += 8) {
              const v8bf b0 = fetch(i + 8), b1 = fetch(i + 12);
              product(a0, i);
              if (i + 4 < np) product(a1, i + 4);
              a0 = b0;
              a1 = b1;
            }
          }
#pragma unroll
          for (int f = 0; f < 4; ++f) nr[f].merge_halves();
        }
      }
#pragma unroll
      for (int h = 0; h < kTake / 64; ++h) {  // 64 of the voxels, one per lane
        if (h * 64 >= count) break;
        const bool act = h * 64 + lane < count;
        const int c = s_q[base + (act ? h * 64 + lane : 0)];
        int zl, yl, xl;
        cell_at(c, zl, yl, xl);
        // Vector3d(i, j, k): row, column, depth, against barycenters (x, y, z)
        const int px = y0 + yl, py = x0 + xl, pz = z0 + kl + zl;
        const Near me = lane < 32 ? nr[2 * h] : nr[2 * h + 1];
        int emin = me.e1;
        if (slot >= 0 && E > 0) {
          bool exact = act;
          if (listed) {
            const float qx = (float)(px - o4.y), qy = (float)(py - o4.x), qz = (float)(pz - o4.z);
            const float rho = __int_as_float(o4.w);
            const float dd = 1.4143f * fabsf((float)(o4.x - o4.y)), pp = sqrtf(qx * qx + qy * qy + qz * qz);
            const float S = rho * rho + 2.0f * rho * (dd + pp);
            // a squared distance of 1e7 or more is no neighbour (the reference's
            // initial minimum): the FP64 search decides where one could be that far
            const float reach = dd + pp + rho;
            exact = act && emin >= 0 && (me.m2 - me.m1 <= 2.0f * kFilterEps * S + kDecided || reach * reach > 9.9e6f);
          }
          // f(e, r0, r1): the slot's elements, barycenters [r0, r1)
          auto over_elements = [&](auto f) {
            for (int e0 = 0; e0 < E; e0 += 64) {
              const int el = e0 + lane;
              const bool has = el < E && ((cd.emask[(int64_t)g * kElemCap + (el < E ? el : 0)] >> slot) & 1ull);
              for (unsigned long long m = __ballot(has); m; m &= m - 1) {
                const int e = e0 + (int)__builtin_ctzll(m);
                const int32_t* ef = cd.efirst + (int64_t)g * (kElemCap + 1) + e;
                f(e, ef[0], ef[1]);
              }
            }
          };
          unsigned long long todo = __ballot(exact);
          if (__popcll(todo) > kManyExact) {
            // every lane searches for its own voxel, the barycenters uniform
            // (no slot with a list, correction per step: 20000 grains 279 ms, one
            // voxel at a time by the wavefront 985; 4000 26.6 and 83)
            double dmin = 10000000.0;
            int em = -1;
            auto attempt = [&](int r, int e, bool there) {
              const double* q = tri + 3 * (int64_t)r;
              const double dx = px - q[0], dy = py - q[1], dz = pz - q[2];
              const double d = dx * dx + dy * dy + dz * dz;
              if (there && (d < dmin || (d == dmin && e < em))) {
                dmin = d;
                em = e;
              }
            };
            if (listed) {
              for (int t = 0; t < npos; ++t) {
                const int e = cd.tags[first + t] & (kTagEnd - 1);
#pragma unroll
                for (int r = 0; r < kChunk; ++r) {
                  const int src = cd.rsrc[((int64_t)first + t) * kChunk + r];
                  attempt(max(src, 0), e, src >= 0);
                }
              }
            } else {
              over_elements([&](int e, int r0, int r1) {
                for (int r = r0; r < r1; r += 4) {
#pragma unroll
                  for (int u = 0; u < 4; ++u) attempt(min(r + u, r1 - 1), e, true);
                }
              });
            }
            if (exact) emin = em;
            todo = 0;
          }
          for (; todo; todo &= todo - 1) {
            const int who = (int)__builtin_ctzll(todo);
            const double dpx = (double)__builtin_amdgcn_readlane(px, who),
                         dpy = (double)__builtin_amdgcn_readlane(py, who),
                         dpz = (double)__builtin_amdgcn_readlane(pz, who);
            double dmin = 10000000.0;
            int em = -1;
            auto attempt = [&](int r, int e) {
              const double* q = tri + 3 * (int64_t)r;
              const double dx = dpx - q[0], dy = dpy - q[1], dz = dpz - q[2];
              const double d = dx * dx + dy * dy + dz * dz;
              if (d < dmin || (d == dmin && e < em)) {
                dmin = d;
                em = e;
              }
            };
            if (listed) {
              for (int r = lane; r < npos * kChunk; r += 64) {
                const int src = cd.rsrc[(int64_t)first * kChunk + r];
                if (src >= 0) attempt(src, cd.tags[first + r / kChunk] & (kTagEnd - 1));
              }
            } else {
              over_elements([&](int e, int r0, int r1) {
                for (int r = r0 + lane; r < r1; r += 64) attempt(r, e);
              });
            }
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {  // the smallest (distance, element) pair
              const double od = __shfl_xor(dmin, o);
              const int oe = __shfl_xor(em, o);
              if (od < dmin || (od == dmin && (unsigned)oe < (unsigned)em)) {
                dmin = od;
                em = oe;
              }
            }
            if (lane == who) emin = em;
          }
        }
        double w_energy = 1.0, w_mobility = 1.0;
        if (emin >= 0) {
          w_energy = cd.mobility[(int64_t)g * kElemCap + emin];
          w_mobility = cd.energy[(int64_t)g * kElemCap + emin];
        }
        if (act) {
          const double val = (double)in[c];
          double o = (double)out[c];
          o = val + (o - val) * w_energy * w_mobility;
          if (cd.see_on) {
            const uint32_t id = c < oldn ? idl[c] : 0u;
            const bool nb = id == 0u || (id <= (uint32_t)sp.N && state[id] != kDeleted);
            double f = 0;
            if (nb) f = (see_g - cd.see[id]) * w_mobility * cd.dt / cd.tsq;
            o = o - f;
          }
          out[c] = (T)o;
        }
      }
    }
    __syncthreads();  // the queue is refilled for the next run
    u = __builtin_amdgcn_readfirstlane(at[0]);
    starts = __builtin_amdgcn_readfirstlane(at[1]);
  }
}

template <class T>
void correct_classes(const Launch& L, const SimParams& sp, const PlanDev& P, const int32_t* state, const DescDev& din,
                     const DescDev& dout, const IdlDev& il, const TopoDev& topo, const CorrDev& cd, int c0, int c1) {
  if (c0 <= 0 && 0 < c1)
    hipLaunchKernelGGL((k_correct<T, 32, 8>), dim3(tile_grid(L, kCorrGridPerCU, 0, sp.N, 2 * (layers_of(0) / 8 + 1))), dim3(256), 0, L.stream, sp, P, 0,
                     state, din, dout, il, topo, cd);
  if (c0 <= 1 && 1 < c1)
    hipLaunchKernelGGL((k_correct<T, 48, 4>), dim3(tile_grid(L, kCorrGridPerCU, 1, sp.N, 2 * (layers_of(1) / 4 + 1))), dim3(256), 0, L.stream, sp, P, 1,
                     state, din, dout, il, topo, cd);
  if (c0 <= 2 && 2 < c1)
    hipLaunchKernelGGL((k_correct<T, 64, 2>), dim3(tile_grid(L, kCorrGridPerCU, 2, sp.N, 2 * (layers_of(2) / 2 + 1))), dim3(256), 0, L.stream, sp, P, 2,
                     state, din, dout, il, topo, cd);
  if (c0 <= 3 && 3 < c1)
    hipLaunchKernelGGL((k_correct<T, 96, 1>), dim3(tile_grid(L, kCorrGridPerCU, 3, sp.N, layers_of(3) + 1)), dim3(256), 0, L.stream, sp, P, 3,
                     state, din, dout, il, topo, cd);
}

}  // namespace

void launch_elements(const Launch& L, const SimParams& sp, const int32_t* state, const DescDev& dout,
                     const TopoDev& topo, const CorrDev& cd, int32_t* err) {
  hipLaunchKernelGGL(k_clear_counters, dim3(1), dim3(64), 0, L.stream, cd.tri_n, cd.row_n);
  const int blocks = sp.N < L.grid ? sp.N : L.grid;
  hipLaunchKernelGGL(k_elements, dim3(blocks > 0 ? blocks : 1), dim3(kEW), 0, L.stream, sp, state, topo, cd, err);
  hipLaunchKernelGGL(k_tri_scatter, dim3(L.grid), dim3(256), 0, L.stream, topo, cd);
  hipLaunchKernelGGL(k_slots, dim3(sp.N > 0 ? sp.N : 1), dim3(256), 0, L.stream, sp, state, dout, topo, cd);
}

void launch_correction(const Launch& L, const SimParams& sp, const PlanDev& P, const int32_t* state,
                       const DescDev& din, const DescDev& dout, const IdlDev& il_stale, const TopoDev& topo,
                       const CorrDev& cd, bool fp32, int c0, int c1) {
  if (fp32) correct_classes<float>(L, sp, P, state, din, dout, il_stale, topo, cd, c0, c1);
  else correct_classes<double>(L, sp, P, state, din, dout, il_stale, topo, cd, c0, c1);
}

}  // namespace gg
