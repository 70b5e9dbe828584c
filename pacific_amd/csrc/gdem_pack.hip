// gdem_pack.hip -- the sphere step in the packed layout (skin candidate
// lists, memoryless contact models).
//
// A step that keeps its lists is one kernel below kStepSmall particles
// (k_step) and two from there on (k_pairs, k_integ).  Candidates are screened, the
// pairs that may touch are gathered into a queue in LDS and evaluated one per
// lane with the reference's body order (RigidBodyWithCrust.cpp:596-640,
// HookeContactForceModel.cpp:44-114 / HertzContactForceModel.cpp:46-114), and
// each particle sums its own contacts in a fixed order -- detected contacts by
// entry, then received contacts by partner slot, then walls -- (Torsor.cpp:
// 184-189, no floating-point atomics) and applies the leap-frog tail
// (SecondOrderLeapFrog.cpp:44-94 via ParticleKinematics.cpp:62-128), writing
// the other state copy.  In k_step both partners evaluate a pair, with the
// same operands in the same order, so they get the same force bit for bit and
// nothing passes between workgroups inside a step; k_pairs evaluates each
// pair once and stores a record that k_integ adds to both bodies.
//
// A rebuild of the lists (k_pk_count, k_scan, k_pk_scatter, k_pk_cellsort,
// k_pk_sweep, k_pk_lists: the counting sort by cell and the half-stencil sweep,
// LinkedCell.cpp:1019-1103) is launched once per chunk of at most kChunkSteps
// steps and exits at once when it is not due.  When a particle's path passes
// the skin's limit in the middle of a chunk, the remaining step kernels of that
// chunk exit without doing anything (StepWords), the next chunk starts with
// the rebuild and continues from the step that waited: the rebuilds happen at
// exactly the steps at which a check before every step would make them.  The
// chunks are as long as the lists' lives make worth while (ChunkPolicy).
//
// The per-pair arithmetic and the order of every sum are those of the fused
// kernel (gdem_sphere_step.h), so both give bit-identical results.  Contact
// statistics need fixed-order sums over the evaluations; with statistics on,
// gdem_step runs the canonical layout.
//
// Bound: below some 100,000 particles the step is one chain of dependent
// loads and FP64 operations (about 12 us) and launches.  us per step of a call
// (gdem_step alone), with the six launches per step of before (screening,
// contacts, integrator and three rebuild kernels that exit) and now: 1,000
// particles in a box 26 and 15, a touching bed of 30,000 54 to 59 and 26, a gas
// of 100,000 40 and 21.  Many particles stream the state (about 250 B each)
// through k_integ, and both partners' evaluations in one kernel no longer hide
// behind it: at 1M in a gas k_step takes 125 us a step, k_pairs and k_integ 103
// to 109 (six launches 118 to 122); at 400,000 k_step takes 58 and the two 61,
// and in a packing of 500,000 190 to 215 against 220: the line lies at
// kStepSmall.  With the occupancy check off (gdem_set_skin_adapt) a rebuild is
// offered before every step, seven launches: 21 us at 1,000, 30 at 100,000, 119
// at 1M (22, 40 and 124 before).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gdem_binning.h"
#include "gdem_internal.h"
#include "gdem_sphere_step.h"
#include "gdem_sweep.h"

#pragma clang fp contract(off)

namespace gdem {

constexpr int kPB = 256;

static inline int pblocks(int n) { return (n + kPB - 1) / kPB; }

// ---------------------------------------------------------------- layout
// Puts an incoming list into the order its contacts are summed in: partner
// slot, then code (next_incoming's order), so the step walks it as it stands.
__device__ __forceinline__ void sort_incoming(int2* l, int n, int stride) {
  auto key = [](int2 e) { return ((long long)e.x << 7) | (long long)(e.y & 127); };
  for (int i = 1; i < n; ++i) {
    const int2 v = l[(size_t)i * stride];
    int b = i - 1;
    while (b >= 0) {
      const int2 u = l[(size_t)b * stride];
      if (key(u) <= key(v)) break;
      l[(size_t)(b + 1) * stride] = u;
      --b;
    }
    if (b + 1 != i) l[(size_t)(b + 1) * stride] = v;
  }
}

// The screening list of particle t from its candidate lists: entries by
// increasing gap bound, so that a step reads only the entries its paths can
// have closed; an entry carries its place in the order of summation (out
// entries, then in entries by partner slot) in bits 0-5 of its code.  Few
// particles (k_step) screen both lists, many (k_pairs) each pair at its out
// entry, and leave the in-list as the mirror indices of the entries know it.
// touch: its entries that touch or nearly do.  Returns the longer of the two
// lists (the build's counts, before any cut).
// The keys are sorted in a column of LDS (keys, one column per lane).
// COUNTED: the incoming counts are complete.
template <bool COUNTED>
__device__ __forceinline__ int build_screen_list(const StepLists& l, int t, int n,
                                                 uint32_t (*keys)[kPB], int& touch) {
  const int co = l.out_count[t], ci = COUNTED ? l.in_count[t] : 0;
  const int nout = min(co, kListCap), nin = l.both ? min(ci, kListCap) : 0;
  if (l.both) sort_incoming(l.in_list + t, nin, n);
  const int lane = threadIdx.x, cnt = nout + nin;
  auto entry = [&](int k) {
    return k < nout ? l.out_list[(size_t)k * n + t] : l.in_list[(size_t)(k - nout) * n + t];
  };
  touch = 0;
  for (int k = 0; k < cnt; ++k) {
    const uint32_t key = ((uint32_t)entry(k).y & kGapMask) | (uint32_t)k;
    if (!(key & kGapMask)) ++touch;
    int b = k - 1;
    for (; b >= 0 && keys[b][lane] > key; --b) keys[b + 1][lane] = keys[b][lane];
    keys[b + 1][lane] = key;
  }
  for (int k = 0; k < cnt; ++k) {
    const uint32_t key = keys[k][lane];
    l.screen[(size_t)k * n + t] = make_int2(entry((int)(key & 63u)).x, (int)key);
  }
  l.screen_count[t] = cnt;
  l.min_gap[t] = cnt ? gap_bound((int)keys[0][lane], l.gap_unit) : __builtin_huge_valf();
  return max(co, ci);
}

// Largest list length of the build where it comes near the capacity (the only
// case anything is done about): an atomic of every wave on one word would
// take 190 us at 1M particles.
__device__ __forceinline__ void note_peak(int peak, StepWords* w) {
  if (peak > kListCap - kListHeadroom) atomicMax(&w->peak, peak);
}

// Counter `seg` of row j.  Each counter has a cache line of its own: atomics
// on one line are served one after another (64 counters in two lines cost an
// integrating kernel 100 us at 1M particles, spread over 64 lines about 2 us).
__device__ __forceinline__ int32_t* row_word(int32_t* rows, int j, int seg) {
  return rows + ((size_t)j * kRowSegs + seg) * kRowPad;
}

// Largest path length of the launch that will read row j: one integer atomic
// per wave on the workgroup's segment of the row (a non-negative float's bits
// are ordered as integers).
__device__ __forceinline__ void wave_path(float len, int32_t* rows, int j) {
  int b = __float_as_int(len);
  for (int o = 32; o > 0; o >>= 1) b = max(b, __shfl_xor(b, o, 64));
  if ((threadIdx.x & 63) == 0 && b > 0) atomicMax(row_word(rows, j, blockIdx.x % kRowSegs), b);
}
__device__ __forceinline__ float row_path(int32_t* rows, int j) {
  static_assert(kRowSegs == 64, "one lane per segment");
  int b = *row_word(rows, j, threadIdx.x & 63);
  for (int o = 32; o > 0; o >>= 1) b = max(b, __shfl_xor(b, o, 64));
  return __int_as_float(b);
}

// Touching candidates of the last build (row kTouchRow).
__device__ __forceinline__ void wave_touch(int touch, int32_t* rows) {
  for (int o = 32; o > 0; o >>= 1) touch += __shfl_xor(touch, o, 64);
  if ((threadIdx.x & 63) == 0 && touch > 0)
    atomicAdd(row_word(rows, kTouchRow, blockIdx.x % kRowSegs), touch);
}

// World angular velocity of slot s of copy `in` where it is not stored: the
// step that wrote the copy computed it as q (omega_body) q* with the
// orientation q from before its update (SecondOrderLeapFrog.cpp:74-94, then
// ParticleKinematics.cpp:62-104), which the other copy still holds at slot
// so.  The same operations in the same order: the value is bit-identical.
__device__ __forceinline__ v3 world_omega(const Pack& in, const Pack& other, int s, int so) {
  const double4 d = in.D[s];
  const quat q = qmk(mk(other.A[so].w, other.B[so].w, other.D[so].w), other.E[so]);
  return qmulv(q, qleftvec(qconj(q), mk(d.x, d.y, d.z)));
}

// The canonical copy into the packed one.  Thread 0 sets the step words: a
// rebuild is due if the canonical words say so for copy p.  The screening
// lists are made here when the canonical kernels built the candidate lists.
__global__ void __launch_bounds__(kPB) k_to_pack(State s, Pack pk, PackConst k0, PackConst k1,
                                                 StepLists l, float* path, const float* path_in,
                                                 int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  __shared__ uint32_t sh_keys[2 * kListCap][kPB];
  int peak = 0, touch = 0;
  float len = 0.f;
  if (i < n) {
    const double4 pr = s.pos_r[i], vm = s.vel_m[i], wr = s.om_req[i], wb = s.wbf_I[i],
                  q = s.quat[i];
    pk.A[i] = make_double4(pr.x, pr.y, pr.z, q.x);
    pk.B[i] = make_double4(vm.x, vm.y, vm.z, q.y);
    pk.C[i] = make_double4(wr.x, wr.y, wr.z, 0.);
    pk.D[i] = make_double4(wb.x, wb.y, wb.z, q.z);
    pk.E[i] = q.w;
    const double2 rr = make_double2(pr.w, wr.w), mi = make_double2(vm.w, wb.w);
    const Aux ax = s.aux[i];
    k0.rr[i] = rr;
    k0.mi[i] = mi;
    k0.aux[i] = ax;
    k1.rr[i] = rr;
    k1.mi[i] = mi;
    k1.aux[i] = ax;
    len = path_in[i];
    path[i] = len;
    // without a build the lists hold nothing yet; need is set then
    if (!l.words->slot[kChunkSteps].need) peak = build_screen_list<true>(l, i, n, sh_keys, touch);
  }
  note_peak(peak, l.words);
  wave_touch(touch, l.path_rows);
  wave_path(len, l.path_rows, kChunkSteps);
}

__global__ void __launch_bounds__(64) k_step_words(StepWords* w, int32_t* path_rows,
                                                   const SkinWords* words, int p) {
  *row_word(path_rows, kChunkSteps, threadIdx.x) = 0;
  *row_word(path_rows, kTouchRow, threadIdx.x) = 0;
  if (threadIdx.x != 0) return;
  w->slot[kChunkSteps] = StepSlot{0, p, words->need[p] != 0 ? 1 : 0, 0, 1};
  w->target = 0;
  w->peak = 0;
  w->chunks = 0;
  w->rebuilds = 0;
}

__global__ void __launch_bounds__(kPB) k_from_pack(Pack pk, PackConst k, State s, float* path_out,
                                                   const float* path, const StepWords* w,
                                                   SkinWords* words, int p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) words->need[p] = w->slot[kChunkSteps].need;
  if (i >= n) return;
  const double4 a = pk.A[i], b = pk.B[i], c = pk.C[i], d = pk.D[i];
  const double2 rr = k.rr[i], mi = k.mi[i];
  s.pos_r[i] = make_double4(a.x, a.y, a.z, rr.x);
  s.vel_m[i] = make_double4(b.x, b.y, b.z, mi.x);
  s.om_req[i] = make_double4(c.x, c.y, c.z, rr.y);
  s.wbf_I[i] = make_double4(d.x, d.y, d.z, mi.y);
  s.quat[i] = make_double4(a.w, b.w, d.w, pk.E[i]);
  s.aux[i] = k.aux[i];
  path_out[i] = path[i];
}

// ---------------------------------------------------------------- rebuild
// The rebuild kernels read the step words and the copy they name; each exits
// at once unless a rebuild is due.  k_pk_count hands the state of the step
// sequence over from the end of the previous chunk (slot kChunkSteps) to
// slot 0 (with the largest paths of row kChunkSteps to row 0), k_pk_scatter
// clears the need flags and path rows the chunk's steps write.
__global__ void __launch_bounds__(kPB) k_pk_count(Bins b, PosSrc src0, PosSrc src1, Pack pk0,
                                                  Pack pk1, StepWords* w,
                                                  int32_t* path_rows, SkinWords* words,
                                                  int32_t* in_count, int n, Grid g, const int32_t* row_rank,
                                                  unsigned long long* err) {
  const StepSlot sl = w->slot[kChunkSteps];
  const bool open = sl.done < w->target;
  const bool rebuild = open && sl.need;
  if (blockIdx.x == 0 && threadIdx.x < kRowSegs) {
    *row_word(path_rows, 0, threadIdx.x) =
        rebuild ? 0 : *row_word(path_rows, kChunkSteps, threadIdx.x);
    if (rebuild) *row_word(path_rows, kTouchRow, threadIdx.x) = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    w->slot[0] = sl;
    if (rebuild) w->slot[0].wstored = 1;
    if (open) w->chunks += 1;
    if (rebuild) {
      words->rebuilds += 1;
      w->rebuilds += 1;
      w->peak = 0;
    }
  }
  if (!rebuild) return;
  if (!sl.wstored) {
    // the steps after the rebuild read the copy through the new order: the
    // world angular velocity is stored first, from the orientations of the
    // other copy at the slots of the previous order (perm still holds it)
    const Pack& in = sl.cur ? pk1 : pk0;
    const Pack& other = sl.cur ? pk0 : pk1;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
      const v3 w3 = world_omega(in, other, i, sl.rebuilt ? b.perm[i] : i);
      in.C[i] = make_double4(w3.x, w3.y, w3.z, 0.);
    }
  }
  count_pass(b.key, b.slot, b.cnt, n, true, in_count, sl.cur ? src1 : src0, g, row_rank, err);
}

__global__ void __launch_bounds__(kPB) k_pk_scatter(Bins b, StepWords* w, SkinGate gate, int n,
                                                    int32_t* path_rows) {
  const bool rebuild = gate.rebuild();
  if (blockIdx.x == 0) {
    if (threadIdx.x >= 1 && threadIdx.x <= kChunkSteps) w->slot[threadIdx.x].need = 0;
    for (int k = threadIdx.x; k < kChunkSteps * kRowSegs; k += kPB)
      *row_word(path_rows, 1 + k / kRowSegs, k % kRowSegs) = 0;
  }
  if (!rebuild) return;
  scatter_pass(b.key, b.slot, b.local, b.bsum, b.perm, n);
}

__global__ void __launch_bounds__(kPB) k_pk_cellsort(Bins b, PosSrc src0, PosSrc src1,
                                                     SkinGate gate, int ncell, int n) {
  if (!gate.rebuild()) return;
  const PosSrc src = gate.sw->slot[0].cur ? src1 : src0;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += gridDim.x * blockDim.x)
    sort_cell(b.local, b.bsum, b.perm, b.cell_start, src, b.pos, b.ids, c, ncell, n);
}

// The candidate sweep; grid-stride over the particles' workgroups (the grid
// is a multiple of 8, so a workgroup stays on its XCD's range of cells).
// LISTS: the screening lists hold the out entries alone, so each particle's is
// made right after its sweep (the longest incoming list is noted by the sweep).
// Bound by the latency of its loads: without the contact test, which candidates
// never take, it holds 51 registers instead of 140, and seven waves share a
// SIMD instead of three.  1M particles: sweep 173 us and lists 37 us in a kernel
// of their own before, 149 us together.
template <bool LISTS>
__global__ void __launch_bounds__(kPB) k_pk_sweep(DetectArgs d, PosSrc src0, PosSrc src1,
                                                  StepLists l) {
  __shared__ uint32_t sh_keys[LISTS ? kListCap : 1][kPB];
  if (!d.gate.rebuild()) return;
  const PosSrc src = d.gate.sw->slot[0].cur ? src1 : src0;
  const int per = d.nblk8 >> 3;
  for (int b = blockIdx.x; b < d.nblk8; b += gridDim.x) {
    const int t = ((b & 7) * per + (b >> 3)) * kPB + threadIdx.x;
    if (t < d.n) detect_particle<kSweepCandidates>(d, src, t);
    if (LISTS) {
      int touch = 0;
      note_peak(t < d.n ? build_screen_list<false>(l, t, d.n, sh_keys, touch) : 0, l.words);
      wave_touch(touch, l.path_rows);
    }
  }
}

// Screening lists of out and in entries: after the whole sweep.
__global__ void __launch_bounds__(kPB) k_pk_lists(StepLists l, SkinGate gate, int n) {
  __shared__ uint32_t sh_keys[2 * kListCap][kPB];
  if (!gate.rebuild()) return;
  for (int b0 = blockIdx.x * kPB; b0 < n; b0 += gridDim.x * kPB) {
    const int t = b0 + threadIdx.x;
    int touch = 0;
    note_peak(t < n ? build_screen_list<true>(l, t, n, sh_keys, touch) : 0, l.words);
    wave_touch(touch, l.path_rows);
  }
}

// ---------------------------------------------------------------- step
// What one launch of a step works on, from its slot of the step words.
struct StepView {
  Pack in, out;
  PackConst kin, kout;
  const float* path;
  float* path_out;
  bool rebuild;     // lists just rebuilt: the copy is read through perm
  bool copy_const;  // the constants go to the other copy: a rebuild reorders
                    // them, the step after it fills the remaining copy
  bool last;        // closes with the half kick and writes F and T
  bool wstored;     // in.C holds the world angular velocities
  bool moved;       // the other copy is in the order before the last rebuild
  float far;        // no particle's path is longer
};

// False: nothing to do (target reached, or a rebuild is due that this launch
// was not offered).
__device__ __forceinline__ bool step_view(const StepArgs& a, int j_in, int after, StepSlot& sl,
                                          StepView& v) {
  sl = a.w->slot[j_in];
  const int target = a.w->target;
  if (sl.done >= target || (sl.need && !after)) return false;
  v.in = sl.cur ? a.pk1 : a.pk0;
  v.out = sl.cur ? a.pk0 : a.pk1;
  v.kin = sl.cur ? a.kc1 : a.kc0;
  v.kout = sl.cur ? a.kc0 : a.kc1;
  v.path = sl.cur ? a.path1 : a.path0;
  v.path_out = sl.cur ? a.path0 : a.path1;
  v.rebuild = sl.need != 0;
  v.copy_const = v.rebuild || sl.rebuilt;
  v.last = sl.done + 1 == target;
  v.wstored = sl.wstored != 0;
  v.moved = sl.rebuilt != 0;
  v.far = row_path(a.path_rows, j_in);
  return true;
}

// The step words after a launch (the first wave of the grid): done a step, or
// passed on as they are.
__device__ __forceinline__ void step_done(const StepArgs& a, int j_in, int j_out,
                                          const StepSlot& sl, bool did, bool wstored) {
  if (blockIdx.x != 0 || threadIdx.x >= kRowSegs) return;
  StepSlot& o = a.w->slot[j_out];
  if (!did)
    *row_word(a.path_rows, j_out, threadIdx.x) = *row_word(a.path_rows, j_in, threadIdx.x);
  if (threadIdx.x != 0) return;
  if (!did) {
    o = sl;
    return;
  }
  o.done = sl.done + 1;
  o.cur = sl.cur ^ 1;
  o.rebuilt = sl.need ? 1 : 0;
  o.wstored = wstored ? 1 : 0;
}

// Candidates of particle t that may touch it, as a bit mask over their places
// in the order of summation; mine: its path length, r its radius.  The
// screening list is ordered by a lower bound of each pair's gap at the last
// rebuild: the entries beyond the two longest possible paths end the walk,
// and an entry whose gap exceeds the two paths cannot have met, for which
// only the partner's path (4 B) is read instead of its position and radius
// (48 B).  Otherwise apart() decides, as in the canonical screening.  Of L
// lanes that share a particle, this one takes the entries sub, sub + L, ...
template <int L>
__device__ __forceinline__ unsigned long long screen_particle(const StepArgs& a,
                                                              const StepView& vw, int t, v3 X,
                                                              double r, float mine, int sub) {
  unsigned long long may = 0ull;
  const int cnt = a.screen_count[t];
  const int2* l = a.screen + t;
  const float reach = mine + vw.far;
  for (int e0 = sub; e0 < cnt; e0 += 2 * L) {
    int2 en[2];
    float pu[2];
    int su[2];
    double4 q[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
      en[k] = e0 + k * L < cnt ? l[(size_t)(e0 + k * L) * a.lstride] : make_int2(-1, -1);
    if (gap_bound(en[0].y, a.gap_unit) > reach) break;
#pragma unroll
    for (int k = 0; k < 2; ++k) pu[k] = (en[k].x >= 0 && !vw.rebuild) ? vw.path[en[k].x] : 0.f;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      su[k] = en[k].x;
      if (su[k] < 0) continue;
      if (gap_bound(en[k].y, a.gap_unit) > mine + pu[k]) su[k] = -1;
      else if (vw.rebuild) su[k] = a.perm[su[k]];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (su[k] >= 0) {
        const double4 p = vw.in.A[su[k]];
        q[k] = make_double4(p.x, p.y, p.z, vw.kin.rr[su[k]].x);
      }
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (su[k] >= 0 && !apart(a.grid, X, r, q[k])) may |= 1ull << (en[k].y & 63);
  }
  return may;
}

// One candidate pair: particle at slot s of the copy and its entry's partner
// at slot su, world angular velocities W and W2; first: the particle is the
// reference's first body.  f: force on the first body, ta and tb: torques on
// the first and on the second.  Returns whether they touch.
__device__ __forceinline__ bool pair_contact(const StepArgs& a, const Pack& in,
                                             const PackConst& kin, int s, int su, bool first,
                                             v3 W, v3 W2, v3& f, v3& ta, v3& tb) {
  const double4 p1 = in.A[s], p2 = in.A[su];
  const double2 rr = kin.rr[s], rr2 = kin.rr[su];
  const double4 b = in.B[s], b2 = in.B[su];
  const Aux ax = kin.aux[s], ax2 = kin.aux[su];
  const double m = kin.mi[s].x, m2 = kin.mi[su].x;
  const v3 X = mk(p1.x, p1.y, p1.z);
  const v3 V = mk(b.x, b.y, b.z), V2 = mk(b2.x, b2.y, b2.z);
  // either body may have crossed a periodic face since the list was built:
  // the partner is taken at its nearest image
  const int sx = image_shift(a.grid, 0, p2.x - X.x);
  const int sy = image_shift(a.grid, 1, p2.y - X.y);
  const int sz = image_shift(a.grid, 2, p2.z - X.z);
  const double shx = sx * a.grid.size[0], shy = sy * a.grid.size[1], shz = sz * a.grid.size[2];
  // the two bodies in the reference's order
  const v3 A = first ? X : mk(p2.x, p2.y, p2.z);
  const v3 B = first ? mk(p2.x + shx, p2.y + shy, p2.z + shz)
                     : mk(X.x + (-shx), X.y + (-shy), X.z + (-shz));
  const v3 VA = first ? V : V2, VB = first ? V2 : V, WA = first ? W : W2, WB = first ? W2 : W;
  const double rA = first ? rr.x : rr2.x, rB = first ? rr2.x : rr.x;
  const double qA = first ? rr.y : rr2.y, qB = first ? rr2.y : rr.y;
  const double mA = first ? m : m2, mB = first ? m2 : m;
  const Aux xA = first ? ax : ax2, xB = first ? ax2 : ax;
  v3 cp, ov;
  double dist;
  int rc = sphere_sphere(A, rA, xA.crust, B, rB, xB.crust, cp, ov, dist);
  int nbIter = 1;
  if (rc < 0) rc = sphere_sphere_retry(A, rA, xA.crust, B, rB, xB.crust, cp, ov, dist, nbIter);
  if (rc < 0) {
    atomicMin(&a.err[kErrContact], pack_ids(xA.id, xB.id));
    return false;
  }
  if (rc == 0 || !(dist < 0.)) return false;
  const Model& md = a.models[xA.mat * a.model_stride + xB.mat];
  f = contact_force(md, cp, ov, dist, A, VA, WA, mA, qA, B, VB, WB, mB, qB);
  ta = cross(sub(cp, A), f);
  tb = cross(sub(cp, B), neg(f));
  return true;
}

// One queued wall contact of particle t (SimpleObstacle::InterAction,
// Component/src/SimpleObstacle.cpp:222-271).
__device__ __forceinline__ bool wall_contact(const StepArgs& a, const Pack& in,
                                             const PackConst& kin, int s, int wi, v3 W, v3& f,
                                             v3& tq) {
  const Wall& wl = a.walls[wi];
  const double4 p = in.A[s], b = in.B[s];
  const double2 rr = kin.rr[s];
  const Aux ax = kin.aux[s];
  const v3 X = mk(p.x, p.y, p.z);
  v3 c = mk(0., 0., 0.), ov = mk(0., 0., 0.);
  double dist;
  int nbIter = 1;
  int rc = wl.kind == WALL_RECTANGLE ? sphere_rect(wl, X, rr.x, c, ov, dist)
                                     : sphere_wall(wl, X, rr.x, ax.crust, c, ov, dist);
  if (rc < 0) rc = sphere_wall_retry(wl, X, rr.x, ax.crust, c, ov, dist, nbIter);
  if (rc < 0) {
    atomicMin(&a.err[kErrContact], pack_ids(ax.id, -1 - wi));
    return false;
  }
  if (rc == 0 || !(dist < 0.)) return false;
  const Model& md = a.models[ax.mat * a.model_stride + wl.material];
  // the wall's velocity at the contact point (Obstacle.cpp:128-133)
  const v3 wo = mk(wl.origin[0], wl.origin[1], wl.origin[2]);
  const v3 wv = mk(wl.vel[0], wl.vel[1], wl.vel[2]);
  const v3 ww = mk(wl.omega[0], wl.omega[1], wl.omega[2]);
  f = contact_force(md, c, ov, dist, X, mk(b.x, b.y, b.z), W, kin.mi[s].x, rr.y,
                    wo, wv, ww, 1.e20, wl.req);
  tq = cross(sub(c, X), f);
  return true;
}

// Periodic wrap of coordinate x along axis d after the drift; false when x
// may have left the grid along a closed axis (Cell::GetCell then decides).
__device__ __forceinline__ bool wrap_axis(const StepArgs& a, int d, double& x) {
  if (a.grid.periodic[d]) {
    const double lo = a.grid.origin[d], L = a.grid.size[d];
    if (x >= lo + L) x -= L;
    else if (x < lo) x += L;
    return true;
  }
  const double u = x - a.grid.origin[d];
  return u >= 0. && u <= a.gmax[d];
}

// State of one particle that changes at every step.
struct StepState {
  double4 A, B, D;
  double qw;
  double2 mi;
};
__device__ __forceinline__ StepState load_state(const StepView& v, int s) {
  return StepState{v.in.A[s], v.in.B[s], v.in.D[s], v.in.E[s], v.kin.mi[s]};
}

// Weight m (1 - 0/rho) g at the centre (InitializeForce, Particle.cpp:414-419,
// 1409-1416).
__device__ __forceinline__ v3 weight(const StepArgs& a, double m) {
  const double mw = m * (1. - 0. / 1.);
  return mk(a.gravity[0] * mw, a.gravity[1] * mw, a.gravity[2] * mw);
}

// Leap-frog tail of particle t (as force_particle) with force F and torque T:
// writes the other copy, the path length (mine before this step, len after
// it) and the need flag of the next step.
__device__ __forceinline__ void finish_particle(const StepArgs& a, const StepView& vw,
                                                const StepState& st, int t, int s, float mine,
                                                v3 F, v3 T, int j_out, bool store_w,
                                                float& len) {
  const double4 A4 = st.A, B4 = st.B, D4 = st.D;
  const double qw = st.qw, m = st.mi.x, I = st.mi.y;
  const bool last = vw.last, rebuild = vw.rebuild;
  const v3 X = mk(A4.x, A4.y, A4.z), V = mk(B4.x, B4.y, B4.z);
  v3 WBF = mk(D4.x, D4.y, D4.z);
  quat q = qmk(mk(A4.w, B4.w, D4.w), qw);
  v3 Xo = X, Vo, Wo;
  double drift = 0.;
  const quat pc = qconj(q);
  // torque in body frame (ParticleKinematics.cpp:115-117)
  const v3 tq = qmulv(pc, qleftvec(q, T));
  const double mcf = m * 1.;
  // closing half kick, SecondOrderLeapFrog::advanceVelocity (:74-94)
  Vo = add(V, scl(dvd(F, mcf), a.dt_vel));
  WBF = ssprk3_sphere(tq, WBF, I, a.dt_vel);
  if (last) {
    Wo = qmulv(q, qleftvec(pc, WBF));
    a.F[t] = make_double4(F.x, F.y, F.z, 0.);
    a.T[t] = make_double4(T.x, T.y, T.z, 0.);
  } else {
    // next step's kick and drift, SecondOrderLeapFrog::Move (:44-67) and
    // ParticleKinematics::Move (:62-104)
    Vo = add(Vo, scl(dvd(F, mcf), a.dt_vel));
    const v3 dx = scl(Vo, a.dt_disp);
    WBF = ssprk3_sphere(tq, WBF, I, a.dt_vel);
    Wo = qmulv(q, qleftvec(pc, WBF));
    const v3 avg = Wo;
    Xo = add(X, dx);
    const double nOmega = norm(avg);
    quat dq;
    if (nOmega > kEps) {
      const double cc = cos(nOmega * a.dt_disp / 2.);
      const double sn = sin(nOmega * a.dt_disp / 2.);
      dq = qmk(scl(avg, sn * 1. / nOmega), cc);
    } else {
      dq = qmk(mk(0., 0., 0.), 1.);
    }
    q = qmul(dq, q);
    const double depl = norm(dx);
    drift = depl;
    // the record (id, crust) is read only when the drift may exceed a crust
    if (depl > a.crust_min) {
      const Aux ax = vw.kin.aux[s];
      if (depl > ax.crust) atomicMin(&a.err[kErrMotion], (unsigned long long)(uint32_t)ax.id);
    }
    // every axis is wrapped (no short-circuit)
    const bool in0 = wrap_axis(a, 0, Xo.x);
    const bool in1 = wrap_axis(a, 1, Xo.y);
    const bool in2 = wrap_axis(a, 2, Xo.z);
    const bool inside = in0 && in1 && in2;
    if (!inside) {
      int ijk[3];
      if (!cell_of(a.grid, Xo, ijk))
        atomicMin(&a.err[kErrSim], (unsigned long long)(uint32_t)vw.kin.aux[s].id);
    }
  }
  // streaming stores: the new copy would otherwise sit dirty in the L2s
  // until the kernel's end (measured: 5 us per step less at 1M particles)
  const Pack& out = vw.out;
  typedef double nd4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store((nd4){Xo.x, Xo.y, Xo.z, q.v.x}, reinterpret_cast<nd4*>(out.A + t));
  __builtin_nontemporal_store((nd4){Vo.x, Vo.y, Vo.z, q.v.y}, reinterpret_cast<nd4*>(out.B + t));
  if (store_w)
    __builtin_nontemporal_store((nd4){Wo.x, Wo.y, Wo.z, 0.}, reinterpret_cast<nd4*>(out.C + t));
  __builtin_nontemporal_store((nd4){WBF.x, WBF.y, WBF.z, q.v.z}, reinterpret_cast<nd4*>(out.D + t));
  __builtin_nontemporal_store(q.w, out.E + t);
  // path length since the rebuild; need flag of the next step (StepWords)
  len = mine;
  if (!last || rebuild) {
    len = skin_path(mine, rebuild, drift);
    if (len > a.limit) atomicOr(&a.w->slot[j_out].need, 1);
  }
  vw.path_out[t] = len;
  if (vw.copy_const) {
    vw.kout.rr[t] = vw.kin.rr[s];
    vw.kout.mi[t] = st.mi;
    vw.kout.aux[t] = vw.kin.aux[s];
  }
}

// Stages the walls' grown-box test data (bounding box centre and extent) in
// LDS; a barrier has to follow.
template <int BS>
__device__ __forceinline__ void stage_walls(const StepArgs& a, double* bb) {
  for (int k = threadIdx.x; k < 6 * a.nwalls; k += BS) {
    const Wall& wl = a.walls[k / 6];
    const int d = k % 6;
    bb[k] = d < 3 ? wl.bb_centre[d] : wl.bb_ext[d - 3];
  }
}

// Walls whose bounding box grown by r holds X (SimpleObstacle::InterAction's
// InZone test, Component/src/SimpleObstacle.cpp:222-271), as a bit mask.
__device__ __forceinline__ unsigned long long near_walls(const double* bb, int nwalls, v3 X,
                                                         double r) {
  unsigned long long wm = 0ull;
  for (int wi = 0; wi < nwalls; ++wi, bb += 6)
    if (fabs(bb[0] - X.x) <= bb[3] + r && fabs(bb[1] - X.y) <= bb[4] + r &&
        fabs(bb[2] - X.z) <= bb[5] + r)
      wm |= 1ull << wi;
  return wm;
}

// LDS of the contact evaluation of a workgroup of BS lanes.
template <int BS>
struct ContactLds {
  int wave[BS / 64];
  uint8_t part[BS], code[BS], hit[BS];
  int slot[BS];
  double rec[6][BS];
};

// Force and torque of the contacts of a workgroup's particles: lane k < PP
// brings particle t (masks cm, wm of the candidates and walls that may touch;
// lanes without a particle bring none) and gets its sums added to F and T.
// The pairs are queued in LDS, evaluated one per lane in rounds of BS, and each
// particle adds its own in queue order: candidates in the order of summation,
// then walls.  nc counts the contacts, each pair at its out entry.  Every lane
// of the workgroup calls.
template <int BS, bool WALLS>
__device__ __forceinline__ void gather_contacts(const StepArgs& a, const StepView& vw,
                                                ContactLds<BS>& sh, int t,
                                                unsigned long long cm, unsigned long long wm,
                                                v3& F, v3& T, int& nc) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int cnt = __popcll(cm) + (WALLS ? __popcll(wm) : 0);
  int incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) sh.wave[wid] = incl;
  sh.slot[threadIdx.x] = t;
  __syncthreads();
  int next = incl - cnt, nq = 0;  // next: queue position of the next contact
#pragma unroll
  for (int w = 0; w < BS / 64; ++w) {
    if (w < wid) next += sh.wave[w];
    nq += sh.wave[w];
  }
  const int end = next + cnt;
  for (int q0 = 0; q0 < nq; q0 += BS) {
    int pos = next;
    while (pos < end && pos < q0 + BS) {
      int code;
      if (!WALLS || cm) {
        code = __ffsll((long long)cm) - 1;
        cm &= cm - 1ull;
      } else {
        code = 64 + (__ffsll((long long)wm) - 1);
        wm &= wm - 1ull;
      }
      sh.part[pos - q0] = (uint8_t)threadIdx.x;
      sh.code[pos - q0] = (uint8_t)code;
      ++pos;
    }
    __syncthreads();
    if (q0 + (int)threadIdx.x < nq) {
      const int code = sh.code[threadIdx.x];
      const int tt = sh.slot[sh.part[threadIdx.x]];
      const int ss = vw.rebuild ? a.perm[tt] : tt;
      v3 f = mk(0., 0., 0.), tq = f;
      bool hit;
      if (!WALLS || code < 64) {
        const int nout = min(a.out_count[tt], kListCap);
        const int2 en = code < nout ? a.out_list[(size_t)code * a.lstride + tt]
                                    : a.in_list[(size_t)(code - nout) * a.lstride + tt];
        const int su = vw.rebuild ? a.perm[en.x] : en.x;
        const bool first = (en.y & 64) != 0;
        const double4 c1 = vw.in.C[ss], c2 = vw.in.C[su];
        v3 fA, ta, tb;
        hit = pair_contact(a, vw.in, vw.kin, ss, su, first, mk(c1.x, c1.y, c1.z),
                           mk(c2.x, c2.y, c2.z), fA, ta, tb);
        if (hit) {
          f = first ? fA : neg(fA);
          tq = first ? ta : tb;
        }
        nc += hit && code < nout;
      } else {
        const double4 c = vw.in.C[ss];
        hit = wall_contact(a, vw.in, vw.kin, ss, code - 64, mk(c.x, c.y, c.z), f, tq);
        nc += hit;
      }
      sh.hit[threadIdx.x] = hit;
      sh.rec[0][threadIdx.x] = f.x;
      sh.rec[1][threadIdx.x] = f.y;
      sh.rec[2][threadIdx.x] = f.z;
      sh.rec[3][threadIdx.x] = tq.x;
      sh.rec[4][threadIdx.x] = tq.y;
      sh.rec[5][threadIdx.x] = tq.z;
    }
    __syncthreads();
    for (; next < pos; ++next) {
      const int k = next - q0;
      if (!sh.hit[k]) continue;
      F = add(F, mk(sh.rec[0][k], sh.rec[1][k], sh.rec[2][k]));
      T = add(T, mk(sh.rec[3][k], sh.rec[4][k], sh.rec[5][k]));
    }
    __syncthreads();
  }
}

// Adds the contacts counted by a workgroup's lanes to its slot (no atomics).
template <int BS>
__device__ __forceinline__ void count_contacts(const StepArgs& a, int* sh_wave, int nc) {
  for (int o = 32; o > 0; o >>= 1) nc += __shfl_xor(nc, o, 64);
  if ((threadIdx.x & 63) == 0) sh_wave[threadIdx.x >> 6] = nc;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long tot = 0;
    for (int w = 0; w < BS / 64; ++w) tot += (unsigned long long)sh_wave[w];
    if (tot) a.contacts[blockIdx.x] += tot;
  }
}

// One step of fewer than kStepSmall particles in one kernel.  A workgroup of
// BS lanes steps PP particles: BS / PP lanes screen the lists of one particle
// together, all BS lanes evaluate the queued contacts, and the first lane of
// each particle sums and integrates.  after: a rebuild was offered right
// before this launch.
template <int BS, int PP, bool WALLS>
__global__ void __launch_bounds__(BS) k_step(StepArgs a, int j_in, int j_out, int after) {
  constexpr int L = BS / PP;  // lanes per particle
  __shared__ ContactLds<BS> sh;
  __shared__ unsigned long long sh_may[PP];
  __shared__ double sh_bb[WALLS ? 6 * kMaxWalls : 1];
  StepSlot sl;
  StepView vw;
  const bool go = step_view(a, j_in, after, sl, vw);
  step_done(a, j_in, j_out, sl, go, true);
  if (!go) return;
  if (WALLS) stage_walls<BS>(a, sh_bb);
  // PP consecutive slots per workgroup, XCD-aware as logical_index
  const int part = threadIdx.x % PP, sub = threadIdx.x / PP;
  const int t = ((blockIdx.x & 7) * (a.nblk8 >> 3) + (blockIdx.x >> 3)) * PP + part;
  const bool live = t < a.n;
  const bool own = live && sub == 0;  // this lane sums and integrates particle t
  const int s = live ? (vw.rebuild ? a.perm[t] : t) : 0;
  float mine = 0.f;
  v3 X = mk(0., 0., 0.);
  double r = 0.;
  if (threadIdx.x < PP) sh_may[threadIdx.x] = 0ull;
  __syncthreads();  // the masks and the wall boxes
  if (live) {
    const double4 A4 = vw.in.A[s];
    X = mk(A4.x, A4.y, A4.z);
    r = vw.kin.rr[s].x;
    if (!vw.rebuild) mine = vw.path[t];
    const unsigned long long may = screen_particle<L>(a, vw, t, X, r, mine, sub);
    if (may) atomicOr(&sh_may[part], may);
  }
  __syncthreads();
  v3 F = mk(0., 0., 0.), T = F;
  if (own) F = weight(a, vw.kin.mi[s].x);
  int nc = 0;
  gather_contacts<BS, WALLS>(a, vw, sh, t, own ? sh_may[part] : 0ull,
                             WALLS && own ? near_walls(sh_bb, a.nwalls, X, r) : 0ull, F, T, nc);
  count_contacts<BS>(a, sh.wave, nc);
  float len = 0.f;
  if (own) finish_particle(a, vw, load_state(vw, s), t, s, mine, F, T, j_out, true, len);
  wave_path(len, a.path_rows, j_out);
}

// One step of many particles in two kernels.
//
// k_pairs: a workgroup takes `per` times kPB particles.  Path length and
// smallest gap bound decide for most of them; the others are compacted in LDS
// and screened one per lane, and the pairs that may touch are queued in LDS
// and evaluated once, one per lane.  A contact stores its record at the out
// entry, flags it in the particle's out mask and its mirror entry in the
// partner's in mask (integer OR).  The kernel is a chain of latencies, so the
// grid should be resident at once and a workgroup's contacts should fill one
// round of lanes: per is the smaller of the particles per resident workgroup
// and the particles that hold kPB contacts (by the touching candidates of
// the last build); the workgroups that are then not needed exit.
__global__ void __launch_bounds__(kPB) k_pairs(StepArgs a, int j_in, int after) {
  constexpr int N = kPairPer * kPB;
  __shared__ int sh_near, sh_wave[kPB / 64];
  __shared__ uint16_t sh_part[N];  // particles to screen
  __shared__ uint32_t sh_may[N];   // their candidates that may touch
  __shared__ uint32_t sh_om[N];
  __shared__ uint16_t sh_item[kPB];
  __shared__ uint8_t sh_code[kPB];
  StepSlot sl;
  StepView vw;
  if (!step_view(a, j_in, after, sl, vw)) return;
  int touch = *row_word(a.path_rows, kTouchRow, threadIdx.x & 63);
  for (int o = 32; o > 0; o >>= 1) touch += __shfl_xor(touch, o, 64);
  const int fill = touch > 0 ? (int)min((long long)kPairPer, (long long)a.n / touch) : kPairPer;
  const int per = max(1, min(fill, a.n / (kPairGrid * kPB)));
  const int blocks8 = ((a.n + per * kPB - 1) / (per * kPB) + 7) / 8 * 8;
  if ((int)blockIdx.x >= blocks8) return;
  const int t0 = ((blockIdx.x & 7) * (blocks8 >> 3) + (blockIdx.x >> 3)) * (per * kPB);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (threadIdx.x == 0) sh_near = 0;
  __syncthreads();
  for (int q = 0; q < per; ++q) {
    const int t = t0 + q * kPB + threadIdx.x;
    bool near = false;
    if (t < a.n) near = a.min_gap[t] <= (vw.rebuild ? 0.f : vw.path[t]) + vw.far;
    sh_om[q * kPB + threadIdx.x] = 0u;
    const unsigned long long who = __ballot(near);
    if (!who) continue;
    int base = 0;
    if (lane == 0) base = atomicAdd(&sh_near, __popcll(who));
    base = __shfl(base, 0, 64);
    if (near)
      sh_part[base + __popcll(who & ((1ull << lane) - 1ull))] = (uint16_t)(q * kPB + threadIdx.x);
  }
  __syncthreads();
  const int nnear = sh_near;
  int cnt = 0;  // candidates of this lane's particles k = threadIdx.x, + kPB, ...
  for (int k = threadIdx.x; k < nnear; k += kPB) {
    const int t = t0 + sh_part[k];
    const int s = vw.rebuild ? a.perm[t] : t;
    const double4 A4 = vw.in.A[s];
    const uint32_t may =
        (uint32_t)screen_particle<1>(a, vw, t, mk(A4.x, A4.y, A4.z), vw.kin.rr[s].x,
                                     vw.rebuild ? 0.f : vw.path[t], 0);
    sh_may[k] = may;
    cnt += __builtin_popcount(may);
  }
  int incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) sh_wave[wid] = incl;
  __syncthreads();
  int next = incl - cnt, nq = 0;  // next: queue position of this lane's next pair
#pragma unroll
  for (int w = 0; w < kPB / 64; ++w) {
    if (w < wid) next += sh_wave[w];
    nq += sh_wave[w];
  }
  int nc = 0, k = threadIdx.x;
  uint32_t may = k < nnear ? sh_may[k] : 0u;
  // rounds of kPB queued pairs
  for (int q0 = 0; q0 < nq; q0 += kPB) {
    while (next < q0 + kPB) {
      while (!may && (k += kPB) < nnear) may = sh_may[k];
      if (!may) break;
      sh_item[next - q0] = sh_part[k];
      sh_code[next - q0] = (uint8_t)__builtin_ctz(may);
      may &= may - 1u;
      ++next;
    }
    __syncthreads();
    if (q0 + (int)threadIdx.x < nq) {
      const int at = sh_item[threadIdx.x], e = sh_code[threadIdx.x];
      const int t = t0 + at;
      const int s = vw.rebuild ? a.perm[t] : t;
      const int2 en = a.out_list[(size_t)e * a.lstride + t];
      const int su = vw.rebuild ? a.perm[en.x] : en.x;
      v3 W, W2;
      if (vw.wstored) {
        const double4 c = vw.in.C[s], c2 = vw.in.C[su];
        W = mk(c.x, c.y, c.z);
        W2 = mk(c2.x, c2.y, c2.z);
      } else {
        // never on a rebuild: its first kernel stores them
        W = world_omega(vw.in, vw.out, s, vw.moved ? a.perm[s] : s);
        W2 = world_omega(vw.in, vw.out, su, vw.moved ? a.perm[su] : su);
      }
      v3 f, ta, tb;
      if (pair_contact(a, vw.in, vw.kin, s, su, (en.y & 64) != 0, W, W2, f, ta, tb)) {
        PairRec& r = a.rec[(size_t)e * a.lstride + t];
        r.f[0] = f.x; r.f[1] = f.y; r.f[2] = f.z;
        r.ta[0] = ta.x; r.ta[1] = ta.y; r.ta[2] = ta.z;
        r.tb[0] = tb.x; r.tb[1] = tb.y; r.tb[2] = tb.z;
        atomicOr(&sh_om[at], 1u << e);
        const int fi = (en.y >> 7) & 31;  // the mirror entry in the partner's in-list
        if (fi < kListCap) atomicOr(&a.imask[en.x], 1u << fi);
        ++nc;
      }
    }
    __syncthreads();
  }
  if (nq) count_contacts<kPB>(a, sh_wave, nc);
  for (int q = 0; q < per; ++q) {
    const int t = t0 + q * kPB + threadIdx.x;
    if (t < a.n) a.omask[t] = sh_om[q * kPB + threadIdx.x];
  }
}

// Adds one stored pair record to the body it belongs to.
__device__ __forceinline__ void add_record(const PairRec& R, bool first, v3& F, v3& T) {
  const v3 f = mk(R.f[0], R.f[1], R.f[2]);
  if (first) {
    F = add(F, f);
    T = add(T, mk(R.ta[0], R.ta[1], R.ta[2]));
  } else {
    F = add(F, neg(f));
    T = add(T, mk(R.tb[0], R.tb[1], R.tb[2]));
  }
}

// k_integ: each particle sums its flagged records in the fixed order, adds
// the walls and integrates.  HBM bound (it streams the state).  A step
// without walls leaves the world angular velocity to be derived
// (world_omega): 24 B per particle neither read nor written here.
template <bool WALLS>
__global__ void __launch_bounds__(kPB) k_integ(StepArgs a, int j_in, int j_out, int after) {
  __shared__ int sh_wave[kPB / 64];
  __shared__ double sh_bb[WALLS ? 6 * kMaxWalls : 1];
  StepSlot sl;
  StepView vw;
  const bool go = step_view(a, j_in, after, sl, vw);
  const bool store_w = WALLS || vw.last;
  step_done(a, j_in, j_out, sl, go, store_w);
  if (!go) return;
  if (WALLS) {
    stage_walls<kPB>(a, sh_bb);
    __syncthreads();
  }
  const int t = logical_index(a.nblk8);
  float len = 0.f;
  int nwc = 0;
  if (t < a.n) {
    const int s = vw.rebuild ? a.perm[t] : t;
    const StepState st = load_state(vw, s);
    const float mine = vw.rebuild ? 0.f : vw.path[t];
    const uint32_t om = a.omask[t], im = a.imask[t];
    v3 F = weight(a, st.mi.x), T = mk(0., 0., 0.);
    // contact segment: detected contacts by entry, then received contacts in
    // the order (partner slot, code, position)
    for (uint32_t mm = om; mm != 0u; mm &= mm - 1u) {
      const size_t at = (size_t)__builtin_ctz(mm) * a.lstride + t;
      add_record(a.rec[at], (a.out_list[at].y & 64) != 0, F, T);
    }
    if (im != 0u) {
      a.imask[t] = 0u;  // ready for the next pair kernel
      const int nin = min(a.in_count[t], kListCap);
      const int2* il = a.in_list + t;
      long long last = -1;
      const int nlive = __builtin_popcount(im);
      for (int k = 0; k < nlive; ++k) {
        long long key;
        const int f = next_incoming(il, nin, a.lstride, last, key, im);
        if (f < 0) break;
        const int2 en = il[(size_t)f * a.lstride];
        const int e = (en.y >> 7) & 31;
        if (e < kListCap)
          add_record(a.rec[(size_t)e * a.lstride + en.x], (en.y & 64) != 0, F, T);
        last = key;
      }
    }
    if (WALLS) {
      const v3 X = mk(st.A.x, st.A.y, st.A.z);
      unsigned long long wm = near_walls(sh_bb, a.nwalls, X, vw.kin.rr[s].x);
      for (; wm != 0ull; wm &= wm - 1ull) {
        const double4 c = vw.in.C[s];  // with walls every step stores it
        v3 f, tq;
        if (wall_contact(a, vw.in, vw.kin, s, __ffsll((long long)wm) - 1, mk(c.x, c.y, c.z), f,
                         tq)) {
          F = add(F, f);
          T = add(T, tq);
          ++nwc;
        }
      }
    }
    finish_particle(a, vw, st, t, s, mine, F, T, j_out, store_w, len);
  }
  wave_path(len, a.path_rows, j_out);
  if (WALLS) count_contacts<kPB>(a, sh_wave, nwc);
}

// Kick + drift of copy pk in place (SecondOrderLeapFrog::Move via
// ParticleKinematics::Move), from the stored F and T (the opening half of a
// step sequence).
__global__ void __launch_bounds__(kPB) k_move_pack(Pack pk, PackConst k, const double4* Fa,
                                                   const double4* Ta, int n, Grid g, double dtv,
                                                   double dtd, unsigned long long* err,
                                                   float limit, float* path, StepWords* w,
                                                   int32_t* path_rows, int p, int32_t nsteps) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double depl = 0.;
  float far = 0.f;
  if (i == 0) {
    // the step sequence of this call: nsteps steps from copy p
    w->slot[kChunkSteps].done = 0;
    w->slot[kChunkSteps].cur = p;
    w->slot[kChunkSteps].wstored = 1;
    w->target = nsteps;
    w->chunks = 0;
    w->rebuilds = 0;
  }
  if (i < n) {
    const double4 A4 = pk.A[i], B4 = pk.B[i], D4 = pk.D[i];
    const double2 mi = k.mi[i];
    const double4 f4 = Fa[i], t4 = Ta[i];
    const v3 F = mk(f4.x, f4.y, f4.z), T = mk(t4.x, t4.y, t4.z);
    quat q = qmk(mk(A4.w, B4.w, D4.w), pk.E[i]);
    const quat pc = qconj(q);
    const v3 tq = qmulv(pc, qleftvec(q, T));
    const double mcf = mi.x * 1.;
    const v3 V = add(mk(B4.x, B4.y, B4.z), scl(dvd(F, mcf), dtv));
    const v3 dx = scl(V, dtd);
    const v3 WBF = ssprk3_sphere(tq, mk(D4.x, D4.y, D4.z), mi.y, dtv);
    const v3 W = qmulv(q, qleftvec(pc, WBF));
    const v3 avg = W;
    v3 X = add(mk(A4.x, A4.y, A4.z), dx);
    const double nOmega = norm(avg);
    quat dq;
    if (nOmega > kEps) {
      const double cc = cos(nOmega * dtd / 2.);
      const double sn = sin(nOmega * dtd / 2.);
      dq = qmk(scl(avg, sn * 1. / nOmega), cc);
    } else {
      dq = qmk(mk(0., 0., 0.), 1.);
    }
    q = qmul(dq, q);
    depl = norm(dx);
    const Aux ax = k.aux[i];
    if (depl > ax.crust) atomicMin(&err[kErrMotion], (unsigned long long)(uint32_t)ax.id);
    double xo[3] = {X.x, X.y, X.z};
    for (int d = 0; d < 3; ++d) {
      if (!g.periodic[d]) continue;
      const double lo = g.origin[d], L = g.size[d];
      if (xo[d] >= lo + L) xo[d] -= L;
      else if (xo[d] < lo) xo[d] += L;
    }
    X = mk(xo[0], xo[1], xo[2]);
    int ijk[3];
    if (!cell_of(g, X, ijk)) atomicMin(&err[kErrSim], (unsigned long long)(uint32_t)ax.id);
    pk.A[i] = make_double4(X.x, X.y, X.z, q.v.x);
    pk.B[i] = make_double4(V.x, V.y, V.z, q.v.y);
    pk.C[i] = make_double4(W.x, W.y, W.z, 0.);
    pk.D[i] = make_double4(WBF.x, WBF.y, WBF.z, q.v.z);
    pk.E[i] = q.w;
    const float len = skin_path(path[i], false, depl);
    path[i] = len;
    far = len;
    if (len > limit) atomicOr(&w->slot[kChunkSteps].need, 1);
  }
  wave_path(far, path_rows, kChunkSteps);
}

// ---------------------------------------------------------------- launchers
void launch_to_pack(const State& s, const Pack& pk, const PackConst& k0, const PackConst& k1,
                    const StepLists& l, const SkinWords* words, float* path, const float* path_in,
                    int p, int32_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_step_words, dim3(1), dim3(kRowSegs), 0, st, l.words,
                     l.path_rows, words, p);
  hipLaunchKernelGGL(k_to_pack, dim3(pblocks(std::max(n, 1))), dim3(kPB), 0, st, s, pk, k0, k1, l,
                     path, path_in, n);
}

void launch_from_pack(const Pack& pk, const PackConst& k, const State& s, float* path_out,
                      const float* path, const StepWords* w, SkinWords* words, int p, int32_t n,
                      hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_from_pack, dim3(pblocks(n)), dim3(kPB), 0, st, pk, k, s, path_out, path, w,
                     words, p, n);
}

void launch_pack_rebuild(const Bins& b, const PosSrc& src0, const PosSrc& src1, StepWords* w,
                         SkinWords* words, const DetectArgs& d, const StepLists& l,
                         const Pack& pk0, const Pack& pk1, hipStream_t st) {
  // grids this size exit in a microsecond or two when no rebuild is due
  const dim3 block(kPB), grid(std::min(pblocks(d.n), 1024));
  const int32_t ncell = d.grid.ncell;
  hipLaunchKernelGGL(k_pk_count, grid, block, 0, st, b, src0, src1, pk0, pk1, w, l.path_rows, words,
                     d.in_count, d.n, d.grid, d.row_rank, d.err);
  launch_scan(b, ncell, d.gate, st);
  hipLaunchKernelGGL(k_pk_scatter, grid, block, 0, st, b, w, d.gate, d.n, l.path_rows);
  hipLaunchKernelGGL(k_pk_cellsort, dim3(std::min(pblocks(ncell), 1024)), block, 0, st, b, src0,
                     src1, d.gate, ncell, d.n);
  const dim3 sweep(std::min(d.nblk8, 2048));
  if (l.both) {
    hipLaunchKernelGGL(k_pk_sweep<false>, sweep, block, 0, st, d, src0, src1, l);
    hipLaunchKernelGGL(k_pk_lists, grid, block, 0, st, l, d.gate, d.n);
  } else {
    hipLaunchKernelGGL(k_pk_sweep<true>, sweep, block, 0, st, d, src0, src1, l);
  }
}

bool step_in_one(int32_t n) { return n < kStepSmall; }

int step_particles(int32_t n) {
  return n < 32768 ? 64 : n < 65536 ? 128 : kPB;
}

template <int PP, bool WALLS>
static void one_launch(const StepArgs& a, int j_in, int j_out, int after, hipStream_t st,
                       hipEvent_t start, hipEvent_t stop) {
  const dim3 grid(a.nblk8), block(kPB);
  if (start)
    hipExtLaunchKernelGGL((k_step<kPB, PP, WALLS>), grid, block, 0, st, start, stop, 0, a, j_in,
                          j_out, after);
  else
    hipLaunchKernelGGL((k_step<kPB, PP, WALLS>), grid, block, 0, st, a, j_in, j_out, after);
}

template <bool WALLS>
static void step_launch(const StepArgs& a, int j_in, int j_out, int after, hipStream_t st,
                        hipEvent_t start, hipEvent_t stop, hipEvent_t start1, hipEvent_t stop1) {
  if (step_in_one(a.n)) {
    const int pp = step_particles(a.n);
    if (pp == 64) one_launch<64, WALLS>(a, j_in, j_out, after, st, start, stop);
    else if (pp == 128) one_launch<128, WALLS>(a, j_in, j_out, after, st, start, stop);
    else one_launch<kPB, WALLS>(a, j_in, j_out, after, st, start, stop);
    return;
  }
  const dim3 pgrid(a.nblk8), grid(a.nblk8), block(kPB);
  if (start) {
    hipExtLaunchKernelGGL(k_pairs, pgrid, block, 0, st, start1, stop1, 0, a, j_in, after);
    hipExtLaunchKernelGGL(k_integ<WALLS>, grid, block, 0, st, start, stop, 0, a, j_in, j_out,
                          after);
  } else {
    hipLaunchKernelGGL(k_pairs, pgrid, block, 0, st, a, j_in, after);
    hipLaunchKernelGGL(k_integ<WALLS>, grid, block, 0, st, a, j_in, j_out, after);
  }
}

void launch_step(const StepArgs& a, int j_in, int j_out, bool after, hipStream_t st,
                 hipEvent_t start, hipEvent_t stop, hipEvent_t start1, hipEvent_t stop1) {
  if (a.n <= 0) return;
  if (a.nwalls > 0) step_launch<true>(a, j_in, j_out, after, st, start, stop, start1, stop1);
  else step_launch<false>(a, j_in, j_out, after, st, start, stop, start1, stop1);
}

void launch_move_pack(const Pack& pk, const PackConst& k, const double4* F, const double4* T,
                      int32_t n, const Grid& g, double dt_vel, double dt_disp,
                      unsigned long long* err, float limit, float* path, StepWords* w,
                      int32_t* path_rows, int p, int32_t nsteps, hipStream_t st) {
  hipLaunchKernelGGL(k_move_pack, dim3(pblocks(std::max(n, 1))), dim3(kPB), 0, st, pk, k, F, T, n,
                     g, dt_vel, dt_disp, err, limit, path, w, path_rows, p, nsteps);
}

}  // namespace gdem
