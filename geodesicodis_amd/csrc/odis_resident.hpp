// odis_resident.hpp -- many steps per launch with the ocean held on the chip.
//
// k_resident advances one or more instances `count` steps in one launch.  An
// instance's cells are split into W compact patches, one workgroup per (instance, patch), all workgroups resident at
// once.  A workgroup loads the operators and the state of its patch once --
// velocities, histories and operators of its faces and cells in registers,
// the values that neighbouring lanes read (signed fluxes, TRiSK partial
// sums, heights, tide) in LDS -- and writes the state back after the last
// step.  Between steps only the patch boundary leaves the CU: for every face
// shared by two patches each side sends the other its cell's TRiSK partial
// sum and its cell's height.  Both sides update a shared face identically,
// as the patches of k_step do, so the state is the same bit for bit.
//
// Why: a step launched by itself reads and writes everything (128 B per face
// and per cell in FP64) and pays a launch; at 163842 cells that is 20 us, at
// 10242 cells 5.9 us, nearly all of it launch and memory latency.  Held on
// the chip (256 CUs with 512 KB of registers and 160 KB of LDS each), a step
// costs its arithmetic and one exchange with the neighbouring patches.
// Measured, us per step of long runs, one launch per step -> resident:
//   642 cells FP64 5.8 -> 2.8;  10242 FP64 5.9 -> 2.5, FP32 5.5 -> 2.4
//   40962 FP64 8.4 -> 3.2, FP32 6.9 -> 2.6
//   163842 FP64 21.1 -> 4.2, FP32 14.2 -> 2.9
//   256 x 40962 FP32 437 (k_step_il) -> 174;  23 x 10242 FP64 25.6 -> 7.5
// What bounds it now: at small patches the exchange (about 2 us from a
// cell's send to the neighbour's look that sees it), at 641 cells per patch
// that and the FP64 vector units (about 1.5 us of issue per step).
//
// Exchange: an inbox slot per (patch, boundary face).  Each 8-byte word
// carries 4 bytes of data and the 32-bit sequence number of the message,
// written and polled past the L2 (agent scope), so a word that shows the
// awaited number holds the awaited data and nothing else needs ordering or
// flushing.  Message k + 2 is only sent after the receiver's message
// k + 1 was received, which the receiver sent after reading message k; at a
// change of instance (no message after the last step of one, none needed
// before the first of the next) a sender is one message further ahead.  So
// a slot keeps kResDepth messages, by sequence number.
//
// A batch larger than the chip holds at once runs ipl instances at a time,
// each for all the steps, inside one launch: the operators stay in registers
// from one instance to the next.
//
// Progress: workgroups wait for each other, so all of them must be on the
// chip.  The grid is no larger than what the chip holds, resident launches of
// one process that would not fit together follow one another, and the first thing a launch does is to count
// its workgroups in: until the count is complete nothing has been written,
// and if it is not complete in time (another process holds the CUs) one
// workgroup takes the launch back -- one atomic word decides between
// "complete" and "taken back" -- and every workgroup leaves.  The host then
// steps the same steps with one launch each.  After the count every
// workgroup stays on the chip and every wait ends; each wait is bounded by
// time all the same.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <future>
#include <string>
#include <system_error>
#include <type_traits>
#include <vector>

#include "odis_kernels.hpp"

namespace odis {

constexpr int kResDepth = 4;               // messages an inbox slot holds (by sequence number)
constexpr unsigned kResFailed = 0xffffffffu;
constexpr int kResEn = 8;                  // steps whose dissipation integrands are kept before they are summed
constexpr unsigned long long kResTaken = 1ull << 63;   // bit of the arrival word: launch taken back
constexpr long long kResArriveTicks = 20000000;        // 0.2 s of the 100 MHz wall clock
constexpr long long kResWaitTicks = 1000000000;        // 10 s

// Patches of the resident step, cells and faces regrouped by patch:
// a patch's cells with a boundary face first, its faces with both cells in
// the patch ("inner") first, then the boundary faces.
struct ResHost {
  int W = 0;                                 // patches per instance
  int max_cells = 0, max_face = 0, max_bnd = 0;  // of a patch; faces: inner + boundary
  std::vector<int> cptr, fptr, bptr;         // [W + 1] cells; inner faces; boundary faces (slots)
  std::vector<int> cell;                     // [N] device cell
  std::vector<int> face;                     // [inner faces] device face
  std::vector<int> fcell;                    // [inner faces] local cells c0 | c1 << 16
  std::vector<int> bface;                    // [slots] device face
  std::vector<int> bcell;                    // [slots] own local cell | own side << 16 | owner << 17
  std::vector<int> bhalo;                    // [slots] device cell across the face
  std::vector<int> bpeer;                    // [slots] slot of the same face in the other patch
  std::vector<unsigned short> cyc;           // [6][N] by position in `cell`: local faces (inner, then boundary)
};

// pt[cptr[j] .. cptr[j + 1]): the cells of patch j, by recursive bisection of
// the cells along the longest axis of their box.  Compact patches: 640 cells
// have about 210 boundary faces.
struct ResPoint {
  float x[3];
  int cell;
};
inline void bisect_cells(ResPoint *pt, int lo, int hi, int j, int W, std::vector<int> &cptr) {
  if (W == 1) {
    std::sort(pt + lo, pt + hi, [](const ResPoint &p, const ResPoint &q) { return p.cell < q.cell; });
    cptr[j + 1] = hi;
    return;
  }
  float mn[3] = {2, 2, 2}, mx[3] = {-2, -2, -2};
  for (int p = lo; p < hi; p++)
    for (int d = 0; d < 3; d++) {
      mn[d] = std::min(mn[d], pt[p].x[d]);
      mx[d] = std::max(mx[d], pt[p].x[d]);
    }
  int ax = 0;
  for (int d = 1; d < 3; d++)
    if (mx[d] - mn[d] > mx[ax] - mn[ax]) ax = d;
  const int W0 = W / 2, mid = lo + int((long long)(hi - lo) * W0 / W);
  std::nth_element(pt + lo, pt + mid, pt + hi, [ax](const ResPoint &p, const ResPoint &q) {
    return p.x[ax] < q.x[ax] || (p.x[ax] == q.x[ax] && p.cell < q.cell);
  });
  // the halves in parallel on large grids (each writes its own points and ends)
  std::future<void> other;
  if (hi - lo > 16384) {
    try {
      other = std::async(std::launch::async, [=, &cptr] { bisect_cells(pt, lo, mid, j, W0, cptr); });
    } catch (const std::system_error &) {  // no thread to be had: one after the other
    }
  }
  if (!other.valid()) bisect_cells(pt, lo, mid, j, W0, cptr);
  bisect_cells(pt, mid, hi, j + W0, W - W0, cptr);
  if (other.valid()) other.get();
}

// W patches over N cells at xyz[N][3]; gi[2][E] cells of each face, cyc[6][N] face cycle
// of each cell (device order, faces sorted by their lower cell).  Empty
// string on success.
inline std::string build_resident(int N, int E, const std::vector<float> &xyz, const std::vector<int> &gi,
                                  const std::vector<int> &cyc, int W, ResHost &h) {
  h.W = W;
  for (float x : xyz)
    if (!std::isfinite(x)) return "a cell without a place";
  h.cptr.assign(W + 1, 0);
  std::vector<int> patch(N);
  std::vector<ResPoint> pt(N);
  for (int c = 0; c < N; c++)
    pt[c] = {{xyz[size_t(3) * c], xyz[size_t(3) * c + 1], xyz[size_t(3) * c + 2]}, c};
  bisect_cells(pt.data(), 0, N, 0, W, h.cptr);
  for (int j = 0; j < W; j++)
    for (int p = h.cptr[j]; p < h.cptr[j + 1]; p++) patch[pt[p].cell] = j;
  std::vector<int> n_in(W, 0), n_bd(W, 0);
  std::vector<char> edge(N, 0);
  for (int f = 0; f < E; f++) {
    const int a = gi[f], b = gi[size_t(E) + f];
    if (a == b) return "a face with one cell";
    if (patch[a] == patch[b]) {
      n_in[patch[a]]++;
    } else {
      n_bd[patch[a]]++;
      n_bd[patch[b]]++;
      edge[a] = edge[b] = 1;
    }
  }
  h.fptr.assign(W + 1, 0);
  h.bptr.assign(W + 1, 0);
  h.max_cells = h.max_face = h.max_bnd = 0;
  for (int j = 0; j < W; j++) {
    if (n_in[j] < 1) return "a patch without inner faces";
    h.fptr[j + 1] = h.fptr[j] + n_in[j];
    h.bptr[j + 1] = h.bptr[j] + n_bd[j];
    h.max_cells = std::max(h.max_cells, h.cptr[j + 1] - h.cptr[j]);
    h.max_face = std::max(h.max_face, n_in[j] + n_bd[j]);
    h.max_bnd = std::max(h.max_bnd, n_bd[j]);
  }
  if (h.max_cells > 32767 || h.max_face > 65535) return "patch too large for its local indices";
  h.cell.resize(N);
  std::vector<int> loc(N);
  for (int j = 0; j < W; j++) {
    int p = h.cptr[j];
    for (int pass = 0; pass < 2; pass++)
      for (int k = h.cptr[j]; k < h.cptr[j + 1]; k++) {
        const int c = pt[k].cell;
        if (edge[c] != (pass == 0)) continue;
        loc[c] = p - h.cptr[j];
        h.cell[p++] = c;
      }
  }
  h.face.resize(h.fptr[W]);
  h.fcell.resize(h.fptr[W]);
  const int S = h.bptr[W];
  h.bface.resize(S);
  h.bcell.resize(S);
  h.bhalo.resize(S);
  h.bpeer.resize(S);
  std::vector<int> fi(h.fptr.begin(), h.fptr.end() - 1), bi(h.bptr.begin(), h.bptr.end() - 1);
  // local face of each side of a face
  std::vector<unsigned short> lside(size_t(2) * E);
  for (int f = 0; f < E; f++) {
    const int a = gi[f], b = gi[size_t(E) + f], pa = patch[a], pb = patch[b];
    if (pa == pb) {
      const int q = fi[pa]++;
      h.face[q] = f;
      h.fcell[q] = loc[a] | (loc[b] << 16);
      lside[2 * size_t(f)] = lside[2 * size_t(f) + 1] = (unsigned short)(q - h.fptr[pa]);
    } else {
      const int sa = bi[pa]++, sb = bi[pb]++;
      h.bface[sa] = h.bface[sb] = f;
      h.bcell[sa] = loc[a] | ((a < b ? 1 : 0) << 17);
      h.bcell[sb] = loc[b] | (1 << 16) | ((b < a ? 1 : 0) << 17);
      h.bhalo[sa] = b;
      h.bhalo[sb] = a;
      h.bpeer[sa] = sb;
      h.bpeer[sb] = sa;
      lside[2 * size_t(f)] = (unsigned short)(n_in[pa] + sa - h.bptr[pa]);
      lside[2 * size_t(f) + 1] = (unsigned short)(n_in[pb] + sb - h.bptr[pb]);
    }
  }
  h.cyc.resize(size_t(6) * N);
  for (int p = 0; p < N; p++) {
    const int c = h.cell[p];
    for (int q = 0; q < 6; q++) {
      const int f = cyc[size_t(q) * N + c];
      if (f < 0 || f >= E) return "cell cycle out of range";
      const int side = gi[f] == c ? 0 : (gi[size_t(E) + f] == c ? 1 : -1);
      if (side < 0) return "a face of a cell's cycle does not touch the cell";
      h.cyc[size_t(q) * N + p] = lside[2 * size_t(f) + side];
    }
  }
  return std::string();
}

typedef unsigned uint4v __attribute__((ext_vector_type(4)));

template <typename T>
struct ResArgs {
  int E, N, B, W, ipl, nfields, energy_quad, quad_drag, count;  // ipl: instances at a time
  long long n0;                // index of the first step
  unsigned seq0;               // sequence number the launch's messages count from
  unsigned launch;             // number of the launch, from 1
  unsigned long long arrive;   // arrival word once every workgroup of this launch is in
  // operands (device order)
  const T *g_coef, *fcor, *farea, *fdist, *flen, *kite, *area, *cellS;
  const int *info;
  const double *inst, *table;  // table: step s and instance b at 8 + (s B + b) 8
  // patches
  const int *cptr, *fptr, *bptr, *cell, *face, *fcell, *bface, *bcell, *bhalo, *bpeer;
  const unsigned short *cyc;
  int max_cells, max_face, max_bnd;
  // state (instance-major)
  const T *v, *eta, *ts;
  T *v_out, *eta_out, *ts_out, *ring_v, *ring_e;
  double *part;                // [B][count][W] dissipation partials
  uint4v *mail;                // [ipl][kResDepth][kResPlanes][slots]
  int slots;
  unsigned long long *ctl;     // [0] arrival word, [1] a wait ran out of time, [2] first launch taken back
  unsigned *status;            // host memory: the first launch taken back, or kResFailed
};

__device__ __forceinline__ unsigned long long res_get(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A message is two values of T: one 16-byte piece in FP32, two in FP64, each
// of two words (data, tag).  A word is only looked at by itself, so nothing
// is asked of a 16-byte access beyond its aligned 8-byte words being whole.
// The pieces of a box are kept by plane ([plane][slot]), so that a wave's
// look at 64 slots reads whole lines.  Looks and sends are plain 16-byte
// accesses with the agent-scope bit (sc1): with four 8-byte loads a look, each
// of which goes past the L2 by itself, a step of 256 patches took 5.7 us
// instead of 2.6.
template <typename T>
constexpr int kResPlanes = sizeof(T) == 8 ? 2 : 1;

// (The two wait states after the store keep a following vector instruction
// from overwriting its data registers before they are read; the compiler
// adds them after stores of its own, not after inline assembly.)
__device__ __forceinline__ void res_store(uint4v *p, uint4v x) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(x) : "memory");
}

__device__ __forceinline__ void res_send(uint4v *p, int slots, double a, double b, unsigned tag) {
  const unsigned long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  res_store(p, uint4v{unsigned(x), tag, unsigned(x >> 32), tag});
  res_store(p + slots, uint4v{unsigned(y), tag, unsigned(y >> 32), tag});
}
__device__ __forceinline__ void res_send(uint4v *p, int, float a, float b, unsigned tag) {
  res_store(p, uint4v{__float_as_uint(a), tag, __float_as_uint(b), tag});
}
// one look at a message: true when every word carries the tag
__device__ __forceinline__ bool res_look(const uint4v *p, int slots, double &a, double &b, unsigned tag) {
  uint4v x, y;
  asm volatile("global_load_dwordx4 %0, %2, off sc1\n\tglobal_load_dwordx4 %1, %3, off sc1\n\ts_waitcnt vmcnt(0)"
               : "=&v"(x), "=&v"(y)
               : "v"(p), "v"(p + slots)
               : "memory");
  a = __longlong_as_double((long long)(x[0] | (static_cast<unsigned long long>(x[2]) << 32)));
  b = __longlong_as_double((long long)(y[0] | (static_cast<unsigned long long>(y[2]) << 32)));
  return x[1] == tag && x[3] == tag && y[1] == tag && y[3] == tag;
}
__device__ __forceinline__ bool res_look(const uint4v *p, int, float &a, float &b, unsigned tag) {
  uint4v x;
  asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(x) : "v"(p) : "memory");
  a = __uint_as_float(x[0]);
  b = __uint_as_float(x[2]);
  return x[1] == tag && x[3] == tag;
}

// LDS of a workgroup: en (dissipation integrands of kResEn steps), then per
// face the pair of partial sums and l_e v_e, per cell the pair (height,
// tide), the tide fields of the cells and across the boundary, the peers.
template <typename T>
__host__ __device__ inline size_t res_lds_bytes(int NT, int cells, int faces, int bnd, int nf) {
  const size_t t = size_t(3) * faces + size_t(2 + nf) * cells + size_t(nf) * bnd;
  return sizeof(double) * size_t(kResEn) * NT + t * sizeof(T) + sizeof(int) * (size_t(bnd) + 4);
}

template <typename T>
struct alignas(2 * sizeof(T)) ResPair {
  T x, y;
};

// The momentum update of one face from values at hand, operation for
// operation that of face_update's compact form: u0, u1 the tide at the two
// cells, r1, r2 the tendencies of the last two steps.
template <typename T>
struct ResFace {
  T v, r1, r2;                       // state
  T gc0, gc1, fcor, area, dist, len; // operands
};

// QUAD: quadratic drag or its dissipation may be on (else no square root is
// formed at all; chosen at run time it is formed and thrown away).
template <typename T, bool QUAD>
__device__ __forceinline__ double res_face(ResFace<T> &f, T t0, T t1, T e0, T e1, T u0, T u1, T g, T alpha, T dt, T qd,
                                           bool ab3, bool energy_quad, bool quad_drag) {
  const T vt = (t0 - t1) / f.dist;
  const T ve = f.v;
  const T sp = ve * ve + vt * vt;
  const T en = QUAD && energy_quad ? sqrt(sp) * sp : sp;
  const double energy = double(f.area) * double(en);
  const T ge = f.gc0 * e0 + f.gc1 * e1;
  T f0 = -g * ge + f.fcor * vt;
  if (QUAD && quad_drag) f0 -= qd * sqrt(sp) * ve;
  const T fu = f.gc0 * u0 + f.gc1 * u1;
  const T drag = -alpha * ve + fu;
  T upd;
  if (ab3)
    upd = (T(23. / 12.) * f0 + T(-16. / 12.) * f.r1 + T(5. / 12.) * f.r2) * dt;
  else
    upd = f0 * dt;
  f.r2 = f.r1;
  f.r1 = f0;
  f.v = (ve + upd) + dt * drag;
  return energy;
}

// Six values of a cell's faces, each a register of its own (an array would be
// held as one six-wide register).
template <typename T>
struct Six {
  T a0, a1, a2, a3, a4, a5;
  template <int I>
  __device__ __forceinline__ T &at() {
    if constexpr (I == 0) return a0;
    else if constexpr (I == 1) return a1;
    else if constexpr (I == 2) return a2;
    else if constexpr (I == 3) return a3;
    else if constexpr (I == 4) return a4;
    else return a5;
  }
};

template <int I>
using Int = std::integral_constant<int, I>;

// f(Int<0>), ..., f(Int<N - 1>)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F &&f) {
  if constexpr (I < N) {
    f(Int<I>());
    each<N, I + 1>(f);
  }
}

// TRiSK partial sums of a cell with K faces (trisk_partials of k_step), each
// handed to put(p, sum) before the next is formed when LEAN: 16 wavefronts
// hide the chains, and six of them at once would not fit the registers
template <typename T, int K, bool LEAN, typename Put>
__device__ __forceinline__ void res_partials(Six<T> &F, Six<T> &R, Put put) {
  each<K>([&](auto P) {
    constexpr int p = decltype(P)::value;
    T S = R.template at<p>();
    T acc = (S - T(0.5)) * F.template at<(p + 1) % K>();
    each<K - 2>([&](auto J) {
      constexpr int j = decltype(J)::value + 2;
      S += R.template at<(p + j - 1) % K>();
      acc += (S - T(0.5)) * F.template at<(p + j) % K>();
    });
    put(P, acc);
    if (LEAN) __builtin_amdgcn_sched_barrier(0);
  });
}

// A wait ran out of time: every workgroup of the launch is told to leave.
__device__ __forceinline__ void res_fail(unsigned long long *ctl, unsigned *status) {
  __hip_atomic_store(ctl + 1, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(status, kResFailed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Wait for the workgroups counted in; false when the launch was taken back,
// or follows one that failed (the host then knows by `status`, which stays as
// that one left it).  One lane of each workgroup.
__device__ __forceinline__ bool res_all_here(unsigned long long *ctl, unsigned long long arrive, unsigned launch,
                                             unsigned *status) {
  if (res_get(ctl + 1)) return false;
  const long long t0 = wall_clock64();
  unsigned long long w = res_get(ctl);
  while (!(w & kResTaken) && w < arrive) {
    if (wall_clock64() - t0 > kResArriveTicks) {
      unsigned long long seen = w;
      if (__hip_atomic_compare_exchange_strong(ctl, &seen, w | kResTaken, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        w |= kResTaken;
      else
        w = seen;
    } else {
      __builtin_amdgcn_s_sleep(1);
      w = res_get(ctl);
    }
  }
  if (!(w & kResTaken)) return true;
  unsigned long long none = 0;  // the first launch to be taken back tells the host
  if (__hip_atomic_compare_exchange_strong(ctl + 2, &none, (unsigned long long)launch, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    __hip_atomic_store(status, launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  return false;
}

__device__ __forceinline__ double lane_value(double x, int lane) {
  const long long v = __double_as_longlong(x);
  const unsigned lo = unsigned(__builtin_amdgcn_readlane(int(v), lane));
  const unsigned hi = unsigned(__builtin_amdgcn_readlane(int(v >> 32), lane));
  return __longlong_as_double((long long)((static_cast<unsigned long long>(hi) << 32) | lo));
}

// a value that is the same in every lane, held in scalar registers
__device__ __forceinline__ double uniform(double x) { return lane_value(x, 0); }

// FI faces per lane and one cell, NT lanes.  Faces: inner face q in slot
// q / NT of lane q % NT; the boundary faces in the last slot of the last
// lanes.  Two barriers a step: faces (the boundary faces last, from the
// neighbours' messages, which are under way during the inner ones), barrier,
// cells (those with a boundary face in the first lanes, sent at once),
// barrier.
//
// The kernel's arguments are read from the kernarg segment where they are
// used (`hide` keeps the compiler from holding all of them, and addresses
// made of them, in registers across the step loop), and the kite fractions
// are made opaque every step, or their 30 partial sums per cell would be
// kept: with both the FP64 kernel fits 128 registers, 16 wavefronts per CU.
template <typename T, int NT, int FI, int WPS, bool QUAD>
__global__ __launch_bounds__(NT, WPS) void k_resident(ResArgs<T> args) {
  constexpr bool LEAN = sizeof(T) == 8 ? NT == 1024 : WPS == 8;
  typedef const ResArgs<T> __attribute__((address_space(4))) * ArgPtr;
  ArgPtr ka = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
  auto hide = [&] { asm volatile("" : "+s"(ka)); };
  extern __shared__ __align__(16) unsigned char res_lds[];
  const int tid = threadIdx.x;
  const int W = ka->W, nf = ka->nfields, max_bnd = ka->max_bnd;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int li = tile / W, j = tile - li * W;
  double *en = reinterpret_cast<double *>(res_lds);                    // [kResEn][NT]
  ResPair<T> *lt = reinterpret_cast<ResPair<T> *>(en + kResEn * NT);   // [faces] partial sums: inner, outer cell
  ResPair<T> *lc = lt + ka->max_face;                                  // [cells] height, tide of the step
  T *lv = reinterpret_cast<T *>(lc + ka->max_cells);                   // [faces] l_e v_e
  T *ls = lv + ka->max_face;                                           // [nf][cells] tide fields
  T *lh = ls + size_t(nf) * ka->max_cells;                             // [nf][bnd] tide fields across the boundary
  int *peer = reinterpret_cast<int *>(lh + size_t(nf) * max_bnd);      // [bnd]
  int *bad = peer + max_bnd;
  const int max_cells = ka->max_cells;
  if (tid == 0) {
    *bad = 0;
    __hip_atomic_fetch_add(ka->ctl, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const int c_lo = ka->cptr[j], nc = ka->cptr[j + 1] - c_lo;
  const int f_lo = ka->fptr[j], ni = ka->fptr[j + 1] - f_lo;
  const int b_lo = ka->bptr[j], nb = ka->bptr[j + 1] - b_lo;
  const int bq = tid - (NT - nb);        // boundary face of this lane's last slot
  const bool bnd = bq >= 0;
  // face of slot u: an inner face (past the last: the last again, nothing
  // stored) or the lane's boundary face
  auto is_bnd = [&](int u) { return u == FI - 1 && bnd; };
  auto face_id = [&](int u) {
    return is_bnd(u) ? ka->bface[b_lo + bq] : ka->face[f_lo + min(tid + u * NT, ni - 1)];
  };
  // operators
  ResFace<T> f[FI];
  int fc[FI];                            // local cells c0 | c1 << 16; boundary face: own cell, side, owner
  int halo = 0;
#pragma unroll
  for (int u = 0; u < FI; ++u) {
    const int e = face_id(u), E = ka->E;
    fc[u] = is_bnd(u) ? ka->bcell[b_lo + bq] : ka->fcell[f_lo + min(tid + u * NT, ni - 1)];
    f[u].gc0 = ka->g_coef[e];
    f[u].gc1 = ka->g_coef[E + e];
    f[u].fcor = ka->fcor[e];
    f[u].area = ka->farea[e];
    f[u].dist = ka->fdist[e];
    f[u].len = ka->flen[e];
  }
  if (bnd) {
    halo = ka->bhalo[b_lo + bq];
    for (int k = 0; k < nf; ++k) lh[k * max_bnd + bq] = ka->cellS[size_t(k) * ka->N + halo];
    peer[bq] = ka->bpeer[b_lo + bq];
  }
  Six<T> R;
  T area, eta, r1, r2;
  int lq[3], info;
  const bool has_cell = tid < nc;
  {
    const int p = min(tid, nc - 1), N = ka->N;
    const int c = ka->cell[c_lo + p];
    info = ka->info[c];
    each<6>([&](auto Q) { R.template at<Q.value>() = ka->kite[size_t(Q.value) * N + c]; });
#pragma unroll
    for (int q = 0; q < 3; ++q)
      lq[q] = int(ka->cyc[size_t(2 * q) * N + c_lo + p]) | (int(ka->cyc[size_t(2 * q + 1) * N + c_lo + p]) << 16);
    area = ka->area[c];
    if (has_cell)
      for (int k = 0; k < nf; ++k) ls[k * max_cells + p] = ka->cellS[size_t(k) * N + c];
  }
  // every workgroup on the chip, or none goes on
  if (tid == 0 && !res_all_here(ka->ctl, ka->arrive, ka->launch, ka->status)) *bad = 1;
  __syncthreads();
  if (*bad) return;  // nothing written

  const int slots = ka->slots;
  const size_t box_step = size_t(slots) * kResPlanes<T>;
  uint4v *const box = ka->mail + size_t(li) * kResDepth * box_step;
  const int count = ka->count, B = ka->B;
  const long long n0 = ka->n0;
  const bool e_quad = ka->energy_quad != 0, q_drag = ka->quad_drag != 0;
  unsigned seq = ka->seq0;
#pragma unroll 1
  for (int b = li; b < B; b += ka->ipl, seq += unsigned(count)) {
    hide();
    const double *ip = ka->inst + b * 8;
    const T g = T(uniform(ip[0])), alpha = T(uniform(ip[1])), dt = T(uniform(ip[2])), qd = T(uniform(ip[4])),
            h = T(uniform(ip[5]));
    const bool load = uniform(ip[3]) != 0.0;
    const double *coef = ka->table + 8 + size_t(b) * 8 + (tid & 7);  // step s: + s B 8; lane k: factor k % 8
    double mine = *coef;
    T t_far = T(0), e_far = T(0);
    {
      const int E = ka->E, N = ka->N;
      const int s1 = int((n0 + 2) % 3), s2 = int((n0 + 1) % 3);
      const T *v = ka->v + size_t(b) * E, *rv = ka->ring_v + size_t(b) * 3 * E, *ts = ka->ts + size_t(b) * 2 * E;
#pragma unroll
      for (int u = 0; u < FI; ++u) {
        const int e = face_id(u), q = tid + u * NT;
        f[u].v = v[e];
        f[u].r1 = rv[size_t(s1) * E + e];
        f[u].r2 = rv[size_t(s2) * E + e];
        const T t0 = ts[e], t1 = ts[E + e];
        if (is_bnd(u)) {
          const bool outer = (fc[u] >> 16) & 1;
          if (outer) lt[ni + bq].y = t1;
          else lt[ni + bq].x = t0;
          t_far = outer ? t0 : t1;
          e_far = ka->eta[size_t(b) * N + halo];
        } else if (q < ni) {
          lt[q] = ResPair<T>{t0, t1};
        }
      }
      const int c = ka->cell[c_lo + min(tid, nc - 1)];
      const T *re = ka->ring_e + size_t(b) * 3 * N;
      eta = ka->eta[size_t(b) * N + c];
      r1 = re[size_t(s1) * N + c];
      r2 = re[size_t(s2) * N + c];
    }
    T ck[kMaxForcing];                    // the tide's factors: the same in every lane
#pragma unroll
    for (int k = 0; k < kMaxForcing; ++k) ck[k] = k < nf ? T(lane_value(mine, k)) : T(0);
    if (has_cell) {
      T x = T(0);
#pragma unroll
      for (int k = 0; k < kMaxForcing; ++k)
        if (k < nf) x += ck[k] * ls[k * max_cells + tid];
      lc[tid] = ResPair<T>{eta, x};
    }
    T u_far = T(0);                       // tide across the boundary face
    if (bnd)
#pragma unroll
      for (int k = 0; k < kMaxForcing; ++k)
        if (k < nf) u_far += ck[k] * lh[k * max_bnd + bq];
    double *part = ka->part + size_t(b) * count * W + j;
    hide();
    __syncthreads();

#pragma unroll 1
    for (int s = 0; s < count; ++s) {
      const bool ab3 = (n0 + s >= 2) || load;
      const bool last = s + 1 == count;
      if (!last) coef += size_t(B) * 8;
      mine = *coef;  // the next step's, under way meanwhile
      int lane = tid;
      if (LEAN) {
        asm volatile("" : "+v"(lane), "+v"(info), "+v"(lq[0]), "+v"(lq[1]), "+v"(lq[2]));
#pragma unroll
        for (int u = 0; u < FI; ++u) asm volatile("" : "+v"(fc[u]), "+v"(f[u].area));
      }
      double local = 0.0;
#pragma unroll
      for (int u = 0; u < FI; ++u) {
        const int q = lane + u * NT;
        T t0, t1, e0, e1, u0, u1;
        if (is_bnd(u)) {
          if (s > 0) {  // the message of step s - 1
            const unsigned tag = seq + unsigned(s);
            const uint4v *p = box + size_t(tag & (kResDepth - 1)) * box_step + (b_lo + bq);
            int spins = 0;
            long long since = 0;
            while (!res_look(p, slots, t_far, e_far, tag)) {
              if ((++spins & 1023) == 0) {
                const long long now = wall_clock64();
                if (since == 0) since = now;
                if (now - since > kResWaitTicks || res_get(ka->ctl + 1)) {
                  res_fail(ka->ctl, ka->status);
                  *bad = 1;
                  break;
                }
              }
            }
          }
          const bool outer = (fc[u] >> 16) & 1;
          const ResPair<T> t = lt[ni + bq], c = lc[fc[u] & 0xffff];
          t0 = outer ? t_far : t.x, t1 = outer ? t.y : t_far;
          e0 = outer ? e_far : c.x, e1 = outer ? c.x : e_far;
          u0 = outer ? u_far : c.y, u1 = outer ? c.y : u_far;
        } else {
          const ResPair<T> t = lt[min(q, ni - 1)], c0 = lc[fc[u] & 0xffff], c1 = lc[fc[u] >> 16];
          t0 = t.x, t1 = t.y, e0 = c0.x, e1 = c1.x, u0 = c0.y, u1 = c1.y;
        }
        const double e = res_face<T, QUAD>(f[u], t0, t1, e0, e1, u0, u1, g, alpha, dt, qd, ab3, e_quad, q_drag);
        const bool b_here = is_bnd(u);
        if (b_here || q < ni) {
          if (!b_here || (fc[u] >> 17)) local += e;
          lv[b_here ? ni + bq : q] = f[u].len * f[u].v;
        }
      }
      en[(s & (kResEn - 1)) * NT + lane] = local;
      __syncthreads();
      if (*bad) return;
      // read from the first lanes here, where all lanes are active
#pragma unroll
      for (int k = 0; k < kMaxForcing; ++k) ck[k] = k < nf ? T(lane_value(mine, k)) : T(0);
      if (has_cell) {
        const unsigned tag = seq + unsigned(s) + 1;  // the message of this step
        uint4v *out = box + size_t(tag & (kResDepth - 1)) * box_step;
        Six<T> F;
        Six<int> l;
        each<6>([&](auto Q) {
          constexpr int q = Q.value;
          asm volatile("" : "+v"(R.template at<q>()));
          l.template at<q>() = (lq[q >> 1] >> ((q & 1) * 16)) & 0xffff;
          const T x = lv[l.template at<q>()];
          F.template at<q>() = ((info >> (3 + q)) & 1) ? -x : x;
        });
        const int k6 = info & 7, db = info >> 3;
        // divergence and continuity, as divergence() and continuity_with()
        T sum = F.a0;
        sum += F.a1;
        sum += F.a2;
        sum += F.a3;
        sum += F.a4;
        if (k6 == 6) sum += F.a5;
        const T f0 = h * (-sum / area);
        T upd;
        if (ab3)
          upd = (T(23. / 12.) * f0 + T(-16. / 12.) * r1 + T(5. / 12.) * r2) * dt;
        else
          upd = f0 * dt;
        r2 = r1;
        r1 = f0;
        eta = eta + upd;
        auto put = [&](auto Q, T t) {
          const int q = l.template at<Q.value>();
          T *at = &lt[q].x + ((db >> Q.value) & 1);
          *at = t;
          if (q >= ni && !last) res_send(out + peer[q - ni], slots, t, eta, tag);
        };
        if (k6 == 6)
          res_partials<T, 6, LEAN>(F, R, put);
        else
          res_partials<T, 5, LEAN>(F, R, put);
        T x = T(0);
#pragma unroll
        for (int k = 0; k < kMaxForcing; ++k)
          if (k < nf) x += ck[k] * ls[k * max_cells + lane];
        lc[lane] = ResPair<T>{eta, x};
      }
      if (bnd) {
        u_far = T(0);
#pragma unroll
        for (int k = 0; k < kMaxForcing; ++k)
          if (k < nf) u_far += ck[k] * lh[k * max_bnd + bq];
      }
      // dissipation partials of up to kResEn steps: wave w the steps w, w + NT / 64, ...
      if ((s & (kResEn - 1)) == kResEn - 1 || last) {
        const int sb = s & ~(kResEn - 1);
        for (int k = lane >> 6; k <= s - sb; k += NT / 64) {
          double x = 0.0;
#pragma unroll 4
          for (int q = 0; q < NT / 64; ++q) x += en[k * NT + q * 64 + (lane & 63)];
          for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
          if ((lane & 63) == 0) part[size_t(sb + k) * W] = x;
        }
      }
      __syncthreads();
    }
    // the state back: v, the two live history slots, height, partial sums
    hide();
    {
      const int E = ka->E, N = ka->N;
      const long long n1 = n0 + count;
      const int w1 = int((n1 + 2) % 3), w2 = int((n1 + 1) % 3);
      T *v = ka->v_out + size_t(b) * E, *rv = ka->ring_v + size_t(b) * 3 * E, *ts = ka->ts_out + size_t(b) * 2 * E;
#pragma unroll
      for (int u = 0; u < FI; ++u) {
        const int e = face_id(u), q = tid + u * NT;
        const bool b_here = is_bnd(u);
        if (b_here) {
          const bool outer = (fc[u] >> 16) & 1;
          const ResPair<T> t = lt[ni + bq];
          ts[(outer ? E : 0) + e] = outer ? t.y : t.x;
        } else if (q < ni) {
          const ResPair<T> t = lt[q];
          ts[e] = t.x;
          ts[E + e] = t.y;
        }
        if (b_here ? (fc[u] >> 17) != 0 : q < ni) {
          v[e] = f[u].v;
          rv[size_t(w1) * E + e] = f[u].r1;
          rv[size_t(w2) * E + e] = f[u].r2;
        }
      }
      if (has_cell) {
        const int c = ka->cell[c_lo + tid];
        T *re = ka->ring_e + size_t(b) * 3 * N;
        ka->eta_out[size_t(b) * N + c] = eta;
        re[size_t(w1) * N + c] = r1;
        re[size_t(w2) * N + c] = r2;
      }
    }
    __syncthreads();  // the next instance's values go to the same LDS
  }
}

// Dissipation series of the steps of a resident launch: a workgroup of one
// wave per (step, instance) adds the W partials in a fixed order.
__global__ __launch_bounds__(64) void k_resident_series(const double *__restrict__ part, int W, int count, long long n0,
                                                        const double *__restrict__ dconst, double *series,
                                                        int *nonfinite, int cap) {
  const int s = blockIdx.x, b = blockIdx.y;
  const double *p = part + (size_t(b) * count + s) * W;
  double x = 0.0;
  for (int q = threadIdx.x; q < W; q += 64) x += p[q];
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  if (threadIdx.x == 0) {
    const double d = x * dconst[b];
    series[size_t(b) * cap + size_t((n0 + s) % cap)] = d;
    if (!isfinite(d)) nonfinite[b] = 1;
  }
}

}  // namespace odis
