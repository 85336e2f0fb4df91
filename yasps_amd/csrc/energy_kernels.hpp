// Element kernel machinery shared by the library's energies (energies.hip) and run-time
// generated user energies (yasps_amd/usercode.py): gather of an element's vertex data
// through the union view (vertices driven by affine bodies included), energy / gradient /
// packed Hessian from Kind<ID>::eval, PSD projection with the reference's rules, and the
// scatter into block storage for segments of any size (hessianKernelNoProject.pyx:37-264
// semantics). A translation unit specialises Kind<ID> for its energies (A vertices of W
// values, N = A W, P element parameters, S scene parameters, and
//   __device__ static void eval(x, p, s, E, g, H)
// with H the packed upper triangle) and instantiates eval_energy<ID> / energy_values<ID>.
//
// Vertices of an affine union child follow x = t + A r (JOIN of the body's A (9, row-major)
// and t (3) through a vertex -> body connectivity, one_bunny_partial_abd.py:127-144).
// The map is linear, so the projection acts on the Hessian in vertex positions and the
// chain rule maps it to the body's segments (differentiator.pyx:795-801): with slot
// entries s -> (position entry i(s), coefficient c(s)), g_s = c(s) g_i(s) and
// H_st = c(s) c(t) H_i(s)i(t): t entries map to x_j with c = 1, A entries (j, l) to x_j
// with c = r_l.
#pragma once
#include "common.hpp"
#include "dense.hpp"
#include "element_common.hpp"

#include <algorithm>
#include <type_traits>

namespace ysp {
namespace {

constexpr unsigned kEB = 64;
constexpr int kSlotsMax = 16;

template <int ID>
struct Kind;


// Quadratic form of a linear map of the element's vertex data, y = J x + c with J 6 x 12:
// E = y^T Q y / 2 + l^T y, g = J^T (Q y + l), H = J^T spd(Q) J (the projection acts on the
// inner Hessian: the map is linear). Scene parameters are read from memory in place
// (element_eval), not copied per element.
constexpr int kQfRows = 6;
template <int N>
__device__ __forceinline__ void project_packed(double (&H)[N * (N + 1) / 2], uint32_t method);

template <>
struct Kind<YSP_ENERGY_QUADRATIC_FORM> {
  static constexpr int A = 4, W = 3, N = 12, P = 0, S = kQfRows * 12 + kQfRows * kQfRows + 2 * kQfRows;
};

__device__ __forceinline__ void quadratic_form_eval(const double (&x)[12], const double* __restrict__ sp,
                                                    uint32_t method, double& E, double (&g)[12],
                                                    double (&H)[78]) {
  const double* J = sp;
  const double* Q = sp + kQfRows * 12;
  const double* lin = Q + kQfRows * kQfRows;
  const double* off = lin + kQfRows;
  double y[kQfRows], qy[kQfRows];
#pragma unroll
  for (int i = 0; i < kQfRows; ++i) {
    double acc = off[i];
#pragma unroll
    for (int j = 0; j < 12; ++j) acc += J[12 * i + j] * x[j];
    y[i] = acc;
  }
  E = 0.0;
#pragma unroll
  for (int i = 0; i < kQfRows; ++i) {
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < kQfRows; ++k) acc += Q[kQfRows * i + k] * y[k];
    qy[i] = acc + lin[i];
    E += y[i] * (0.5 * acc + lin[i]);
  }
#pragma unroll
  for (int j = 0; j < 12; ++j) {
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < kQfRows; ++i) acc += J[12 * i + j] * qy[i];
    g[j] = acc;
  }
  double Qp[kQfRows * (kQfRows + 1) / 2];
#pragma unroll
  for (int i = 0; i < kQfRows; ++i)
#pragma unroll
    for (int k = i; k < kQfRows; ++k) Qp[upper_index<kQfRows>(i, k)] = Q[kQfRows * i + k];
  if (method != 0) project_packed<kQfRows>(Qp, method);
  double JQ[kQfRows][12];                       // spd(Q) J
#pragma unroll
  for (int i = 0; i < kQfRows; ++i)
#pragma unroll
    for (int j = 0; j < 12; ++j) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < kQfRows; ++k)
        acc += Qp[i <= k ? upper_index<kQfRows>(i, k) : upper_index<kQfRows>(k, i)] * J[12 * k + j];
      JQ[i][j] = acc;
    }
#pragma unroll
  for (int a = 0; a < 12; ++a)
#pragma unroll
    for (int b = a; b < 12; ++b) {
      double acc = 0.0;
#pragma unroll
      for (int i = 0; i < kQfRows; ++i) acc += J[12 * i + a] * JQ[i][b];
      H[upper_index<12>(a, b)] = acc;
    }
}

struct AffineView {
  uint32_t mask;                                  // bit c: union child c is affine
  const uint32_t* body[YSP_MAX_UNION_CHILDREN];   // vertex -> body
  const double* rest[YSP_MAX_UNION_CHILDREN];     // rest position r per vertex
};

// Union child of instance v and its index inside the child.
__device__ __forceinline__ uint32_t union_child(const UnionView& U, uint32_t v, uint32_t& local) {
  uint32_t total = 0;
  for (uint32_t c = 0; c < U.nc; ++c) {
    const uint32_t cnt = U.counts[c];
    if (v < total + cnt) {
      local = v - total;
      return c;
    }
    total += cnt;
  }
  local = 0;
  return 0;
}

// ----------------------------------------------------------------- projection
// hessianKernelHeader.pyx:79-252 for N >= 4: the packed-Schur PSD test on the element
// Hessian; a failing matrix H becomes V max(L, 0) V^T (method 2) or V |L| V^T (method 1),
// formed as H plus the change of its negative eigenvalues (dense.hpp), so that what the
// projection leaves alone keeps its bits.
template <int N>
__device__ __forceinline__ bool is_psd(const double (&H)[N * (N + 1) / 2]) {
  double L[N * (N + 1) / 2];
#pragma unroll
  for (int r = 0; r < N; ++r)
#pragma unroll
    for (int c = 0; c <= r; ++c) L[r * (r + 1) / 2 + c] = H[upper_index<N>(c, r)];
  return psd_test_packed<N>(L);
}

template <int N>
__device__ __forceinline__ void project_packed(double (&H)[N * (N + 1) / 2], uint32_t method) {
  if (is_psd<N>(H)) return;
  double D[N * (N + 1) / 2];
#pragma unroll
  for (int i = 0; i < N * (N + 1) / 2; ++i) D[i] = H[i];
  clamp_change_packed<N>(D, method);
#pragma unroll
  for (int i = 0; i < N * (N + 1) / 2; ++i) H[i] += D[i];
}

// 4-vertex kinds whose energy depends on vertex differences only (barriers, dihedral
// bending, SNH): their 12x12 Hessians annihilate the three translations, so a failing
// Hessian is projected in the 9-dimensional complement, M = (U x I3)^T H (U x I3) with U
// the orthonormal 4x3 basis orthogonal to (1,1,1,1): the same result as the 12x12
// decomposition up to the rounding-level translation eigenvalues, on a 9x9 matrix (0.42 of
// the work and 81 instead of 144 eigenvector registers). The PSD test stays on the full
// 12x12 matrix, as the reference runs it.
template <int ID>
__host__ __device__ constexpr bool translation_free() {
  return ID == YSP_ENERGY_POINT_TRIANGLE || ID == YSP_ENERGY_EDGE_EDGE ||
         ID == YSP_ENERGY_BENDING || ID == YSP_ENERGY_SNH;
}

__device__ __forceinline__ double basis4(int a, int k) {
  // columns of U: (1,-1,0,0)/sqrt2, (1,1,-2,0)/sqrt6, (1,1,1,-3)/sqrt12
  constexpr double c0 = 0.70710678118654752440, c1 = 0.40824829046386301637,
                   c2 = 0.28867513459481288225;
  return k == 0 ? (a == 0 ? c0 : (a == 1 ? -c0 : 0.0))
       : k == 1 ? (a <= 1 ? c1 : (a == 2 ? -2.0 * c1 : 0.0))
                : (a <= 2 ? c2 : -3.0 * c2);
}

// Elements that the evaluation does not scatter itself are held: an indefinite Hessian for
// the projection kernel, an element whose slots are not one W-wide slot per vertex
// (vertices driven by affine bodies, a repeated target vertex) for the general scatter,
// or both. Slot i of a launch's list is elem[i] (element, kHeld* flags) with the packed
// Hessian and the gradient in data, 8 slots interleaved: component c of slot i at
// held_at<N>(i, c). A lane per slot then reads whole 64-byte pieces (one slot after the
// other took 137 us to project what is indefinite of 122,000 hinges, this takes 116), and a
// wavefront per slot shares its lines with the 7 slots beside it. general lists the slots of
// the second kind.
constexpr uint32_t kHeldIndefinite = 1u << 31, kHeldGeneral = 1u << 30;
constexpr uint32_t kHeldElement = kHeldGeneral - 1;
template <int N>
__host__ __device__ constexpr int held_doubles() {
  return N * (N + 1) / 2 + N;
}
template <int N>
__device__ __forceinline__ size_t held_at(uint32_t slot, int c) {
  return static_cast<size_t>(slot / 8) * (8 * held_doubles<N>()) + 8 * c + slot % 8;
}
struct Held {
  uint32_t* counts;              // [2]: slots, general slots
  uint32_t* elem;
  uint32_t* general;
  double* data;
};

template <int N>
__device__ __forceinline__ double hget(const double (&H)[N * (N + 1) / 2], int i, int j) {
  return i <= j ? H[upper_index<N>(i, j)] : H[upper_index<N>(j, i)];
}

// Per-workgroup sums of the contended destinations of the general scatter (atomic mode):
// every element of an affine body adds into the same (A, A), (A, t), (t, t) blocks and the
// same 12 gradient entries of that body, so a device-scope FP64 atomic per element and
// entry serialises on a few addresses. Blocks coupling two affine groups and gradient
// segments of affine groups are summed in LDS instead (a few slots keyed by the
// destination's offset, found by all, with a sum for each wavefront) and leave with one
// global atomic per entry and workgroup, the wavefronts' sums added in order. A destination
// that finds no free slot takes the global atomic directly. The assembled bits are not
// reproducible: the list's order past one evaluation wavefront, which destinations find a
// slot when there are more than slots, and every global atomic follow the schedule.
constexpr unsigned kGB = 1024, kGW = kGB / 64;
// Lists up to this length go to one workgroup: fewer sums depend on the schedule then (spread
// over workgroups, the iteration counts of two solves of a small stiff scene differed in 5 of 25
// pairs, in one workgroup in none; no guarantee, see above). Longer ones are spread over the
// chip: with 256 elements a workgroup 7,000 tets and 42,000 pairs took 344 us each, spread 64.
constexpr uint32_t kGRun = 256;
constexpr uint32_t kHotEmpty = 0xffffffffu;
constexpr int kHotBlocks = 8, kHotBlockMax = 81, kHotGrad = 4, kHotGradMax = 9;
struct HotTable {
  uint32_t bkey[kHotBlocks];    // value offset of the block in S.blocks
  uint32_t bsize[kHotBlocks];   // h * w
  uint32_t bdiag[kHotBlocks];   // offset in S.diag_blocks, kHotEmpty without one
  uint32_t gkey[kHotGrad];      // gradient offset
  uint32_t gsize[kHotGrad];
  double bval[kGW][kHotBlocks][kHotBlockMax];
  double gval[kGW][kHotGrad][kHotGradMax];
};

__device__ __forceinline__ int hot_slot(uint32_t* keys, int cap, uint32_t key) {
  for (int j = 0; j < cap; ++j) {
    const uint32_t cur = __hip_atomic_load(keys + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (cur == key) return j;
    if (cur == kHotEmpty) {
      const uint32_t old = atomicCAS(keys + j, kHotEmpty, key);
      if (old == kHotEmpty || old == key) return j;
    }
  }
  return -1;
}

__device__ __forceinline__ void hot_init(HotTable& t) {
  for (uint32_t i = threadIdx.x; i < kGW * kHotBlocks * kHotBlockMax; i += kGB) (&t.bval[0][0][0])[i] = 0.0;
  for (uint32_t i = threadIdx.x; i < kGW * kHotGrad * kHotGradMax; i += kGB) (&t.gval[0][0][0])[i] = 0.0;
  if (threadIdx.x < kHotBlocks) t.bkey[threadIdx.x] = kHotEmpty;
  if (threadIdx.x < kHotGrad) t.gkey[threadIdx.x] = kHotEmpty;
  __syncthreads();
}

__device__ __forceinline__ void hot_flush(HotTable& t, const ScatterArgs& S) {
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kHotBlocks * kHotBlockMax; i += kGB) {
    const uint32_t j = i / kHotBlockMax, o = i % kHotBlockMax;
    if (t.bkey[j] == kHotEmpty || o >= t.bsize[j]) continue;
    double v = 0.0;
    for (unsigned w = 0; w < kGW; ++w) v += t.bval[w][j][o];
    atomic_add_f64(S.blocks + t.bkey[j] + o, v);
    if (t.bdiag[j] != kHotEmpty) atomic_add_f64(S.diag_blocks + t.bdiag[j] + o, v);
  }
  for (uint32_t i = threadIdx.x; i < kHotGrad * kHotGradMax; i += kGB) {
    const uint32_t j = i / kHotGradMax, o = i % kHotGradMax;
    if (t.gkey[j] == kHotEmpty || o >= t.gsize[j]) continue;
    double v = 0.0;
    for (unsigned w = 0; w < kGW; ++w) v += t.gval[w][j][o];
    atomic_add_f64(S.gradient + t.gkey[j] + o, v);
  }
}

// The general scatter: one wavefront per held element, any slot sizes, vertices of affine
// bodies. Slot groups by |perm| in first-occurrence order (hessianKernelNoProject.pyx:
// 93-163); lanes hold the slots while the groups are found, then the entries of one block
// after the other, with the element's Hessian, gradient and slots in LDS. (One lane per
// element with run-time indices put Hessian and slots in scratch memory: 1.2 ms for 7,000
// tets of affine bodies, 0.9 ms for 42,000 point-triangle and 0.8 ms for the edge-edge
// pairs of the same scene; these lists now take 64 us each.)
template <int N, int KT>
struct ElementLds {
  double h[N * (N + 1) / 2 + N];     // packed Hessian, then the gradient
  double r[8][3];                    // rest positions of affine vertices
  uint32_t idx[KT];
  uint32_t members[KT];              // per group: its slots
  uint32_t diag[KT];                 // per group: offset in the diagonal blocks
  uint8_t size[KT], col[KT], xbase[KT], amode[KT], aff[KT], head[KT];
};

// LDS written by some lanes of a wavefront and then read by others of the same wavefront.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Position entry and coefficient of entry k of slot i (identity unless the slot is the
// affine matrix of an affine vertex).
template <typename L>
__device__ __forceinline__ int xmap(const L& el, int i, int k, double& c) {
  if (el.amode[i]) {
    c = el.r[el.xbase[i] / 3][k % 3];
    return el.xbase[i] + k / 3;
  }
  c = 1.0;
  return el.xbase[i] + k;
}

template <int A, int W, int KT>
__global__ void __launch_bounds__(kGB)
    energy_scatter_kernel(UnionView P, AffineView AF, const uint32_t* __restrict__ e2v,
                          ScatterArgs S, int* __restrict__ flags, Held held) {
  constexpr int N = A * W, NH = N * (N + 1) / 2;
  static_assert(KT <= 64 && A <= 8, "slots and vertices of an element");
  __shared__ HotTable table;
  __shared__ ElementLds<N, KT> els[kGB / 64];
  const bool hot = AF.mask && !S.block_staging;    // uniform over the grid
  ElementLds<N, KT>& el = els[threadIdx.x / 64];
  const int lane = threadIdx.x % 64;
  const uint32_t count = held.counts[1];
  // a workgroup's run of the list
  const uint32_t per = count <= kGRun ? kGRun : (count + gridDim.x - 1) / gridDim.x;
  if (blockIdx.x * per >= count) return;
  if (hot) hot_init(table);
  const uint32_t end = min(count, (blockIdx.x + 1) * per);
  for (uint32_t i0 = blockIdx.x * per + threadIdx.x / 64; i0 < end; i0 += kGB / 64) {
    const uint32_t slot = held.general[i0];
    const uint32_t e = held.elem[slot] & kHeldElement;
    const int K = static_cast<int>(S.K);
    bool ok = K <= KT && !(S.block_staging && (W != 3 || AF.mask));
    // lane i: slot i
    uint32_t ii = 0, sz = 0;
    int place = -1;
    if (ok && lane < K) {
      const size_t o = static_cast<size_t>(e) * S.K + lane;
      ii = S.seg_idx[o];
      sz = S.seg_size[o];
      const int pm = S.perm[o];
      place = pm == 0 ? -1 : (pm < 0 ? -pm : pm) - 1;
    }
    for (int i = lane; i < held_doubles<N>(); i += 64) el.h[i] = held.data[held_at<N>(slot, i)];
    uint32_t col = 0, total = 0, members = 0;
#pragma unroll
    for (int j = 0; j < KT; ++j) {
      const uint32_t sj = __shfl(sz, j);
      const int pj = __shfl(place, j);
      if (j < lane) col += sj;
      total += sj;
      if (pj >= 0 && pj == place) members |= 1u << j;
    }
    const bool leads = members && __ffs(members) - 1 == lane;
    const uint64_t heads = __ballot(leads);
    const int ng = __popcll(heads);
    uint32_t xbase = col;
    bool amode = false, aff = false;
    if (AF.mask) {
      // slots of vertex a: [a Kv, (a + 1) Kv); an affine vertex owns A then t
      const int Kv = K / A;
      if (Kv * A != K || W != 3) ok = false;
      if (ok && lane < K) {
        const int a = lane / Kv, q = lane % Kv;
        uint32_t local;
        const uint32_t c = union_child(P, e2v[static_cast<size_t>(e) * A + a], local);
        aff = (AF.mask >> c) & 1u;
        xbase = 3 * a;
        amode = aff && q == 0;
        if (q == 0)
          for (int k = 0; k < 3; ++k)
            el.r[a][k] = aff ? AF.rest[c][3 * static_cast<size_t>(local) + k] : 0.0;
        const int want = aff ? (q == 0 ? 9 : (q == 1 ? 3 : -1)) : (q == 0 ? 3 : -1);
        if (want > 0 && sz != static_cast<uint32_t>(want)) ok = false;
        if (want < 0 && ii >= 2) ok = false;
      }
    } else if (total != static_cast<uint32_t>(N)) {
      ok = false;                                  // slots tile the DoFs
    }
    if (__any(!ok)) {
      if (lane == 0) atomicOr(flags, 1);
      continue;
    }
    if (lane < KT) {
      el.idx[lane] = ii;
      el.size[lane] = static_cast<uint8_t>(sz);
      el.col[lane] = static_cast<uint8_t>(col);
      el.xbase[lane] = static_cast<uint8_t>(xbase);
      el.amode[lane] = amode;
      el.aff[lane] = aff;
    }
    if (leads) {
      const int g = lanes_below(heads);
      el.head[g] = static_cast<uint8_t>(lane);
      el.members[g] = members;
      if (ii >= 2 && S.diag_blocks && !S.block_staging) el.diag[g] = diag_offset(S, ii - 2, sz);
    }
    // destinations of the block pairs, in coordinate order (at most 64 of them here)
    const uint32_t cstart = S.coord_outer[e];
    const int nt = __popcll(__ballot(leads && ii >= 2));
    const uint32_t pairs = nt * (nt + 1) / 2;
    uint32_t dest = 0;
    if (!S.block_staging && static_cast<uint32_t>(lane) < pairs) dest = S.lookups[cstart + lane];
    wave_lds_fence();
    // gradient
    for (int i = 0; i < K; ++i) {
      const int n = el.size[i];
      const uint32_t t = el.idx[i];
      if (S.grad_staging) {
        if (lane < n) {
          double c;
          const int x = xmap(el, i, lane, c);
          S.grad_staging[static_cast<size_t>(e) * S.grad_local + el.col[i] + lane] = c * el.h[NH + x];
        }
        continue;
      }
      if (t < 2) continue;
      int gs = -1;
      if (hot && el.aff[i] && n <= kHotGradMax) {
        if (lane == 0) {
          gs = hot_slot(table.gkey, kHotGrad, t - 2);
          if (gs >= 0) table.gsize[gs] = n;
        }
        gs = __shfl(gs, 0);
      }
      if (lane < n) {
        double c;
        const int x = xmap(el, i, lane, c);
        const double v = c * el.h[NH + x];
        if (gs >= 0) table.gval[threadIdx.x / 64][gs][lane] += v;
        else atomic_add_f64(S.gradient + (t - 2) + lane, v);
      }
    }
    // Hessian blocks of every valid group pair, in coordinate order
    uint32_t at = 0;
    for (int gi = 0; gi < ng; ++gi) {
      const int fi = el.head[gi];
      const uint32_t ti = el.idx[fi];
      if (ti < 2) continue;
      const int h = el.size[fi];
      for (int gj = gi; gj < ng; ++gj) {
        const int fj = el.head[gj];
        const uint32_t tj = el.idx[fj];
        if (tj < 2) continue;
        const int w = el.size[fj];
        const uint32_t coord = cstart + at;
        const uint32_t off = at < 64 ? __shfl(dest, static_cast<int>(at))
                                     : (S.block_staging ? 0u : S.lookups[coord]);
        ++at;
        double* dst = S.block_staging ? S.block_staging + 9 * static_cast<size_t>(coord) : S.blocks + off;
        double* dd = !S.block_staging && gi == gj && S.diag_blocks ? S.diag_blocks + el.diag[gi] : nullptr;
        int hs = -1;
        if (hot && el.aff[fi] && el.aff[fj] && h * w <= kHotBlockMax) {
          if (lane == 0) {
            hs = hot_slot(table.bkey, kHotBlocks, off);
            if (hs >= 0) {
              table.bsize[hs] = h * w;
              table.bdiag[hs] = dd ? el.diag[gi] : kHotEmpty;
            }
          }
          hs = __shfl(hs, 0);
        }
        const bool tr = !(ti < tj);
        const uint32_t inv = 65536u / w + 1;       // t / w for t < 144, w <= 12
        for (int t = lane; t < h * w; t += 64) {
          const int k = static_cast<int>((t * inv) >> 16), l = t - k * w;
          double v = 0.0;
          for (uint32_t ma = el.members[gi]; ma; ma &= ma - 1) {
            const int a = __ffs(ma) - 1;
            if (el.size[a] == 0) continue;
            double ca;
            const int xa = xmap(el, a, k, ca);
            for (uint32_t mb = el.members[gj]; mb; mb &= mb - 1) {
              const int b = __ffs(mb) - 1;
              if (el.size[b] == 0) continue;
              double cb;
              const int xb = xmap(el, b, l, cb);
              const int lo = min(xa, xb), hi = max(xa, xb);
              v += ca * cb * el.h[upper_index<N>(lo, hi)];
            }
          }
          // stored block: rows of the lower global index; (l, k) of a transposed block
          const int o = tr ? l * h + k : k * w + l;
          if (S.block_staging) {
            dst[o] = v;
          } else if (hs >= 0) {
            table.bval[threadIdx.x / 64][hs][o] += v;
          } else {
            atomic_add_f64(dst + o, v);
            if (dd) atomic_add_f64(dd + o, v);
          }
        }
      }
    }
    wave_lds_fence();                              // before the next element overwrites el
  }
  if (hot) hot_flush(table, S);
}

template <int ID>
__device__ __forceinline__ void gather(const UnionView& P, const uint32_t* e2v, uint32_t e,
                                       double (&x)[Kind<ID>::N]) {
  using T = Kind<ID>;
#pragma unroll
  for (int a = 0; a < T::A; ++a) {
    const uint32_t v = e2v[static_cast<size_t>(e) * T::A + a];
    const double* row = union_row(P, v);
#pragma unroll
    for (int i = 0; i < T::W; ++i) x[T::W * a + i] = row[i];
  }
}

// Scene parameters of one element; Baraff-Witkin picks its stretch coefficients from
// the current F (helpers.py:252-253: 0.01 below unit stretch, else 1).
template <int ID>
__device__ __forceinline__ void scene_params(const double* sp, const double* x, const double* p,
                                             double (&s)[Kind<ID>::S]) {
#pragma unroll
  for (int i = 0; i < Kind<ID>::S; ++i) s[i] = sp[i];
  if constexpr (ID == YSP_ENERGY_BARAFF_WITKIN) bw_stretch_coefficients(x, p, s[3], s[4]);
}

// Energy, gradient and packed Hessian of one element (not projected, but for the quadratic
// form, whose projection acts on its inner Hessian).
template <int ID>
__device__ __forceinline__ void element_eval(const double (&x)[Kind<ID>::N], const double* p,
                                             const double* sp, uint32_t method, double& E,
                                             double (&g)[Kind<ID>::N],
                                             double (&H)[Kind<ID>::N * (Kind<ID>::N + 1) / 2]) {
  if constexpr (ID == YSP_ENERGY_QUADRATIC_FORM) {
    quadratic_form_eval(x, sp, method, E, g, H);
  } else {
    double s[Kind<ID>::S];
    scene_params<ID>(sp, x, p, s);
    Kind<ID>::eval(x, p, s, E, g, H);
  }
}

// ----------------------------------------------------------------- vertex fast path
// Elements without affine vertices whose slots are one W-wide slot per local vertex (or
// padding): slot bookkeeping and scatter at compile-time vertex indices, so that no
// per-element array is indexed at run time (such an array would be placed in scratch
// memory). An element whose layout is anything else (a target vertex repeated inside
// the element) goes to a queue for the general kernel.
template <int NV>
struct VSlots {
  uint32_t idx[NV];   // seg_idx of the vertex's slot, 0 without one
  bool has[NV];       // the vertex owns a W-wide slot
  bool target[NV];    // ... with a target index (>= 2) in a group
  int rank[NV];       // rank of its group among the element's target groups
  int ntarget;
  bool ok;
};

template <int KT, int NV, int W>
__device__ __forceinline__ void load_vslots(const ScatterArgs& S, uint32_t e, VSlots<NV>& vs) {
  const uint32_t K = S.K;
  vs.ok = K <= static_cast<uint32_t>(KT);
  int grp[NV];
#pragma unroll
  for (int a = 0; a < NV; ++a) {
    vs.idx[a] = 0;
    vs.has[a] = false;
    grp[a] = -1;
  }
  int placement[KT];
  int ng = 0;
  uint32_t col = 0;
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    if (!vs.ok || static_cast<uint32_t>(i) >= K) continue;
    const size_t o = static_cast<size_t>(e) * K + i;
    const uint32_t ii = S.seg_idx[o];
    const uint32_t sz = S.seg_size[o];
    const int pm = S.perm[o];
    // a union's padding slot (index 0) holds no DoFs, whatever its size (the size makes
    // a vertex of a small child as wide as the union's widest child, e.g. next to
    // affine bodies)
    if (ii == 0) continue;
    int g = -1;
    if (pm != 0) {
      const int p = (pm < 0 ? -pm : pm) - 1;
#pragma unroll
      for (int k = 0; k < KT; ++k)
        if (k < ng && placement[k] == p) g = k;
      if (g < 0) {
        g = ng++;
#pragma unroll
        for (int k = 0; k < KT; ++k)
          if (k == g) placement[k] = p;
      }
    }
    if (sz == W) {
      const uint32_t v = col / W;
      if (v >= static_cast<uint32_t>(NV)) vs.ok = false;
#pragma unroll
      for (int a = 0; a < NV; ++a)
        if (v == static_cast<uint32_t>(a)) {
          vs.idx[a] = ii;
          vs.has[a] = true;
          grp[a] = g;
        }
    } else if (sz != 0) {
      vs.ok = false;
    }
    col += sz;
  }
  if (col != static_cast<uint32_t>(NV * W)) vs.ok = false;      // slots tile the DoFs
  vs.ntarget = 0;
#pragma unroll
  for (int a = 0; a < NV; ++a) {
    vs.target[a] = vs.has[a] && vs.idx[a] >= 2 && grp[a] >= 0;
    vs.ntarget += vs.target[a];
  }
#pragma unroll
  for (int a = 0; a < NV; ++a) {
    int r = 0;
#pragma unroll
    for (int b = 0; b < NV; ++b) {
      r += vs.target[b] && grp[b] < grp[a];
      if (b > a && vs.target[a] && vs.target[b] && grp[a] == grp[b]) vs.ok = false;
    }
    vs.rank[a] = r;
  }
}

// Gradient segments and Hessian blocks of vertex-layout elements (the semantics of the
// general scatter: pair of target-group ranks lo <= hi at coordinate coordStart +
// lo*n - lo(lo-1)/2 + (hi-lo), block oriented with the rows of the smaller target index).
// A wavefront calls these together (one per workgroup, lanes without an element with
// take == false): the lanes' segments or blocks meet in LDS, and consecutive lanes then
// write consecutive entries. Each lane writing its own block made 64 requests of every
// store or atomic where this makes 8 to 14: evaluating 27,000 hinges with atomics took 168 us,
// now 52, projecting four lists of such elements 100 us each, now 49. Staged, projecting 122,000
// hinges went from 113 to 90 us and the evaluations stayed as they were.
constexpr uint32_t kNowhere = 0xffffffffu;
template <int W>
struct WaveScatter {
  double v[kEB * W * W];
  uint32_t at[kEB], diag[kEB];
};

// put(destination of a lane's first entry, entry, value) for C entries of every lane that has
// a destination; lane-major in v.
template <int C, typename Put>
__device__ __forceinline__ void wave_put(const double* v, const uint32_t* at, Put put) {
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const uint32_t f = i * kEB + threadIdx.x, l = f / C, o = f % C;
    if (at[l] != kNowhere) put(at[l], o, v[f]);
  }
}

template <int NV, int W, int N>
__device__ __forceinline__ void scatter_vertex_gradient(const ScatterArgs& S, uint32_t e, bool take,
                                                        const VSlots<NV>& vs, const double (&g)[N],
                                                        WaveScatter<W>& w) {
#pragma unroll
  for (int a = 0; a < NV; ++a) {
    const bool mine = take && vs.has[a] && (S.grad_staging || vs.idx[a] >= 2);
    w.at[threadIdx.x] = !mine ? kNowhere : (S.grad_staging ? e : vs.idx[a] - 2);
#pragma unroll
    for (int k = 0; k < W; ++k) w.v[threadIdx.x * W + k] = g[W * a + k];
    wave_lds_fence();
    if (S.grad_staging)
      wave_put<W>(w.v, w.at, [&](uint32_t el, uint32_t o, double v) {
        S.grad_staging[static_cast<size_t>(el) * S.grad_local + W * a + o] = v;
      });
    else
      wave_put<W>(w.v, w.at,
                  [&](uint32_t d, uint32_t o, double v) { atomic_add_f64(S.gradient + d + o, v); });
    wave_lds_fence();
  }
}

// block(a, b, B): the W x W block of local vertices a <= b, called where take holds.
template <int NV, int W, typename BlockFn>
__device__ __forceinline__ void scatter_vertex_blocks(const ScatterArgs& S, uint32_t e, bool take,
                                                      const VSlots<NV>& vs, WaveScatter<W>& w,
                                                      BlockFn block) {
  if (!__any(take)) return;
  const uint32_t cstart = S.coord_outer[e];
  const int n = vs.ntarget;
#pragma unroll
  for (int a = 0; a < NV; ++a)
#pragma unroll
    for (int b = a; b < NV; ++b) {
      const bool mine = take && vs.target[a] && vs.target[b];
      uint32_t at = kNowhere, diag = kNowhere;
      if (mine) {
        double B[W][W];
        block(a, b, B);
        const int lo = min(vs.rank[a], vs.rank[b]), hi = max(vs.rank[a], vs.rank[b]);
        const uint32_t coord = cstart + static_cast<uint32_t>(lo * n - lo * (lo - 1) / 2 + (hi - lo));
        const bool tr = !(vs.idx[a] < vs.idx[b]);   // includes the diagonal block a == b
        at = S.block_staging ? coord : S.lookups[coord];
        if (a == b && S.diag_blocks && !S.block_staging) diag = diag_offset(S, vs.idx[a] - 2, W);
#pragma unroll
        for (int k = 0; k < W; ++k)
#pragma unroll
          for (int l = 0; l < W; ++l)
            w.v[threadIdx.x * (W * W) + (tr ? l * W + k : k * W + l)] = B[k][l];
      }
      w.at[threadIdx.x] = at;
      w.diag[threadIdx.x] = diag;
      wave_lds_fence();
      if (S.block_staging) {
        wave_put<W * W>(w.v, w.at, [&](uint32_t c, uint32_t o, double v) {
          S.block_staging[9 * static_cast<size_t>(c) + o] = v;
        });
      } else {
        wave_put<W * W>(w.v, w.at,
                        [&](uint32_t d, uint32_t o, double v) { atomic_add_f64(S.blocks + d + o, v); });
        if (a == b && S.diag_blocks)
          wave_put<W * W>(w.v, w.diag, [&](uint32_t d, uint32_t o, double v) {
            atomic_add_f64(S.diag_blocks + d + o, v);
          });
      }
      wave_lds_fence();
    }
}

// Evaluation of elements [first, last): gradient and Hessian, PSD test, scatter of what
// needs nothing else. The projection lives in a kernel of its own (below): with the
// eigensolver inlined behind the generated code every kind's kernel held both register
// sets and two copies of the scatter. Hessians of up to kProjectInline rows are projected in
// place all the same: 600,000 indefinite point pairs (6 x 6) took 311 us staged and 539 us with
// atomics when they were held, 175 and 398 us in place (one kernel with Jacobi sweeps and
// without the scatter through LDS: 210 and 1,313). The next size, 9 x 9 (point to edge), is
// better held: 613 us against 781 in one kernel.
constexpr int kProjectInline = 6;
template <int ID>
__host__ __device__ constexpr bool projects_later() {
  return ID != YSP_ENERGY_QUADRATIC_FORM && Kind<ID>::N > kProjectInline;
}

template <int ID, int KT>
__global__ void __launch_bounds__(kEB)
    energy_eval_kernel(UnionView P, const uint32_t* __restrict__ e2v, uint32_t first, uint32_t last,
                       const double* __restrict__ ep, const double* __restrict__ sp,
                       uint32_t method, ScatterArgs SA, int* __restrict__ flags, Held held) {
  using T = Kind<ID>;
  __shared__ WaveScatter<T::W> ws;
  // staged blocks are 3 x 3: a launch of any other width is refused whole (no lane alone:
  // the lanes that stay would read LDS words that those which left never wrote)
  if (SA.block_staging && T::W != 3) {
    if (threadIdx.x == 0) atomicOr(flags, 1);
    return;
  }
  const uint32_t i = first + blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = i < last;                    // the wavefront scatters together
  const uint32_t e = live ? i : last - 1;
  VSlots<T::A> vs;
  load_vslots<KT, T::A, T::W>(SA, e, vs);
  double x[T::N];
  gather<ID>(P, e2v, e, x);
  const double* p = ep + static_cast<size_t>(e) * T::P;
  double E, g[T::N], H[T::N * (T::N + 1) / 2];
  element_eval<ID>(x, p, sp, method, E, g, H);
  bool psd = true;
  if constexpr (ID != YSP_ENERGY_QUADRATIC_FORM)
    if (method != 0) {
      if constexpr (projects_later<ID>()) psd = is_psd<T::N>(H);
      else project_packed<T::N>(H, method);
    }
  const bool vertex = live && vs.ok, done = vertex && psd;
  scatter_vertex_gradient<T::A, T::W, T::N>(SA, e, vertex, vs, g, ws);
  scatter_vertex_blocks<T::A, T::W>(SA, e, done, vs, ws, [&](int a, int b, double (&B)[T::W][T::W]) {
#pragma unroll
    for (int k = 0; k < T::W; ++k)
#pragma unroll
      for (int l = 0; l < T::W; ++l) B[k][l] = hget<T::N>(H, T::W * a + k, T::W * b + l);
  });
  if (!live || done) return;
  const uint32_t slot = wave_reserve(held.counts, 1u);
  held.elem[slot] = e | (psd ? 0u : kHeldIndefinite) | (vs.ok ? 0u : kHeldGeneral);
#pragma unroll
  for (int i = 0; i < T::N * (T::N + 1) / 2; ++i) held.data[held_at<T::N>(slot, i)] = H[i];
  if (!vs.ok) {
    held.general[wave_reserve(held.counts + 1, 1u)] = slot;
#pragma unroll
    for (int i = 0; i < T::N; ++i)
      held.data[held_at<T::N>(slot, T::N * (T::N + 1) / 2 + i)] = g[i];
  }
}

// Projection of the held indefinite Hessians: scattered (vertex layouts) or written back
// for the general scatter. kFree: in the translation-free complement of four vertices.
template <int A, int W, int KT, bool kFree>
__global__ void __launch_bounds__(kEB)
    energy_project_kernel(uint32_t method, ScatterArgs SA, Held held) {
  constexpr int N = A * W, P = N * (N + 1) / 2;
  __shared__ WaveScatter<W> ws;
  const uint32_t count = held.counts[0], slot0 = blockIdx.x * blockDim.x;
  if (slot0 >= count) return;
  const uint32_t slot = min(slot0 + threadIdx.x, count - 1);
  const uint32_t word = held.elem[slot];
  const bool mine = slot0 + threadIdx.x < count && (word & kHeldIndefinite);
  if (!__any(mine)) return;                      // the wavefront scatters together
  constexpr int R = kFree ? 9 : N;               // dimension of the eigenproblem
  double D[R * (R + 1) / 2];                     // then the change of its spectrum
  if constexpr (kFree) {
    static_assert(A == 4 && W == 3, "four vertices");
    double H[P];
#pragma unroll
    for (int i = 0; i < P; ++i) H[i] = held.data[held_at<N>(slot, i)];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int l = k; l < 3; ++l)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            if (k == l && j < i) continue;
            double acc = 0.0;
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
              for (int b = 0; b < 4; ++b)
                acc += basis4(a, k) * basis4(b, l) * hget<12>(H, 3 * a + i, 3 * b + j);
            D[upper_index<9>(3 * k + i, 3 * l + j)] = acc;
          }
  } else {
#pragma unroll
    for (int i = 0; i < P; ++i) D[i] = held.data[held_at<N>(slot, i)];
  }
  clamp_change_packed<R>(D, method);
  // the Hessian again: not kept in registers across the eigensolver (the compiler must not
  // know that it is the same slot)
  uint32_t again = slot;
  asm volatile("" : "+v"(again));
  double* data = held.data + held_at<N>(again, 0);
  auto block = [&](int a, int b, double (&B)[W][W]) {
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j) {
        const int r = W * a + i, c = W * b + j;
        double v = data[8 * (r <= c ? upper_index<N>(r, c) : upper_index<N>(c, r))];
        if constexpr (kFree) {
#pragma unroll
          for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int l = 0; l < 3; ++l) {
              const double w = basis4(a, k) * basis4(b, l);
              if (w != 0.0) v = fma(w, hget<9>(D, 3 * k + i, 3 * l + j), v);
            }
        } else {
          v += hget<R>(D, r, c);
        }
        B[i][j] = v;
      }
  };
  if (mine && (word & kHeldGeneral)) {
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int b = a; b < A; ++b) {
        double B[W][W];
        block(a, b, B);
#pragma unroll
        for (int i = 0; i < W; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j)
            if (a < b || j >= i) data[8 * upper_index<N>(W * a + i, W * b + j)] = B[i][j];
      }
  }
  const bool take = mine && !(word & kHeldGeneral);
  if (!__any(take)) return;
  const uint32_t e = word & kHeldElement;
  VSlots<A> vs;
  load_vslots<KT, A, W>(SA, e, vs);
  scatter_vertex_blocks<A, W>(SA, e, take, vs, ws, block);
}

template <int ID>
__global__ void __launch_bounds__(kEB)
    energy_value_kernel(UnionView P, const uint32_t* __restrict__ e2v, uint32_t n,
                        const double* __restrict__ ep, const double* __restrict__ sp,
                        double* __restrict__ energy) {
  using T = Kind<ID>;
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  double x[T::N];
  gather<ID>(P, e2v, e, x);
  const double* p = ep + static_cast<size_t>(e) * T::P;
  double E, g[T::N], H[T::N * (T::N + 1) / 2];
  element_eval<ID>(x, p, sp, 0, E, g, H);
  energy[e] = E;
}

// Elements per round of evaluation, projection and general scatter: what a round holds (at
// most 94 MB) stays in the Infinity Cache between its kernels.
constexpr uint32_t kHeldRound = 131072;

template <int ID>
int launch_eval(const UnionView& U, const AffineView& AF, const uint32_t* e2v, uint32_t n,
                const double* ep, const double* sp, uint32_t method, const ScatterArgs& SA,
                int* flags, uint32_t* elem, uint32_t* general, double* data, hipStream_t s) {
  using T = Kind<ID>;
  auto run = [&](auto kt) {
    constexpr int KT = decltype(kt)::value;
    for (uint32_t first = 0, round = 0; first < n; first += kHeldRound, ++round) {
      const uint32_t m = std::min(kHeldRound, n - first);
      const Held held{reinterpret_cast<uint32_t*>(flags) + 1 + 2 * round, elem, general, data};
      const dim3 g(grid_for(m, kEB)), b(kEB);
      hipLaunchKernelGGL((energy_eval_kernel<ID, KT>), g, b, 0, s, U, e2v, first, first + m, ep, sp,
                         method, SA, flags, held);
      if constexpr (projects_later<ID>()) {
        if (method != 0)
          hipLaunchKernelGGL((energy_project_kernel<T::A, T::W, KT, (translation_free<ID>() &&
                                                                     T::A == 4 && T::W == 3)>),
                             g, b, 0, s, method, SA, held);
      }
      // usually nothing to do, or everything that an affine body drives
      hipLaunchKernelGGL((energy_scatter_kernel<T::A, T::W, KT>),
                         dim3(std::min<unsigned>(grid_for(m, kGW), AF.mask ? 256 : 64)), dim3(kGB),
                         0, s, U, AF, e2v, SA, flags, held);
    }
  };
  if (SA.K <= 8) run(std::integral_constant<int, 8>());
  else run(std::integral_constant<int, kSlotsMax>());
  return YSP_OK;
}


template <int ID>
void launch_values(const UnionView& U, const uint32_t* e2v, uint32_t n, const double* ep,
                   const double* sp, double* energy, hipStream_t s) {
  hipLaunchKernelGGL(energy_value_kernel<ID>, dim3(grid_for(n, kEB)), dim3(kEB), 0, s, U, e2v, n,
                     ep, sp, energy);
}


int check_view(const ysp_union_f64* u, uint32_t width, const char* who) {
  if (!u || u->num_children == 0 || u->num_children > YSP_MAX_UNION_CHILDREN || u->width != width) {
    ysp_set_error(__FILE__, __LINE__, who);
    return YSP_ERR_ARG;
  }
  return YSP_OK;
}

// Body of ysp_eval_element_energy for energy ID (flags: an unsupported slot layout, the
// elements queued for the general kernel; checked at the next ysp_check_deferred).
template <int ID>
int eval_energy(const ysp_union_f64* positions, const ysp_affine_children* affine,
                const uint32_t* elem2v, uint32_t n, const double* element_params,
                const double* scene_params, uint32_t projection_method,
                const ysp_scatter_args* out, void* stream, const char* who) {
  if (!out || projection_method > 2 || out->max_num_indices > static_cast<uint32_t>(kSlotsMax)) {
    ysp_set_error(__FILE__, __LINE__, who);
    return YSP_ERR_ARG;
  }
  if (n == 0) return YSP_OK;
  if (int rc = check_view(positions, Kind<ID>::W, who)) return rc;
  hipStream_t s = as_stream(stream);
  if (n > kHeldElement) {
    ysp_set_error(__FILE__, __LINE__, who);
    return YSP_ERR_ARG;
  }
  const ElementScratchOrder order(s);
  if (order.rc != YSP_OK) return order.rc;
  const uint32_t rounds = (n + kHeldRound - 1) / kHeldRound, most = std::min(n, kHeldRound);
  int* flag = static_cast<int*>(scratch(34, (1 + 2 * rounds) * sizeof(int)));
  uint32_t* elem = static_cast<uint32_t*>(scratch(46, 2 * sizeof(uint32_t) * most));
  double* data = static_cast<double*>(
      scratch(130, sizeof(double) * held_doubles<Kind<ID>::N>() * (static_cast<size_t>(most) + 8)));
  if (!flag || !elem || !data) return YSP_ERR_HIP;
  YSP_CHECK(hipMemsetAsync(flag, 0, (1 + 2 * rounds) * sizeof(int), s));
  const UnionView U = make_view(positions);
  const ScatterArgs SA = make_scatter(out);
  AffineView AF{};
  if (affine) {
    AF.mask = affine->mask & ((1u << positions->num_children) - 1u);
    for (int c = 0; c < YSP_MAX_UNION_CHILDREN; ++c) {
      AF.body[c] = affine->vertex_body[c];
      AF.rest[c] = affine->rest_position[c];
      if (((AF.mask >> c) & 1u) && !AF.rest[c]) {
        ysp_set_error(__FILE__, __LINE__, "element energy: affine child without rest data");
        return YSP_ERR_ARG;
      }
    }
  }
  launch_eval<ID>(U, AF, elem2v, n, element_params, scene_params, projection_method, SA, flag,
                  elem, elem + most, data, s);
  YSP_CHECK_LAUNCH();
  return defer_flag_check(flag, s, "element energy: slot layout does not match the element's vertices");
}

// Body of ysp_element_energy_values for energy ID: energy[e] of every element.
template <int ID>
int energy_values(const ysp_union_f64* positions, const uint32_t* elem2v, uint32_t n,
                  const double* element_params, const double* scene_params, double* energy,
                  void* stream, const char* who) {
  if (n == 0) return YSP_OK;
  if (int rc = check_view(positions, Kind<ID>::W, who)) return rc;
  launch_values<ID>(make_view(positions), elem2v, n, element_params, scene_params, energy,
                    as_stream(stream));
  YSP_CHECK_LAUNCH();
  return YSP_OK;
}

}  // namespace
}  // namespace ysp
