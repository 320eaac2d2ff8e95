// HEOM Liouvillian apply on gfx950: one table-driven gather kernel serves the
// forward operator (tfqmr_double/calc_ax_tfqmr_omp.f90, td/calcderiv_omp.f90)
// and its real transpose (bicg/calc_atrx_bicg_omp.f90 in the reference's
// BiCG convention).
//
// Mapping: the d*d elements of one output ADO are spread over min(d*d, 256)
// lanes of a 256-thread workgroup.  Element (i, j) lives at complex offset
// i + j*d (the reference's Fortran order), so consecutive lanes read
// consecutive rows: a column of a neighbour block is one coalesced segment.
// The ADO's own block is staged in LDS for the H commutator; neighbour blocks
// are gathered straight from HBM/L2, one element per lane per term, because c
// and c^+ are signed partial permutations: (c X)(i, j) = s_i * X(p_i, j).
//
// An ADO below the top tier has one coupling per drawer (72 to 112), a
// top-tier ADO one per drawer it holds (2 to 4), so the two run apart:
// "heavy" workgroups take one ADO each, its couplings staged in LDS and
// sliced over the lanes (256 / (d*d) slices at d = 4, one at d = 16), four
// gathered at a time; "light" workgroups take 256 / (d*d) top-tier ADOs at a
// time and a run of such groups, so the operator maps and H are staged once.
#include "heomq_kernels.hpp"

#include <algorithm>

namespace heomq {

template <typename T> struct V2;
template <> struct V2<double> { using type = double2; };
template <> struct V2<float> { using type = float2; };

constexpr int kMaxOps = 12;   // 2 * norbs * nspin for norbs <= 3
constexpr int kStage = 128;   // couplings staged in LDS at once

// One coupling with its record: coefficients with the entry's signs, the
// neighbour, the operator (0xff: no term) and the dagger flag.
template <typename T>
struct Coupling {
  T clr, cli, crr, cri;
  int32_t nbr;
  uint8_t op, dag;
};

template <typename T>
__device__ inline Coupling<T> to_coupling(const DevOperator& op, const DevEntry en) {
  const double2* r = reinterpret_cast<const double2*>(op.rec + en.rec);
  const double2 l = r[0], q = r[1];
  const T sl = (en.flags & 2) ? (T)-1 : (T)1, sr = (en.flags & 4) ? (T)-1 : (T)1;
  return Coupling<T>{sl * (T)l.x, sl * (T)l.y, sr * (T)q.x, sr * (T)q.y, en.nbr, en.op, (uint8_t)(en.flags & 1)};
}

// Couplings cs[0], cs[stride], .. (nv of them, at most U) of element (i, j):
// every neighbour element is loaded before any is used.  smap[o * 2 * D + i] = (p_i + 1) * s_i of the left factor,
// smap[o * 2 * D + D + j] the same of the right factor, 0 for no term.
template <int D, typename T, bool TRANS, int U>
__device__ inline void add_couplings(const Coupling<T>* cs, int stride, int nv, const int8_t* smap,
                                     const typename V2<T>::type* __restrict__ xv, int i, int j, int64_t trace_pos,
                                     int trace_elem, T& ar, T& ai) {
  using V = typename V2<T>::type;
  V vl[U], vr[U];
  int ml[U], mr[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    vl[u] = V{0, 0};
    vr[u] = V{0, 0};
    ml[u] = mr[u] = 0;
    if (u >= nv) continue;
    const Coupling<T>& c = cs[u * stride];
    if (c.op == 0xff) continue;
    ml[u] = smap[c.op * 2 * D + i];
    mr[u] = smap[c.op * 2 * D + D + j];
    const V* __restrict__ xn = xv + (int64_t)c.nbr * (D * D);
    const int pl = (ml[u] < 0 ? -ml[u] : ml[u]) - 1, pr = (mr[u] < 0 ? -mr[u] : mr[u]) - 1;
    const int el = c.dag ? j + pl * D : pl + j * D, er = c.dag ? pr + i * D : i + pr * D;
    if (ml[u] != 0 && !(TRANS && c.nbr == trace_pos && el == trace_elem)) vl[u] = xn[el];
    if (mr[u] != 0 && !(TRANS && c.nbr == trace_pos && er == trace_elem)) vr[u] = xn[er];
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u >= nv) break;
    __builtin_amdgcn_sched_barrier(0);   // one coupling's coefficients in registers at a time
    const Coupling<T>& c = cs[u * stride];
    const T cj = c.dag ? (T)-1 : (T)1;
    const T sl = ml[u] < 0 ? (T)-1 : (T)1, sr = mr[u] < 0 ? (T)-1 : (T)1;   // a zero element where there is no term
    const T lx = sl * vl[u].x, ly = sl * cj * vl[u].y, rx = sr * vr[u].x, ry = sr * cj * vr[u].y;
    ar += c.clr * lx - c.cli * ly;
    ai += c.clr * ly + c.cli * lx;
    ar += c.crr * rx - c.cri * ry;
    ai += c.crr * ry + c.cri * rx;
  }
}

// One coupling of KC elements (i, j0 + q dj) of a lane (d = 64), every
// neighbour element loaded before any is used; smap as above.
template <int D, typename T, bool TRANS, int KC>
__device__ inline void add_coupling_elems(const Coupling<T>& c, const int8_t* smap,
                                          const typename V2<T>::type* __restrict__ xv, int i, int j0, int dj,
                                          int64_t trace_pos, int trace_elem, T* ar, T* ai) {
  using V = typename V2<T>::type;
  if (c.op == 0xff) return;   // block-uniform
  const V* __restrict__ xn = xv + (int64_t)c.nbr * (D * D);
  const bool zero = TRANS && c.nbr == trace_pos;
  const int ml = smap[c.op * 2 * D + i], pl = (ml < 0 ? -ml : ml) - 1;
  V vl[KC], vr[KC];
  int mr[KC];
#pragma unroll
  for (int q = 0; q < KC; ++q) {
    const int j = j0 + q * dj;
    mr[q] = smap[c.op * 2 * D + D + j];
    const int pr = (mr[q] < 0 ? -mr[q] : mr[q]) - 1;
    const int el = c.dag ? j + pl * D : pl + j * D, er = c.dag ? pr + i * D : i + pr * D;
    vl[q] = V{0, 0};
    vr[q] = V{0, 0};
    if (ml != 0 && !(zero && el == trace_elem)) vl[q] = xn[el];
    if (mr[q] != 0 && !(zero && er == trace_elem)) vr[q] = xn[er];
  }
  const T cj = c.dag ? (T)-1 : (T)1, sl = ml < 0 ? (T)-1 : (T)1;
#pragma unroll
  for (int q = 0; q < KC; ++q) {
    const T sr = mr[q] < 0 ? (T)-1 : (T)1;   // a zero element where there is no term
    const T lx = sl * vl[q].x, ly = sl * cj * vl[q].y, rx = sr * vr[q].x, ry = sr * cj * vr[q].y;
    ar[q] += c.clr * lx - c.cli * ly;
    ai[q] += c.clr * ly + c.cli * lx;
    ar[q] += c.crr * rx - c.cri * ry;
    ai[q] += c.crr * ry + c.cri * rx;
  }
}

// What a workgroup stages once: the operators' maps and, for d <= 16, H by
// rows with the row index fastest (16 rows of one column index are
// consecutive: no bank conflicts).
template <int D>
struct DenseLds {
  static constexpr bool kH = D <= 16;
  int8_t smap[kMaxOps * 2 * D];
  uint8_t hn[kH ? D : 1];
  uint8_t hc[kH ? D * D : 1];
  double2 hv[kH ? D * D : 1];
  __device__ void stage(const DevOperator& op) {
    for (int k = threadIdx.x; k < op.nop * 2 * D; k += 256) {
      const int o = k / (2 * D), r = k % (2 * D), side = r / D, i = r % D;
      const int8_t* m = op.opmap + (o * 4 + 2 * side) * D;
      smap[k] = m[i] < 0 ? (int8_t)0 : (int8_t)((m[i] + 1) * m[D + i]);
    }
    if (kH) {
      if (threadIdx.x < D) hn[threadIdx.x] = (uint8_t)op.hnnz[threadIdx.x];
      for (int k = threadIdx.x; k < D * D; k += 256) {
        const int i = k % D, t = k / D;
        if (t >= op.hnnz[i]) continue;
        hc[k] = (uint8_t)op.hcol[i * D + t];
        hv[k] = reinterpret_cast<const double2*>(op.hval)[i * D + t];
      }
    }
  }
  // i hsign (H X - X H)(i, j) + gamma X(i, j) of the block `self` (LDS)
  template <typename T>
  __device__ void same_tier(const DevOperator& op, const typename V2<T>::type* self, T gr, T gi, int i, int j, T& ar,
                            T& ai) const {
    using V = typename V2<T>::type;
    const V xe = self[i + j * D];
    T cr = 0, ci = 0;
    const int ni = kH ? (int)hn[i] : op.hnnz[i];
#pragma unroll 1
    for (int t = 0; t < ni; ++t) {            // (H X)(i, j)
      const int c = kH ? (int)hc[t * D + i] : op.hcol[i * D + t];
      const double2 h = kH ? hv[t * D + i] : reinterpret_cast<const double2*>(op.hval)[i * D + t];
      const V v = self[c + j * D];
      cr += (T)h.x * v.x - (T)h.y * v.y;
      ci += (T)h.x * v.y + (T)h.y * v.x;
    }
    const int nj = kH ? (int)hn[j] : op.hnnz[j];
#pragma unroll 1
    for (int t = 0; t < nj; ++t) {            // (X H)(i, j) = sum_k X(i, k) conj(H(j, k))
      const int c = kH ? (int)hc[t * D + j] : op.hcol[j * D + t];
      const double2 h = kH ? hv[t * D + j] : reinterpret_cast<const double2*>(op.hval)[j * D + t];
      const V v = self[i + c * D];
      cr -= (T)h.x * v.x + (T)h.y * v.y;
      ci -= (T)h.x * v.y - (T)h.y * v.x;
    }
    const T hs = (T)op.hsign;
    ar += gr * xe.x - gi * xe.y - hs * ci;
    ai += gr * xe.y + gi * xe.x + hs * cr;
  }
};

// Blocks [0, n_heavy) take one ADO below the top tier each; the rest take
// `run` groups of 256 / min(d*d, 256) consecutive top-tier ADOs.
//
// Bound by the latency of the dependent loads (entry -> record -> neighbour
// element) and, at d = 16, by HBM and the Infinity Cache: every top-tier block
// is read by its own workgroup and by the three heavy ADOs above it.  Staging
// the couplings in LDS takes entry and record out of the element's chain, and
// the couplings in flight (4 heavy and 3 light at d = 16, 2 and 2 at d = 4)
// are the most that keep 80 VGPRs without scratch, 6 waves per SIMD.  FP64
// forward, with one ADO per workgroup slot and its couplings walked one by one
// before: 1415 -> 513 us at two-impurity size (M = 112, L = 3; 962 MB, 1.9
// TB/s), 71 -> 15 us and 441 -> 216 us at the single impurity's M = 72, L = 3
// and 4.  At d = 64 a lane has 16 elements; KC of them share a walk over the
// couplings, with 2 KC gathers in flight, and the couplings are staged once
// where they fit.  Three orbitals, M = 48, FP64 (KC = 8) forward at L = 1 / 2 / 3:
// 284 / 389 / 1612 us with one element at a time, 122 / 156 / 1034 us now (KC = 4:
// 140 / 186 / 1032; KC = 16, with 500 bytes of scratch a lane: 117 / 152 / 1354);
// FP32 (KC = 4, four workgroups per CU) 265 / 358 / 934 -> 135 / 176 / 671 us (KC =
// 8: 119 / 151 / 828).  Ordering the heavy workgroups among the light ones by their
// neighbours' place gave 597 against 622 us at an earlier stage, for a table
// built per context: not kept.
template <int D, typename T, bool TRANS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 16 ? 6 : 2)))
k_apply(const DevOperator op, const T* __restrict__ x, T* __restrict__ y, int64_t trace_pos, int run) {
  using V = typename V2<T>::type;
  constexpr int E = D * D;
  constexpr int LANES = E < 256 ? E : 256;
  constexpr int EPT = E / LANES;
  constexpr int APB = 256 / LANES;   // ADOs of a light group, slices of a heavy ADO
  constexpr int U = D == 4 ? 2 : 4, UL = D == 4 ? 2 : 3;   // couplings in flight, heavy and light
  constexpr int KC = EPT > 1 ? (sizeof(T) == 8 ? 8 : 4) : 1;   // d = 64: elements of a lane in flight instead
  __shared__ V xs[EPT == 1 ? 512 : E];
  __shared__ DenseLds<D> tab;
  __shared__ Coupling<T> s_c[kStage];
  const int tid = threadIdx.x;
  const int slot = APB > 1 ? tid / LANES : 0, lane = tid - slot * LANES;   // one ADO per group: uniform addresses
  const V* __restrict__ xv = reinterpret_cast<const V*>(x);
  V* __restrict__ yv = reinterpret_cast<V*>(y);
  const int64_t n_heavy = op.n_heavy;
  const int light_max = op.light_max;
  tab.stage(op);

  if ((int64_t)blockIdx.x < n_heavy) {   // block-uniform
    const int64_t a = blockIdx.x;
    for (int e = tid; e < E; e += 256) {
      V v = xv[a * E + e];
      if (TRANS && a == trace_pos && e == op.trace_elem) v = V{0, 0};
      xs[e] = v;
    }
    const T gr = (T)op.gam[2 * a], gi = (T)op.gam[2 * a + 1];
    const int64_t p0 = op.rowptr[a], p1 = op.rowptr[a + 1];
    auto stage_heavy = [&](int64_t q0) {
      const int n = (int)(p1 - q0 < kStage ? p1 - q0 : kStage);
      __syncthreads();   // the previous stage is read
      if (tid < n) s_c[tid] = to_coupling<T>(op, op.ent[q0 + tid]);
      __syncthreads();
      return n;
    };
    if constexpr (EPT > 1) {
      int n = 0;
      for (int k0 = 0; k0 < EPT; k0 += KC) {
        T ar[KC] = {}, ai[KC] = {};
        for (int64_t q0 = p0; q0 < p1; q0 += kStage) {
          if (k0 == 0 || p1 - p0 > kStage) n = stage_heavy(q0);   // one stage serves every pass where all couplings fit
          for (int c = 0; c < n; ++c)
            add_coupling_elems<D, T, TRANS, KC>(s_c[c], tab.smap, xv, lane % D, (lane + k0 * LANES) / D, LANES / D,
                                                trace_pos, op.trace_elem, ar, ai);
        }
        if (k0 == 0) __syncthreads();   // xs is staged (also for an ADO without couplings)
#pragma unroll
        for (int q = 0; q < KC; ++q) {
          const int e = lane + (k0 + q) * LANES;
          tab.template same_tier<T>(op, xs, gr, gi, e % D, e / D, ar[q], ai[q]);
          yv[a * E + e] = V{ar[q], ai[q]};
        }
      }
    } else {
      const int e = lane;
      T ar = 0, ai = 0;
      for (int64_t q0 = p0; q0 < p1; q0 += kStage) {
        const int n = stage_heavy(q0);
        for (int c0 = slot; c0 < n; c0 += APB * U) {
          const int nv = (n - c0 + APB - 1) / APB;
          add_couplings<D, T, TRANS, U>(s_c + c0, APB, nv < U ? nv : U, tab.smap, xv, e % D, e / D, trace_pos,
                                        op.trace_elem, ar, ai);
        }
      }
      __syncthreads();   // xs and the tables are staged (also for an ADO without couplings)
      if (slot == 0) tab.template same_tier<T>(op, xs, gr, gi, e % D, e / D, ar, ai);
      if (APB > 1) {   // sum the slices (fixed pairing)
        __syncthreads();   // slice 0 has read xs
        xs[tid] = V{ar, ai};
        __syncthreads();
        for (int half = APB / 2; half > 0; half >>= 1) {
          if (slot < half) {
            const V o = xs[tid + half * LANES];
            xs[tid].x += o.x;
            xs[tid].y += o.y;
          }
          __syncthreads();
        }
        ar = xs[tid].x;
        ai = xs[tid].y;
      }
      if (slot == 0) yv[a * E + e] = V{ar, ai};
    }
    return;
  }

  // Light groups: the couplings of the whole run are staged first (`per` of
  // each ADO; more than that only in a run of one, restaged chunk by chunk).
  // A group's own elements are loaded one group ahead and staged in
  // alternating buffers, so a group has one barrier.
  const int64_t g0 = ((int64_t)blockIdx.x - n_heavy) * run;
  const int64_t groups = (op.n_ado - n_heavy + APB - 1) / APB;
  const int nr = (int)(groups - g0 < run ? groups - g0 : run);
  const int64_t a0 = n_heavy + g0 * APB;
  const int per = light_max < kStage / APB ? light_max : kStage / APB;
  auto stage_light = [&](int c0) {
    for (int k = tid; k < nr * APB * per; k += 256) {
      const int64_t sa = a0 + k / per;
      int64_t p = 0, pe = 0;
      if (sa < op.n_ado) {
        p = op.rowptr[sa] + c0 + k % per;
        pe = op.rowptr[sa + 1];
      }
      s_c[k] = to_coupling<T>(op, p < pe ? op.ent[p] : DevEntry{0, 0, 0, 0xff});
    }
  };
  V own{0, 0};
  if (EPT == 1 && a0 + slot < op.n_ado) own = xv[(a0 + slot) * E + lane];
  stage_light(0);
  __syncthreads();   // couplings and tables are staged
  for (int r = 0; r < nr; ++r) {
    const int64_t a = a0 + (int64_t)r * APB + slot;
    const bool active = a < op.n_ado;
    V* xr = EPT == 1 ? &xs[(r & 1) * 256] : xs;
    if (EPT == 1) {
      xr[tid] = TRANS && a == trace_pos && lane == op.trace_elem ? V{0, 0} : own;
      if (r + 1 < nr && a + APB < op.n_ado) own = xv[(a + APB) * E + lane];
    } else {
      __syncthreads();   // the previous group has read xs
      for (int f = tid; f < E; f += 256)
        xs[f] = TRANS && a == trace_pos && f == op.trace_elem ? V{0, 0} : xv[a * E + f];
    }
    V g{0, 0};
    if (active) g = V{(T)op.gam[2 * a], (T)op.gam[2 * a + 1]};
    if constexpr (EPT > 1) {
      for (int k0 = 0; k0 < EPT; k0 += KC) {
        T ar[KC] = {}, ai[KC] = {};
        for (int c0 = 0; c0 < light_max; c0 += per) {
          if (per < light_max) {   // uniform
            __syncthreads();
            stage_light(c0);
            __syncthreads();
          }
          for (int u = 0; u < per; ++u)
            add_coupling_elems<D, T, TRANS, KC>(s_c[r * per + u], tab.smap, xv, lane % D, (lane + k0 * LANES) / D,
                                                LANES / D, trace_pos, op.trace_elem, ar, ai);
        }
        if (k0 == 0) __syncthreads();   // xs is staged
#pragma unroll
        for (int q = 0; q < KC; ++q) {
          const int e = lane + (k0 + q) * LANES;
          tab.template same_tier<T>(op, xs, g.x, g.y, e % D, e / D, ar[q], ai[q]);
          yv[a * E + e] = V{ar[q], ai[q]};
        }
      }
    } else {
      const int e = lane;
      T ar = 0, ai = 0;
      for (int c0 = 0; c0 < light_max; c0 += per) {
        if (per < light_max) {   // uniform
          __syncthreads();
          stage_light(c0);
          __syncthreads();
        }
        if (active)
          for (int u = 0; u < per; u += UL)
            add_couplings<D, T, TRANS, UL>(&s_c[(r * APB + slot) * per + u], 1, per - u < UL ? per - u : UL, tab.smap,
                                           xv, e % D, e / D, trace_pos, op.trace_elem, ar, ai);
      }
      __syncthreads();   // xs is staged
      if (active) {
        tab.template same_tier<T>(op, xr + slot * E, g.x, g.y, e % D, e / D, ar, ai);
        yv[a * E + e] = V{ar, ai};
      }
    }
  }
}

// Forward trace row: y(d,d,trace_pos) = tr x0 (calc_ax_tfqmr_omp.f90:492-495).
template <typename T>
__global__ void k_trace_fwd(const T* __restrict__ x, T* __restrict__ y, int d, int64_t pos, int elem) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  T sr = 0, si = 0;
  for (int i = 0; i < d; ++i) {
    sr += x[2 * (i + i * d)];
    si += x[2 * (i + i * d) + 1];
  }
  const int64_t o = 2 * ((int64_t)pos * d * d + elem);
  y[o] = sr;
  y[o + 1] = si;
}

// Transposed trace row: z0(i,i) += w(d,d,trace_pos).
template <typename T>
__global__ void k_trace_trn(const T* __restrict__ w, T* __restrict__ z, int d, int64_t pos, int elem) {
  const int i = threadIdx.x;
  if (i >= d || blockIdx.x != 0) return;
  const int64_t o = 2 * ((int64_t)pos * d * d + elem);
  z[2 * (i + i * d)] += w[o];
  z[2 * (i + i * d) + 1] += w[o + 1];
}

// Light workgroups take up to kLightRunMax groups each (fewer when their
// couplings would not fit the stage) while at least kLightBlocksMin workgroups
// remain: 16 per CU, so a run never leaves the chip idle.
constexpr int kLightRunMax = 8, kLightBlocksMin = 4096;

template <int D, typename T>
static hipError_t launch_d(const DevOperator& op, const T* x, T* y, int64_t trace_pos, hipStream_t s) {
  constexpr int E = D * D;
  constexpr int LANES = E < 256 ? E : 256;
  constexpr int APB = 256 / LANES;
  if (op.n_ado <= 0) return hipSuccess;
  const int64_t groups = (op.n_ado - op.n_heavy + APB - 1) / APB;
  const int64_t fit = std::max<int64_t>(1, kStage / (APB * (int64_t)op.light_max));   // runs whose couplings fit the stage
  const int run = (int)std::min({fit, (int64_t)kLightRunMax, std::max<int64_t>(1, groups / kLightBlocksMin)});
  const int64_t blocks = op.n_heavy + (groups + run - 1) / run;
  if (op.transposed)
    hipLaunchKernelGGL((k_apply<D, T, true>), dim3((unsigned)blocks), dim3(256), 0, s, op, x, y, trace_pos, run);
  else
    hipLaunchKernelGGL((k_apply<D, T, false>), dim3((unsigned)blocks), dim3(256), 0, s, op, x, y, trace_pos, run);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  if (trace_pos >= 0) {
    if (op.transposed)
      hipLaunchKernelGGL((k_trace_trn<T>), dim3(1), dim3(64), 0, s, x, y, D, trace_pos, op.trace_elem);
    else
      hipLaunchKernelGGL((k_trace_fwd<T>), dim3(1), dim3(64), 0, s, x, y, D, trace_pos, op.trace_elem);
    err = hipGetLastError();
  }
  return err;
}

template <typename T>
static hipError_t launch_any(const DevOperator& op, const T* x, T* y, int64_t trace_pos, hipStream_t s) {
  switch (op.d) {
    case 4: return launch_d<4, T>(op, x, y, trace_pos, s);
    case 16: return launch_d<16, T>(op, x, y, trace_pos, s);
    case 64: return launch_d<64, T>(op, x, y, trace_pos, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_apply_f64(const DevOperator& op, const double* x, double* y, int64_t trace_pos, hipStream_t s) {
  return launch_any<double>(op, x, y, trace_pos, s);
}
hipError_t launch_apply_f32(const DevOperator& op, const float* x, float* y, int64_t trace_pos, hipStream_t s) {
  return launch_any<float>(op, x, y, trace_pos, s);
}

// ---------------------------------------------------------------------------
// BiCG convention around the same operator (tier-0 block only; element (i, j)
// at i + j*d; lower triangle i > j).
// ---------------------------------------------------------------------------
// x0: real diagonal, upper = conj(lower)^T (calc_ax_bicg_omp.f90:70-77)
__global__ void k_bicg_herm_in(int d, double* __restrict__ x) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= d * d) return;
  const int i = e % d, j = e / d;
  if (i == j) x[2 * e + 1] = 0.0;
  else if (i < j) {   // upper element reads the lower one, which no thread writes
    const int t = j + i * d;
    x[2 * e] = x[2 * t];
    x[2 * e + 1] = -x[2 * t + 1];
  }
}
// y0 (or w0): upper triangle zeroed, diagonal real (calc_ax_bicg_omp.f90:330-337;
// calc_atrx_bicg_omp.f90:103-110)
__global__ void k_bicg_lower(int d, double* __restrict__ y) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= d * d) return;
  const int i = e % d, j = e / d;
  if (i == j) y[2 * e + 1] = 0.0;
  else if (i < j) { y[2 * e] = 0.0; y[2 * e + 1] = 0.0; }
}
// z0 folded onto its lower triangle: the transpose of k_bicg_herm_in
// (lower += conj(upper)^T, diagonal real, upper zero); each lower thread owns
// its mirror element
__global__ void k_bicg_fold(int d, double* __restrict__ z) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= d * d) return;
  const int i = e % d, j = e / d;
  if (i == j) z[2 * e + 1] = 0.0;
  else if (i > j) {
    const int t = j + i * d;
    z[2 * e] += z[2 * t];
    z[2 * e + 1] -= z[2 * t + 1];
    z[2 * t] = 0.0;
    z[2 * t + 1] = 0.0;
  }
}

hipError_t launch_herm_from_lower_f64(int d, double* x, hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_herm_in, dim3((d * d + 255) / 256), dim3(256), 0, s, d, x);
  return hipGetLastError();
}

hipError_t launch_lower_tier0_f64(int d, double* x, hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_lower, dim3((d * d + 255) / 256), dim3(256), 0, s, d, x);
  return hipGetLastError();
}

hipError_t launch_apply_bicg_f64(const DevOperator& op, double* x, double* y, hipStream_t s) {
  const int d = op.d;
  hipLaunchKernelGGL(k_bicg_herm_in, dim3((d * d + 255) / 256), dim3(256), 0, s, d, x);
  if (hipError_t e = hipGetLastError()) return e;
  DevOperator o = op;
  o.trace_elem = 0;   // y(1,1) of tier 0 = tr rho0 (calc_ax_bicg_omp.f90:321-324)
  if (hipError_t e = launch_any<double>(o, x, y, 0, s)) return e;
  hipLaunchKernelGGL(k_bicg_lower, dim3((d * d + 255) / 256), dim3(256), 0, s, d, y);
  return hipGetLastError();
}

hipError_t launch_apply_transpose_bicg_f64(const DevOperator& op, double* w, double* z, hipStream_t s) {
  const int d = op.d;
  hipLaunchKernelGGL(k_bicg_lower, dim3((d * d + 255) / 256), dim3(256), 0, s, d, w);
  if (hipError_t e = hipGetLastError()) return e;
  DevOperator o = op;
  o.trace_elem = 0;   // w(1,1) is the trace row's dual: kept out of L^T, added to the diagonal of z0
  if (hipError_t e = launch_any<double>(o, w, z, 0, s)) return e;
  hipLaunchKernelGGL(k_bicg_fold, dim3((d * d + 255) / 256), dim3(256), 0, s, d, z);
  return hipGetLastError();
}

}  // namespace heomq
