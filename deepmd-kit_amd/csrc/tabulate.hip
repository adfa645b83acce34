// Tabulated (compressed) se_a embedding: tabulate_fusion_se_a forward, grad,
// grad_grad.
//
// Semantics (reference): source/lib/src/tabulate.cc:45-73 (locate_xx: two
// strides + linear extrapolation), :122-158 (quintic and its derivative),
// :162-232 (forward with the is_sorted padding fold: the first slot whose x
// equals the last slot's x and whose em[1:4] are zero stands for all the
// remaining slots, weight nnei - j), :234-341 (grad), :343-447 (grad_grad).
//
// Four basis functions (the se_a env matrix, op and fused model alike): one
// wavefront an atom (several in the backward where atoms are few), channels on
// the lanes, see k_tab4_fwd / k_tab4_bwd below; the backward of narrow nets puts
// the slots there (k_tab4_bwd_narrow).
// Other basis dimensions (9, 16, 25) and grad_grad: one workgroup an atom;
// forward and grad_grad put the L channels on the threads and walk the
// neighbours, grad puts the neighbours on the threads and walks the channels,
// with dy for the atom staged in LDS.
#include "dpk_common.h"

namespace dpk {
namespace {

template <typename T>
struct TabInfo {
  T lower, upper, vmax, stride0, stride1;
  int first;    // int((upper - lower) / stride0)
  int tail;     // table index of the high tail
  int last;     // nspline - 1: interval indices are clamped to the table
};

template <typename T>
TabInfo<T> make_info(const T* h, int nspline) {
  TabInfo<T> ti;
  ti.lower = h[0];
  ti.upper = h[1];
  ti.vmax = h[2];
  ti.stride0 = h[3];
  ti.stride1 = h[4];
  ti.first = (int)((ti.upper - ti.lower) / ti.stride0);
  T bxx = std::nextafter(ti.vmax, ti.lower);
  ti.tail = ti.first + (int)((bxx - ti.upper) / ti.stride1);
  ti.last = nspline - 1;
  return ti;
}

template <typename T>
__device__ __forceinline__ void locate(const TabInfo<T>& ti, T xx, int& idx, T& x, T& ext) {
  ext = T(0);
  if (xx < ti.lower) {
    idx = 0;
    x = T(0);
    ext = xx - ti.lower;
  } else if (xx < ti.upper) {
    idx = (int)((xx - ti.lower) / ti.stride0);
    x = xx - ((T)idx * ti.stride0 + ti.lower);
  } else if (xx < ti.vmax) {
    idx = ti.first + (int)((xx - ti.upper) / ti.stride1);
    x = xx - ((T)(idx - ti.first) * ti.stride1 + ti.upper);
  } else {
    idx = ti.tail;
    x = ti.vmax - ((T)(idx - ti.first) * ti.stride1 + ti.upper);
    ext = xx - ti.vmax;
  }
  idx = idx < 0 ? 0 : (idx > ti.last ? ti.last : idx);
}

// value (with extrapolation) and first derivative of channel k's piece
template <typename T>
__device__ __forceinline__ void piece(const T* __restrict__ c, T x, T ext, T& val, T& grd) {
  const T a0 = c[0], a1 = c[1], a2 = c[2], a3 = c[3], a4 = c[4], a5 = c[5];
  grd = a1 + (T(2) * a2 + (T(3) * a3 + (T(4) * a4 + T(5) * a5 * x) * x) * x) * x;
  val = a0 + (a1 + (a2 + (a3 + (a4 + a5 * x) * x) * x) * x) * x + grd * ext;
}

template <typename T>
__device__ __forceinline__ bool fold_hit(const T* __restrict__ em_x, const T* __restrict__ em,
                                         int nnei, int nd, int jj, T last) {
  return em_x[jj] == last && em[jj * nd + 1] == T(0) && em[jj * nd + 2] == T(0) &&
         em[jj * nd + 3] == T(0);
}

template <typename T, int ND>
__global__ void k_tab_fwd(T* __restrict__ out, const T* __restrict__ table, TabInfo<T> ti,
                          const T* __restrict__ em_x, const T* __restrict__ em, int nnei, int L) {
  const int ii = blockIdx.x;
  const T* ex = em_x + (size_t)ii * nnei;
  const T* e = em + (size_t)ii * nnei * ND;
  const T last = ex[nnei - 1];
  for (int k = threadIdx.x; k < L; k += blockDim.x) {
    T acc[ND];
    for (int m = 0; m < ND; ++m) acc[m] = T(0);
    for (int jj = 0; jj < nnei; ++jj) {
      const bool unloop = fold_hit<T>(ex, e, nnei, ND, jj, last);
      int idx;
      T x, ext, val, grd;
      locate<T>(ti, ex[jj], idx, x, ext);
      piece<T>(table + (size_t)idx * L * 6 + 6 * k, x, ext, val, grd);
      const T sc = unloop ? T(nnei - jj) * val : val;
      for (int m = 0; m < ND; ++m) acc[m] += sc * e[jj * ND + m];
      if (unloop) break;
    }
    for (int m = 0; m < ND; ++m) out[((size_t)ii * ND + m) * L + k] = acc[m];
  }
}

template <typename T, int ND>
__global__ void k_tab_grad(T* __restrict__ dx_out, T* __restrict__ dem_out,
                           const T* __restrict__ table, TabInfo<T> ti,
                           const T* __restrict__ em_x, const T* __restrict__ em,
                           const T* __restrict__ dy, int nnei, int L) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* dys = reinterpret_cast<T*>(smem);  // [ND][L]
  __shared__ int first;
  const int ii = blockIdx.x;
  const T* ex = em_x + (size_t)ii * nnei;
  const T* e = em + (size_t)ii * nnei * ND;
  const T last = ex[nnei - 1];
  for (int q = threadIdx.x; q < ND * L; q += blockDim.x) dys[q] = dy[(size_t)ii * ND * L + q];
  if (threadIdx.x == 0) first = nnei;
  __syncthreads();
  for (int jj = threadIdx.x; jj < nnei; jj += blockDim.x)
    if (fold_hit<T>(ex, e, nnei, ND, jj, last)) atomicMin(&first, jj);
  __syncthreads();
  const int f = first;
  for (int jj = threadIdx.x; jj < nnei; jj += blockDim.x) {
    T gx = T(0), gm[ND];
    for (int m = 0; m < ND; ++m) gm[m] = T(0);
    if (jj <= f) {
      T ll[ND];
      for (int m = 0; m < ND; ++m) ll[m] = e[jj * ND + m];
      int idx;
      T x, ext;
      locate<T>(ti, ex[jj], idx, x, ext);
      const T* row = table + (size_t)idx * L * 6;
      for (int k = 0; k < L; ++k) {
        T val, grd;
        piece<T>(row + 6 * k, x, ext, val, grd);
        T dot = T(0);
        for (int m = 0; m < ND; ++m) dot += ll[m] * dys[m * L + k];
        gx += grd * dot;
        for (int m = 0; m < ND; ++m) gm[m] += val * dys[m * L + k];
      }
      const T w = jj == f ? T(nnei - jj) : T(1);
      gx *= w;
      for (int m = 0; m < ND; ++m) gm[m] *= w;
    }
    dx_out[(size_t)ii * nnei + jj] = gx;
    for (int m = 0; m < ND; ++m) dem_out[((size_t)ii * nnei + jj) * ND + m] = gm[m];
  }
}

template <typename T, int ND>
__global__ void k_tab_gg(T* __restrict__ out, const T* __restrict__ table, TabInfo<T> ti,
                         const T* __restrict__ em_x, const T* __restrict__ em,
                         const T* __restrict__ dzx, const T* __restrict__ dzem, int nnei, int L) {
  const int ii = blockIdx.x;
  const T* ex = em_x + (size_t)ii * nnei;
  const T* e = em + (size_t)ii * nnei * ND;
  const T* hx = dzx + (size_t)ii * nnei;
  const T* hm = dzem + (size_t)ii * nnei * ND;
  const T last = ex[nnei - 1];
  for (int k = threadIdx.x; k < L; k += blockDim.x) {
    T acc[ND];
    for (int m = 0; m < ND; ++m) acc[m] = T(0);
    for (int jj = 0; jj < nnei; ++jj) {
      const bool unloop = fold_hit<T>(ex, e, nnei, ND, jj, last);
      int idx;
      T x, ext, val, grd;
      locate<T>(ti, ex[jj], idx, x, ext);
      piece<T>(table + (size_t)idx * L * 6 + 6 * k, x, ext, val, grd);
      const T sc = unloop ? T(nnei - jj) : T(1);
      const T gx = hx[jj] * grd;
      for (int m = 0; m < ND; ++m) acc[m] += sc * (val * hm[jj * ND + m] + gx * e[jj * ND + m]);
      if (unloop) break;
    }
    for (int m = 0; m < ND; ++m) out[((size_t)ii * ND + m) * L + k] = acc[m];
  }
}

__global__ void k_zero_any(unsigned char* __restrict__ p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

int zero_bytes(void* p, size_t n, hipStream_t st) {
  if (n == 0) return DPK_OK;
  hipLaunchKernelGGL(k_zero_any, dim3(cdiv((long long)n, 256)), dim3(256), 0, st,
                     static_cast<unsigned char*>(p), n);
  DPK_LAUNCHED();
  return DPK_OK;
}

constexpr int kMaxTabNets = 16;
constexpr int kMaxTabTypes = 16;

template <typename T>
struct TabSet {
  TabInfo<T> ti[kMaxTabNets];
  long long off[kMaxTabNets];  // element offset of net k's table
  int ntypes;
  int sec[kMaxTabTypes + 1];
};

// Four basis functions.  What bounds these kernels is the table: 6 L values a
// slot, which no other slot shares unless it falls into the same interval
// (2.4 KB a slot at L = 100 in FP32, 2.0 GB a call for 12,288 x 92 slots, from
// L1 and L2).  One wavefront takes one atom and puts the channels on its lanes,
// CPL adjacent ones each, so that a row is read with 16-byte loads over
// consecutive addresses, four rows in flight; a slot's interval is found once,
// by one lane, and reaches the others through v_readlane.  (One channel a
// thread, with every thread locating every slot -- or, in the backward, one
// slot a thread, each lane reading a row of its own -- was bound by its
// instructions and by the cache's address coalescing.)  The sum over the slots
// is taken in their order by one lane a channel; the backward's five sums over
// the channels are folded across the lanes for four slots together.
// Measured at 12,288 x 92 x 100, FP32: forward 207 -> 119 us (17 TB/s of
// table), backward 202 -> 151.  What bounds them now is the L2 bandwidth of the
// rows, and below some thousand atoms a wavefront's own pace: the forward gives
// channels beyond 64 CPL to other workgroups (100 x 92 slots of 256: 47 -> 28 us),
// the backward, whose slots don't meet, shares an atom (tab_split).  Spreading an
// atom's slots in the forward, whose sums then meet, gains nothing (1,001 atoms:
// 18.1 and 18.3 us).
template <typename T>
struct Tab4 {
  const T* em;        // [natoms, nnei, 4]
  const T* emx;       // [natoms, nnei], or null: em[..., 0]
  const int* atype;   // null: one table
  const int* net_of;
  const T* tables;
  const T* dy;        // backward: [natoms, 4, L]
  T* out;             // forward: [natoms, 4, L]; backward: d em [natoms, nnei, 4]
  T* dx;              // backward: d em_x [natoms, nnei], or null: added to d em[..., 0]
  T scale;
  int natoms, nnei, L;
  int lp;             // backward: log2 of the wavefronts an atom
  TabSet<T> ts;
};

__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// the 6 CPL coefficients of a lane's channels; VEC: the address is aligned to
// the widest load that 6 CPL values fill (16 bytes, 8 for one FP32 channel)
template <typename T, int CPL, bool VEC>
__device__ __forceinline__ void load_row(const T* __restrict__ p, T (&a)[6 * CPL]) {
  if constexpr (!VEC) {
#pragma unroll
    for (int i = 0; i < 6 * CPL; ++i) a[i] = p[i];
  } else {
    constexpr int W = sizeof(T) == 8 ? 2 : (CPL == 2 ? 4 : 2);
    typedef __attribute__((ext_vector_type(W))) T vec;
#pragma unroll
    for (int i = 0; i < 6 * CPL / W; ++i) {
      const vec v = reinterpret_cast<const vec*>(p)[i];
#pragma unroll
      for (int w = 0; w < W; ++w) a[W * i + w] = v[w];
    }
  }
}

// A chunk of up to 64 slots, one a lane: intervals, rows and the fold.
template <typename T>
struct Slots {
  T r[4], x, ext;
  int idx, cnt;            // slots to take (the last one with the fold's weight)
  bool stop;
  unsigned long long far;  // slots outside the table (extrapolated)
  __device__ __forceinline__ void take(const Tab4<T>& A, const TabInfo<T>& ti, const T* e,
                                       const T* ex, T last, int c0, int nb, int lane) {
    const int j = c0 + lane;
    const bool in = j < nb;
    T xx = last;
#pragma unroll
    for (int m = 0; m < 4; ++m) r[m] = in ? e[(size_t)j * 4 + m] : T(0);
    if (in) xx = ex != nullptr ? ex[j] : r[0];
    const unsigned long long hit =
        __ballot(in && xx == last && r[1] == T(0) && r[2] == T(0) && r[3] == T(0));
    stop = hit != 0;
    cnt = stop ? __ffsll(hit) : (nb - c0 < 64 ? nb - c0 : 64);
    locate<T>(ti, xx, idx, x, ext);
    far = __ballot(in && ext != T(0));
  }
};

template <typename T, int CPL, bool VEC>
__global__ void __launch_bounds__(256) k_tab4_fwd(Tab4<T> A) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int atom = blockIdx.x * 4 + wave;
  if (atom >= A.natoms) return;
  int tc = A.atype != nullptr ? A.atype[atom] : 0;
  tc = __builtin_amdgcn_readfirstlane(tc < 0 ? 0 : tc);
  const T* ea = A.em + (size_t)atom * A.nnei * 4;
  const int L = A.L;
  // (each of the grid's rows of workgroups takes a run of 64 CPL channels)
  for (int kc = blockIdx.y * 64 * CPL; kc < L; kc += gridDim.y * 64 * CPL) {
    const int k0 = kc + lane * CPL;
    const int kl = k0 < L ? k0 : 0;
    T acc[CPL][4];
#pragma unroll
    for (int q = 0; q < CPL; ++q)
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[q][m] = T(0);
    for (int t = 0; t < A.ts.ntypes; ++t) {
      const int b0 = A.ts.sec[t], nb = A.ts.sec[t + 1] - b0;
      if (nb <= 0) continue;
      const int net =
          A.net_of != nullptr ? __builtin_amdgcn_readfirstlane(A.net_of[tc * A.ts.ntypes + t]) : 0;
      const TabInfo<T>& ti = A.ts.ti[net];
      const T* tab = A.tables + A.ts.off[net];
      const T* e = ea + (size_t)b0 * 4;
      const T* ex = A.emx != nullptr ? A.emx + (size_t)atom * A.nnei + b0 : nullptr;
      const T last = ex != nullptr ? ex[nb - 1] : e[(size_t)(nb - 1) * 4];
      Slots<T> s;
      s.stop = false;
      for (int c0 = 0; c0 < nb && !s.stop; c0 += 64) {
        s.take(A, ti, e, ex, last, c0, nb, lane);
        for (int j = 0; j < s.cnt; j += 4) {
          T a[4][6 * CPL];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int l = j + u < s.cnt ? j + u : s.cnt - 1;
            load_row<T, CPL, VEC>(
                tab + (size_t)__builtin_amdgcn_readlane(s.idx, l) * L * 6 + 6 * kl, a[u]);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int l = j + u;
            if (l >= s.cnt) break;
            const T x = lane_value(s.x, l);
            const bool far = (s.far >> l) & 1;
            const T ext = far ? lane_value(s.ext, l) : T(0);
            const T w = s.stop && l == s.cnt - 1 ? T(nb - c0 - l) : T(1);
            const T e0 = lane_value(s.r[0], l), e1 = lane_value(s.r[1], l),
                    e2 = lane_value(s.r[2], l), e3 = lane_value(s.r[3], l);
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
              const T* c = a[u] + 6 * q;
              T val = c[0] + (c[1] + (c[2] + (c[3] + (c[4] + c[5] * x) * x) * x) * x) * x;
              if (far)
                val += (c[1] + (T(2) * c[2] + (T(3) * c[3] + (T(4) * c[4] + T(5) * c[5] * x) * x) *
                                                  x) * x) * ext;
              const T sc = w * val;
              acc[q][0] += sc * e0;
              acc[q][1] += sc * e1;
              acc[q][2] += sc * e2;
              acc[q][3] += sc * e3;
            }
          }
        }
      }
    }
    if (k0 < L)
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < CPL; ++q)
          A.out[((size_t)atom * 4 + m) * L + k0 + q] = acc[q][m] * A.scale;
  }
}

// Sums over the 64 lanes: two values side by side (v_permlane32_swap, then
// v_permlane16_swap of two such pairs), then the 16 lanes of a row.
__device__ __forceinline__ float half_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float quarter_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double half_sum(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                   (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                   (unsigned)__double2hiint(b), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double quarter_sum(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                   (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                   (unsigned)__double2hiint(b), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
template <int CTRL>
__device__ __forceinline__ float row_turn(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double row_turn(double v) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false),
      __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false));
}
// the four values' sums: in row 0 v0, row 1 v2, row 2 v1, row 3 v3
template <typename T>
__device__ __forceinline__ T sum4(T v0, T v1, T v2, T v3) {
  T s = quarter_sum(half_sum(v0, v1), half_sum(v2, v3));
  s += row_turn<0x128>(s);  // row_ror:8, 4, 2, 1
  s += row_turn<0x124>(s);
  s += row_turn<0x122>(s);
  s += row_turn<0x121>(s);
  return s;
}

// ONE: the channels fit the lanes, dy stays in registers.
template <typename T, int CPL, bool VEC, bool ONE>
__global__ void __launch_bounds__(256) k_tab4_bwd(Tab4<T> A) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // 1 << lp wavefronts share an atom: each takes every (1 << lp)-th four slots
  const int unit = blockIdx.x * 4 + wave, atom = unit >> A.lp, mask = (1 << A.lp) - 1,
            part = unit & mask;
  if (atom >= A.natoms) return;
  int tc = A.atype != nullptr ? A.atype[atom] : 0;
  tc = __builtin_amdgcn_readfirstlane(tc < 0 ? 0 : tc);
  const T* ea = A.em + (size_t)atom * A.nnei * 4;
  const int L = A.L, row = lane >> 4, c = lane & 15;
  int turn = 0;  // fours of the chunks before
  T dy[CPL][4];
  auto load_dy = [&](int k0) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int q = 0; q < CPL; ++q)
        dy[q][m] = k0 < L ? A.dy[((size_t)atom * 4 + m) * L + k0 + q] * A.scale : T(0);
  };
  if constexpr (ONE) load_dy(lane * CPL);
  for (int t = 0; t < A.ts.ntypes; ++t) {
    const int b0 = A.ts.sec[t], nb = A.ts.sec[t + 1] - b0;
    if (nb <= 0) continue;
    const int net =
        A.net_of != nullptr ? __builtin_amdgcn_readfirstlane(A.net_of[tc * A.ts.ntypes + t]) : 0;
    const TabInfo<T>& ti = A.ts.ti[net];
    const T* tab = A.tables + A.ts.off[net];
    const T* e = ea + (size_t)b0 * 4;
    const T* ex = A.emx != nullptr ? A.emx + (size_t)atom * A.nnei + b0 : nullptr;
    const T last = ex != nullptr ? ex[nb - 1] : e[(size_t)(nb - 1) * 4];
    T* od = A.out + ((size_t)atom * A.nnei + b0) * 4;
    T* ox = A.dx != nullptr ? A.dx + (size_t)atom * A.nnei + b0 : nullptr;
    Slots<T> s;
    s.stop = false;
    int c0 = 0;
    for (; c0 < nb && !s.stop; c0 += 64) {
      s.take(A, ti, e, ex, last, c0, nb, lane);
      const int first = (part - turn) & mask;
      turn += (s.cnt + 3) / 4;
      for (int j = 4 * first; j < s.cnt; j += 4 << A.lp) {
        T v[4][5];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int q = 0; q < 5; ++q) v[u][q] = T(0);
        for (int kc = 0; kc < (ONE ? 1 : L); kc += 64 * CPL) {
          const int k0 = kc + lane * CPL, kl = k0 < L ? k0 : 0;
          if constexpr (!ONE) load_dy(k0);
          T a[4][6 * CPL];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int l = j + u < s.cnt ? j + u : s.cnt - 1;
            load_row<T, CPL, VEC>(
                tab + (size_t)__builtin_amdgcn_readlane(s.idx, l) * L * 6 + 6 * kl, a[u]);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int l = j + u < s.cnt ? j + u : s.cnt - 1;
            const T x = lane_value(s.x, l);
            const bool far = (s.far >> l) & 1;
            const T e0 = lane_value(s.r[0], l), e1 = lane_value(s.r[1], l),
                    e2 = lane_value(s.r[2], l), e3 = lane_value(s.r[3], l);
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
              const T* k = a[u] + 6 * q;
              // (the forms of `piece`: bonded pairs share an interval and nearly an
              // x, so another rounding here would show in the virial)
              const T d = k[1] + (T(2) * k[2] +
                                  (T(3) * k[3] + (T(4) * k[4] + T(5) * k[5] * x) * x) * x) * x;
              T p = k[0] + (k[1] + (k[2] + (k[3] + (k[4] + k[5] * x) * x) * x) * x) * x;
              if (far) p += d * lane_value(s.ext, l);
              v[u][0] += d * (e0 * dy[q][0] + e1 * dy[q][1] + e2 * dy[q][2] + e3 * dy[q][3]);
#pragma unroll
              for (int m = 0; m < 4; ++m) v[u][1 + m] += p * dy[q][m];
            }
          }
        }
        T r[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) r[q] = sum4<T>(v[0][q], v[1][q], v[2][q], v[3][q]);
        const int l = j + (((row & 1) << 1) | (row >> 1));  // the slot of this row of lanes
        if (l < s.cnt && c < 5) {
          const T w = s.stop && l == s.cnt - 1 ? T(nb - c0 - l) : T(1);
          const T o = c == 0 ? r[1] : (c == 1 ? r[2] : (c == 2 ? r[3] : (c == 3 ? r[4] : r[0])));
          if (ox != nullptr) {
            if (c < 4) od[(size_t)(c0 + l) * 4 + c] = o * w;
            else ox[c0 + l] = o * w;
          } else if (c < 4) {
            od[(size_t)(c0 + l) * 4 + c] = c == 0 ? (o + r[0]) * w : o * w;
          }
        }
      }
      if (s.stop) {  // the slots that the fold stands for
        const int z = c0 + s.cnt, q0 = lane + 64 * part, step = 64 << A.lp;
        for (int q = 4 * z + q0; q < 4 * nb; q += step) od[q] = T(0);
        if (ox != nullptr)
          for (int q = z + q0; q < nb; q += step) ox[q] = T(0);
      }
    }
  }
}

// Backward of narrow nets: a slot a lane, the channels in turn, dy in LDS; one
// workgroup an atom: up to 16 channels, and 32 where the slots fill a wavefront.
// (Channels on the lanes leave half of them idle and fold every slot's sums across
// all: 12,288 x 92 slots of 8 / 16 / 32 / 48 channels in FP32 114 us each, this 27 /
// 51 / 92 / 130; 20 slots of 32 channels 31, this 41.)
constexpr int kNarrow = 32;

template <typename T>
__global__ void __launch_bounds__(128) k_tab4_bwd_narrow(Tab4<T> A) {
  __shared__ __align__(4 * sizeof(T)) T dys[kNarrow][4];
  __shared__ int first[kMaxTabTypes];
  const int atom = blockIdx.x, L = A.L;
  int tc = A.atype != nullptr ? A.atype[atom] : 0;
  tc = tc < 0 ? 0 : tc;
  const T* ea = A.em + (size_t)atom * A.nnei * 4;
  const T* xa = A.emx != nullptr ? A.emx + (size_t)atom * A.nnei : nullptr;
  for (int q = threadIdx.x; q < 4 * L; q += blockDim.x)
    dys[q % L][q / L] = A.dy[(size_t)atom * 4 * L + q] * A.scale;
  if (threadIdx.x < (unsigned)A.ts.ntypes) first[threadIdx.x] = A.nnei;
  __syncthreads();
  for (int t = 0; t < A.ts.ntypes; ++t) {  // the blocks' folds
    const int b0 = A.ts.sec[t], b1 = A.ts.sec[t + 1];
    if (b1 <= b0) continue;
    const T last = xa != nullptr ? xa[b1 - 1] : ea[(size_t)(b1 - 1) * 4];
    for (int j = b0 + threadIdx.x; j < b1; j += blockDim.x) {
      const T* r = ea + (size_t)j * 4;
      if ((xa != nullptr ? xa[j] : r[0]) == last && r[1] == T(0) && r[2] == T(0) && r[3] == T(0))
        atomicMin(&first[t], j);
    }
  }
  __syncthreads();
  for (int t = 0; t < A.ts.ntypes; ++t) {
    const int b0 = A.ts.sec[t], b1 = A.ts.sec[t + 1];
    if (b1 <= b0) continue;
    const int net = A.net_of != nullptr ? A.net_of[tc * A.ts.ntypes + t] : 0;
    const TabInfo<T>& ti = A.ts.ti[net];
    const T* tab = A.tables + A.ts.off[net];
    for (int j = b0 + threadIdx.x; j < b1; j += blockDim.x) {
      const T* r = ea + (size_t)j * 4;
      T gx = T(0), gm[4] = {T(0), T(0), T(0), T(0)};
      if (j <= first[t]) {
        int idx;
        T x, ext;
        locate<T>(ti, xa != nullptr ? xa[j] : r[0], idx, x, ext);
        const T* row = tab + (size_t)idx * L * 6;
        const T r0 = r[0], r1 = r[1], r2 = r[2], r3 = r[3];
#pragma clang loop unroll_count(sizeof(T) == 4 ? 2 : 1)
        for (int k = 0; k < L; ++k) {
          T val, grd;
          piece<T>(row + 6 * k, x, ext, val, grd);
          const T d0 = dys[k][0], d1 = dys[k][1], d2 = dys[k][2], d3 = dys[k][3];
          gx += grd * (r0 * d0 + r1 * d1 + r2 * d2 + r3 * d3);
          gm[0] += val * d0;
          gm[1] += val * d1;
          gm[2] += val * d2;
          gm[3] += val * d3;
        }
        const T w = j == first[t] ? T(b1 - j) : T(1);
        gx *= w;
        for (int m = 0; m < 4; ++m) gm[m] *= w;
      }
      const size_t s = (size_t)atom * A.nnei + j;
      if (A.dx != nullptr) A.dx[s] = gx;
      else gm[0] += gx;
      for (int m = 0; m < 4; ++m) A.out[s * 4 + m] = gm[m];
    }
  }
}

// Wavefronts an atom of the backward (log2): several, of eight slots and more
// each, while they fit the chip together (16 a CU).  FP32, 100 channels, with 1 / 2
// / 4 / 8 us: 100 atoms of 200 slots 59 / 35 / 23 / 16, 1,001 of 92 33 / 25 / 22 /
// 24, of 200 61 / 44 / 40 / 42, 12,288 of 92 151 / 153 / 164 / 207.
inline int tab_split(int natoms, int nnei, int ncu) {
  int lp = 0;
  while (lp < 3 && (2l << lp) * natoms <= 16l * ncu && (16 << lp) <= nnei) ++lp;
  return lp;
}

// Channels a lane: two for wide nets (16-byte loads, lanes filled), one where
// 64 lanes hold all of them, or where L is odd (the rows are then aligned to
// one channel only).  Tables that are not aligned are read value by value.
template <typename T>
int launch_tab4(bool fwd, Tab4<T>& A, hipStream_t st) {
  if (A.natoms == 0) return DPK_OK;
  const dim3 b(256);
  const size_t at = reinterpret_cast<size_t>(A.tables);
  if (!fwd && (A.L <= 16 || (A.L <= kNarrow && A.nnei >= 64))) {
    hipLaunchKernelGGL((k_tab4_bwd_narrow<T>), dim3(A.natoms), dim3(A.nnei >= 128 ? 128 : 64), 0,
                       st, A);
    DPK_LAUNCHED();
    return DPK_OK;
  }
  A.lp = 0;
  if (!fwd) {
    int dev = 0, ncu = 0;
    const int rc = device_cus(&dev, &ncu);
    if (rc != DPK_OK) return rc;
    A.lp = tab_split(A.natoms, A.nnei, ncu);
  }
  const dim3 g(cdiv((long long)A.natoms << A.lp, 4));
#define DPK_TAB4(CPL, VEC)                                                                 \
  do {                                                                                     \
    if (fwd)                                                                               \
      hipLaunchKernelGGL((k_tab4_fwd<T, CPL, VEC>), dim3(g.x, cdiv(A.L, 64 * CPL)), b, 0, st, A); \
    else if (A.L <= 64 * CPL)                                                              \
      hipLaunchKernelGGL((k_tab4_bwd<T, CPL, VEC, true>), g, b, 0, st, A);                   \
    else hipLaunchKernelGGL((k_tab4_bwd<T, CPL, VEC, false>), g, b, 0, st, A);               \
  } while (0)
  if (at % 16 != 0 && (sizeof(T) == 8 || at % 8 != 0)) DPK_TAB4(1, false);
  else if (A.L > 64 && A.L % 2 == 0 && at % 16 == 0) DPK_TAB4(2, true);
  else DPK_TAB4(1, true);
#undef DPK_TAB4
  DPK_LAUNCHED();
  return DPK_OK;
}

// the operator's arguments: one table, every slot in one block
template <typename T>
Tab4<T> op_args(const T* table, const TabInfo<T>& ti, const T* em_x, const T* em, int nloc,
                int nnei, int L) {
  Tab4<T> A{};
  A.em = em;
  A.emx = em_x;
  A.tables = table;
  A.scale = T(1);
  A.natoms = nloc;
  A.nnei = nnei;
  A.L = L;
  A.ts.ti[0] = ti;
  A.ts.ntypes = 1;
  A.ts.sec[1] = nnei;
  return A;
}

int block_for(int L) { return L >= 256 ? 256 : (L > 128 ? 256 : (L > 64 ? 128 : 64)); }

template <typename T>
int check(const T* info, int nloc, int nnei, int L, int nd, int nspline) {
  DPK_REQUIRE(nspline > 0, DPK_ERR_ARG, "tabulate: empty table");
  DPK_REQUIRE(info != nullptr, DPK_ERR_ARG, "tabulate: table_info must be a host array");
  DPK_REQUIRE(nloc >= 0 && nnei >= 0 && L > 0, DPK_ERR_ARG, "tabulate: bad sizes");
  DPK_REQUIRE(nd == 4 || nd == 9 || nd == 16 || nd == 25, DPK_ERR_ARG,
              "The environment basis dimension must be 4, 9, 16, or 25, got %d", nd);
  DPK_REQUIRE(info[3] > T(0) && info[4] > T(0), DPK_ERR_ARG, "tabulate: strides must be > 0");
  return DPK_OK;
}

template <typename T>
int tab_fwd(T* out, const T* table, int nspline, const T* info, const T* em_x, const T* em, int nloc,
            int nnei, int L, int nd, dpk_stream_t stream) {
  clear_error();
  int rc = check<T>(info, nloc, nnei, L, nd, nspline);
  if (rc) return rc;
  hipStream_t st = as_stream(stream);
  if (nloc == 0) return DPK_OK;
  if (nnei == 0) return zero_bytes(out, sizeof(T) * (size_t)nloc * nd * L, st);
  TabInfo<T> ti = make_info<T>(info, nspline);
  if (nd == 4) {
    Tab4<T> A = op_args<T>(table, ti, em_x, em, nloc, nnei, L);
    A.out = out;
    return launch_tab4<T>(true, A, st);
  }
  dim3 g(nloc), b(block_for(L));
  switch (nd) {
    case 9: hipLaunchKernelGGL((k_tab_fwd<T, 9>), g, b, 0, st, out, table, ti, em_x, em, nnei, L); break;
    case 16: hipLaunchKernelGGL((k_tab_fwd<T, 16>), g, b, 0, st, out, table, ti, em_x, em, nnei, L); break;
    default: hipLaunchKernelGGL((k_tab_fwd<T, 25>), g, b, 0, st, out, table, ti, em_x, em, nnei, L); break;
  }
  DPK_LAUNCHED();
  return DPK_OK;
}

template <typename T>
int tab_grad(T* dx, T* dem, const T* table, int nspline, const T* info, const T* em_x, const T* em,
             const T* dy, int nloc, int nnei, int L, int nd, dpk_stream_t stream) {
  clear_error();
  int rc = check<T>(info, nloc, nnei, L, nd, nspline);
  if (rc) return rc;
  if (nloc == 0 || nnei == 0) return DPK_OK;
  hipStream_t st = as_stream(stream);
  TabInfo<T> ti = make_info<T>(info, nspline);
  size_t lds = sizeof(T) * (size_t)nd * L;
  DPK_REQUIRE(lds <= 60 * 1024, DPK_ERR_UNSUPPORTED, "tabulate grad: nd*L too large for LDS");
  if (nd == 4) {
    Tab4<T> A = op_args<T>(table, ti, em_x, em, nloc, nnei, L);
    A.dy = dy;
    A.out = dem;
    A.dx = dx;
    return launch_tab4<T>(false, A, st);
  }
  dim3 g(nloc), b(nnei >= 128 ? 128 : 64);
  switch (nd) {
    case 9: hipLaunchKernelGGL((k_tab_grad<T, 9>), g, b, lds, st, dx, dem, table, ti, em_x, em, dy, nnei, L); break;
    case 16: hipLaunchKernelGGL((k_tab_grad<T, 16>), g, b, lds, st, dx, dem, table, ti, em_x, em, dy, nnei, L); break;
    default: hipLaunchKernelGGL((k_tab_grad<T, 25>), g, b, lds, st, dx, dem, table, ti, em_x, em, dy, nnei, L); break;
  }
  DPK_LAUNCHED();
  return DPK_OK;
}

template <typename T>
int tab_gg(T* out, const T* table, int nspline, const T* info, const T* em_x, const T* em, const T* dzx,
           const T* dzem, int nloc, int nnei, int L, int nd, dpk_stream_t stream) {
  clear_error();
  int rc = check<T>(info, nloc, nnei, L, nd, nspline);
  if (rc) return rc;
  hipStream_t st = as_stream(stream);
  if (nloc == 0) return DPK_OK;
  if (nnei == 0) return zero_bytes(out, sizeof(T) * (size_t)nloc * nd * L, st);
  TabInfo<T> ti = make_info<T>(info, nspline);
  dim3 g(nloc), b(block_for(L));
  switch (nd) {
    case 4: hipLaunchKernelGGL((k_tab_gg<T, 4>), g, b, 0, st, out, table, ti, em_x, em, dzx, dzem, nnei, L); break;
    case 9: hipLaunchKernelGGL((k_tab_gg<T, 9>), g, b, 0, st, out, table, ti, em_x, em, dzx, dzem, nnei, L); break;
    case 16: hipLaunchKernelGGL((k_tab_gg<T, 16>), g, b, 0, st, out, table, ti, em_x, em, dzx, dzem, nnei, L); break;
    default: hipLaunchKernelGGL((k_tab_gg<T, 25>), g, b, 0, st, out, table, ti, em_x, em, dzx, dzem, nnei, L); break;
  }
  DPK_LAUNCHED();
  return DPK_OK;
}

// ---------------------------------------------------------------------------
// Compressed embedding inside the fused model: the per-type-block loop of
// deepmd/pt/model/descriptor/se_a.py:795-843 (one tabulate_fusion_se_a call
// per (centre type, neighbour type) table, summed, divided by nnei) over the
// env matrix em [natoms, nnei, 4] in place: em_x of a slot is em[slot][0] and
// the padding fold applies per type block (the block's last slot).  Tables of
// all nets are concatenated; their infos travel by value (Tab4).
template <typename T>
int tabemb(bool fwd, void* out, const void* em, const void* gxyz, const int* atype,
           const void* tables, const long long* off, const int* nspline, const double* info,
           const int* net_of, int ntypes, int nnets, const int* sec_host, int L, int natoms,
           int nnei, hipStream_t st) {
  DPK_REQUIRE(ntypes > 0 && ntypes <= kMaxTabTypes && nnets > 0 && nnets <= kMaxTabNets,
              DPK_ERR_UNSUPPORTED, "tab_embed: ntypes=%d nnets=%d (<= %d tables)", ntypes, nnets,
              kMaxTabNets);
  DPK_REQUIRE(L > 0 && nnei > 0 && natoms >= 0, DPK_ERR_ARG, "tab_embed: bad sizes");
  Tab4<T> A{};
  TabSet<T>& ts = A.ts;
  ts.ntypes = ntypes;
  for (int t = 0; t <= ntypes; ++t) ts.sec[t] = sec_host[t];
  DPK_REQUIRE(ts.sec[ntypes] == nnei, DPK_ERR_ARG, "tab_embed: sum(sel)=%d != nnei=%d",
              ts.sec[ntypes], nnei);
  for (int k = 0; k < nnets; ++k) {
    T h[6];
    for (int q = 0; q < 6; ++q) h[q] = (T)info[6 * k + q];
    DPK_REQUIRE(nspline[k] > 0 && h[3] > T(0) && h[4] > T(0), DPK_ERR_ARG,
                "tab_embed: table %d is empty or has a non-positive stride", k);
    ts.ti[k] = make_info<T>(h, nspline[k]);
    ts.off[k] = off[k];
  }
  if (!fwd)
    DPK_REQUIRE(sizeof(T) * 4 * (size_t)L <= 32 * 1024, DPK_ERR_UNSUPPORTED,
                "tab_embed: L=%d too large", L);
  A.em = static_cast<const T*>(em);
  A.atype = atype;
  A.net_of = net_of;
  A.tables = static_cast<const T*>(tables);
  A.dy = static_cast<const T*>(gxyz);
  A.out = static_cast<T*>(out);
  A.scale = T(1) / T(nnei);
  A.natoms = natoms;
  A.nnei = nnei;
  A.L = L;
  return launch_tab4<T>(fwd, A, st);
}

int tabemb_common(bool fwd, void* out, int prec, const void* em, const void* gxyz,
                  const int* atype, const void* tables, const long long* off, const int* nspline,
                  const double* info, const int* net_of, int ntypes, int nnets,
                  const int* sec_host, int L, int natoms, int nnei, dpk_stream_t stream) {
  clear_error();
  DPK_REQUIRE(off && nspline && info && sec_host, DPK_ERR_ARG,
              "tab_embed: table offsets, sizes, infos and sections are host arrays");
  hipStream_t st = as_stream(stream);
  if (prec == DPK_PREC_F64)
    return tabemb<double>(fwd, out, em, gxyz, atype, tables, off, nspline, info, net_of, ntypes,
                          nnets, sec_host, L, natoms, nnei, st);
  if (prec == DPK_PREC_F32)
    return tabemb<float>(fwd, out, em, gxyz, atype, tables, off, nspline, info, net_of, ntypes,
                         nnets, sec_host, L, natoms, nnei, st);
  set_error("tab_embed: precision %d unsupported (FP64 or FP32 tables)", prec);
  return DPK_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace dpk

using namespace dpk;

extern "C" int dpk_tab_embed_fwd(void* xyz, int prec, const void* em, const int* atype,
                                 const void* tables, const long long* table_off,
                                 const int* nspline, const double* info, const int* net_of,
                                 int ntypes, int nnets, const int* sec_host, int L, int natoms,
                                 int nnei, dpk_stream_t stream) {
  return tabemb_common(true, xyz, prec, em, nullptr, atype, tables, table_off, nspline, info,
                       net_of, ntypes, nnets, sec_host, L, natoms, nnei, stream);
}

extern "C" int dpk_tab_embed_bwd(void* net_deriv, int prec, const void* em, const void* gxyz,
                                 const int* atype, const void* tables, const long long* table_off,
                                 const int* nspline, const double* info, const int* net_of,
                                 int ntypes, int nnets, const int* sec_host, int L, int natoms,
                                 int nnei, dpk_stream_t stream) {
  return tabemb_common(false, net_deriv, prec, em, gxyz, atype, tables, table_off, nspline, info,
                       net_of, ntypes, nnets, sec_host, L, natoms, nnei, stream);
}

extern "C" int dpk_tabulate_fusion_se_a_f64(double* out, const double* table, int nspline,
                                            const double* info, const double* em_x,
                                            const double* em, int nloc, int nnei, int L, int nd,
                                            dpk_stream_t s) {
  return tab_fwd<double>(out, table, nspline, info, em_x, em, nloc, nnei, L, nd, s);
}
extern "C" int dpk_tabulate_fusion_se_a_f32(float* out, const float* table, int nspline,
                                            const float* info,
                                            const float* em_x, const float* em, int nloc,
                                            int nnei, int L, int nd, dpk_stream_t s) {
  return tab_fwd<float>(out, table, nspline, info, em_x, em, nloc, nnei, L, nd, s);
}
extern "C" int dpk_tabulate_fusion_se_a_grad_f64(double* dx, double* dem, const double* table,
                                                 int nspline, const double* info, const double* em_x,
                                                 const double* em, const double* dy, int nloc,
                                                 int nnei, int L, int nd, dpk_stream_t s) {
  return tab_grad<double>(dx, dem, table, nspline, info, em_x, em, dy, nloc, nnei, L, nd, s);
}
extern "C" int dpk_tabulate_fusion_se_a_grad_f32(float* dx, float* dem, const float* table,
                                                 int nspline, const float* info, const float* em_x,
                                                 const float* em, const float* dy, int nloc,
                                                 int nnei, int L, int nd, dpk_stream_t s) {
  return tab_grad<float>(dx, dem, table, nspline, info, em_x, em, dy, nloc, nnei, L, nd, s);
}
extern "C" int dpk_tabulate_fusion_se_a_grad_grad_f64(double* out, const double* table,
                                                      int nspline, const double* info, const double* em_x,
                                                      const double* em, const double* dzx,
                                                      const double* dzem, int nloc, int nnei,
                                                      int L, int nd, dpk_stream_t s) {
  return tab_gg<double>(out, table, nspline, info, em_x, em, dzx, dzem, nloc, nnei, L, nd, s);
}
extern "C" int dpk_tabulate_fusion_se_a_grad_grad_f32(float* out, const float* table,
                                                      int nspline, const float* info, const float* em_x,
                                                      const float* em, const float* dzx,
                                                      const float* dzem, int nloc, int nnei,
                                                      int L, int nd, dpk_stream_t s) {
  return tab_gg<float>(out, table, nspline, info, em_x, em, dzx, dzem, nloc, nnei, L, nd, s);
}
