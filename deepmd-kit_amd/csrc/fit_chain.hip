// The FP64 energy fitting in one call: descriptor, tanh layers, energy
// and the backward down to dE/dxyz, all atom types in every launch.
//
// The math is that of fitting.hip (se_a.py:844-850, fitting.py:734-899); a
// layer is one kernel, a matrix product with its epilogue:
//   forward   z = y_{l-1} W_l;  y_l = tanh(z + b) idt + res(y_{l-1}),
//             sd_l = idt (1 - tanh^2)      (last layer: g_z = w_out sd instead)
//   backward  m = g_z_l W_l^T;  g_y_{l-1} = m + res^T(g_y_l),
//             g_z_{l-1} = g_y_{l-1} sd_{l-1}
//   dE/dD = g_z_1 W_1^T
// Rows are slots (atoms grouped by type); a tile belongs to one type and takes
// that type's weights, so a step of three layers is 9 launches whatever the
// number of types (three products forward, the energy, three back, and the
// descriptor's two) instead of 31 with two.
//
// What bounds it: with few atoms the launches and the length of the sum over
// K, else the FP64 pipe (64 cycles a v_mfma_f64_16x16x4).  Both operands come
// straight from memory into registers, four steps of eight K values ahead: W is
// laid out once in the order the lanes read it (dpk.h), and a lane's two K values
// of A are adjacent.
// Measured, fitting kernels of a step (descriptor apart), against hipBLASLt
// products and elementwise kernels a type: water of 81 atoms 266 -> 43 us, of
// 1,536 atoms 255 -> 127; Cu of 5,324 atoms 380 -> 372 (one type: 12 launches
// -> 7).  With many rows of wide layers the library's products are faster (Cu of
// 13,500 atoms 1,081 against 986, 131,072 9,509 against 8,391): the model calls
// this up to the rows of Fitting.chain_rows.  FP32 stays with the library: there this kernel took 559 us against
// 591 at 12,288 atoms and 1972 against 1290 at 37,700.
#include "dpk_common.h"
#include "tanh64.h"

namespace dpk {
namespace {
namespace chain {

typedef __attribute__((ext_vector_type(4))) double v4d;
typedef __attribute__((ext_vector_type(2))) double v2d;

constexpr int kMaxSeg = 16, kMaxLayers = 8;
enum { EPI_STORE = 0, EPI_FWD = 1, EPI_BWD = 2 };

struct Seg {
  const double *w, *b, *idt, *wout;
  int row0, rows, tile0, res;
};

struct Args {
  const double* A;         // [n, K]
  int K, N, nseg, ntiles, cols;
  const double* prev;      // forward: y_{l-1}; backward: g_y_l (null: w_out)
  int ldprev;
  const double* sd_in;     // backward: sd_{l-1}
  double *y, *sd, *gz;     // forward: y, sd (or, last layer, gz); backward: y = g_y (may be null), gz
  Seg seg[kMaxSeg];
};

// One value of the product through the epilogue.
template <int EPI>
__device__ __forceinline__ void finish(const Args& G, const Seg& s, int row, int col, double v,
                                       const double* tab) {
  const size_t o = (size_t)row * G.N + col;
  if constexpr (EPI == EPI_STORE) {
    G.y[o] = v;
  } else if constexpr (EPI == EPI_FWD) {
    const double t = tanh64(v + s.b[col], tab);
    const double k = s.idt != nullptr ? s.idt[col] : 1.0;
    double yv = t * k;
    if (s.res != 0)
      yv += G.prev[(size_t)row * G.ldprev + (s.res == 2 && col >= G.ldprev ? col - G.ldprev : col)];
    const double d = k * (1.0 - t * t);
    G.y[o] = yv;
    if (G.gz != nullptr) G.gz[o] = s.wout[col] * d;
    else G.sd[o] = d;
  } else {
    if (s.res != 0) {
      const double* gn = G.prev != nullptr ? G.prev + (size_t)row * G.ldprev : s.wout;
      v += gn[col];
      if (s.res == 2) v += gn[col + G.N];
    }
    if (G.y != nullptr) G.y[o] = v;
    G.gz[o] = v * G.sd_in[o];
  }
}

// A wavefront's tile is 16 MT x 16 NT.  KS = 1: the workgroup's four take a
// 2 x 2 of them; KS = 4: they share one tile, a quarter of K each, and add
// their parts in LDS in a fixed order.
template <int MT, int NT, int KS, int EPI>
__global__ void __launch_bounds__(256) k_gemm(Args G) {
  constexpr int W2 = KS == 1 ? 2 : 1, TM = 16 * MT * W2, P = 4;
  __shared__ double tab[32];
  __shared__ double part[KS == 1 ? 1 : KS][KS == 1 ? 1 : MT * NT * 4][64];
  if constexpr (EPI == EPI_FWD) {
    if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
    if (KS == 1) __syncthreads();
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  // consecutive workgroups go to the eight XCDs in turn: each XCD takes a
  // contiguous run of tiles, whose rows of A stay in its L2
  const int per = (G.ntiles + 7) / 8;
  const int tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per || tile >= G.ntiles) return;
  const int rt = tile / G.cols, ct = tile % G.cols;
  int k = 0;
  while (k + 1 < G.nseg && rt >= G.seg[k + 1].tile0) ++k;
  const Seg& s = G.seg[k];
  const int wm = KS == 1 ? wave >> 1 : 0, wn = KS == 1 ? wave & 1 : 0;
  const int rbase = (rt - s.tile0) * TM + wm * 16 * MT;
  const int col0 = (ct * W2 + wn) * 16 * NT;
  const int groups = G.K / 8;
  const int s0 = KS == 1 ? 0 : groups * wave / KS, s1 = KS == 1 ? groups : groups * (wave + 1) / KS;
  const double* ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r = rbase + 16 * i + c;
    ap[i] = G.A + (size_t)(s.row0 + (r < s.rows ? r : s.rows - 1)) * G.K + 2 * g;
  }
  const double* bp = s.w + (size_t)(col0 / 16) * groups * 128 + 2 * lane;
  v4d acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  v2d a[P][MT], b[P][NT];
  auto load = [&](int p, int q) {
    q = q < s1 ? q : (s1 > 0 ? s1 - 1 : 0);
#pragma unroll
    for (int i = 0; i < MT; ++i) a[p][i] = *reinterpret_cast<const v2d*>(ap[i] + 8 * q);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      b[p][j] = *reinterpret_cast<const v2d*>(bp + ((size_t)j * groups + q) * 128);
  };
#pragma unroll
  for (int p = 0; p < P; ++p) load(p, s0 + p);
  for (int q = s0; q < s1; q += P) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      if (q + p < s1) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[p][i][u], b[p][j][u],
                                                             acc[i][j], 0, 0, 0);
      }
      load(p, q + p + P);
    }
  }
  if constexpr (KS == 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = rbase + 16 * i + g + 4 * r;
          if (row < s.rows)
            finish<EPI>(G, s, s.row0 + row, col0 + 16 * j + c, acc[i][j][r], tab);
        }
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][(i * NT + j) * 4 + r][lane] = acc[i][j][r];
    __syncthreads();
    for (int q = wave; q < MT * NT * 4; q += 4) {
      double v = part[0][q][lane];
#pragma unroll
      for (int w = 1; w < KS; ++w) v += part[w][q][lane];
      const int ij = q >> 2, row = rbase + 16 * (ij / NT) + g + 4 * (q & 3);
      if (row < s.rows)
        finish<EPI>(G, s, s.row0 + row, col0 + 16 * (ij % NT) + c, v, tab);
    }
  }
}

// atom_e[order[i]] = y_i . w_out + ebias of the slot's type; a wavefront a row
struct EnergyArgs {
  double* atom_e;
  const double* y;
  const int* order;
  int n, h, nseg;
  const double* wout[kMaxSeg];
  double ebias[kMaxSeg];
  int row0[kMaxSeg + 1];
};
__global__ void __launch_bounds__(256) k_energy(EnergyArgs E) {
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= E.n) return;
  int k = 0;
  while (k + 1 < E.nseg && row >= E.row0[k + 1]) ++k;
  const double* y = E.y + (size_t)row * E.h;
  double acc = 0.0;
  for (int ch = 4 * lane; ch < E.h; ch += 256)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc += y[ch + q] * E.wout[k][ch + q];
  acc = wave_sum(acc);
  if (lane == 0) E.atom_e[E.order[row]] = acc + E.ebias[k];
}

// Tile of a product of `rows` by N: 64 x 64 by the workgroup where that still
// gives every CU two of them, else 32 x 32 and at last 16 x 16 with K split
// over the wavefronts -- larger tiles read less, smaller ones fill the chip.
// (64 x 64 from one a CU: Cu of 5,324 atoms 75 us slower; never: 28 slower;
// 32 x 32 only from four a CU: water of 1,536 atoms 18 slower.)
int tile_of(const int* rows, int nseg, int N, int ncu) {
  for (int t : {64, 32}) {
    if (N % t != 0) continue;
    long tiles = 0;
    for (int k = 0; k < nseg; ++k) tiles += (rows[k] + t - 1) / t;
    if (tiles * (N / t) >= (t == 64 ? 2 : 1) * (long)ncu) return t;
  }
  return 16;
}

template <int EPI>
int product(Args& G, int ncu, hipStream_t st) {
  int rows[kMaxSeg];
  for (int k = 0; k < G.nseg; ++k) rows[k] = G.seg[k].rows;
  const int t = tile_of(rows, G.nseg, G.N, ncu);
  int tiles = 0;
  for (int k = 0; k < G.nseg; ++k) {
    G.seg[k].tile0 = tiles;
    tiles += (rows[k] + t - 1) / t;
  }
  G.cols = G.N / t;
  const long all = (long)tiles * G.cols;
  DPK_REQUIRE(all < (1L << 30), DPK_ERR_UNSUPPORTED, "fit_chain: too many rows");
  G.ntiles = (int)all;
  const dim3 grid((unsigned)(8 * ((all + 7) / 8))), b(256);
  if (t == 64) hipLaunchKernelGGL((k_gemm<2, 2, 1, EPI>), grid, b, 0, st, G);
  else if (t == 32) hipLaunchKernelGGL((k_gemm<2, 2, 4, EPI>), grid, b, 0, st, G);
  else hipLaunchKernelGGL((k_gemm<1, 1, 4, EPI>), grid, b, 0, st, G);
  DPK_LAUNCHED();
  return DPK_OK;
}

// doubles of the workspace: dE/dD, y (two), sd of the layers but the last,
// g_y (two), g_z (two)
size_t ws_values(int n, int L, const int* w) {
  int h = 0;
  for (int l = 1; l <= L; ++l) h = w[l] > h ? w[l] : h;
  return (size_t)n * (w[0] + (size_t)(L + 5) * h);
}

int run(int L, const int* w, const int* res, const void* const* params,
        const double* ebias, int nseg, const int* segs, double* atom_e, void* gxyz,
        const void* xyz, const int* order, int n, int d3, int m2, void* desc, void* ws,
        hipStream_t st) {
  int dev = 0, ncu = 0, rc = device_cus(&dev, &ncu);
  if (rc != DPK_OK) return rc;
  int hmax = 0;
  for (int l = 1; l <= L; ++l) hmax = w[l] > hmax ? w[l] : hmax;
  const size_t blk = (size_t)n * hmax;
  double* gd = static_cast<double*>(ws);
  double* at = gd + (size_t)n * w[0];
  double *y[2] = {at, at + blk}, *gy[2] = {at + 2 * blk, at + 3 * blk},
    *gz[2] = {at + 4 * blk, at + 5 * blk}, *sd = at + 6 * blk;
  rc = dpk_fit_descriptor_fwd(desc, DPK_PREC_F64, xyz, order, n, d3, m2, st);
  if (rc != DPK_OK) return rc;
  // params of type t: four pointers a layer (W, W^T, b, idt), then w_out
  auto par = [&](int t, int l, int q) {
    return static_cast<const double*>(params[(size_t)t * (4 * L + 1) + 4 * l + q]);
  };
  auto fill = [&](Args& G, int l, int q) {
    G.nseg = 0;
    for (int k = 0; k < nseg; ++k) {
      const int t = segs[3 * k], a = segs[3 * k + 1], b = segs[3 * k + 2];
      if (b <= a) continue;
      Seg& s = G.seg[G.nseg++];
      s.w = par(t, l, q);
      s.b = par(t, l, 2);
      s.idt = par(t, l, 3);
      s.wout = par(t, L, 0);
      s.row0 = a;
      s.rows = b - a;
      s.res = res[t * L + l];
    }
  };
  int cur = 0;
  for (int l = 0; l < L; ++l) {
    Args G{};
    fill(G, l, 0);
    G.A = l == 0 ? static_cast<const double*>(desc) : y[1 - cur];
    G.K = w[l];
    G.N = w[l + 1];
    G.prev = l == 0 ? nullptr : y[1 - cur];
    G.ldprev = w[l];
    G.y = y[cur];
    if (l == L - 1) G.gz = gz[0];
    else G.sd = sd + (size_t)l * blk;
    if ((rc = product<EPI_FWD>(G, ncu, st)) != DPK_OK) return rc;
    cur = 1 - cur;
  }
  EnergyArgs E{};
  E.atom_e = atom_e;
  E.y = y[1 - cur];
  E.order = order;
  E.n = n;
  E.h = w[L];
  for (int k = 0; k < nseg; ++k) {
    if (segs[3 * k + 2] <= segs[3 * k + 1]) continue;
    E.wout[E.nseg] = par(segs[3 * k], L, 0);
    E.ebias[E.nseg] = ebias[segs[3 * k]];
    E.row0[E.nseg++] = segs[3 * k + 1];
  }
  hipLaunchKernelGGL(k_energy, dim3(cdiv(n, 4)), dim3(256), 0, st, E);
  DPK_LAUNCHED();
  int gi = 0, zi = 0;
  for (int l = L - 1; l > 0; --l) {
    Args G{};
    fill(G, l, 1);
    G.A = gz[zi];
    G.K = w[l + 1];
    G.N = w[l];
    G.prev = l == L - 1 ? nullptr : gy[1 - gi];
    G.ldprev = w[l + 1];
    G.y = l > 1 ? gy[gi] : nullptr;
    G.sd_in = sd + (size_t)(l - 1) * blk;
    G.gz = gz[1 - zi];
    if ((rc = product<EPI_BWD>(G, ncu, st)) != DPK_OK) return rc;
    gi = 1 - gi;
    zi = 1 - zi;
  }
  Args G{};
  fill(G, 0, 1);
  G.A = gz[zi];
  G.K = w[1];
  G.N = w[0];
  G.y = gd;
  if ((rc = product<EPI_STORE>(G, ncu, st)) != DPK_OK) return rc;
  return dpk_fit_descriptor_bwd(gxyz, DPK_PREC_F64, gd, xyz, order, n, d3, m2, st);
}

}  // namespace chain
}  // namespace
}  // namespace dpk

using namespace dpk;

extern "C" size_t dpk_fit_chain_f64_workspace_bytes(int n, int nlayers, const int* widths) {
  if (n <= 0 || nlayers < 1 || nlayers > chain::kMaxLayers || widths == nullptr) return 0;
  return chain::ws_values(n, nlayers, widths) * sizeof(double);
}

extern "C" int dpk_fit_chain_f64(int nlayers, const int* widths, const int* res,
                                 const void* const* params, const double* ebias, int nseg,
                                 const int* segs, double* atom_energy, double* gxyz,
                                 const double* xyz, const int* order, int n, int d3, int m2,
                                 double* desc, void* ws, size_t ws_bytes, dpk_stream_t stream) {
  clear_error();
  DPK_REQUIRE(nlayers >= 1 && nlayers <= chain::kMaxLayers && nseg >= 1 && nseg <= chain::kMaxSeg,
              DPK_ERR_UNSUPPORTED, "fit_chain: %d layers, %d segments (at most %d, %d)", nlayers,
              nseg, chain::kMaxLayers, chain::kMaxSeg);
  DPK_REQUIRE(widths && res && params && ebias && segs, DPK_ERR_ARG, "fit_chain: null tables");
  DPK_REQUIRE(widths[0] == d3 * m2, DPK_ERR_ARG, "fit_chain: %d inputs for a descriptor of %d x %d",
              widths[0], d3, m2);
  for (int l = 0; l <= nlayers; ++l)
    DPK_REQUIRE(widths[l] > 0 && widths[l] % 16 == 0, DPK_ERR_UNSUPPORTED,
                "fit_chain: width %d is not a multiple of 16", widths[l]);
  int at = 0;
  for (int k = 0; k < nseg; ++k) {
    DPK_REQUIRE(segs[3 * k] >= 0 && segs[3 * k + 1] == at && segs[3 * k + 2] >= at, DPK_ERR_ARG,
                "fit_chain: segment %d [%d, %d) does not follow row %d", k, segs[3 * k + 1],
                segs[3 * k + 2], at);
    at = segs[3 * k + 2];
    if (segs[3 * k + 2] == segs[3 * k + 1]) continue;
    for (int l = 0; l < nlayers; ++l) {
      const int r = res[segs[3 * k] * nlayers + l];
      DPK_REQUIRE(r == 0 || (l > 0 && (r == 1 ? widths[l] == widths[l + 1]
                                              : r == 2 && 2 * widths[l] == widths[l + 1])),
                  DPK_ERR_ARG, "fit_chain: resnet %d from width %d to %d", r, widths[l],
                  widths[l + 1]);
    }
  }
  DPK_REQUIRE(at == n && n >= 0, DPK_ERR_ARG, "fit_chain: segments of %d rows for n = %d", at, n);
  if (n == 0) return DPK_OK;
  DPK_REQUIRE(atom_energy && gxyz && xyz && order && desc && ws, DPK_ERR_ARG,
              "fit_chain: null buffer");
  DPK_REQUIRE(ws_bytes >= dpk_fit_chain_f64_workspace_bytes(n, nlayers, widths), DPK_ERR_ARG,
              "fit_chain: workspace of %zu bytes is too small", ws_bytes);
  return chain::run(nlayers, widths, res, params, ebias, nseg, segs, atom_energy, gxyz, xyz, order,
                    n, d3, m2, desc, ws, as_stream(stream));
}
