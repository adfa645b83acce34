// FP64 se_e2_a embedding net + R^T G contraction (forward) and its recomputing
// backward (dE/d em per slot); the math of embed.hip in double precision.
//
// What bounds it: the FP64 pipe.  On gfx950 a v_mfma_f64_16x16x4 holds it for
// 64 cycles and a v_fma_f64 for 4, and the two do not overlap (measured: 4 of
// the one and 64 of the other take 580 cycles together, 276 and 295 alone),
// so every FP64 operation that is left out is time.  Hence:
//  * type blocks are computed up to their last real neighbour, when the list
//    is given: the padding rows' sum comes from a host table, and in the
//    backward one of them stands for all where they are the same;
//  * the contractions with the four env-matrix components use
//    v_mfma_f64_4x4x4_4b (16 cycles): its four blocks are the four groups of
//    four channels (forward) or slots (backward), so no row of the 16 x 16
//    form is padding, and an accumulator block is one double per lane;
//  * channels are counted in steps of four (S1 = ceil(d1 / 4) of them per
//    resnet copy): widths (25, 50, 100) take 7 / 14 / 28 steps instead of the
//    8 / 16 / 32 of (32, 64, 128);
//  * tanh = 1 - 2 / (e^2x + 1) with e^2x = 2^(n/32) p(r): n to the nearest,
//    2^(j/32) from a table of 32 doubles in LDS (64 banks: no conflicts), p of
//    degree 5 (relative error 1.4e-16), the power of two and the clamp in
//    integer operations, which do not hold the FP64 pipe; v_rcp_f64
//    (4.6e-8) and one cubic step.  13 FP64 operations and a reciprocal.
//
// Organisation.  A tile of 16 slots per wavefront; lane (g = lane / 16, c =
// lane % 16).  An activation register t of a lane is channel 4 t + g of slot
// c: that is the A and the B layout of the MFMA alike, so layer 2 (and, in
// the backward, layer 3) is W (A) x activations (B) and stays in that layout,
// and layer 3 of the forward is activations (A) x W (B), whose result --
// slots 4 i + g, channel c -- is the operand the contraction needs; only y2
// (the resnet copy of layer 3) is turned through LDS for it.
//
// The workgroup holds every net's weights in LDS in fragment order (one
// conflict-free 8-byte read a lane and MFMA) when they fit, else lanes read
// them from memory through the caches.  Workgroups are persistent (one a CU);
// `split` wavefronts share an atom, taking every split-th tile of it and
// adding their parts in LDS in a fixed order, so that a few hundred atoms
// fill the chip as well as many thousands.
//
// Measured (forward / backward, us), against one wavefront an atom, every
// slot, 16 x 16 contractions and the library exp: water of 81 atoms 285 / 292
// -> 28 / 42, of 1,536 atoms 414 / 461 -> 115 / 179 (sel 46 + 92, two nets of
// 25, 50, 100); Cu of 5,324 atoms 926 / 1379 -> 651 / 1016 (sel 200, 32, 64,
// 128), where the FP64 pipe's own work is about 0.45 / 0.75 ms.
#include "dpk_common.h"
#include "tanh64.h"

namespace dpk {
namespace {

typedef __attribute__((ext_vector_type(4))) double v4d;

constexpr int kMaxTypes = 16;
constexpr int P1 = 32, P2 = 64, P3 = 128;  // internal widths of the packed parameters
// offsets of the packed parameters (include/dpk.h), in doubles
constexpr int O_B1 = P1, O_W2 = 2 * P1, O_B2 = O_W2 + P2 * P1, O_I2 = O_B2 + P2,
              O_W3 = O_I2 + P2, O_B3 = O_W3 + P3 * P2, O_I3 = O_B3 + P3, NET = O_I3 + P3;

struct EmbArgs {
  const double* em;
  const double* gxyz;    // backward
  const int* atype;
  const double* params;
  const int* net_of;
  const int* ch_out;
  const int* nlist;      // may be null: every slot is computed
  const double* pad;     // may be null
  double* out;
  int ntypes, nnets, d3, natoms, nnei, split;
  int res2, res3, idt;   // general kernels only
  ActSpec act;
  int sec[kMaxTypes + 1];
};

struct Act2 {
  double f, d;
};
// any other activation: one copy of the code for all places
__device__ __noinline__ Act2 act_general(ActSpec a, double z) {
  Act2 r;
  act_fd<double>(a, z, r.f, r.d);
  return r;
}

__device__ __forceinline__ v4d mma16(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ double mma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Channel steps: S1 of layer 1, 2 S1 of layer 2, 4 S1 of layer 3; step t,
// channel 4 t + g.  Internal (packed) channel of step t: 32 (t / S1) + 4 (t %
// S1) + g.  G (general): S1 = 8, run-time resnet modes, time steps and
// activation; otherwise tanh, doubling resnets, no time steps.
template <int S1_, bool G_>
struct Shape {
  static constexpr int S1 = S1_;
  static constexpr bool G = G_;
  static constexpr int S2 = 2 * S1, S3 = 4 * S1;
  static constexpr int B2 = (S2 + 3) / 4, B3 = S1;  // 16-channel blocks
  // one net in LDS, in doubles
  static constexpr int oW2 = 0, oW3 = B2 * S1 * 64, oV = oW3 + B3 * S2 * 64;
  static constexpr int vW1 = oV, vB1 = vW1 + 4 * S1, vB2 = vB1 + 4 * S1, vB3 = vB2 + 16 * B2,
                       vI2 = vB3 + 16 * B3, vI3 = vI2 + (G ? 16 * B2 : 0),
                       size = vI3 + (G ? 16 * B3 : 0);
  __device__ static __forceinline__ int inner(int n) {  // channel n -> internal channel
    const int t = n >> 2;
    return S1 == 8 ? n : 32 * (t / S1) + 4 * (t % S1) + (n & 3);
  }
};

// Parameters of a net, from LDS (fragment order) or from memory.
template <class SH, bool LDS>
struct Net {
  const double* p;
  int lane;
  // between 16-channel blocks: the next block's weights are not read (and held
  // in registers) early
  __device__ __forceinline__ void fence() const {
    if constexpr (!LDS) asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ double w2(int m, int ks) const {
    if constexpr (LDS) return p[SH::oW2 + (m * SH::S1 + ks) * 64 + lane];
    const int n = 16 * m + (lane & 15);
    if (n >= 4 * SH::S2) return 0.0;
    return p[O_W2 + SH::inner(n) * P1 + 4 * ks + (lane >> 4)];
  }
  __device__ __forceinline__ double w3(int m, int ks) const {
    if constexpr (LDS) return p[SH::oW3 + (m * SH::S2 + ks) * 64 + lane];
    return p[O_W3 + SH::inner(16 * m + (lane & 15)) * P2 + 32 * (ks / SH::S1) +
             4 * (ks % SH::S1) + (lane >> 4)];
  }
  __device__ __forceinline__ double w1(int n) const { return p[LDS ? SH::vW1 + n : n]; }
  __device__ __forceinline__ double b1(int n) const { return p[LDS ? SH::vB1 + n : O_B1 + n]; }
  __device__ __forceinline__ double b2(int n) const {
    return LDS ? p[SH::vB2 + n] : (n < 4 * SH::S2 ? p[O_B2 + SH::inner(n)] : 0.0);
  }
  __device__ __forceinline__ double b3(int n) const {
    return p[LDS ? SH::vB3 + n : O_B3 + SH::inner(n)];
  }
  __device__ __forceinline__ double i2(int n) const {
    return p[LDS ? SH::vI2 + n : O_I2 + SH::inner(n)];
  }
  __device__ __forceinline__ double i3(int n) const {
    return p[LDS ? SH::vI3 + n : O_I3 + SH::inner(n)];
  }
};

template <class SH>
__device__ __forceinline__ void stage_nets(double* w, const double* params, int nnets) {
  for (int k = 0; k < nnets; ++k) {
    double* o = w + (size_t)k * SH::size;
    const double* p = params + (size_t)k * NET;
    for (int q = threadIdx.x; q < SH::size; q += blockDim.x) {
      double v = 0.0;
      if (q < SH::oW3) {
        const int l = q & 63, ks = (q >> 6) % SH::S1, n = 16 * ((q >> 6) / SH::S1) + (l & 15);
        if (n < 4 * SH::S2) v = p[O_W2 + SH::inner(n) * P1 + 4 * ks + (l >> 4)];
      } else if (q < SH::oV) {
        const int r = q - SH::oW3, l = r & 63, ks = (r >> 6) % SH::S2;
        const int n = 16 * ((r >> 6) / SH::S2) + (l & 15);
        v = p[O_W3 + SH::inner(n) * P2 + SH::inner(4 * ks + (l >> 4))];
      } else if (q < SH::vB1) {
        v = p[q - SH::vW1];
      } else if (q < SH::vB2) {
        v = p[O_B1 + q - SH::vB1];
      } else if (q < SH::vB3) {
        if (q - SH::vB2 < 4 * SH::S2) v = p[O_B2 + SH::inner(q - SH::vB2)];
      } else if (q < SH::vI2) {
        v = p[O_B3 + SH::inner(q - SH::vB3)];
      } else if (q < SH::vI3) {
        if (q - SH::vI2 < 4 * SH::S2) v = p[O_I2 + SH::inner(q - SH::vI2)];
      } else {
        v = p[O_I3 + SH::inner(q - SH::vI3)];
      }
      o[q] = v;
    }
  }
}

// activation f and (DERIV) its derivative d at z
template <class SH, bool DERIV>
__device__ __forceinline__ void act64(const EmbArgs& A, const double* tab, double z, double& f,
                                      double& d) {
  if constexpr (SH::G) {
    if (A.act.id != DPK_ACT_TANH) {
      const Act2 r = act_general(A.act, z);
      f = r.f;
      d = r.d;
      return;
    }
  }
  f = tanh64(z, tab);
  if constexpr (DERIV) d = __fma_rn(-f, f, 1.0);
}

// Layers 1 and 2 for the lane's slot (s), with the tangents d/ds (DERIV).
template <class SH, bool LDS, bool DERIV>
__device__ __forceinline__ void layers12(const EmbArgs& A, const Net<SH, LDS>& net,
                                         const double* tab, double s, int g, double (&y2)[SH::S2],
                                         double (&d2)[DERIV ? SH::S2 : 1]) {
  double y1[SH::S1], d1[DERIV ? SH::S1 : 1];
#pragma unroll
  for (int t = 0; t < SH::S1; ++t) {
    const double w = net.w1(4 * t + g);
    double d = 0.0;
    act64<SH, DERIV>(A, tab, __fma_rn(s, w, net.b1(4 * t + g)), y1[t], d);
    if constexpr (DERIV) d1[t] = d * w;
  }
#pragma unroll
  for (int m = 0; m < SH::B2; ++m) {
    v4d acc, da = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = 4 * m + i < SH::S2 ? net.b2(16 * m + 4 * i + g) : 0.0;
#pragma unroll
    for (int ks = 0; ks < SH::S1; ++ks) {
      const double w = net.w2(m, ks);
      acc = mma16(w, y1[ks], acc);
      if constexpr (DERIV) da = mma16(w, d1[ks], da);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 4 * m + i;
      if (t >= SH::S2) continue;
      double f, d = 0.0;
      act64<SH, DERIV>(A, tab, acc[i], f, d);
      if constexpr (DERIV) d *= da[i];
      if constexpr (SH::G) {
        if (A.idt) {
          const double k = net.i2(16 * m + 4 * i + g);
          f *= k;
          if constexpr (DERIV) d *= k;
        }
        if (A.res2 == 2) {
          f += y1[t % SH::S1];
          if constexpr (DERIV) d += d1[t % SH::S1];
        }
      } else {
        f += y1[t % SH::S1];
        if constexpr (DERIV) d += d1[t % SH::S1];
      }
      y2[t] = f;
      if constexpr (DERIV) d2[t] = d;
    }
    net.fence();
  }
}

// Whether the env-matrix rows of the slots [b, e) are all that of slot b.
__device__ __forceinline__ bool same_rows(const double* em, int b, int e, int lane) {
  const long long* r = reinterpret_cast<const long long*>(em);
  bool same = true;
  for (int q = 4 * b + lane; q < 4 * e; q += 64) same = same && r[q] == r[4 * b + (lane & 3)];
  return __ballot(!same) == 0;
}

// Walks the tiles (16 slots from s0, up to b1) of an atom that fall to
// wavefront `sub` of `split`.  Forward: a block ends at its last real
// neighbour.  Backward (BWD): the padding rows after it are one slot more
// where they are all the same (fold), for all of which that slot stands;
// else they are computed like any other.
template <bool BWD, class F>
__device__ __forceinline__ void for_tiles(const EmbArgs& A, int atom, int sub, int lane,
                                          F&& body) {
  int turn = sub;  // tiles until this wavefront's next one
  const int ti = A.atype[atom] < 0 ? 0 : A.atype[atom];
  for (int t = 0; t < A.ntypes; ++t) {
    const int b0 = A.sec[t];
    int b1 = A.sec[t + 1];
    const int end = b1;
    bool fold = false;
    if (A.nlist != nullptr) {
      b1 = block_end(A.nlist + (size_t)atom * A.nnei, b0, b1, lane);
      if (BWD && b1 < end) {
        fold = same_rows(A.em + (size_t)atom * A.nnei * 4, b1, end, lane);
        b1 = fold ? b1 + 1 : end;
      }
    }
    const int net = A.net_of[ti * A.ntypes + t];
    int s0 = b0 + 16 * turn;
    for (; s0 < b1; s0 += 16 * A.split) body(net, s0, b1, fold ? end : b1);
    turn = (s0 - b0 - ((b1 - b0 + 15) / 16) * 16) / 16;
  }
}

// --------------------------------------------------------------- forward --
// Scratch of a wavefront: its 4 x 16 B3 partial sums, and before that the
// 16 x 17 tile that turns y2.
template <class SH>
constexpr int kFwdScratch = (4 * 16 * SH::B3 > 16 * 17 ? 4 * 16 * SH::B3 : 16 * 17);

template <class SH, bool LDS, int NW>
__global__ void __launch_bounds__(64 * NW) k_fwd64(EmbArgs A) {
  extern __shared__ __align__(16) double sm[];
  double* tab = sm;                                     // [32]
  double* scr = sm + 32;                                // [NW][kFwdScratch]
  double* nets = scr + (size_t)NW * kFwdScratch<SH>;    // LDS: [nnets][SH::size]
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  if constexpr (LDS) stage_nets<SH>(nets, A.params, A.nnets);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  const int per = NW / A.split, sub = wave % A.split, mine = wave / A.split;
  double* tile = scr + (size_t)wave * kFwdScratch<SH>;
  const double* part = scr + (size_t)(wave - sub) * kFwdScratch<SH>;
  const double inv = 1.0 / (double)A.nnei;
  const int sn = 16 * SH::B3;  // channels of a partial row
  for (int base = blockIdx.x * per; base < A.natoms; base += gridDim.x * per) {
    const int atom = base + mine;
    if (atom < A.natoms) {
      const double* e = A.em + (size_t)atom * A.nnei * 4;
      double acc[SH::B3], accy[SH::B2];
#pragma unroll
      for (int m = 0; m < SH::B3; ++m) acc[m] = 0.0;
#pragma unroll
      for (int m = 0; m < SH::B2; ++m) accy[m] = 0.0;
      for_tiles<false>(A, atom, sub, lane, [&](int k, int s0, int b1, int) {
        asm volatile("" ::: "memory");  // weights are read every tile, not kept in registers
        const Net<SH, LDS> net{LDS ? nets + (size_t)k * SH::size : A.params + (size_t)k * NET,
                               lane};
        const double s = s0 + c < b1 ? e[(s0 + c) * 4] : 0.0;
        double rT[4];  // component c % 4 of slot 4 i + g
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int sl = s0 + 4 * i + g;
          rT[i] = sl < b1 ? e[sl * 4 + (c & 3)] : 0.0;
        }
        double y2[SH::S2], none[1];
        layers12<SH, LDS, false>(A, net, tab, s, g, y2, none);
        if (!SH::G || A.res3 == 2) {
#pragma unroll
          for (int m = 0; m < SH::B2; ++m) {  // turn y2: slots on the registers
#pragma unroll
            for (int i = 0; i < 4; ++i)
              tile[c * 17 + 4 * i + g] = 4 * m + i < SH::S2 ? y2[4 * m + i < SH::S2 ? 4 * m + i : 0] : 0.0;
            wave_sync();
#pragma unroll
            for (int i = 0; i < 4; ++i) accy[m] = mma4(rT[i], tile[(4 * i + g) * 17 + c], accy[m]);
            wave_sync();
          }
        }
#pragma unroll
        for (int m = 0; m < SH::B3; ++m) {
          const double b = net.b3(16 * m + c);
          v4d z = {b, b, b, b};
#pragma unroll
          for (int ks = 0; ks < SH::S2; ++ks) z = mma16(y2[ks], net.w3(m, ks), z);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            double f, d;
            act64<SH, false>(A, tab, z[i], f, d);
            if constexpr (SH::G) {
              if (A.idt) f *= net.i3(16 * m + c);
            }
            acc[m] = mma4(rT[i], f, acc[m]);
          }
          net.fence();
        }
      });
      if (A.pad != nullptr && A.nlist != nullptr && sub == 0 && A.atype[atom] >= 0) {
        const int ti = A.atype[atom];
        for (int t = 0; t < A.ntypes; ++t) {
          const int b1 = block_end(A.nlist + (size_t)atom * A.nnei, A.sec[t], A.sec[t + 1], lane);
          if (b1 >= A.sec[t + 1]) continue;
          const double* pt = A.pad + (((size_t)ti * A.nnei + b1) * 4 + g) * P3;
#pragma unroll
          for (int m = 0; m < SH::B3; ++m) acc[m] += pt[SH::inner(16 * m + c)];
        }
      }
      // lane (g, c): component g, channels 16 m + c of the wavefront's tiles;
      // the resnet part of channel n is that of channel n mod 4 S2 of y2
#pragma unroll
      for (int m = 0; m < SH::B3; ++m) tile[g * sn + 16 * m + c] = acc[m];
      wave_sync();
#pragma unroll
      for (int m = 0; m < SH::B2; ++m) {
        const int n = 16 * m + c;
        if (n < 4 * SH::S2) {
          tile[g * sn + n] += accy[m];
          tile[g * sn + n + 4 * SH::S2] += accy[m];
        }
      }
    }
    if (A.split > 1) __syncthreads();
    else wave_sync();
    if (atom < A.natoms) {
      double* o = A.out + (size_t)atom * 4 * A.d3;
      for (int q = sub * 64 + lane; q < 4 * sn; q += 64 * A.split) {
        double v = 0.0;
        for (int w = 0; w < A.split; ++w) v += part[(size_t)w * kFwdScratch<SH> + q];
        const int tc = A.ch_out[SH::inner(q % sn)];
        if (tc >= 0) o[(q / sn) * A.d3 + tc] = v * inv;
      }
    }
    if (A.split > 1) __syncthreads();
    else wave_sync();
  }
}

// -------------------------------------------------------------- backward --
// Scratch of a wavefront: its atom's dE/dxyz / nnei, rows of gs (4 more than
// the channels: the four rows a read touches lie in different banks).
template <class SH>
constexpr int kGs = 16 * SH::B3 + 4;

template <class SH, bool LDS, int NW>
__global__ void __launch_bounds__(64 * NW) k_bwd64(EmbArgs A) {
  extern __shared__ __align__(16) double sm[];
  double* tab = sm;
  double* scr = sm + 32;
  double* nets = scr + (size_t)NW * 4 * kGs<SH>;
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  if constexpr (LDS) stage_nets<SH>(nets, A.params, A.nnets);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  double* gx = scr + (size_t)wave * 4 * kGs<SH>;
  const double inv = 1.0 / (double)A.nnei;
  const long units = (long)A.natoms * A.split;
  for (long u = (long)blockIdx.x * NW + wave; u < units; u += (long)gridDim.x * NW) {
    // (the turn of the parts goes round: a wavefront's units are all sizes)
    const int atom = (int)(u / A.split), sub = (int)((u + atom) % A.split);
    const double* e = A.em + (size_t)atom * A.nnei * 4;
    double* nd = A.out + (size_t)atom * A.nnei * 4;
    wave_sync();
    for (int q = lane; q < 4 * 16 * SH::B3; q += 64) {
      const int n = q % (16 * SH::B3), cc = q / (16 * SH::B3), tc = A.ch_out[SH::inner(n)];
      gx[cc * kGs<SH> + n] =
          tc >= 0 ? A.gxyz[(size_t)atom * 4 * A.d3 + cc * A.d3 + tc] * inv : 0.0;
    }
    wave_sync();
    for_tiles<true>(A, atom, sub, lane, [&](int k, int s0, int b1, int end) {
      asm volatile("" ::: "memory");  // weights are read every tile, not kept in registers
      const Net<SH, LDS> net{LDS ? nets + (size_t)k * SH::size : A.params + (size_t)k * NET,
                             lane};
      const int slot = s0 + c;
      const double s = slot < b1 ? e[slot * 4] : 0.0;
      double y2[SH::S2], d2[SH::S2];
      layers12<SH, LDS, true>(A, net, tab, s, g, y2, d2);
      double dR = 0.0, Mx = 0.0;  // component g of slot c
#pragma unroll
      for (int m = 0; m < SH::B3; ++m) {
        v4d z, dz = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] = net.b3(16 * m + 4 * i + g);
#pragma unroll
        for (int ks = 0; ks < SH::S2; ++ks) {
          const double w = net.w3(m, ks);
          z = mma16(w, y2[ks], z);
          dz = mma16(w, d2[ks], dz);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = (4 * m + i) % SH::S2;
          double f, d;
          act64<SH, true>(A, tab, z[i], f, d);
          if constexpr (SH::G) {
            d *= dz[i];
            if (A.idt) {
              const double ts = net.i3(16 * m + 4 * i + g);
              f *= ts;
              d *= ts;
            }
            if (A.res3 == 2) {
              f += y2[t];
              d += d2[t];
            }
          } else {
            f += y2[t];
            d = __fma_rn(d, dz[i], d2[t]);
          }
          const double ga = gx[(c & 3) * kGs<SH> + 16 * m + 4 * i + g];
          dR = mma4(ga, f, dR);
          Mx = mma4(ga, d, Mx);
        }
        net.fence();
      }
      const double R = slot < b1 ? e[slot * 4 + g] : 0.0;
      double ds = R * Mx;
      ds += __shfl_xor(ds, 16, 64);
      ds += __shfl_xor(ds, 32, 64);
      const double v = g == 0 ? dR + ds : dR;
      if (slot < b1) nd[slot * 4 + g] = v;
      if (end > b1 && b1 <= s0 + 16) {  // slot b1 - 1 stands for the padding after it
        const double w = __shfl(v, 16 * g + (b1 - 1 - s0), 64);
        for (int q = b1 + c; q < end; q += 16) nd[q * 4 + g] = w;
      }
    });
  }
}

constexpr int kLdsMax = 160 * 1024;

// Wavefronts a workgroup: two nets of (25, 50, 100) fit in LDS beside the
// scratch of eight.  Twelve and sixteen gave nothing where they fit (Cu of
// 5,324 atoms: forward 656 and 692 us against 667, backward 1065 and 1104
// against 1038): two wavefronts a SIMD keep the FP64 pipe busy.
constexpr int kWaves = 8;

// `split`: the least work in the fullest round of wavefronts, rounds(split) *
// tiles(split) -- with few atoms their tiles are spread over several
// wavefronts, and with many a finer split evens out the last round (5,324 Cu
// atoms of 12 tiles on 2,048 wavefronts: 3 rounds of 12 tiles whole, 11 of 3
// split by four).  Tiles an atom: sel is set about a tenth above the
// neighbours a system has.
int choose_split(int natoms, int tiles, int waves) {
  int best = 1;
  long cost = -1;
  for (int s = 1; s <= kWaves; s *= 2) {
    const long c = (((long)natoms * s + waves - 1) / waves) * ((tiles + s - 1) / s);
    if (cost < 0 || c < cost) {
      cost = c;
      best = s;
    }
  }
  return best;
}

template <class SH, bool LDS>
int launch64(bool fwd, EmbArgs& A, hipStream_t st) {
  constexpr int NW = kWaves;
  static int ncu[64];
  int dev = 0;
  DPK_HIP(hipGetDevice(&dev));
  DPK_REQUIRE(dev >= 0 && dev < 64, DPK_ERR_ARG, "embed: device %d out of range", dev);
  if (ncu[dev] == 0)
    DPK_HIP(hipDeviceGetAttribute(&ncu[dev], hipDeviceAttributeMultiprocessorCount, dev));
  const size_t lds =
      sizeof(double) * (32 + (size_t)NW * (fwd ? kFwdScratch<SH> : 4 * kGs<SH>) +
                        (LDS ? (size_t)A.nnets * SH::size : 0));
  int tiles = 0;
  for (int t = 0; t < A.ntypes; ++t) tiles += (9 * (A.sec[t + 1] - A.sec[t]) / 10 + 15) / 16;
  A.split = choose_split(A.natoms, tiles, ncu[dev] * NW);
  const long want = ((long)A.natoms * A.split + NW - 1) / NW;
  // LDS: one workgroup a CU; without, the register budget's two
  const long room = (long)ncu[dev] * (LDS ? 1 : 2);
  const unsigned grid = (unsigned)(want < room ? want : room);
  if (fwd)
    hipLaunchKernelGGL((k_fwd64<SH, LDS, NW>), dim3(grid), dim3(64 * NW), lds, st, A);
  else
    hipLaunchKernelGGL((k_bwd64<SH, LDS, NW>), dim3(grid), dim3(64 * NW), lds, st, A);
  DPK_LAUNCHED();
  return DPK_OK;
}

template <class SH>
int launch_shape(bool fwd, EmbArgs& A, hipStream_t st) {
  const size_t most = 32 + (size_t)kWaves * (kFwdScratch<SH> > 4 * kGs<SH> ? kFwdScratch<SH>
                                                                            : 4 * kGs<SH>);
  if (sizeof(double) * (most + (size_t)A.nnets * SH::size) <= kLdsMax)
    return launch64<SH, true>(fwd, A, st);
  return launch64<SH, false>(fwd, A, st);
}

}  // namespace

int embed_f64(bool fwd, void* out, const void* em, const void* gx, const int* atype,
              const void* params, const int* net_of, const int* ch_out, int ntypes, int nnets,
              int res2, int res3, int has_idt, const ActSpec& act, int d3, const int* sec_host,
              int natoms, int nnei, const int* nlist, const double* pad, hipStream_t st) {
  EmbArgs A;
  A.em = static_cast<const double*>(em);
  A.gxyz = static_cast<const double*>(gx);
  A.atype = atype;
  A.params = static_cast<const double*>(params);
  A.net_of = net_of;
  A.ch_out = ch_out;
  A.nlist = nlist;
  A.pad = pad;
  A.out = static_cast<double*>(out);
  A.ntypes = ntypes;
  A.nnets = nnets;
  A.d3 = d3;
  A.natoms = natoms;
  A.nnei = nnei;
  A.split = 1;
  A.res2 = res2;
  A.res3 = res3;
  A.idt = has_idt;
  A.act = act;
  for (int t = 0; t <= ntypes; ++t) A.sec[t] = sec_host[t];
  if (act.id != DPK_ACT_TANH || has_idt || res2 != 2 || res3 != 2)
    return launch_shape<Shape<8, true>>(fwd, A, st);
  // doubling resnets: d3 = 4 d1, so d3 <= 112 leaves the eighth step of every
  // copy empty
  if (d3 <= 112) return launch_shape<Shape<7, false>>(fwd, A, st);
  return launch_shape<Shape<8, false>>(fwd, A, st);
}

}  // namespace dpk
