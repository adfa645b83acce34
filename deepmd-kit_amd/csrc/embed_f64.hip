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
// The workgroup holds the weights in LDS in fragment order (one conflict-free
// 8-byte read a lane and MFMA): of every net where they fit together (one of
// width 128, two of 100), else a group of nets at a time, the atoms that use it
// dealt to the wavefronts (k_fwd64 / k_bwd64, ALL false).  Workgroups are
// persistent (one a CU); `split` wavefronts share an atom, taking every
// split-th tile of it and adding their parts in LDS in a fixed order, so that
// a few hundred atoms fill the chip as well as many thousands.
//
// Groups, against fragments read from memory through the caches (activations
// spilled: 900 to 1,500 bytes a lane), forward / backward us: two nets of 128,
// water of 375 atoms 154 / 178 -> 73 / 104, 1,536 482 / 577 -> 152 / 233, 5,184
// 1,352 / 1,593 -> 380 / 581; four nets of 100: 81 atoms 34 / 42 -> 34 / 48, 375
// 62 / 75 -> 70 / 91, 1,536 210 / 236 -> 136 / 196, 5,184 580 / 643 -> 327 / 473;
// sixteen of 128, 14,374 atoms of four types: 3,990 / 5,224 -> 1,096 / 1,720;
// gelu, two nets of 100, 1,536 atoms 728 / 888 -> 416 / 528.
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
  int room;              // nets that fit in LDS together
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
// S1) + g.  Kinds: tanh with doubling resnets and no time steps; G (general, S1
// = 8): run-time resnet modes and time steps, with tanh or any activation.
enum { kPlain = 0, kTanh = 1, kAny = 2 };
template <int S1_, int KIND_>
struct Shape {
  static constexpr int S1 = S1_, KIND = KIND_;
  static constexpr bool G = KIND != kPlain;
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

// Parameters of a net in LDS.
template <class SH>
struct Net {
  const double* p;
  int lane;
  // between 16-channel blocks: the next block's weights are not read (and held
  // in registers) early
  __device__ __forceinline__ void fence() const { __builtin_amdgcn_sched_barrier(0); }
  __device__ __forceinline__ double w2(int m, int ks) const {
    return p[SH::oW2 + (m * SH::S1 + ks) * 64 + lane];
  }
  __device__ __forceinline__ double w3(int m, int ks) const {
    return p[SH::oW3 + (m * SH::S2 + ks) * 64 + lane];
  }
  __device__ __forceinline__ double w1(int n) const { return p[SH::vW1 + n]; }
  __device__ __forceinline__ double b1(int n) const { return p[SH::vB1 + n]; }
  __device__ __forceinline__ double b2(int n) const { return p[SH::vB2 + n]; }
  __device__ __forceinline__ double b3(int n) const { return p[SH::vB3 + n]; }
  __device__ __forceinline__ double i2(int n) const { return p[SH::vI2 + n]; }
  __device__ __forceinline__ double i3(int n) const { return p[SH::vI3 + n]; }
};

// Nets list[p0 .. p1) (list null: nets p0 .. p1) to LDS in fragment order, a
// fragment (64 values) a wavefront and load, all of a wavefront's loads of a
// net in flight together.
template <class SH, int NW>
__device__ __forceinline__ void stage_nets(double* w, const double* params,
                                           const unsigned short* list, int p0, int p1, int wave,
                                           int lane) {
  constexpr int F2 = SH::B2 * SH::S1, F3 = SH::B3 * SH::S2;
  const int g = lane >> 4, c = lane & 15;
  for (int q = p0; q < p1; ++q) {
    const int k = list != nullptr ? __builtin_amdgcn_readfirstlane(list[q]) : q;
    double* o = w + (size_t)(q - p0) * SH::size;
    const double* p = params + (size_t)k * NET;
#pragma unroll
    for (int i = 0; i < (F2 + NW - 1) / NW; ++i) {
      const int f = wave + NW * i, n = 16 * (f / SH::S1) + c;
      if (f < F2)
        o[SH::oW2 + f * 64 + lane] =
            n < 4 * SH::S2 ? p[O_W2 + SH::inner(n) * P1 + 4 * (f % SH::S1) + g] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < (F3 + NW - 1) / NW; ++i) {
      const int f = wave + NW * i;
      if (f < F3)
        o[SH::oW3 + f * 64 + lane] = p[O_W3 + SH::inner(16 * (f / SH::S2) + c) * P2 +
                                       SH::inner(4 * (f % SH::S2) + g)];
    }
    for (int i = SH::oV + threadIdx.x; i < SH::size; i += 64 * NW) {
      double v = 0.0;
      if (i < SH::vB1) {
        v = p[i - SH::vW1];
      } else if (i < SH::vB2) {
        v = p[O_B1 + i - SH::vB1];
      } else if (i < SH::vB3) {
        if (i - SH::vB2 < 4 * SH::S2) v = p[O_B2 + SH::inner(i - SH::vB2)];
      } else if (i < SH::vI2) {
        v = p[O_B3 + SH::inner(i - SH::vB3)];
      } else if (i < SH::vI3) {
        if (i - SH::vI2 < 4 * SH::S2) v = p[O_I2 + SH::inner(i - SH::vI2)];
      } else {
        v = p[O_I3 + SH::inner(i - SH::vI3)];
      }
      o[i] = v;
    }
  }
}

// Nets that don't fit in LDS together are taken in groups of `room`: a
// workgroup lists the nets that its atoms use, stages a group, works off the
// type blocks that use one of its nets, and goes on to the next.
constexpr int kMaxNets = kMaxTypes * kMaxTypes;
struct Groups {
  unsigned short list[kMaxNets];  // the nets used, ascending
  unsigned short at[kMaxNets];    // a net's place in the list (kMaxNets: not used)
  unsigned types;                 // the types of the atoms, a bit each
};

// Lists the nets of the workgroup's atoms, `per` of them a turn of the grid
// (virtual atoms count as type 0), and returns how many there are.
__device__ __forceinline__ int list_nets(const EmbArgs& A, Groups& G, int per) {
  if (threadIdx.x == 0) G.types = 0;
  for (int q = threadIdx.x; q < kMaxNets; q += blockDim.x) G.at[q] = kMaxNets;
  __syncthreads();
  unsigned m = 0;
  for (int q = threadIdx.x;; q += blockDim.x) {
    const long base = ((long)blockIdx.x + (long)(q / per) * gridDim.x) * per;
    if (base >= A.natoms) break;
    const long atom = base + q % per;
    if (atom < A.natoms) m |= 1u << (A.atype[atom] < 0 ? 0 : A.atype[atom]);
  }
  if (m != 0) atomicOr(&G.types, m);
  __syncthreads();
  for (int q = threadIdx.x; q < A.ntypes * A.ntypes; q += blockDim.x) {
    const int t = q % A.ntypes;
    if ((G.types >> (q / A.ntypes) & 1) && A.sec[t + 1] > A.sec[t]) G.at[A.net_of[q]] = 0;
  }
  __syncthreads();
  int n = 0;
  for (int k = 0; k < A.nnets; ++k) {  // (every thread counts)
    const bool use = G.at[k] < kMaxNets;
    if (use && threadIdx.x == 0) G.list[n] = (unsigned short)k;
    n += use;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += blockDim.x) G.at[G.list[q]] = (unsigned short)q;
  __syncthreads();
  return n;
}

// The blocks (a bit each) of centre type ti that use a net of the group [p0,
// p1); earlier: whether a former group had one.
__device__ __forceinline__ unsigned group_blocks(const EmbArgs& A, const Groups& G, int p0, int p1,
                                                 int ti, bool& earlier) {
  unsigned m = 0;
  earlier = false;
  for (int t = 0; t < A.ntypes; ++t) {
    if (A.sec[t + 1] <= A.sec[t]) continue;
    const int at = __builtin_amdgcn_readfirstlane(G.at[A.net_of[ti * A.ntypes + t]]);
    earlier = earlier || at < p0;
    if (at >= p0 && at < p1) m |= 1u << t;
  }
  return m;
}

// The centre types (a bit each) that have a block in the group.
__device__ __forceinline__ unsigned group_types(const EmbArgs& A, const Groups& G, int p0, int p1,
                                                int lane) {
  bool has = false;
  if (lane < A.ntypes)
    for (int t = 0; t < A.ntypes; ++t) {
      const int at = G.at[A.net_of[lane * A.ntypes + t]];
      has = has || (A.sec[t + 1] > A.sec[t] && at >= p0 && at < p1);
    }
  return (unsigned)__ballot(has);
}

// Of the workgroup's atoms q0 .. q0 + 63 (`per` of them a turn of the grid)
// those of the given types, a bit each; first: atom of the bit 0, or past the
// end.
__device__ __forceinline__ int atom_at(int q, int per) {
  return (int)((blockIdx.x + (long)(q / per) * gridDim.x) * per + q % per);
}
__device__ __forceinline__ unsigned long long atoms_of(const EmbArgs& A, unsigned types, int q0,
                                                       int per, int lane) {
  const int atom = atom_at(q0 + lane, per);
  bool take = false;
  if (atom < A.natoms) take = types >> (A.atype[atom] < 0 ? 0 : A.atype[atom]) & 1;
  return __ballot(take);
}
__device__ __forceinline__ int nth_bit(unsigned long long m, int n) {
  for (; n > 0; --n) m &= m - 1;
  return __ffsll(m) - 1;
}

// activation f and (DERIV) its derivative d at z
template <class SH, bool DERIV>
__device__ __forceinline__ void act64(const EmbArgs& A, const double* tab, double z, double& f,
                                      double& d) {
  if constexpr (SH::KIND == kAny) {
    const Act2 r = act_general(A.act, z);
    f = r.f;
    d = r.d;
    return;
  }
  f = tanh64(z, tab);
  if constexpr (DERIV) d = __fma_rn(-f, f, 1.0);
}

// Layers 1 and 2 for the lane's slot (s), with the tangents d/ds (DERIV).
template <class SH, bool DERIV>
__device__ __forceinline__ void layers12(const EmbArgs& A, const Net<SH>& net,
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
// wavefront `sub` of `split`, in the blocks of the mask.  Forward: a block ends
// at its last real neighbour.  Backward (BWD): the padding rows after it are one slot more
// where they are all the same (fold), for all of which that slot stands;
// else they are computed like any other.
template <bool BWD, class F>
__device__ __forceinline__ void for_tiles(const EmbArgs& A, int atom, int ti, unsigned blocks,
                                          int sub, int lane, F&& body) {
  int turn = sub;  // tiles until this wavefront's next one
  for (int t = 0; t < A.ntypes; ++t) {
    if (!(blocks >> t & 1)) continue;
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

// A workgroup's LDS, in doubles: the table and (nets in groups) their list, the
// scratch, the nets.
constexpr int kHeadAll = 32, kHead = 32 + (int)((sizeof(Groups) + 15) / 16 * 2);

// ALL: the nets fit in LDS together (one group)
template <class SH, bool ALL, int NW>
__global__ void __launch_bounds__(64 * NW) k_fwd64(EmbArgs A) {
  extern __shared__ __align__(16) double sm[];
  double* tab = sm;                                     // [32]
  Groups& groups = *reinterpret_cast<Groups*>(sm + kHeadAll);
  double* scr = sm + (ALL ? kHeadAll : kHead);          // [NW][kFwdScratch]
  double* nets = scr + (size_t)NW * kFwdScratch<SH>;    // [room][SH::size]
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  const int per = NW / A.split, sub = wave % A.split, mine = wave / A.split;
  double* tile = scr + (size_t)wave * kFwdScratch<SH>;
  const double* part = scr + (size_t)(wave - sub) * kFwdScratch<SH>;
  const double inv = 1.0 / (double)A.nnei;
  const int sn = 16 * SH::B3;  // channels of a partial row
  const bool dyn = !ALL && A.split == 1;
  const int used = ALL ? A.nnets : list_nets(A, groups, per);
  int p0 = 0, p1 = 0;
  do {
    p0 = p1;
    p1 = ALL || p0 + A.room > used ? used : p0 + A.room;
    if (!ALL) __syncthreads();  // the wavefronts are done with the nets before
    stage_nets<SH, NW>(nets, A.params, ALL ? nullptr : groups.list, p0, p1, wave, lane);
    __syncthreads();
    // one turn: an atom for every `split` wavefronts, or (work false) none
    auto turn = [&](int atom, bool work) {
      int ti = 0;
      unsigned blocks = ~0u;
      bool earlier = false;
      if (work) {
        ti = A.atype[atom] < 0 ? 0 : A.atype[atom];
        if constexpr (!ALL) blocks = group_blocks(A, groups, p0, p1, ti, earlier);
      }
      if (work) {
        const double* e = A.em + (size_t)atom * A.nnei * 4;
        double acc[SH::B3], accy[SH::B2];
#pragma unroll
        for (int m = 0; m < SH::B3; ++m) acc[m] = 0.0;
#pragma unroll
        for (int m = 0; m < SH::B2; ++m) accy[m] = 0.0;
        for_tiles<false>(A, atom, ti, blocks, sub, lane, [&](int k, int s0, int b1, int) {
          asm volatile("" ::: "memory");  // weights are read every tile, not kept in registers
          const Net<SH> net{nets + (size_t)((ALL ? k : groups.at[k]) - p0) * SH::size, lane};
          const double s = s0 + c < b1 ? e[(s0 + c) * 4] : 0.0;
          double rT[4];  // component c % 4 of slot 4 i + g
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int sl = s0 + 4 * i + g;
            rT[i] = sl < b1 ? e[sl * 4 + (c & 3)] : 0.0;
          }
          double y2[SH::S2], none[1];
          layers12<SH, false>(A, net, tab, s, g, y2, none);
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
          for (int t = 0; t < A.ntypes; ++t) {
            if (!(blocks >> t & 1)) continue;
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
      if (work) {
        double* o = A.out + (size_t)atom * 4 * A.d3;
        for (int q = sub * 64 + lane; q < 4 * sn; q += 64 * A.split) {
          double v = 0.0;
          for (int w = 0; w < A.split; ++w) v += part[(size_t)w * kFwdScratch<SH> + q];
          const int tc = A.ch_out[SH::inner(q % sn)];
          if (tc < 0) continue;
          double* r = o + (q / sn) * A.d3 + tc;
          *r = earlier ? *r + v * inv : v * inv;
        }
      }
      if (A.split > 1) __syncthreads();
      else wave_sync();
    };
    if constexpr (ALL) {
      for (int base = blockIdx.x * per; base < A.natoms; base += gridDim.x * per)
        turn(base + mine, base + mine < A.natoms);
    } else {
      const unsigned types = group_types(A, groups, p0, p1, lane);
      int dealt = 0;  // whole atoms go to the wavefronts in turn
      for (int q0 = 0; atom_at(q0, per) < A.natoms; q0 += 64) {
        const unsigned long long m = atoms_of(A, types, q0, per, lane);
        const int n = __popcll(m), off = A.split == 1 ? (mine - dealt) & (per - 1) : mine;
        for (int i = 0; i < n; i += per)
          turn(atom_at(q0 + nth_bit(m, i + off < n ? i + off : 0), per), i + off < n);
        dealt += n;
      }
    }
  } while (!ALL && p1 < used);
}

// -------------------------------------------------------------- backward --
// Scratch of a wavefront: its atom's dE/dxyz / nnei, rows of gs (4 more than
// the channels: the four rows a read touches lie in different banks).
template <class SH>
constexpr int kGs = 16 * SH::B3 + 4;

template <class SH, bool ALL, int NW>
__global__ void __launch_bounds__(64 * NW) k_bwd64(EmbArgs A) {
  extern __shared__ __align__(16) double sm[];
  double* tab = sm;
  Groups& groups = *reinterpret_cast<Groups*>(sm + kHeadAll);
  double* scr = sm + (ALL ? kHeadAll : kHead);
  double* nets = scr + (size_t)NW * 4 * kGs<SH>;
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  double* gx = scr + (size_t)wave * 4 * kGs<SH>;
  const double inv = 1.0 / (double)A.nnei;
  const long units = (long)A.natoms * A.split;
  const int used = ALL ? A.nnets : list_nets(A, groups, NW / A.split);
  int p0 = 0, p1 = 0;
  do {
    p0 = p1;
    p1 = ALL || p0 + A.room > used ? used : p0 + A.room;
    if (!ALL) __syncthreads();
    stage_nets<SH, NW>(nets, A.params, ALL ? nullptr : groups.list, p0, p1, wave, lane);
    __syncthreads();
    // part `sub` of an atom's tiles
    auto unit = [&](int atom, int sub) {
      const int ti = A.atype[atom] < 0 ? 0 : A.atype[atom];
      unsigned blocks = ~0u;
      if constexpr (!ALL) {
        bool earlier;
        blocks = group_blocks(A, groups, p0, p1, ti, earlier);
      }
      const double* e = A.em + (size_t)atom * A.nnei * 4;
      double* nd = A.out + (size_t)atom * A.nnei * 4;
      wave_sync();
      for (int q = lane; q < 4 * 16 * SH::B3; q += 64) {
        const int n = q % (16 * SH::B3), cc = q / (16 * SH::B3), tc = A.ch_out[SH::inner(n)];
        gx[cc * kGs<SH> + n] =
            tc >= 0 ? A.gxyz[(size_t)atom * 4 * A.d3 + cc * A.d3 + tc] * inv : 0.0;
      }
      wave_sync();
      for_tiles<true>(A, atom, ti, blocks, sub, lane, [&](int k, int s0, int b1, int end) {
        asm volatile("" ::: "memory");  // weights are read every tile, not kept in registers
        const Net<SH> net{nets + (size_t)((ALL ? k : groups.at[k]) - p0) * SH::size, lane};
        const int slot = s0 + c;
        const double s = slot < b1 ? e[slot * 4] : 0.0;
        double y2[SH::S2], d2[SH::S2];
        layers12<SH, true>(A, net, tab, s, g, y2, d2);
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
    };
    // (the turn of the parts goes round: a wavefront's units are all sizes)
    if constexpr (ALL) {
      for (long u = (long)blockIdx.x * NW + wave; u < units; u += (long)gridDim.x * NW) {
        const int atom = (int)(u / A.split);
        unit(atom, (int)((u + atom) % A.split));
      }
    } else {
      const unsigned types = group_types(A, groups, p0, p1, lane);
      const int per = NW / A.split;
      int dealt = 0;
      for (int q0 = 0; atom_at(q0, per) < A.natoms; q0 += 64) {
        const unsigned long long m = atoms_of(A, types, q0, per, lane);
        const int n = __popcll(m) * A.split;
        for (int i = (wave - dealt) & (NW - 1); i < n; i += NW) {
          const int atom = atom_at(q0 + nth_bit(m, i / A.split), per);
          unit(atom, (i + atom) % A.split);
        }
        dealt += n;
      }
    }
  } while (!ALL && p1 < used);
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
// neighbours a system has.  Nets in groups: a group's blocks may hold any
// number of tiles, so the atoms that use a group (all, or with a net a centre
// and neighbour type `share` of them) are split only while the chip is not full.
int choose_split(const EmbArgs& A, int tiles, int ncu) {
  const long waves = (long)ncu * kWaves;
  int best = 1;
  if (A.room < A.nnets) {
    const bool pairs = A.nnets > A.ntypes;  // a net a centre and neighbour type
    const double share = pairs && A.room < A.ntypes ? (double)A.room / A.ntypes : 1.0;
    while (best < kWaves && A.natoms * share * 2 * best <= (double)waves) best *= 2;
    return best;
  }
  long cost = -1;
  for (int s = 1; s <= kWaves; s *= 2) {
    const long c = (((long)A.natoms * s + waves - 1) / waves) * ((tiles + s - 1) / s);
    if (cost < 0 || c < cost) {
      cost = c;
      best = s;
    }
  }
  return best;
}

template <class SH>
int launch64(bool fwd, EmbArgs& A, hipStream_t st) {
  constexpr int NW = kWaves;
  int dev = 0, ncu = 0;
  const int rc = device_cus(&dev, &ncu);
  if (rc != DPK_OK) return rc;
  constexpr int kMost = NW * (kFwdScratch<SH> > 4 * kGs<SH> ? kFwdScratch<SH> : 4 * kGs<SH>);
  constexpr int kRoom = (kLdsMax / 8 - kHead - kMost) / SH::size;
  static_assert(kRoom >= 1, "a net fits in LDS beside the scratch");
  A.room = kRoom < A.nnets ? kRoom : A.nnets;
  const bool all = A.room == A.nnets;
  const size_t lds =
      sizeof(double) * ((all ? kHeadAll : kHead) + (size_t)NW * (fwd ? kFwdScratch<SH> : 4 * kGs<SH>) +
                        (size_t)A.room * SH::size);
  int tiles = 0;
  for (int t = 0; t < A.ntypes; ++t) tiles += (9 * (A.sec[t + 1] - A.sec[t]) / 10 + 15) / 16;
  A.split = choose_split(A, tiles, ncu);
  const long want = ((long)A.natoms * A.split + NW - 1) / NW;
  const unsigned grid = (unsigned)(want < ncu ? want : ncu);  // one workgroup a CU
  const auto kernel = fwd ? (all ? k_fwd64<SH, true, NW> : k_fwd64<SH, false, NW>)
                          : (all ? k_bwd64<SH, true, NW> : k_bwd64<SH, false, NW>);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * NW), lds, st, A);
  DPK_LAUNCHED();
  return DPK_OK;
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
  A.room = nnets;
  if (act.id != DPK_ACT_TANH) return launch64<Shape<8, kAny>>(fwd, A, st);
  if (has_idt || res2 != 2 || res3 != 2) return launch64<Shape<8, kTanh>>(fwd, A, st);
  // doubling resnets: d3 = 4 d1, so d3 <= 112 leaves the eighth step of every
  // copy empty
  if (d3 <= 112) return launch64<Shape<7, kPlain>>(fwd, A, st);
  return launch64<Shape<8, kPlain>>(fwd, A, st);
}

}  // namespace dpk
