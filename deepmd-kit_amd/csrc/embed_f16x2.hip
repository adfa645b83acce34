// FP16X2 se_e2_a embedding net + R^T G contraction (forward) and its
// recomputing backward (dE/d em per slot): FP16 weights, every data operand
// split into two FP16 values (hi = fp16(x), lo = fp16(x - hi)), FP32
// accumulation; the math of embed.hip.  Reference: deepmd/pt/model/descriptor/
// se_a.py:784-858, deepmd/pt/model/network/mlp.py:188-219.
//
// What bounds it: instruction issue.  A SIMD issues a plain VALU instruction
// in 4 cycles, an exp2 / rcp in 8, a 16x16x32 MFMA in 8 (measured, the matrix
// core itself being busy for 16); a tile of 16 slots costs 112 exp2 / rcp, 60
// (forward) or 104 (backward) MFMAs and 269 or 484 others, of which the issue
// takes about 80% of the time.  What keeps the count down:
//  * with r = 1 / (1 + e^2x), 1 - tanh^2 x = 4 (r - r^2) is one FMA, its 4
//    applied once a tile;
//  * tangents carry constant factors (below) so that no operand is scaled
//    before it is packed;
//  * the forward's layer 3 has the slots on the rows (A = y2, B = W3^T), so
//    its result is the next contraction's operand as it stands; only the four
//    blocks of y2 (the resnet copies) are re-laid, by an identity MFMA; hi
//    and lo parts share one 16x16x32 instruction;
//  * the backward adds up the gx of the two channels that carry one resnet
//    copy once an atom.
// Measured in one run, against all of G re-laid, every copy contracted and one
// workgroup per resident slot: 131,072 Cu atoms (12 tiles an atom) forward 2.26 ->
// 1.94 ms, backward 3.57 -> 3.10 (under the profiler 1.99 and 3.16).  Three
// wavefronts a SIMD for the backward and five for the forward gain nothing.
//
// Precision.  The split operands are tanh, not r (whose 1/2 would cancel in the
// sums; 32 FMAs a tile: forward 1.88 -> 1.94 ms, backward 3.05 -> 3.10, a step of
// 131,072 Cu atoms 7.68 -> 7.78), and tangents
// at one to two times their value (layers12); the resnet copies have an
// accumulator of their own.  Errors against 64 bits, 2-norms, weights exact in
// FP16 and scaled by 1 / 0.3 / 0.1 (nets of 32, 64, 128), r and quarter-scale
// tangents -> now: xyz 1.1 / 1.5 / 2.0e-7 -> 1.0 / 1.3 / 1.6e-7, dE/d em 2.8 / 3.5
// / 3.7e-7 -> 2.0 / 1.8 / 1.7e-7, its radial part 3.6 / 9.3 / 27e-7 -> 2.7 / 2.6 /
// 4.1e-7; without resnets (20, 30, 100) at 0.1: 5.4e-7, 1.0e-6, 1.8e-4 -> 3.0e-7,
// 3.0e-7, 2.2e-5.
// One wavefront an atom, or several where atoms are few (split_of), 16 slots a
// tile; lane (g = lane / 16, c = lane % 16).
#include <atomic>

#include "dpk_common.h"
#include "half16.h"
#include "embed_image.h"

namespace dpk {
namespace {

using namespace bfimg;
using E = h16::F16x2;
using h16::v2u;
using h16::v4f;
using h16::v4u;

constexpr int kMaxTypes = 16;
struct Block2 {  // type blocks of a row; nlist / pad as in embed.hip's BlockInfo
  int ntypes;
  int sec[kMaxTypes + 1];
  const int* nlist;
  const float* pad;
};

template <int RES2_, int RES3_, bool IDT_>
struct Net2 {
  static constexpr int RES2 = RES2_, RES3 = RES3_;
  static constexpr bool IDT = IDT_;
};

__device__ __forceinline__ v4u pack8(const float a[4], const float b[4]) {
  return v4u{E::pack2(a[0], a[1]), E::pack2(a[2], a[3]), E::pack2(b[0], b[1]),
             E::pack2(b[2], b[3])};
}
__device__ __forceinline__ v2u pack4(const float a[4]) {
  return v2u{E::pack2(a[0], a[1]), E::pack2(a[2], a[3])};
}
// lo = fp16(x - hi) of the values packed in hi: v_fma_mix_f32 twice and one
// conversion a pair (v_fma_mixlo / mixhi_f16 write the halves themselves but
// issue at half rate: 8 cycles each against 12 for the three)
__device__ __forceinline__ unsigned lo2(float a, float b, unsigned hi) {
  return E::pack2(h16::sub_f16_lo(a, hi), h16::sub_f16_hi(b, hi));
}
__device__ __forceinline__ v2u lo4(const float a[4], v2u hi) {
  return v2u{lo2(a[0], a[1], hi[0]), lo2(a[2], a[3], hi[1])};
}
__device__ __forceinline__ v4u lo8(const float a[4], const float b[4], v4u hi) {
  return v4u{lo2(a[0], a[1], hi[0]), lo2(a[2], a[3], hi[1]), lo2(b[0], b[1], hi[2]),
             lo2(b[2], b[3], hi[3])};
}
__device__ __forceinline__ v4u lds8(const unsigned char* p) {
  return *reinterpret_cast<const v4u*>(p);
}

constexpr v4f kZero4 = {0.f, 0.f, 0.f, 0.f};

// Forward of one net: the layer-3 bias of channel c four times over, after the
// net image in LDS (one 16-byte read starts a lane's accumulator).  Two nets
// with it leave room for two workgroups a CU instead of three (128,625 water
// atoms: 1.33 ms against 1.09 without).
constexpr int kBias4 = P3 * 16;

// Resident nets: copied to LDS once per (persistent) workgroup, w1 (which only
// the tangents use) as S1 w1.
template <bool BIAS4, int S1>
__device__ __forceinline__ void stage(unsigned char* dst, const unsigned char* src, int nnets) {
  constexpr int kOut = NET_BYTES + (BIAS4 ? kBias4 : 0);
  for (int k = 0; k < nnets; ++k) {
    const int4* s4 = reinterpret_cast<const int4*>(src + (size_t)k * NET_BYTES);
    int4* d4 = reinterpret_cast<int4*>(dst + k * kOut);
    for (int q = threadIdx.x; q < NET_BYTES / 16; q += blockDim.x) {
      int4 v = s4[q];
      if (S1 != 1 && q < (V_W1 + P1) / 4) {
        v.x = __float_as_int(S1 * __int_as_float(v.x));
        v.y = __float_as_int(S1 * __int_as_float(v.y));
        v.z = __float_as_int(S1 * __int_as_float(v.z));
        v.w = __float_as_int(S1 * __int_as_float(v.w));
      }
      d4[q] = v;
    }
    if constexpr (BIAS4) {
      const float* b = reinterpret_cast<const float*>(src + (size_t)k * NET_BYTES) + V_B3K;
      float* o = reinterpret_cast<float*>(dst + k * kOut + NET_BYTES);
      for (int q = threadIdx.x; q < 4 * P3; q += blockDim.x) o[q] = b[q >> 2];
    }
  }
  __syncthreads();
}

// Layers 1-2 for the lane's slot (channels 16 m + 4 g + i): y2 and, for the
// backward, t2 = (dy2/ds) K / 2.  With K = 2 log2 e the image's weights are
// K W; t1 = 8 w1 (r - r^2) = 2 dy1/ds goes through them as it is, and
// K W t1 (r2 - r2^2) = (K / 2) (dy2/ds without the resnet), to which the
// resnet adds (K / 4) t1.  The factor 2 of t1 sets the scale at which all
// tangents are split: 2, 1.4 and (k_bwd2) 1.04 of the derivatives, so that
// their low parts stay out of FP16's subnormals as far as those of the values
// do and no derivative below 62,900 overflows.  SCALED: w1 is 8 w1 already.
template <bool TANGENT, bool SCALED, class C>
__device__ __forceinline__ void layers12(const unsigned char* nb, float s, int g, int c,
                                         float y2[4][4], float t2[4][4]) {
  constexpr bool FOLD = C::RES2 == 2 && !C::IDT;  // y2 = (1 + y1) - 2 r2
  const float* vec = reinterpret_cast<const float*>(nb);
  float y1[2][4], e1[2][4], t1[2][4];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = 16 * m + 4 * g + i;
      const float r = tanh_r(__builtin_fmaf(s, vec[V_W1K + ch], vec[V_B1K + ch]));
      y1[m][i] = __builtin_fmaf(-2.0f, r, 1.0f);
      if (FOLD) e1[m][i] = __builtin_fmaf(-2.0f, r, 2.0f);
      if (TANGENT)
        t1[m][i] = __builtin_fmaf(-r, r, r) * (SCALED ? vec[V_W1 + ch] : 8.0f * vec[V_W1 + ch]);
    }
  const v4u B1 = pack8(y1[0], y1[1]), B1l = lo8(y1[0], y1[1], B1);
  v4u T1, T1l;
  if constexpr (TANGENT) {
    T1 = pack8(t1[0], t1[1]);
    T1l = lo8(t1[0], t1[1], T1);
    if constexpr (C::RES2 == 2) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) t1[m][i] *= K2L2E / 4;
    }
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const v4u a = lds8(nb + OFF_W2 + ((16 * m + c) * W2S + 8 * g) * 2);
    v4f acc = E::mfma32(a, B1, *reinterpret_cast<const v4f*>(vec + V_B2K + 16 * m + 4 * g));
    acc = E::mfma32(a, B1l, acc);
    v4f tac;
    if constexpr (TANGENT) {
      tac = E::mfma32(a, T1, kZero4);
      tac = E::mfma32(a, T1l, tac);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float idt = C::IDT ? vec[V_IDT2 + 16 * m + 4 * g + i] : 1.0f;
      const float r = tanh_r(acc[i]);
      if constexpr (FOLD) {
        y2[m][i] = __builtin_fmaf(-2.0f, r, e1[m & 1][i]);
      } else {
        const float t = __builtin_fmaf(-2.0f, r, 1.0f);
        y2[m][i] = (C::IDT ? t * idt : t) + (C::RES2 == 2 ? y1[m & 1][i] : 0.0f);
      }
      if constexpr (TANGENT) {
        const float w = C::IDT ? __builtin_fmaf(-r, r, r) * idt : __builtin_fmaf(-r, r, r);
        t2[m][i] = C::RES2 == 2 ? __builtin_fmaf(w, tac[i], t1[m & 1][i]) : w * tac[i];
      }
    }
  }
}

// tanh (with time steps: idt tanh) from r; idt2 = -2 idt
template <class C>
__device__ __forceinline__ float tanh3(float r, float idt, float idt2) {
  return C::IDT ? __builtin_fmaf(r, idt2, idt) : __builtin_fmaf(-2.0f, r, 1.0f);
}

template <bool RESIDENT, bool BIAS4, class C>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_fwd2(
    float* __restrict__ xyz, const float* __restrict__ em, const int* __restrict__ atype,
    const unsigned char* __restrict__ nets, const int* __restrict__ net_of,
    const int* __restrict__ ch_out, Block2 bi, int nnets, int d3, int natoms, int nnei, int lp) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  if (RESIDENT) stage<BIAS4, 1>(lds, nets, nnets);
  constexpr int kNet = NET_BYTES + (BIAS4 ? kBias4 : 0);
  const float id[4] = {c == 4 * g ? 1.f : 0.f, c == 4 * g + 1 ? 1.f : 0.f,
                       c == 4 * g + 2 ? 1.f : 0.f, c == 4 * g + 3 ? 1.f : 0.f};
  const v2u ident = pack4(id);
  // 1 << lp wavefronts an atom, each with every (1 << lp)-th tile
  const int apw = 4 >> lp, part = wave & ((1 << lp) - 1);
  for (int base = blockIdx.x * apw; base < natoms; base += gridDim.x * apw) {
    const int atom = base + (wave >> lp);
    const bool valid = atom < natoms;
    int ti = valid ? atype[atom] : 0;
    ti = ti < 0 ? 0 : ti;
    const float* e = em + (size_t)(valid ? atom : 0) * nnei * 4;
    // xyz nnei = accY + acc: sums over slots of R y2 and R tanh.  Rows 0-3 are
    // R's hi parts, rows 4-7 its lo parts (added once an atom).
    v4f acc[8], accY[4];
#pragma unroll
    for (int m = 0; m < 8; ++m) acc[m] = kZero4;
#pragma unroll
    for (int m = 0; m < 4; ++m) accY[m] = kZero4;
    int tix = 0;  // tiles of the blocks before this one
    for (int t = 0; t < bi.ntypes; ++t) {
      const int net = net_of[ti * bi.ntypes + t];
      const unsigned char* nb = RESIDENT ? lds + (size_t)net * kNet
                                         : nets + (size_t)net * NET_BYTES;
      const float* vec = reinterpret_cast<const float*>(nb);
      const int b0 = bi.sec[t];
      int b1 = valid ? bi.sec[t + 1] : b0;
      if (bi.nlist != nullptr && valid) {
        b1 = block_end(bi.nlist + (size_t)atom * nnei, b0, b1, lane);
        // a virtual centre's rows are zero, not padding rows
        if (bi.pad != nullptr && b1 < bi.sec[t + 1] && part == 0 && g == 0 && atype[atom] >= 0) {
          const float* pt = bi.pad + ((size_t)ti * nnei + b1) * 4 * P3;
#pragma unroll
          for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][i] += pt[i * P3 + 16 * m + c];
        }
      }
      const int first = (part - tix) & ((1 << lp) - 1);
      tix += (b1 - b0 + 15) >> 4;
      for (int s0 = b0 + 16 * first; s0 < b1; s0 += 16 << lp) {
        // weights are re-read from LDS every tile rather than hoisted into
        // registers across the loop (that would halve the occupancy)
        asm volatile("" ::: "memory");
        const int slot = s0 + c;
        const float s = slot < b1 ? e[slot * 4] : 0.f;
        float rr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int sl = s0 + 4 * g + i;
          rr[i] = (c < 8 && sl < b1) ? e[sl * 4 + (c & 3)] : 0.f;
        }
        v2u rT = pack4(rr);
        const v2u rl = lo4(rr, rT);
        if (c >= 4) rT = rl;
        const v4u RT = {rT[0], rT[1], rT[0], rT[1]};  // against (hi, lo) of the same slots
        float y2[4][4], t2[4][4];
        layers12<false, false, C>(nb, s, g, c, y2, t2);
        const v4u B2[2] = {pack8(y2[0], y2[1]), pack8(y2[2], y2[3])};
        const v4u B2l[2] = {lo8(y2[0], y2[1], B2[0]), lo8(y2[2], y2[3], B2[1])};
        if constexpr (C::RES3 == 2) {
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const int p = m >> 1, h = 2 * (m & 1);
            const v4f a = E::mfma16(v2u{B2[p][h], B2[p][h + 1]}, ident, kZero4);
            const v4f b = E::mfma16(v2u{B2l[p][h], B2l[p][h + 1]}, ident, kZero4);
            accY[m] = E::mfma32(RT, v4u{E::pack2(a[0], a[1]), E::pack2(a[2], a[3]),
                                        E::pack2(b[0], b[1]), E::pack2(b[2], b[3])},
                                accY[m]);  // exact: a and b hold FP16 values
          }
        }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const unsigned char* row = nb + OFF_W3 + ((16 * m + c) * W3S + 8 * g) * 2;
          const v4u a0 = lds8(row), a1 = lds8(row + 64);
          v4f u;
          if constexpr (BIAS4) {
            u = *reinterpret_cast<const v4f*>(nb + NET_BYTES + (16 * m + c) * 16);
          } else {
            const float b = vec[V_B3K + 16 * m + c];
            u = v4f{b, b, b, b};
          }
          u = E::mfma32(B2[0], a0, u);
          u = E::mfma32(B2[1], a1, u);
          u = E::mfma32(B2l[0], a0, u);
          u = E::mfma32(B2l[1], a1, u);  // row 4 g + i = slot, column c = channel
          const float idt = C::IDT ? vec[V_IDT3 + 16 * m + c] : 1.0f, idt2 = -2.0f * idt;
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = tanh3<C>(tanh_r(u[i]), idt, idt2);
          const v2u vh = pack4(v), vl = lo4(v, vh);
          acc[m] = E::mfma32(RT, v4u{vh[0], vh[1], vl[0], vl[1]}, acc[m]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    float* part_lds = reinterpret_cast<float*>(lds + (RESIDENT ? nnets * kNet : 0));
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = acc[m][i] + accY[m & 3][i];
        acc[m][i] = v + __shfl_xor(v, 16, 64);
      }
    if (lp > 0) {  // the other wavefronts' sums, in their order
      __syncthreads();
      if (g == 0)
#pragma unroll
        for (int m = 0; m < 8; ++m)
          *reinterpret_cast<v4f*>(part_lds + ((wave * 8 + m) * 16 + c) * 4) = acc[m];
      __syncthreads();
      if (part == 0 && g == 0)
        for (int w = wave + 1; w < wave + (1 << lp); ++w)
#pragma unroll
          for (int m = 0; m < 8; ++m)
            acc[m] += *reinterpret_cast<const v4f*>(part_lds + ((w * 8 + m) * 16 + c) * 4);
    }
    const float inv = 1.0f / (float)nnei;
    float* o = xyz + (size_t)(valid ? atom : 0) * 4 * d3;
    if (valid && part == 0 && g == 0)
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int tc = ch_out[16 * m + c];
        if (tc >= 0)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i * d3 + tc] = acc[m][i] * inv;
      }
  }
}

template <bool RESIDENT, class C>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_bwd2(
    float* __restrict__ net_deriv, const float* __restrict__ em, const float* __restrict__ gxyz,
    const int* __restrict__ atype, const unsigned char* __restrict__ nets,
    const int* __restrict__ net_of, const int* __restrict__ ch_out, Block2 bi, int nnets, int d3,
    int natoms, int nnei, int lp) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  if (RESIDENT) stage<false, 8>(lds, nets, nnets);
  // 1 << lp wavefronts an atom, each with every (1 << lp)-th tile
  const int apw = 4 >> lp, part = wave & ((1 << lp) - 1);
  for (int base = blockIdx.x * apw; base < natoms; base += gridDim.x * apw) {
    const int atom = base + (wave >> lp);
    const bool valid = atom < natoms;
    int ti = valid ? atype[atom] : 0;
    ti = ti < 0 ? 0 : ti;
    const size_t aoff = (size_t)(valid ? atom : 0);
    const float* e = em + aoff * nnei * 4;
    float* nd = net_deriv + aoff * nnei * 4;
    // A operand gx[c][ch] / nnei for channel-block pairs, scaled by a power of
    // two q chosen from the atom's largest |gx| so that the 16-bit operands
    // keep their full significand (dE/dxyz / nnei can sit in FP16's subnormal
    // range); the results are multiplied by 1 / q.  Rows 0-3 the components,
    // rows 4-7 their lo parts: one MFMA forms gx_hi B and gx_lo B.
    float amax = 0.f;
    if (valid)  // the atom's 4 d3 values, read by the whole wavefront
      for (int q0 = lane; q0 < 4 * d3; q0 += 64) amax = fmaxf(amax, fabsf(gxyz[aoff * 4 * d3 + q0]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    // every lane holds the maximum: keep q and 1/q in scalar registers
    amax = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(amax)));
    const float q = h16::pow2_scale(amax / (float)nnei);
    const float qin = q / (float)nnei;
    const float unq = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(1.0f / q)));
    const int comp = c & 3;
    v4u gxa[4], gxc[2];  // gxc: summed over the channels of one resnet copy
    float cl[2][4], ch[2][4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      float lo[4], hi[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[i] = hi[i] = 0.f;
        if (c < 8 && valid) {
          const int t0 = ch_out[32 * p + 4 * g + i], t1 = ch_out[32 * p + 16 + 4 * g + i];
          if (t0 >= 0) lo[i] = gxyz[aoff * 4 * d3 + comp * d3 + t0] * qin;
          if (t1 >= 0) hi[i] = gxyz[aoff * 4 * d3 + comp * d3 + t1] * qin;
        }
      }
      gxa[p] = pack8(lo, hi);
      const v4u l = lo8(lo, hi, gxa[p]);
      if (c >= 4) gxa[p] = l;
      if constexpr (C::RES3 == 2) {  // channels 32 p.. of p and p + 2 carry the same copies
        const int k = p & 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          cl[k][i] = p < 2 ? lo[i] : cl[k][i] + lo[i];
          ch[k][i] = p < 2 ? hi[i] : ch[k][i] + hi[i];
        }
        if (p >= 2) {
          gxc[k] = pack8(cl[k], ch[k]);
          const v4u l2 = lo8(cl[k], ch[k], gxc[k]);
          if (c >= 4) gxc[k] = l2;
        }
      }
    }
    int tix = 0;  // tiles of the blocks before this one
    for (int t = 0; t < bi.ntypes; ++t) {
      const unsigned char* nb =
          (RESIDENT ? lds : nets) + (size_t)net_of[ti * bi.ntypes + t] * NET_BYTES;
      const float* vec = reinterpret_cast<const float*>(nb);
      const int b0 = bi.sec[t];
      int b1 = valid ? bi.sec[t + 1] : b0;
      if (bi.nlist != nullptr && valid) {
        // slots after the last real neighbour move no atom: dE/d em = 0
        b1 = block_end(bi.nlist + (size_t)atom * nnei, b0, b1, lane);
        for (int z = b1 + lane + 64 * part; z < bi.sec[t + 1]; z += 64 << lp)
          *reinterpret_cast<float4*>(nd + z * 4) = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      const int first = (part - tix) & ((1 << lp) - 1);
      tix += (b1 - b0 + 15) >> 4;
      for (int s0 = b0 + 16 * first; s0 < b1; s0 += 16 << lp) {
        asm volatile("" ::: "memory");
        const int slot = s0 + c;
        const float s = slot < b1 ? e[slot * 4] : 0.f;
        float y2[4][4], t2[4][4];
        layers12<true, RESIDENT, C>(nb, s, g, c, y2, t2);
        const v4u B2[2] = {pack8(y2[0], y2[1]), pack8(y2[2], y2[3])};
        const v4u B2l[2] = {lo8(y2[0], y2[1], B2[0]), lo8(y2[2], y2[3], B2[1])};
        const v4u T2[2] = {pack8(t2[0], t2[1]), pack8(t2[2], t2[3])};
        const v4u T2l[2] = {lo8(t2[0], t2[1], T2[0]), lo8(t2[2], t2[3], T2[1])};
        // dR[comp][slot c] = gx y2 + gx tanh;
        // dE/ds = sum_comp R[comp] (8 / K^2) Mx[comp], Mx = gx (K W3 t2) (r3 - r3^2)
        //         + (K / 4) gx t2 (the resnet copies)
        v4f dR = kZero4, Mx = kZero4, dRc = kZero4;
        if constexpr (C::RES3 == 2) {
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            dRc = E::mfma32(gxc[p], B2[p], dRc);
            Mx = E::mfma32(gxc[p], T2[p], Mx);
            dRc = E::mfma32(gxc[p], B2l[p], dRc);
            Mx = E::mfma32(gxc[p], T2l[p], Mx);
          }
          Mx *= K2L2E / 4;
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          float v[2][4], dv[2][4];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int m = 2 * p + h;
            const unsigned char* row = nb + OFF_W3 + ((16 * m + c) * W3S + 8 * g) * 2;
            const v4u a0 = lds8(row), a1 = lds8(row + 64);
            v4f u = E::mfma32(a0, B2[0], *reinterpret_cast<const v4f*>(vec + V_B3K + 16 * m + 4 * g));
            v4f tu = E::mfma32(a0, T2[0], kZero4);
            u = E::mfma32(a1, B2[1], u);
            tu = E::mfma32(a1, T2[1], tu);
            u = E::mfma32(a0, B2l[0], u);
            tu = E::mfma32(a0, T2l[0], tu);
            u = E::mfma32(a1, B2l[1], u);
            tu = E::mfma32(a1, T2l[1], tu);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float idt = C::IDT ? vec[V_IDT3 + 16 * m + 4 * g + i] : 1.0f;
              const float r = tanh_r(u[i]);
              v[h][i] = tanh3<C>(r, idt, -2.0f * idt);
              const float d = __builtin_fmaf(-r, r, r) * tu[i];
              dv[h][i] = C::IDT ? d * idt : d;
            }
          }
          const v4u vh = pack8(v[0], v[1]), dh = pack8(dv[0], dv[1]);
          dR = E::mfma32(gxa[p], vh, dR);
          Mx = E::mfma32(gxa[p], dh, Mx);
          dR = E::mfma32(gxa[p], lo8(v[0], v[1], vh), dR);
          Mx = E::mfma32(gxa[p], lo8(dv[0], dv[1], dh), Mx);
          __builtin_amdgcn_sched_barrier(0);
        }
        dR += dRc;
        // lanes g = 1 hold rows 4-7 (the gx_lo products): fold them into ds
        // and dR of the lanes g = 0 (the components are the same)
        float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
        if (g < 2 && slot < b1) r = *reinterpret_cast<const float4*>(e + slot * 4);
        float ds = (8.0f / (K2L2E * K2L2E)) *
                   (r.x * Mx[0] + r.y * Mx[1] + r.z * Mx[2] + r.w * Mx[3]);
        ds += __shfl_xor(ds, 16, 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) dR[i] += __shfl_xor(dR[i], 16, 64);
        if (g == 0 && slot < b1)
          *reinterpret_cast<float4*>(nd + slot * 4) =
              make_float4((dR[0] + ds) * unq, dR[1] * unq, dR[2] * unq, dR[3] * unq);
      }
    }
  }
}

constexpr int kResidentMaxBytes = 64 * 1024;
constexpr int kPartSums = 4 * 8 * 16 * 16;  // forward, split atoms: four wavefronts' sums

// Workgroups of a persistent grid per resident slot: with one, a slow XCD or a
// ragged last round holds the launch; with eight, finished slots take what is
// left, and a net is still copied to LDS once for several groups of atoms.
// Forward + backward us (before tanh took r's place: 1-2% less than now) with 1 /
// 4 / 8 a slot, or one a group: Cu (one net)
// 8,788 atoms 356 / 333 / 331 / 332, 20,000 782 / 705 / 704 / 705, 131,072 5,227 /
// 4,703 / 4,748 / 4,658; water (two nets) 8,788 275 / 275 / 276 / 274, 49,000 1,468 /
// 1,418 / 1,399 / 1,435, 131,072 3,974 / 3,828 / 3,792 / 3,917.
constexpr int kGridRounds = 8;

// Wavefronts an atom (log2).  One wavefront alone works off its tiles at its
// own latency, so few atoms leave the chip idle: four wavefronts an atom up to
// two atoms a CU, two up to six, as long as each has a tile.  Forward +
// backward us with 1 / 2 / 4 wavefronts an atom (Cu rows of 12 tiles): 500
// atoms 75 / 48 / 41, 1,000 79 / 62 / 61, 1,500 103 / 81 / 80, 2,048 106 / 101 /
// 110, 4,096 172 / 182 / 200; water rows of 8: 500 56 / 38 / 33, 1,000 59 / 48 /
// 53, 1,500 75 / 65 / 71, 2,048 78 / 79 / 89.
inline int split_of(int natoms, int nnei, int ncu) {
  const int lp = natoms <= 2 * ncu ? 2 : natoms <= 6 * ncu ? 1 : 0;
  return nnei > 32 ? lp : nnei > 16 && lp > 0 ? 1 : 0;
}

template <bool RESIDENT, class C>
int launch2(bool fwd, void* out, const void* em, const void* gx, const int* atype,
            const void* image, const int* net_of, const int* ch_out, const Block2& bi, int nnets,
            int d3, int natoms, int nnei, hipStream_t st) {
  // resident workgroups per device, cached per (device, direction, nnets, split)
  constexpr int kDev = 64, kRes = kResidentMaxBytes / NET_BYTES + 1;
  static std::atomic<int> cache[kDev][2][kRes][2];
  int dev = 0, ncu = 0;
  const int rc = device_cus(&dev, &ncu);
  if (rc != DPK_OK) return rc;
  DPK_REQUIRE(dev >= 0 && dev < kDev, DPK_ERR_ARG, "embed: device %d out of range", dev);
  const int lp = split_of(natoms, nnei, ncu);
  const bool bias4 = RESIDENT && fwd && nnets == 1;
  const size_t lds = (RESIDENT ? (size_t)nnets * NET_BYTES + (bias4 ? kBias4 : 0) : 0) +
                     (fwd && lp > 0 ? kPartSums : 0);
  const auto kfwd = bias4 ? k_fwd2<RESIDENT, RESIDENT, C> : k_fwd2<RESIDENT, false, C>;
  std::atomic<int>& kept = cache[dev][fwd ? 0 : 1][RESIDENT ? nnets : 0][lp > 0];
  int slots = kept.load(std::memory_order_relaxed);
  if (slots == 0) {
    int per_cu = 0;
    if (fwd)
      DPK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfwd, 256, lds));
    else
      DPK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bwd2<RESIDENT, C>, 256, lds));
    slots = ncu * (per_cu < 1 ? 1 : per_cu);
    kept.store(slots, std::memory_order_relaxed);
  }
  const int groups = cdiv(natoms, 4 >> lp);
  const int pct = tune(DPK_TUNE_EMBED_GRID_PCT);
  const long want = pct == 0 ? groups : ((long)kGridRounds * slots * pct + 99) / 100;
  const int grid = groups < want ? groups : (int)(want > 0 ? want : 1);
  const unsigned char* img = static_cast<const unsigned char*>(image);
  if (fwd)
    hipLaunchKernelGGL(kfwd, dim3(grid), dim3(256), lds, st,
                       static_cast<float*>(out), static_cast<const float*>(em), atype, img,
                       net_of, ch_out, bi, nnets, d3, natoms, nnei, lp);
  else
    hipLaunchKernelGGL((k_bwd2<RESIDENT, C>), dim3(grid), dim3(256), lds, st,
                       static_cast<float*>(out), static_cast<const float*>(em),
                       static_cast<const float*>(gx), atype, img, net_of, ch_out, bi, nnets, d3,
                       natoms, nnei, lp);
  DPK_LAUNCHED();
  return DPK_OK;
}

}  // namespace

int embed_f16x2(bool fwd, void* out, const void* em, const void* gx, const int* atype,
                const void* image, const int* net_of, const int* ch_out, int ntypes, int nnets,
                int res2, int res3, int has_idt, int d3, const int* sec_host, int natoms,
                int nnei, const int* nlist, const float* pad, hipStream_t st) {
  DPK_REQUIRE(ntypes > 0 && ntypes <= kMaxTypes, DPK_ERR_ARG, "embed: ntypes=%d", ntypes);
  Block2 bi;
  bi.ntypes = ntypes;
  bi.nlist = nlist;
  bi.pad = pad;
  for (int t = 0; t <= ntypes; ++t) bi.sec[t] = sec_host[t];
  const bool resident = (size_t)nnets * NET_BYTES <= (size_t)kResidentMaxBytes;
#define DPK_F16X2(R2, R3, I)                                                                      \
  return resident                                                                                 \
             ? launch2<true, Net2<R2, R3, I>>(fwd, out, em, gx, atype, image, net_of, ch_out, bi, \
                                              nnets, d3, natoms, nnei, st)                        \
             : launch2<false, Net2<R2, R3, I>>(fwd, out, em, gx, atype, image, net_of, ch_out,    \
                                               bi, nnets, d3, natoms, nnei, st)
  switch ((res2 ? 4 : 0) + (res3 ? 2 : 0) + (has_idt ? 1 : 0)) {
    case 0: DPK_F16X2(0, 0, false);
    case 1: DPK_F16X2(0, 0, true);
    case 2: DPK_F16X2(0, 2, false);
    case 3: DPK_F16X2(0, 2, true);
    case 4: DPK_F16X2(2, 0, false);
    case 5: DPK_F16X2(2, 0, true);
    case 6: DPK_F16X2(2, 2, false);
    default: DPK_F16X2(2, 2, true);
  }
#undef DPK_F16X2
}

}  // namespace dpk
