// Device helpers shared by the HIP translation units and by the kernels the
// library compiles at run time (hipRTC): MFMA tiles, accumulator layout,
// float32 tanh, row sums, integer powers.  Self-contained (no includes), so
// that its text can be compiled by hipRTC as it is.
#ifndef TDX_DEV_H
#define TDX_DEV_H

namespace tdx {

typedef float f4_t __attribute__((ext_vector_type(4)));
typedef double d4_t __attribute__((ext_vector_type(4)));

template <typename T> struct V4;
template <> struct V4<float> { typedef f4_t type; };
template <> struct V4<double> { typedef d4_t type; };

__device__ __forceinline__ f4_t mma16(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ d4_t mma16(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// float32 products on the bf16 matrix units.  A float32 value is split into
// three bf16 pieces, x = h + m + l (each the rounding of what is left: 24
// significant bits, exact above 2^-110), and a product of two values is the
// six piece products that reach 2^-24 of it, m m' + h l' + l h' first, then
// h m' + m h', then h h', summed in the float32 accumulator.  What bounds it:
// a 16x16x32 bf16 MFMA takes 16 cycles and VALU work of other wavefronts runs
// beside it; a float32 16x16x4 takes 32 and shares the VALU's multipliers, so
// 16x16x32 in float32 costs 256 cycles that add to the VALU's, in six bf16
// products 96 that mostly do not.  Measured against 64 bits, relative error
// of sums over K = 32: 3.6e-8 (float32 MFMA 1.03e-7), K = 128: 6e-8 (2.0e-7).
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef unsigned u4_t __attribute__((ext_vector_type(4)));
typedef unsigned u2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
typedef float f16_t __attribute__((ext_vector_type(16)));

// Eight float32 values (one lane's k-slots of a 32-deep product) in pieces.
struct Bf3 {
  u4_t h, m, l;
};

// The pieces of NP pairs of values (2k in the low half, 2k + 1 in the high).
// The remainder x - h is a dot product of the packed pieces with (-1, 0) or
// (0, -1) on top of x: exact, and one instruction where unpacking and
// subtracting are two.  Stage by stage over the pairs, so that the dot
// products' latencies overlap.  An infinite or NaN value, or one that rounds to
// infinity, makes its remainder, and its pair partner's, NaN (image_pair takes
// such weights out first).
template <int NP>
__device__ __forceinline__ void bf3_pairs(const float (&x)[2 * NP], unsigned (&h)[NP],
                                          unsigned (&m)[NP], unsigned (&l)[NP]) {
#if defined(__AMDGCN__)
  typedef float f2_t __attribute__((ext_vector_type(2)));
  // in registers: as a packed literal it would be read as an inline constant
  unsigned e0 = 0x0000BF80u, e1 = 0xBF800000u;
  asm("" : "+v"(e0), "+v"(e1));
  const bf2_t n0 = __builtin_bit_cast(bf2_t, e0), n1 = __builtin_bit_cast(bf2_t, e1);
  float r[2 * NP];
  auto round = [&](const float (&v)[2 * NP], unsigned (&p)[NP]) {
#pragma unroll
    for (int k = 0; k < NP; ++k)
      p[k] = __builtin_bit_cast(unsigned,
                                __builtin_convertvector(f2_t{v[2 * k], v[2 * k + 1]}, bf2_t));
  };
  auto rest = [&](const float (&v)[2 * NP], const unsigned (&p)[NP]) {
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const bf2_t b = __builtin_bit_cast(bf2_t, p[k]);
      r[2 * k] = __builtin_amdgcn_fdot2_f32_bf16(b, n0, v[2 * k], false);
      r[2 * k + 1] = __builtin_amdgcn_fdot2_f32_bf16(b, n1, v[2 * k + 1], false);
    }
  };
  round(x, h);
  rest(x, h);
  round(r, m);
  rest(r, m);
  round(r, l);
#else
  for (int k = 0; k < NP; ++k) h[k] = m[k] = l[k] = 0;  // device code only
#endif
}
__device__ __forceinline__ Bf3 bf3_split(f4_t a, f4_t b) {
  const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  unsigned h[4], m[4], l[4];
  bf3_pairs<4>(x, h, m, l);
  return Bf3{u4_t{h[0], h[1], h[2], h[3]}, u4_t{m[0], m[1], m[2], m[3]},
             u4_t{l[0], l[1], l[2], l[3]}};
}
// Four values in the low k-slots, zeros in the others.
__device__ __forceinline__ Bf3 bf3_split(f4_t a) {
  const float x[4] = {a[0], a[1], a[2], a[3]};
  unsigned h[2], m[2], l[2];
  bf3_pairs<2>(x, h, m, l);
  return Bf3{u4_t{h[0], h[1], 0, 0}, u4_t{m[0], m[1], 0, 0}, u4_t{l[0], l[1], 0, 0}};
}
__device__ __forceinline__ f4_t mma_bf(u4_t a, u4_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a),
                                                 __builtin_bit_cast(bf8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f16_t mma_bf(u4_t a, u4_t b, f16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8_t, a),
                                                 __builtin_bit_cast(bf8_t, b), c, 0, 0, 0);
}
// The five small products of a 16x16x32 (or 32x32x16) step.  They need an
// accumulator of their own: the unit aligns its addends to the largest and
// cuts off below (towards minus infinity), so small products added to a
// large accumulator leave a bias (1.2e-9 of the sum of magnitudes per step,
// which long sums of cancelling terms pile up) where the leading ones, added
// alone, leave none.
template <typename V>
__device__ __forceinline__ V mma3_small(const Bf3 &a, const Bf3 &b, V c) {
  c = mma_bf(a.l, b.h, c);
  c = mma_bf(a.h, b.l, c);
  c = mma_bf(a.m, b.m, c);
  c = mma_bf(a.m, b.h, c);
  return mma_bf(a.h, b.m, c);
}
// c + a b for one step of a long sum: the small products from zero, added
// after.  Error against 64 bits over K = 16384, of the sum of magnitudes:
// 1.0e-8 (float32 MFMA 2.5e-8; all six in one accumulator 2.3e-8 with a bias
// of 0.9e-8), with cancelling terms 0.9e-9 (2.2e-9; 2.3e-9).
template <typename V>
__device__ __forceinline__ V mma3(const Bf3 &a, const Bf3 &b, V c) {
  const V s = mma3_small(a, b, V{});
  return mma_bf(a.h, b.h, c) + s;
}

// c + a[0] b[0] + a[1] b[1]: two steps, one sum of small products.
template <typename V>
__device__ __forceinline__ V mma3_pair(const Bf3 (&a)[2], const Bf3 (&b)[2], V c) {
  const V s = mma3_small(a[1], b[1], mma3_small(a[0], b[0], V{}));
  return mma_bf(a[1].h, b[1].h, mma_bf(a[0].h, b[0].h, c)) + s;
}

// Row of the 16x16 MFMA accumulator held in register i of a lane in
// quarter q (= lane / 16); the column is lane % 16.  The f32 and f64
// 16x16x4 instructions place rows differently.
template <typename T> __device__ __forceinline__ int crow(int q, int i);
template <> __device__ __forceinline__ int crow<float>(int q, int i) { return 4 * q + i; }
template <> __device__ __forceinline__ int crow<double>(int q, int i) { return q + 4 * i; }

// tanh in float32 without branches: for |x| < 0.625 an odd polynomial
// x + x^3 q(x^2) (q fitted by weighted least squares to (tanh x - x)/x^3,
// max error 0.8 ulp on that interval in float32 Horner form); otherwise
// 1 - 2/(1 + 2^(2|x| log2 e)) with the sign restored (about 2 ulp; exp2
// overflows to inf for large |x| and gives exactly 1).
__device__ __forceinline__ float dtanh(float x) {
  const float ax = fabsf(x);
  const float x2 = x * x;
  float p = 0.002142803743481636f;
  p = fmaf(p, x2, -0.008177093230187893f);
  p = fmaf(p, x2, 0.021700501441955566f);
  p = fmaf(p, x2, -0.05394670367240906f);
  p = fmaf(p, x2, 0.1333320587873459f);
  p = fmaf(p, x2, -0.3333333134651184f);
  const float small = fmaf(x * x2, p, x);
  const float e = __builtin_amdgcn_exp2f(ax * 2.8853900817779268f);
  const float r = __builtin_amdgcn_rcpf(1.0f + e);
  const float large = copysignf(fmaf(-2.0f, r, 1.0f), x);
  return ax < 0.625f ? small : large;
}
__device__ __forceinline__ double dtanh(double x) { return tanh(x); }

// Sum over the 16 lanes of a row of the wavefront (lanes 16k .. 16k+15);
// every lane of the row receives the sum.  Float: DPP lane swizzles
// (quad xor 1, quad xor 2, half-row mirror, row mirror) fused into adds.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float rowsum16(float v) {
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x141>(v);
  v += dpp_f<0x140>(v);
  return v;
}
__device__ __forceinline__ double rowsum16(double v) {
  v += __shfl_xor(v, 1);
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 4);
  v += __shfl_xor(v, 8);
  return v;
}
__device__ __forceinline__ float dpow(float x, float p) { return powf(x, p); }
__device__ __forceinline__ double dpow(double x, double p) { return pow(x, p); }

// x ** p for integer p with the special cases torch uses for a scalar
// exponent (copy for 1, x*x for 2, x*x*x for 3, reciprocals for -1/-2).
template <typename T>
__device__ __forceinline__ T ipow(T x, int p) {
  switch (p) {
    case 0: return T(1);
    case 1: return x;
    case 2: return x * x;
    case 3: return (x * x) * x;
    case -1: return T(1) / x;
    case -2: return T(1) / (x * x);
    default: return dpow(x, T(p));
  }
}


__device__ __forceinline__ float dsin(float x) { return sinf(x); }
__device__ __forceinline__ double dsin(double x) { return sin(x); }
__device__ __forceinline__ float dcos(float x) { return cosf(x); }
__device__ __forceinline__ double dcos(double x) { return cos(x); }
__device__ __forceinline__ float dexp(float x) { return expf(x); }
__device__ __forceinline__ double dexp(double x) { return exp(x); }
__device__ __forceinline__ float dlog(float x) { return logf(x); }
__device__ __forceinline__ double dlog(double x) { return log(x); }
__device__ __forceinline__ float dsqrt(float x) { return sqrtf(x); }
__device__ __forceinline__ double dsqrt(double x) { return sqrt(x); }

// Table access by word index: records (i) and real values (r).
template <typename T>
struct PtrTab {
  const int32_t *I;
  const T *R;
  __device__ __forceinline__ int i(int k) const { return I[k]; }
  __device__ __forceinline__ T r(int k) const { return R[k]; }
};

// A callable power of a residual program (the reference applies it to the
// term's running product, tedeous/derivative.py:54-55, 128-129, 317-318):
// the chain of one-argument operations at word ref of g's records -- n,
// then n (op, arg) pairs, op TDX_AD_OP_*, arg a real's index or the integer
// power -- applied to x in order; v its value, d its derivative (dual
// numbers).
template <typename T, typename G>
__device__ __forceinline__ void chain_apply(const G &g, int ref, T x, T &v, T &d) {
  const int n = g.i(ref);
  v = x;
  d = T(1);
  for (int k = 0; k < n; ++k) {
    const int op = g.i(ref + 1 + 2 * k), arg = g.i(ref + 2 + 2 * k);
    switch (op) {
      case TDX_AD_OP_ADD: v = v + g.r(arg); break;
      case TDX_AD_OP_SUB: v = v - g.r(arg); break;
      case TDX_AD_OP_RSUB: v = g.r(arg) - v; d = -d; break;
      case TDX_AD_OP_MUL: v = g.r(arg) * v; d = g.r(arg) * d; break;
      case TDX_AD_OP_DIV: v = v / g.r(arg); d = d / g.r(arg); break;
      case TDX_AD_OP_RDIV: {
        const T nv = g.r(arg) / v;
        d = -(nv / v) * d;
        v = nv;
      } break;
      case TDX_AD_OP_POWI:
        d = (arg == 0 ? T(0) : T(arg) * ipow(v, arg - 1)) * d;
        v = ipow(v, arg);
        break;
      case TDX_AD_OP_POWR: {
        const T p = g.r(arg);
        d = (p * dpow(v, p - T(1))) * d;
        v = dpow(v, p);
      } break;
      case TDX_AD_OP_NEG: v = -v; d = -d; break;
      case TDX_AD_OP_SIN: d = dcos(v) * d; v = dsin(v); break;
      case TDX_AD_OP_COS: d = -dsin(v) * d; v = dcos(v); break;
      case TDX_AD_OP_EXP: v = dexp(v); d = v * d; break;
      case TDX_AD_OP_LOG: d = d / v; v = dlog(v); break;
      case TDX_AD_OP_TANH: v = dtanh(v); d = (T(1) - v * v) * d; break;
      case TDX_AD_OP_SQRT: v = dsqrt(v); d = d / (T(2) * v); break;
      default: break;
    }
  }
}
}  // namespace tdx

#endif  // TDX_DEV_H
