// Matrix-core (MFMA) GEMMs for the STE / LRE backward of the LUT conv.
//
// Both estimators differentiate y[n,o,l] = sum_k f(x_nkl, w_ok) as a dense
// product of mapped operands (STE: the quantized values, LRE: 256-entry slope
// tables indexed by the other operand's LUT index):
//   col[n,k,l] = sum_o go[n,o,l] * Tx[wi(o,k)]          (backward-data, then fold)
//   gw[o,k]    = sum_{n,l} go[n,o,l] * Tw[xi(n,k,l)]     (backward-weight)
// with xi read straight from the saved quantized image (implicit im2col;
// out-of-image taps take index pad_index, so LRE's Tw[128] border rule
// holds).  Reference: csrc/claude/bgemm_lre_backward_claude.cu:443-524 (cuBLAS
// SGEMMs) and nn/bgemm_int8.py:184-207,277-290 (cuDNN convolution_backward).
//
// Two engines over BM x BN block tiles (64 or 128 each), 32-deep k-tiles and
// 256 threads as 2 x 2 waves:
// - split-bf16 (the layer paths): fp32 operands split exactly into three
//   bf16 parts and multiplied on v_mfma_f32_16x16x32_bf16 as the six part
//   products of order <= 2 (three when a table is bf16 already); see the
//   "split-bf16 operand planes" section below.  Backward-weight, and for
//   atx_conv_bwd_data the column GEMM (its A operand from bf16 weight planes
//   prepared per call) and the tap GEMM (both operands from planes, the image
//   gradient without columns).
// - fp32 (v_mfma_f32_16x16x4f32, plain fp32 products): the backward-data
//   GEMM of atx_conv_bwd_data_col (no workspace for the planes) and layers
//   whose go spans exceed the split path's 32-bit buffer offsets.  The
//   256-entry table lives in LDS; operand tiles go HBM -> registers while
//   the previous tile is multiplied, then through the table into a second
//   LDS buffer ([BK][B + 16], bank 16k + i: conflict-free MFMA reads); one
//   barrier per k-tile.
// The backward-data GEMMs fold the batch into their columns (c = n*L + l),
// so small images waste no tile width.

#include "atx_internal.h"
#include "atx_tiles.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace atx {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int BK = 32;          // contraction depth of one k-tile
constexpr int GT = 256;         // threads per block (2 x 2 waves)

template <int B> struct KMajor {          // [BK][B + 16]: bank(k, i) = 16k + i
  static constexpr int LD = B + 16;
  static constexpr int SIZE = BK * LD;
  __device__ static int at(int m, int k) { return k * LD + m; }
};

// ------------------------------------------------ split-bf16 operand planes
// gfx950's bf16 matrix cores (v_mfma_f32_16x16x32_bf16: a 16 x 16 x 32 block
// in 16 cycles) do 16 times the products per cycle of its fp32 ones
// (v_mfma_f32_16x16x4f32: 16 x 16 x 4 in 32).  An fp32 value a splits exactly
// into three bf16 parts a = ah + am + al by truncation: ah is a with its low
// 16 bits cleared, r = a - ah is exact in fp32 with at most 16 significant
// bits, am is r truncated the same way and al = r - am has at most 8.  The
// product a*b is taken as the six part products of order <= 2,
//   ah*bh + ah*bm + am*bh + ah*bl + am*bm + al*bh,
// each exact in fp32 (8 x 8 significant bits), summed in fp32.  The dropped
// products am*bl + al*bm + al*bl stay below 2^-20 |a b| (|am| < 2^-7 |a|,
// |al| < 2^-14 |a|), on average about 2^-23 |a b|, the size of an fp32
// product's own rounding.  An operand whose values are bf16 already (the
// STE's quantized integers, or any table whose m and l parts are all zero)
// has only its h part: three products, each exact, instead of six.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Which part products a tile multiply takes.
enum PartProducts { PROD6 = 0, A_EXACT = 1, B_EXACT = 2 };

// Operand tile of B rows x BK contraction elements as three bf16 planes
// (h, m, l) of B x 64 bytes.  Row r is stored at s = r ^ ((r >> 2) & 1) and
// its four 16-byte units (8 contraction elements each) are XOR-swizzled by
// (s >> 1) & 3: the MFMA fragment reads (8 lanes = rows 0..7 of one unit)
// and the loaders' 8-byte stores (16 lanes = two rows r, r + 1 or r, r + 4,
// eight 8-byte groups each) are then bank-conflict-free.
template <int B> struct Planes {
  static constexpr int PLANE = B * 64;
  static constexpr int SIZE = 3 * PLANE;
  // byte offset of contraction elements k..k+3 (k % 4 == 0) of row r
  __device__ static int at(int r, int k) {
    const int s = r ^ ((r >> 2) & 1);
    return s * 64 + ((((k >> 3) ^ (s >> 1)) & 3) << 4) + ((k & 4) << 1);
  }
};

// Parts of four consecutive contraction elements, two bf16 per dword (the
// lower element in the low half): P[0] = h, P[1] = m, P[2] = l.
template <bool FULL>
__device__ __forceinline__ void split4(const float (&v)[4], uint2 (&P)[3]) {
  unsigned h[4], m[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = __float_as_uint(v[e]);
    if constexpr (FULL) {
      const float r = bf16_rest(v[e]);
      m[e] = __float_as_uint(r);
      l[e] = __float_as_uint(r - __uint_as_float(m[e] & 0xffff0000u));
    }
  }
  P[0] = make_uint2(__builtin_amdgcn_perm(h[1], h[0], 0x07060302u),
                    __builtin_amdgcn_perm(h[3], h[2], 0x07060302u));
  if constexpr (FULL) {
    P[1] = make_uint2(__builtin_amdgcn_perm(m[1], m[0], 0x07060302u),
                      __builtin_amdgcn_perm(m[3], m[2], 0x07060302u));
    P[2] = make_uint2(__builtin_amdgcn_perm(l[1], l[0], 0x07060302u),
                      __builtin_amdgcn_perm(l[3], l[2], 0x07060302u));
  }
}

// Split table: entry i = (h | m << 16, l) of tab[i]; entry 256 is zero (the
// index of invalid elements).  Returns whether every entry is bf16 exactly
// (all m and l parts zero).  Needs GT == 256 threads; ends with a barrier.
__device__ __forceinline__ bool split_table(uint2* stab, const float* tab, int t) {
  const float v = tab[t];
  const unsigned u = __float_as_uint(v);
  const float r = bf16_rest(v);
  const unsigned ru = __float_as_uint(r);
  const unsigned lo = __float_as_uint(r - __uint_as_float(ru & 0xffff0000u));
  stab[t] = make_uint2((u >> 16) | (ru & 0xffff0000u), lo >> 16);
  if (t == 0) stab[256] = make_uint2(0u, 0u);
  return __syncthreads_or(r != 0.0f) == 0;
}

// Whether every entry of a 256-entry table is bf16 exactly (GT == 256
// threads; ends with a barrier).
__device__ __forceinline__ bool table_exact(const float* tab, int t) {
  const float v = tab[t];
  return __syncthreads_or(bf16_rest(v) != 0.0f) == 0;
}

// Parts of four table entries (indices into a split table) in split4's order.
template <bool FULL>
__device__ __forceinline__ void lookup4(const uint2* stab, const unsigned (&idx)[4],
                                        uint2 (&P)[3]) {
  uint2 e[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) e[i] = stab[idx[i]];
  P[0] = make_uint2(__builtin_amdgcn_perm(e[1].x, e[0].x, 0x05040100u),
                    __builtin_amdgcn_perm(e[3].x, e[2].x, 0x05040100u));
  if constexpr (FULL) {
    P[1] = make_uint2(__builtin_amdgcn_perm(e[1].x, e[0].x, 0x07060302u),
                      __builtin_amdgcn_perm(e[3].x, e[2].x, 0x07060302u));
    P[2] = make_uint2(__builtin_amdgcn_perm(e[1].y, e[0].y, 0x05040100u),
                      __builtin_amdgcn_perm(e[3].y, e[2].y, 0x05040100u));
  }
}

template <int B, bool FULL>
__device__ __forceinline__ void put_parts(char* s, int r, int k, const uint2 (&P)[3]) {
  const int off = Planes<B>::at(r, k);
  *(uint2*)(s + off) = P[0];
  if constexpr (FULL) {
    *(uint2*)(s + Planes<B>::PLANE + off) = P[1];
    *(uint2*)(s + 2 * Planes<B>::PLANE + off) = P[2];
  }
}

// Index of an image element (int8: v + 128, uint8: v, fp32: quant_index).
template <typename T> __device__ __forceinline__ unsigned img_index(unsigned raw, int offset);
template <> __device__ __forceinline__ unsigned img_index<int8_t>(unsigned raw, int) {
  return (raw + 128u) & 255u;
}
template <> __device__ __forceinline__ unsigned img_index<uint8_t>(unsigned raw, int) {
  return raw & 255u;
}
template <> __device__ __forceinline__ unsigned img_index<float>(unsigned raw, int offset) {
  return quant_index(__uint_as_float(raw), offset);
}

// ------------------------------------------------------------- operand loaders
// Each loader owns a BK x B slice of one operand: fetch() issues the global
// loads of k-tile p0 into registers, stash() maps them through the LDS table
// (if any) and stores them into an LDS tile.  fetch() has no branches: an
// element outside the operand loads element 0 instead and its validity bit
// zeroes it in stash(), so the compiler never waits for a load before the
// MFMAs that follow.  VEC: the operand's quads are 16-byte (4-byte for
// bytes) aligned and never straddle a row, so one vector load covers them.

// Backward-data A: A(m = k, p = o) = tx[wq[o*K + k]], KMajor.
template <int B, bool VEC> struct DataA {
  using Lay = KMajor<B>;
  static constexpr int QPR = B / 4, NQ = BK * B / (4 * GT), PSTEP = GT / QPR;
  const uint8_t* wq; int K;
  int mq, pr, gm;
  unsigned raw[NQ], ok;
  __device__ void init(int t, int m0) {
    mq = (t % QPR) * 4; pr = t / QPR; gm = m0 + mq;
  }
  __device__ void fetch(int p0, int pe) {
    ok = 0;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int p = p0 + pr + i * PSTEP;
      const long long row = (long long)p * K;
      if constexpr (VEC) {
        const bool v = p < pe && gm < K;
        raw[i] = *(const unsigned*)(wq + (v ? row + gm : 0));
        ok |= (v ? 15u : 0u) << (4 * i);
      } else {
        raw[i] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool v = p < pe && gm + e < K;
          raw[i] |= (unsigned)wq[v ? row + gm + e : 0] << (8 * e);
          ok |= (v ? 1u : 0u) << (4 * i + e);
        }
      }
    }
  }
  __device__ void stash(float* s, const float* tab) const {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      floatx4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = tab[(raw[i] >> (8 * e)) & 255u];
        v[e] = (ok >> (4 * i + e)) & 1u ? x : 0.0f;
      }
      *(floatx4*)&s[Lay::at(mq, pr + i * PSTEP)] = v;
    }
  }
  __device__ void advance() {}
};

// Backward-data B: B(p = o, j = c) = go[n][o][l] (* sx * sw[o] when SCALED)
// with c = n*L + l, KMajor.  The scale product is rounded to fp32 first and
// then applied, the order of the layer's `y * (scale_x * scale_w)`.
template <int B, bool VEC, bool SCALED> struct DataB {
  using Lay = KMajor<B>;
  static constexpr int QPR = B / 4, NQ = BK * B / (4 * GT), PSTEP = GT / QPR;
  const float* go; int O, L, NL;
  const float* sx; const float* sw;
  int jq, pr;
  float sx0;
  long long base[4];        // go offset of column c + e at o = 0 (-1: no column)
  floatx4 raw[NQ];
  float sc[NQ];
  unsigned ok;
  __device__ void init(int t, int n0) {
    jq = (t % QPR) * 4; pr = t / QPR;
    if constexpr (SCALED) sx0 = sx[0];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = n0 + jq + e;
      if (c < NL) {
        const int n = c / L;
        base[e] = (long long)n * O * L + (c - n * L);
      } else {
        base[e] = -1;
      }
    }
  }
  __device__ void fetch(int p0, int pe) {
    ok = 0;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int o = p0 + pr + i * PSTEP;
      const long long ol = (long long)o * L;
      if constexpr (SCALED) sc[i] = sw[o < pe ? o : 0];
      if constexpr (VEC) {
        const bool v = o < pe && base[0] >= 0;
        raw[i] = *(const floatx4*)(go + (v ? base[0] + ol : 0));
        ok |= (v ? 15u : 0u) << (4 * i);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool v = o < pe && base[e] >= 0;
          raw[i][e] = go[v ? base[e] + ol : 0];
          ok |= (v ? 1u : 0u) << (4 * i + e);
        }
      }
    }
  }
  __device__ void stash(float* s, const float*) const {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      floatx4 v;
      float f = 1.0f;
      if constexpr (SCALED) f = sx0 * sc[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = SCALED ? raw[i][e] * f : raw[i][e];
        v[e] = (ok >> (4 * i + e)) & 1u ? x : 0.0f;
      }
      *(floatx4*)&s[Lay::at(jq, pr + i * PSTEP)] = v;
    }
  }
  __device__ void advance() {}
};

// Backward-weight A: A(m = o, p = r) = go[n][o][l] with r = n*L + l, read by
// buffer loads from a descriptor that starts at image n0 (the image of the
// block's first contraction row) and ends at the end of go: rows r >= P lie
// past its end and read 0, so they add nothing whatever the B operand holds,
// and rows o >= O read other images' values, whose results the epilogue
// drops.  The go scale sx * sw[o] is applied to the results instead (it is
// constant along the contraction).  VEC (L % 4 == 0): a quad of rows lies
// in one image, one 16-byte load.  Offsets are 32-bit: the host keeps a
// block's images within 2^31 bytes of go.
template <int B, bool VEC> struct WeightA {
  static constexpr int NQ = B / 32;        // quads per thread (rows m, m+32, ...)
  __amdgpu_buffer_rsrc_t res;
  int O, L;
  int pq, mr, m0;
  int n, l;                 // row p0 + pq: image (from n0) and position
  floatx4 raw[NQ];
  __device__ void init(const float* go, long long go_elems, int t, int mbase, int pb) {
    pq = (t & 7) * 4; mr = t >> 3; m0 = mbase;
    const int n0 = pb / L;
    const long long base = (long long)n0 * O * L;
    const long long bytes = (go_elems - base) * 4;
    res = buffer_rsrc(go + base, (int)(unsigned)(bytes < 0xffffffffLL ? bytes : 0xffffffffLL));
    const int r = pb + pq - n0 * L;
    n = r / L;
    l = r - n * L;
  }
  __device__ void fetch(int, int) {
    const int rowb = 32 * L * 4;           // bytes between a thread's rows o, o + 32
    const unsigned ob = (unsigned)(m0 + mr);
    if constexpr (VEC) {
      const unsigned off = (((unsigned)n * O + ob) * L + l) * 4u;
#pragma unroll
      for (int i = 0; i < NQ; ++i)
        raw[i] = __builtin_bit_cast(floatx4,
                                    __builtin_amdgcn_raw_buffer_load_b128(res, off, i * rowb, 0));
    } else {
      unsigned off[4];
      int en = n, el = l;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        off[e] = (((unsigned)en * O + ob) * L + el) * 4u;
        if (++el == L) { el = 0; ++en; }
      }
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          raw[i][e] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(res, off[e], i * rowb, 0));
    }
  }
  template <bool FULL> __device__ void put(char* s, const uint2*) const {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const float v[4] = {raw[i][0], raw[i][1], raw[i][2], raw[i][3]};
      uint2 P[3];
      split4<FULL>(v, P);
      put_parts<B, FULL>(s, mr + 32 * i, pq, P);
    }
  }
  __device__ void advance() {
    l += BK;
    while (l >= L) { l -= L; ++n; }
  }
};

// Backward-weight B: B(p = r, j = k) = tw[index of image tap k at output
// position r] (implicit im2col).  Out-of-image taps use `pad`.  Taps k >= K
// and rows r >= P (whose A values are 0) take the pad entry; the table's
// entries are finite, so those products are 0 or dropped by the epilogue.
template <int B, typename T> struct WeightB {
  static constexpr int NQ = B / 32;
  const T* img; atx_conv_geom g; int K, L, offset, pad;
  int pq, jr;
  int coff[NQ], dh[NQ], dw[NQ];     // per tap: c*H*W, kh*DH - PH, kw*DW - PW
  unsigned kv;                      // bit i: tap i < K
  int n, oh, ow;                    // output position of row p0 + pq
  unsigned raw[NQ][4], in;          // in: element read from the image
  __device__ void init(int t, int n0, int pb) {
    pq = (t & 7) * 4; jr = t >> 3;
    const int KK = g.KH * g.KW;
    kv = 0;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int k = n0 + jr + 32 * i;
      const int kc = k < K ? k : 0;
      const int c = kc / KK, tt = kc - c * KK;
      const int kh = tt / g.KW, kw = tt - kh * g.KW;
      coff[i] = c * g.H * g.W;
      dh[i] = kh * g.DH - g.PH;
      dw[i] = kw * g.DW - g.PW;
      if (k < K) kv |= 1u << i;
    }
    const int r = pb + pq;
    n = r / L;
    const int l = r - n * L;
    oh = l / g.OW;
    ow = l - oh * g.OW;
  }
  __device__ void fetch(int p0, int pe) {
    const int r = p0 + pq;
    in = 0;
    int en = n, eh = oh, ew = ow;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool rv = r + e < pe;
      const long long nb = (long long)en * g.C * g.H * g.W;
      const int ih0 = eh * g.SH, iw0 = ew * g.SW;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int ih = ih0 + dh[i], iw = iw0 + dw[i];
        const bool inside = rv && ((kv >> i) & 1u) && (unsigned)ih < (unsigned)g.H &&
                            (unsigned)iw < (unsigned)g.W;
        const T x = img[inside ? nb + coff[i] + ih * g.W + iw : 0];
        if constexpr (sizeof(T) == 4) raw[i][e] = __float_as_uint((float)x);
        else raw[i][e] = (unsigned)(unsigned char)x;
        in |= (inside ? 1u : 0u) << (4 * i + e);
      }
      if (++ew == g.OW) { ew = 0; if (++eh == g.OH) { eh = 0; ++en; } }
    }
  }
  template <bool FULL> __device__ void put(char* s, const uint2* stab) const {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      unsigned idx[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        idx[e] = (in >> (4 * i + e)) & 1u ? img_index<T>(raw[i][e], offset) : (unsigned)pad;
      uint2 P[3];
      lookup4<FULL>(stab, idx, P);
      put_parts<B, FULL>(s, jr + 32 * i, pq, P);
    }
  }
  __device__ void advance() {
    ow += BK;
    while (ow >= g.OW) {
      ow -= g.OW;
      if (++oh == g.OH) { oh = 0; ++n; }
    }
  }
};

// Backward-weight B from the forward's row-offset operand: B(p = r, j = k) =
// tw[xt[slot(k, r)][r] >> 8] (xt as the LUT GEMM reads it: [Kpad][Rpad]
// uint16, slot(k, r) = (k & ~3) | ((k - (r >> 2)) & 3), padding taps and
// rows hold offset 0).  A thread's four rows are one quad and the quad index
// moves by BK / 4 = 8 per k-tile, so each of its taps stays in one slot: one
// 8-byte load per (tap, k-tile) and a bit-field extract per element.  Taps
// k >= K and rows r >= P read padding (finite table entries): their results
// are dropped or multiplied by A's zeros.
template <int B> struct WeightBRows {
  static constexpr int NQ = B / 32;
  const uint16_t* xt; long long Rpad; int K, Kpad;
  int pq, jr;
  const uint16_t* src[NQ];          // slot row of tap i, at the thread's current quad
  uint2 raw[NQ];
  __device__ void init(int t, int n0, int pb) {
    pq = (t & 7) * 4; jr = t >> 3;
    const int r0 = pb + pq;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int k = n0 + jr + 32 * i;
      const int slot = k < Kpad ? ((k & ~3) | ((k - (r0 >> 2)) & 3)) : 0;
      src[i] = xt + (long long)slot * Rpad + r0;
    }
  }
  __device__ void fetch(int, int) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) raw[i] = *(const uint2*)src[i];
  }
  template <bool FULL> __device__ void put(char* s, const uint2* stab) const {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const unsigned w[2] = {raw[i].x, raw[i].y};
      unsigned idx[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) idx[e] = (w[e >> 1] >> (16 * (e & 1) + 8)) & 255u;
      uint2 P[3];
      lookup4<FULL>(stab, idx, P);
      put_parts<B, FULL>(s, jr + 32 * i, pq, P);
    }
  }
  __device__ void advance() {
#pragma unroll
    for (int i = 0; i < NQ; ++i) src[i] += BK;
  }
};

// ---------------------------------------- backward-data loaders (bf16 planes)
// Backward-data A from prepared planes [3][Kp][Opad] (the h, m, l parts of
// tx[wq[o][k]], zero for k >= K and o >= O; Kp, Opad multiples of 128 and
// 32): A(m = k, p = o).  Row m of a k-tile is 64 contiguous bytes per
// plane; a thread copies 16-byte units (three planes, or only the h plane
// when the table is bf16 exactly).  Buffer loads: rows past the planes read
// 0.
template <int B> struct PlaneA {
  static constexpr int NU = 3 * B * 4 / GT;   // 16-byte units per thread, three planes
  const uint16_t* planes; int pbytes;        // the planes and their size
  __amdgpu_buffer_rsrc_t res;
  int Kp, Opad, m0, t;
  bool full;
  u32x4 raw[NU];
  __device__ void init(int tid, int mbase) {
    t = tid; m0 = mbase;
    res = buffer_rsrc(planes, pbytes);
  }
  __device__ void fetch(int p0, int) {
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      if (j >= NU / 3 && !full) break;
      const int u = t + GT * j;
      const int q = u / (4 * B), row = (u >> 2) % B, unit = u & 3;
      const unsigned off = (((unsigned)q * Kp + m0 + row) * Opad + p0 + 8 * unit) * 2u;
      raw[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(res, off, 0, 0));
    }
  }
  template <bool FULL> __device__ void put(char* s, const uint2*) const {
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      if (j >= NU / 3 && !FULL) break;
      const int u = t + GT * j;
      const int q = u / (4 * B), row = (u >> 2) % B, unit = u & 3;
      *(u32x4*)(s + q * Planes<B>::PLANE + Planes<B>::at(row, 8 * unit)) = raw[j];
    }
  }
  __device__ void advance() {}
};

// Backward-data B: B(p = o, col = c) = go[n][o][l] * fp32(sx * sw[o]) with
// c = n*L + l (the product of scales rounded first, the order of the layer's
// `y * (scale_x * scale_w)`).  A thread holds four columns x four
// consecutive o (o-quad oq = t & 7, column quad cq = t >> 3) and stores each
// column's four contraction elements as 8-byte plane groups.  Buffer loads
// from a descriptor starting at the block's first image: columns past N*L
// read 0 (offset 2^31, past the descriptor), o >= O reads the next image's
// values or 0 (the A planes are 0 there).  VEC (L % 4 == 0): a column quad
// lies in one image, one 16-byte load per o.
template <int B, bool VEC, bool SCALED> struct GoCols {
  static_assert(B == 128, "GoCols covers 128 columns with 256 threads");
  __amdgpu_buffer_rsrc_t res;
  int O, L;                 // L: positions of go per image
  int Lc;                   // columns per image
  int W, OW, first;         // W > 0: column q is go's position (q / W) * OW + q % W + first
  const float* sx; const float* sw;
  int oq, cq;
  unsigned off[4];          // byte offset of column 4cq + e at o = 0 (VEC: off[0] only)
  floatx4 raw[4];           // raw[i][e]: o = p0 + 4oq + i, column 4cq + e
  float sc[4];
  __device__ void init(const float* go, long long go_elems, int tid, int n0, int NL) {
    oq = tid & 7; cq = tid >> 3;
    const int nb = n0 / Lc;
    const long long base = (long long)nb * O * L;
    const long long bytes = (go_elems - base) * 4;
    res = buffer_rsrc(go + base, (int)(bytes < 0x7fffffffLL ? bytes : 0x7fffffffLL));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = n0 + 4 * cq + e;
      const int n = c / Lc;
      int l = c - n * Lc;
      if (!VEC && W > 0) l = l / W * OW + l % W + first;
      off[e] = c < NL ? (unsigned)(((long long)(n - nb) * O * L + l) * 4) : 0x80000000u;
    }
  }
  __device__ void fetch(int p0, int) {
    const int ob = p0 + 4 * oq;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned ol = (unsigned)(ob + i) * L * 4u;
      if constexpr (SCALED) sc[i] = sx[0] * sw[ob + i < O ? ob + i : 0];
      if constexpr (VEC) {
        raw[i] = __builtin_bit_cast(floatx4,
                                    __builtin_amdgcn_raw_buffer_load_b128(res, off[0] + ol, 0, 0));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          raw[i][e] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(res, off[e] + ol, 0, 0));
      }
    }
    // The last, partial k-tile reads rows o >= O (the next image's), whose
    // weight planes are zero: zero them here too, so that a non-finite go
    // there cannot add 0 * inf = NaN.  p0 is the tile start (wave-uniform).
    if (p0 + 32 > O) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (ob + i >= O) raw[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  }
  template <bool FULL> __device__ void put(char* s, const uint2*) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = SCALED ? raw[i][e] * sc[i] : raw[i][e];
      uint2 P[3];
      split4<FULL>(v, P);
      put_parts<B, FULL>(s, 4 * cq + e, 4 * oq, P);
    }
  }
  __device__ void advance() {}
};

// ------------------------------------------------------------------ epilogues
// out[n][k][l] of the backward-data GEMM (rows m = k, columns c = n*L + l).
// With `mask`, the fake-quant STE is applied on the way out:
// v = (mask ? v : 0) / max(scale, 1e-12) (the 1x1 stride-1 conv, whose
// columns are the image gradient itself).
struct DataOut {
  float* col; int K, L, NL;
  const uint8_t* mask; const float* scale;
  long long split_stride;   // elements per partial slice (blockIdx.z = slice)
};
// ws[s][o][k] of the backward-weight GEMM, times the go scale sx * sw[o]
// when sw is given.
struct WeightOut {
  float* ws; int O, K; long long sst;
  const float* sx; const float* sw;
  __device__ void store(int m, int c, float v, int s) const {
    if (m < O && c < K) {
      if (sw) v *= sx[0] * sw[m];
      ws[(long long)s * sst + (long long)m * K + c] = v;
    }
  }
};

// ----------------------------------------------------------------- main kernel
// TR: the MFMA takes the B fragment as its first operand, so the 16x16
// result block is stored transposed (lane holds columns 4*(lane >> 4) + r of
// row lane & 15); the products and their order are the same.
template <int BM, int BN, class LA, class LB, bool TR = false>
__device__ __forceinline__ void mma_tile(const float* As, const float* Bs,
                                         floatx4 (&acc)[BM / 32][BN / 32]) {
  constexpr int TM = BM / 32, TN = BN / 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < BK; kk += 4) {
    float a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = As[LA::Lay::at(wm * (BM / 2) + i * 16 + li, kk + lk)];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = Bs[LB::Lay::at(wn * (BN / 2) + j * 16 + li, kk + lk)];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = TR ? __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], a[i], acc[i][j], 0, 0, 0)
                       : __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
  }
}

// acc = sum over the contraction range [pb, pe) of A tile x B tile.
// Double-buffered: the global loads of k-tile i+1 are in flight while tile i
// is multiplied; one barrier per k-tile.
template <int BM, int BN, bool TR = false, class LA, class LB>
__device__ __forceinline__ void gemm_tiles(LA& la, LB& lb, const float* tab, int pb, int pe,
                                           floatx4 (&acc)[BM / 32][BN / 32], float* As0,
                                           float* As1, float* Bs0, float* Bs1) {
#pragma unroll
  for (int i = 0; i < BM / 32; ++i)
#pragma unroll
    for (int j = 0; j < BN / 32; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  if (pb >= pe) return;

  la.fetch(pb, pe);
  lb.fetch(pb, pe);
  la.stash(As0, tab);
  lb.stash(Bs0, tab);
  __syncthreads();
  float *Ac = As0, *An = As1, *Bc = Bs0, *Bn = Bs1;
  for (int p0 = pb; p0 + BK < pe; p0 += BK) {
    la.advance(); lb.advance();
    la.fetch(p0 + BK, pe);
    lb.fetch(p0 + BK, pe);
    // Keep the next tile's loads ahead of the MFMAs and their consumers
    // behind them: the scheduler would otherwise sink the loads, or hoist
    // the stash's use of them, and expose the load latency.
    __builtin_amdgcn_sched_barrier(0);
    mma_tile<BM, BN, LA, LB, TR>(Ac, Bc, acc);
    __builtin_amdgcn_sched_barrier(0);
    la.stash(An, tab);
    lb.stash(Bn, tab);
    __syncthreads();
    float* x = Ac; Ac = An; An = x;
    x = Bc; Bc = Bn; Bn = x;
  }
  mma_tile<BM, BN, LA, LB, TR>(Ac, Bc, acc);
}

// acc += A tile x B tile from split-bf16 planes (one 32-deep MFMA step).
// Lane (i = lane & 15, g = lane >> 4) reads 16 bytes (contraction elements
// 8g..8g+7) of row i of each 16-row block; the result blocks have the fp32
// path's layout (lane holds rows 4g + r of column i).  The part products are
// added smallest first.
// TR: the B fragment is the MFMA's first operand, so each 16x16 result block
// comes out transposed (lane holds columns 4*(lane >> 4) + r of row
// lane & 15), the layout of the data epilogue's vector path.
template <int BM, int BN, int PR, bool TR = false>
__device__ __forceinline__ void mma_planes(const char* As, const char* Bs,
                                           floatx4 (&acc)[BM / 32][BN / 32]) {
  constexpr int TM = BM / 32, TN = BN / 32;
  constexpr int NA = PR == A_EXACT ? 1 : 3;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, k8 = 8 * (lane >> 4);
  // A parts stay in registers; the B parts are read one at a time, each
  // taking its products with the A parts of total order <= 2 (smallest
  // first: B part q with A parts 2 - q .. 0).
  u32x4 a[NA][TM];
#pragma unroll
  for (int q = 0; q < NA; ++q)
#pragma unroll
    for (int i = 0; i < TM; ++i)
      a[q][i] = *(const u32x4*)(As + q * Planes<BM>::PLANE +
                                Planes<BM>::at(wm * (BM / 2) + i * 16 + li, k8));
  constexpr int NB = PR == B_EXACT ? 1 : 3;
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    u32x4 b[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      b[j] = *(const u32x4*)(Bs + q * Planes<BN>::PLANE +
                             Planes<BN>::at(wn * (BN / 2) + j * 16 + li, k8));
#pragma unroll
    for (int qa = (PR == A_EXACT ? 0 : 2 - q); qa >= 0; --qa)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = TR ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                               __builtin_bit_cast(bf16x8, b[j]), __builtin_bit_cast(bf16x8, a[qa][i]),
                               acc[i][j], 0, 0, 0)
                         : __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                               __builtin_bit_cast(bf16x8, a[qa][i]), __builtin_bit_cast(bf16x8, b[j]),
                               acc[i][j], 0, 0, 0);
  }
}

// acc = sum over the contraction range [pb, pe) on split-bf16 planes.  One
// LDS tile per operand: the loaders' global loads of k-tile i+1 are in
// flight while tile i is multiplied, then stored as planes after a barrier
// (two barriers per k-tile; the kernels run two blocks per CU, so one
// block's MFMAs cover the other's stores).
template <int BM, int BN, int PR, bool TR = false, class LA, class LB>
__device__ __forceinline__ void gemm_planes(LA& la, LB& lb, const uint2* stab, int pb, int pe,
                                            floatx4 (&acc)[BM / 32][BN / 32], char* As,
                                            char* Bs) {
#pragma unroll
  for (int i = 0; i < BM / 32; ++i)
#pragma unroll
    for (int j = 0; j < BN / 32; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  if (pb >= pe) return;
  la.fetch(pb, pe);
  lb.fetch(pb, pe);
  for (int p0 = pb;; p0 += BK) {
    la.template put<PR != A_EXACT>(As, stab);
    lb.template put<PR != B_EXACT>(Bs, stab);
    __syncthreads();
    const bool more = p0 + BK < pe;
    if (more) {
      la.advance(); lb.advance();
      la.fetch(p0 + BK, pe);
      lb.fetch(p0 + BK, pe);
    }
    __builtin_amdgcn_sched_barrier(0);
    mma_planes<BM, BN, PR, TR>(As, Bs, acc);
    if (!more) break;
    __syncthreads();
  }
}

// Data-GEMM epilogue: out[n][m][l] for column c = n*L + l (rows m), with the
// optional per-tensor fake-quant STE (mask ? v : 0) / max(scale, 1e-12).
// VEC (L % 4 == 0, out 16-byte and mask 4-byte aligned): the tiles are
// multiplied with TR (transposed 16x16 blocks), so a lane holds the four
// consecutive columns c0..c0+3 of one row m; the quad lies in one image and
// is wholly inside N*L or wholly outside, so it is one 16-byte store and one
// 4-byte mask load.  Otherwise the blocks are untransposed and every element
// is stored on its own.
template <int BM, int BN, bool VEC>
__device__ __forceinline__ void data_epilogue(const DataOut& ep,
                                              const floatx4 (&acc)[BM / 32][BN / 32], int m0,
                                              int n0) {
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6, wm = wave >> 1, wn = wave & 1;
  constexpr int TM = BM / 32;
  const float sdiv = ep.mask ? fmaxf(ep.scale[0], 1e-12f) : 1.0f;
  if constexpr (VEC) {
#pragma unroll
  for (int j = 0; j < BN / 32; ++j) {
    const int c0 = n0 + wn * (BN / 2) + j * 16 + 4 * (lane >> 4);
    {
      const bool cv = c0 < ep.NL;
      const int cc = cv ? c0 : 0;
      const int n = cc / ep.L;
      const long long off = (long long)n * ep.K * ep.L + (cc - n * ep.L);
      if (ep.mask) {
        unsigned mk[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = m0 + wm * (BM / 2) + i * 16 + (lane & 15);
          mk[i] = *(const unsigned*)(ep.mask + (cv && m < ep.K ? off + (long long)m * ep.L : 0));
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = m0 + wm * (BM / 2) + i * 16 + (lane & 15);
          floatx4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = ((mk[i] >> (8 * r)) & 255u ? acc[i][j][r] : 0.0f) / sdiv;
          if (cv && m < ep.K) *(floatx4*)(ep.col + off + (long long)m * ep.L) = v;
        }
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = m0 + wm * (BM / 2) + i * 16 + (lane & 15);
          if (cv && m < ep.K) *(floatx4*)(ep.col + off + (long long)m * ep.L) = acc[i][j];
        }
      }
    }
  }
  } else {
    // untransposed blocks (lane holds rows 4*(lane >> 4) + r of column
    // lane & 15): per element, 16 consecutive columns per store
#pragma unroll
    for (int j = 0; j < BN / 32; ++j) {
      const int c = n0 + wn * (BN / 2) + j * 16 + (lane & 15);
      const bool cv = c < ep.NL;
      const int cc = cv ? c : 0;
      const int n = cc / ep.L;
      const long long off = (long long)n * ep.K * ep.L + (cc - n * ep.L);
      if (ep.mask) {
        unsigned char mk[TM][4];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + r;
            mk[i][r] = ep.mask[cv && m < ep.K ? off + (long long)m * ep.L : 0];
          }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + r;
            if (cv && m < ep.K)
              ep.col[off + (long long)m * ep.L] = (mk[i][r] ? acc[i][j][r] : 0.0f) / sdiv;
          }
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + r;
            if (cv && m < ep.K) ep.col[off + (long long)m * ep.L] = acc[i][j][r];
          }
      }
    }
  }
}


// VB: go quads (L % 4 == 0) are 16-byte loads and the output quads 16-byte
// stores (data_epilogue VEC).
template <int BM, int BN, bool VA, bool VB, bool SC>
__global__ void __launch_bounds__(GT, 2)
data_gemm_kernel(DataA<BM, VA> la, DataB<BN, VB, SC> lb, DataOut ep,
                 const float* __restrict__ tx, int O, int o_chunk) {
  __shared__ float tab[256];
  __shared__ __align__(16) float As[2][KMajor<BM>::SIZE];
  __shared__ __align__(16) float Bs[2][KMajor<BN>::SIZE];
  const int t = threadIdx.x;
  tab[t] = tx[t];
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  la.init(t, m0);
  lb.init(t, n0);
  __syncthreads();
  // contraction slice of this block (grid.z splits O; each slice writes its
  // own partial output, summed afterwards in a fixed order)
  const int ob = blockIdx.z * o_chunk, oe = min(O, ob + o_chunk);
  ep.col += (long long)blockIdx.z * ep.split_stride;
  floatx4 acc[BM / 32][BN / 32];
  gemm_tiles<BM, BN, VB>(la, lb, tab, ob, oe, acc, As[0], As[1], Bs[0], Bs[1]);
  data_epilogue<BM, BN, VB>(ep, acc, m0, n0);
}

// planes[q][k][o] (q = h, m, l part of tx[wq[o*K + k]]; zero for k >= K or
// o >= O) over Kp x Opad, the A operand of the plane data GEMMs.  A thread
// writes eight consecutive o of one k per plane (16 bytes).
__global__ void __launch_bounds__(GT)
weight_planes_kernel(const uint8_t* __restrict__ wq, const float* __restrict__ tx, int O, int K,
                     int Kp, int Opad, uint16_t* __restrict__ planes) {
  __shared__ uint2 stab[257];
  split_table(stab, tx, threadIdx.x);
  const long long idx = (long long)blockIdx.x * GT + threadIdx.x;
  const int per_row = Opad / 8;
  if (idx >= (long long)Kp * per_row) return;
  const int k = (int)(idx / per_row), o8 = (int)(idx - (long long)k * per_row) * 8;
  uint2 P[2][3];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    unsigned ix[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int o = o8 + 4 * h + e;
      ix[e] = k < K && o < O ? wq[(long long)o * K + k] : 256u;
    }
    lookup4<true>(stab, ix, P[h]);
  }
  const long long plane = (long long)Kp * Opad;
#pragma unroll
  for (int q = 0; q < 3; ++q)
    *(uint4*)(planes + q * plane + (long long)k * Opad + o8) =
        make_uint4(P[0][q].x, P[0][q].y, P[1][q].x, P[1][q].y);
}

// Backward-data GEMM on split-bf16 planes: A from weight_planes_kernel's
// planes (three parts, or one when the table is bf16 exactly), B = go (six
// part products, or three).  VB (L % 4 == 0): 16-byte go loads and the
// transposed epilogue.  Two blocks per CU.
template <int BM, bool VB, bool SC>
__global__ void __launch_bounds__(GT, 2)
data_planes_kernel(PlaneA<BM> la, GoCols<128, VB, SC> lb, DataOut ep,
                   const float* __restrict__ go, long long go_elems,
                   const float* __restrict__ tx, int O, int o_chunk) {
  __shared__ __align__(16) char As[Planes<BM>::SIZE];
  __shared__ __align__(16) char Bs[Planes<128>::SIZE];
  const int t = threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * 128;
  la.init(t, m0);
  lb.init(go, go_elems, t, n0, ep.NL);
  const bool exact = table_exact(tx, t);
  la.full = !exact;
  const int ob = blockIdx.z * o_chunk, oe = min(O, ob + o_chunk);
  ep.col += (long long)blockIdx.z * ep.split_stride;
  floatx4 acc[BM / 32][4];
  if (exact) gemm_planes<BM, 128, A_EXACT, VB>(la, lb, nullptr, ob, oe, acc, As, Bs);
  else gemm_planes<BM, 128, PROD6, VB>(la, lb, nullptr, ob, oe, acc, As, Bs);
  data_epilogue<BM, 128, VB>(ep, acc, m0, n0);
}

// -------------------------------- backward-data on position-major go planes
// go' = go * fp32(sx * sw[o]) split once into bf16 parts, laid out for the
// data GEMM's B operand: planes[p][ob][q][32] (p = n*L + l, ob = o / 32, part
// q = h, m, l; zero for o >= O), 192 contiguous bytes per (p, ob).  Bound by
// HBM: 4 bytes read and 6 written per element.  Block: 64 positions x 32
// channels, transposed through LDS so that both sides are whole lines.
__global__ void __launch_bounds__(256)
go_planes_kernel(const float* __restrict__ go, int N, int O, int L, int nOb,
                 const float* __restrict__ sx, const float* __restrict__ sw,
                 uint16_t* __restrict__ planes) {
  constexpr int ROW = 208;                 // LDS bytes per position (13 units: no conflicts)
  __shared__ __align__(16) char tile[64 * ROW];
  const int t = threadIdx.x, ob = blockIdx.y;
  const int P = N * L;
  const int pl = t & 63, o8 = (t >> 6) * 8;
  const int p = blockIdx.x * 64 + pl;
  if (p < P) {
    const int n = p / L, l = p - n * L;
    const float* src = go + (long long)n * O * L + l;
    uint2 h[2][3];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int o = ob * 32 + o8 + 4 * f + e;
        v[e] = o < O ? src[(long long)o * L] : 0.0f;
        if (sw && o < O) v[e] *= sx[0] * sw[o];
      }
      split4<true>(v, h[f]);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
      *(uint4*)(tile + pl * ROW + q * 64 + o8 * 2) =
          make_uint4(h[0][q].x, h[0][q].y, h[1][q].x, h[1][q].y);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int u = t + 256 * j, row = u / 12, part = u - row * 12;
    const long long pr = (long long)blockIdx.x * 64 + row;
    if (pr < P)
      *(uint4*)((char*)planes + (pr * nOb + ob) * 192 + part * 16) =
          *(const uint4*)(tile + row * ROW + part * 16);
  }
}

// Pixels of one residue class (h = ph mod SH, w = pw mod SW) of the image and
// the taps that reach them: rows i0 + a*istep (a < nI), columns j0 + b*jstep
// (b < nJ); pixel (ph + SH*hc, pw + SW*wc) reads output (hc + dh0 - a*dhs, wc
// + dw0 - b*dws).  With stride 1 there is one class and every tap reaches it.
struct TapClass {
  int ph, pw, Hc, Wc;
  int i0, istep, nI, j0, jstep, nJ;
  int dh0, dhs, dw0, dws;
};
struct TapClasses { TapClass c[4]; int n; };

// Image gradient gx[n][c][h][w] = sum over (tap, o) (before the STE): M = c,
// columns = the pixels of a class (blockIdx.z / splits), contraction over the
// class's taps and 32-channel blocks, split into `splits` partial images
// (blockIdx.z % splits).  A = rows c*KK + tap of the weight planes, B = the go
// planes' (shifted position, ob) rows, zero outside go.
//
// What bounded the kernel this replaces (go read, scaled and split in the
// k-loop) was its loader: sixteen 4-byte loads with tap arithmetic, ~120 VALU
// instructions and twelve LDS stores per thread and k-tile, against 48 MFMAs
// per wave.  Both operands are now copied as they lie, by loads that write LDS
// themselves (16 bytes a lane, no registers, no LDS store instructions) into
// the second of two stages while the first is multiplied: one barrier per
// k-tile.  A wave owns 32 rows x 64 columns; BM = 64: four waves, two blocks
// per CU; BM = 128: eight waves share the columns' planes.
struct TapArgs {
  const uint16_t* wplanes; const uint16_t* gplanes;
  int wbytes, gbytes;                      // sizes of the planes
  int Kp, KK, nOb;                         // weight plane rows, taps, 32-channel blocks
  int splits;
  TapClasses classes;
  atx_conv_geom g;
};

// One k-tile's planes of both operands.
template <int BM> struct TapStage {
  static constexpr int BYTES = Planes<BM>::SIZE + Planes<128>::SIZE;
};

using lds_ptr = __attribute__((address_space(3))) void*;

// Copies for one k-tile: a wave's 1 KiB pieces are 16 rows of one plane.  Lane
// i writes bytes 16 i of the piece, that is row s = 16 piece + i / 4 of the
// plane in its stored order (Planes): source row r = s ^ ((s >> 2) & 1), unit
// (i & 3) ^ ((s >> 1) & 3).
template <int BM> struct TapLoader {
  static constexpr int NW = BM / 16;       // waves
  static constexpr int GB = 8 / NW;        // column pieces per wave
  __amdgpu_buffer_rsrc_t wr, gr;
  int a, b, ob;                            // tap (a, b) of the class, channel block
  unsigned wrow, unit;                     // weight row (m0 + r) * KK, byte of the unit
  int base[GB], hc[GB], wc[GB];            // image's first position, or -1; pixel
  int wave;
  bool full;
  __device__ void init(const TapArgs& p, const TapClass& k, int m0, int n0, int cols, int tile,
                       bool full_) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    full = full_;
    const int lane = threadIdx.x & 63, s = lane >> 2;          // within a piece
    const int r = s ^ ((s >> 2) & 1);
    unit = (unsigned)(((lane & 3) ^ ((s >> 1) & 3)) << 4);
    wr = buffer_rsrc(p.wplanes, p.wbytes);
    gr = buffer_rsrc(p.gplanes, p.gbytes);
    const int tap = tile / p.nOb;
    ob = tile - tap * p.nOb;
    a = tap / k.nJ;
    b = tap - a * k.nJ;
    wrow = (unsigned)(m0 + 16 * wave + r) * p.KK;
    const int HWc = k.Hc * k.Wc;
#pragma unroll
    for (int j = 0; j < GB; ++j) {
      const int c = n0 + 16 * (wave + NW * j) + r;
      const int n = c / HWc, q = c - n * HWc;
      hc[j] = q / k.Wc;
      wc[j] = q - hc[j] * k.Wc;
      base[j] = c < cols ? n * p.g.OH * p.g.OW : -1;
    }
  }
  // Issues the copies of the current k-tile into `st` and steps to the next.
  __device__ __forceinline__ void load(const TapArgs& p, const TapClass& k, char* st) {
    const int tap = (k.i0 + a * k.istep) * p.g.KW + k.j0 + b * k.jstep;
    const unsigned woff = ((wrow + tap) * (unsigned)p.nOb + ob) * 64u + unit;
    const int wplane = p.Kp * p.nOb * 64;
    char* as = st + 1024 * wave;
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q == 0 || full)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(as + q * Planes<BM>::PLANE), 16,
                                                 (int)woff, q * wplane, 0, 0);
    const int dh = k.dh0 - a * k.dhs, dw = k.dw0 - b * k.dws;
    char* bs = st + Planes<BM>::SIZE + 1024 * wave;
#pragma unroll
    for (int j = 0; j < GB; ++j) {
      const int oh = hc[j] + dh, ow = wc[j] + dw;
      const bool v = base[j] >= 0 && (unsigned)oh < (unsigned)p.g.OH &&
                     (unsigned)ow < (unsigned)p.g.OW;
      const unsigned off =
          v ? (unsigned)((base[j] + oh * p.g.OW + ow) * p.nOb + ob) * 192u + unit : 0x80000000u;
#pragma unroll
      for (int q = 0; q < 3; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            gr, (lds_ptr)(bs + 1024 * NW * j + q * Planes<128>::PLANE), 16, (int)off, 64 * q, 0, 0);
    }
    if (++ob == p.nOb) {
      ob = 0;
      if (++b == k.nJ) { b = 0; ++a; }
    }
  }
};

// part += the k-tile's products for the wave's 32 rows x 64 columns (part
// products smallest first, as mma_planes).
template <int BM, bool EXACT, bool TR>
__device__ __forceinline__ void mma_stage(const char* st, floatx4 (&part)[2][4]) {
  constexpr int NA = EXACT ? 1 : 3;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = (wave >> 1) * 32 + (lane & 15), col = (wave & 1) * 64 + (lane & 15);
  const int k8 = 8 * (lane >> 4);
  const char* As = st;
  const char* Bs = st + Planes<BM>::SIZE;
  u32x4 a[NA][2];
#pragma unroll
  for (int q = 0; q < NA; ++q)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      a[q][i] = *(const u32x4*)(As + q * Planes<BM>::PLANE + Planes<BM>::at(row + 16 * i, k8));
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    u32x4 b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      b[j] = *(const u32x4*)(Bs + q * Planes<128>::PLANE + Planes<128>::at(col + 16 * j, k8));
#pragma unroll
    for (int qa = EXACT ? 0 : 2 - q; qa >= 0; --qa)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bf16x8 x = __builtin_bit_cast(bf16x8, a[qa][i]);
          const bf16x8 y = __builtin_bit_cast(bf16x8, b[j]);
          part[i][j] = TR ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(y, x, part[i][j], 0, 0, 0)
                          : __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, part[i][j], 0, 0, 0);
        }
  }
}

// acc += a tap's sums in the columns whose output the tap reads.  With a
// non-finite entry in the table, the zeros that stand for outputs outside go
// give products of NaN, and the tap adds nothing there (nor does it with a
// finite table, where the products are zero).
template <bool TR>
__device__ __forceinline__ void add_reached(floatx4 (&acc)[2][4], const floatx4 (&part)[2][4],
                                            const TapArgs& p, const TapClass& k, int n0,
                                            int tap) {
  const int a = tap / k.nJ, b = tap - a * k.nJ, HWc = k.Hc * k.Wc;
  const int dh = k.dh0 - a * k.dhs, dw = k.dw0 - b * k.dws;
  const int lane = threadIdx.x & 63;
  const int c0 = n0 + ((threadIdx.x >> 6) & 1) * 64 + (TR ? 4 * (lane >> 4) : lane & 15);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {            // TR: the block's columns; else its rows
      const int q = (c0 + 16 * j + (TR ? e : 0)) % HWc, hc = q / k.Wc, wc = q - hc * k.Wc;
      const bool in = (unsigned)(hc + dh) < (unsigned)p.g.OH &&
                      (unsigned)(wc + dw) < (unsigned)p.g.OW;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        acc[i][j][e] = in ? acc[i][j][e] + part[i][j][e] : acc[i][j][e];
    }
}

// acc += the products of `tiles` k-tiles.  A tap's sum, or at most FLUSH
// k-tiles of it, is accumulated on its own and then added: one chain over all
// taps and channels doubled the error of 9 x 128 terms against per-tap sums
// (5.2e-7 against 2.0e-7 of the result).
constexpr int FLUSH = 2;
template <int BM, bool EXACT, bool TR, bool FINITE>
__device__ __forceinline__ void tap_sums(TapLoader<BM>& ld, const TapArgs& p, const TapClass& k,
                                         int n0, int tiles, floatx4 (&acc)[2][4], char* st0,
                                         char* st1) {
  floatx4 part[2][4];
  int run = 0, ob = ld.ob, tap = ld.a * k.nJ + ld.b;
  ld.load(p, k, st0);
  auto step = [&](char* cur, char* nxt, int left) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's copies are in LDS
    __syncthreads();                                   // every wave's; the other stage is read
    if (left > 1) ld.load(p, k, nxt);
    if (run == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) part[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    mma_stage<BM, EXACT, TR>(cur, part);
    if (++ob == p.nOb) ob = 0;
    if (++run == FLUSH || ob == 0 || left == 1) {
      run = 0;
      if constexpr (FINITE) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] += part[i][j];
      } else {
        add_reached<TR>(acc, part, p, k, n0, tap);
      }
      if (ob == 0) ++tap;
    }
  };
  for (; tiles > 1; tiles -= 2) {
    step(st0, st1, tiles);
    step(st1, st0, tiles - 1);
  }
  if (tiles > 0) step(st0, st1, tiles);
}

// VO: one class and H*W % 4 == 0 (transposed blocks, 16-byte stores).
template <int BM, bool VO>
__global__ void __launch_bounds__(BM * 4, BM == 64 ? 2 : 1)
tap_planes_kernel(const TapArgs p, DataOut ep, const float* __restrict__ tx) {
  __shared__ __align__(16) char st0[TapStage<BM>::BYTES];
  __shared__ __align__(16) char st1[TapStage<BM>::BYTES];
  const int t = threadIdx.x;
  const int ci = blockIdx.z / p.splits, sl = blockIdx.z - ci * p.splits;
  const TapClass k = p.classes.c[ci];
  const int cols = p.g.N * k.Hc * k.Wc;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * 128;
  if (n0 >= cols) return;
  const int tiles = k.nI * k.nJ * p.nOb;
  const int chunk = (tiles + p.splits - 1) / p.splits;
  const int tb = min(tiles, sl * chunk), te = min(tiles, tb + chunk);
  ep.col += (long long)sl * ep.split_stride;
  floatx4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  bool rest = false, wild = false;         // each wave reads the whole table: no barrier
#pragma unroll
  for (int e = 0; e < 256; e += 64) {
    const float v = tx[e + (t & 63)];
    rest |= bf16_rest(v) != 0.0f;
    wild |= !__builtin_isfinite(v);
  }
  const bool exact = !__any(rest), finite = !__any(wild);
  if (tb < te) {
    TapLoader<BM> ld;
    ld.init(p, k, m0, n0, cols, tb, !exact);
    const int n = te - tb;
    if (exact && finite) tap_sums<BM, true, VO, true>(ld, p, k, n0, n, acc, st0, st1);
    else if (finite) tap_sums<BM, false, VO, true>(ld, p, k, n0, n, acc, st0, st1);
    else if (exact) tap_sums<BM, true, VO, false>(ld, p, k, n0, n, acc, st0, st1);
    else tap_sums<BM, false, VO, false>(ld, p, k, n0, n, acc, st0, st1);
  }
  // epilogue, with the fused STE (mask ? v : 0) / max(scale, 1e-12)
  const int lane = t & 63, wave = t >> 6;
  const int rb = m0 + (wave >> 1) * 32, cb = n0 + (wave & 1) * 64;
  const float sdiv = ep.mask ? fmaxf(ep.scale[0], 1e-12f) : 1.0f;
  if constexpr (VO) {                      // lane: columns c .. c + 3 of one row per block
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = cb + 16 * j + 4 * (lane >> 4);
      if (c >= cols) continue;
      const int n = c / ep.L;
      const long long off = (long long)n * ep.K * ep.L + (c - n * ep.L);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = rb + 16 * i + (lane & 15);
        if (m >= ep.K) continue;
        const long long at = off + (long long)m * ep.L;
        floatx4 v = acc[i][j];
        if (ep.mask) {
          const unsigned mk = *(const unsigned*)(ep.mask + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = ((mk >> (8 * e)) & 255u ? v[e] : 0.0f) / sdiv;
        }
        *(floatx4*)(ep.col + at) = v;
      }
    }
  } else {                                 // lane: rows m .. m + 3 of one column per block
    const int HWc = k.Hc * k.Wc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = cb + 16 * j + (lane & 15);
      if (c >= cols) continue;
      const int n = c / HWc, q = c - n * HWc;
      const int hc = q / k.Wc, wc = q - hc * k.Wc;
      const long long off = (long long)n * ep.K * ep.L +
                            (long long)(k.ph + p.g.SH * hc) * p.g.W + k.pw + p.g.SW * wc;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = rb + 16 * i + 4 * (lane >> 4) + e;
          if (m >= ep.K) continue;
          const long long at = off + (long long)m * ep.L;
          const float v = acc[i][j][e];
          ep.col[at] = ep.mask ? (ep.mask[at] ? v : 0.0f) / sdiv : v;
        }
    }
  }
}

template <class LB> __device__ __forceinline__ void set_pad(LB&, const float*) {}
template <int B, typename T>
__device__ __forceinline__ void set_pad(WeightB<B, T>& lb, const float* pad_dev) {
  if (pad_dev) lb.pad = (int)quant_index(pad_dev[0], 0);
}

// Backward-weight GEMM on split-bf16 planes: A = go (six part products),
// B = the table (three when every table entry is bf16 exactly).
template <int BM, int BN, bool VA, class LB>
__global__ void __launch_bounds__(GT, 2)
weight_gemm_kernel(WeightA<BM, VA> la, LB lb, WeightOut ep, const float* __restrict__ go,
                   long long go_elems, const float* __restrict__ tw,
                   const float* __restrict__ pad_dev, int P, int p_chunk) {
  __shared__ uint2 stab[257];
  __shared__ __align__(16) char As[Planes<BM>::SIZE];
  __shared__ __align__(16) char Bs[Planes<BN>::SIZE];
  const int t = threadIdx.x;
  set_pad(lb, pad_dev);
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int s = blockIdx.z;
  const int pb = s * p_chunk, pe = min(P, pb + p_chunk);
  la.init(go, go_elems, t, m0, pb);
  lb.init(t, n0, pb);
  const bool exact = split_table(stab, tw, t);
  floatx4 acc[BM / 32][BN / 32];
  if (exact) gemm_planes<BM, BN, B_EXACT>(la, lb, stab, pb, pe, acc, As, Bs);
  else gemm_planes<BM, BN, PROD6>(la, lb, stab, pb, pe, acc, As, Bs);
  const int lane = t & 63, wave = t >> 6, wm = wave >> 1, wn = wave & 1;
#pragma unroll
  for (int i = 0; i < BM / 32; ++i)
#pragma unroll
    for (int j = 0; j < BN / 32; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        ep.store(m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + r,
                 n0 + wn * (BN / 2) + j * 16 + (lane & 15), acc[i][j][r], s);
}

// gw[i] = sum_s ws[s][i]; optional per-channel term (the uint8 layer's weight
// zero point): gw -= (zsum[o] * (zsx * scale[o])) * zzx, each product and the
// difference rounded on its own; optional fused per-channel fake-quant
// backward: gw = mask ? gw / max(scale[o], 1e-12) : 0 with o = i / K.  A block
// sums 256 / G consecutive elements over G groups of slices (group g takes
// slices g, g + G, ...), then adds the G partials in group order:
// deterministic.
template <bool VEC>
__global__ void __launch_bounds__(256)
split_sum_kernel(const float* __restrict__ ws, int S, long long numel, int K, int G,
                 const uint8_t* __restrict__ mask, const float* __restrict__ scale,
                 float* __restrict__ out, const float* __restrict__ zsum,
                 const float* __restrict__ zsx, const float* __restrict__ zzx) {
  // VEC: each item is four consecutive elements (16-byte loads and stores;
  // numel % 4 == 0); every element keeps the same summation order.
  constexpr int W = VEC ? 4 : 1;
  typedef float floatw __attribute__((ext_vector_type(W)));
  __shared__ floatw part[256];
  const int t = threadIdx.x;
  const int epb = 256 / G;
  const int e = t % epb, grp = t / epb;
  const long long i = ((long long)blockIdx.x * epb + e) * W;   // first element
  floatw a = 0.0f;
  if (i < numel)
    for (int s = grp; s < S; s += G) a += *(const floatw*)(ws + (long long)s * numel + i);
  part[t] = a;
  __syncthreads();
  if (grp == 0 && i < numel) {
    for (int g = 1; g < G; ++g) a += part[g * epb + e];
    if (mask || zsum) {
      long long o = i / K, r = i - o * K;
#pragma unroll
      for (int j = 0; j < W; ++j) {
        float v = a[j];
        if (zsum) {
#pragma clang fp contract(off)
          v = v - (zsum[o] * (zsx[0] * scale[o])) * zzx[0];
        }
        if (mask) v = (mask[i + j] ? v : 0.0f) / fmaxf(scale[o], 1e-12f);
        a[j] = v;
        if (++r == K) { r = 0; ++o; }
      }
    }
    *(floatw*)(out + i) = a;
  }
}

// Launch of split_sum_kernel: enough groups that the grid has >= 1024 blocks.
int launch_split_sum(const float* ws, int S, long long numel, int K,
                            const uint8_t* mask, const float* scale, float* out,
                            hipStream_t stream, const float* zsum, const float* zsx,
                            const float* zzx) {
  const bool vec = numel % 4 == 0 && ((uintptr_t)ws & 15) == 0 && ((uintptr_t)out & 15) == 0;
  const long long items = vec ? numel / 4 : numel;
  int G = 1;
  while (G < 64 && G < S && cdiv(items, 256 / G) < 1024) G *= 2;
  const long long blocks = cdiv(items, 256 / G);
  ATX_REQUIRE(blocks <= 0x7fffffffLL, "split_sum: too many elements");
  if (vec)
    hipLaunchKernelGGL(split_sum_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, stream,
                       ws, S, numel, K, G, mask, scale, out, zsum, zsx, zzx);
  else
    hipLaunchKernelGGL(split_sum_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, stream,
                       ws, S, numel, K, G, mask, scale, out, zsum, zsx, zzx);
  return check_launch("split_sum_kernel");
}

inline int tile_of(int extent) { return extent <= 64 ? 64 : 128; }

// Split of the weight-gradient contraction, every split at least four
// k-tiles deep.  Cost in k-tiles: rounds of 512 blocks (two per CU) x
// (k-tiles per block + 4 for the block's prologue and epilogue) + 2 + S x
// O*K / 1.5e6 for writing and summing the S partial slices.  Any S, not just
// powers of two: one round with many k-tiles per block beats several rounds
// with few (each block's pipeline start and epilogue are paid per round).
static int weight_splits(int O, int K, long long P) {
  const long long tiles = cdiv(O, tile_of(O)) * cdiv(K, tile_of(K));
  const long long kt = cdiv(P, BK);                 // k-tiles of the contraction
  const long long smax = std::max<long long>(1, std::min<long long>(P / (4 * BK), 4096));
  double best = 0.0;
  long long pick = 1;
  for (long long s = 1; s <= smax; ++s) {
    const long long kc = cdiv(kt, s), sr = cdiv(kt, kc);
    // each split's rows of go within 1 GiB (32-bit buffer offsets)
    if ((double)kc * BK * O * 4.0 > (double)(1LL << 30) && s < smax) continue;
    const double cost = (double)cdiv(tiles * sr, 512) * (kc + 4) +
                        (sr > 1 ? 2.0 + (double)sr * O * K / 1.5e6 : 0.0);
    if (best == 0.0 || cost < best) { best = cost; pick = sr; }
  }
  return (int)pick;
}

struct DataArgs {
  const float* go; const uint8_t* wq; const float* tx; int N, O, K, L;
  const float* sx; const float* sw;          // optional go scale sx * sw[o]
  float* out; const uint8_t* mask; const float* scale;
  int splits, o_chunk;                       // contraction split (1 = none)
  float* partials;                           // [splits][N*K*L] when splits > 1
  uint16_t* planes;                          // bf16 weight planes (null: fp32 kernels)
  // A padded 1x1 conv (or null; with planes): only go's positions inside the
  // image are columns, and out is the image gradient.
  const atx_conv_geom* crop = nullptr;
  int columns() const { return crop ? crop->H * crop->W : L; }   // per image
};

// Bytes of the bf16 weight planes [3][Kp][Opad] (Kp = K rounded up to 128,
// Opad = O rounded up to 32; a multiple of 256 bytes).
static long long weight_planes_bytes(int K, int O) {
  return 3LL * cdiv(K, 128) * 128 * cdiv(O, BK) * BK * 2;
}

// go spans of at most 2^31 bytes per block (32-bit buffer offsets): the
// images a block's 128 columns touch, two partial images included.
static bool planes_fit(long long cols_per_image, int O, long long out_per_image) {
  return (cdiv(128, cols_per_image) + 2) * (long long)O * out_per_image * 4 < (1LL << 31);
}

static int launch_weight_planes(const uint8_t* wq, const float* tx, int O, int K,
                                uint16_t* planes, hipStream_t stream) {
  const int Kp = (int)(cdiv(K, 128) * 128), Opad = (int)(cdiv(O, BK) * BK);
  const long long items = (long long)Kp * (Opad / 8);
  hipLaunchKernelGGL(weight_planes_kernel, dim3((unsigned)cdiv(items, GT)), dim3(GT), 0, stream,
                     wq, tx, O, K, Kp, Opad, planes);
  return check_launch("weight_planes_kernel");
}

// Split of the backward-data contraction over O into deterministic partial
// slices, each at least four k-tiles deep.  Cost in k-tiles, as for the
// weight gradient: rounds of 512 blocks x (k-tiles per block + 4) + 2 + S x
// N*K*L / 1.5e6 for writing and summing the partials (the output is the
// col buffer or the image gradient, so a split pays only when the tiles
// leave most of a round idle).
static int data_splits(int N, int O, int K, int L) {
  const long long blocks = cdiv((long long)N * L, 128) * cdiv(K, tile_of(K));
  const long long numel = (long long)N * K * L;
  if (numel > 0x7fffffffLL) return 1;
  const long long kt = cdiv(O, BK);
  const long long smax = std::max<long long>(1, std::min<long long>(kt / 4, 64));
  double best = 0.0;
  long long pick = 1;
  for (long long s = 1; s <= smax; ++s) {
    const long long kc = cdiv(kt, s), sr = cdiv(kt, kc);
    const double cost = (double)cdiv(blocks * sr, 512) * (kc + 4) +
                        (sr > 1 ? 2.0 + (double)sr * numel / 1.5e6 : 0.0);
    if (s == 1 || cost < best) { best = cost; pick = sr; }
  }
  return (int)pick;
}

template <int BM, bool VA, bool VB, bool SC>
static void launch_data(const DataArgs& a, hipStream_t stream) {
  constexpr int BN = 128;
  const int NL = a.N * a.L;
  DataA<BM, VA> la{};
  la.wq = a.wq; la.K = a.K;
  DataB<BN, VB, SC> lb{};
  lb.go = a.go; lb.O = a.O; lb.L = a.L; lb.NL = NL; lb.sx = a.sx; lb.sw = a.sw;
  const bool split = a.splits > 1;
  DataOut ep{split ? a.partials : a.out, a.K, a.L, NL, split ? nullptr : a.mask,
             split ? nullptr : a.scale, (long long)NL * a.K};
  dim3 grid((unsigned)cdiv(NL, BN), (unsigned)cdiv(a.K, BM), (unsigned)a.splits);
  hipLaunchKernelGGL((data_gemm_kernel<BM, BN, VA, VB, SC>), grid, dim3(GT), 0, stream, la, lb,
                     ep, a.tx, a.O, a.o_chunk);
}

template <int BM, bool VB, bool SC>
static void launch_data_planes(const DataArgs& a, hipStream_t stream) {
  const int Lc = a.columns(), NL = a.N * Lc;
  PlaneA<BM> la{};
  la.planes = a.planes; la.pbytes = (int)weight_planes_bytes(a.K, a.O);
  la.Kp = (int)(cdiv(a.K, 128) * 128); la.Opad = (int)(cdiv(a.O, BK) * BK);
  GoCols<128, VB, SC> lb{};
  lb.O = a.O; lb.L = a.L; lb.Lc = Lc; lb.sx = a.sx; lb.sw = a.sw;
  if (a.crop) {
    lb.W = a.crop->W; lb.OW = a.crop->OW;
    lb.first = a.crop->PH * a.crop->OW + a.crop->PW;
  }
  const bool split = a.splits > 1;
  DataOut ep{split ? a.partials : a.out, a.K, Lc, NL, split ? nullptr : a.mask,
             split ? nullptr : a.scale, (long long)NL * a.K};
  dim3 grid((unsigned)cdiv(NL, 128), (unsigned)cdiv(a.K, BM), (unsigned)a.splits);
  hipLaunchKernelGGL((data_planes_kernel<BM, VB, SC>), grid, dim3(GT), 0, stream, la, lb, ep,
                     a.go, (long long)a.N * a.O * a.L, a.tx, a.O, a.o_chunk);
}

template <int BM, bool SC>
static void dispatch_data_vec(const DataArgs& a, hipStream_t stream) {
  const bool va = a.K % 4 == 0 && (uintptr_t)a.wq % 4 == 0;
  const float* out = a.splits > 1 ? a.partials : a.out;
  const bool vb = !a.crop && a.L % 4 == 0 && (uintptr_t)a.go % 16 == 0 &&
                  (uintptr_t)out % 16 == 0 &&
                  (a.splits > 1 || (uintptr_t)a.mask % 4 == 0);
  if (a.planes) {
    if (vb) launch_data_planes<BM, true, SC>(a, stream);
    else launch_data_planes<BM, false, SC>(a, stream);
    return;
  }
  if (va && vb) launch_data<BM, true, true, SC>(a, stream);
  else if (va) launch_data<BM, true, false, SC>(a, stream);
  else if (vb) launch_data<BM, false, true, SC>(a, stream);
  else launch_data<BM, false, false, SC>(a, stream);
}

// Runs the backward-data GEMM into a.out; with a.splits > 1 the partial
// slices go to a.partials and are summed into a.out (with the optional
// per-tensor STE mask) by split_sum_kernel.
static int run_data_gemm(DataArgs a, hipStream_t stream) {
  if (a.splits < 1) a.splits = 1;
  a.o_chunk = (int)(cdiv(cdiv(a.O, a.splits), BK) * BK);
  a.splits = (int)cdiv(a.O, a.o_chunk);
  if (a.planes && !planes_fit(a.columns(), a.O, a.L)) a.planes = nullptr;
  if (a.planes) {
    const int rc = launch_weight_planes(a.wq, a.tx, a.O, a.K, a.planes, stream);
    if (rc) return rc;
  }
  const bool sc = a.sw != nullptr;
  if (tile_of(a.K) == 64) {
    if (sc) dispatch_data_vec<64, true>(a, stream); else dispatch_data_vec<64, false>(a, stream);
  } else {
    if (sc) dispatch_data_vec<128, true>(a, stream); else dispatch_data_vec<128, false>(a, stream);
  }
  int rc = check_launch("data_gemm_kernel");
  if (rc || a.splits == 1) return rc;
  const long long numel = (long long)a.N * a.K * a.columns();
  // split_sum's per-channel scale index i / K: K = numel makes it per tensor
  return launch_split_sum(a.partials, a.splits, numel, (int)numel, a.mask, a.scale, a.out,
                          stream);
}

template <int BM, int BN, bool VA, typename T>
static void launch_weight(const float* go, const T* img, atx_conv_geom g, int O, int K, int L,
                          int P, int chunk, int S, int offset, int pad_index,
                          const float* pad_dev, const float* tw, const float* go_sx,
                          const float* go_sw, float* ws, hipStream_t stream) {
  WeightA<BM, VA> la{};
  la.O = O; la.L = L;
  WeightB<BN, T> lb{};
  lb.img = img; lb.g = g; lb.K = K; lb.L = L; lb.offset = offset; lb.pad = pad_index;
  WeightOut ep{ws, O, K, (long long)O * K, go_sx, go_sw};
  dim3 grid((unsigned)cdiv(K, BN), (unsigned)cdiv(O, BM), (unsigned)S);
  hipLaunchKernelGGL((weight_gemm_kernel<BM, BN, VA, WeightB<BN, T>>), grid, dim3(GT), 0,
                     stream, la, lb, ep, go, (long long)P * O, tw, pad_dev, P, chunk);
}

template <bool VA, typename T>
static void dispatch_weight_tiles(const float* go, const T* img, atx_conv_geom g, int O, int K,
                                  int L, int P, int chunk, int S, int offset, int pad_index,
                                  const float* pad_dev, const float* tw, const float* go_sx,
                                  const float* go_sw, float* ws, hipStream_t stream) {
  const int bm = tile_of(O), bn = tile_of(K);
#define ATX_LW(M_, N_)                                                                       \
  launch_weight<M_, N_, VA, T>(go, img, g, O, K, L, P, chunk, S, offset, pad_index, pad_dev, \
                               tw, go_sx, go_sw, ws, stream)
  if (bm == 64 && bn == 64) ATX_LW(64, 64);
  else if (bm == 64) ATX_LW(64, 128);
  else if (bn == 64) ATX_LW(128, 64);
  else ATX_LW(128, 128);
#undef ATX_LW
}

template <typename T>
static void dispatch_weight(const float* go, const T* img, atx_conv_geom g, int O, int K, int L,
                            int P, int chunk, int S, int offset, int pad_index,
                            const float* pad_dev, const float* tw, const float* go_sx,
                            const float* go_sw, float* ws, hipStream_t stream) {
  if (L % 4 == 0 && (uintptr_t)go % 16 == 0)
    dispatch_weight_tiles<true, T>(go, img, g, O, K, L, P, chunk, S, offset, pad_index, pad_dev,
                                   tw, go_sx, go_sw, ws, stream);
  else
    dispatch_weight_tiles<false, T>(go, img, g, O, K, L, P, chunk, S, offset, pad_index,
                                    pad_dev, tw, go_sx, go_sw, ws, stream);
}

template <int BM, int BN, bool VA>
static void launch_weight_rows(const float* go, const uint16_t* xt, long long Rpad, int O,
                               int K, int L, int P, int chunk, int S, const float* tw,
                               const float* go_sx, const float* go_sw, float* ws,
                               hipStream_t stream) {
  WeightA<BM, VA> la{};
  la.O = O; la.L = L;
  WeightBRows<BN> lb{};
  lb.xt = xt; lb.Rpad = Rpad; lb.K = K; lb.Kpad = (K + 3) & ~3;
  WeightOut ep{ws, O, K, (long long)O * K, go_sx, go_sw};
  dim3 grid((unsigned)cdiv(K, BN), (unsigned)cdiv(O, BM), (unsigned)S);
  hipLaunchKernelGGL((weight_gemm_kernel<BM, BN, VA, WeightBRows<BN>>), grid, dim3(GT), 0,
                     stream, la, lb, ep, go, (long long)P * O, tw, (const float*)nullptr, P,
                     chunk);
}

template <bool VA>
static void dispatch_weight_rows(const float* go, const uint16_t* xt, long long Rpad, int O,
                                 int K, int L, int P, int chunk, int S, const float* tw,
                                 const float* go_sx, const float* go_sw, float* ws,
                                 hipStream_t stream) {
  const int bm = tile_of(O), bn = tile_of(K);
#define ATX_LWR(M_, N_) \
  launch_weight_rows<M_, N_, VA>(go, xt, Rpad, O, K, L, P, chunk, S, tw, go_sx, go_sw, ws, stream)
  if (bm == 64 && bn == 64) ATX_LWR(64, 64);
  else if (bm == 64) ATX_LWR(64, 128);
  else if (bn == 64) ATX_LWR(128, 64);
  else ATX_LWR(128, 128);
#undef ATX_LWR
}

// Residue classes of a stride of 1 or 2 per axis, most taps first.
static TapClasses tap_classes(const atx_conv_geom& g) {
  TapClasses t{};
  const auto axis = [](int r, int S, int K, int Pd, int D, int size, int& i0, int& istep, int& nI,
                       int& d0, int& ds, int& ext) {
    ext = size > r ? (size - r + S - 1) / S : 0;
    nI = 0;
    istep = S == 2 && (D & 1) ? 2 : 1;     // taps of one parity of i*D
    i0 = 0;
    for (int i = 0; i < K; ++i)
      if ((r + Pd - i * D) % S == 0) { if (nI++ == 0) i0 = i; }
    d0 = (r + Pd - i0 * D) / S;            // exact for a reaching tap
    ds = istep * D / S;
  };
  for (int ph = 0; ph < g.SH; ++ph)
    for (int pw = 0; pw < g.SW; ++pw) {
      TapClass c{};
      c.ph = ph; c.pw = pw;
      axis(ph, g.SH, g.KH, g.PH, g.DH, g.H, c.i0, c.istep, c.nI, c.dh0, c.dhs, c.Hc);
      axis(pw, g.SW, g.KW, g.PW, g.DW, g.W, c.j0, c.jstep, c.nJ, c.dw0, c.dws, c.Wc);
      int at = t.n++;
      for (; at > 0 && t.c[at - 1].nI * t.c[at - 1].nJ < c.nI * c.nJ; --at) t.c[at] = t.c[at - 1];
      t.c[at] = c;
    }
  return t;
}

static long long go_planes_bytes(long long P, int O) { return P * cdiv(O, BK) * 192; }

// Split of the tap GEMM's contraction (partial images summed by split_sum):
// the cost of data_splits over the tiles and the deepest class's k-tiles.
static int tap_splits(const atx_conv_geom& g, int O) {
  const TapClasses t = tap_classes(g);
  const long long numel = (long long)g.N * g.C * g.H * g.W;
  const long long mt = cdiv(g.C, 64), nob = cdiv(O, BK);
  const long long kt = (long long)t.c[0].nI * t.c[0].nJ * nob;
  double work = 0.0;                       // k-tiles of all blocks
  long long blocks = 0;
  for (int i = 0; i < t.n; ++i) {
    const long long b = cdiv((long long)g.N * t.c[i].Hc * t.c[i].Wc, 128) * mt;
    blocks += b;
    work += (double)b * t.c[i].nI * t.c[i].nJ * nob;
  }
  const long long smax = std::max<long long>(1, std::min<long long>(kt / 4, 64));
  double best = 0.0;
  long long pick = 1;
  for (long long s = 1; s <= smax; ++s) {
    const double rounds = std::max((double)cdiv(blocks * s, 512) * 4.0 + work / 512.0,
                                   (double)cdiv(kt, s) + 4.0);
    const double idle = (double)cdiv(blocks * s, 512) * 512.0 / (blocks * s);
    const double cost = rounds * (t.n == 1 ? idle : 1.0) +
                        (s > 1 ? 2.0 + (double)s * numel / 1.5e6 : 0.0);
    if (s == 1 || cost < best) { best = cost; pick = s; }
  }
  return (int)pick;
}

// Images per pass of the tap GEMM (32-bit plane offsets, pixel counts and
// output indices), 0 when one image does not fit.
static int tap_images(const atx_conv_geom& g, int O) {
  const long long L = (long long)g.OH * g.OW, HW = (long long)g.H * g.W;
  const long long lim = 0x7fffffffLL - 4096;
  const long long n = std::min(std::min(lim / go_planes_bytes(L, O), lim / (HW * g.C)), lim / HW);
  return (int)std::min<long long>(n, g.N);
}

// 1e8 products, or (stride 1) 512 output tiles: a large image of few channels.
static bool tap_size(const atx_conv_geom& g, int O) {
  const double K = (double)g.C * g.KH * g.KW, P = (double)g.N * g.OH * g.OW;
  return P * O * K >= 1e8 ||
         (g.SH == 1 && g.SW == 1 && (double)g.N * g.H * g.W * cdiv(g.C, 64) >= 512 * 128);
}

// Times of the two ways to an image gradient in microseconds, least-squares
// fits to 220 convs (the 3x3 layers of the ResNets, small C or O, and random
// ones: kernels of 2 to 7, strides 1 and 2, dilations, C and O from 1 to 512),
// each with a bf16-exact and a general table; they are off by 14% and 13% (rms).
// Both count the padding they multiply.
//
// The tap GEMM pads C to a tile of 64 or 128 rows for each tap and go to 32
// channels: k-tile rounds (64 rows: two blocks per CU, 128: one), blocks, the
// planes (4 bytes read, 6 written and 6 read per value), gx with its mask and
// partials, and stride 2's scattered stores.
static double tap_cost(const atx_conv_geom& g, int O) {
  const TapClasses t = tap_classes(g);
  const double P = (double)g.N * g.OH * g.OW, img = (double)g.N * g.C * g.H * g.W;
  const long long nob = cdiv(O, BK), S = tap_splits(g, O);
  const long long slots = g.C <= 64 ? 512 : 256, mt = cdiv(g.C, g.C <= 64 ? 64 : 128);
  double blocks = 0.0, work = 0.0;
  for (int i = 0; i < t.n; ++i) {
    const double b = (double)cdiv((long long)g.N * t.c[i].Hc * t.c[i].Wc, 128) * mt;
    blocks += b;
    work += b * t.c[i].nI * t.c[i].nJ * nob / slots;
  }
  const double chain = (double)cdiv((long long)t.c[0].nI * t.c[0].nJ * nob, S);
  const double rounds = t.n == 1 ? std::ceil(blocks * S / slots) : 1.0;
  return 15.6 + 0.92 * std::max(work, chain * rounds) + 2.9 * blocks * S / slots +
         0.31e-6 * P * (4.0 * O + 192.0 * nob) + 0.18e-6 * img * (5.0 + (S > 1 ? 8.0 * S : 0.0)) +
         (t.n > 1 ? 3.2e-6 * img : 0.0);
}

// Share of a tile's rows and channels that are not padding.
static double tap_fill(const atx_conv_geom& g, int O) {
  const double tile = g.C <= 64 ? 64.0 : 128.0;
  return g.C / (std::ceil(g.C / tile) * tile) * O / (cdiv(O, BK) * (double)BK);
}

// The column GEMM pads C KH KW to its row tile (64 or 128) and O to 32; then
// the columns, written and folded (more per pixel with stride 2).
static double column_cost(const atx_conv_geom& g, int O) {
  const int K = g.C * g.KH * g.KW, L = g.OH * g.OW;
  const double P = (double)g.N * L, img = (double)g.N * g.C * g.H * g.W;
  const long long S = data_splits(g.N, O, K, L), nob = cdiv(O, BK);
  const double tile = tile_of(K) / 64.0;
  const double blocks = (double)cdiv((long long)g.N * L, 128) * cdiv(K, tile_of(K));
  return 13.7 + 0.42 * std::ceil(blocks * S / 512.0) * (cdiv(nob, S) + 4.0) * tile +
         0.79 * blocks * nob * tile / 512.0 + 0.04e-6 * P * O * 4.0 +
         0.22e-6 * (P * K * (4.0 + (S > 1 ? 8.0 * S : 0.0)) + 5.0 * img) +
         0.19e-6 * img * g.KH * g.KW + (g.SH > 1 || g.SW > 1 ? 1.0e-6 * img : 0.0);
}

// The tap GEMM serves convs of at least two taps, strides of 1 or 2 and
// tap_size() where the estimates above favour it; with tiles filled to 90%
// also where it is estimated up to 1.2 times as long, about the estimates'
// error, since it is the faster there more often (128 -> 256 with stride 2 at
// 16 x 16, batch 128: 66 against 77 us, both estimated 72).  A 1x1 conv's
// columns are its gradient, or (stride 2) most of its pixels have no tap: the
// column GEMM there reads go once per 128 rows and writes the result, which
// the go planes' pass does not beat (1024 -> 256 at 14 x 14, batch 64: 74
// against 85 us).  Below 1e8 products the extra launch costs more than the
// loop saves (1.8e6 to 5.5e6 products: 14-18 us against 17-19; 3e8: 27.5
// against 24.6).  Above, LRE tables, tap GEMM against column GEMM plus col2im:
// batch 64 at 56 x 56 x 64 137 / 296 us, 28 x 28 x 128 126 / 175, 14 x 14 x 256
// 129 / 139, 7 x 7 x 512 119 / 135, stride 2 at 56 x 56 x 128 205 / 242; few
// output channels (64 -> 8 at 56 x 56) 82 / 248.  The columns win where padding
// is most of the tap GEMM's work: 3 -> 64 at 64 x 64 125 / 38, 4 -> 512 1337 /
// 172, 7x7 stride 2 of 3 -> 64 at 224 x 224, batch 32 803 / 241, 24 -> 24 with
// stride 2 66 / 48.  Over 220 further random convs with both tables the tap
// GEMM wherever tap_size() holds takes 50.6 ms, the faster way of each 31.0
// and the rule's picks 31.7.
static bool tap_gemm(const atx_conv_geom& g, int O) {
  const long long K = (long long)g.C * g.KH * g.KW, L = (long long)g.OH * g.OW;
  return g.KH * g.KW > 1 && (g.SH == 1 || g.SH == 2) && (g.SW == 1 || g.SW == 2) && O > 0 &&
         g.N > 0 && K > 0 && L > 0 && g.H > 0 && g.W > 0 &&
         tap_size(g, O) && weight_planes_bytes((int)K, O) < 0x7fffffffLL &&
         (double)g.KH * g.KW * cdiv(O, BK) < 1e8 && cdiv(g.C, 64) <= 65535 &&
         cdiv(O, BK) <= 65535 && tap_images(g, O) > 0 &&
         tap_cost(g, O) < column_cost(g, O) * (tap_fill(g, O) >= 0.9 ? 1.2 : 1.0);
}

// Workspace of one pass: [weight planes][go planes][split partials].
static long long tap_workspace_bytes(const atx_conv_geom& g, int O) {
  const int S = tap_splits(g, O);
  return weight_planes_bytes(g.C * g.KH * g.KW, O) +
         (go_planes_bytes((long long)g.N * g.OH * g.OW, O) + 255) / 256 * 256 +
         (S > 1 ? (long long)S * g.N * g.C * g.H * g.W * 4 : 0);
}

static int run_tap_images(const float* go, const uint8_t* wq, const float* tx,
                        const atx_conv_geom& g, int O, const float* sx, const float* sw,
                        const uint8_t* mask, const float* scale, float* gx, char* ws,
                        hipStream_t stream) {
  const int KK = g.KH * g.KW, K = g.C * KK, L = g.OH * g.OW, P = g.N * L, HW = g.H * g.W;
  const int nob = (int)cdiv(O, BK), S = tap_splits(g, O);
  uint16_t* wplanes = (uint16_t*)ws;
  uint16_t* gplanes = (uint16_t*)(ws + weight_planes_bytes(K, O));
  float* partials = (float*)((char*)gplanes + (go_planes_bytes(P, O) + 255) / 256 * 256);
  int rc = launch_weight_planes(wq, tx, O, K, wplanes, stream);
  if (rc) return rc;
  hipLaunchKernelGGL(go_planes_kernel, dim3((unsigned)cdiv(P, 64), (unsigned)nob), dim3(256), 0,
                     stream, go, g.N, O, L, nob, sx, sw, gplanes);
  rc = check_launch("go_planes_kernel");
  if (rc) return rc;
  const TapClasses classes = tap_classes(g);
  const bool split = S > 1;
  float* out = split ? partials : gx;
  const long long numel = (long long)g.N * g.C * HW;
  DataOut ep{out, g.C, HW, g.N * HW, split ? nullptr : mask, split ? nullptr : scale, numel};
  TapArgs p{};
  p.wplanes = wplanes; p.gplanes = gplanes;
  p.wbytes = (int)weight_planes_bytes(K, O); p.gbytes = (int)go_planes_bytes(P, O);
  p.Kp = (int)(cdiv(K, 128) * 128); p.KK = KK; p.nOb = nob;
  p.splits = S; p.classes = classes; p.g = g;
  const bool vo = classes.n == 1 && HW % 4 == 0 && (uintptr_t)out % 16 == 0 &&
                  (split || (uintptr_t)mask % 4 == 0);
  long long ct = 0;
  for (int i = 0; i < classes.n; ++i)
    ct = std::max(ct, cdiv((long long)g.N * classes.c[i].Hc * classes.c[i].Wc, 128));
  const auto launch = [&](auto bm) {
    constexpr int BM = decltype(bm)::value;
    const dim3 grid((unsigned)ct, (unsigned)cdiv(g.C, BM), (unsigned)(classes.n * S));
    if (vo)
      hipLaunchKernelGGL((tap_planes_kernel<BM, true>), grid, dim3(BM * 4), 0, stream, p, ep, tx);
    else
      hipLaunchKernelGGL((tap_planes_kernel<BM, false>), grid, dim3(BM * 4), 0, stream, p, ep, tx);
  };
  if (g.C <= 64) launch(std::integral_constant<int, 64>{});
  else launch(std::integral_constant<int, 128>{});
  rc = check_launch("tap_planes_kernel");
  if (rc || !split) return rc;
  return launch_split_sum(partials, S, numel, (int)numel, mask, scale, gx, stream);
}

// Images of the next pass over g.N: at most tap_images(); and when the last
// round of blocks would be nearly empty, only those that fill the rounds
// before it, so that the rest, a pass with a split contraction, ends sooner
// (128 x 128 x 28 x 28, 3.06 rounds: 252 -> 225 us; 83 x 100 x 30 x 30, 2.28
// rounds: 179 -> 164).
static int tap_pass(const atx_conv_geom& g, int O) {
  atx_conv_geom part = g;
  part.N = tap_images(g, O);
  if (g.SH > 1 || g.SW > 1) return part.N;           // classes of unequal depth share the rounds
  const long long HW = (long long)g.H * g.W;
  const long long slots = g.C <= 64 ? 512 : 256, mt = cdiv(g.C, g.C <= 64 ? 64 : 128);
  const long long full = cdiv(part.N * HW, 128) * mt / slots;
  const long long n = full * slots / mt * 128 / HW;
  if (full < 1 || n < 1 || n >= part.N || tap_splits(part, O) > 1) return part.N;
  const double whole = tap_cost(part, O);
  atx_conv_geom tail = g;
  tail.N = part.N - (int)n;
  part.N = (int)n;
  return tap_cost(part, O) + tap_cost(tail, O) < whole ? part.N : part.N + tail.N;
}

// All images, in passes.
static int run_tap_gemm(const float* go, const uint8_t* wq, const float* tx, atx_conv_geom g,
                        int O, const float* sx, const float* sw, const uint8_t* mask,
                        const float* scale, float* gx, char* ws, hipStream_t stream) {
  const long long gi = (long long)O * g.OH * g.OW, xi = (long long)g.C * g.H * g.W;
  const int N = g.N;
  for (int n = 0; n < N;) {
    g.N = N - n;
    g.N = tap_pass(g, O);
    const int rc = run_tap_images(go + n * gi, wq, tx, g, O, sx, sw, mask ? mask + n * xi : nullptr,
                                  scale, gx + n * xi, ws, stream);
    if (rc) return rc;
    n += g.N;
  }
  return ATX_OK;
}

}  // namespace atx

using namespace atx;

extern "C" {

int atx_conv_bwd_data_col(const float* go, const uint8_t* wq, const float* tx, int N, int O,
                          int K, int L, float* col, hipStream_t stream) {
  ATX_REQUIRE(N >= 0 && O >= 0 && K >= 0 && L >= 0, "atx_conv_bwd_data_col: negative size");
  if ((long long)N * K * L == 0) return ATX_OK;
  ATX_REQUIRE(col, "atx_conv_bwd_data_col: null output");
  if (O == 0) {
    // Empty contraction: the split-sum kernel with S = 0 writes zeros.
    return launch_split_sum(nullptr, 0, (long long)N * K * L, K, nullptr, nullptr, col, stream);
  }
  ATX_REQUIRE(go && wq && tx, "atx_conv_bwd_data_col: null pointer");
  ATX_REQUIRE((long long)N * L < 0x7fffffffLL && cdiv(K, 64) <= 65535,
              "atx_conv_bwd_data_col: sizes too large");
  // no workspace here: the fp32 kernels (table lookups in the loaders)
  const DataArgs a{go, wq, tx, N, O, K, L, nullptr, nullptr, col, nullptr, nullptr, 1, 0,
                   nullptr, nullptr};
  return run_data_gemm(a, stream);
}

// A 1x1, stride-1, unpadded conv's columns are its image gradient.
static bool direct_columns(const atx_conv_geom& g) {
  return g.KH == 1 && g.KW == 1 && g.SH == 1 && g.SW == 1 && g.PH == 0 && g.PW == 0;
}

// A padded 1x1, stride-1 conv's columns inside the image are its gradient: the
// GEMM reads go's positions there (scalar loads).  Against columns and col2im,
// 64 x 64 x 56 x 56 -> 64 with padding 1: 65 -> 43 us, 64 x 256 x 28 x 28 ->
// 256: 97 -> 78.
static bool cropped_columns(const atx_conv_geom& g, int O) {
  return g.KH == 1 && g.KW == 1 && g.SH == 1 && g.SW == 1 && !direct_columns(g) && g.H > 0 &&
         g.W > 0 && planes_fit((long long)g.H * g.W, O, (long long)g.OH * g.OW);
}

// Workspace of atx_conv_bwd_data: [bf16 weight planes][split partials][col
// (unless direct or cropped)], or the tap GEMM's (tap_workspace_bytes).
long long atx_conv_bwd_data_workspace_bytes(atx_conv_geom g, int O) {
  const int K = g.C * g.KH * g.KW, L = g.OH * g.OW;
  if (g.N <= 0 || K <= 0 || L <= 0 || O <= 0) return 0;
  const long long planes = weight_planes_bytes(K, O);
  if (tap_gemm(g, O)) {
    long long bytes = 0;
    for (int n = g.N; n > 0;) {            // the passes of run_tap_gemm
      g.N = n;
      g.N = tap_pass(g, O);
      bytes = std::max(bytes, tap_workspace_bytes(g, O));
      n -= g.N;
    }
    return bytes;
  }
  const bool crop = cropped_columns(g, O);
  const int Lc = crop ? g.H * g.W : L;
  const long long numel = (long long)g.N * K * Lc;
  const int S = data_splits(g.N, O, K, Lc);
  return planes + ((S > 1 ? S : 0) + (crop || direct_columns(g) ? 0 : 1)) * numel * 4;
}

int atx_conv_bwd_data(const float* go, const uint8_t* wq, const float* tx, atx_conv_geom g,
                      int O, const float* go_sx, const float* go_sw, const uint8_t* mask,
                      const float* scale, float* gx, float* workspace, hipStream_t stream) {
  ATX_REQUIRE(O >= 0 && g.N >= 0 && g.C >= 0 && g.H >= 0 && g.W >= 0 && g.KH > 0 && g.KW > 0,
              "atx_conv_bwd_data: bad geometry");
  ATX_REQUIRE((go_sx == nullptr) == (go_sw == nullptr),
              "atx_conv_bwd_data: go_sx and go_sw come together");
  ATX_REQUIRE(!mask || scale, "atx_conv_bwd_data: mask needs scale");
  const long long img = (long long)g.N * g.C * g.H * g.W;
  if (img == 0) return ATX_OK;
  ATX_REQUIRE(gx, "atx_conv_bwd_data: null output");
  const int K = g.C * g.KH * g.KW;
  const int L = g.OH * g.OW;
  // the bf16 weight planes lead the workspace (absent when O, K or L is 0)
  uint16_t* planes = nullptr;
  float* rest = workspace;
  if (O > 0 && K > 0 && L > 0) {
    ATX_REQUIRE(workspace, "atx_conv_bwd_data: null workspace");
    planes = (uint16_t*)workspace;
    rest = (float*)((char*)workspace + weight_planes_bytes(K, O));
  }
  if (tap_gemm(g, O)) {
    ATX_REQUIRE(go && wq && tx, "atx_conv_bwd_data: null pointer");
    return run_tap_gemm(go, wq, tx, g, O, go_sx, go_sw, mask, scale, gx, (char*)workspace, stream);
  }
  const bool crop = O > 0 && L > 0 && cropped_columns(g, O);
  const int Lc = crop ? g.H * g.W : L;
  const long long numel = (long long)g.N * K * Lc;
  const int S = (O > 0 && numel > 0) ? data_splits(g.N, O, K, Lc) : 1;
  float* partials = S > 1 ? rest : nullptr;
  float* col = rest ? rest + (S > 1 ? S * numel : 0) : nullptr;
  ATX_REQUIRE(S == 1 || rest, "atx_conv_bwd_data: null workspace");
  if (crop || direct_columns(g)) {
    if (O == 0 || L == 0)
      return launch_split_sum(nullptr, 0, img, 1, nullptr, nullptr, gx, stream);
    ATX_REQUIRE(go && wq && tx, "atx_conv_bwd_data: null pointer");
    ATX_REQUIRE((long long)g.N * L < 0x7fffffffLL && cdiv(K, 64) <= 65535,
                "atx_conv_bwd_data: sizes too large");
    const DataArgs a{go, wq, tx, g.N, O, K, L, go_sx, go_sw, gx, mask, scale, S, 0, partials,
                     planes, crop ? &g : nullptr};
    return run_data_gemm(a, stream);
  }
  ATX_REQUIRE(rest, "atx_conv_bwd_data: null workspace");
  if ((long long)K * L == 0 || O == 0) {
    if (numel) {
      int rc = launch_split_sum(nullptr, 0, numel, 1, nullptr, nullptr, col, stream);
      if (rc) return rc;
    }
  } else {
    ATX_REQUIRE(go && wq && tx, "atx_conv_bwd_data: null pointer");
    ATX_REQUIRE((long long)g.N * L < 0x7fffffffLL && cdiv(K, 64) <= 65535,
                "atx_conv_bwd_data: sizes too large");
    const DataArgs a{go, wq, tx, g.N, O, K, L, go_sx, go_sw, col, nullptr, nullptr, S, 0,
                     partials, planes};
    int rc = run_data_gemm(a, stream);
    if (rc) return rc;
  }
  return atx_col2im(col, g, mask, scale, gx, stream);
}

long long atx_conv_bwd_weight_workspace_bytes(int O, int K, long long P) {
  if (O <= 0 || K <= 0 || P <= 0) return 0;
  return (long long)weight_splits(O, K, P) * O * K * 4;
}

int atx_conv_bwd_weight(const float* go, const void* img, int dtype, atx_conv_geom g, int O,
                        int pad_index, const float* pad_dev, const float* tw,
                        const float* go_sx, const float* go_sw,
                        const uint8_t* mask_w, const float* scale_w, float* gw,
                        float* workspace, hipStream_t stream) {
  ATX_REQUIRE(O >= 0 && dtype >= 0 && dtype <= 3, "atx_conv_bwd_weight: bad arguments");
  ATX_REQUIRE((go_sx == nullptr) == (go_sw == nullptr),
              "atx_conv_bwd_weight: go_sx and go_sw come together");
  const int f32_offset = dtype == 3 ? 0 : 128;   // 3: fp32 unsigned quantized values
  if (dtype == 3) dtype = 2;
  ATX_REQUIRE(pad_index >= 0 && pad_index <= 255, "atx_conv_bwd_weight: bad pad_index");
  const int K = g.C * g.KH * g.KW;
  const int L = g.OH * g.OW;
  const long long P = (long long)g.N * L;
  ATX_REQUIRE(P < 0x7fffffffLL, "atx_conv_bwd_weight: N*L too large");
  if ((long long)O * K == 0) return ATX_OK;
  ATX_REQUIRE(gw && tw && (!mask_w || scale_w), "atx_conv_bwd_weight: null pointer");
  if (P == 0) {
    // Empty contraction: the split-sum kernel with S = 0 writes zeros.
    return launch_split_sum(nullptr, 0, (long long)O * K, K, nullptr, scale_w, gw, stream);
  }
  ATX_REQUIRE(go && img && workspace, "atx_conv_bwd_weight: null operand/workspace");
  ATX_REQUIRE(cdiv(O, 64) <= 65535, "atx_conv_bwd_weight: too many output channels");
  ATX_REQUIRE((long long)O * L < (1LL << 28), "%s: one image's output gradient exceeds 1 GiB",
              __func__);
  const int S = weight_splits(O, K, P);
  const int chunk = (int)(cdiv(cdiv(P, S), BK) * BK);
  const int Sreal = (int)cdiv(P, chunk);
  if (dtype == 0)
    dispatch_weight<int8_t>(go, (const int8_t*)img, g, O, K, L, (int)P, chunk, Sreal, 128,
                            pad_index, pad_dev, tw, go_sx, go_sw, workspace, stream);
  else if (dtype == 1)
    dispatch_weight<uint8_t>(go, (const uint8_t*)img, g, O, K, L, (int)P, chunk, Sreal, 0,
                             pad_index, pad_dev, tw, go_sx, go_sw, workspace, stream);
  else
    dispatch_weight<float>(go, (const float*)img, g, O, K, L, (int)P, chunk, Sreal,
                           f32_offset, pad_index, pad_dev, tw, go_sx, go_sw, workspace, stream);
  int rc = check_launch("weight_gemm_kernel");
  if (rc) return rc;
  return launch_split_sum(workspace, Sreal, (long long)O * K, K, mask_w, scale_w, gw, stream);
}

int atx_conv_bwd_weight_rows(const float* go, const uint16_t* xt, int Rpad, int N, int K,
                             int L, int O, const float* tw, const float* go_sx,
                             const float* go_sw, const uint8_t* mask_w, const float* scale_w,
                             float* gw, float* workspace, hipStream_t stream) {
  ATX_REQUIRE(N >= 0 && K >= 0 && L >= 0 && O >= 0, "atx_conv_bwd_weight_rows: negative size");
  ATX_REQUIRE((go_sx == nullptr) == (go_sw == nullptr),
              "atx_conv_bwd_weight_rows: go_sx and go_sw come together");
  const long long P = (long long)N * L;
  ATX_REQUIRE(P < 0x7fffffffLL, "atx_conv_bwd_weight_rows: N*L too large");
  ATX_REQUIRE(Rpad >= P && Rpad % ATX_ROW_TILE == 0, "atx_conv_bwd_weight_rows: bad Rpad %d",
              Rpad);
  if ((long long)O * K == 0) return ATX_OK;
  ATX_REQUIRE(gw && tw && (!mask_w || scale_w), "atx_conv_bwd_weight_rows: null pointer");
  if (P == 0)
    return launch_split_sum(nullptr, 0, (long long)O * K, K, nullptr, scale_w, gw, stream);
  ATX_REQUIRE(go && xt && workspace, "atx_conv_bwd_weight_rows: null operand/workspace");
  ATX_REQUIRE(cdiv(O, 64) <= 65535, "atx_conv_bwd_weight_rows: too many output channels");
  ATX_REQUIRE((long long)O * L < (1LL << 28), "%s: one image's output gradient exceeds 1 GiB",
              __func__);
  const int S = weight_splits(O, K, P);
  const int chunk = (int)(cdiv(cdiv(P, S), BK) * BK);
  const int Sreal = (int)cdiv(P, chunk);
  if (L % 4 == 0 && (uintptr_t)go % 16 == 0)
    dispatch_weight_rows<true>(go, xt, Rpad, O, K, L, (int)P, chunk, Sreal, tw, go_sx, go_sw,
                               workspace, stream);
  else
    dispatch_weight_rows<false>(go, xt, Rpad, O, K, L, (int)P, chunk, Sreal, tw, go_sx, go_sw,
                                workspace, stream);
  int rc = check_launch("weight_gemm_kernel<rows>");
  if (rc) return rc;
  return launch_split_sum(workspace, Sreal, (long long)O * K, K, mask_w, scale_w, gw, stream);
}

}  // extern "C"
