// LUT GEMM forward for gfx950: y[n,o,l] = sum_k LUT[xi(n,k,l)][wi(o,k)].
//
// Kernel structure ("expanded tables" in byte planes, added by the matrix
// cores):
//   A workgroup owns a tile of ATX_ROW_TILE (2048) rows r = n*L + l and
//   ATX_COL_TILE (32) output channels.  For every k it builds, in LDS, the
//   table E_k[v][o] = LUT16[v][wi(o,k)] (256 rows x 32 channels) from the
//   transposed 16-bit LUT image (L2-resident, 128 KiB), each row as two
//   16-channel chunks of high bytes and two of low bytes.  A lane looks a
//   row's 16 channels up with two 16-byte LDS reads, and one sparse matrix
//   product (v_smfmac_i32_16x16x128_i8) adds them: its 4:2-sparse operand is a
//   fixed selection matrix (row i picks byte i of every chunk, weighted by the
//   plane), so 64 lanes' 32 bytes - 16 rows x 4 taps x 16 channels x 2 planes
//   - go into 16 x 16 int32 sums.  The high plane's weight 256 does not fit an
//   int8, so a second product adds the high bytes once more (-128 each).
//
//   What bounds it: the LDS reads (2 bytes per lookup; conflict-free 16-byte
//   reads measure 122 TB/s = 61 T lookups/s), then the table build.  Reads
//   plus both products measure 44-46 T lookups/s; with one VALU add per
//   lookup in their place (packed pairs, 1.26 VALU instructions per lookup)
//   the same loop measured 30.7 T.  Whole kernel, K = 2304, 65536 rows x 64
//   channels: 537 -> 406 us with upper-half tables (24 T), 558 -> 441 us with
//   full ones; K = 1024, 12544 x 256: 201 -> 145 us; K = 64, 200704 x 256: 222
//   -> 167 us.  Timed copies (100352 x 128, K = 1152, full tables, 650 us):
//   without the LUT-row loads 505, without the table writes as well 410.  The
//   LUT rows (64 KiB per quad from L1 / L2 at 64 bytes a clock) and the LDS
//   reads do not overlap fully; that is what is left.
//
//   LDS layout.  gfx950's LDS has 64 banks (256 bytes per clock); it serves a
//   16-byte read in passes of 16 lanes, 0-3, 12-15 and 20-27 the first, then
//   4-11, 16-19 and 28-31, and the same of the upper half.  Four consecutive
//   tables share each 256-byte line: line v holds row v of tap t in quarter t
//   (channel half cg at + 32, plane at + 16; 0 = high).  Lane (j, g) = (lane &
//   15, lane >> 4) reads tap (j & 3) ^ g, channel half (j >> 3) ^ c and plane
//   (g & 1) ^ h in its read (c, h): the lanes of a pass read sixteen different
//   positions of a line, whatever their rows, so no two share a bank.  The
//   activation operand is pre-encoded as the byte offset v*256 + ((v >> 1) &
//   3)*16 ("row offset"), of which this kernel takes the byte v: one v_perm
//   puts it above the lane's position bits.
//
//   Table build: two quad buffers (128 KiB).  While quad j is read, the wave
//   transposes its share of quad j+1 (entries loaded during quad j-1) with
//   v_perm into chunks, stores them, and then loads the entries of quad j+2,
//   one channel per two reads: a burst of sixteen loads at one place stalled
//   the wave's reads behind the address unit (c. 15% of the kernel).  A wave
//   builds one tap; its lanes cover 128 consecutive rows of both channel
//   halves, so a load instruction touches two LUT rows (eight rows of 64 bytes
//   each measured twice the time), and the four lanes of a store pass write
//   four different positions (two halves, planes in the order of lane bit 0).
//   One barrier per quad (four k-steps) orders build and reads.
//
//   Threads: 512 (8 waves, 2 per SIMD).  Wave w owns rows 256w .. 256w+255 of
//   the tile; lane (j, g) the rows 64h + 4j + m (h, m = 0..3) x 8 channels =
//   128 int32 accumulators of its 256 registers.  Four consecutive rows per
//   lane let the epilogue store every (channel, h) as one 16-byte vector,
//   eight lanes one 128-byte line (sixteen consecutive rows per lane, 16-byte
//   pieces 64 bytes apart, measured 10-40% slower).
//
// Reference: bgemm_lut_u8_kernel / bgemm_mainloop
// (csrc/claude/bgemm_lut_kernels.cuh:183-387) computes the same sum with a
// 16-bit LUT gathered through L1 and fp32 accumulation.

#include "atx_internal.h"
#include "atx_tiles.h"

#include <algorithm>
#include <mutex>
#include <stdlib.h>
#include <string.h>
#include <type_traits>

namespace atx {

constexpr int RT = ATX_ROW_TILE;   // rows per workgroup (2048)
constexpr int OT = ATX_COL_TILE;   // channels per workgroup (32)
constexpr int RPL = 16;            // rows per lane
constexpr int RPW = 16 * RPL;      // rows per wave (256)
constexpr int NWAVE = RT / RPW;    // waves per workgroup (8)
constexpr int NT = 64 * NWAVE;     // threads per workgroup (512)
constexpr int TPL = 4;             // tables per LDS line (quarters)
constexpr int LINE = 256;          // bytes per LDS line
constexpr int QTAB = 256 * LINE;   // one quad of tables (64 KiB)
constexpr int SMEM_BYTES = 2 * QTAB;          // two quad buffers (128 KiB)
static_assert(QTAB == 1 << 16, "quad buffer select is bit 16 of a read address");
static_assert(OT == 32 && NWAVE == 8, "tile geometry");
static_assert(TPL * OT * 2 == LINE, "four 64-byte table rows per line");

// K limit of exact int32 partial sums (entries up to 65535).
constexpr int KMAX_U16 = 32768;

struct GemmParams {
  const uint16_t* xt; int Rpad;
  const uint8_t* wt; int Opad;
  const uint16_t* lut16t;
  const float* lutf32t;
  int K, R, L, O;
  int k_chunk, splits, tiles_r, tiles_o;
  // Rows per tile: RT, or fewer (a multiple of RPW) when R / RT leaves the
  // last tile mostly empty, so every tile carries about R / tiles_r rows.
  // Waves whose rows lie past the tile (wave * RPW >= rt) build tables but
  // accumulate and store nothing.
  int rt;
  int out_kind;                 // ATX_OUT_*; splits > 1 => raw int32 partials
  void* y;
  long long split_stride;       // elements per partial slice
  const float* sx; const float* sw; const float* bias;
  // Stream-K schedule (sk_per > 0) of G workgroups: workgroup w first runs
  // the whole tiles w, w + G, ... below sk_dp (sk_dp = G * full rounds),
  // then quads [w * sk_per, (w + 1) * sk_per) of the tile-major (tile, quad)
  // space of the remaining tiles, nqt quads per tile; a remaining tile cut by
  // a workgroup boundary adds its int32 sums into slot
  // floor(tail tile * nqt / sk_per) of skws.
  int sk_per, nqt, sk_dp, sk_g;
  int* skws;
  // Device flag (or null): nonzero when every activation index of the rows
  // below R is at least 128 (x >= 0 before an int8 fake-quant).  The tables
  // are then built for rows 128..255 only (upper-half tables).
  const int* x_upper;
  bool sgn;                     // signed (int16) table entries
};

// ------------------------------------------------------------------ prepare
__global__ void lut_prepare_kernel(const float* __restrict__ lut,
                                   uint16_t* __restrict__ out16t,
                                   float* __restrict__ outf32t,
                                   int* __restrict__ flags) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;   // 65536 entries
  const float v = lut[i];
  const float r = __builtin_rintf(v);
  const bool is_int = (v == r);
  const bool ok16 = is_int && fabsf(v) <= 32767.0f;
  const bool oku16 = is_int && v >= 0.0f && v <= 65535.0f;
  if (!ok16) flags[0] = 1;     // benign race: every writer stores 1
  if (!oku16) flags[1] = 1;
  const unsigned short v16 =
      (ok16 || oku16) ? (unsigned short)(unsigned)(int)r : (unsigned short)0;
  const int t = ((i & 255) << 8) | (i >> 8);             // [x][w] -> [w][x]
  out16t[t] = v16;
  outf32t[t] = v;
}

// ------------------------------------------------------------- operand pack
// xt[slot][r] = row_offset(x[n][operand_tap(slot, r)][l]) for r < R
// (r = n*L + l); 0 for r >= R and taps >= K.  The four rows of a quad (one tap)
// are one 8-byte store; when L % 4 == 0 the quad is four consecutive elements
// of one x row, read with one 4- (u8) or 16-byte (fp32) load (`vec`: L % 4 ==
// 0 and the pointers aligned for it).
//
// A thread owns one quad of rows and one quad of slots (blockIdx.y = slot
// quad): the four taps' loads are in flight together and go out as four
// 8-byte pieces.  Bound by HBM: 4 (fp32) or 1 byte read, 2 written per element
// and 1 more for the fp32 operand's index image.  16 x 1152 x 784 fp32: 52 us
// with one tap per thread, 25 us now (4.0 TB/s); the u8 operand 3.6 -> 6 TB/s.
template <typename T>
__global__ void __launch_bounds__(256)
pack_x_quads_kernel(const T* __restrict__ x, int N, int K, int L, int offset,
                    uint8_t* __restrict__ xq, uint16_t* __restrict__ xt, int Rpad, bool vec,
                    int* __restrict__ upper) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= (Rpad >> 2)) return;
  const int R = N * L;
  const int r0 = q << 2;
  long long base[4];
  unsigned valid = 0;
  if (R > 0) {
    const int rr = min(r0, R - 1);
    int n = rr / L, l = rr - n * L;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (r0 + e < R) valid |= 1u << e;
      base[e] = (long long)n * K * L + l;
      if (++l == L) { l = 0; ++n; }
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) base[e] = 0;
  }
  bool low = false;             // some index of rows < R and taps < K is < 128
  for (int k4 = blockIdx.y * 4; k4 < K; k4 += gridDim.y * 4) {
    unsigned v[4];                                 // the taps' four indices, a byte each
    if constexpr (sizeof(T) == 4) {
      float f[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k4 | ((q + u) & 3);          // this quad's tap of slot k4 + u
        const long long kl = (long long)min(k, K - 1) * L;
        if (vec) {
          float4 w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (k < K && valid) w = *(const float4*)(x + base[0] + kl);
          f[u][0] = w.x; f[u][1] = w.y; f[u][2] = w.z; f[u][3] = w.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) f[u][e] = k < K && ((valid >> e) & 1u) ? x[base[e] + kl] : 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        v[u] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u] |= quant_index(f[u][e], offset) << (8 * e);
        const int k = k4 | ((q + u) & 3);
        if (xq && k < K && valid) {
          const long long kl = (long long)k * L;
          if (vec) {
            *(unsigned*)(xq + base[0] + kl) = v[u];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if ((valid >> e) & 1u) xq[base[e] + kl] = (uint8_t)(v[u] >> (8 * e));
          }
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k4 | ((q + u) & 3);
        const long long kl = (long long)min(k, K - 1) * L;
        if (vec) {
          v[u] = (k < K && valid) ? *(const unsigned*)(x + base[0] + kl) : 0u;
        } else {
          v[u] = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (k < K && ((valid >> e) & 1u)) v[u] |= (unsigned)x[base[e] + kl] << (8 * e);
        }
      }
    }
    uint16_t* dst = xt + (long long)k4 * Rpad + r0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k4 | ((q + u) & 3);
      unsigned off[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool live = k < K && ((valid >> e) & 1u);
        const unsigned idx = (v[u] >> (8 * e)) & 255u;
        off[e] = live ? row_offset(idx) : 0u;
        low |= live && idx < 128u;
      }
      *(uint2*)(dst + (long long)u * Rpad) =
          make_uint2(off[0] | (off[1] << 16), off[2] | (off[3] << 16));
    }
  }
  if (upper && low) upper[0] = 0;        // benign race: every writer stores 0
}

// Strided operands of the plain (torch.mm-layout) LUT GEMM.  Row operand:
// X[r][k] at X + r*sr + k*sk -> xt[slot][r] = row_offset(index), as pack_x
// (quads of rows share a tap); column operand: Y[c][k] at Y + c*sc + k*sk ->
// wt[k][c] = index.  index = clamp(rint(v) + offset, 0, 255) for fp32, the
// byte for uint8; the optional u8 images get q[r*K + k] / q[c*K + k].
template <typename T>
__global__ void pack_rows_strided_kernel(const T* __restrict__ x, int R, int K, long long sr,
                                         long long sk, int offset, uint8_t* __restrict__ xq,
                                         uint16_t* __restrict__ xt, int Rpad,
                                         int* __restrict__ upper) {
  const int q0 = blockIdx.x * blockDim.x + threadIdx.x;
  const int qstride = gridDim.x * blockDim.x;
  const int nquad = Rpad >> 2;
  bool low = false;             // some index of rows < R and taps < K is < 128
  for (int slot = blockIdx.y; slot < operand_rows(K); slot += gridDim.y) {
    const int k = operand_tap(slot, q0 << 2);
    uint16_t* dst = xt + (long long)slot * Rpad;
    for (int q = q0; q < nquad; q += qstride) {
      const int r0 = q << 2;
      unsigned off[4] = {0u, 0u, 0u, 0u};
      if (k < K) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = r0 + e;
          if (r < R) {
            unsigned v;
            if constexpr (sizeof(T) == 4) v = quant_index((float)x[r * sr + k * sk], offset);
            else v = (unsigned)x[r * sr + k * sk];
            if (xq) xq[(long long)r * K + k] = (uint8_t)v;
            off[e] = row_offset(v);
            low |= v < 128u;
          }
        }
      }
      *(uint2*)(dst + r0) = make_uint2(off[0] | (off[1] << 16), off[2] | (off[3] << 16));
    }
  }
  if (upper && low) upper[0] = 0;        // benign race: every writer stores 0
}

template <typename T>
__global__ void pack_cols_strided_kernel(const T* __restrict__ y, int C, int K, long long sc,
                                         long long sk, int offset, uint8_t* __restrict__ yq,
                                         uint8_t* __restrict__ wt, int Opad) {
  const long long total = (long long)K * Opad;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const int k = (int)(i / Opad);
    const int c = (int)(i - (long long)k * Opad);
    unsigned v = 0;
    if (c < C) {
      if constexpr (sizeof(T) == 4) v = quant_index((float)y[c * sc + k * sk], offset);
      else v = (unsigned)y[c * sc + k * sk];
      if (yq) yq[(long long)c * K + k] = (uint8_t)v;
    }
    wt[i] = (uint8_t)v;
  }
}

// The strided packs of operands contiguous along k (a linear layer's weight
// [N, K], activations [M, K]): rows are far apart in memory, so lanes read along
// k and a 64 x 64 tile of indices is turned in LDS; both sides then move whole
// lines.  4096 x 1024 fp32: 34 -> 8.9 us; the columns of 1000 x 1024: 10.8 -> 5.5.
constexpr int TT = 64;                 // tile side
constexpr int TP = TT + 4;             // LDS bytes per tile row

// tile[i][k] = index of X[i0 + i][k0 + k] (0 past R, K), the u8 image on the way.
template <typename T>
__device__ __forceinline__ void load_tile(unsigned char* tile, const T* __restrict__ x, int R,
                                          int K, long long sr, int i0, int k0, int offset,
                                          uint8_t* __restrict__ xq) {
  const int k = threadIdx.x & 63, k1 = k0 + k, i1 = threadIdx.x >> 6;
  const T* src = x + (long long)(i0 + i1) * sr + k1;
  uint8_t* dq = xq + (long long)(i0 + i1) * K + k1;
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
    unsigned v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = i0 + i1 + 4 * (8 * h + j);
      v[j] = 0;
      if (r < R && k1 < K) {
        if constexpr (sizeof(T) == 4) v[j] = __float_as_uint(*src);
        else v[j] = *src;
      }
      src += 4 * sr;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = i1 + 4 * (8 * h + j);
      const bool live = i0 + i < R && k1 < K;
      if constexpr (sizeof(T) == 4) v[j] = live ? quant_index(__uint_as_float(v[j]), offset) : 0u;
      if (xq && live) *dq = (uint8_t)v[j];
      dq += 4LL * K;
      tile[i * TP + k] = (unsigned char)v[j];
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
pack_rows_turned_kernel(const T* __restrict__ x, int R, int K, long long sr, int offset,
                        uint8_t* __restrict__ xq, uint16_t* __restrict__ xt, int Rpad,
                        int* __restrict__ upper) {
  __shared__ unsigned char tile[TT * TP];
  const int r0 = blockIdx.x * TT, k0 = blockIdx.y * TT;
  load_tile(tile, x, R, K, sr, r0, k0, offset, xq);
  __syncthreads();
  const int rq = threadIdx.x & 15, k4 = (threadIdx.x >> 4) * 4;      // row quad, tap quad
  const int q = (r0 >> 2) + rq;
  if (k0 + k4 >= operand_rows(K)) return;
  bool low = false;             // some index of rows < R and taps < K is < 128
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int k = k4 | ((q + u) & 3);            // this quad's tap of slot k4 + u
    unsigned off[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool live = r0 + 4 * rq + e < R && k0 + k < K;
      const unsigned idx = tile[(4 * rq + e) * TP + k];
      off[e] = live ? row_offset(idx) : 0u;
      low |= live && idx < 128u;
    }
    *(uint2*)(xt + (long long)(k0 + k4 + u) * Rpad + r0 + 4 * rq) =
        make_uint2(off[0] | (off[1] << 16), off[2] | (off[3] << 16));
  }
  if (upper && low) upper[0] = 0;        // benign race: every writer stores 0
}

template <typename T>
__global__ void __launch_bounds__(256)
pack_cols_turned_kernel(const T* __restrict__ y, int C, int K, long long sc, int offset,
                        uint8_t* __restrict__ yq, uint8_t* __restrict__ wt, int Opad) {
  __shared__ unsigned char tile[TT * TP];
  const int c0 = blockIdx.x * TT, k0 = blockIdx.y * TT;
  load_tile(tile, y, C, K, sc, c0, k0, offset, yq);
  __syncthreads();
  const int c4 = (threadIdx.x & 15) * 4;
  if (c0 + c4 >= Opad) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int k = (threadIdx.x >> 4) + 16 * j;
    if (k0 + k >= K) break;
    unsigned v = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) v |= (unsigned)tile[(c4 + e) * TP + k] << (8 * e);
    *(unsigned*)(wt + (long long)(k0 + k) * Opad + c0 + c4) = v;
  }
}

template <typename T>
__global__ void pack_w_kernel(const T* __restrict__ w, int O, int K, int offset,
                              uint8_t* __restrict__ wq, uint8_t* __restrict__ wt,
                              int Opad) {
  const long long total = (long long)K * Opad;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const int k = (int)(i / Opad);
    const int o = (int)(i - (long long)k * Opad);
    unsigned v = 0;
    if (o < O) {
      const long long src = (long long)o * K + k;
      if constexpr (sizeof(T) == 4) {
        v = quant_index((float)w[src], offset);
        if (wq) wq[src] = (uint8_t)v;
      } else {
        v = (unsigned)w[src];
      }
    }
    if (wt) wt[i] = (uint8_t)v;
  }
}

// ------------------------------------------------------------- main kernel
using v4i = int __attribute__((ext_vector_type(4)));
using v8i = int __attribute__((ext_vector_type(8)));

constexpr int RD = 4;              // table reads (32-byte pairs) in flight per lane
static_assert(8 % RD == 0, "a row quad's reload follows a whole ring");

// The lane's accumulators: acc[4 h + m][c][q] is row 64 h + 4 j + m of the
// wave, channel 16 ((j >> 3) ^ c) + 4 g + q of the tile (j = lane & 15, g =
// lane >> 4).
using Acc = v4i[RPL][2];

// Selection operand of the sparse matrix product (16 x 128, 4:2 sparse):
// row i has one entry in each of the 16-byte chunks a lane group reads, at
// byte i, so the product adds, for every channel i, the chunks' bytes i of
// the four lane groups.  The weights undo the byte split: a high byte counts
// -256 (two products of -128: an int8 holds no 256) and a low byte -1.
// Lane group g and register half h of the table operand hold plane
// (g & 1) ^ h (0 high, 1 low).  In the instruction's layout lane group ga of
// this operand covers half ga >> 1, lane group 2 (ga & 1) in its bytes 0-7
// and 2 (ga & 1) + 1 in bytes 8-15; a group of four k has two value slots,
// whose positions are in idx.
struct Select { v4i both, high; int idx; };

__device__ __forceinline__ Select make_select(int lane) {
  const int i = lane & 15, half = lane >> 5, pos = i & 3;
  const int shift = 8 * (2 * ((i >> 2) & 1) + (pos == 3));
  const unsigned hi = 0x80u << shift;                   // -128
  const unsigned lo = 0xffu << shift;                   // -1
  const unsigned b0 = half ? lo : hi, b1 = half ? hi : lo;
  const unsigned h0 = half ? 0u : hi, h1 = half ? hi : 0u;
  const bool up = (i >> 3) != 0;
  Select s;
  s.both = v4i{up ? 0 : (int)b0, up ? (int)b0 : 0, up ? 0 : (int)b1, up ? (int)b1 : 0};
  s.high = v4i{up ? 0 : (int)h0, up ? (int)h0 : 0, up ? 0 : (int)h1, up ? (int)h1 : 0};
  s.idx = (int)(((pos < 3 ? (unsigned)pos : 0u) | 12u) * 0x11111111u);
  return s;
}

// Byte code of a table entry: the 16-bit entry with its low byte (and, for
// unsigned tables, its high byte) offset to a signed byte.  Summed with the
// weights above T entries give -(sum - code_bias T).
__device__ __forceinline__ unsigned code_xor(bool sgn) { return sgn ? 0x00800080u : 0x80808080u; }
__device__ __forceinline__ int code_bias(bool sgn) { return sgn ? 128 : 32768 + 128; }

// LUT16T entries v0 .. v0+3 (UPPER: v0, v0+1) of the lane's sixteen channels.
template <bool UPPER> struct Src { unsigned d[16][UPPER ? 1 : 2]; };

// Loads them: w holds the sixteen weight indices; base is v0 in byte 0 and,
// for a tap past the end, bit 30 (the address then lies past the image and
// the entries read 0).
template <bool UPPER>
__device__ __forceinline__ void load_src(Src<UPPER>& s, int c, __amdgpu_buffer_rsrc_t lut,
                                         const v4i w, unsigned base) {
  const unsigned sel = 0x03020000u | (unsigned)(4 + (c & 3)) << 8;
  const unsigned off = __builtin_amdgcn_perm((unsigned)w[c >> 2], base, sel) << 1;
  if constexpr (UPPER) {
    s.d[c][0] = __builtin_amdgcn_raw_buffer_load_b32(lut, (int)off, 0, 0);
  } else {
    const uint2 v = __builtin_bit_cast(
        uint2, __builtin_amdgcn_raw_buffer_load_b64(lut, (int)off, 0, 0));
    s.d[c][0] = v.x;
    s.d[c][1] = v.y;
  }
}

// Chunks of two table rows (e: v0 + 2u, o: v0 + 2u + 1) in both planes.
struct Chunks { unsigned e0[4], e1[4], o0[4], o1[4]; };

// Channels 4k .. 4k + 3 of entries u: bytes transposed into the rows' chunks
// (sel0 / sel1 pick the planes' bytes).
template <bool UPPER>
__device__ __forceinline__ void transpose4(Chunks& t, const Src<UPPER>& s, int u, int k,
                                           unsigned sel0, unsigned sel1, unsigned xk) {
  const unsigned d0 = s.d[4 * k][u] ^ xk, d1 = s.d[4 * k + 1][u] ^ xk;
  const unsigned d2 = s.d[4 * k + 2][u] ^ xk, d3 = s.d[4 * k + 3][u] ^ xk;
  const unsigned p01 = __builtin_amdgcn_perm(d1, d0, 0x05010400u);
  const unsigned p23 = __builtin_amdgcn_perm(d3, d2, 0x05010400u);
  const unsigned q01 = __builtin_amdgcn_perm(d1, d0, 0x07030602u);
  const unsigned q23 = __builtin_amdgcn_perm(d3, d2, 0x07030602u);
  t.e0[k] = __builtin_amdgcn_perm(p23, p01, sel0);
  t.e1[k] = __builtin_amdgcn_perm(p23, p01, sel1);
  t.o0[k] = __builtin_amdgcn_perm(q23, q01, sel0);
  t.o1[k] = __builtin_amdgcn_perm(q23, q01, sel1);
}

// Stores the chunks: the lane's first plane at wa, the other at wb.
__device__ __forceinline__ void store_chunks(unsigned char* smem, const Chunks& t, int u,
                                             unsigned wa, unsigned wb) {
  *(uint4*)(smem + wa + (2 * u) * LINE) = make_uint4(t.e0[0], t.e0[1], t.e0[2], t.e0[3]);
  *(uint4*)(smem + wb + (2 * u) * LINE) = make_uint4(t.e1[0], t.e1[1], t.e1[2], t.e1[3]);
  *(uint4*)(smem + wa + (2 * u + 1) * LINE) = make_uint4(t.o0[0], t.o0[1], t.o0[2], t.o0[3]);
  *(uint4*)(smem + wb + (2 * u + 1) * LINE) = make_uint4(t.o1[0], t.o1[1], t.o1[2], t.o1[3]);
}

// The lane's eight channels of an output tile: index, and for fp32 kinds the
// factor and bias (ATX_OUT_F32: 1 and none).
struct OutChannels { int o[8]; float sc[8], b[8]; };

__device__ __forceinline__ OutChannels out_channels(const GemmParams& p, int oc, int lane,
                                                    bool raw) {
  OutChannels t;
  const bool dq = !raw && p.out_kind == ATX_OUT_DEQUANT;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    t.o[e] = oc + 16 * (((lane >> 3) & 1) ^ (e >> 2)) + 4 * (lane >> 4) + (e & 3);
    const int o = min(t.o[e], p.O - 1);
    t.sc[e] = dq ? p.sx[0] * p.sw[o] : 1.0f;
    t.b[e] = dq && p.bias ? p.bias[o] : 0.0f;
  }
  return t;
}

// One output value's bits: the int32 sum (`raw`), or fp32 sc * sum [+ bias].
__device__ __forceinline__ int out_bits(int v, float sc, float b, bool raw, bool bias) {
  if (raw) return v;
  const float t = (float)v * sc;
  return __builtin_bit_cast(int, bias ? b + t : t);
}

// Writes the lane's accumulators: rows r + 64 h .. + 3 (r a multiple of 4) of
// its channels, to y as int32 (`raw`: split-K partials too) or fp32.
// Rows beyond R and channels beyond O are dropped.  With L % 4 == 0 four rows
// never straddle two images and are one 16-byte store; otherwise rows are
// stored one by one, stepping (n, l) across image boundaries.
__device__ __forceinline__ void store_tile(const GemmParams& p, int* y, const Acc& acc, int r,
                                           int oc, int lane, bool raw) {
  const bool bias = !raw && p.out_kind == ATX_OUT_DEQUANT && p.bias;
  const OutChannels t = out_channels(p, oc, lane, raw);
  const bool vec = (p.L & 3) == 0;
#pragma unroll
  for (int h = 0; h < RPL / 4; ++h) {
    const int rq = r + 64 * h;
    if (rq >= p.R) break;
    int n = rq / p.L, l = rq - n * p.L;
    if (vec) {
      const long long ybase = (long long)n * p.O * p.L + l;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (t.o[e] >= p.O) continue;
        int v[4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
          v[m] = out_bits(acc[4 * h + m][e >> 2][e & 3], t.sc[e], t.b[e], raw, bias);
        *(int4*)(y + ybase + (long long)t.o[e] * p.L) = make_int4(v[0], v[1], v[2], v[3]);
      }
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (rq + m >= p.R) break;
        const long long ybase = (long long)n * p.O * p.L + l;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (t.o[e] < p.O)
            y[ybase + (long long)t.o[e] * p.L] =
                out_bits(acc[4 * h + m][e >> 2][e & 3], t.sc[e], t.b[e], raw, bias);
        if (++l == p.L) { l = 0; ++n; }
      }
    }
  }
}

// Sums of one tile segment: rows tile tr, channels tile to, k in [kb, ke).
template <bool UPPER>
__device__ __forceinline__ void lut_tile(const GemmParams& p, unsigned char* smem, int tr,
                                         int to, int kb, int ke, Acc& acc) {
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int j16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int b = 0; b < RPL; ++b)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[b][c] = v4i{0, 0, 0, 0};
  if (kb >= ke) return;

  // Reads: lane (j, g) reads the tap of quarter t = (j & 3) ^ g, which for its
  // rows (64 h + 4 j + m) sits in operand slot (t - j) & 3.  t and the channel
  // half j >> 3 differ between the lanes of a read pass that share a plane.
  const int tq = (j16 & 3) ^ g;
  unsigned mask = (unsigned)(tq << 6 | (j16 >> 3) << 5 | (g & 1) << 4);
  const Select sel = make_select(lane);

  // Table build: wave w builds table t = w & 3 of the quad for its rows
  // vh .. vh + 127 (vh = 128 (w >> 2); UPPER: 64 rows of 128..255); lane bit
  // 1 is the channel half, the other bits the group of four (UPPER: two) rows
  // v0.  The four lanes of a store pass write four 16-byte positions: two
  // channel halves, and the planes in the order of lane bit 0.
  const int bt = wave & 3, bcg = (lane >> 1) & 1, vg = (lane >> 2) << 1 | (lane & 1);
  const int v0 = UPPER ? 128 + 64 * (wave >> 2) + 2 * vg : 128 * (wave >> 2) + 4 * vg;
  const unsigned wline = (unsigned)(v0 * LINE + bt * 64 + bcg * 32);
  unsigned wa = wline + (vg & 1) * 16, wb = wline + (~vg & 1) * 16;
  const unsigned sel0 = (vg & 1) ? 0x05040100u : 0x07060302u;   // low / high bytes
  const unsigned sel1 = (vg & 1) ? 0x07060302u : 0x05040100u;
  const unsigned xk = code_xor(p.sgn);
  const __amdgpu_buffer_rsrc_t lutr = buffer_rsrc(p.lut16t, 256 * 256 * 2);

  const int n = ke - kb;
  const int nq = (n + TPL - 1) / TPL;
  const int slot_bytes = p.Rpad * 2;                    // one k-row of the operand
  const int xoff = ((tq - j16) & 3) * slot_bytes + (wave * RPW + j16 * 4) * 2;
  const uint16_t* __restrict__ xtile = p.xt + (long long)tr * p.rt;
  // wave-uniform: does this wave own rows of the tile?
  const bool active = __builtin_amdgcn_readfirstlane(wave) * RPW < p.rt;
  // Quads past the chunk read through an empty view (0); a wave past the tile,
  // whose rows can lie past the operand's padded rows when a short last tile
  // ends near Rpad, reads none.
  auto load_x = [&](int j, int h) {                     // rows 64 h + 4 j16 .. + 3
    // (readfirstlane: a select, not a branch)
    const int bytes = __builtin_amdgcn_readfirstlane(j < nq ? TPL * slot_bytes : 0);
    const __amdgpu_buffer_rsrc_t xs =
        buffer_rsrc(xtile + (long long)(kb + TPL * j) * p.Rpad, bytes);
    return __builtin_bit_cast(
        uint2, __builtin_amdgcn_raw_buffer_load_b64(xs, xoff, 128 * h, 0));
  };
  // The lane's sixteen weight indices of quad j (0 past the chunk).
  const uint8_t* __restrict__ wtile = p.wt + to * OT;
  const int woff = bt * p.Opad + bcg * 16;
  auto load_w = [&](int j) {
    const int taps = min(TPL, n - TPL * j);
    const __amdgpu_buffer_rsrc_t ws =
        buffer_rsrc(wtile + (long long)(kb + TPL * min(j, nq - 1)) * p.Opad,
                    taps > 0 ? (taps - 1) * p.Opad + OT : 0);
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ws, woff, 0, 0));
  };
  auto src_base = [&](int j) {
    return (unsigned)v0 | (TPL * j + bt < n ? 0u : 0x40000000u);
  };

  Src<UPPER> src;
  v4i wreg;
  constexpr int NU = UPPER ? 1 : 2;                     // row pairs a lane builds
  Chunks t;
  // Part i of a table build: channels 4k .. 4k + 3 of row pair u.
  auto piece = [&](int i) __attribute__((always_inline)) {
    const int u = i / 4, k = i % 4;
    transpose4<UPPER>(t, src, u, k, sel0, sel1, xk);
    if (k == 3) store_chunks(smem, t, u, wa, wb);
  };
  auto load_all = [&](const v4i w, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 16; ++c) load_src<UPPER>(src, c, lutr, w, src_base(j));
  };
  wreg = load_w(1);
  load_all(load_w(0), 0);
#pragma unroll
  for (int i = 0; i < 4 * NU; ++i) piece(i);            // quad 0 -> buffer 0
  load_all(wreg, 1);

  if (!active) {                                        // tables only
    __syncthreads();
    for (int j = 0; j < nq; ++j) {
      wreg = load_w(j + 2);
      wa ^= QTAB;
      wb ^= QTAB;
#pragma unroll
      for (int i = 0; i < 4 * NU; ++i) piece(i);
      load_all(wreg, j + 2);
      __syncthreads();
    }
    return;
  }

  uint2 x[4];                                           // row offsets
#pragma unroll
  for (int h = 0; h < 4; ++h) x[h] = load_x(0, h);
  __syncthreads();
  for (int j = 0; j < nq; ++j) {
    // Table of quad j + 1: its entries were loaded during the previous quad;
    // the entry loads of quad j + 2 follow once the registers are free, one
    // channel per read pair, so neither the address unit's queue nor the
    // stores' waits stall the reads.
    wreg = load_w(j + 2);
    const unsigned base = src_base(j + 2);
    wa ^= QTAB;
    wb ^= QTAB;
    v8i ring[RD];
    auto read = [&](int i) __attribute__((always_inline)) {
      const int b = i >> 1, c = i & 1;
      const unsigned xd = (b & 2) ? x[b >> 2].y : x[b >> 2].x;
      const unsigned a = __builtin_amdgcn_perm(xd, mask, (b & 1) ? 0x03020700u : 0x03020500u) ^
                         (c << 5);
      const v4i lo = *(const v4i*)(smem + a);
      const v4i hi = *(const v4i*)(smem + (a ^ 16));
      ring[i % RD] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto sum = [&](int i, const v4i w) __attribute__((always_inline)) {
      v4i& a = acc[i >> 1][i & 1];
      a = __builtin_amdgcn_smfmac_i32_16x16x128_i8(w, ring[i % RD], a, sel.idx, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < RD; ++i) read(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * RPL; i += 2) {              // row block i / 2
      sum(i, sel.both);
      sum(i + 1, sel.both);
      sum(i, sel.high);
      if (i + RD < 2 * RPL) read(i + RD);
      sum(i + 1, sel.high);
      if (i + 1 + RD < 2 * RPL) read(i + 1 + RD);
      if (i / 2 < 4 * NU) piece(i / 2);
      if (i >= 16) {
        load_src<UPPER>(src, i - 16, lutr, wreg, base);
        load_src<UPPER>(src, i - 15, lutr, wreg, base);
      }
      if ((i + RD) % 8 == 0 && i + RD < 2 * RPL + 8)    // a row quad has been read
        x[(i + RD) / 8 - 1] = load_x(j + 1, (i + RD) / 8 - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    mask ^= QTAB;
    __syncthreads();
  }
  const int total = code_bias(p.sgn) * (TPL * nq);      // mod 2^32, as the sums
#pragma unroll
  for (int b = 0; b < RPL; ++b)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[b][c][q] = (int)((unsigned)total - (unsigned)acc[b][c][q]);
}

// Slot layout of a cut tile (stream-K): value (h, m, e) of thread tid at
// ((RQ * h + m) * 8 + e) * NT + tid, so each atomic of a wave covers 256
// contiguous bytes.
__device__ __forceinline__ long long sk_index(int j, int e, int tid) {
  return (long long)(j * 8 + e) * NT + tid;
}

// Slot of stream-K boundary b (quad position (b + 1) * per), or -1 when that
// boundary does not open a cut tile: the tile containing it must start at or
// after boundary b's predecessor (its first boundary is this one).
// Returns the tail tile index (0-based among the remaining tiles).
__device__ __forceinline__ int sk_slot_tile(const GemmParams& p, int b, long long total) {
  const long long B = (long long)(b + 1) * p.sk_per;
  if (B >= total || B % p.nqt == 0) return -1;
  const long long t = B / p.nqt;
  return (t * p.nqt) / p.sk_per == b ? (int)t : -1;
}

__global__ void __launch_bounds__(NT, 1)
lut_gemm_kernel(const GemmParams p) {
  __shared__ __align__(16) unsigned char smem[SMEM_BYTES];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int lb = logical_block();
  Acc acc;
  // the wave's rows lie in the tile
  const bool has_rows = __builtin_amdgcn_readfirstlane(wave) * RPW < p.rt;
  const int rlane = wave * RPW + (lane & 15) * 4;       // the lane's first row in the tile
  const bool upper = p.x_upper && __builtin_amdgcn_readfirstlane(*p.x_upper) != 0;
  if (upper && tid < 2 * (LINE / 16)) {      // row 0 (line 0) of both quad buffers
    // a zero entry as the table build codes it (planes alternate)
    const unsigned xk = code_xor(p.sgn);
    const unsigned z = (tid & 1) ? 0x80808080u : (xk >> 24) * 0x01010101u;
    const int c = tid % (LINE / 16);
    *(uint4*)(smem + (tid < LINE / 16 ? 0 : QTAB) + 16 * c) = make_uint4(z, z, z, z);
  }
  // Segments: one tile's k-chunk (split-K), or (stream-K) whole tiles first
  // (the full rounds), then this workgroup's run of the remaining tiles'
  // quads, tile segment by tile segment.
  const long long total = ((long long)p.tiles_r * p.tiles_o - p.sk_dp) * p.nqt;
  long long it = (long long)lb * p.sk_per;
  const long long end = min(total, it + p.sk_per);
  int whole = p.sk_per ? lb : p.sk_dp;                   // next whole tile
  for (bool first = true;; first = false) {
    int tile, kb, ke;
    int* slot = nullptr;
    int* y = (int*)p.y;
    if (p.sk_per == 0) {
      if (!first) break;
      const int nt = p.tiles_o * p.tiles_r, s = lb / nt;
      tile = lb - s * nt;
      kb = s * p.k_chunk;
      ke = min(p.K, kb + p.k_chunk);
      if (p.splits > 1) y += (long long)s * p.split_stride;
    } else if (whole < p.sk_dp) {
      tile = whole;
      whole += p.sk_g;
      kb = 0;
      ke = p.K;
    } else if (it < end) {
      const int tt = (int)(it / p.nqt);                  // tail tile
      const int q0 = (int)(it - (long long)tt * p.nqt);
      const int q1 = (int)min((long long)p.nqt, q0 + (end - it));
      tile = p.sk_dp + tt;
      kb = TPL * q0;
      ke = min(p.K, TPL * q1);
      if (q0 != 0 || q1 != p.nqt)
        slot = p.skws + (((long long)tt * p.nqt) / p.sk_per) * (long long)(RPL * 8 * NT);
      it += q1 - q0;
    } else {
      break;
    }
    const int to = tile % p.tiles_o, tr = tile / p.tiles_o;
    if (!first) __syncthreads();             // the previous segment's tables are read
    if (upper) lut_tile<true>(p, smem, tr, to, kb, ke, acc);
    else lut_tile<false>(p, smem, tr, to, kb, ke, acc);
    // ---- epilogue: registers -> HBM, every wave at once (no LDS staging).
    if (!has_rows) continue;                 // (a slot's rows of this wave stay zero)
    if (slot) {
#pragma unroll
      for (int b = 0; b < RPL; ++b)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          __hip_atomic_fetch_add(slot + sk_index(b, e, tid), acc[b][e >> 2][e & 3],
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      store_tile(p, y, acc, tr * p.rt + rlane, to * OT, lane,
                 p.splits > 1 || p.out_kind == ATX_OUT_I32);
    }
  }
}

// Zeroes the slots of the cut tiles (block b = slot b).
__global__ void __launch_bounds__(NT)
sk_clear_kernel(const GemmParams p) {
  const long long total = ((long long)p.tiles_r * p.tiles_o - p.sk_dp) * p.nqt;
  if (sk_slot_tile(p, blockIdx.x, total) < 0) return;
  int* slot = p.skws + (long long)blockIdx.x * (RPL * 8 * NT);
  for (int j = 0; j < RPL * 8; ++j) slot[(long long)j * NT + threadIdx.x] = 0;
}

// Epilogue of the cut tiles: each thread reloads the sums it would have held
// and stores them as the main kernel does.
__global__ void __launch_bounds__(NT)
sk_finish_kernel(const GemmParams p) {
  const long long total = ((long long)p.tiles_r * p.tiles_o - p.sk_dp) * p.nqt;
  const int tt = sk_slot_tile(p, blockIdx.x, total);
  if (tt < 0) return;
  const int tile = p.sk_dp + tt;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int* slot = p.skws + (long long)blockIdx.x * (RPL * 8 * NT);
  Acc acc;
#pragma unroll
  for (int b = 0; b < RPL; ++b)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[b][e >> 2][e & 3] = slot[sk_index(b, e, tid)];
  const int to = tile % p.tiles_o, tr = tile / p.tiles_o;
  if (wave * RPW >= p.rt) return;            // rows past the tile
  store_tile(p, (int*)p.y, acc, tr * p.rt + wave * RPW + (lane & 15) * 4, to * OT, lane,
             p.out_kind == ATX_OUT_I32);
}

// Split-K reduction: exact int64 sum of int32 partials, then the epilogue.
// One output per thread (any size / alignment).
__global__ void split_reduce1_kernel(const int* __restrict__ ws, int S,
                                     long long numel, int O, int L, int out_kind,
                                     void* __restrict__ y, const float* sx,
                                     const float* sw, const float* bias, U8Terms u8) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < numel;
       i += (long long)gridDim.x * blockDim.x) {
    long long a = 0;
    for (int s = 0; s < S; ++s) a += ws[(long long)s * numel + i];
    if (out_kind == ATX_OUT_I32) {
      ((int*)y)[i] = (int)a;
    } else if (out_kind == ATX_OUT_F32) {
      ((float*)y)[i] = (float)a;
    } else if (out_kind == OUT_DEQUANT_U8) {
      const long long nl = i / L;              // n * O + o
      const int o = (int)(nl % O), l = (int)(i - nl * L);
      const long long n = nl / O;
      const float z = u8.zx[0], zo = u8.zw[o];
      ((float*)y)[i] = u8_dequant((float)a, u8.xs[n * L + l], zo, z * u8.ws[o],
                                  (u8.K * z) * zo, sx[0] * sw[o], bias, bias ? bias[o] : 0.f);
    } else {
      const int o = (int)((i / L) % O);
      const float sc = sx[0] * sw[o];
      const float t = (float)a * sc;
      ((float*)y)[i] = bias ? bias[o] + t : t;
    }
  }
}

// Four consecutive outputs per thread (16-byte partial loads); numel % 4 == 0.
__global__ void split_reduce_kernel(const int* __restrict__ ws, int S,
                                    long long numel, int O, int L, int out_kind,
                                    void* __restrict__ y, const float* sx,
                                    const float* sw, const float* bias, U8Terms u8) {
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < (numel >> 2);
       q += (long long)gridDim.x * blockDim.x) {
    const long long i = q << 2;
    long long a[4] = {0, 0, 0, 0};
    for (int s = 0; s < S; ++s) {
      const int4 v = *(const int4*)(ws + (long long)s * numel + i);
      a[0] += v.x; a[1] += v.y; a[2] += v.z; a[3] += v.w;
    }
    if (out_kind == ATX_OUT_I32) {
      *(int4*)((int*)y + i) = make_int4((int)a[0], (int)a[1], (int)a[2], (int)a[3]);
    } else if (out_kind == ATX_OUT_F32) {
      *(float4*)((float*)y + i) =
          make_float4((float)a[0], (float)a[1], (float)a[2], (float)a[3]);
    } else if (out_kind == OUT_DEQUANT_U8) {
      long long nl = i / L;                    // n * O + o
      int l = (int)(i - nl * L), o = (int)(nl % O);
      long long n = nl / O;
      const float z = u8.zx[0], kz = u8.K * z, s0 = sx[0];
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float zo = u8.zw[o];
        f[e] = u8_dequant((float)a[e], u8.xs[n * L + l], zo, z * u8.ws[o], kz * zo,
                          s0 * sw[o], bias, bias ? bias[o] : 0.f);
        if (++l == L) { l = 0; if (++o == O) { o = 0; ++n; } }
      }
      *(float4*)((float*)y + i) = make_float4(f[0], f[1], f[2], f[3]);
    } else {
      long long nl = i / L;                    // n * O + o
      int l = (int)(i - nl * L), o = (int)(nl % O);
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sc = sx[0] * sw[o];
        const float t = (float)a[e] * sc;
        f[e] = bias ? bias[o] + t : t;
        if (++l == L) { l = 0; if (++o == O) o = 0; }
      }
      *(float4*)((float*)y + i) = make_float4(f[0], f[1], f[2], f[3]);
    }
  }
}

// Split plan shared by the workspace query and the launch.  sk_per > 0
// selects the stream-K schedule (PLAN_CUS workgroups, sk_per quads each).
struct Plan { int tiles_r, tiles_o, splits, k_chunk, sk_per, nqt, sk_dp, rt; };

// Compute units of a full MI355X (one resident workgroup each: the kernel's
// 8 waves hold 2 waves per SIMD at its register budget).  A constant, not a
// device query, so the workspace query and the launch always agree.
constexpr int PLAN_CUS = 256;

// Plan by a cost model in microseconds, over the rows per tile rt (2048, 1792,
// 1536, 1280, 1024, 768 or 512, keeping ceil(R / rt) tiles inside the operand's
// padded rows) and the split-K count S, with x = rt / 2048:
//   ceil(tiles(rt) * S / CUs) rounds x (k-chunk x step x (0.75 + 0.25 x)
//     + 3.7 + 5.9 x: table prologue and output stores)
//   + for S > 1: 3.6 for the reduce launch and S x R*O x 1.31e-6 for writing
//     and re-reading one int32 partial slice,
// step = 0.62 (a k-step of a full tile), 0.44 with the upper-half tables
// (`upper`; the tables' loads and stores halve).  The flag's value is on the
// device, so every call that passes one (the int8 layers, the GEMM-level ops)
// is planned as if it were set: for signed operands a plan at most 3% dearer by
// the model (19 x 675 x 621 -> 83), the same at most sizes.  A least-squares
// fit to a sweep of (rt, S) over 38 shapes (19 ResNet-50 layers at batch 64, 10
// ResNet-18 layers at 128, GEMM and small shapes), both table heights: its
// picks take 13.29 ms over the sweep, the best pair of each shape 13.24, the
// model fitted to the kernel's earlier sums (0.95 us a step) 13.62.
// k-chunks are whole quads of tables (multiples of 4); S is at least
// ceil(K / kmax), the exact-int32 bound of one pass, and the smallest cost
// wins (ties: the larger rt, then the smaller S).
// Stream-K (K <= kmax, at the default rt): floor(tiles / CUs) full rounds of
// whole tiles, then the T = tail tiles * ceil(K/4) quads of the rest dealt
// out evenly, per = ceil(T / CUs) quads per workgroup, which ends the
// partial last round.  Cost, fitted to the same sweep: the rounds and quads at
// the step above, a tile's fixed cost per tail segment a workgroup runs
// (ceil(per / nqt) + 1 at most), 42 for the clear / finish launches and their
// traffic, 0.07 per cut tile (its 256 KiB slot and atomics).  It is taken when
// cheaper than the best split-K plan: 5 of the 38 with full tables (K = 1024,
// 12544 x 512: 327 against 340 us; K = 2304, 12544 x 256: 361 against 370).
// The upper-half tables' constant is 60: with the slots cold, as within a
// network, stream-K took 15 us more than split-K at K = 1152, 50176 x 128.
// ATX_LUT_SCHEDULE (environment: auto | split | stream_k) overrides the
// choice; ATX_LUT_ROWS and ATX_LUT_SPLITS force the rows per tile and the
// split count (split-K plans), for measurement.
// ws_limit >= 0 caps the workspace: split counts whose int32 partials exceed
// it are not considered; when even the smallest admissible split count (set
// by the int32-exactness bound) needs more, the plan's splits is -1.
constexpr long long SK_SLOT_BYTES = (long long)(PLAN_CUS - 1) * RT * OT * 4;

static Plan make_plan(int N, int K, int L, int O, int kmax, long long ws_limit = -1,
                      bool upper = false) {
  Plan pl;
  const long long R = (long long)N * L;
  pl.tiles_r = (int)cdiv(R, RT);
  // the fewest whole waves of rows that cover R in tiles_r tiles
  pl.rt = R > 0 ? (int)std::min<long long>(RT, cdiv(cdiv(R, pl.tiles_r), RPW) * RPW) : RT;
  pl.tiles_o = (int)cdiv(O, OT);
  pl.sk_per = 0;
  pl.sk_dp = 0;
  pl.nqt = (int)cdiv(K, TPL);
  if (K <= 0) { pl.splits = 1; pl.k_chunk = 1; return pl; }
  const char* sched = getenv("ATX_LUT_SCHEDULE");
  const bool force_sk = sched && !strcmp(sched, "stream_k");
  const char* force_rows = getenv("ATX_LUT_ROWS");
  const char* force_s = getenv("ATX_LUT_SPLITS");
  const long long cus = PLAN_CUS;
  const int smin = (int)cdiv(K, kmax);
  const int fs = force_s ? std::max(smin, atoi(force_s)) : 0;
  const double step = upper ? 0.437 : 0.623;               // us per k-step of a full tile
  const double slice = (double)R * O * 1.31e-6;
  const auto step_cost = [&](int rt) { return step * (0.753 + 0.247 * rt / RT); };
  const auto tile_cost = [&](int rt) { return 3.66 + 5.93 * rt / RT; };
  const long long rows_cap = cdiv(R, RT) * RT;
  static const int kRows[] = {2048, 1792, 1536, 1280, 1024, 768, 512};
  int cand[8], nc = 0;
  if (force_rows) {
    const int rt = atoi(force_rows);
    if (rt >= RPW && rt <= RT && rt % RPW == 0 && R > 0 && cdiv(R, rt) * rt <= rows_cap)
      cand[nc++] = rt;
  }
  if (nc == 0) {
    if (force_sk || R <= 0) {
      cand[nc++] = pl.rt;
    } else {
      cand[nc++] = pl.rt;
      for (int rt : kRows)
        if (rt < pl.rt && cdiv(R, rt) * rt <= rows_cap) cand[nc++] = rt;
    }
  }
  long long best_kc = cdiv(cdiv(K, smin), TPL) * TPL;
  int best_rt = pl.rt;
  double best_cost = 0.0;
  bool found = false;
  for (int c = 0; c < nc; ++c) {
    const int rt = cand[c];
    const long long tiles = cdiv(R, rt) * pl.tiles_o;
    // least cost of S or more splits (no workgroup idle): ends the search early
    const double work = tiles * (K * step_cost(rt)) / cus;
    const double per_s = tiles * tile_cost(rt) / cus + slice;
    for (int S = fs ? fs : smin; S <= (fs ? fs : std::max(smin, 64)); ++S) {
      const long long kc = cdiv(cdiv(K, S), TPL) * TPL;
      if (S > smin && kc < 8 && !fs) break;
      if (found && S > 1 && work + S * per_s >= best_cost) break;
      const long long splits = cdiv(K, kc);
      if (ws_limit >= 0 && splits > 1 && splits * R * O * 4 > ws_limit) continue;
      const double cost = (double)cdiv(tiles * splits, cus) *
                              (kc * step_cost(rt) + tile_cost(rt)) +
                          (splits > 1 ? 3.6 + splits * slice : 0.0);
      if (!found || cost < best_cost) {
        best_kc = kc; best_cost = cost; best_rt = rt; found = true;
      }
    }
  }
  if (!found) { pl.splits = -1; pl.k_chunk = 1; return pl; }
  pl.k_chunk = (int)std::min<long long>(best_kc, kmax);
  pl.splits = (int)cdiv(K, pl.k_chunk);
  // stream-K at the default rows per tile, when forced or cheaper
  const long long tiles = (long long)pl.tiles_r * pl.tiles_o;
  const bool split_only = (sched && !strcmp(sched, "split")) || force_rows || force_s;
  if (!split_only && K <= kmax && tiles % cus != 0 && (ws_limit < 0 || SK_SLOT_BYTES <= ws_limit)) {
    const long long rounds = tiles / cus;
    const long long tail = tiles - rounds * cus;
    const long long T = tail * pl.nqt;
    const long long per = cdiv(T, cus);
    if (per >= 2) {
      const long long cuts = std::min<long long>(tail, cdiv(T, per) - 1);
      const double sk_cost = rounds * (K * step_cost(pl.rt) + tile_cost(pl.rt)) +
                             4.0 * per * step_cost(pl.rt) +
                             tile_cost(pl.rt) * (double)(cdiv(per, pl.nqt) + 1) +
                             (upper ? 60.0 : 42.0) + 0.07 * cuts;
      if (force_sk || sk_cost < best_cost) {
        pl.sk_per = (int)per;
        pl.sk_dp = (int)(rounds * cus);
        return pl;                       // default rows per tile
      }
    }
  }
  pl.rt = best_rt;
  pl.tiles_r = R > 0 ? (int)cdiv(R, best_rt) : pl.tiles_r;
  return pl;
}

// ------------------------------------------------ no-allocation scratch
// Device memory of atx_lut_gemm_noalloc: a file-scope array, one copy per GPU
// for the life of the process.  Host code never uses its name as an address:
// the device address of this GPU's copy comes from hipGetSymbolAddress (with
// that device current) and is cached per device.
static __device__ __align__(256) unsigned char scratch[ATX_NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_addr[MAX_DEVICES];

// Address of the current device's scratch array; the stream must belong to
// the current device (the address is only valid there).
static int noalloc_scratch(hipStream_t stream, void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess)
    return set_error(ATX_ELAUNCH, "atx_lut_gemm_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= MAX_DEVICES)
    return set_error(ATX_ERANGE, "atx_lut_gemm_noalloc: device %d out of range", dev);
  if (stream != nullptr) {
    int sdev = -1;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess)
      return set_error(ATX_ELAUNCH, "atx_lut_gemm_noalloc: hipStreamGetDevice: %s",
                       hipGetErrorString(e));
    if (sdev != dev)
      return set_error(ATX_EINVAL,
                       "atx_lut_gemm_noalloc: the stream belongs to device %d, the current "
                       "device is %d", sdev, dev);
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_addr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return set_error(ATX_ELAUNCH, "atx_lut_gemm_noalloc: hipGetSymbolAddress: %s",
                       hipGetErrorString(e));
    g_scratch_addr[dev] = p;
  }
  *out = g_scratch_addr[dev];
  return ATX_OK;
}

}  // namespace atx

using namespace atx;

extern "C" {

int atx_lut_prepare(const float* lut, uint16_t* out16t, float* outf32t,
                    int* flags, hipStream_t stream) {
  ATX_REQUIRE(lut && out16t && outf32t && flags, "atx_lut_prepare: null pointer");
  hipLaunchKernelGGL(lut_prepare_kernel, dim3(256), dim3(256), 0, stream, lut,
                     out16t, outf32t, flags);
  return check_launch("lut_prepare_kernel");
}

int atx_pack_x_f32(const float* x, int N, int K, int L, int offset, uint8_t* xq,
                   uint16_t* xt, int Rpad, int* upper, hipStream_t stream) {
  ATX_REQUIRE(N >= 0 && K >= 0 && L >= 0, "atx_pack_x_f32: negative size");
  ATX_REQUIRE(Rpad >= (long long)N * L && Rpad % RT == 0,
              "atx_pack_x_f32: Rpad must be a multiple of %d covering N*L", RT);
  if ((long long)K * Rpad == 0) return ATX_OK;
  // an empty x (N*L == 0) only writes the zero padding rows
  ATX_REQUIRE(xt && ((long long)N * L == 0 || x), "atx_pack_x_f32: null pointer");
  const dim3 grid((unsigned)cdiv(Rpad / 4, 256),
                  (unsigned)std::min(operand_rows(K) / 4, 65535));
  const bool vec = L % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)xq % 4 == 0;
  hipLaunchKernelGGL(pack_x_quads_kernel<float>, grid, dim3(256), 0, stream, x, N, K, L,
                     offset, xq, xt, Rpad, vec, upper);
  return check_launch("pack_x_quads_kernel<float>");
}

int atx_pack_x_u8(const uint8_t* xq, int N, int K, int L, uint16_t* xt, int Rpad,
                  int* upper, hipStream_t stream) {
  ATX_REQUIRE(N >= 0 && K >= 0 && L >= 0, "atx_pack_x_u8: negative size");
  ATX_REQUIRE(Rpad >= (long long)N * L && Rpad % RT == 0,
              "atx_pack_x_u8: Rpad must be a multiple of %d covering N*L", RT);
  if ((long long)K * Rpad == 0) return ATX_OK;
  ATX_REQUIRE(xt && ((long long)N * L == 0 || xq), "atx_pack_x_u8: null pointer");
  ATX_REQUIRE(operand_rows(K) / 4 <= 65535, "atx_pack_x_u8: K too large");
  const dim3 grid((unsigned)cdiv(Rpad / 4, 256), (unsigned)(operand_rows(K) / 4));
  const bool vec = L % 4 == 0 && (uintptr_t)xq % 4 == 0;
  hipLaunchKernelGGL(pack_x_quads_kernel<uint8_t>, grid, dim3(256), 0, stream, xq, N, K, L, 0,
                     (uint8_t*)nullptr, xt, Rpad, vec, upper);
  return check_launch("pack_x_quads_kernel<u8>");
}

int atx_pack_w_f32(const float* w, int O, int K, int offset, uint8_t* wq,
                   uint8_t* wt, int Opad, hipStream_t stream) {
  ATX_REQUIRE(O >= 0 && K >= 0, "atx_pack_w_f32: negative size");
  ATX_REQUIRE(Opad >= O && Opad % OT == 0,
              "atx_pack_w_f32: Opad must be a multiple of %d covering O", OT);
  if ((long long)K * Opad == 0) return ATX_OK;
  // an empty w (O == 0) only writes the padding columns
  ATX_REQUIRE((wt || wq) && (O == 0 || w), "atx_pack_w_f32: null pointer");
  hipLaunchKernelGGL(pack_w_kernel<float>, dim3(elem_grid((long long)K * Opad, 256)),
                     dim3(256), 0, stream, w, O, K, offset, wq, wt, Opad);
  return check_launch("pack_w_kernel<float>");
}

int atx_pack_w_u8(const uint8_t* wq, int O, int K, uint8_t* wt, int Opad,
                  hipStream_t stream) {
  ATX_REQUIRE(O >= 0 && K >= 0, "atx_pack_w_u8: negative size");
  ATX_REQUIRE(Opad >= O && Opad % OT == 0,
              "atx_pack_w_u8: Opad must be a multiple of %d covering O", OT);
  if ((long long)K * Opad == 0) return ATX_OK;
  ATX_REQUIRE(wt && (O == 0 || wq), "atx_pack_w_u8: null pointer");
  hipLaunchKernelGGL(pack_w_kernel<uint8_t>, dim3(elem_grid((long long)K * Opad, 256)),
                     dim3(256), 0, stream, wq, O, K, 0, (uint8_t*)nullptr, wt, Opad);
  return check_launch("pack_w_kernel<u8>");
}

int atx_pack_rows_strided(const void* x, int dtype, int R, int K, long long sr, long long sk,
                          int offset, uint8_t* xq, uint16_t* xt, int Rpad, int* upper,
                          hipStream_t stream) {
  ATX_REQUIRE(R >= 0 && K >= 0 && (dtype == 0 || dtype == 1),
              "atx_pack_rows_strided: bad arguments");
  ATX_REQUIRE(Rpad >= R && Rpad % RT == 0,
              "atx_pack_rows_strided: Rpad must be a multiple of %d covering R", RT);
  if ((long long)K * Rpad == 0) return ATX_OK;
  ATX_REQUIRE(xt && (R == 0 || x), "atx_pack_rows_strided: null pointer");
  // contiguous along k (and not along the rows too): turned in LDS
  if (sk == 1 && sr != 1 && K > 1 && cdiv(K, TT) <= 65535) {
    const dim3 tiles((unsigned)(Rpad / TT), (unsigned)cdiv(K, TT));
    if (dtype == 0)
      hipLaunchKernelGGL(pack_rows_turned_kernel<float>, tiles, dim3(256), 0, stream,
                         (const float*)x, R, K, sr, offset, xq, xt, Rpad, upper);
    else
      hipLaunchKernelGGL(pack_rows_turned_kernel<uint8_t>, tiles, dim3(256), 0, stream,
                         (const uint8_t*)x, R, K, sr, 0, xq, xt, Rpad, upper);
    return check_launch("pack_rows_turned_kernel");
  }
  dim3 grid((unsigned)std::min<long long>(cdiv(Rpad / 4, 256), 1024),
            (unsigned)std::min(operand_rows(K), 65535));
  if (dtype == 0)
    hipLaunchKernelGGL(pack_rows_strided_kernel<float>, grid, dim3(256), 0, stream,
                       (const float*)x, R, K, sr, sk, offset, xq, xt, Rpad, upper);
  else
    hipLaunchKernelGGL(pack_rows_strided_kernel<uint8_t>, grid, dim3(256), 0, stream,
                       (const uint8_t*)x, R, K, sr, sk, 0, xq, xt, Rpad, upper);
  return check_launch("pack_rows_strided_kernel");
}

int atx_pack_cols_strided(const void* y, int dtype, int C, int K, long long sc, long long sk,
                          int offset, uint8_t* yq, uint8_t* wt, int Opad, hipStream_t stream) {
  ATX_REQUIRE(C >= 0 && K >= 0 && (dtype == 0 || dtype == 1),
              "atx_pack_cols_strided: bad arguments");
  ATX_REQUIRE(Opad >= C && Opad % OT == 0,
              "atx_pack_cols_strided: Opad must be a multiple of %d covering C", OT);
  if ((long long)K * Opad == 0) return ATX_OK;
  ATX_REQUIRE(wt && (C == 0 || y), "atx_pack_cols_strided: null pointer");
  if (sk == 1 && sc != 1 && K > 1 && (uintptr_t)wt % 4 == 0 && cdiv(K, TT) <= 65535) {
    const dim3 tiles((unsigned)cdiv(Opad, TT), (unsigned)cdiv(K, TT));
    if (dtype == 0)
      hipLaunchKernelGGL(pack_cols_turned_kernel<float>, tiles, dim3(256), 0, stream,
                         (const float*)y, C, K, sc, offset, yq, wt, Opad);
    else
      hipLaunchKernelGGL(pack_cols_turned_kernel<uint8_t>, tiles, dim3(256), 0, stream,
                         (const uint8_t*)y, C, K, sc, 0, yq, wt, Opad);
    return check_launch("pack_cols_turned_kernel");
  }
  const dim3 grid(elem_grid((long long)K * Opad, 256));
  if (dtype == 0)
    hipLaunchKernelGGL(pack_cols_strided_kernel<float>, grid, dim3(256), 0, stream,
                       (const float*)y, C, K, sc, sk, offset, yq, wt, Opad);
  else
    hipLaunchKernelGGL(pack_cols_strided_kernel<uint8_t>, grid, dim3(256), 0, stream,
                       (const uint8_t*)y, C, K, sc, sk, 0, yq, wt, Opad);
  return check_launch("pack_cols_strided_kernel");
}

long long atx_lut_gemm_workspace_bytes(int N, int K, int L, int O) {
  if (N <= 0 || K <= 0 || L <= 0 || O <= 0) return 0;
  // the launch plans with or without an x_upper flag: enough for either
  long long bytes = 0;
  for (int upper = 0; upper < 2; ++upper) {
    const Plan pl = make_plan(N, K, L, O, KMAX_U16, -1, upper != 0);
    if (pl.sk_per > 0) bytes = std::max(bytes, SK_SLOT_BYTES);
    else if (pl.splits > 1) bytes = std::max(bytes, (long long)pl.splits * N * O * L * 4);
  }
  return bytes;
}

}  // extern "C"

namespace atx {

// The body of atx_lut_gemm / atx_lut_gemm_noalloc.  ws_limit < 0: the
// workspace holds atx_lut_gemm_workspace_bytes() (caller-sized); otherwise
// the plan is restricted to schedules whose workspace fits ws_limit bytes,
// and `scratch()` supplies it (called only when a launch needs it).
template <typename ScratchFn>
static int lut_gemm_run(const uint16_t* xt, int Rpad, const uint8_t* wt, int Opad, int N, int K,
                        int L, int O, const uint16_t* lut16t, const float* lutf32t,
                        int lut_class, atx_gemm_epilogue ep, void* y, void* workspace,
                        long long ws_limit, ScratchFn scratch, hipStream_t stream) {
  ATX_REQUIRE_EPILOGUE(ep, "atx_lut_gemm");
  ATX_REQUIRE(N >= 0 && K >= 0 && L >= 0 && O >= 0, "atx_lut_gemm: negative size");
  const long long R = (long long)N * L;
  ATX_REQUIRE(R <= 0x7fffffffLL - RT, "atx_lut_gemm: N*L too large");
  ATX_REQUIRE(Rpad >= R && Rpad % RT == 0, "atx_lut_gemm: bad Rpad %d", Rpad);
  // Four k-rows of the row-offset operand are addressed with 32-bit offsets.
  if ((long long)Rpad > (1LL << 27))
    return set_error(ATX_ERANGE, "atx_lut_gemm: Rpad %d exceeds 2^27 rows", Rpad);
  ATX_REQUIRE(Opad >= O && Opad % OT == 0, "atx_lut_gemm: bad Opad %d", Opad);
  ATX_REQUIRE(ep.out_kind >= ATX_OUT_F32 && ep.out_kind <= ATX_OUT_DEQUANT,
              "atx_lut_gemm: bad out_kind");
  ATX_REQUIRE(lut_class >= ATX_LUT_I16 && lut_class <= ATX_LUT_F32,
              "atx_lut_gemm: bad lut_class");
  ATX_REQUIRE(!(lut_class == ATX_LUT_F32 && ep.out_kind == ATX_OUT_I32),
              "atx_lut_gemm: int32 output needs an integer LUT");
  ATX_REQUIRE(ep.out_kind != ATX_OUT_DEQUANT || (ep.scale_x && ep.scale_w),
              "atx_lut_gemm: dequant epilogue needs scale_x and scale_w");
  if (R * O == 0) return ATX_OK;
  ATX_REQUIRE(y, "atx_lut_gemm: null output");
  // K == 0 is an empty contraction: every sum is 0 and only the epilogue runs.
  ATX_REQUIRE(K == 0 || (xt && wt), "atx_lut_gemm: null operand");

  GemmParams p{};
  p.xt = xt; p.Rpad = Rpad; p.wt = wt; p.Opad = Opad;
  p.lut16t = lut16t; p.lutf32t = lutf32t;
  p.K = K; p.R = (int)R; p.L = L; p.O = O;
  p.out_kind = ep.out_kind; p.y = y;
  p.sx = ep.scale_x; p.sw = ep.scale_w; p.bias = ep.bias;
  p.x_upper = ep.x_upper;
  p.sgn = lut_class == ATX_LUT_I16;

  if (lut_class == ATX_LUT_F32) {
    ATX_REQUIRE(lutf32t, "atx_lut_gemm: fp32 class needs the fp32 image");
    int rc = timing_mark(false, stream);
    if (rc == ATX_OK)
      rc = lut_gemm_f32_tiled(xt, Rpad, wt, Opad, lutf32t, N, K, L, O, ep.out_kind, ep.scale_x,
                              ep.scale_w, ep.bias, (float*)y, stream);
    return rc == ATX_OK ? timing_mark(true, stream) : rc;
  }
  ATX_REQUIRE(lut16t, "atx_lut_gemm: integer class needs the 16-bit image");
  const Plan pl = make_plan(N, K, L, O, KMAX_U16, ws_limit, ep.x_upper != nullptr);
  if (pl.splits < 0)
    return set_error(ATX_ERANGE,
                     "atx_lut_gemm_noalloc: K = %d needs %lld bytes of int32 partial sums "
                     "(R = %lld rows x O = %d), more than the %lld-byte scratch buffer; "
                     "call atx_lut_gemm with a workspace", K,
                     (long long)cdiv(K, KMAX_U16) * R * O * 4, R, O, ws_limit);
  if (ws_limit >= 0 && (pl.sk_per > 0 || pl.splits > 1)) {
    const int rc = scratch(&workspace);
    if (rc != ATX_OK) return rc;
  }
  p.tiles_r = pl.tiles_r; p.tiles_o = pl.tiles_o; p.rt = pl.rt;
  p.splits = pl.splits; p.k_chunk = pl.k_chunk;
  const long long numel = R * O;
  if (pl.sk_per > 0) {
    ATX_REQUIRE(workspace, "atx_lut_gemm: stream-K plan needs a workspace of %lld bytes",
                (long long)(PLAN_CUS - 1) * RT * OT * 4);
    p.sk_per = pl.sk_per; p.nqt = pl.nqt; p.skws = (int*)workspace;
    p.sk_dp = pl.sk_dp; p.sk_g = PLAN_CUS;
    p.splits = 1;
    const long long T = ((long long)pl.tiles_r * pl.tiles_o - pl.sk_dp) * pl.nqt;
    const unsigned Gt = (unsigned)cdiv(T, pl.sk_per);         // tail workgroups, <= PLAN_CUS
    const unsigned G = pl.sk_dp > 0 ? (unsigned)PLAN_CUS : Gt;
    if (Gt > 1) {
      hipLaunchKernelGGL(sk_clear_kernel, dim3(Gt - 1), dim3(NT), 0, stream, p);
      int rc = check_launch("sk_clear_kernel");
      if (rc != ATX_OK) return rc;
    }
    int rc = timing_mark(false, stream);
    if (rc != ATX_OK) return rc;
    hipLaunchKernelGGL(lut_gemm_kernel, dim3(G), dim3(NT), 0, stream, p);
    rc = check_launch("lut_gemm_kernel");
    if (rc == ATX_OK) rc = timing_mark(true, stream);
    if (rc != ATX_OK || Gt <= 1) return rc;
    hipLaunchKernelGGL(sk_finish_kernel, dim3(Gt - 1), dim3(NT), 0, stream, p);
    return check_launch("sk_finish_kernel");
  }
  if (pl.splits > 1) {
    ATX_REQUIRE(workspace, "atx_lut_gemm: split-K plan needs a workspace of %lld bytes",
                (long long)pl.splits * numel * 4);
    p.y = workspace;
    p.split_stride = numel;
  }
  const long long blocks = (long long)pl.tiles_r * pl.tiles_o * pl.splits;
  ATX_REQUIRE(blocks < 0x7fffffffLL, "atx_lut_gemm: grid too large");
  int rc = timing_mark(false, stream);
  if (rc != ATX_OK) return rc;
  hipLaunchKernelGGL(lut_gemm_kernel, dim3((unsigned)blocks), dim3(NT), 0, stream, p);
  rc = check_launch("lut_gemm_kernel");
  if (rc == ATX_OK) rc = timing_mark(true, stream);
  if (rc != ATX_OK || pl.splits == 1) return rc;
  return launch_split_reduce((const int*)workspace, pl.splits, numel, O, L, ep, y, stream);
}

int launch_split_reduce(const int* ws, int S, long long numel, int O, int L,
                        const atx_gemm_epilogue& ep, void* y, hipStream_t stream,
                        const U8Terms& u8) {
  if (numel % 4 == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)ws & 15) == 0)
    hipLaunchKernelGGL(split_reduce_kernel, dim3(elem_grid(numel / 4, 256)), dim3(256), 0,
                       stream, ws, S, numel, O, L, ep.out_kind, y, ep.scale_x, ep.scale_w,
                       ep.bias, u8);
  else
    hipLaunchKernelGGL(split_reduce1_kernel, dim3(elem_grid(numel, 256)), dim3(256), 0,
                       stream, ws, S, numel, O, L, ep.out_kind, y, ep.scale_x, ep.scale_w,
                       ep.bias, u8);
  return check_launch("split_reduce_kernel");
}

}  // namespace atx

extern "C" {

int atx_lut_gemm(const uint16_t* xt, int Rpad, const uint8_t* wt, int Opad,
                 int N, int K, int L, int O, const uint16_t* lut16t,
                 const float* lutf32t, int lut_class, atx_gemm_epilogue ep,
                 void* y, void* workspace, hipStream_t stream) {
  return lut_gemm_run(xt, Rpad, wt, Opad, N, K, L, O, lut16t, lutf32t, lut_class, ep, y,
                      workspace, -1, [](void**) { return ATX_OK; }, stream);
}

int atx_lut_gemm_noalloc(const uint16_t* xt, int Rpad, const uint8_t* wt, int Opad,
                         int N, int K, int L, int O, const uint16_t* lut16t,
                         const float* lutf32t, int lut_class, atx_gemm_epilogue ep,
                         void* y, hipStream_t stream) {
  return lut_gemm_run(xt, Rpad, wt, Opad, N, K, L, O, lut16t, lutf32t, lut_class, ep, y,
                      nullptr, ATX_NOALLOC_SCRATCH_BYTES,
                      [stream](void** ws) { return noalloc_scratch(stream, ws); }, stream);
}

}  // extern "C"
