// Quantized linear for the DeltaNet layer's projections on gfx950: y = x W^T with W in
// the reference's 4-bit affine layout (cpp/src/model.cpp:356-372, mx::quantized_matmul
// with transpose = true, group 64; python/mlp_kernel.py:54-56): uint32 words of 8 values,
// value i in nibble i (low nibble first), element = nibble * scale + bias per group of
// 64, scales and biases bf16. Up to four matrices that read the same x run in one launch
// (in_proj_qkv, in_proj_z, in_proj_a, in_proj_b of one layer), and an optional prologue
// applies the layer's GatedRMSNorm (model.cpp:350-354) to the recurrence output before
// out_proj, so norm and projection are one launch.
//
// HBM-bound at decode (M = B * L rows of x, 1..4): every weight byte is read once.
// Mapping: a workgroup of 4 or 8 waves stages its operand in LDS, then each wave takes 4 output
// rows at a time, one per 16-lane DPP row; lane m of a row reads the row's 16-byte pieces m, m + 16,
// m + 32, ... (each 32 nibbles = half a group), so a load instruction reads 4 x 256
// contiguous bytes; the rows' scale and bias words come 16 bytes a lane, ahead of the
// weights, and reach the lanes that use them through the wave's LDS rows. A nibble v becomes the bf16 value 128 + v with one and-or
// ((w >> 4i) & 0x000F000F | 0x43004300 gives nibbles i and i + 4 of the word as two bf16),
// v_dot2 multiplies pairs by the operand staged in the same pair order, and scale and
// bias are applied once per half-group: sum x (q s + b) = s * sum x (128 + q) +
// (b - 128 s) * sum x. The row total is a DPP row sum; the result is rounded to bf16 once.
//
// More rows (verify blocks, batched decode, prefill windows) run on MFMA with the
// same arithmetic: qprep writes the operand once into the workspace in the MFMA fragment
// order (the norm prologue applied there, as above) together with each row's sum x per
// 64-value group, then in qgemm each lane's weight row gives B fragments straight from its
// nibble words and the operand fragments come from the workspace; per group
// acc = sum x (128 + q) (fp32, MFMA), then y += s * acc + (b - 128 s) * sum x. In qgemm a
// workgroup's 4 waves split K and add their partial sums in LDS at the end, so each wave
// reads a quarter of the operand; calls of many weight rows and one m group (up to 48 rows,
// e.g. 8 layers of in_proj at once) take qgemm_ns instead, whose workgroup of 256 weight rows
// reads the operand into LDS once for its four waves; calls of more than 48 rows and enough
// tiles take qgemm_big, whose workgroups share 128 x 256 or 64 x 128 tiles through LDS.
#include "../../include/gdn.h"
#include "gdn_device_math.h"
#include "gdn_internal.h"

#include <algorithm>
#include <mutex>

namespace gdn {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// global-memory pointers: a plain pointer that passed through a struct can lose its
// address space and compile to flat loads, which also count against the LDS wait counter
typedef const u32x2 __attribute__((address_space(1))) g_u32x2;
typedef const u32x4 __attribute__((address_space(1))) g_u32x4;

constexpr int kThreads = 256;

struct QParams {
  int M, K, R, tiles, nseg;
  int passes;            // row passes per workgroup: a tile is 16 x passes rows
  const uint16_t* x;     // (L, M, K) bf16, or NULL with the norm prologue
  const float* xf;       // (L, M, K) fp32 recurrence output (norm prologue)
  const uint16_t* z;     // (L, M, K) bf16 gate (norm prologue)
  const float* gamma;    // (L, 128) fp32 (norm prologue)
  float eps;
  const uint32_t* w[GDN_QLINEAR_MAX_SEGS];
  const uint16_t* s[GDN_QLINEAR_MAX_SEGS];
  const uint16_t* b[GDN_QLINEAR_MAX_SEGS];
  uint16_t* y[GDN_QLINEAR_MAX_SEGS];
  int n[GDN_QLINEAR_MAX_SEGS];
  int row0[GDN_QLINEAR_MAX_SEGS];  // first global row of each segment
  // MFMA path: the operand in fragment order, (L, mtiles, K / 32) blocks of 64 lanes x 8
  // bf16; lane 16 g4 + mm of block f = 2 g + s holds row 16 mt + mm, values
  // k = 64 g + 16 g4 + 8 s + (0, 4, 1, 5, 2, 6, 3, 7) (the nibble pair order); rows past M
  // are zeros
  uint16_t* xfrag;
  // MFMA path: sum x of each 64-value group, fp32, (L, K / 64, 16 mtiles): row-contiguous
  // per group, so a workgroup's m tiles of one group are one run
  float* xsum;
  int mtiles;
  // MFMA path: xfrag in 32-row fragments instead (qgemm_big_kernel): (L, mtiles / 2, K / 64, 4)
  // blocks of 64 lanes x 8 bf16; lane 32 h + mm of block s of group g holds row 32 mb + mm,
  // values k = 64 g + 32 h + 8 s + (0, 4, 1, 5, 2, 6, 3, 7)
  int frag32;
  int mgroups;  // MFMA path: groups of MT m-tiles (the grid is layers x tiles x mgroups)
  int remap;    // MFMA path: XCD-aware workgroup order (see qgemm_tile)
  int layers;   // qgemm_big_kernel's leftover rows
};

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, a), __builtin_bit_cast(bf2, b), c, false);
}

__device__ __forceinline__ uint32_t pack_bf2(float lo, float hi) {
  return (uint32_t)f2bf(lo) | ((uint32_t)f2bf(hi) << 16);
}

// Operand chunk c (32 values) of row mm to LDS: four 16-byte words, word i holding the pairs
// (v[8i+j], v[8i+j+4]), j = 0..3, the order the nibble pairs come out in; plus the sum of the
// 32 values.
__device__ __forceinline__ void stage_chunk(const QParams& p, u32x4* xs, float* xsum, int nch, int layer, int mm, int c) {
  const uint16_t* src = p.x + ((size_t)layer * p.M + mm) * p.K + 32 * c;
  float v[32];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const u16x8 xx = *reinterpret_cast<const u16x8*>(src + 8 * q);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[8 * q + e] = bf2f(xx[e]);
  }
  float sum = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e) sum += v[e];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u32x4 q;
#pragma unroll
    for (int j = 0; j < 4; ++j) q[j] = pack_bf2(v[8 * i + j], v[8 * i + j + 4]);
    xs[(mm * 4 + i) * nch + c] = q;
  }
  xsum[mm * nch + c] = sum;
}

// The GatedRMSNorm of (xf, z) (model.cpp:350-354) as the operand: h = o * rsqrt(mean(o^2) +
// eps) * gamma (fp32), times silu(fp32(z)), rounded to bf16 (the activation dtype out_proj
// takes). A lane takes 8 values; the 16 lanes of a DPP row hold a 128-value head, whose sum of
// squares is 8 terms a lane and a row sum.
struct NormIn {
  f4 o[2];
  u16x8 z;
};
__device__ __forceinline__ NormIn norm_load(const QParams& p, size_t at) {
  NormIn n;
  n.o[0] = *reinterpret_cast<const f4*>(p.xf + at);
  n.o[1] = *reinterpret_cast<const f4*>(p.xf + at + 4);
  n.z = *reinterpret_cast<const u16x8*>(p.z + at);
  return n;
}
__device__ __forceinline__ void gated_rmsnorm8(const NormIn& n, const f4 (&gm)[2], float eps, float (&v)[8]) {
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += n.o[e / 4][e % 4] * n.o[e / 4][e % 4];
  ss = row16_sum(ss);
  const float rs = 1.0f / sqrtf(ss / 128.0f + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float zf = bf2f(n.z[e]);
    const float h = n.o[e / 4][e % 4] * rs * gm[e / 4][e % 4];
    v[e] = rbf(h * (zf * d_sigmoidf(zf)));
  }
}

// (a & m) | c: with m and c in VGPRs (opaque values from nibble_consts) the compiler selects
// one v_and_or_b32 for it -- with literal constants it cannot (a VOP3 takes no literal on
// this target and at most one SGPR) and emits a separate AND and OR. Written out in C, not
// as inline asm, so that the compiler also sees the instruction and keeps the wait states
// an MFMA reading its result needs.
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t c) { return (a & m) | c; }
struct NibbleConsts {
  uint32_t mask, bias;  // 0x000F000F, 0x43004300
};
__device__ __forceinline__ NibbleConsts nibble_consts() {
  NibbleConsts k;
  k.mask = 0x000F000Fu;
  k.bias = 0x43004300u;
  asm volatile("" : "+v"(k.mask), "+v"(k.bias));  // (emits nothing: keeps them opaque VGPR values)
  return k;
}

// A weight row's segment: its nibble words, scales, biases and output column. Every
// candidate is read as a value first and held opaque (the empty asm), then selected: a
// select between loads of the argument arrays is otherwise folded into one load at a
// run-time index, for which the compiler copies the kernel arguments to scratch.
struct RowPtrs {
  const uint32_t* w;
  const uint16_t *s, *b;
  uint16_t* y;
  int ystride;
};
__device__ __forceinline__ RowPtrs row_ptrs(const QParams& p, int layer, int row) {
  const uint32_t* wv[GDN_QLINEAR_MAX_SEGS];
  const uint16_t *sv[GDN_QLINEAR_MAX_SEGS], *bv[GDN_QLINEAR_MAX_SEGS];
  uint16_t* yv[GDN_QLINEAR_MAX_SEGS];
  int nv[GDN_QLINEAR_MAX_SEGS], rv[GDN_QLINEAR_MAX_SEGS];
#pragma unroll
  for (int q = 0; q < GDN_QLINEAR_MAX_SEGS; ++q) {
    wv[q] = p.w[q];
    sv[q] = p.s[q];
    bv[q] = p.b[q];
    yv[q] = p.y[q];
    nv[q] = p.n[q];
    rv[q] = p.row0[q];
    asm volatile("" : "+s"(wv[q]), "+s"(sv[q]), "+s"(bv[q]), "+s"(yv[q]), "+s"(nv[q]), "+s"(rv[q]));
  }
  int sg = 0;
#pragma unroll
  for (int q = 1; q < GDN_QLINEAR_MAX_SEGS; ++q) sg += (q < p.nseg && row >= rv[q]) ? 1 : 0;
  const uint32_t* wseg = wv[0];
  const uint16_t *sseg = sv[0], *bseg = bv[0];
  uint16_t* yseg = yv[0];
  int nseg = nv[0], r0 = rv[0];
#pragma unroll
  for (int q = 1; q < GDN_QLINEAR_MAX_SEGS; ++q) {
    if (sg == q) {
      wseg = wv[q];
      sseg = sv[q];
      bseg = bv[q];
      yseg = yv[q];
      nseg = nv[q];
      r0 = rv[q];
    }
  }
  const int G = p.K / 64;
  const size_t lrow = (size_t)layer * nseg + (row - r0);
  RowPtrs r;
  r.w = wseg + lrow * (p.K / 8);
  r.s = sseg + lrow * G;
  r.b = bseg + lrow * G;
  r.y = yseg + (size_t)layer * p.M * nseg + (row - r0);
  r.ystride = nseg;
  return r;
}

// W waves. NM: the operand's rows, 1 (no branch between the pieces' products) or up to
// GDN_QLINEAR_GEMV_ROWS.
template <int J, bool NORM, int W, int NM>
__global__ __launch_bounds__(64 * W) void qlinear_kernel(QParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // each wave's scale and bias words of its current 4 rows: [wave][row][scale, bias][group]
  __shared__ __attribute__((aligned(16))) uint16_t sbs[W][4][2][J * 8];
  const int layer = blockIdx.x / p.tiles;
  const int tile = blockIdx.x % p.tiles;
  constexpr int K = J * 512, nch = K / 32;
  u32x4* xs = reinterpret_cast<u32x4*>(smem);                 // [M][4][nch]
  float* xsum = reinterpret_cast<float*>(xs + p.M * 4 * nch);  // [M][nch]
  const int tid = threadIdx.x;
  const int lane = tid & 63, m = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int passes = p.passes;

  const int mc = m < J ? m : J - 1;  // the 8 groups whose scale and bias words the lane loads

  // ---- stage the operand ----
  if (NORM) {
    // a wave's 64 pieces of 8 values are 4 heads; a row's J of them go to the waves in turn,
    // their loads issued ahead of the arithmetic. Piece q is word q % 4 of chunk q / 4.
    constexpr int kMine = (J + W - 1) / W;
    const float* g = p.gamma + (size_t)layer * 128 + 8 * m;
    const f4 gm[2] = {*reinterpret_cast<const f4*>(g), *reinterpret_cast<const f4*>(g + 4)};
    for (int mm = 0; mm < p.M; ++mm) {
      const size_t base = ((size_t)layer * p.M + mm) * K + 8 * lane;
      NormIn in[kMine];
#pragma unroll
      for (int i = 0; i < kMine; ++i) in[i] = norm_load(p, base + 512 * min(wave + W * i, J - 1));
#pragma unroll
      for (int i = 0; i < kMine; ++i) {
        if (wave + W * i >= J) break;
        const int q = 64 * (wave + W * i) + lane;
        float v[8];
        gated_rmsnorm8(in[i], gm, p.eps, v);
        u32x4 wd;
#pragma unroll
        for (int e = 0; e < 4; ++e) wd[e] = pack_bf2(v[e], v[e + 4]);
        xs[(mm * 4 + (q & 3)) * nch + (q >> 2)] = wd;
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += v[e];
        sum += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0xB1, 0xF, 0xF, true));
        sum += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0x4E, 0xF, 0xF, true));
        if ((q & 3) == 0) xsum[mm * nch + (q >> 2)] = sum;
      }
    }
  } else {
    for (int t = tid; t < p.M * nch; t += 64 * W) stage_chunk(p, xs, xsum, nch, layer, t / nch, t % nch);
  }
  __syncthreads();

  // ---- passes of 4 rows per wave ----
  const NibbleConsts nk = nibble_consts();
  for (int pass = 0; pass < passes; ++pass) {
    // (the operand is read from LDS again in every pass: without branches between the products
    // the compiler would hold all of it in registers, 253 at K = 5120)
    if (NM == 1) asm volatile("" ::: "memory");
    const int grow = (tile * passes + pass) * (4 * W) + wave * 4 + (lane >> 4);
    const bool valid = grow < p.R;
    const int row = valid ? grow : p.R - 1;
    // the row's segment, selected here in the kernel's body: through row_ptrs the selection held
    // more registers than there are scalar ones and took about 85 vector instructions a pass more,
    // with K a variable (M = 2, 48 layers of in_proj 384-393 us against 376; K = 1024, 248,320
    // rows 38 us against 33)
    int sg = 0;
#pragma unroll
    for (int q = 1; q < GDN_QLINEAR_MAX_SEGS; ++q) sg += (q < p.nseg && row >= p.row0[q]) ? 1 : 0;
    const uint32_t* wseg = p.w[0];
    const uint16_t *sseg = p.s[0], *bseg = p.b[0];
    uint16_t* yseg = p.y[0];
    int nseg = p.n[0], r0 = p.row0[0];
#pragma unroll
    for (int q = 1; q < GDN_QLINEAR_MAX_SEGS; ++q) {
      if (sg == q) {
        wseg = p.w[q];
        sseg = p.s[q];
        bseg = p.b[q];
        yseg = p.y[q];
        nseg = p.n[q];
        r0 = p.row0[q];
      }
    }
    // the row's scale and bias words, 16 bytes a lane (groups 8 mc .. + 7; lanes past the row's
    // K / 512 chunks repeat the last), first: they arrive before the weights
    const size_t lrow = (size_t)layer * nseg + (row - r0);
    const u32x4* wr = reinterpret_cast<const u32x4*>(wseg + lrow * (K / 8));
    const u32x4 swd = *reinterpret_cast<const u32x4*>(sseg + lrow * (K / 64) + 8 * mc);
    const u32x4 bwd = *reinterpret_cast<const u32x4*>(bseg + lrow * (K / 64) + 8 * mc);
    u32x4 wv[J];
#pragma unroll
    for (int j = 0; j < J; ++j) wv[j] = __builtin_nontemporal_load(wr + m + 16 * j);
    // through this wave's LDS rows (written and read by this wave only: no barrier) to the
    // lanes that use them: piece m + 16 j is in group m / 2 + 8 j
    uint16_t* srl = &sbs[wave][lane >> 4][0][0];
    uint16_t* brl = &sbs[wave][lane >> 4][1][0];
    *reinterpret_cast<u32x4*>(srl + 8 * mc) = swd;
    *reinterpret_cast<u32x4*>(brl + 8 * mc) = bwd;
    float y[NM] = {};
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int c = m + 16 * j;
      const float sc = bf2f(srl[(m >> 1) + 8 * j]);
      const float off = bf2f(brl[(m >> 1) + 8 * j]) - 128.0f * sc;
      uint32_t pr[4][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t wd = wv[j][i];
#pragma unroll
        for (int q = 0; q < 4; ++q) pr[i][q] = and_or(wd >> (4 * q), nk.mask, nk.bias);
      }
#pragma unroll
      for (int mm = 0; mm < NM; ++mm) {
        if (NM == 1 || mm < p.M) {
          float acc = 0.0f;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const u32x4 xq = xs[(mm * 4 + i) * nch + c];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc = dot2(pr[i][q], xq[q], acc);
          }
          y[mm] = __builtin_fmaf(sc, acc, __builtin_fmaf(off, xsum[mm * nch + c], y[mm]));
        }
      }
    }
#pragma unroll
    for (int mm = 0; mm < NM; ++mm) {
      if (NM == 1 || mm < p.M) {
        const float tot = row16_sum(y[mm]);
        if (m == 0 && valid) yseg[((size_t)layer * p.M + mm) * nseg + (row - r0)] = f2bf(tot);
      }
    }
  }
}

// MFMA path, step 1: the operand (normalised when NORM) into the workspace's fragment
// order. Workgroup = 16 rows x 128 HH values of a layer (K / (128 HH) fastest, then row tiles);
// thread (r, j) takes the 8 values 8 j of each of the HH 128-value heads of row r, so a 16-lane
// DPP row holds one head of one row and reads its contiguous bytes, and the head's sum of squares
// is 8 terms per thread and a row sum. The 4 HH KB pass through LDS and leave in the workspace's
// order, 256 bytes or more at a time. (One thread per 8 values storing its own 16 bytes, its
// place found with 64-bit divisions, took 47-49 us for in_proj's 4096 rows, 14 us for 1024.)
template <bool NORM, int HH>
__global__ __launch_bounds__(kThreads) void qprep_kernel(QParams p) {
  __shared__ __attribute__((aligned(16))) u32x4 tile[HH * (256 + 256 / 16)];  // 16 bytes of padding every 256
  const int nch = p.K / 32, rows = 16 * p.mtiles;
  const int npc = p.K / (128 * HH), piece = blockIdx.x % npc, mtl = blockIdx.x / npc;
  const int mtile = mtl % p.mtiles, layer = mtl / p.mtiles;
  const int r = threadIdx.x >> 4, j = threadIdx.x & 15;
  const int mrow = 16 * mtile + r;
  const bool live = mrow < p.M;
  const size_t base = ((size_t)layer * p.M + (live ? mrow : 0)) * p.K + 128 * HH * piece + 8 * j;
  f4 gm[2];
  NormIn in[HH];
  u16x8 x[HH];
#pragma unroll
  for (int hh = 0; hh < HH; ++hh) {
    if (NORM) in[hh] = norm_load(p, base + 128 * hh);
    else x[hh] = *reinterpret_cast<const u16x8*>(p.x + base + 128 * hh);
  }
  if (NORM) {
    const float* g = p.gamma + (size_t)layer * 128 + 8 * j;
    gm[0] = *reinterpret_cast<const f4*>(g);
    gm[1] = *reinterpret_cast<const f4*>(g + 4);
  }
#pragma unroll
  for (int hh = 0; hh < HH; ++hh) {
    float v[8];
    if (NORM) {
      gated_rmsnorm8(in[hh], gm, p.eps, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = live ? v[e] : 0.0f;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = live ? bf2f(x[hh][e]) : 0.0f;
    }
    u32x4 q;
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = pack_bf2(v[e], v[e + 4]);
    // its place among the workgroup's 256 HH 16-byte pieces: 32-value piece c of its values,
    // quarter jq of it
    const int c = 4 * hh + (j >> 2), jq = j & 3;
    const int at = p.frag32 ? (8 * (c >> 1) + 2 * jq + (c & 1)) * 16 + r
                            : (2 * (c >> 1) + (jq & 1)) * 64 + 16 * (2 * (c & 1) + (jq >> 1)) + r;
    tile[at + (at >> 4)] = q;
    // the group's sum x: the 64 values of (row, group) are the 8 values of each of 8
    // consecutive threads, added in a fixed order (each thread's 8 in sequence, then a
    // butterfly over the 8 threads)
    float sx = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) sx += v[e];
    sx += __shfl_xor(sx, 1, 8);
    sx += __shfl_xor(sx, 2, 8);
    sx += __shfl_xor(sx, 4, 8);
    if ((j & 7) == 0)
      p.xsum[((size_t)layer * (p.K / 64) + 2 * HH * piece + 2 * hh + (j >> 3)) * rows + mrow] = sx;
  }
  __syncthreads();
  u32x4* out = reinterpret_cast<u32x4*>(p.xfrag);
#pragma unroll
  for (int i = 0; i < HH; ++i) {
    const int at = 256 * i + threadIdx.x;
    const u32x4 q = tile[at + (at >> 4)];
    if (p.frag32) {
      const int run = at >> 4;  // 16 rows of (group, block, half): 256 bytes
      out[((size_t)layer * (p.mtiles / 2) + mtile / 2) * nch * 128 + (size_t)piece * (512 * HH) + (run >> 1) * 64 +
          (run & 1) * 32 + (mtile & 1) * 16 + (at & 15)] = q;
    } else {
      out[((size_t)layer * p.mtiles + mtile) * nch * 64 + (size_t)piece * (256 * HH) + at] = q;
    }
  }
}

__device__ __forceinline__ f4 mfma(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A nibble word (values k .. k + 7) as a B fragment: bf16 128 + v, pairs (i, i + 4).
__device__ __forceinline__ bf8 nibbles_bf16(uint32_t wd, NibbleConsts k) {
  u32x4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = and_or(wd >> (4 * q), k.mask, k.bias);
  return __builtin_bit_cast(bf8, r);
}

// MFMA path, step 2. Workgroup = 16 NT weight rows (the output columns) x 16 MT operand
// rows; wave w takes the groups g = 4 i + w, i < G / 4, of the G = K / 64 groups (a multiple
// of 4 for every supported K), so the four groups of a weight row's 128-byte line are asked
// for by the four waves together and the line is fetched once (when each wave took a
// contiguous quarter of K, a line's four groups were read at four different times and
// lines were fetched again after eviction). Lane (g4, nn) = (l / 16, l % 16) takes the
// nibble words 8 g + 2 g4 + s of its row 16 nt + nn (loaded by another lane, see below) and
// gets C rows m = 4 g4 + i of column nn.
// Memory: the weight stream comes from HBM once, so what bounds the kernel is how many of
// its bytes each wave keeps in flight: every load is issued kRing groups ahead (the ring
// below), and the workgroup's scale and bias pairs are staged in LDS once at the start
// (they would otherwise be two more loads per row tile and group at the same depth).
constexpr int kRing = 2;  // groups in flight per wave (G / 4 is a multiple of it)
// F32: the operand is in qgemm_big_kernel's 32-row fragments (its leftover rows): this lane's
// values are block 2 (g4 % 2) + s of group g there, lane 32 (g4 / 2) + 16 (mt % 2) + nn.
template <int MT, int NT>
struct QgemmLds {
  static constexpr int kRows = 16 * NT;
  static constexpr int kMaxG = 8192 / 64;
  // scale | bias << 16 per (row, group), rows kMaxG + 1 words apart at most (a row stride
  // of G + 1 words puts the 16 rows a wave reads at once on distinct banks); at the end the
  // partial sums of waves 1..3
  union {
    uint32_t sb[kRows * (kMaxG + 1)];
    f4 red[3][MT * NT][64];
  };
  // the operand's group sums for this workgroup's MT m tiles, all groups: [group][16 MT]
  __attribute__((aligned(16))) float xs_l[kMaxG * 16 * MT];
};
template <int MT, int NT, bool F32>
__device__ __forceinline__ void qgemm_tile(const QParams& p, int bid, int nwg, QgemmLds<MT, NT>& sm) {
  constexpr int kRows = 16 * NT;
  // Workgroup = (layer, weight tile, m group), m groups fastest. Workgroups are dispatched to
  // the 8 XCDs round robin; the ids are renumbered (p.remap) so that each XCD runs a
  // contiguous range: with several m groups, all m groups of a weight tile on one XCD, one
  // after another, so its weight rows come from HBM once and from that XCD's L2 after; with
  // 8 layers or more, whole layers per XCD, so a layer's operand is read from HBM into one
  // L2 instead of all eight.
  if (p.remap) bid = (bid & 7) * (nwg >> 3) + (bid >> 3);
  const int mg = bid % p.mgroups, lt = bid / p.mgroups;
  const int layer = lt / p.tiles, tile = lt % p.tiles;
  const int mt0 = mg * MT;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, nn = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, G = K / 64, nch = K / 32, sbs = G + 1;
  const int ng = G / 4;  // this wave's groups: 4 i + wave, i < ng

  // Weight loads are laid out for the memory path, not for the MFMA: lane 4 r + c reads the
  // 8-byte chunk c (words 2 c, 2 c + 1) of row r's group, so the 32 bytes of a row's group
  // come from one lane quad in one L1 access (with lane 16 c + r reading them, the four
  // lanes of every quad hit four rows: four times the L1 accesses, and the address path
  // saturates). The B fragment wants chunk g4 of row nn in lane 16 g4 + nn, so each loaded
  // word pair crosses lanes with ds_bpermute before its nibbles are expanded.
  const int bsrc = (4 * nn + g4) * 4;  // byte address of the lane that loaded (nn, g4)
  g_u32x2* wr[NT];
  uint16_t* yr[NT];
  int ystride[NT];
  bool valid[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int grow = (tile * NT + nt) * 16 + nn;
    valid[nt] = grow < p.R;
    const RowPtrs rp = row_ptrs(p, layer, valid[nt] ? grow : p.R - 1);
    yr[nt] = rp.y;
    ystride[nt] = rp.ystride;
    const int lrow = (tile * NT + nt) * 16 + (lane >> 2);
    const RowPtrs rl = row_ptrs(p, layer, lrow < p.R ? lrow : p.R - 1);
    wr[nt] = (g_u32x2*)(rl.w) + (lane & 3);  // + 4 g: words 8 g + 2 c, +1
  }
  const bf8* xa = reinterpret_cast<const bf8*>(p.xfrag + ((size_t)layer * p.mtiles + mt0) * nch * 512) +
                  (F32 ? 128 * (g4 & 1) + 32 * (g4 >> 1) + nn : lane);
  const NibbleConsts nk = nibble_consts();

  // A ring of kRing slots, one group each (operand fragments and nibble words): slot j
  // holds groups j, j + kRing, ... and is reloaded with the group kRing ahead right after
  // its products, so every load is issued kRing groups before its use. (Loads complete in
  // issue order: a nearer load issued after a farther one would wait for it.) Loads past
  // the wave's last group reload that group, unused.
  struct Slot {
    bf8 a[MT][2];
    u32x2 w[NT];
  };
  auto load = [&](int g, Slot& sl) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        sl.a[mt][s] = F32 ? xa[((size_t)(mt / 2) * nch * 2 + 4 * g + s) * 64 + 16 * (mt & 1)]
                          : xa[((size_t)mt * nch + 2 * g + s) * 64];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sl.w[nt] = wr[nt][4 * g];
  };
  Slot R[kRing];
#pragma unroll
  for (int j = 0; j < kRing; ++j) load(4 * j + wave, R[j]);  // (ng >= kRing)

  // the scale and bias pairs of the workgroup's rows, all groups: thread t takes row
  // t / (256 / kRows), four groups at a time (8-byte loads: G and the block starts are
  // multiples of 4)
  {
    constexpr int tpr = kThreads / kRows;
    const int r = threadIdx.x / tpr, j = threadIdx.x % tpr;
    const int grow = tile * kRows + r;
    const RowPtrs rp = row_ptrs(p, layer, grow < p.R ? grow : p.R - 1);
    for (int g = 4 * j; g < G; g += 4 * tpr) {
      const u32x2 sv = *(g_u32x2*)(rp.s + g);
      const u32x2 bv = *(g_u32x2*)(rp.b + g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t s16 = (sv[e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
        const uint32_t b16 = (bv[e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
        sm.sb[r * sbs + g + e] = s16 | (b16 << 16);
      }
    }
    // the group sums: 4 MT float4 per group, contiguous in xsum
    const float* xsg = p.xsum + (size_t)layer * G * (16 * p.mtiles) + 16 * mt0;
    for (int q = threadIdx.x; q < 4 * MT * G; q += kThreads) {
      const int g = q / (4 * MT), o = 4 * (q % (4 * MT));
      *reinterpret_cast<f4*>(&sm.xs_l[g * 16 * MT + o]) = *reinterpret_cast<const f4*>(xsg + (size_t)g * 16 * p.mtiles + o);
    }
  }
  __syncthreads();

  f4 y[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) y[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};

  // the wave's i-th group from slot sl, then sl reloaded with its (i + kRing)-th
  auto step = [&](int i, Slot& sl) {
    const int g = 4 * i + wave;
    f4 xs[MT];  // sum x of the group for this lane's rows 4 g4 .. + 3 of each m tile
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xs[mt] = *reinterpret_cast<const f4*>(&sm.xs_l[g * 16 * MT + 16 * mt + 4 * g4]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint32_t sbv = sm.sb[(16 * nt + nn) * sbs + g];
      const float sc = __builtin_bit_cast(float, sbv << 16);
      const float off = __builtin_bit_cast(float, sbv & 0xFFFF0000u) - 128.0f * sc;
      const uint32_t w0 = (uint32_t)__builtin_amdgcn_ds_bpermute(bsrc, (int)sl.w[nt][0]);
      const uint32_t w1 = (uint32_t)__builtin_amdgcn_ds_bpermute(bsrc, (int)sl.w[nt][1]);
      const bf8 b0 = nibbles_bf16(w0, nk), b1 = nibbles_bf16(w1, nk);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        f4 acc = mfma(sl.a[mt][0], b0, f4{0.f, 0.f, 0.f, 0.f});
        acc = mfma(sl.a[mt][1], b1, acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[mt][nt][i] = __builtin_fmaf(sc, acc[i], __builtin_fmaf(off, xs[mt][i], y[mt][nt][i]));
      }
    }
    load(4 * min(i + kRing, ng - 1) + wave, sl);
  };
  for (int ib = 0; ib < ng; ib += kRing) {
#pragma unroll
    for (int j = 0; j < kRing; ++j) step(ib + j, R[j]);
  }

  // the four waves' partial sums (fixed order: wave 0 + 1 + 2 + 3), rounded to bf16 once
  __syncthreads();  // every wave is done with the scale and bias pairs
  if (wave > 0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) sm.red[wave - 1][mt * NT + nt][lane] = y[mt][nt];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        f4 t = y[mt][nt];
#pragma unroll
        for (int w = 0; w < 3; ++w) t = t + sm.red[w][mt * NT + nt][lane];
        if (valid[nt]) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int m = (mt0 + mt) * 16 + 4 * g4 + i;
            if (m < p.M) yr[nt][(size_t)m * ystride[nt]] = f2bf(t[i]);
          }
        }
      }
  }
}

template <int MT, int NT>
__global__ __launch_bounds__(kThreads) void qgemm_kernel(QParams p) {
  __shared__ __attribute__((aligned(16))) QgemmLds<MT, NT> sm;
  qgemm_tile<MT, NT, false>(p, blockIdx.x, gridDim.x, sm);
}

// MFMA path for calls of many weight rows and few operand rows (one m group of up to 48 rows;
// 8 layers or more of in_proj per call): workgroup = 256 weight rows, wave w owns 64 of them
// (kNsTiles 16-row tiles) over the whole of K, and the four waves share the operand, which
// passes through an LDS ring once per workgroup (qgemm_kernel reads it from L2 once per 64
// rows). A step is two groups. Direct-to-LDS loads (`global_load_lds_dwordx4`: lane l's 16
// bytes land at the destination + 16 l, no VGPRs) fill the ring kNsAhead steps ahead: each
// wave issues one of the step's four 1 KB blocks of every m tile, waits for its own loads,
// and one barrier per step then makes the slot whole for all four. Each wave also loads the
// scale words of its rows, 8 groups at a time, into its own pair of LDS buffers (read by that
// wave only: no barrier). The weight words stay in a register ring, loaded and moved into
// fragment order as in qgemm_kernel. Loads complete in issue order and the waits count them,
// so every step issues the same loads (past the last step they repeat it), and no lane is
// masked off in the loop (a divergent branch there split the loop into blocks, after which
// the compiler sank a step's FMAs to its end with every MFMA result live). Per group
// y += s * sum x (128 + q) as in qgemm_kernel, each wave adding its groups in order; the
// bias term sum_g (b_g - 128 s_g) sum x_g is made after the loop as MFMA products (below),
// and each row is rounded once.
constexpr int kNsTiles = 4;
constexpr int kNsRows = 4 * 16 * kNsTiles;  // weight rows per workgroup
constexpr int kNsAhead = 2;                 // steps between a load and its use
typedef __attribute__((address_space(3))) void lds_void;
// Direct-to-LDS loads written as asm: the compiler, which cannot tell which LDS bytes such a
// load writes, otherwise waits for every one in flight (vmcnt(0)) at points in the loop, which
// would undo the ring. The asm statements have a memory clobber (no memory access moves
// across them); the kernel waits for them itself. M0 carries the LDS destination and is
// restored after the load has been issued (the load takes it at issue), so the compiler's
// view of M0 is never disturbed.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p);
}
__device__ __forceinline__ void dma16(const void* src, uint32_t lds) {
  uint32_t m0_saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(m0_saved)
               : "v"(src), "s"(lds)
               : "memory");
}
// four consecutive 1 KB blocks from a wave-uniform address (the instruction offset moves both
// addresses); voff = 16 x lane
__device__ __forceinline__ void dma16x4(const void* src, uint32_t voff, uint32_t lds) {
  uint32_t m0_saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024\n\t"
               "global_load_lds_dwordx4 %1, %2 offset:2048\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(m0_saved)
               : "v"(voff), "s"(src), "s"(lds)
               : "memory");
}
// two consecutive blocks from one uniform address, a lane's source offsets v0 and v1
__device__ __forceinline__ void dma16x2(const void* src, uint32_t v0, uint32_t v1, uint32_t lds) {
  uint32_t m0_saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\t"
               "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(m0_saved)
               : "v"(v0), "v"(v1), "s"(src), "s"(lds)
               : "memory", "scc");
}
// one block where `skip` (wave-uniform) is 0; the branch is inside the asm, so that the
// compiler's basic block -- and the order of the products and sums in it -- stays whole
__device__ __forceinline__ void dma16_unless(int skip, const void* src, uint32_t voff, uint32_t lds) {
  uint32_t m0_saved;
  asm volatile("s_cmp_lg_u32 %4, 0\n\ts_cbranch_scc1 1f\n\t"
               "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0\n1:"
               : "=&s"(m0_saved)
               : "v"(voff), "s"(src), "s"(lds), "s"(skip)
               : "memory", "scc");
}

template <int MT>
__global__ __launch_bounds__(kThreads) void qgemm_ns_kernel(QParams p) {
  constexpr int NT = kNsTiles, D = kNsAhead, S = D + 1;
  constexpr int kSlot = MT * 4 * 1024;     // a slot: [m tile][group of the step][k step] 1 KB operand blocks
  constexpr int kPerStep = MT + 2 * NT;    // vector-memory instructions per wave and step
  constexpr int kMaxG = 8192 / 64;
  __shared__ __attribute__((aligned(16))) unsigned char ring[S * kSlot];
  __shared__ __attribute__((aligned(16))) uint16_t sbl[4][2][64 * 8];  // scale words: [wave][buffer][row][8 groups]
  __shared__ __attribute__((aligned(16))) float xs_all[kMaxG * 16 * MT];  // the sums x: [group][16 MT]

  int bid = blockIdx.x;
  if (p.remap) bid = (bid & 7) * (int)(gridDim.x >> 3) + (bid >> 3);
  const int layer = bid / p.tiles, tile = bid % p.tiles;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, nn = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, G = K / 64, nch = K / 32, nsteps = G / 2, nblk = G / 8;
  const int rbase = (tile * 4 + wave) * 16 * NT;
  const int bsrc = (4 * nn + g4) * 4;  // as in qgemm_kernel
  g_u32x2* wr[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int lrow = rbase + 16 * nt + (lane >> 2);
    const RowPtrs rl = row_ptrs(p, layer, lrow < p.R ? lrow : p.R - 1);
    wr[nt] = (g_u32x2*)(rl.w) + (lane & 3);
  }
  // lane l loads the scale words of the wave's row l
  const RowPtrs rsb = row_ptrs(p, layer, min(rbase + lane, p.R - 1));
  const char* s_src = reinterpret_cast<const char*>(rsb.s);
  const char* xa = reinterpret_cast<const char*>(p.xfrag + (size_t)layer * MT * nch * 512) + 16 * lane;
  // the layer's sums x, all groups, for the bias products after the loop (one barrier: the
  // loop issues no load before it)
  {
    const f4* src = reinterpret_cast<const f4*>(p.xsum + (size_t)layer * G * 16 * MT);
    for (int q = threadIdx.x; q < G * 4 * MT; q += kThreads) reinterpret_cast<f4*>(xs_all)[q] = src[q];
  }
  __syncthreads();
  const NibbleConsts nk = nibble_consts();

  // step j's loads: the wave's block (group 2 j + wave / 2, k step wave % 2) of every m tile
  // and its share of the sums into ring slot sl; its weight words into ws
  const uint32_t ring_l = lds_addr(ring);
  auto issue_op = [&](int j, int sl) {
    const uint32_t dst = ring_l + sl * kSlot;
#pragma unroll
    for (int i = 0; i < MT; ++i) dma16(xa + ((size_t)i * nch + 4 * j + wave) * 1024, dst + (4 * i + wave) * 1024);
  };
  struct WStep {
    u32x2 w[2][NT];
  };
  auto issue_w = [&](int j, WStep& ws) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      g_u32x2* wj = wr[nt] + 8 * j;
      ws.w[0][nt] = wj[0];
      ws.w[1][nt] = wj[4];
    }
  };
  // scale and bias words of groups 8 blk .. + 7 into buffer buf
  const uint32_t sbl_l = lds_addr(&sbl[wave][0][0]);
  auto issue_sb = [&](int blk, int buf) { dma16(s_src + 16 * blk, sbl_l + buf * 1024); };

  f4 y[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) y[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int j, const unsigned char* slot, const uint16_t* sbw, const WStep& ws) {
    // the scale words of the step's two groups, one 4-byte read per tile
    uint32_t sw[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sw[nt] = *reinterpret_cast<const uint32_t*>(sbw + (16 * nt + nn) * 8 + ((2 * j) & 7));
#pragma unroll
    for (int gg = 0; gg < 2; ++gg) {
      bf8 a[MT][2];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int s = 0; s < 2; ++s) a[mt][s] = *reinterpret_cast<const bf8*>(slot + (4 * mt + 2 * gg + s) * 1024 + 16 * lane);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float sc = __builtin_bit_cast(float, gg ? sw[nt] & 0xFFFF0000u : sw[nt] << 16);
        const uint32_t w0 = (uint32_t)__builtin_amdgcn_ds_bpermute(bsrc, (int)ws.w[gg][nt][0]);
        const uint32_t w1 = (uint32_t)__builtin_amdgcn_ds_bpermute(bsrc, (int)ws.w[gg][nt][1]);
        const bf8 b0 = nibbles_bf16(w0, nk), b1 = nibbles_bf16(w1, nk);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          f4 acc = mfma(a[mt][0], b0, f4{0.f, 0.f, 0.f, 0.f});
          acc = mfma(a[mt][1], b1, acc);
#pragma unroll
          for (int i = 0; i < 4; ++i) y[mt][nt][i] = __builtin_fmaf(sc, acc[i], y[mt][nt][i]);
        }
      }
    }
  };

  WStep W[2];
  issue_sb(0, 0);
#pragma unroll
  for (int j = 0; j < D; ++j) {
    issue_op(j, j);
    issue_w(j, W[j]);
  }
  int sl = 0;  // ring slot of step j
  for (int j0 = 0; j0 < nsteps; j0 += 4) {  // nsteps is a multiple of 4 (G of 8)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = j0 + r;
      // step j's loads are done once no more than the loads issued after them are in flight:
      // step j + 1's, and also the scale words issued at step 4 b after step 4 b + 2's (in
      // flight at steps 4 b + 1 and 4 b + 2); then every wave's are (the barrier). The wait
      // and the barrier are one asm statement with a memory clobber, so no load moves across
      // them.
      if (r == 1 || r == 2)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kPerStep + 1) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kPerStep) : "memory");
      compute(j, ring + sl * kSlot, &sbl[wave][(j >> 2) & 1][0], W[r & 1]);
      __builtin_amdgcn_sched_barrier(0);
      // refill what step j - 1 read (every wave is past it: the barrier above)
      const int jn = min(j + D, nsteps - 1);
      issue_op(jn, sl == 0 ? S - 1 : sl - 1);
      issue_w(jn, W[r & 1]);
      if (r == 0) issue_sb(min((j >> 2) + 1, nblk - 1), ((j >> 2) + 1) & 1);
      sl = sl == S - 1 ? 0 : sl + 1;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the repeated loads, before the LDS goes away
  // this lane's output rows, their scale and bias words: found here rather than held in
  // registers through the loop
  uint16_t* yr[NT];
  const uint16_t *srow[NT], *brow[NT];
  int ystride[NT];
  bool valid[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int grow = rbase + 16 * nt + nn;
    valid[nt] = grow < p.R;
    const RowPtrs rp = row_ptrs(p, layer, valid[nt] ? grow : p.R - 1);
    yr[nt] = rp.y;
    ystride[nt] = rp.ystride;
    srow[nt] = rp.s;
    brow[nt] = rp.b;
  }

  // The bias term sum_g (b_g - 128 s_g) sum x_g = Yb - 128 Ys, Yb = sum_g b_g sum x_g and
  // Ys = sum_g s_g sum x_g, on MFMA after the loop (it was two FMAs per element and group):
  // A = the sums x of 16 operand rows x 32 groups, each split into three bf16 terms (exact to
  // about 2^-24 of it), B = the rows' bias / scale words of the same groups (bf16, exact);
  // groups past G are zeros. Lane (g4, r) takes groups 32 ks + 8 g4 .. + 7.
  {
    f4 yb[MT][NT], ysc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) yb[mt][nt] = ysc[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < (G + 31) / 32; ++ks) {
      const int g0 = 32 * ks + 8 * g4;
      const bool live = g0 < G;  // G is a multiple of 16: all eight or none
      bf8 bb[NT], bs[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        u32x4 vb{}, vs{};
        if (live) {
          const u32x2 b0 = *(g_u32x2*)(brow[nt] + g0), b1 = *(g_u32x2*)(brow[nt] + g0 + 4);
          const u32x2 s0 = *(g_u32x2*)(srow[nt] + g0), s1 = *(g_u32x2*)(srow[nt] + g0 + 4);
          vb = u32x4{b0[0], b0[1], b1[0], b1[1]};
          vs = u32x4{s0[0], s0[1], s1[0], s1[1]};
        }
        bb[nt] = __builtin_bit_cast(bf8, vb);
        bs[nt] = __builtin_bit_cast(bf8, vs);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = live ? xs_all[(g0 + i) * 16 * MT + 16 * mt + nn] : 0.0f;
        bf8 hi, mid, lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float h = rbf(v[i]);
          const float r1 = v[i] - h;
          const float m1 = rbf(r1);
          hi[i] = __builtin_bit_cast(__bf16, (uint16_t)(__builtin_bit_cast(uint32_t, h) >> 16));
          mid[i] = __builtin_bit_cast(__bf16, (uint16_t)(__builtin_bit_cast(uint32_t, m1) >> 16));
          lo[i] = (__bf16)(r1 - m1);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          yb[mt][nt] = mfma(hi, bb[nt], yb[mt][nt]);
          yb[mt][nt] = mfma(mid, bb[nt], yb[mt][nt]);
          yb[mt][nt] = mfma(lo, bb[nt], yb[mt][nt]);
          ysc[mt][nt] = mfma(hi, bs[nt], ysc[mt][nt]);
          ysc[mt][nt] = mfma(mid, bs[nt], ysc[mt][nt]);
          ysc[mt][nt] = mfma(lo, bs[nt], ysc[mt][nt]);
        }
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) y[mt][nt][i] += __builtin_fmaf(-128.0f, ysc[mt][nt][i], yb[mt][nt][i]);
  }

#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (valid[nt]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = mt * 16 + 4 * g4 + i;
          if (m < p.M) yr[nt][(size_t)m * ystride[nt]] = f2bf(y[mt][nt][i]);
        }
      }
    }
}

// MFMA path for many operand rows: an LDS-tiled product on v_mfma_f32_32x32x16_bf16.
// Workgroup = 4 waves as WN x WK over a tile of 32 MTW operand rows x 64 WN weight rows of one
// matrix; the WK wave sets take every WK-th group of K and add their sums in LDS at the end.
// Two workgroups share a CU (80 KB of LDS each), so that one's barriers fall into the other's
// products. A step is WK groups: its operand blocks (16 KB) and nibble words (8 KB) pass
// through a ring of kBigSlots LDS slots filled by direct-to-LDS loads ahead of their use; each
// wave's scale words come 8 groups at a time into its own pair of buffers. Per group and
// 32 x 32 tile: four products into acc = sum x (16 + q), then y += s acc (16 FMAs a lane
// beside 128 cycles of MFMA); the bias term is made on MFMA, as qgemm_ns_kernel does. Nibble q is the bf16 16 + q here (q in the mantissa's upper
// four bits: one shift more per word than 128 + q): the terms of the offset are summed apart
// from the products that cancel them, so their size is what the fp32 sums round at, and with
// 128 the outputs lay further from the exact product than qgemm_kernel's, which cancels them
// group by group (with 16 they lie as near or nearer, see the bias term in the kernel).
typedef float f16v __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f16v mfma32(bf8 a, bf8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// Nibble word (values k .. k + 7) as a B fragment: bf16 16 + v, pairs (i, i + 4).
__device__ __forceinline__ NibbleConsts nibble16_consts() {
  NibbleConsts k;
  k.mask = 0x00780078u;
  k.bias = 0x41804180u;
  asm volatile("" : "+v"(k.mask), "+v"(k.bias));
  return k;
}
__device__ __forceinline__ bf8 nibbles16_bf16(uint32_t wd, NibbleConsts k) {
  u32x4 r;
  r[0] = and_or(wd << 3, k.mask, k.bias);
#pragma unroll
  for (int q = 1; q < 4; ++q) r[q] = and_or(wd >> (4 * q - 3), k.mask, k.bias);
  return __builtin_bit_cast(bf8, r);
}
constexpr int kBigSlots = 3;
constexpr int kRestTiles = 2;  // 16-row tiles of a workgroup of leftover rows
template <int WN, int WK, int MTW>
struct BigCfg {
  static constexpr int NTW = 2;                    // 32-row weight tiles of a wave
  static constexpr int kRows = 64 * WN;            // weight rows of the tile
  static constexpr int kABytes = MTW * WK * 4096;  // operand bytes of a step
  static constexpr int kWBytes = WN * WK * 2048;   // nibble bytes of a step
  static constexpr int kSlot = kABytes + kWBytes;
  static constexpr int kPerStep = 6;               // loads of a wave and step: 4 + 2
  static constexpr int kSbStride = 8 / WK;         // steps an 8-group block of scale words lasts
  static constexpr size_t kLds = kBigSlots * kSlot + 4 * 2 * 1024;
  static_assert(WN * WK == 4 && MTW * WK == 4, "4 waves share each step's loads evenly");
};

// The rows past each matrix's whole tiles (r: in_proj_a and in_proj_b are all such rows) are
// qgemm_kernel's tiles, in the first `nrest` workgroups of the same launch: in a launch of
// their own the in_proj's 96 rows took 17 us after 1024 operand rows and 40 us after 4096, here
// they run beside the first tiles.
template <int WN, int WK, int MTW, bool REST>
__global__ __launch_bounds__(kThreads, 2) void qgemm_big_kernel(QParams p, QParams r, int nrest) {
  using C = BigCfg<WN, WK, MTW>;
  constexpr int NTW = C::NTW;
  __shared__ __attribute__((aligned(16))) unsigned char smem[C::kLds];
  unsigned char* const ring = smem;
  uint16_t* const sbl_all = reinterpret_cast<uint16_t*>(smem + kBigSlots * C::kSlot);  // [wave][2][64 rows][8 groups]
  // Workgroups are dispatched to the XCDs round robin: each XCD takes a contiguous range of
  // tile ids, in which panels of 8 weight tiles run weight tile fastest, so the tiles one XCD
  // runs at once share their weight and operand slices through its L2.
  int bid = blockIdx.x;
  if (REST && bid < nrest) {
    static_assert(sizeof(QgemmLds<4, kRestTiles>) <= C::kLds, "the leftover rows' tiles fit the same LDS");
    if (bid < r.tiles * r.mgroups * r.layers)
      qgemm_tile<4, kRestTiles, true>(r, bid, 0, *reinterpret_cast<QgemmLds<4, kRestTiles>*>(smem));
    return;
  }
  if (REST) bid -= nrest;  // (a multiple of 8: the XCDs keep their turns)
  if (p.remap) bid = (bid & 7) * (int)((gridDim.x - (REST ? nrest : 0)) >> 3) + (bid >> 3);
  const int per_layer = p.tiles * p.mgroups;
  const int layer = bid / per_layer;
  int rem = bid % per_layer;
  const int panel = rem / (8 * p.mgroups);
  const int width = min(8, p.tiles - 8 * panel);
  rem -= panel * 8 * p.mgroups;
  const int tile = 8 * panel + rem % width, mg = rem / width;

  // the tile's matrix (row0 counts whole tiles here) and its base addresses, wave-uniform
  const uint32_t* wseg = p.w[0];
  const uint16_t *sseg = p.s[0], *bseg = p.b[0];
  uint16_t* yseg = p.y[0];
  int nseg = p.n[0], t0 = 0;
#pragma unroll
  for (int q = 1; q < GDN_QLINEAR_MAX_SEGS; ++q) {
    if (q < p.nseg && tile >= p.row0[q]) {
      wseg = p.w[q];
      sseg = p.s[q];
      bseg = p.b[q];
      yseg = p.y[q];
      nseg = p.n[q];
      t0 = p.row0[q];
    }
  }
  const int lane = threadIdx.x & 63, h = lane >> 5, nn = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave % WK, wn = wave / WK;
  const int G = p.K / 64, nsteps = G / WK, nblk = G / 8;
  const int mblk = p.mtiles / 2;  // the operand's 32-row blocks
  const int mb0 = mg * MTW;
  const int nbase = (tile - t0) * C::kRows + 64 * wn;  // this wave's first row of the matrix
  const size_t wrow = (size_t)p.K / 2;                 // bytes of a weight row
  const char* const wb = reinterpret_cast<const char*>(wseg) + (size_t)layer * nseg * wrow;
  const char* const sb = reinterpret_cast<const char*>(sseg) + (size_t)layer * nseg * (2 * G);
  const char* const bb = reinterpret_cast<const char*>(bseg) + (size_t)layer * nseg * (2 * G);

  // this wave's loads of a step: the four blocks of one (group, operand block) and the nibble
  // words of its own 64 rows and group in two loads of 32 rows, a lane pair the 32 bytes of a
  // row (the halves of rows 4..7 of every 8 swapped: eight lanes of a read then hit distinct
  // banks). Offsets of lanes in a matrix: 32 bits (the host checks it).
  const int a_kg = wave / MTW, a_mb = wave % MTW;
  const char* const a_src = reinterpret_cast<const char*>(p.xfrag) +
                            (((size_t)layer * mblk + min(mb0 + a_mb, mblk - 1)) * G + a_kg) * 4096;
  uint32_t w_off[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t)
    w_off[t] = (uint32_t)(min(nbase + 32 * t + (lane >> 1), nseg - 1) * wrow) + 16 * ((lane & 1) ^ ((lane >> 3) & 1));
  const uint32_t s_off = (uint32_t)min(nbase + lane, nseg - 1) * (2 * G);
  const uint32_t ring_l = lds_addr(ring);
  const uint32_t sb_l = lds_addr(sbl_all) + wave * 2048;
  auto issue = [&](int j, int sl) {
    const uint32_t dst = ring_l + sl * C::kSlot;
    dma16x4(a_src + (size_t)j * (WK * 4096), 16 * lane, dst + (a_kg * MTW + a_mb) * 4096);
    dma16x2(wb + (j * WK + wk) * 32, w_off[0], w_off[1], dst + C::kABytes + (wk * WN + wn) * 2048);
  };

  f16v y[MTW][NTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) y[mt][nt][i] = 0.0f;
  const NibbleConsts nk = nibble16_consts();

  dma16_unless(0, sb, s_off, sb_l);  // the first 8 groups' scale words
#pragma unroll
  for (int j = 0; j < kBigSlots; ++j) issue(min(j, nsteps - 1), j);

  // The bias term sum_g (b_g - 16 s_g) sum x_g, 16 groups at a time: y += on MFMA, A = the sums x
  // of 32 operand rows x 16 groups, each split into three bf16 terms (exact to about 2^-24 of
  // it), B = the rows' biases and their scales times -16 (exact in bf16). A block's term is added
  // just before its groups' products, which cancel most of it, so that y stays near its final
  // size. With K split, the wave set wk adds every WK-th block, before the products of WK blocks'
  // groups (the first while the ring fills). Shares of the outputs off the exact product's
  // rounding at operands N(0, 1), then N(0.1, 1): large tiles (in_proj M = 1024) 0.5e-3, 1.2e-3;
  // small tiles (M = 333) 0.8e-3, 1.4e-3; qgemm_kernel 1.2e-3, 1.5e-3. With the whole term first,
  // as the small tiles had it, 1.0e-3 and 3.0e-3, for 1 us less of 99 (out_proj M = 333: 2.7e-3,
  // whole term first 2.8e-3, qgemm_kernel 3.3e-3). Past a mean of about 0.2 qgemm_kernel's sums,
  // which cancel group by group, lie nearer: N(1, 1) 4.0e-3 against 6.3e-3 and 6.4e-3.
  const int rows = 16 * p.mtiles, nks = G / 16;
  const float* const xs0 = p.xsum + (size_t)layer * G * rows;
  struct BiasBlock {
    u32x4 s[NTW], b[NTW];
    float v[MTW][8];
  };
  // the lane, opaque: the addresses below are made from it at each use and hold no registers in
  // the loop
  auto opaque_lane = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  auto load_rows = [&](int ks, int l, BiasBlock& q) {
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      const uint32_t off = (uint32_t)min(nbase + 32 * nt + (l & 31), nseg - 1) * (2 * G) + 16 * (l >> 5) + 32 * ks;
      q.s[nt] = *reinterpret_cast<const u32x4*>(sb + off);
      q.b[nt] = *reinterpret_cast<const u32x4*>(bb + off);
    }
  };
  auto load_sums = [&](int ks, int l, int mt, BiasBlock& q) {
    const uint32_t off = (uint32_t)(16 * ks + 8 * (l >> 5)) * rows + 32 * min(mb0 + mt, mblk - 1) + (l & 31);
#pragma unroll
    for (int i = 0; i < 8; ++i) q.v[mt][i] = xs0[off + (uint32_t)(i * rows)];
  };
  // (with `sums`, inside the loop, the sums are loaded here, an operand block at a time: no
  // registers for all of them beside the loop's)
  auto add_bias = [&](BiasBlock& q, int ks, int l, bool sums) {
    bf8 b0[NTW], s0[NTW];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      b0[nt] = __builtin_bit_cast(bf8, q.b[nt]);
      u32x4 t;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = -16.0f * __builtin_bit_cast(float, q.s[nt][e] << 16);
        const float hi = -16.0f * __builtin_bit_cast(float, q.s[nt][e] & 0xFFFF0000u);
        t[e] = (__builtin_bit_cast(uint32_t, lo) >> 16) | (__builtin_bit_cast(uint32_t, hi) & 0xFFFF0000u);
      }
      s0[nt] = __builtin_bit_cast(bf8, t);
    }
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      if (sums) load_sums(ks, l, mt, q);
      bf8 x3[3];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float hv = rbf(q.v[mt][i]);
        const float r1 = q.v[mt][i] - hv;
        const float m1 = rbf(r1);
        x3[0][i] = __builtin_bit_cast(__bf16, (uint16_t)(__builtin_bit_cast(uint32_t, hv) >> 16));
        x3[1][i] = __builtin_bit_cast(__bf16, (uint16_t)(__builtin_bit_cast(uint32_t, m1) >> 16));
        x3[2][i] = (__bf16)(r1 - m1);
      }
#pragma unroll
      for (int t = 2; t >= 0; --t)
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          y[mt][nt] = mfma32(x3[t], b0[nt], y[mt][nt]);
          y[mt][nt] = mfma32(x3[t], s0[nt], y[mt][nt]);
        }
      if (sums && mt % 2) __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (WK > 1 && wk < nks) {
    BiasBlock q;
    load_rows(wk, lane, q);
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) load_sums(wk, lane, mt, q);
    add_bias(q, wk, lane, false);
  }

  // The loop. A step's 2 MTW tiles in sequence, each tile's FMAs between the next one's MFMAs
  // (the last tile's in the next step). Left to itself the compiler issues a tile's four MFMAs
  // and then all its FMAs, so the order is held by schedule barriers. The step's one barrier
  // stands before its last two tiles, behind which nothing reads the step's slot any more:
  // there every wave's loads of the next step are done (all but the newest step's are, in each
  // wave, by its wait), so the last tiles already read the next step's first operands, and the
  // slot is refilled with the step kBigSlots ahead.
  constexpr int T = MTW * NTW;
  static_assert(T >= 4 && NTW == 2, "the operand blocks of a step are read before its last two tiles");
  bf8 b[NTW][4], a[2][4];
  float sc[NTW], slast = 0.0f;
  u32x4 wd[NTW];
  f16v acc[2] = {f16v{}, f16v{}};  // tile t in acc[t & 1]
  auto read_a = [&](const unsigned char* slot, int mt, int s) {
    a[mt & 1][s] = *reinterpret_cast<const bf8*>(slot + ((wk * MTW + mt) * 4 + s) * 1024 + 16 * lane);
  };
  auto read_w = [&](const unsigned char* slot, int nt) {
    wd[nt] = *reinterpret_cast<const u32x4*>(slot + C::kABytes + ((wk * WN + wn) * NTW + nt) * 1024 + 32 * nn +
                                             16 * (h ^ ((nn >> 2) & 1)));
  };
  auto read_s = [&](int j, int nt) {
    return bf2f(sbl_all[wave * 1024 + ((j / C::kSbStride) & 1) * 512 + ((j * WK + wk) & 7) + (32 * nt + nn) * 8]);
  };
  auto add = [&](f16v& yt, const f16v& v, float c, int q) {
#pragma unroll
    for (int i = 4 * q; i < 4 * q + 4; ++i) yt[i] = __builtin_fmaf(c, v[i], yt[i]);
  };
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * C::kPerStep) : "memory");
#pragma unroll
  for (int nt = 0; nt < NTW; ++nt) {
    read_w(ring, nt);
    sc[nt] = read_s(0, nt);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) read_a(ring, 0, s);
#pragma unroll
  for (int s = 0; s < 4; ++s) b[0][s] = nibbles16_bf16(wd[0][s], nk);
  int sl = 0;
  for (int j0 = 0; j0 < nsteps; j0 += 16) {  // the steps of WK bias blocks
  const int ks = j0 / 16 * WK + wk;
  if (WK == 1 || (j0 > 0 && ks < nks)) {
    BiasBlock q;
    const int l = opaque_lane();
    load_rows(ks, l, q);
    add_bias(q, ks, l, true);
  }
  const int j1 = WK == 1 ? j0 + 16 : min(j0 + 16, nsteps);
  for (int j = j0; j < j1; ++j) {
    const unsigned char* slot = ring + sl * C::kSlot;
    const int sn = sl == kBigSlots - 1 ? 0 : sl + 1;
    const unsigned char* next = ring + sn * C::kSlot;
    float scn[NTW];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int mt = t / NTW, nt = t % NTW;
      if (t == T - 2) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::kPerStep) : "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        acc[t & 1] = mfma32(a[mt & 1][s], b[nt][s], s == 0 ? f16v{} : acc[t & 1]);
        if (t == 0) {
          add(y[MTW - 1][NTW - 1], acc[(T - 1) & 1], slast, s);
          b[1][s] = nibbles16_bf16(wd[1][s], nk);
        } else {
          add(y[(t - 1) / NTW][(t - 1) % NTW], acc[(t - 1) & 1], sc[(t - 1) % NTW], s);
        }
        // LDS reads, at most one a product: the next operand block's over this one's two tiles
        if (mt + 1 < MTW) {
          if (s % 2 == 0) read_a(slot, mt + 1, 2 * nt + s / 2);
        } else if (nt == 0) {
          if (s < NTW) read_w(next, s);
          else read_a(next, 0, s - NTW);
          if (s == 0) {
            const int blk = min(j / C::kSbStride + 1, nblk - 1);
            dma16_unless(j & (C::kSbStride - 1), sb + 16 * blk, s_off, sb_l + (blk & 1) * 1024);
          }
          if (s == 1) issue(min(j + kBigSlots, nsteps - 1), sl);
        } else {
          if (s < NTW) read_a(next, 0, 2 + s);
          else scn[s - NTW] = read_s(min(j + 1, nsteps - 1), s - NTW);
          b[0][s] = nibbles16_bf16(wd[0][s], nk);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    slast = sc[NTW - 1];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) sc[nt] = scn[nt];
    sl = sn;
  }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) y[MTW - 1][NTW - 1][i] = __builtin_fmaf(slast, acc[(T - 1) & 1][i], y[MTW - 1][NTW - 1][i]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the repeated loads, before the LDS is used again

  // the wave sets' partial sums, in a fixed order
  if (WK > 1) {
    f4* red = reinterpret_cast<f4*>(ring);  // [set - 1][wave of the set][tile][4][64]
    const int w0 = wn * T * 4 * 64 + lane;
    constexpr int kSet = WN * T * 4 * 64;
    __syncthreads();
    if (wk > 0) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f16v& v = y[t / NTW][t % NTW];
          red[(wk - 1) * kSet + w0 + (t * 4 + i) * 64] = f4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        }
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int q = 0; q < WK - 1; ++q)
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f4 r = red[q * kSet + w0 + (t * 4 + i) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[t / NTW][t % NTW][4 * i + e] += r[e];
        }
  }
#pragma unroll
  for (int nt = 0; nt < NTW; ++nt) {
    const int n = nbase + 32 * nt + nn;
    if (n < nseg) {
      uint16_t* yr = yseg + (size_t)layer * p.M * nseg + n;
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int m = 32 * (mb0 + mt) + 8 * (i / 4) + 4 * h + (i & 3);
          if (m < p.M) yr[(size_t)m * nseg] = f2bf(y[mt][nt][i]);
        }
    }
  }
}

template <bool NORM, int W, int NM>
hipError_t launch_j(int J, const QParams& p, dim3 grid, size_t smem, hipStream_t stream) {
  switch (J) {
#define GDN_QL_CASE(j) \
  case j:              \
    hipLaunchKernelGGL((qlinear_kernel<j, NORM, W, NM>), grid, dim3(64 * W), smem, stream, p); break;
    GDN_QL_CASE(2) GDN_QL_CASE(4) GDN_QL_CASE(8) GDN_QL_CASE(10) GDN_QL_CASE(12) GDN_QL_CASE(16)
#undef GDN_QL_CASE
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

bool qlinear_k_supported(int k) {
  return k == 1024 || k == 2048 || k == 4096 || k == 5120 || k == 6144 || k == 8192;
}

bool qlinear_uses_gemv(int m, int k) {
  return m <= GDN_QLINEAR_GEMV_ROWS && (size_t)m * (k / 32) * (4 * 16 + 4) <= 65536;
}

namespace {
// MFMA path: m-tiles of 16 rows per workgroup (1..4), the m-tile count rounded up to a
// multiple of it (the padding rows are zeros in the workspace)
int qgemm_mt(int m) { return std::min(4, (m + 15) / 16); }
int qgemm_mtiles(int m) {
  const int mt = qgemm_mt(m);
  return ((m + 15) / 16 + mt - 1) / mt * mt;
}

template <int MT>
hipError_t launch_gemm_mt(int NT, const QParams& p, dim3 grid, hipStream_t stream) {
  switch (NT) {
    case 1: hipLaunchKernelGGL((qgemm_kernel<MT, 1>), grid, dim3(kThreads), 0, stream, p); break;
    case 2: hipLaunchKernelGGL((qgemm_kernel<MT, 2>), grid, dim3(kThreads), 0, stream, p); break;
    default: hipLaunchKernelGGL((qgemm_kernel<MT, 4>), grid, dim3(kThreads), 0, stream, p); break;
  }
  return hipGetLastError();
}

// The weight rows qgemm_big_kernel takes of an n-row matrix, in whole tiles of `rows`; a last
// partial tile where it is at least 5/8 full.
int big_tiles(int n, int rows) { return n / rows + (n % rows >= rows * 5 / 8 ? 1 : 0); }

// Workgroups of qgemm_big_kernel<WN, WK, MTW> on the busiest CU, or the whole call's (per_cu = 1)
template <int WN, int WK, int MTW>
size_t big_workgroups(const QParams& p, int n_layers, int per_cu) {
  size_t t = 0;
  for (int q = 0; q < p.nseg; ++q) t += big_tiles(p.n[q], BigCfg<WN, WK, MTW>::kRows);
  return (t * n_layers * ((p.mtiles / 2 + MTW - 1) / MTW) + per_cu - 1) / per_cu;
}

// Which form of the product a call of more than 48 rows takes: 0 qgemm_kernel, 1 the 128 x 256
// tiles, 2 the 64 x 128 ones (K split in two). Measured at K = 5120 (and 6/5 of it at 6144), a
// CU with n workgroups takes about 85 n + 8 us with the large tiles and 27.5 n us with the small
// ones; large / small tiles over rotated operands: in_proj M = 333 105 / 101 us, M = 512 114 /
// 124, M = 700 162 / 165, M = 1024 194 / 240; out_proj M = 512 122 / 68, M = 1024 133 / 111,
// M = 1536 141 / 147, M = 2048 200 / 187, M = 4096 346 / 376 (qgemm_kernel at M = 512 and 1024
// 75 and 126). With few small tiles most CUs stand idle and qgemm_kernel's 64 x 64 tiles split
// over more workgroups are faster: out_proj M = 128 (80 tiles) 37 us against 45; from 120 on
// the small tiles are as fast or faster (out_proj M = 160 to 192, 120 tiles: 45 us both; in_proj
// M = 64, 128 tiles: 38 against 45). But where qgemm_kernel's 64 x 32 tiles are exactly two
// workgroups a CU it is faster up to 16 m groups: at N = 4096, M = 256 the 128 small tiles take
// 36.2 us for K = 5120 and 52.7 for K = 8192, qgemm_kernel 28.6 and 40.4; N = 16384, M = 64,
// K = 5120 39.5 and 36.0; N = 1024, M = 1024 39.3 and 33.3; N = 512, M = 2048 42.2 and 47.9.
int big_form(const QParams& p, int n_layers) {
  constexpr int kCUs = 256;
  if (big_workgroups<2, 2, 2>(p, n_layers, 1) < 100) return 0;
  if (p.mtiles / 4 <= 16 && (size_t)n_layers * ((p.R + 31) / 32) * (p.mtiles / 4) == 2 * kCUs) return 0;
  const size_t large = big_workgroups<4, 1, 4>(p, n_layers, kCUs), small = big_workgroups<2, 2, 2>(p, n_layers, kCUs);
  return big_workgroups<4, 1, 4>(p, n_layers, 1) > 0 && 170 * large + 16 <= 55 * small ? 1 : 2;
}

template <int WN, int WK, int MTW>
hipError_t launch_big(QParams p, int n_layers, hipStream_t stream) {
  using C = BigCfg<WN, WK, MTW>;
  int t = 0;
  for (int q = 0; q < p.nseg; ++q) {
    p.row0[q] = t;
    t += big_tiles(p.n[q], C::kRows);
  }
  p.tiles = t;
  p.mgroups = (p.mtiles / 2 + MTW - 1) / MTW;
  const size_t nwg = (size_t)n_layers * p.tiles * p.mgroups;
  p.remap = nwg % 8 == 0;
  QParams r = p;  // the rows past the whole tiles
  r.nseg = 0;
  r.R = 0;
  for (int q = 0; q < p.nseg; ++q) {
    const int done = std::min(p.n[q], big_tiles(p.n[q], C::kRows) * C::kRows);
    if (done == p.n[q]) continue;
    const int i = r.nseg++;
    r.w[i] = p.w[q] + (size_t)done * (p.K / 8);
    r.s[i] = p.s[q] + (size_t)done * (p.K / 64);
    r.b[i] = p.b[q] + (size_t)done * (p.K / 64);
    r.y[i] = p.y[q] + done;
    r.n[i] = p.n[q];
    r.row0[i] = r.R;
    r.R += p.n[q] - done;
  }
  r.layers = n_layers;
  r.tiles = (r.R + 16 * kRestTiles - 1) / (16 * kRestTiles);
  r.mgroups = p.mtiles / 4;
  r.remap = 0;
  const size_t nrest = ((size_t)n_layers * r.tiles * r.mgroups + 7) / 8 * 8;
  const dim3 grid((unsigned)(nrest + nwg));
  if (nrest) hipLaunchKernelGGL((qgemm_big_kernel<WN, WK, MTW, true>), grid, dim3(kThreads), 0, stream, p, r, (int)nrest);
  else hipLaunchKernelGGL((qgemm_big_kernel<WN, WK, MTW, false>), grid, dim3(kThreads), 0, stream, p, r, 0);
  return hipGetLastError();
}
}  // namespace

// The no-allocation entry point's workspace: one array per device, held until the process
// ends. Host code never passes `scratch` itself to a kernel (on the host it names a
// stand-in, not device memory): its device address comes from hipGetSymbolAddress, once per
// device with that device current, and only that address is used.
static __device__ __align__(256) unsigned char scratch[GDN_QLINEAR_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mutex[kMaxScratchDevices];
void* g_scratch_ptr[kMaxScratchDevices];
}  // namespace

// Only a successful lookup is kept: a failure (e.g. before the device's context is usable)
// is returned to this call, and the next call on that device looks the symbol up again.
hipError_t qlinear_scratch(void** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mutex[dev]);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return hipSuccess;
}

// the operand in fragment order (1 KB per 16 rows x 32 values), then its group sums (fp32
// per row and 64 values)
size_t qlinear_xfrag_bytes(int n_layers, int m, int k) {
  const size_t b = (size_t)n_layers * qgemm_mtiles(m) * (k / 32) * 1024;
  return (b + 255) / 256 * 256;
}
size_t qlinear_workspace_bytes(int n_layers, int m, int k) {
  if (qlinear_uses_gemv(m, k)) return 0;
  const size_t xs = (size_t)n_layers * 16 * qgemm_mtiles(m) * (k / 64) * 4;
  return qlinear_xfrag_bytes(n_layers, m, k) + (xs + 255) / 256 * 256;
}

hipError_t launch_qlinear(const gdn_qlinear_args& a, hipStream_t stream) {
  QParams p{};
  p.M = a.m;
  p.K = a.k;
  p.nseg = a.n_segs;
  p.x = static_cast<const uint16_t*>(a.x);
  p.xf = a.norm_x;
  p.z = static_cast<const uint16_t*>(a.norm_z);
  p.gamma = a.norm_gamma;
  p.eps = a.norm_eps;
  int R = 0;
  for (int q = 0; q < GDN_QLINEAR_MAX_SEGS; ++q) {
    const int qq = q < a.n_segs ? q : 0;  // unused slots repeat segment 0 (never selected)
    p.w[q] = static_cast<const uint32_t*>(a.segs[qq].w);
    p.s[q] = static_cast<const uint16_t*>(a.segs[qq].scales);
    p.b[q] = static_cast<const uint16_t*>(a.segs[qq].biases);
    p.y[q] = static_cast<uint16_t*>(a.segs[qq].y);
    p.n[q] = a.segs[qq].n;
    p.row0[q] = R;
    if (q < a.n_segs) R += a.segs[q].n;
  }
  p.R = R;
  const bool norm = a.norm_x != nullptr;
  if (qlinear_uses_gemv(a.m, a.k)) {
    // Waves and passes of 4 rows a wave per workgroup. Calls of few rows take single passes, which
    // put all of their weights in flight at once: in_proj at M = 1 10.7 us in one pass of 4 waves,
    // 15.8 in four; M = 4 21.6 us in one pass of 8 waves, 22.8 of 4 waves (each wave reads the
    // whole operand from LDS), 30 in four passes of 4. Calls of many rows fill the chip anyway and
    // stage the operand less often in taller tiles. At K = 5120: M = 1 one pass of 4 waves up to
    // 7 layers of in_proj (115,360 rows; 51.2 us, in four 57), then two (24 layers 162, in four
    // 166; at K = 8192 four: 140,000 rows 98.4, in two 100.9); M = 2 one pass up to 5 (82,400
    // rows; 47.0, in two 47.5), then two (7 layers 63.8; in one 66.4, in four 64.8), from 131,072
    // rows four (48 layers 376; in two 392); M = 3 and 4 8 waves in one pass up to 5 layers (M = 4
    // 68.9, in two 69.2), then two (7 layers 90.3, in one 92.2), but in one to 131,072 rows where
    // the operand's LDS leaves a CU few workgroups (M = 4, K = 6144, 120,000 rows: 108 against
    // 112). At K = 1024 a pass is short against the staging: from 65,536 rows 4 waves and several
    // passes (69,632 rows: M = 1 10.1 us in four, 11.0 in one; M = 4 15.6 in two, 16.8 in one of 8
    // waves; 248,320 rows: M = 4 45.2 in four, 46.3 in two of 8 waves).
    // With the norm every workgroup normalises the whole operand: the tallest tiles that still make
    // 320 workgroups, where one layer's 5120 rows take single passes (out_proj M = 1 9.0 us
    // against 38 in 8 passes; 48 layers 2.8 us a layer in 8 passes, 3.2 in one).
    const size_t rows = (size_t)a.n_layers * R;
    const bool shortk = a.k == 1024 && rows >= 65536;
    const int W = norm || (a.m > 2 && !shortk) ? 8 : 4;
    if (norm) {
      p.passes = 8;
      while (p.passes > 1 && rows < (size_t)320 * 4 * W * p.passes) p.passes /= 2;
    } else if (W == 8) {
      p.passes = rows < (a.m * a.k > 20480 ? 131072 : 98304) ? 1 : 2;
    } else if (a.m == 1) {
      p.passes = rows < 131072 && !shortk ? 1 : a.k > 1024 && a.k < 8192 ? 2 : 4;
    } else {
      p.passes = rows < 98304 && !shortk ? 1 : rows < 131072 ? 2 : 4;
    }
    p.tiles = (R + 4 * W * p.passes - 1) / (4 * W * p.passes);
    const dim3 grid((unsigned)((size_t)a.n_layers * p.tiles));
    const size_t smem = (size_t)p.M * (a.k / 32) * (4 * 16 + 4);
    const int J = a.k / 512;
    if (norm) return a.m == 1 ? launch_j<true, 8, 1>(J, p, grid, smem, stream) : launch_j<true, 8, 4>(J, p, grid, smem, stream);
    if (W == 8) return launch_j<false, 8, 4>(J, p, grid, smem, stream);
    return a.m == 1 ? launch_j<false, 4, 1>(J, p, grid, smem, stream) : launch_j<false, 4, 4>(J, p, grid, smem, stream);
  }
  // MFMA path: the operand into the workspace, then the product
  const int MT = qgemm_mt(a.m);
  p.mtiles = qgemm_mtiles(a.m);
  p.xfrag = static_cast<uint16_t*>(a.workspace);
  p.xsum = reinterpret_cast<float*>(static_cast<char*>(a.workspace) + qlinear_xfrag_bytes(a.n_layers, a.m, a.k));
  // qgemm_ns_kernel and qgemm_big_kernel load scales and biases 16 bytes a lane, the latter at
  // 32-bit offsets in a matrix
  bool sb16 = true, off32 = true;
  for (int q = 0; q < a.n_segs; ++q) {
    sb16 = sb16 && reinterpret_cast<uintptr_t>(a.segs[q].scales) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(a.segs[q].biases) % 16 == 0;
    off32 = off32 && (size_t)a.segs[q].n * (a.k / 2) <= UINT32_MAX;
  }
  const int big = sb16 && off32 && p.mtiles > 3 ? big_form(p, a.n_layers) : 0;
  p.frag32 = big != 0;
  // One head a thread: with two, the calls of few rows had half the workgroups and each did two
  // norms in sequence (out_proj M = 5 13.9 us against 13.1, M = 333 47.6 against 45.7); from 4096
  // workgroups of two they are enough (out_proj M = 4096 333 us against 336).
  const size_t np = (size_t)a.n_layers * p.mtiles * (a.k / 256);
  if (np < 4096) {
    const dim3 gp((unsigned)(2 * np));
    if (norm) hipLaunchKernelGGL((qprep_kernel<true, 1>), gp, dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL((qprep_kernel<false, 1>), gp, dim3(kThreads), 0, stream, p);
  } else {
    const dim3 gp((unsigned)np);
    if (norm) hipLaunchKernelGGL((qprep_kernel<true, 2>), gp, dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL((qprep_kernel<false, 2>), gp, dim3(kThreads), 0, stream, p);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (big == 1) return launch_big<4, 1, 4>(p, a.n_layers, stream);
  if (big == 2) return launch_big<2, 2, 2>(p, a.n_layers, stream);

  // one m group and enough 256-row workgroups for two per CU: the operand-sharing kernel
  const int ns_tiles = (R + kNsRows - 1) / kNsRows;
  if (p.mtiles == MT && MT <= 3 && sb16 && (size_t)a.n_layers * ns_tiles >= 512) {
    p.tiles = ns_tiles;
    p.mgroups = 1;
    const size_t nwg = (size_t)a.n_layers * ns_tiles;
    p.remap = a.n_layers >= 8 && nwg % 8 == 0;
    const dim3 grid((unsigned)nwg);
    switch (MT) {
      case 1: hipLaunchKernelGGL(qgemm_ns_kernel<1>, grid, dim3(kThreads), 0, stream, p); break;
      case 2: hipLaunchKernelGGL(qgemm_ns_kernel<2>, grid, dim3(kThreads), 0, stream, p); break;
      default: hipLaunchKernelGGL(qgemm_ns_kernel<3>, grid, dim3(kThreads), 0, stream, p); break;
    }
    return hipGetLastError();
  }
  // weight rows per workgroup: 64, 32 or 16 -- the most that still gives 512 workgroups
  const int gy = p.mtiles / MT;
  int NT = 4;
  while (NT > 1 && (size_t)a.n_layers * ((R + 16 * NT - 1) / (16 * NT)) * gy < 512) NT /= 2;
  p.tiles = (R + 16 * NT - 1) / (16 * NT);
  p.mgroups = gy;
  const size_t nwg = (size_t)a.n_layers * p.tiles * gy;
  p.remap = (gy > 1 || a.n_layers >= 8) && nwg % 8 == 0;
  const dim3 grid((unsigned)nwg);
  switch (MT) {
    case 1: return launch_gemm_mt<1>(NT, p, grid, stream);
    case 2: return launch_gemm_mt<2>(NT, p, grid, stream);
    case 3: return launch_gemm_mt<3>(NT, p, grid, stream);
    default: return launch_gemm_mt<4>(NT, p, grid, stream);
  }
}

}  // namespace gdn
