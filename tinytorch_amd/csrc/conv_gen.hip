// Direct convolution over channel chunks (gfx950): forward, input gradient of
// any stride, and weight gradient, for the shapes whose input rows of all
// channels do not fit in LDS at once or that the whole-slab kernels of
// conv.hip run slowly.  Replaces there
//
//   forward  out = W * im2col(x) + bias, NCHW   reference src/ops_spatial.c:71-127
//   dX       col2im(W^T * Gperm)                reference src/autograd.c:515-539,406-434
//   dW, db   Gperm * im2col(x)^T, sum g         reference src/autograd.c:456-513
//
// without an im2col or column-gradient matrix in memory.
//
// One scheme serves all three.  fp32 matrix instructions are slow against
// everything else on the chip (v_mfma_f32_32x32x2_f32: 64 cycles for two
// 32-float operand reads), so single-float LDS reads at computed addresses
// keep the matrix pipe fed, and what has to be kept low is the traffic into
// LDS and the instructions that order it.  A workgroup stages, per chunk of
// the summed index, the rows of the input that its tile touches -- once, not
// once a tap -- and the matching block of the other operand; tiles are small
// (20-30 KB of LDS), so that four or five workgroups share a CU and one
// multiplies while another waits for its loads (two buffers a workgroup, with
// half as many resident, measured 10-40 % slower throughout).  It reads
//
//   A  four consecutive summed indices of a row as one 16-byte read
//      (forward / dX: weights of 32 output channels; dW: the output gradient
//      of 32 filters), rows 4 mod 8 floats apart so that eight lanes cover
//      the 32 banks;
//   B  slab[lane_base + tab[k]]: the lane's own offset (forward / dX: its
//      pixel; dW: its tap) plus the summed index's (its tap; its pixel) from a
//      table in LDS, four at a time.
//
// Lane half h of a wave takes the h-th half of a chunk's summed indices, so
// every table and A read is contiguous and no index is padded but the last
// few of a chunk that is no multiple of 8.
//
// Input rows are staged with their horizontal padding in place (rows of
// exactly the columns the taps can reach, zeros outside the image), a lane a
// column and, for rows below 64 columns, several rows a load; output pixels
// are numbered through (image, row, column), so a tile may span images and
// small images waste nothing.
//
// The input gradient of a stride s is s x s independent stride-1
// convolutions of the output gradient, one for each residue of (h, w) mod s,
// each with the taps that reach it: no product is formed with an inserted
// zero.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include "tt_rt.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

inline hipStream_t stream() { return (hipStream_t)ttrt_stream(); }

constexpr int NT = 256;          // threads a workgroup (4 waves)
constexpr int MAXP = 16;         // row pieces of a slab channel (loads a channel)
constexpr int MAXA = 26;         // 4-byte loads a thread and chunk for A
constexpr int MAXA4 = 13;        // 16-byte ones
constexpr long LDS_MAX = 160L * 1024;

typedef __attribute__((address_space(3))) float lds_float;

// n / d for 0 <= n < 2^24, 0 < d < 2^16, rcp = 1 / d: the estimate is within 1
// of the quotient.
__host__ __device__ inline int fdiv(int n, int d, float rcp) {
  int q = (int)((float)n * rcp);
  const int r = n - q * d;
  q += (r >= d) - (r < 0);
  return q;
}

// v, which the compiler then cannot compare ahead of time: the loads below
// are skipped by scalar compares of constants with it, and kept as masks
// those would fill the scalar registers
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// a value every lane has alike, in a scalar register
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// LDS byte address of p (wave-uniform)
__device__ __forceinline__ unsigned lds_addr(const float *p) {
  return __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_float *)p);
}

// Direct loads: lane l's 4 (16) bytes at base + voff go to LDS at lds + 4 l
// (16 l); base and lds are wave-uniform.  _if: only in the lanes with voff >=
// 0, the others write nothing (a compare and a mask, with no branch and no
// mask kept in registers between calls).
__device__ __forceinline__ void dma4(const float *base, int voff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds), "v"(voff), "s"(base)
               : "memory");
}

__device__ __forceinline__ void dma4_if(const float *base, int voff, unsigned lds) {
  unsigned long long keep;
  asm volatile("s_mov_b32 m0, %1\n\t"
               "v_cmp_le_i32 vcc, 0, %2\n\t"
               "s_and_saveexec_b64 %0, vcc\n\t"
               "global_load_lds_dword %2, %3\n\t"
               "s_mov_b64 exec, %0"
               : "=&s"(keep)
               : "s"(lds), "v"(voff), "s"(base)
               : "memory", "vcc");
}

__device__ __forceinline__ void dma16_if(const float *base, int voff, unsigned lds) {
  unsigned long long keep;
  asm volatile("s_mov_b32 m0, %1\n\t"
               "v_cmp_le_i32 vcc, 0, %2\n\t"
               "s_and_saveexec_b64 %0, vcc\n\t"
               "global_load_lds_dwordx4 %2, %3\n\t"
               "s_mov_b64 exec, %0"
               : "=&s"(keep)
               : "s"(lds), "v"(voff), "s"(base)
               : "memory", "vcc");
}

__device__ __forceinline__ const float *uniform(const float *p) {
  const uintptr_t u = (uintptr_t)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return reinterpret_cast<const float *>(((uintptr_t)hi << 32) | lo);
}

__device__ __forceinline__ void loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// workgroup ids are dealt round robin to the 8 XCDs: neighbouring tiles
// (shared input rows, shared weights) go to one XCD's L2
__device__ __forceinline__ int xcd_order(int pid, int n) {
  const int q = n >> 3, r = n & 7, xcd = pid & 7;
  return xcd * q + min(xcd, r) + (pid >> 3);
}

// A stride-1 view of the taps along one axis: output index o of the tap's
// grid reads input o * is + lo + t, t < n; grid size no, output o at
// o0 + o * os.
struct Axis {
  int n, lo, is, no, o0, os, k0, ks;  // tap t is kernel index k0 + t * ks
};

// forward: every tap; dX: the taps that reach the outputs of residue a
__host__ __device__ inline Axis axis_fwd(int K, int s, int p, int out) {
  return Axis{K, -p, s, out, 0, 1, 0, 1};
}
__host__ __device__ inline Axis axis_dx(int K, int s, int p, int size, int a) {
  // h = a + s o takes g at o + (a + p - k) / s for k = a + p (mod s); the
  // taps in ascending order of that row are k descending
  const int kf = (a + p) % s;
  const int n = kf < K ? (K - 1 - kf) / s + 1 : 0;
  const int kl = kf + (n - 1) * s;
  const int no = a < size ? (size - a + s - 1) / s : 0;
  return Axis{n, n ? (a + p - kl) / s : 0, 1, no, a, s, kl, -s};
}
__device__ inline Axis uniform(const Axis &a) {
  return Axis{uni(a.n), uni(a.lo), a.is, uni(a.no), a.o0, a.os, uni(a.k0), a.ks};
}

// The slab rows of output pixels [p0, p1): pixels are numbered through
// (image, row, column) of an N x no_h x no_w grid.
struct Rows {
  int na, ho, ra, rf, total;  // first image, its first output row, slab rows of
                              // it, of a whole image, in all
};

__device__ __forceinline__ Rows rows_of(const Axis &ah, int now, int p0, int p1) {
  Rows r;
  const int img = ah.no * now;
  r.na = uni(p0 / img);
  r.ho = uni((p0 - r.na * img) / now);
  const int nb = uni((p1 - 1) / img), hb = uni((p1 - 1 - nb * img) / now);
  r.rf = (ah.no - 1) * ah.is + ah.n;
  r.ra = ((nb == r.na ? hb : ah.no - 1) - r.ho) * ah.is + ah.n;
  r.total = nb == r.na ? r.ra : r.ra + (nb - r.na - 1) * r.rf + hb * ah.is + ah.n;
  return r;
}

// slab row of output pixel p, as an offset in floats (rows of rw)
__device__ __forceinline__ int pixel_offset(const Rows &r, const Axis &ah, const Axis &aw, int rw,
                                            int p, int *n, int *ho, int *wo) {
  const int img = ah.no * aw.no;
  *n = p / img;
  const int q = p - *n * img;
  *ho = q / aw.no;
  *wo = q - *ho * aw.no;
  const int row = *n == r.na ? (*ho - r.ho) * ah.is
                             : r.ra + (*n - r.na - 1) * r.rf + *ho * ah.is;
  return row * rw + *wo * aw.is;
}

// Floats between the rows of a slab: a row of up to 64 columns lies against
// the next, a longer one takes whole 64-column pieces.
__host__ __device__ inline int row_stride(int rw) { return rw <= 64 ? rw : (rw + 63) / 64 * 64; }

// A lane's part of the staging of one slab channel: for each piece (a load of
// 64 lanes, `step` floats apart in LDS) the byte offset of its element in
// image na's first channel, -1 outside the image (a zero) or -2 outside the
// slab.
struct Pieces {
  int off[MAXP];
  int n, step;
};

__device__ __forceinline__ void piece_offsets(Pieces &pc, const Rows &r, const Axis &ah,
                                              const Axis &aw, int rw, int C, int H, int W,
                                              int lane) {
  const int rpi = rw <= 64 ? 64 / rw : 1;               // rows a piece
  const int cpr = rw <= 64 ? 1 : (rw + 63) / 64;        // pieces a row
  pc.n = uni(rw <= 64 ? (r.total + rpi - 1) / rpi : r.total * cpr);
  pc.step = uni(rw <= 64 ? rpi * rw : 64);
  const int ls = rw <= 64 ? lane / rw : 0;
  const int lc = lane - ls * rw;
  const float rcp_rf = 1.0f / (float)max(r.rf, 1);
  int row = ls, col = lc, piece = 0;
#pragma unroll
  for (int i = 0; i < MAXP; i++) {
    pc.off[i] = -2;
    if (i >= opaque(pc.n)) continue;
    const bool in = ls < rpi && row < r.total && col < rw;
    int n = 0, hi = r.ho * ah.is + ah.lo + row;
    if (r.total > r.ra && row >= r.ra) {
      const int q = fdiv(row - r.ra, r.rf, rcp_rf);
      n = q + 1;
      hi = ah.lo + (row - r.ra) - q * r.rf;
    }
    const int wi = col + aw.lo;
    const bool ok = (unsigned)hi < (unsigned)H && (unsigned)wi < (unsigned)W;
    pc.off[i] = !in ? -2 : ok ? 4 * (n * C * H * W + hi * W + wi) : -1;
    if (rw <= 64) {
      row += rpi;
    } else if (++piece == cpr) {
      piece = 0;
      row++;
      col = lane;
    } else {
      col += 64;
    }
  }
}

// zeros into n floats (a multiple of 4, 16-byte aligned) of LDS
__device__ __forceinline__ void zero_lds(float *p, int n, int tid) {
  for (int i = 4 * tid; i < n; i += 4 * NT)
    *reinterpret_cast<float4 *>(p + i) = make_float4(0.f, 0.f, 0.f, 0.f);
}

struct ConvG {
  const float *x, *w, *bias;
  float *out, *rout;
  int N, C, H, W;      // the input (dX: the output gradient, C its filters)
  int F, OH, OW;       // the output (dX: the input gradient)
  int HH, WW, sh, sw, ph, pw;
  int ck, cs, lda;     // channels a chunk, floats a slab channel, A's row stride (largest)
  int close;           // quads a wave sums in one chain
  int ftiles;
};

// One step of four summed indices a lane half: A's four (a 16-byte read a
// 32-row block), the table's four offsets, and B's at the lane's offsets off.
template <int MI, int NJ>
__device__ __forceinline__ void read_quad(float (*a)[4], float (*b)[4], const float *al, int astep,
                                          const char *xs, const int *off, const int *tl) {
  const int4 k = *reinterpret_cast<const int4 *>(tl);
#pragma unroll
  for (int i = 0; i < MI; i++) {
    const float4 v = *reinterpret_cast<const float4 *>(al + i * astep);
    a[i][0] = v.x; a[i][1] = v.y; a[i][2] = v.z; a[i][3] = v.w;
  }
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    b[j][0] = *reinterpret_cast<const float *>(xs + (off[j] + k.x));
    b[j][1] = *reinterpret_cast<const float *>(xs + (off[j] + k.y));
    b[j][2] = *reinterpret_cast<const float *>(xs + (off[j] + k.z));
    b[j][3] = *reinterpret_cast<const float *>(xs + (off[j] + k.w));
  }
  __builtin_amdgcn_sched_barrier(0);  // every read of the step ahead of its products
}

template <int MI, int NJ>
__device__ __forceinline__ void mul_quad(float (*a)[4], float (*b)[4], f32x16 (*acc)[NJ]) {
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][s], b[j][s], acc[i][j], 0, 0, 0);
}

template <int MI, int NJ>
__device__ __forceinline__ void clear(f32x16 (&a)[MI][NJ]) {
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int q = 0; q < 16; q++) a[i][j][q] = 0.f;
}

// The products of a few quads are summed by themselves and then added to the
// tile's sums: a chain of all of them rounds as often as it is long.  Relative
// error against 64 bits in one chain, closed as now, and of the GEMM that ran
// these before:
//   forward, a chunk a chain: 32 x 64 x 56 x 56 -> 128 4.3e-7, 1.6e-7, 4.3e-7
//     (145 -> 150 us); 2 x 115 x 10 x 27 -> 28, 5 x 5, stride 2: 4.5e-7,
//     1.5e-7, 1.8e-7
//   dX, 32 x 64 x 56 x 56 -> 128: 6.0e-7, 1.7e-7, 2.1e-7 (167 -> 172 us); few
//     filters, whose GEMM summed few products a tap, close every 32 products:
//     50 x 24 x 45 x 37 -> 40, 5 x 5, stride 2: 2.9e-7, 1.2e-7, 1.3e-7 (31 ->
//     32 us)
//   dW, 32 pixels a chain: 4.8e-7, 1.6e-7, 9.9e-7 and 2.6e-7, 1.4e-7, 3.3e-7
template <int MI, int NJ>
__device__ __forceinline__ void add(f32x16 (&a)[MI][NJ], const f32x16 (&b)[MI][NJ]) {
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int q = 0; q < 16; q++) a[i][j][q] += b[i][j][q];
}

// A wave's outputs of a 32 x P tile of the input gradient (WP pixels from wn * WP
// on; of KW waves with the same pixels, the rows that wave wk stores), a lane an
// element, from memory and the taps in range alone.  The arguments are read and
// the tile found again here: kept for it through conv_gen_kernel's loop, they
// took that loop's scalar registers (21 -> 48 spilled, 6-10 % slower).
template <int P, int WP, int KW>
__device__ __forceinline__ void dx_block_by_taps(int wn, int wk) {
  typedef const __attribute__((address_space(4))) ConvG Args;
  unsigned long long at = (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr();
  int bx = blockIdx.x, bz = blockIdx.z;
  asm volatile("" : "+s"(at), "+s"(bx), "+s"(bz));
  Args &g = *reinterpret_cast<Args *>(at);
  const int a = bz / g.sw, H = g.H, W = g.W, C = g.C, F = g.F, taps = g.HH * g.WW;
  const Axis ah = axis_dx(g.HH, g.sh, g.ph, g.OH, a);
  const Axis aw = axis_dx(g.WW, g.sw, g.pw, g.OW, bz - a * g.sw);
  const int pid = xcd_order(bx, gridDim.x), pt = pid / g.ftiles;
  const int f0 = (pid - pt * g.ftiles) * 32, p0 = pt * P + wn * WP;
  const int img = ah.no * aw.no, px = g.N * img;
#pragma unroll 1
  for (int e = threadIdx.x & 63; e < 32 * WP; e += 64) {
    const int r = e / WP, f = f0 + r, p = p0 + e % WP;
    if (f >= F || p >= px || (KW > 1 && (4 * (r >> 3) + (r & 3)) * KW / 16 != wk)) continue;
    const int n = p / img, ho = (p - n * img) / aw.no, wo = p - n * img - ho * aw.no;
    float v = 0.f;
#pragma unroll 1
    for (int c = 0; c < C; c++) {
      const float *const gi = g.x + ((long)n * C + c) * H * W;
      const float *const wi = g.w + ((long)c * F + f) * taps;
      float s = 0.f;
#pragma unroll 1
      for (int i = 0; i < ah.n; i++)
#pragma unroll 1
        for (int j = 0; j < aw.n; j++) {
          const int hi = ho + ah.lo + i, wj = wo + aw.lo + j;
          if ((unsigned)hi < (unsigned)H && (unsigned)wj < (unsigned)W)
            s += wi[(ah.k0 + i * ah.ks) * g.WW + aw.k0 + j * aw.ks] * gi[hi * W + wj];
        }
      v += s;
    }
    g.out[((long)n * F + f) * g.OH * g.OW + (ah.o0 + ho * ah.os) * g.OW + aw.o0 + wo * aw.os] = v;
  }
}

// Forward (DX false) and input gradient (DX true).  Waves: WN of them tile BF =
// 32 output channels by P = 32 NJ WN pixels, and KW of them share a tile's
// summed indices.  VA: 16-byte loads of the weights.
//
// Bound: the matrix pipe; staging of the next chunk runs under it.
template <int WN, int NJ, int KW, bool DX, bool VA>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
conv_gen_kernel(const ConvG g) {
  static_assert(WN * KW == NT / 64, "four waves");
  constexpr int BF = 32, P = 32 * NJ * WN;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int wk = wave / WN, wn = wave % WN;

  Axis ah, aw;
  if constexpr (DX) {
    const int a = uni(blockIdx.z / g.sw);
    ah = uniform(axis_dx(g.HH, g.sh, g.ph, g.OH, a));
    aw = uniform(axis_dx(g.WW, g.sw, g.pw, g.OW, blockIdx.z - a * g.sw));
  } else {
    ah = axis_fwd(g.HH, g.sh, g.ph, g.OH);
    aw = axis_fwd(g.WW, g.sw, g.pw, g.OW);
  }
  const int T = ah.n * aw.n;
  const int px = g.N * ah.no * aw.no;
  const int pid = xcd_order(blockIdx.x, gridDim.x);
  const int pt = uni(pid / g.ftiles), f0 = (pid - pt * g.ftiles) * BF;
  const int p0 = pt * P, p1 = min(px, p0 + P);
  if (p0 >= px) return;
  const int rw = (aw.no - 1) * aw.is + aw.n, rs = row_stride(rw);
  const Rows r = rows_of(ah, aw.no, p0, p1);

  // ---- LDS: A, slab, tables, bias ----
  const int lda = g.ck * T + 4;
  const int asz = BF * g.lda;
  const int stage_sz = asz + g.ck * g.cs;
  const int tab0 = KW > 1 ? max(stage_sz, NT * 16) : stage_sz;  // KW: the waves' sums
  int *tab = reinterpret_cast<int *>(smem + tab0);
  int *wtab = tab + (g.lda - 4);  // dX: the weights' offsets
  float *bias = reinterpret_cast<float *>(wtab + (DX ? g.lda - 4 : 0));

  const int nchunk = T ? uni((g.C + g.ck - 1) / g.ck) : 0;
  const int taps = g.HH * g.WW;
  const int wf = DX ? taps : g.C * taps, wc = DX ? g.F * taps : taps;
  for (int k = tid; k < g.ck * T; k += NT) {
    const int c = k / T, t = k - c * T, i = t / aw.n, j = t - i * aw.n;
    tab[k] = 4 * (c * g.cs + i * rs + j);
    if constexpr (DX)
      wtab[k] = c * wc + (ah.k0 + i * ah.ks) * g.WW + aw.k0 + j * aw.ks;
  }
  for (int f = tid; f < BF; f += NT) bias[f] = g.bias && f0 + f < g.F ? g.bias[f0 + f] : 0.f;

  // ---- staging ----
  Pieces pc;
  pc.n = 0;
  if (nchunk) piece_offsets(pc, r, ah, aw, rw, g.C, g.H, g.W, lane);
  constexpr int NA = VA ? MAXA4 : MAXA, E = VA ? 4 : 1;
  const int na = uni((BF * lda + NT * E - 1) / (NT * E));
  // byte offset of the thread's weights in a chunk of clim channels, -1: none
  int aoff[NA];
  auto a_offsets = [&](int clim) {
    const int lim = clim * T, df = uni(NT * E / lda), dj = NT * E - df * lda;
    int f = tid * E / lda, j = tid * E - f * lda;
    const int n = opaque(na);
#pragma unroll
    for (int i = 0; i < NA; i++) {
      aoff[i] = -1;
      if (i < n) {
        const int o = DX ? wtab[min(j, lim - 1)] : j;
        if (f < BF && f0 + f < g.F && j < lim) aoff[i] = 4 * (f * wf + o);
        f += df;
        j += dj;
        const bool wrap = j >= lda;
        f += wrap;
        j -= wrap ? lda : 0;
      }
    }
  };
  if (nchunk) {
    if constexpr (DX) __syncthreads();  // wtab
    a_offsets(min(g.ck, g.C));
  }
  const float *const x0 = g.x + (long)r.na * g.C * g.H * g.W;
  const float *const w0 = g.w + (long)f0 * wf;

  const float *const xw = uniform(x0 + (long)wave * g.H * g.W);
  auto stage = [&](int ch) {
    const unsigned as = lds_addr(smem);
    const int cn = min(g.ck, g.C - ch * g.ck);
    const float *const wb = uniform(w0 + (long)ch * g.ck * wc);
    const int n = opaque(na);
#pragma unroll
    for (int i = 0; i < NA; i++) {
      const unsigned dst = as + 4u * (unsigned)((i * NT + wave * 64) * E);
      if (i < n) {
        if constexpr (VA) dma16_if(wb, aoff[i], dst);
        else dma4_if(wb, aoff[i], dst);
      }
    }
    const float *xb = xw + (long)(ch * g.ck) * g.H * g.W;
    unsigned xd = as + 4u * (unsigned)(asz + wave * g.cs);
    for (int c = wave; c < cn; c += NT / 64) {
      unsigned dst = xd;
      const int pn = opaque(pc.n);
#pragma unroll
      for (int i = 0; i < MAXP; i++) {
        if (i < pn) dma4_if(xb, pc.off[i], dst);
        dst += 4u * (unsigned)pc.step;
      }
      xb += (long)(NT / 64) * g.H * g.W;
      xd += 4u * (NT / 64) * (unsigned)g.cs;
    }
  };
  // the last chunk's missing channels: zeros in both operands (LDS may hold an
  // earlier chunk's, and a zero must not meet an infinity)
  auto blank = [&]() {
    float *const as = smem;
    const int cn = g.C % g.ck, kn = cn * T, miss = g.ck * T - kn;
    for (int q = tid; q < BF * miss; q += NT) {
      const int f = q / miss;
      as[f * lda + kn + (q - f * miss)] = 0.f;
    }
    for (int q = cn * g.cs + tid; q < g.ck * g.cs; q += NT) as[asz + q] = 0.f;
  };

  int pix[NJ], opix[NJ];  // the lane's pixels: slab offset (bytes), output offset
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int p = p0 + (wn * NJ + j) * 32 + l32;
    int n, ho, wo;
    pix[j] = 4 * pixel_offset(r, ah, aw, rs, min(p, p1 - 1), &n, &ho, &wo);
    opix[j] = p < p1 ? n * g.F * g.OH * g.OW + (ah.o0 + ho * ah.os) * g.OW + aw.o0 + wo * aw.os
                     : -1;
  }

  f32x16 acc[1][NJ];
  clear(acc);

  auto multiply = [&](int ch) {
    const float *const as = smem;
    const char *const xs = reinterpret_cast<const char *>(as + asz);
    const int kh = (min(g.ck, g.C - ch * g.ck) * T + 7) / 8 * 4;  // indices a lane half
    const float *const al = as + l32 * lda + h * kh;
    const int *const tl = tab + h * kh;
    for (int q = 4 * wk; q < kh;) {
      const int end = min(kh, q + 4 * KW * g.close);
      f32x16 part[1][NJ];
      clear(part);
      for (; q < end; q += 4 * KW) {
        float a[1][4], bb[NJ][4];
        read_quad<1, NJ>(a, bb, al + q, 0, xs, pix, tl + q);
        mul_quad<1, NJ>(a, bb, part);
      }
      add(acc, part);
    }
  };

  const bool ragged = nchunk && g.C % g.ck;
  if (nchunk) {
    // the padding, which no load writes (dX: the missing channels' weights too,
    // whose sums are looked at below)
    const int z0 = DX && f0 + BF > g.F ? 0 : asz;
    zero_lds(smem + z0, asz - z0 + g.ck * g.cs, tid);
    __syncthreads();
  }
  for (int ch = 0; ch < nchunk; ch++) {
    if (ch) __syncthreads();  // every wave is done with the last chunk
    if (ragged && ch + 1 == nchunk) {
      if (ch) a_offsets(g.C % g.ck);
      blank();
    }
    stage(ch);
    loads_done();
    __syncthreads();
    multiply(ch);
  }

  // ---- the KW waves' sums of a tile, added in wave order ----
  if constexpr (KW > 1) {
    static_assert(NJ == 1, "one 32 x 32 block a wave");
    __syncthreads();
    float *const red = smem + wave * 1024;
#pragma unroll
    for (int q = 0; q < 16; q++) red[q * 64 + lane] = acc[0][0][q];
    __syncthreads();
    // wave wk stores rows q = wk * 16 / KW .. of the sum
#pragma unroll
    for (int q = 0; q < 16; q++) {
      float v = smem[wn * 1024 + q * 64 + lane];
#pragma unroll
      for (int k = 1; k < KW; k++) v += smem[(k * WN + wn) * 1024 + q * 64 + lane];
      acc[0][0][q] = v;
    }
  } else {
    if (!nchunk) __syncthreads();  // the bias
  }

  // dX adds only the taps that reach an output; the slab's zeros stand for the
  // others, and times an infinite or NaN weight they are not zero.  Such a weight
  // leaves no sum of its output channel finite: a wave with a sum that is not
  // forms its outputs again tap by tap.
  if constexpr (DX) {
    float z = 0.f;
#pragma unroll
    for (int q = 0; q < 16; q++)
#pragma unroll
      for (int j = 0; j < NJ; j++) z = __builtin_fmaf(acc[0][j][q], 0.f, z);
    if (__ballot(z != 0.f)) {  // NaN
      dx_block_by_taps<P, 32 * NJ, KW>(wn, wk);
      return;
    }
  }

  // ---- bias, relu, store: row 8 (q / 4) + 4 h + q % 4 of a block ----
  const int ohw = g.OH * g.OW;
#pragma unroll
  for (int q = 0; q < 16; q++) {
    if (KW > 1 && (q * KW) / 16 != wk) continue;
    const int fl = 8 * (q >> 2) + 4 * h + (q & 3);
    if (f0 + fl >= g.F) continue;
    const float bv = bias[fl];
    const long fo = (long)(f0 + fl) * ohw;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      if (opix[j] < 0) continue;
      const float v = acc[0][j][q] + bv;
      g.out[fo + opix[j]] = v;
      if (g.rout) g.rout[fo + opix[j]] = v > 0.f ? v : 0.f;
    }
  }
}

struct ConvGW {
  const float *g, *x;
  float *dw, *db;      // or the partials: row stride ld, the bias column at db
  int N, C, H, W, F, OH, OW, HH, WW, sh, sw, ph, pw;
  int cs, nch;         // floats a slab channel, channels staged (at most)
  int ftiles, ctiles;
  int per;             // pixels a split (a multiple of PC)
  long ld, dbs, zs;    // floats between rows of dw, elements of db, splits
};

constexpr int PC = 64;       // pixels a chunk of the weight gradient

// The chunk's output gradient in LDS: a row of PC floats a filter, its 16-byte
// blocks permuted (block b of filter f at b ^ (f & 15)) so that the reads of
// one block of 16 filters cover the banks.
__device__ __forceinline__ int g_block(int f, int b) { return f * PC + 4 * (b ^ (f & 15)); }

// Weight gradient: a workgroup forms BF filters x BN columns (channel, tap)
// over a range of output pixels, in chunks of PC; the splits' sums go to
// partials that conv_gen_dw_reduce adds in order.  db is summed on the VALU
// from the same A operands by the waves of the first column tile.
// VG: 16-byte loads of the output gradient (whole images of a multiple of 4
// pixels), else a load a pixel.
template <int WM, int WN, int MI, int NJ, bool VG>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
conv_gen_dw_kernel(const ConvGW g) {
  static_assert(WM * WN == NT / 64, "four waves");
  constexpr int BF = 32 * MI * WM, BN = 32 * NJ * WN;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;

  const Axis ah = axis_fwd(g.HH, g.sh, g.ph, g.OH), aw = axis_fwd(g.WW, g.sw, g.pw, g.OW);
  const int T = ah.n * aw.n, K = g.C * T;
  const int img = g.OH * g.OW;
  const int px = g.N * img;
  // splits outermost in the order of an XCD: its tiles share x and g
  const int pid = xcd_order(blockIdx.x, gridDim.x);
  const int tiles = g.ftiles * g.ctiles;
  const int z = uni(pid / tiles), tile = pid - z * tiles;
  const int ct = uni(tile / g.ftiles), f0 = (tile - ct * g.ftiles) * BF;
  const int col0 = ct * BN;
  const int c0 = uni(col0 / T), cn = uni(min(g.C - 1, (col0 + BN - 1) / T)) - c0 + 1;
  const int pbeg = z * g.per, pend = min(px, pbeg + g.per);
  const int nchunk = (pend - pbeg + PC - 1) / PC;
  const int rw = (aw.no - 1) * aw.is + aw.n, rs = row_stride(rw);

  constexpr int asz = BF * PC;
  const int slab_sz = (g.nch * g.cs + 3) / 4 * 4;  // then the pixel table
  auto stage = [&](int ch) {
    float *const xs = smem + asz;
    const unsigned as = lds_addr(smem);
    const int p0 = pbeg + ch * PC, p1 = min(pend, p0 + PC);
    const Rows r = rows_of(ah, aw.no, p0, p1);
    // the output gradient: a load a filter, a lane a pixel
    const int p = p0 + lane;
    int n, ho, wo;
    const int po = 4 * pixel_offset(r, ah, aw, rs, min(p, p1 - 1), &n, &ho, &wo);
    if (wave == 0) reinterpret_cast<int *>(xs + slab_sz)[lane] = po;
    // (past the range: pixel p1 - 1 again, against zeros)
    const float *const gb0 = g.g + ((long)r.na * g.F + f0) * img;
    if constexpr (VG) {
      // four filters a load, 16 lanes each: lane l takes the block that
      // position l % 16 of its filter's row holds
      const int fl = lane >> 4, f = wave * 4 + fl;  // f & 15 is the same in every load
      const int pb = min(p0 + 4 * ((lane & 15) ^ f), p1 - 4);
      const int nb = pb / img;
      const int go = 4 * (((nb - r.na) * g.F + fl) * img + pb - nb * img);
      const float *gb = uniform(gb0 + (long)(wave * 4) * img);
      unsigned gd = as + 4u * (unsigned)(wave * 4 * PC);
      const int fn = g.F - f0 - fl;
#pragma unroll
      for (int q = 0; q < BF / 16; q++) {
        dma16_if(gb, q * 16 + wave * 4 < fn ? go : -1, gd);
        gb += 16L * img;
        gd += 4u * 16 * PC;
      }
    } else {
      const float *gb = uniform(gb0 + (long)wave * img);
      const int fn = min(BF, g.F - f0);
      unsigned gd = as + 4u * (unsigned)(wave * PC);
      const int go = 4 * ((n - r.na) * g.F * img + ho * aw.no + wo);
      int pb[4];  // the load of filter f takes the pixel that lane l's place holds
#pragma unroll
      for (int k = 0; k < 4; k++) pb[k] = __shfl(go, (((lane >> 2) ^ (wave + 4 * k)) << 2) | (lane & 3));
      for (int f = wave, k = 0; f < fn; f += NT / 64, k++) {
        const int o = (k & 2) ? ((k & 1) ? pb[3] : pb[2]) : ((k & 1) ? pb[1] : pb[0]);
        dma4(gb, o, gd);
        gb += (long)(NT / 64) * img;
        gd += 4u * (NT / 64) * PC;
      }
    }
    Pieces pc;
    piece_offsets(pc, r, ah, aw, rw, g.C, g.H, g.W, lane);
    const float *xb = uniform(g.x + ((long)r.na * g.C + c0 + wave) * g.H * g.W);
    unsigned xd = as + 4u * (unsigned)(asz + wave * g.cs);
    for (int c = wave; c < cn; c += NT / 64) {
      unsigned dst = xd;
      const int pn = opaque(pc.n);
#pragma unroll
      for (int i = 0; i < MAXP; i++) {
        if (i < pn) dma4_if(xb, pc.off[i], dst);
        dst += 4u * (unsigned)pc.step;
      }
      xb += (long)(NT / 64) * g.H * g.W;
      xd += 4u * (NT / 64) * (unsigned)g.cs;
    }
    // rows outside the image: zeros (the buffer may hold an earlier chunk's)
    const int hl = r.ho * ah.is + ah.lo;
    if (r.total > r.ra || hl < 0 || hl + r.total > g.H) {
#pragma unroll
      for (int i = 0; i < MAXP; i++) {
        if (pc.off[i] == -1)
          for (int c = wave; c < cn; c += NT / 64) xs[c * g.cs + i * pc.step + lane] = 0.f;
      }
    }
  };

  int ko[NJ];  // the lane's columns: byte offset of their tap in the slab
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int col = min(col0 + (wn * NJ + j) * 32 + l32, K - 1);
    const int c = col / T, t = col - c * T, i = t / aw.n;
    ko[j] = 4 * ((c - c0) * g.cs + i * rs + (t - i * aw.n));
  }

  f32x16 acc[MI][NJ];
  clear(acc);
  float sum[MI];
#pragma unroll
  for (int i = 0; i < MI; i++) sum[i] = 0.f;
  const bool want_db = g.db && ct == 0 && wn == 0;

  auto multiply = [&](int ch) {
    const char *const xs = reinterpret_cast<const char *>(smem + asz);
    const int *const tab = reinterpret_cast<const int *>(smem + asz + slab_sz);
    const int np = min(pend - (pbeg + ch * PC), PC);
    const int kh = (np + 7) / 8 * 4;
    const float *const al = smem + (wm * MI * 32 + l32) * PC;
    const int *const tl = tab + h * kh;
    auto quad = [&](int q, bool edge, f32x16 (&acc)[MI][NJ]) {
      float a[MI][4], bb[NJ][4];
      read_quad<MI, NJ>(a, bb, al + 4 * (((h * kh + q) >> 2) ^ (l32 & 15)), 32 * PC, xs, ko, tl + q);
      if (edge) {  // pixels past the range: zeros in both operands
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const bool in = h * kh + q + s < np;
#pragma unroll
          for (int i = 0; i < MI; i++) a[i][s] = in ? a[i][s] : 0.f;
#pragma unroll
          for (int j = 0; j < NJ; j++) bb[j][s] = in ? bb[j][s] : 0.f;
        }
      }
      if (want_db) {
#pragma unroll
        for (int i = 0; i < MI; i++) sum[i] += (a[i][0] + a[i][1]) + (a[i][2] + a[i][3]);
      }
      mul_quad<MI, NJ>(a, bb, acc);
    };
    if (np == PC) {
      for (int q0 = 0; q0 < PC / 2; q0 += PC / 4) {
        f32x16 part[MI][NJ];
        clear(part);
        for (int q = q0; q < q0 + PC / 4; q += 4) quad(q, false, part);
        add(acc, part);
      }
    } else {
      for (int q = 0; q < kh; q += 4) quad(q, true, acc);
    }
  };

  zero_lds(smem + asz, slab_sz, tid);  // the padding columns, which no load writes
  __syncthreads();
  for (int ch = 0; ch < nchunk; ch++) {
    if (ch) __syncthreads();
    stage(ch);
    loads_done();
    __syncthreads();
    multiply(ch);
  }

  float *const dw = g.dw + z * g.zs;
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int f = f0 + (wm * MI + i) * 32 + 8 * (q >> 2) + 4 * h + (q & 3);
      if (f >= g.F) continue;
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const int col = col0 + (wn * NJ + j) * 32 + l32;
        if (col < K) dw[f * g.ld + col] = acc[i][j][q];
      }
    }
  if (want_db) {
#pragma unroll
    for (int i = 0; i < MI; i++) {
      const float v = sum[i] + __shfl_xor(sum[i], 32);
      const int f = f0 + (wm * MI + i) * 32 + l32;
      if (h == 0 && f < g.F) (g.db + z * g.zs)[f * g.dbs] = v;
    }
  }
}

// dw, db = the sum of Z partials of F rows of K + 1 (the last column db's) in
// a fixed order: 64 outputs a workgroup, the splits dealt to its four waves,
// four chains each.
__global__ void __launch_bounds__(NT) conv_gen_dw_reduce(const float *__restrict__ part, float *dw,
                                                         float *db, int Z, int F, int K) {
  __shared__ float s[NT];
  const long n = (long)F * (K + 1);
  const long o = (long)blockIdx.x * 64 + (threadIdx.x & 63);
  const int w = threadIdx.x >> 6, per = (Z + 3) / 4;
  float v = 0.f;
  if (o < n) {
    const int z1 = min(Z, (w + 1) * per);
    int z = w * per;
    float a = 0.f, b = 0.f, c = 0.f, d = 0.f;
    for (; z + 4 <= z1; z += 4) {
      a += part[z * n + o];
      b += part[(z + 1) * n + o];
      c += part[(z + 2) * n + o];
      d += part[(z + 3) * n + o];
    }
    v = (a + b) + (c + d);
    for (; z < z1; z++) v += part[z * n + o];
  }
  s[threadIdx.x] = v;
  __syncthreads();
  if (w || o >= n) return;
  v = ((s[threadIdx.x] + s[threadIdx.x + 64]) + s[threadIdx.x + 128]) + s[threadIdx.x + 192];
  const int f = (int)(o / (K + 1)), k = (int)(o - (long)f * (K + 1));
  if (k < K) dw[(long)f * K + k] = v;
  else if (db) db[f] = v;
}

// ---------------------------------------------------------------- host

bool big_lds(const void *fn) {
  static const void *done[64];
  static int ndone = 0;
  for (int i = 0; i < ndone; i++)
    if (done[i] == fn) return true;
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_MAX) !=
      hipSuccess)
    return false;
  if (ndone < 64) done[ndone++] = fn;
  return true;
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Most slab rows, and row pieces, that P consecutive pixels touch.
struct SlabMax {
  long rows, pieces, cs, imgs;
};
SlabMax slab_max(const Axis &ah, const Axis &aw, int N, int P) {
  SlabMax m{0, 0, 0, 0};
  if (!ah.n || !aw.n || ah.no <= 0 || aw.no <= 0) return m;
  const long img = (long)ah.no * aw.no;
  const long px = img * N;
  const long L = P < px ? P : px;
  long rows = (L + aw.no - 2) / aw.no + 1;          // output rows touched
  if (rows > (long)N * ah.no) rows = (long)N * ah.no;
  long ni = (L - 2 + img) / img + 1;                // images touched
  if (ni > N) ni = N;
  if (ni > rows) ni = rows;
  // a run of q output rows of one image spans (q - 1) is + n slab rows
  m.rows = rows * ah.is + ni * (ah.n > ah.is ? ah.n - ah.is : 0);
  const long rw = (long)(aw.no - 1) * aw.is + aw.n;
  m.pieces = rw <= 64 ? (m.rows + 64 / rw - 1) / (64 / rw) : m.rows * ((rw + 63) / 64);
  // one float a channel more than a multiple of 8: taps of neighbouring
  // channels fall on different banks
  m.cs = (m.rows * row_stride((int)rw) + 7) / 8 * 8 + 1;
  m.imgs = ni;
  return m;
}

// ---- plans ----
struct Tile {
  int p, kw;  // pixels a tile (of 32 output channels), waves sharing its summed indices
};
constexpr int NTILE = 4;
constexpr Tile TILES[NTILE] = {{256, 1}, {128, 1}, {64, 2}, {32, 4}};
constexpr int CUS = 256;

struct GenPlan {
  int tile = -1, ck = 0;
  long lds = 0, cs = 0, lda = 0, ptiles = 0, ftiles = 0;
};

int g_force_tile = -1, g_force_ck = 0;  // ttk_conv_gen_force

// The largest tile that leaves the CUs enough workgroups, and the most
// channels a chunk whose LDS leaves room for as many of them a CU as the grid
// has, up to five.  Measured (us): 128-pixel tiles from about 400 of them
// (128 x 32 x 16 x 16 -> 64: 512 tiles, 19.9 against 21 with 64 pixels; 93 x
// 32 x 19 x 19 -> 32: 263 tiles, 18.9 against 17.5), 256 only for taps beyond
// 3 x 3, whose slab halo is the larger part (404 x 16 x 16 x 16 -> 32, 5 x 5:
// 36.4 against 38.8; 3 x 3 no difference).  Tiles of 64 output channels were
// no faster where the channels fill them.
GenPlan plan_gen(const ConvG &g, bool dx, bool va) {
  const int ncls = dx ? g.sh * g.sw : 1;
  const long ftiles = (g.F + 31) / 32;
  GenPlan best;
  for (int t = 0; t < NTILE; t++) {
    if (g_force_tile >= 0 && t != g_force_tile) continue;
    const Tile &tl = TILES[t];
    long tmax = 0, cs = 0, pieces = 0, imgs = 0, ptiles = 0;
    for (int a = 0; a < (dx ? g.sh : 1); a++)
      for (int b = 0; b < (dx ? g.sw : 1); b++) {
        const Axis ah = dx ? axis_dx(g.HH, g.sh, g.ph, g.OH, a) : axis_fwd(g.HH, g.sh, g.ph, g.OH);
        const Axis aw = dx ? axis_dx(g.WW, g.sw, g.pw, g.OW, b) : axis_fwd(g.WW, g.sw, g.pw, g.OW);
        const SlabMax m = slab_max(ah, aw, g.N, tl.p);
        const long T = (long)ah.n * aw.n;
        const long pt = ((long)g.N * ah.no * aw.no + tl.p - 1) / tl.p;
        if (T > tmax) tmax = T;
        if (m.cs > cs) cs = m.cs;
        if (m.pieces > pieces) pieces = m.pieces;
        if (m.imgs > imgs) imgs = m.imgs;
        if (pt > ptiles) ptiles = pt;
      }
    if (pieces > MAXP || imgs * g.C * g.H * g.W * 4 >= 0x7fffffffL) continue;
    const long tiles = ptiles * ftiles * ncls;
    long per_cu = (tiles + CUS - 1) / CUS;
    if (per_cu > 5) per_cu = 5;
    GenPlan p;
    for (int ck = 8; ck <= 64; ck *= 2) {
      if (g_force_ck && ck != g_force_ck) continue;
      if (ck > 8 && ck >= 2 * ((g.C + 7) / 8 * 8)) continue;
      const long lda = ck * tmax + 4;
      const long e = va ? 4 : 1, na = (32 * lda + NT * e - 1) / (NT * e);
      if (na > (va ? MAXA4 : MAXA)) continue;
      long fl = 32 * lda + ck * cs;
      if (tl.kw > 1 && fl < NT * 16) fl = NT * 16;
      const long lds = 4 * (fl + (dx ? 2 : 1) * ck * tmax + 32);
      if (lds > LDS_MAX || (p.tile >= 0 && (lds * per_cu > LDS_MAX || ck * tmax > 160))) continue;
      p.tile = t;
      p.ck = ck;
      p.lds = lds;
      p.cs = cs;
      p.lda = lda;
      p.ptiles = ptiles;
      p.ftiles = ftiles;
    }
    if (p.tile < 0) continue;
    best = p;
    if (g_force_tile >= 0) break;
    if (t == 0 ? tmax > 9 && tiles >= 384 : t == 1 ? tiles >= 400 : tiles >= CUS) break;
  }
  return best;
}

template <int WN, int NJ, int KW, bool DX>
int launch_gen(const ConvG &g, const GenPlan &p, bool va) {
  auto kern = va && !DX ? conv_gen_kernel<WN, NJ, KW, DX, !DX>
                        : conv_gen_kernel<WN, NJ, KW, DX, false>;
  if (p.lds > 64 * 1024 && !big_lds((const void *)kern)) return -1;
  const dim3 grid((unsigned)(p.ftiles * p.ptiles), 1, DX ? (unsigned)(g.sh * g.sw) : 1u);
  hipLaunchKernelGGL(kern, grid, dim3(NT), (size_t)p.lds, stream(), g);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

struct DwPlan {
  int tile = -1, nch = 0, per = 0, splits = 0;
  long lds = 0, cs = 0, ftiles = 0, ctiles = 0;
};
TTPlanCache<GenPlan> g_gen_plans;  // tag: dX, 16-byte weights, the forced plans
TTPlanCache<DwPlan> g_dw_plans;
int g_force_tag = 0;

template <bool DX>
const GenPlan &gen_plan(const ConvG &g, const int q[13], bool va) {
  return g_gen_plans.get(q, 4 * g_force_tag + 2 * DX + va, [&] { return plan_gen(g, DX, va); });
}

template <bool DX>
int run_gen(ConvG g, const int q[13], bool dry) {
  const bool va = !DX && (g.C * g.HH * g.WW) % 4 == 0 && (dry || aligned16(g.w));
  const GenPlan &p = gen_plan<DX>(g, q, va);
  if (p.tile < 0 || p.ftiles * p.ptiles >= 0x7fffffffL) return -1;
  if (dry) return 0;
  if (ttk_fail_direct_conv()) return -3;
  g.ck = p.ck;
  g.close = !DX ? p.ck * g.HH * g.WW : g.C > 96 ? 10 : 4;
  g.cs = (int)p.cs;
  g.lda = (int)p.lda;
  g.ftiles = (int)p.ftiles;
  switch (p.tile) {
    case 0: return launch_gen<4, 2, 1, DX>(g, p, va);
    case 1: return launch_gen<4, 1, 1, DX>(g, p, va);
    case 2: return launch_gen<2, 1, 2, DX>(g, p, va);
    default: return launch_gen<1, 1, 4, DX>(g, p, va);
  }
}

// what every kernel here indexes in 32 bits
bool geo_ok(const int q[13]) {
  const long N = q[0], C = q[1], H = q[2], W = q[3], F = q[4], HH = q[5], WW = q[6], Ho = q[11],
             Wo = q[12];
  if (N <= 0 || C <= 0 || H <= 0 || W <= 0 || F <= 0 || HH <= 0 || WW <= 0 || q[7] <= 0 ||
      q[8] <= 0 || q[9] < 0 || q[10] < 0 || Ho <= 0 || Wo <= 0)
    return false;
  const long lim = 0x7fffffffL;
  return H < 32768 && W < 32768 && q[7] <= 16 && q[8] <= 16 && N * C * H * W < lim &&
         N * F * Ho * Wo < lim && F * C * HH * WW * 4 < lim;
}

struct DwTile {
  int bf, bn;
};
constexpr int NDW = 3;
constexpr DwTile DWTILES[NDW] = {{32, 128}, {64, 64}, {128, 64}};

int g_force_dw = -1, g_force_splits = 0;

// The tile whose filters fit F (128 of them only where the pixels still give
// every CU several workgroups of several chunks: 32 x 64 x 56 x 56 -> 128,
// 183 us against 204 with 64), and splits for about five workgroups a CU
// (41 x 41 x 64 x 63 -> 26, stride 2: 768 workgroups 35 us, 384 38; 93 x 32 x
// 19 x 19 -> 32: 525 32 us, 384 36).
DwPlan plan_dw(const ConvGW &g) {
  DwPlan p;
  const Axis ah = axis_fwd(g.HH, g.sh, g.ph, g.OH), aw = axis_fwd(g.WW, g.sw, g.pw, g.OW);
  const long T = (long)g.HH * g.WW, K = T * g.C, px = (long)g.N * g.OH * g.OW;
  const SlabMax m = slab_max(ah, aw, g.N, PC);
  if (m.pieces > MAXP || m.imgs * g.C * g.H * g.W * 4 >= 0x7fffffffL ||
      (m.imgs * g.F + 16) * g.OH * g.OW * 4 >= 0x7fffffffL)
    return p;
  const long work = (px + PC - 1) / PC * ((g.F + 127) / 128) * ((K + 63) / 64);
  for (int t = g.F <= 32 ? 0 : g.F <= 64 || work < 8 * CUS ? 1 : 2; t >= 0; t--) {
    if (g_force_dw >= 0 && t != g_force_dw) continue;
    const DwTile &tl = DWTILES[t];
    const long ftiles = (g.F + tl.bf - 1) / tl.bf, ctiles = (K + tl.bn - 1) / tl.bn;
    long nch = (tl.bn + T - 2) / T + 1;
    if (nch > g.C) nch = g.C;
    const long lds = 4 * (tl.bf * PC + (nch * m.cs + 3) / 4 * 4 + PC);
    if (lds > LDS_MAX) continue;
    const long tiles = ftiles * ctiles, chunks = (px + PC - 1) / PC;
    long s = (5 * CUS + tiles - 1) / tiles;
    if (s > chunks) s = chunks;
    if (g_force_splits) s = g_force_splits < chunks ? g_force_splits : chunks;
    const long per = (chunks + s - 1) / s;
    p.tile = t;
    p.nch = (int)nch;
    p.per = (int)(per * PC);
    p.splits = (int)((chunks + per - 1) / per);
    p.lds = lds;
    p.cs = m.cs;
    p.ftiles = ftiles;
    p.ctiles = ctiles;
    return p;
  }
  return p;
}

template <int WM, int WN, int MI, int NJ>
int launch_dw(const ConvGW &g, const DwPlan &p) {
  const bool vg = (g.OH * g.OW) % 4 == 0 && aligned16(g.g);
  auto kern = vg ? conv_gen_dw_kernel<WM, WN, MI, NJ, true> : conv_gen_dw_kernel<WM, WN, MI, NJ, false>;
  if (p.lds > 64 * 1024 && !big_lds((const void *)kern)) return -1;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.ftiles * p.ctiles * p.splits)), dim3(NT),
                     (size_t)p.lds, stream(), g);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

ConvG gen_args(const int q[13], bool dx) {
  ConvG g{};
  g.N = q[0];
  g.C = dx ? q[4] : q[1];
  g.H = dx ? q[11] : q[2];
  g.W = dx ? q[12] : q[3];
  g.F = dx ? q[1] : q[4];
  g.OH = dx ? q[2] : q[11];
  g.OW = dx ? q[3] : q[12];
  g.HH = q[5]; g.WW = q[6];
  g.sh = q[7]; g.sw = q[8];
  g.ph = q[9]; g.pw = q[10];
  return g;
}

ConvGW dw_args(const int q[13]) {
  ConvGW g{};
  g.N = q[0]; g.C = q[1]; g.H = q[2]; g.W = q[3]; g.F = q[4]; g.HH = q[5]; g.WW = q[6];
  g.sh = q[7]; g.sw = q[8]; g.ph = q[9]; g.pw = q[10]; g.OH = q[11]; g.OW = q[12];
  return g;
}

template <bool DX>
double gen_us(const int q[13]) {
  const ConvG g = gen_args(q, DX);
  const GenPlan &p = gen_plan<DX>(g, q, !DX && (g.C * g.HH * g.WW) % 4 == 0);
  const Tile &tl = TILES[p.tile];
  const int ncls = DX ? g.sh * g.sw : 1;
  const double taps = (double)g.HH * g.WW;
  const double tmax = DX ? ((g.HH + g.sh - 1) / g.sh) * (double)((g.WW + g.sw - 1) / g.sw) : taps;
  const double per = tt_per_cu((double)p.ftiles * p.ptiles * ncls);
  const double nch = (g.C + p.ck - 1) / p.ck;
  const double quads = g.C * taps / ncls / 8 / tl.kw * (tl.p == 256 ? 2 : 1);
  const double stage = p.ck * (32 * tmax + p.cs);
  const double resident = DX ? 2.9 : 1.7;
  return (DX ? 7.8 : 6.5) + nch * (DX ? 1.44 : 0.99) * (per > resident ? per / resident : 1) +
         per * (quads * (DX ? 0.116 : 0.104) + nch * stage * (DX ? 7.7e-5 : 9.6e-5));
}

}  // namespace

// Estimated microseconds of the kernel (what: 0 forward, 1 weight gradient, 2
// input gradient) of a shape that it covers: a launch, the busiest CU's chunks
// one after another -- a round trip each where few workgroups hide it -- its
// MFMAs and staged floats, and the splits' partials.  Fitted to 960 shapes (1-64
// images, 1-128 channels, 7-64 a side, 4-256 filters, 1x1 to 5x5, stride 1 and
// 2, up to 40 GFLOP): the ratio to the measured time has a standard deviation of
// 0.16, 0.17 and 0.15.
extern "C" double ttk_conv_gen_us(const int q[13], int what) {
  if (what != 1) return what == 2 ? gen_us<true>(q) : gen_us<false>(q);
  const ConvGW g = dw_args(q);
  const DwPlan &p = g_dw_plans.get(q, g_force_tag, [&] { return plan_dw(g); });
  const double per = tt_per_cu((double)p.ftiles * p.ctiles * p.splits);
  const double gr = DWTILES[p.tile].bf * PC * (g.OH * g.OW % 4 ? 4 : 1);  // 4- or 16-byte loads
  const double part = 4e-6 * g.F * ((double)g.C * g.HH * g.WW + 1) * p.splits;  // MB
  return 5.5 + per * (p.per / PC) *
                   (0.41 + (p.tile == 2 ? 2.04 : 1.02) + 1.26e-4 * p.nch * p.cs + 1.6e-5 * gr) +
         (p.splits > 1 ? 4.8 + 0.49 * part : 0);
}

extern "C" void ttk_conv_gen_force(int tile, int ck, int dw, int splits) {
  g_force_tile = tile;
  g_force_ck = ck;
  g_force_tag++;  // no plan of the cache is for these
  g_force_dw = dw;
  g_force_splits = splits;
}

extern "C" int ttk_conv_gen_fwd(const float *x, const float *w, const float *bias, float *out,
                                float *rout, const int q[13]) {
  if (!geo_ok(q)) return -1;
  ConvG g = gen_args(q, false);
  g.x = x; g.w = w; g.bias = bias; g.out = out; g.rout = rout;
  return run_gen<false>(g, q, !out);
}

extern "C" int ttk_conv_gen_dx(const float *gr, const float *w, float *dx, const int q[13]) {
  if (!geo_ok(q)) return -1;
  ConvG g = gen_args(q, true);
  g.x = gr; g.w = w; g.out = dx;
  return run_gen<true>(g, q, !dx);
}

extern "C" int ttk_conv_gen_dw(const float *gr, const float *x, float *dw, float *db,
                               const int q[13]) {
  if (!geo_ok(q)) return -1;
  ConvGW g = dw_args(q);
  g.g = gr; g.x = x;
  const DwPlan &p = g_dw_plans.get(q, g_force_tag, [&] { return plan_dw(g); });
  if (p.tile < 0 || p.ftiles * p.ctiles * p.splits >= 0x7fffffffL) return -1;
  const int K = g.C * g.HH * g.WW;
  const long n = (long)g.F * (K + 1);
  if (n * p.splits >= 0x7fffffffL * 4) return -1;
  if (!dw) return 0;
  float *part = nullptr;
  if (p.splits > 1) {
    part = (float *)ttrt_alloc(sizeof(float) * (size_t)(n * p.splits));
    if (!part) return -2;
    g.dw = part;
    g.db = part + K;
    g.ld = g.dbs = K + 1;
    g.zs = n;
  } else {
    g.dw = dw;
    g.db = db;
    g.ld = K;
    g.dbs = 1;
    g.zs = 0;
  }
  g.nch = p.nch;
  g.cs = (int)p.cs;
  g.per = p.per;
  g.ftiles = (int)p.ftiles;
  g.ctiles = (int)p.ctiles;
  int rc;
  switch (p.tile) {
    case 0: rc = launch_dw<1, 4, 1, 1>(g, p); break;
    case 1: rc = launch_dw<2, 2, 1, 1>(g, p); break;
    default: rc = launch_dw<2, 2, 2, 1>(g, p); break;
  }
  if (rc == 0 && part) {
    hipLaunchKernelGGL(conv_gen_dw_reduce, dim3((unsigned)((n + 63) / 64)), dim3(NT), 0, stream(),
                       part, dw, db, p.splits, g.F, K);
    if (hipGetLastError() != hipSuccess) rc = -3;
  }
  ttrt_free(part);  // stream-ordered
  return rc;
}
