// Dense-circulant variant of the periodic operators on the matrix cores.
//
// With periodic boundaries every operator of src/x3d_operator_1d.f90 is a
// circulant matrix C = A^-1 B (A the tridiagonal left-hand side, B the
// stencil); column j of C is column 0 shifted by j, so C[i][j] = c[(i-j) mod n]
// with c = A^-1 (B e_0).  Applying it to all lines of a direction is a GEMM
// with K = n:
//   y/z lines:  OUT[i][col] = sum_k C[i][k] IN[k][col]   (IN viewed as n x N)
//   x lines:    OUT[l][i]   = sum_k IN[l][k] C[i][k]     (IN viewed as L x n)
// computed with v_mfma_f32_32x32x16_f16 in three split-precision terms,
// x = x_hi + x_lo (fp16 each, together ~22 bits):
//   C_hi IN_hi + C_hi IN_lo + C_lo IN_hi, accumulated in FP32.
// fp16 keeps three more bits per half than bf16 but has a narrow exponent
// range, so C is scaled by a power of two on the host and each work-group
// scales its input block by the power of two that brings its largest value
// just under 2^14 (exact scalings, undone on the FP32 result).
// Inputs and outputs are FP32 fields of the precision form.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "x3d_line.h"

namespace x3d {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// hi/lo fp16 halves of eight FP32 values
__device__ __forceinline__ void split8(const float (&x)[8], f16x8& hi, f16x8& lo)
{
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const _Float16 h = (_Float16)x[v];
    hi[v] = h;
    lo[v] = (_Float16)(x[v] - (float)h);
  }
}

// One fragment of C for the 32x32x16 operand layout (lane l: row l % 32,
// k = 8 (l / 32) + v): hi and lo halves of 8 values, for one block offset
// row0 - k0, a multiple of 16 (mod n).
struct CircFrag {
  f16x8 hi, lo;
};

// The block offsets 16 p whose fragments are not all zero: p = lo .. lo + count
// - 1, circularly.  The entries of C fall off like beta^|i - j|, and an entry
// 2^-35 below the largest is zero in both fp16 halves, so of the n / 16
// offsets a staggered derivative keeps 4, the first derivative 6 and an
// interpolation 18 (all of them for short lines).
struct CircBand {
  int lo, count;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 ld4(const float* base, unsigned boff, unsigned uniform = 0)
{
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(field_rsrc(base), boff, uniform, 0));
}

// The fp16 halves of x, hi in the low 16 bits.
__device__ __forceinline__ unsigned split_word(float x)
{
  const _Float16 h = (_Float16)x;
  const _Float16 l = (_Float16)(x - (float)h);
  return (unsigned)__builtin_bit_cast(unsigned short, h) | ((unsigned)__builtin_bit_cast(unsigned short, l) << 16);
}

// y/z: OUT = C IN, IN rows k at stride rs, columns [32 bx, 32 bx + 32) of slab
// by (slab stride ss); x: OUT = IN C^T, IN lines [32 bx, 32 bx + 32) of n
// contiguous points.  A tile is one such block of 32 lines, tile = by nbx +
// bx; n = 128 NB.  Work-groups are persistent, each of NW wavefronts owns RB
// blocks of 32 output points of every tile and walks the 16-point input blocks
// that its rows' band reaches; a fragment of C outside the band is skipped.
// What bounds it is HBM, 8 B per point, for the derivatives (4-6 offsets), and
// the LDS reads of the fragments, 18 offsets of 2 KB per row block, for the
// interpolations.  512^3, ms per operator, walking all 32 offsets with one
// 4-wavefront work-group per compute unit -> this: x derivatives 0.79 -> 0.19
// (5.6 TB/s), y/z 0.84 -> 0.24, interpolations 0.79-0.84 -> 0.30-0.35.
// (Fragments carried in registers from one row block to the next: 2% faster,
// but spills at 1024 points.  Neighbouring tiles grouped per XCD: no change.)
// STAGE (where 32 rows of n + 4 words and the band's fragments fit the LDS):
// the tile is read once, by 16-byte loads (x: the 32 lines are one contiguous
// run; y/z: 32-column rows of 128 B), into registers while the tile before it
// is multiplied; it is scaled and split once, when it is copied to LDS, and
// the MFMA operands come from there.  Otherwise it is read from memory twice,
// once for the block maximum and once per MFMA step, and split there.
// A tile that holds an infinity or a NaN walks all offsets, with zero
// fragments outside the band, so that 0 * Inf and 0 * NaN reach the whole
// line as in the dense product.
template <int NB, int NW, bool XDIR, bool STAGE>
__global__ __launch_bounds__(64 * NW) void k_circ_mfma(const float* __restrict__ in, float* __restrict__ out,
                                                       const CircFrag* __restrict__ tab, CircBand band, int ntiles,
                                                       int nbx, unsigned rs, unsigned ss, float inv_cscale)
{
  constexpr int n = 128 * NB, NT = 64 * NW, RB = n / (32 * NW), N16 = n / 16;
  static_assert(RB >= 1 && RB * 32 * NW == n, "whole row blocks per wavefront");
  constexpr int Q = 8 * n / NT;  // 16-byte loads of a tile per thread
  __shared__ float wmax[NW];
  __shared__ unsigned wbits[NW];
  // the operator's fragments (64 lanes x 32 B per offset) are read by every
  // wavefront at every step: copied once per work-group to LDS
  extern __shared__ unsigned char smem_raw[];
  CircFrag* ltab = reinterpret_cast<CircFrag*>(smem_raw);
  unsigned* blk = reinterpret_cast<unsigned*>(smem_raw + (size_t)band.count * 64 * sizeof(CircFrag));
  constexpr int P = n + 4;  // block row pitch in words (16-byte multiple)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lc = lane & 31, lk8 = 8 * (lane >> 5), lk = 4 * (lane >> 5);
  // byte offsets (FP32 fields are below 4 GiB): 32-bit ones of buffer
  // instructions, which leave the registers to two work-groups per compute unit
  auto first = [&](int tile) {  // the tile's first point
    if constexpr (XDIR) return (unsigned)tile * (32u * n * 4u);
    else return (unsigned)(tile / nbx) * (ss * 4u) + (unsigned)(tile % nbx) * 128u;
  };
  f32x4 x[STAGE ? Q : 1];
  auto fetch = [&](int tile) {
    if constexpr (STAGE) {
      // load u is point row (or run) u * NT / 8 further on: a uniform step
      const unsigned q = threadIdx.x;
      const unsigned off = first(tile) + (XDIR ? 16u * q : (q >> 3) * (rs * 4u) + 16u * (q & 7u));
#pragma unroll
      for (int u = 0; u < Q; ++u)
        x[u] = ld4(in, off, u * (XDIR ? NT * 16u : (NT / 8) * rs * 4u));
    }
  };
  int tile = blockIdx.x;
  if (tile < ntiles) fetch(tile);
  for (int q = threadIdx.x; q < band.count * 64; q += NT) ltab[q] = tab[q];
  // this wavefront's rows are the 16-blocks R0 .. R0 + 2 RB - 1; row block
  // R0 + 2 r takes input block k16 through offset p = R0 + 2 r - k16, entry
  // t = p - lo of the table (mod N16)
  const int R0 = __builtin_amdgcn_readfirstlane(wave) * RB * 2;
  const int reach = 2 * (RB - 1) + band.count;
  for (; tile < ntiles; tile += gridDim.x) {
    const unsigned t0 = first(tile);
    const unsigned base = XDIR ? t0 + (unsigned)lc * (n * 4u) : t0 + (unsigned)lc * 4u;  // this lane's line
    const unsigned ps = XDIR ? 4u : rs * 4u;                                             // between its points
    // the block's largest magnitude, and the largest bit pattern of one (which
    // an infinity or a NaN lifts to 0x7F800000 or more)
    float m = 0.f;
    unsigned mb = 0u;
    auto see = [&](float v) {
      m = fmaxf(m, fabsf(v));
      mb = max(mb, __float_as_uint(v) & 0x7FFFFFFFu);
    };
    if constexpr (STAGE) {
#pragma unroll
      for (int u = 0; u < Q; ++u) {
        see(x[u].x);
        see(x[u].y);
        see(x[u].z);
        see(x[u].w);
      }
    } else {
      if constexpr (XDIR) {
        // the 32 lines are one contiguous run
        for (unsigned q = threadIdx.x; q < 8 * n; q += NT) {
          const f32x4 y = ld4(in, t0 + 16u * q);
          see(y.x);
          see(y.y);
          see(y.z);
          see(y.w);
        }
      } else {
        // thread (lc, g) scans points g, g + NT / 32, ...
        for (int k = threadIdx.x >> 5; k < n; k += NT / 32) see(ld(in, base + (unsigned)k * ps));
      }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      m = fmaxf(m, __shfl_xor(m, d));
      mb = max(mb, (unsigned)__shfl_xor((int)mb, d));
    }
    if (lane == 0) {
      wmax[wave] = m;
      wbits[wave] = mb;
    }
    // (also: every wavefront is done with the previous tile's block)
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      m = fmaxf(m, wmax[w]);
      mb = max(mb, wbits[w]);
    }
    int e = 0;
    if (m > 0.f) (void)frexpf(m, &e);  // m = f 2^e, f in [0.5, 1)
    const float scale = ldexpf(1.f, 14 - e), unscale = ldexpf(inv_cscale, e - 14);
    if constexpr (STAGE) {
#pragma unroll
      for (int u = 0; u < Q; ++u) {
        const int q = threadIdx.x + NT * u;
        const unsigned w0 = split_word(x[u].x * scale), w1 = split_word(x[u].y * scale);
        const unsigned w2 = split_word(x[u].z * scale), w3 = split_word(x[u].w * scale);
        if constexpr (XDIR) {
          const int l = (4 * q) / n, k = 4 * q - l * n;
          *reinterpret_cast<u32x4*>(blk + l * P + k) = u32x4{w0, w1, w2, w3};
        } else {
          const int k = q >> 3, c4 = 4 * (q & 7);
          blk[(c4 + 0) * P + k] = w0;
          blk[(c4 + 1) * P + k] = w1;
          blk[(c4 + 2) * P + k] = w2;
          blk[(c4 + 3) * P + k] = w3;
        }
      }
    }
    // (the block and, the first time, the fragments)
    __syncthreads();
    if (tile + (int)gridDim.x < ntiles) fetch(tile + gridDim.x);
    f32x16 acc[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[r][v] = 0.f;
    const bool all = __builtin_amdgcn_readfirstlane((int)(mb >= 0x7F800000u)) != 0;
    // input block of step s: ascending from the lowest that the first row
    // block reaches
    auto block = [&](int s) {
      const int k16 = R0 - (band.lo + band.count - 1) + s;
      return 16 * (k16 < 0 ? k16 + N16 : (k16 >= N16 ? k16 - N16 : k16));
    };
    auto operand = [&](int k0, f16x8& fh, f16x8& fl) {
      if constexpr (STAGE) {
        const u32x4* row = reinterpret_cast<const u32x4*>(blk + lc * P + k0 + lk8);
        const u32x4 a = row[0], b = row[1];
        // low and high halves of word pairs
        const u32x4 h{__builtin_amdgcn_perm(a.y, a.x, 0x05040100u), __builtin_amdgcn_perm(a.w, a.z, 0x05040100u),
                      __builtin_amdgcn_perm(b.y, b.x, 0x05040100u), __builtin_amdgcn_perm(b.w, b.z, 0x05040100u)};
        const u32x4 l{__builtin_amdgcn_perm(a.y, a.x, 0x07060302u), __builtin_amdgcn_perm(a.w, a.z, 0x07060302u),
                      __builtin_amdgcn_perm(b.y, b.x, 0x07060302u), __builtin_amdgcn_perm(b.w, b.z, 0x07060302u)};
        fh = __builtin_bit_cast(f16x8, h);
        fl = __builtin_bit_cast(f16x8, l);
      } else {
        float y[8];
        if constexpr (XDIR) {
          const f32x4 a = ld4(in, base + (unsigned)(k0 + lk8) * 4u), b = ld4(in, base + (unsigned)(k0 + lk8) * 4u + 16u);
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            y[v] = a[v] * scale;
            y[v + 4] = b[v] * scale;
          }
        } else {
#pragma unroll
          for (int v = 0; v < 8; ++v) y[v] = ld(in, base + (unsigned)(k0 + lk8 + v) * ps) * scale;
        }
        split8(y, fh, fl);
      }
    };
    auto multiply = [&](f32x16& d, const f16x8& fh, const f16x8& fl, const CircFrag& cf) {
      if constexpr (XDIR) {
        // D[line][i] = sum_k IN[line][k] C^T[k][i]
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(fh, cf.hi, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(fl, cf.hi, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(fh, cf.lo, d, 0, 0, 0);
      } else {
        // D[i][col] = sum_k C[i][k] IN[k][col]
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(cf.hi, fh, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(cf.hi, fl, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(cf.lo, fh, d, 0, 0, 0);
      }
    };
    const int steps = all || reach > N16 ? N16 : reach;
    for (int s = 0; s < steps; ++s) {
      f16x8 fh, fl;
      operand(block(s), fh, fl);
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        int t = 2 * r + band.count - 1 - s;
        t = t < 0 ? t + N16 : (t >= N16 ? t - N16 : t);
        CircFrag cf;
        if (t < band.count) {
          cf = ltab[t * 64 + lane];
        } else {
          if (!all) continue;
#pragma unroll
          for (int v = 0; v < 8; ++v) cf.hi[v] = cf.lo[v] = (_Float16)0.f;
        }
        multiply(acc[r], fh, fl, cf);
      }
    }
    // D layout: column lc; row 8 (v / 4) + 4 (lane / 32) + v % 4
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int b0 = 16 * (R0 + 2 * r);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = 8 * (v >> 2) + lk + (v & 3);
        // x: row = line within the block, column = output point b0 + lc (the
        // uniform part of each offset in a scalar register)
        const unsigned off = XDIR ? t0 + (unsigned)(lk * n + lc) * 4u : base + (unsigned)lk * ps;
        const unsigned at = XDIR ? (unsigned)((row - lk) * n + b0) * 4u : (unsigned)(b0 + row - lk) * ps;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, acc[r][v] * unscale), field_rsrc(out), off,
                                              (int)at, 0);
      }
    }
  }
}

// ---- host ----------------------------------------------------------------------
// First column of C = A^-1 B: the stencil applied to the periodic delta at 0,
// then the reference's periodic Thomas sweeps and Sherman-Morrison correction
// with the operator's own tables (src/thomas.f90:34-84).
static std::vector<double> circ_column(const x3d_ctx* c, int op, int dir, int kind)
{
  const OpHost& o = c->op[op];
  const int n = o.n;
  const Coef<double> k = stencil_coef(c->sc[dir], kind);
  auto e = [n](int i) { i %= n; if (i < 0) i += n; return i == 0 ? 1.0 : 0.0; };
  std::vector<double> t(n);
  for (int i = 0; i < n; ++i) {
    switch (kind) {
      case K_D: t[i] = k.a * (e(i + 1) - e(i - 1)) + k.b * (e(i + 2) - e(i - 2)); break;
      case K_DVP: t[i] = k.a * (e(i + 1) - e(i)) + k.b * (e(i + 2) - e(i - 1)); break;
      case K_DPV: t[i] = k.a * (e(i) - e(i - 1)) + k.b * (e(i + 1) - e(i - 2)); break;
      case K_IVP:
        t[i] = k.a * (e(i + 1) + e(i)) + k.b * (e(i + 2) + e(i - 1)) + k.c * (e(i + 3) + e(i - 2)) +
               k.d * (e(i + 4) + e(i - 3));
        break;
      default:
        t[i] = k.a * (e(i) + e(i - 1)) + k.b * (e(i + 1) + e(i - 2)) + k.c * (e(i + 2) + e(i - 3)) +
               k.d * (e(i + 3) + e(i - 4));
        break;
    }
  }
  for (int i = 1; i < n; ++i) t[i] = t[i] - t[i - 1] * o.s[i];
  t[n - 1] = t[n - 1] * o.w[n - 1];
  for (int i = n - 2; i >= 0; --i) t[i] = (t[i] - o.f[i] * t[i + 1]) * o.w[i];
  const double ss = (t[0] - o.alfa * t[n - 1]) / (1.0 + o.p[0] - o.alfa * o.p[n - 1]);
  for (int i = 0; i < n; ++i) t[i] = t[i] - ss * o.p[i];
  return t;
}

}  // namespace x3d

using namespace x3d;

extern "C" int x3d_apply_circ_mfma(x3d_ctx* c, int op, float* out, const float* in)
{
  if (!c || op < 0 || op >= X3D_NOPS || !out || !in || out == in) return X3D_ERR_ARG;
  if (!c->op[op].circulant) return X3D_ERR_UNSUPPORTED;
  const int dir = op < 6 ? op / 2 : (op - 6) % 3;
  static const int kinds[4] = {K_DVP, K_DPV, K_IVP, K_IPV};
  const int kind = op < 6 ? K_D : kinds[(op - 6) / 3];
  if (stretch_which(c, dir, kind) >= 0) return X3D_ERR_UNSUPPORTED;  // stretched y-derivatives: the line solvers
  const int n = dir == 0 ? c->nx : dir == 1 ? c->ny : c->nz;
  // the kernel's tiles: 4 wavefronts x RB blocks of 32 along the line, and
  // 32 columns (y/z) or 32 lines (x) per work-group
  const int cols = dir == 0 ? c->ny * c->nz : dir == 1 ? c->nx : c->nx * c->ny;
  if (n % 128 || n > 1024 || cols % 32) return X3D_ERR_UNSUPPORTED;
  if (!c->circ_tab[op]) {
    const std::vector<double> col = circ_column(c, op, dir, kind);
    // scale C by the power of two that brings its largest entry under 2^10
    double cmax = 0.0;
    for (double v : col) cmax = std::fmax(cmax, std::fabs(v));
    int ce = 0;
    if (cmax > 0.0) (void)std::frexp(cmax, &ce);
    const double cs = std::ldexp(1.0, 10 - ce);
    c->circ_scale[op] = (float)std::ldexp(1.0, ce - 10);
    std::vector<CircFrag> h((size_t)(n / 16) * 64);
    const int n16 = n / 16;
    int first = 0, last = 0;  // offsets in use, -n16 / 2 .. n16 / 2 - 1
    for (int p = -n16 / 2; p < n16 - n16 / 2; ++p) {
      const int d = 16 * p;
      bool used = false;
      for (int l = 0; l < 64; ++l) {
        CircFrag f;
        for (int v = 0; v < 8; ++v) {
          int idx = (d + (l & 31) - 8 * (l >> 5) - v) % n;
          if (idx < 0) idx += n;
          const double x = col[idx] * cs;
          const _Float16 hi = (_Float16)x;
          f.hi[v] = hi;
          f.lo[v] = (_Float16)(x - (double)hi);
          used = used || f.hi[v] != (_Float16)0.f || f.lo[v] != (_Float16)0.f;
        }
        h[(size_t)(p + n16 / 2) * 64 + l] = f;
      }
      if (used && p < first) first = p;
      if (used && p > last) last = p;
    }
    // the device table holds the offsets first .. last
    const CircFrag* from = h.data() + (size_t)(first + n16 / 2) * 64;
    const size_t bytes = (size_t)(last - first + 1) * 64 * sizeof(CircFrag);
    void* p = nullptr;
    X3D_CHECK_HIP(hipMalloc(&p, bytes));
    const hipError_t e = hipMemcpy(p, from, bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      (void)hipFree(p);
      return hip_status(e);
    }
    c->circ_tab[op] = p;
    c->circ_lo[op] = first;
    c->circ_count[op] = last - first + 1;
  }
  const CircFrag* tab = static_cast<const CircFrag*>(c->circ_tab[op]);
  const CircBand band{c->circ_lo[op], c->circ_count[op]};
  const long long nxy = (long long)c->nx * c->ny;
  const int ntiles = cols / 32 * (dir == 1 ? c->nz : 1);
  const int nbx = cols / 32;
  const unsigned rs = (unsigned)(dir == 1 ? c->nx : nxy), ss = (unsigned)nxy;
  const float inv = c->circ_scale[op];  // undoes the host scaling of C
  const size_t tsmem = (size_t)band.count * 64 * sizeof(CircFrag);
  const size_t bsmem = (size_t)32 * (n + 4) * sizeof(float);
  // the input block too where both fit (and the wavefronts' maxima, 64 B)
  const bool stage = tsmem + bsmem <= 160 * 1024 - 256;
  const size_t smem = tsmem + (stage ? bsmem : 0);
  // a wavefront per 64 output points (32 up to 384); as many persistent
  // work-groups as the LDS and 16 wavefronts per compute unit allow.  (384 by 6
  // wavefronts of 64 points, which the four SIMDs do not share evenly, against
  // 12 of 32: interpolation of 384 x 192 x 80 48 -> 18 us, derivative 23 -> 12)
  int& ncu = c->ncu;
  if (ncu <= 0) X3D_CHECK_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
  const int nw = n <= 384 ? n / 32 : n / 64;
  const int per_cu = (int)std::max<size_t>(1, std::min<size_t>(16 / nw, (160 * 1024) / (smem + 256)));
  const dim3 grid((unsigned)std::min(ntiles, ncu * per_cu));
#define X3D_MFMA_RUN(NB, NW, XD, ST)                                                                             \
  do {                                                                                                           \
    if (smem > 65536)                                                                                            \
      X3D_CHECK_HIP(hipFuncSetAttribute((const void*)k_circ_mfma<NB, NW, XD, ST>,                                \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));                 \
    hipLaunchKernelGGL((k_circ_mfma<NB, NW, XD, ST>), grid, dim3(64 * NW), smem, c->stream, in, out, tab, band, ntiles, \
                       nbx, rs, ss, inv);                                                                                   \
  } while (0)
#define X3D_NB(NB)                                              \
  case NB: {                                                    \
    constexpr int NW = NB <= 3 ? 4 * NB : 2 * NB;               \
    if (stage) {                                                \
      if (dir == 0) X3D_MFMA_RUN(NB, NW, true, true);           \
      else X3D_MFMA_RUN(NB, NW, false, true);                   \
    } else {                                                    \
      if (dir == 0) X3D_MFMA_RUN(NB, NW, true, false);          \
      else X3D_MFMA_RUN(NB, NW, false, false);                  \
    }                                                           \
  } break;
  switch (n / 128) {  // (the line lengths of a grid: 640 and 896 are not among them)
    X3D_NB(1) X3D_NB(2) X3D_NB(3) X3D_NB(4) X3D_NB(6) X3D_NB(8)
    default: return X3D_ERR_UNSUPPORTED;
  }
#undef X3D_NB
#undef X3D_MFMA_RUN
  X3D_CHECK_HIP(hipGetLastError());
  return X3D_OK;
}
