// Split-precision grouped GEMM for gfx950: FP64 operands emulated with
// integer slices on the INT8 matrix cores (Ozaki-style error-free splitting).
//
// 1. slice_once_kernel (real data, K up to 2048) or slice_max_kernel and
//    slice_kernel, once per operand: for every row r of every block (rows =
//    the GEMM's M modes for A, N modes for B; the K modes are the columns),
//    E_r = the smallest integer with max_k |x_rk| < 2^E_r, and
//        x_rk = 2^E_r / 127 * sum_{i=0..S-1} v_i,rk * 254^(-i) + residue,
//    v_i in [-127, 127] (int8), |residue| <= 2^E_r / 127 * 254^(1-S) / 2:
//    y = 127 * (x / 2^E) (|y| < 127; one rounding, 2^-53 relative), then
//    v = rint(y), y = (y - v) * 254 (|y| <= 127), S times. With S = 6 the
//    residue is 3.7e-15 of the row maximum (the 7-bit digits of a power-of-two
//    radix would need 7 digits, 28 products, for the same order).
//    The operand is read in place through its mode strides (no permutation
//    pass). Each slice plane holds K padded to a multiple of 32 (zeros) in
//    16-byte chunks, chunk-major: chunk c of row r at byte (c*R + r)*16, so
//    that 64 consecutive rows of one chunk are one contiguous 1 KB run for
//    both the writer and the GEMM's loads.
// 2. split_gemm_kernel: C = sum_{pairs} alpha_p * A_p B_p, where for every
//    pair the products v^A_i v^B_j with i + j <= S - 1 (21 of them) run on
//    v_mfma_i32_32x32x32_i8, summed per level L = i + j in INT32 -- exact,
//    since |sum| <= S * 127^2 * K < 2^31 for K <= 2 * kSplitKChunk (the
//    planner cuts longer pairs into K chunks) -- and recombined in FP64
//    after the pair's K loop:
//        C_mn += alpha * 2^(EA_m+EB_n) / 127^2 * sum_L 254^(-L) S_L,mn.
//    The error is that of the two representations plus the dropped levels
//    L >= S (same order), about 1e-13 relative Frobenius for N(0,1) data;
//    no rounding occurs in the products or the INT32 sums.
//    Complex data have two slice sets per operand (re, im) under one exponent
//    per row; a kernel of its own forms both components of C in one pass.
// Tiles: 64 x 64 per workgroup of four waves, 32 x 32 per wave64; K steps of 32
// (two chunks) in a ring of LDS stages.
// Stages are fetched with global_load_lds_dwordx4 (HBM/L2 -> LDS without
// registers): one wave instruction moves the 64 rows of one (plane, chunk),
// issued a full K step ahead of the MFMAs that consume it. In LDS a stage is
// [plane][chunk][row] x 16 bytes, so a lane's MFMA operand (row l%32, chunk
// l/32) is read with consecutive lanes on consecutive 16-byte slots (no bank
// conflicts). The MFMA is issued as D = B^T A^T so that each lane's
// accumulators run down a column of C (contiguous column-major stores).
#include <utility>

#include "itg_internal.h"

namespace itg {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;
constexpr int kXcds = 8;
constexpr double kInvRadix = 1.0 / kSliceRadix;               // rounded: 2^-53 relative
constexpr double kInvLead2 = 1.0 / (kSliceLead * kSliceLead);  // rounded: 2^-53 relative
constexpr int kNonFinite = 0x7fff;   // row exponent of a row holding Inf / NaN
constexpr int kZeroRow = -0x40000000;  // partial exponent of an all-zero K range
static_assert(kSliceRows == 64 && kSliceKPart % 64 == 0, "slice tiling");

__device__ inline int64_t mode_offset(uint32_t idx, int n, const int32_t* dim,
                                      const int32_t* str) {
  int64_t o = 0;
#pragma unroll
  for (int i = 0; i < kSliceModes; ++i) {
    if (i >= n) break;
    if (i + 1 < n) {
      const uint32_t q = idx / (uint32_t)dim[i];
      o += (int64_t)(idx - q * (uint32_t)dim[i]) * str[i];
      idx = q;
    } else {
      o += (int64_t)idx * str[i];
    }
  }
  return o;
}

// Magnitude used for the row scale: |x| (real) or max(|re|, |im|) (complex,
// whose two parts share one scale per row so that their slice products land
// on the same INT32 grid).
template <int CPLX>
__device__ inline double elem_mag(const double* x, int64_t o) {
  if (CPLX) {
    const double2 v = reinterpret_cast<const double2*>(x)[o];
    const double m = fmax(fabs(v.x), fabs(v.y));
    return (isfinite(v.x) && isfinite(v.y)) ? m : INFINITY;
  }
  const double v = x[o];
  return isfinite(v) ? fabs(v) : INFINITY;
}

// Exponent recorded for a magnitude m: kNonFinite for Inf (elem_mag maps
// NaN to Inf), kZeroRow for 0, else e with m = f 2^e, f in [0.5, 1), so
// m < 2^e. Monotonic in m, so the exponent of a maximum is the maximum of
// the exponents.
__device__ inline int mag_exponent(double m) {
  int e = kZeroRow;
  if (!isfinite(m))
    e = kNonFinite;
  else if (m > 0.0)
    (void)frexp(m, &e);
  return e;
}

// Offset of K multi-index k (K mode 0 fastest), advanced one element at a
// time without divisions.
struct KWalk {
  int64_t off;
  int32_t c[kSliceModes];
  __device__ void init(uint32_t k, const SliceBlock& d) {
    off = 0;
#pragma unroll
    for (int i = 0; i < kSliceModes; ++i) {
      c[i] = 0;
      if (i >= d.nkm) continue;
      if (i + 1 < d.nkm) {
        const uint32_t q = k / (uint32_t)d.kdim[i];
        c[i] = (int32_t)(k - q * (uint32_t)d.kdim[i]);
        k = q;
      } else {
        c[i] = (int32_t)k;
      }
      off += (int64_t)c[i] * d.kstr[i];
    }
  }
  __device__ void step(const SliceBlock& d) {
    off += d.kstr[0];
    if (++c[0] == d.kdim[0]) {
      c[0] = 0;
      off -= (int64_t)d.kdim[0] * d.kstr[0];
#pragma unroll
      for (int i = 1; i < kSliceModes; ++i) {
        if (i >= d.nkm) break;
        off += d.kstr[i];
        if (++c[i] < d.kdim[i]) break;
        c[i] = 0;
        off -= (int64_t)d.kdim[i] * d.kstr[i];
      }
    }
  }
};

// Workgroup -> (block, 64-row tile rt, K part kp) of the slicing grid.
struct SliceTile {
  int64_t b;
  int r0, kp;
};
__device__ inline SliceTile slice_tile(const SliceBlock* blocks, const int2* wgmap, int64_t wg) {
  SliceTile t;
  const int2 m = wgmap[wg];
  t.b = m.x;
  const int kparts = blocks[t.b].kparts;
  t.kp = m.y % kparts;
  t.r0 = (m.y / kparts) * kSliceRows;
  return t;
}

// srow[i] = element offset of row min(r0 + i, R - 1) of block d (threads
// 0..kSliceRows-1 write; the caller synchronises).
__device__ inline void load_row_offsets(const SliceBlock& d, int r0, int tid, int64_t* srow) {
  if (tid < kSliceRows)
    srow[tid] = mode_offset((uint32_t)min(r0 + tid, d.R - 1), d.nrm, d.rdim, d.rstr);
}

// Pass 1: for each row of a (64 rows) x (kSliceKPart) tile, the exponent of
// the largest magnitude in the tile's K range (kZeroRow if all are zero,
// kNonFinite if any is Inf/NaN), stored as partial kp of the row. The source
// is contiguous either along the rows (operand stored rows-fastest) or along
// K; threads run along the contiguous direction so that loads coalesce.
template <int CPLX>
__global__ void __launch_bounds__(kThreads)
    slice_max_kernel(const SliceBlock* __restrict__ blocks, const int2* __restrict__ wgmap,
                     SliceOperands ops) {
  __shared__ int ered[4][kSliceRows];  // partial exponents: [thread part][row]
  __shared__ int64_t srow[kSliceRows];
  const SliceTile t = slice_tile(blocks, wgmap, blockIdx.x);
  const SliceBlock& d = blocks[t.b];
  const int tid = threadIdx.x;
  const double* x = ops.src[d.side] + (CPLX ? 2 : 1) * d.off;
  int32_t* pmax = ops.pmax[d.side];
  const int k_lo = t.kp * kSliceKPart, k_hi = min(d.K, k_lo + kSliceKPart);
  const bool kfast = d.nkm == 1 && d.kstr[0] == 1;
  // Every load below is unconditional, from an offset clamped into the block
  // (rows past R onto row R-1, K past the range onto its first element), and
  // the value is dropped afterwards: conditional loads end up in branches of
  // their own and serialise.
  load_row_offsets(d, t.r0, tid, srow);
  __syncthreads();
  if (!kfast) {
    // lanes along the rows; thread part p walks its quarter of the K range,
    // 16 elements at a time: the 16 offsets first, then 16 loads in flight
    constexpr int kQ = kSliceKPart / 4, kU = 16;
    const int row = tid % kSliceRows, part = tid / kSliceRows;
    double m = 0.0;
    const int ka = k_lo + part * kQ, kb = min(k_hi, ka + kQ);
    if (t.r0 + row < d.R && ka < kb && d.nkm == 1) {
      // one K mode (the usual case once adjacent modes are merged): the K
      // offset of element k is k * kstr for the whole wave, so all kQ loads
      // go out before the first is used (k past the range re-reads the
      // range's last element, which leaves the maximum unchanged)
      const int64_t ro = srow[row], ks = d.kstr[0];
      double v[kQ];
#pragma unroll
      for (int u = 0; u < kQ; ++u)
        v[u] = elem_mag<CPLX>(x, ro + (int64_t)min(ka + u, kb - 1) * ks);
#pragma unroll
      for (int u = 0; u < kQ; ++u) m = fmax(m, v[u]);
    } else if (t.r0 + row < d.R && ka < kb) {
      const int64_t ro = srow[row];
      KWalk w;
      w.init((uint32_t)ka, d);
      const int64_t o0 = w.off;
      for (int k = ka; k < kb; k += kU) {
        int64_t o[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          o[u] = (k + u < kb) ? w.off : o0;
          w.step(d);
        }
        double v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) v[u] = elem_mag<CPLX>(x, ro + o[u]);
#pragma unroll
        for (int u = 0; u < kU; ++u) m = fmax(m, (k + u < kb) ? v[u] : 0.0);
      }
    }
    ered[part][row] = mag_exponent(m);
  } else {
    // lanes along K (two elements each: the part is 128 wide); a wave takes
    // rows wave, wave+4, ... and issues the loads of all of them before
    // reducing
    static_assert(kSliceKPart == 128, "two K elements per lane");
    const int lane = tid & 63, wave = tid >> 6;
    constexpr int kRowsW = kSliceRows / 4;
    const int k0 = k_lo + lane, k1 = k0 + 64;
    const int c0 = min(k0, k_hi - 1), c1 = min(k1, k_hi - 1);
    double m[kRowsW];
#pragma unroll
    for (int i = 0; i < kRowsW; ++i) {
      const int64_t ro = srow[wave + 4 * i];
      const double a = elem_mag<CPLX>(x, ro + c0);
      const double b = elem_mag<CPLX>(x, ro + c1);
      m[i] = fmax(k0 < k_hi ? a : 0.0, k1 < k_hi ? b : 0.0);
    }
    // The 16 rows' exponents are reduced over the 64 lanes by a butterfly
    // that halves the rows a lane holds at each of the strides 32, 16, 8, 4
    // (15 lane exchanges instead of 16 x 6) and then reduces the quads;
    // lane l ends with row (l >> 2) of the wave.
    int w[kRowsW];
#pragma unroll
    for (int i = 0; i < kRowsW; ++i) w[i] = mag_exponent(m[i]);
#pragma unroll
    for (int n = kRowsW, b = 32; n > 1; n >>= 1, b >>= 1) {
      const bool hi = (lane & b) != 0;
#pragma unroll
      for (int j = 0; j < n / 2; ++j) {
        const int send = hi ? w[j] : w[j + n / 2];
        const int keep = hi ? w[j + n / 2] : w[j];
        w[j] = max(keep, __shfl_xor(send, b));
      }
    }
    w[0] = max(w[0], __shfl_xor(w[0], 2));
    w[0] = max(w[0], __shfl_xor(w[0], 1));
    if ((lane & 3) == 0) {
      const int row = wave + 4 * (lane >> 2);
      ered[0][row] = w[0];
      ered[1][row] = ered[2][row] = ered[3][row] = kZeroRow;
    }
  }
  __syncthreads();
  if (tid < kSliceRows && t.r0 + tid < d.R)
    pmax[d.pmax_off + (int64_t)t.kp * d.R + t.r0 + tid] =
        max(max(ered[0][tid], ered[1][tid]), max(ered[2][tid], ered[3][tid]));
}

// The S digits of 16 values x of a row with exponent e (kNonFinite: all zero),
// 16 bytes to each of the planes at dst, pstride apart.
template <int S>
__device__ __forceinline__ void slice_digits(const double (&x)[16], int e, int8_t* dst,
                                             int64_t pstride) {
  uint32_t packed[S][4];
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int w = 0; w < 4; ++w) packed[i][w] = 0u;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    // x / 2^E is exact (|.| < 1), the scale by 127 rounds once
    double y = ldexp(e == kNonFinite ? 0.0 : x[j], -e) * kSliceLead;
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const double v = rint(y);
      y = (y - v) * kSliceRadix;
      packed[i][j >> 2] |= ((uint32_t)((int32_t)v & 0xff)) << (8 * (j & 3));
    }
  }
#pragma unroll
  for (int i = 0; i < S; ++i)
    *reinterpret_cast<v4i*>(dst + i * pstride) =
        v4i{(int)packed[i][0], (int)packed[i][1], (int)packed[i][2], (int)packed[i][3]};
}

// Pass 2: row exponent E = max of the row's partials (0 for an all-zero row),
// then the S slices of every element of the tile.
// Slice sets per element: 1 (real) or 2 (re, im: complex); set s of block b
// starts at planes + sets*plane_off + s*S*R*Kpad.
template <int S, int CPLX>
__global__ void __launch_bounds__(kThreads)
    slice_kernel(const SliceBlock* __restrict__ blocks, const int2* __restrict__ wgmap,
                 SliceOperands ops) {
  __shared__ int32_t sexp[kSliceRows];
  __shared__ int64_t srow[kSliceRows];
  const SliceTile t = slice_tile(blocks, wgmap, blockIdx.x);
  const SliceBlock& d = blocks[t.b];
  const int r0 = t.r0;
  const int tid = threadIdx.x;
  const double* x = ops.src[d.side] + (CPLX ? 2 : 1) * d.off;
  int8_t* planes = ops.planes[d.side];
  int32_t* exps = ops.exps[d.side];
  const int32_t* pmax = ops.pmax[d.side];
  load_row_offsets(d, r0, tid, srow);
  if (tid < kSliceRows) {
    int e = kZeroRow;
    if (r0 + tid < d.R)
      for (int p = 0; p < d.kparts; ++p)
        e = max(e, pmax[d.pmax_off + (int64_t)p * d.R + r0 + tid]);
    if (e == kZeroRow) e = 0;
    sexp[tid] = e;
    if (t.kp == 0 && r0 + tid < d.R) exps[d.exp_off + r0 + tid] = e;
  }
  __syncthreads();

  // slice 16 consecutive k of one row per item; consecutive threads take
  // consecutive rows, so the 16-byte chunks they write are adjacent in the
  // chunk-major planes (a K-contiguous source is then read 128 bytes per
  // lane, which the L1 cache serves line by line)
  constexpr int kChunks = kSliceKPart / 16;
  const int ch_end = min(d.Kpad / 16, (t.kp + 1) * kChunks);
  const int64_t pstride = (int64_t)d.R * d.Kpad;
  // A thread has kItems items; for real data the loads of all of them go
  // out before the first item's digits are formed (complex data: one item
  // at a time, for registers). Items past the block (rows >= R, chunks past
  // the K range) load from clamped, valid addresses and store nothing.
  constexpr int kItems = kSliceRows * kChunks / kThreads;
  static_assert(kSliceRows * kChunks % kThreads == 0, "items per thread");
  constexpr int NB = CPLX ? 1 : kItems;
  constexpr int NC = CPLX ? 2 : 1;  // re, im
  for (int i0 = 0; i0 < kItems; i0 += NB) {
    double xr[NB][16], xi[NB][16];  // xi: complex data
    int eq[NB], grq[NB], chq[NB];
    bool lq[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int it = tid + (i0 + q) * kThreads;
      const int row = it % kSliceRows;
      const int ch0 = t.kp * kChunks + it / kSliceRows;
      const int gr = r0 + row;
      lq[q] = gr < d.R && ch0 < ch_end;
      const int ch = min(ch0, ch_end - 1);
      const int e = sexp[row];
      eq[q] = e;
      grq[q] = gr;
      chq[q] = ch;
      const int64_t ro = srow[row];
      KWalk kw;
      kw.init((uint32_t)(ch * 16), d);
      // the 16 offsets first (padding k >= K clamped onto the row's k = 0),
      // then the 16 loads back to back and unconditional
      int64_t off[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        off[j] = ro + (ch * 16 + j < d.K ? kw.off : 0);
        kw.step(d);
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const bool in = ch * 16 + j < d.K;
        if (CPLX) {
          const double2 v = reinterpret_cast<const double2*>(x)[off[j]];
          xr[q][j] = in ? v.x : 0.0;
          xi[q][j] = in ? v.y : 0.0;
        } else {
          const double v = x[off[j]];
          xr[q][j] = in ? v : 0.0;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      if (!lq[q]) continue;
      const int e = eq[q];
      // one slice set at a time (re, then im for complex data), so only one
      // set's packed digits are live: with all at once the complex kernel
      // needed a full register file and ran one wave per SIMD
      int8_t* dst =
          planes + NC * d.plane_off + ((int64_t)chq[q] * d.R + grq[q]) * 16;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        slice_digits<S>(c == 0 ? xr[q] : xi[q], e, dst + c * S * pstride, pstride);
      }
    }
  }
}

// Two values at any multiple of 8 bytes.
struct __attribute__((aligned(8))) Chunk {
  double x, y;
};

// One pass, for blocks whose K fits a workgroup (d.once rows x Kpad / 16 chunks
// <= kOnceChunks): a thread loads the values of its two chunks, the rows'
// exponents are the maxima of their chunks' (LDS), and the slices are formed
// from the values in registers. Bound by memory: 8 bytes read and 6 written per
// value. Four workgroups a CU (114 registers) overlap one's loads with another's
// digits: 256 threads and up to K = 2048 took 132 us for the operands of the U(1)
// chi = 4096 apply's two products (two passes: 186), 512 threads 143, 1024
// threads 174. 16384 x 512: 24 us rows first, 26 us K first (two passes: 40, 59);
// 16384 x 2048: 146 and 112 (161 and 190); 30 x 2000: 7.7 (19). With few rows a
// tile uses only part of each line, so neighbours run on one XCD, whose L2 holds
// the line (16384 x 2048 rows first without that: 236 us), and chunks that are
// contiguous in the operand are read 16 bytes at a time (143 us of the apply's
// 155 with 512 threads). Complex data (two passes) would need twice the registers.
template <int S>
__global__ void __launch_bounds__(kOnceThreads, 4)
    slice_once_kernel(const SliceBlock* __restrict__ blocks, const int2* __restrict__ map,
                      SliceOperands ops) {
  __shared__ int32_t sexp[kOnceThreads];
  __shared__ int64_t srow[kOnceThreads];
  constexpr int NI = kOnceChunks / kOnceThreads;
  static_assert(kOnceChunks / 2 <= kOnceThreads, "Kpad >= 32: at most a row per thread");
  // consecutive tiles to one XCD (workgroup w runs on XCD w % 8)
  const int n = gridDim.x, xcd = blockIdx.x % kXcds, per = n / kXcds, rem = n % kXcds;
  const int2 m = map[xcd * per + min(xcd, rem) + (int)blockIdx.x / kXcds];
  const SliceBlock& d = blocks[m.x];
  const int tid = threadIdx.x;
  const int r0 = m.y * d.once, rows = min(d.once, d.R - r0), chunks = d.Kpad / 16;
  const double* x = ops.src[d.side] + d.off;
  int8_t* planes = ops.planes[d.side] + d.plane_off;
  if (tid < rows) {
    srow[tid] = mode_offset((uint32_t)(r0 + tid), d.nrm, d.rdim, d.rstr);
    sexp[tid] = kZeroRow;
  }
  __syncthreads();
  // Consecutive threads take consecutive rows of a chunk. Every load is
  // unconditional, from a chunk clamped into the tile (one past it stores
  // nothing) and a k clamped into the row (padding).
  double v[NI][16];
  int row[NI], ch[NI];
  bool live[NI];
#pragma unroll
  for (int q = 0; q < NI; ++q) {
    const int it0 = tid + q * kOnceThreads, it = min(it0, rows * chunks - 1);
    live[q] = it0 == it;
    ch[q] = it / rows;
    row[q] = it - ch[q] * rows;
    const int64_t ro = srow[row[q]];
    const int k0 = ch[q] * 16;
    if (d.nkm == 1 && d.kstr[0] == 1 && k0 + 16 <= d.K) {
#pragma unroll
      for (int j = 0; j < 16; j += 2) {
        const Chunk c = *reinterpret_cast<const Chunk*>(x + ro + k0 + j);
        v[q][j] = c.x;
        v[q][j + 1] = c.y;
      }
    } else if (d.nkm == 1) {
      const int64_t ks = d.kstr[0];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[q][j] = x[ro + (int64_t)min(k0 + j, d.K - 1) * ks];
    } else {
      KWalk kw;
      kw.init((uint32_t)k0, d);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        v[q][j] = x[ro + (k0 + j < d.K ? kw.off : 0)];
        kw.step(d);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NI; ++q) {
    double mag = 0.0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (ch[q] * 16 + j >= d.K) v[q][j] = 0.0;
      mag = fmax(mag, isfinite(v[q][j]) ? fabs(v[q][j]) : INFINITY);
    }
    if (live[q]) atomicMax(&sexp[row[q]], mag_exponent(mag));
  }
  __syncthreads();
  const int64_t pstride = (int64_t)d.R * d.Kpad;
#pragma unroll
  for (int q = 0; q < NI; ++q) {
    if (!live[q]) continue;
    int e = sexp[row[q]];
    if (e == kZeroRow) e = 0;
    if (ch[q] == 0) ops.exps[d.side][d.exp_off + r0 + row[q]] = e;
    slice_digits<S>(v[q], e, planes + ((int64_t)ch[q] * d.R + r0 + row[q]) * 16, pstride);
  }
}

constexpr int kBT = kGemmTile;  // rows and columns of a workgroup's tile
constexpr int BKB = 32;  // K bytes per LDS stage (two 16-byte chunks)

typedef const __attribute__((address_space(4))) SplitPair* const_pair_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) void* gbl_ptr_t;

// 16 bytes per lane from global memory straight into LDS; lane l's bytes land
// at lds_base + 16*l (lds_base is wave-uniform, passed through M0).
__device__ inline void load_lds16(const int8_t* g, v4i* lds_base) {
  __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)lds_base, 16, 0, 0);
}

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt left at their maxima).
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | (((N >> 4) & 3) << 14));
}

// Workgroup barrier for the stage ring. __syncthreads() carries a release
// fence, which waits for every outstanding load -- including the LDS fills
// issued for later stages that are meant to stay in flight. Here the caller
// has already waited (vmcnt) for the stage the next step reads; this waits
// for the wave's own LDS reads (so no stage is refilled under a reader),
// then synchronises. The empty asm statements keep the compiler from moving
// memory operations across the barrier.
__device__ inline void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xF | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// f(0), f(1), ... with each argument a compile-time constant.
template <class F, int... N>
__device__ __attribute__((always_inline)) inline void static_for(F f,
                                                                 std::integer_sequence<int, N...>) {
  (f(std::integral_constant<int, N>{}), ...);
}
// The products of S digits by S in the order (0, 0), (0, 1), ..., (0, S - 1),
// (1, 0), ..., (1, S - 2), ...: number of the first one of digit i of the
// first factor, and that digit of product n.
template <int S>
constexpr int digit_first(int i) {
  return i * S - i * (i - 1) / 2;
}
template <int S>
constexpr int digit_row(int n) {
  int i = 0;
  while (n >= digit_first<S>(i + 1)) ++i;
  return i;
}

// The stages of a workgroup's 64 x 64 tile, filled as one sequence over the
// pairs of its group. A stage holds K bytes k..k+31 of the digit planes of
// both operands, [operand][plane][chunk][row] x 16 bytes, SETS * S planes per
// operand; wave w of four fetches chunk w & 1 of the planes of parity w >> 1.
// Past the last step every lane fetches the first row of the last pair again,
// into a stage nobody reads, so that every step issues the same loads and
// waits for the same count. The group has at least one pair.
template <int S, int SETS>
struct StageFill {
  static constexpr int kPlanes = SETS * S;
  static constexpr int kLoads = kPlanes;              // a wave's, per stage
  static constexpr int kOperand = kPlanes * 2 * kBT;  // 16-byte slots of one operand
  static constexpr int kStage = 2 * kOperand;
  const const_pair_t pairs;
  const int8_t *planesA, *planesB;
  const int M, N, p1, wave;
  int p;              // pair, K byte and padded K of the stage to fill next
  int k, kpad;
  const int8_t *a, *b;
  int64_t as, bs;     // plane strides
  uint32_t aoff, boff;  // this lane's row: rows past the block are clamped onto its last
                        // row (they only feed outputs that are never stored)
  v4i* dst;

  __device__ __attribute__((always_inline)) StageFill(const SplitPair* tab, const GemmGroup& g,
                                                      const int8_t* pa, const int8_t* pb, int m0,
                                                      int n0, int lane, int w)
      : pairs((const_pair_t)(uintptr_t)tab), planesA(pa), planesB(pb), M(g.M), N(g.N), p1(g.p1),
        wave(w), p(g.p0), k(0), kpad(0), a(nullptr), b(nullptr), as(0), bs(0),
        aoff((uint32_t)min(m0 + lane, g.M - 1) * 16u),
        boff((uint32_t)min(n0 + lane, g.N - 1) * 16u), dst(nullptr) {}
  __device__ __attribute__((always_inline)) void open() {
    const bool live = p < p1;
    const __attribute__((address_space(4))) SplitPair& pr = pairs[live ? p : p1 - 1];
    as = pr.a_pstride;
    bs = pr.b_pstride;
    a = planesA + SETS * pr.a_planes + pr.a_koff + (wave >> 1) * as + (int64_t)(wave & 1) * M * 16;
    b = planesB + SETS * pr.b_planes + pr.b_koff + (wave >> 1) * bs + (int64_t)(wave & 1) * N * 16;
    k = 0;
    kpad = pr.kpad;
    aoff = live ? aoff : 0u;
    boff = live ? boff : 0u;
  }
  __device__ __attribute__((always_inline)) void stage(v4i* st) { dst = st + wave * kBT; }
  // load t of kLoads into the stage
  __device__ __attribute__((always_inline)) void load(int t) const {
    constexpr int h = kPlanes / 2;
    if (t < h)
      load_lds16(a + 2 * t * as + aoff, dst + t * 4 * kBT);
    else
      load_lds16(b + 2 * (t - h) * bs + boff, dst + kOperand + (t - h) * 4 * kBT);
  }
  __device__ __attribute__((always_inline)) void next() {
    a += (int64_t)M * BKB;
    b += (int64_t)N * BKB;
    k += BKB;
    if (k >= kpad) {
      ++p;
      open();
    }
  }
  // both stages ahead of the first step; the first has landed on return
  __device__ __attribute__((always_inline)) void begin(v4i* lds) {
    open();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      stage(lds + i * kStage);
#pragma unroll
      for (int t = 0; t < kLoads; ++t) load(t);
      next();
    }
    wait_vmcnt<kLoads>();
    stage_barrier();
  }
};
constexpr int kRing = 3;  // LDS stages

// Whether dword q of S digits may be negated behind MFMA q + first of two
// quarters in a row: digit q / 4 after its last product with the old sign
// (first quarter; `old` false: it has none) and before its first with the new
// one, in the quarter that starts at MFMA `now`.
template <int S>
constexpr bool negation_fits(int first, bool old, int now) {
  for (int q = 0; q < 4 * S; ++q) {
    const int i = q / 4, at = q + first;
    if (old && at < digit_first<S>(i + 1) - 1) return false;
    if (at >= now + digit_first<S>(i)) return false;
  }
  return true;
}

// The four digits of a dword negated (a digit is at most 127 in magnitude):
// with l = the low seven bits, each byte is 128 - l with its sign bit flipped
// where the digit was not negative.
__device__ inline int negate_digits(int x) {
  const uint32_t h = 0x80808080u, u = (uint32_t)x;
  return (int)((~(u | h) + 0x01010101u) ^ (~u & h));
}

// Complex split GEMM, both components of C in one pass: 64 x 64 tiles, four
// waves of 32 x 32, one workgroup (one wave per SIMD) per CU. With A = ar + i
// ai and B = br + i bi a K step forms ar br and -ai bi into the levels of Re
// C, ar bi and ai br into those of Im C: 84 MFMAs per 24 fragment reads and
// 48 KB of fills, half of either per MFMA of a pass per component.
// DIFF: exactly one operand is conjugated (+ai bi, -ai br); negim: Im C is
// negated (B conjugated).
// Stages form one sequence over the pairs of the group: step s computes from
// stage s % 3 and fills step s + 2 into the stage step s - 1 read, also across
// the end of a pair, so the fills of the next pair run under this one's
// recombination. The barrier that opens the next stage comes before the last
// quarter of a step's MFMAs, and the next step's first fragments are read
// under that quarter.
// Against a pass per component (a 32 x 32 block of one component per wave, two
// waves per SIMD), MI355X: 7680 x 1536 x 6144 5.68 -> 4.47 ms, 1000^3 0.101 ->
// 0.071, 300^3 33 -> 22 us, 2000 x 64 x 2000 51 -> 48 us. It is bound by power:
// the matrix pipe is busy 73 % of the cycles at 1.8 GHz; the same product of
// zeros takes 3.36 ms, at 2.4 GHz. Without the negations (4 %) or with the
// compiler's instruction order (6 % slower) the balance is the same.
template <int S, bool DIFF>
__global__ void __launch_bounds__(kThreads, 1)
    split_gemm_cplx_kernel(const SplitPair* __restrict__ pairs,
                           const GemmGroup* __restrict__ groups,
                           const GemmTile* __restrict__ tiles, const int8_t* __restrict__ planesA,
                           const int8_t* __restrict__ planesB, const int32_t* __restrict__ expA,
                           const int32_t* __restrict__ expB, double2* __restrict__ Cg, double ga,
                           double beta, int negim, int aim) {
  using Fill = StageFill<S, 2>;
  constexpr int NLD = Fill::kLoads, NL = S;
  constexpr int NP = S * (S + 1) / 2;    // digit products of a quarter step
  static_assert(S + NLD <= NP, "a quarter holds S reads and the fills");
  // The 4 S dwords of ai are negated one behind each MFMA, in place: from
  // MFMA kNeg of the third quarter, digit i after its last product there and
  // before its first in the fourth; with DIFF (third quarter negated, fourth
  // not) also from MFMA kNegDiff of the second.
  constexpr int kNeg = S + 1, kNegDiff = S + 2;
  static_assert(negation_fits<S>(kNeg, true, NP) && negation_fits<S>(kNegDiff, false, NP),
                "negation order");
  __shared__ v4i lds[kRing * Fill::kStage];

  const GemmTile& tt = tiles[blockIdx.x];
  if (tt.g < 0) return;
  const GemmGroup grp = groups[tt.g];
  const int m0 = tt.m0, n0 = tt.n0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave & 1) * 32, wn0 = (wave >> 1) * 32;
  const int l32 = lane & 31, lh = lane >> 5;
  Fill fill(pairs, grp, planesA, planesB, m0, n0, lane, wave);

  double acc_re[16], acc_im[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc_re[r] = acc_im[r] = 0.0;

  // fragment of digit plane i of an operand's stage
  auto frag = [&](const v4i* op, int i, int w0) { return op[(i * 2 + lh) * kBT + w0 + l32]; };

  v4i ar[S], br[S];
  int st = 0;
  if (grp.p0 < grp.p1) {
    fill.begin(lds);
#pragma unroll
    for (int i = 0; i < S; ++i) ar[i] = frag(lds, i, wm0);
#pragma unroll
    for (int i = 0; i < S; ++i) br[i] = frag(lds + Fill::kOperand, i, wn0);
  }

  for (int p = grp.p0; p < grp.p1; ++p) {
    const __attribute__((address_space(4))) SplitPair& pr = fill.pairs[p];
    const int kpad = pr.kpad;
    v16i re[NL], im[NL];
#pragma unroll
    for (int L = 0; L < NL; ++L) re[L] = im[L] = v16i{0};
    const int32_t *xa = expA + pr.a_exp, *xb = expB + pr.b_exp;
    const int ea = xa[(uint32_t)min(m0 + wm0 + l32, grp.M - 1)];
    int eb[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      eb[r] = xb[(uint32_t)min(n0 + wn0 + (r & 3) + 8 * (r >> 2) + 4 * lh, grp.N - 1)];

    for (int k0 = 0; k0 < kpad; k0 += BKB) {
      const v4i* sA = lds + st * Fill::kStage;
      const v4i* sB = sA + Fill::kOperand;
      fill.stage(lds + (st == 0 ? kRing - 1 : st - 1) * Fill::kStage);
      if (++st == kRing) st = 0;
      const v4i* nA = lds + st * Fill::kStage;
      const v4i* nB = nA + Fill::kOperand;
      // One quarter of the step: the digit products a b into lev, with
      // after(n) issued behind MFMA n. A wave issues in order and an MFMA
      // keeps the matrix pipe busy for several issues, so reads, fills and
      // negations placed between MFMAs cost nothing; before a quarter they
      // would leave the pipe idle (the order is pinned).
      auto products = [&](const v4i (&a)[S], const v4i (&b)[S], v16i (&lev)[NL],
                          auto after) __attribute__((always_inline)) {
        static_for([&](auto n) __attribute__((always_inline)) {
          constexpr int i = digit_row<S>(n), j = n - digit_first<S>(i);
          lev[i + j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[j], a[i], lev[i + j], 0, 0, 0);
          after(n);
          __builtin_amdgcn_sched_barrier(0);
        }, std::make_integer_sequence<int, S * (S + 1) / 2>{});
      };
      v4i ai[S], bi[S];
      // dword q of the 4 S dwords of ai
      auto negate = [&](auto q) __attribute__((always_inline)) {
        if constexpr (q >= 0 && q < 4 * S) ai[q / 4][q % 4] = negate_digits(ai[q / 4][q % 4]);
      };
      products(ar, br, re, [&](auto n) __attribute__((always_inline)) {
        if constexpr (n < S) bi[n] = frag(sB, S + n, wn0);
      });
      products(ar, bi, im, [&](auto n) __attribute__((always_inline)) {
        if constexpr (n < S)
          ai[n] = frag(sA, S + n, wm0);
        else if constexpr (n < S + NLD)
          fill.load(n - S);
        if constexpr (DIFF) negate(std::integral_constant<int, n - kNegDiff>{});
      });
      products(ai, br, im, [&](auto n) __attribute__((always_inline)) {
        if constexpr (DIFF) negate(std::integral_constant<int, n + NP - kNegDiff>{});
        negate(std::integral_constant<int, n - kNeg>{});
      });
      fill.next();
      wait_vmcnt<NLD>();
      stage_barrier();
      // the next step's first fragments (past the last step: a stage nobody
      // reads, values unused)
      products(ai, bi, re, [&](auto n) __attribute__((always_inline)) {
        if constexpr (n < S)
          ar[n] = frag(nA, n, wm0);
        else if constexpr (n < 2 * S)
          br[n - S] = frag(nB, n - S, wn0);
        negate(std::integral_constant<int, n + NP - kNeg>{});
      });
    }

    // FP64 recombination of the levels, scaled per row/column
    const double al = ga * (aim ? pr.alpha_im : pr.alpha);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      auto join = [&](const v16i (&lev)[NL]) {
        double h = (double)lev[NL - 1][r];
#pragma unroll
        for (int L = NL - 2; L >= 0; --L) h = fma(h, kInvRadix, (double)lev[L][r]);
        const double v = ldexp(h * kInvLead2, ea + eb[r]);
        return (ea == kNonFinite || eb[r] == kNonFinite) ? __builtin_nan("") : v;
      };
      const double vr = join(re), vi = join(im);
      acc_re[r] = fma(al, vr, acc_re[r]);
      acc_im[r] = fma(al, negim ? -vi : vi, acc_im[r]);
      __builtin_amdgcn_sched_barrier(0);  // one output at a time: few registers
    }
  }
  wait_vmcnt<0>();  // no fill outlives the workgroup

  const int gm = m0 + wm0 + l32;
  if (gm >= grp.M) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int gn = n0 + wn0 + (r & 3) + 8 * (r >> 2) + 4 * lh;
    if (gn >= grp.N) continue;
    const int64_t o = grp.off_c + gm + (int64_t)gn * grp.ldc;
    double2 out = make_double2(acc_re[r], acc_im[r]);
    if (beta != 0.0) {
      const double2 c = Cg[o];
      out.x = fma(beta, c.x, out.x);
      out.y = fma(beta, c.y, out.y);
    }
    Cg[o] = out;
  }
}

// Real split GEMM: 64 x 64 tiles, four waves of 32 x 32, two workgroups (two
// waves per SIMD) per CU. As in the complex kernel the stages form one
// sequence over the pairs of the group and reads and fills are issued between
// MFMAs. A step's first seven fragments are read before it begins: the barrier
// that opens the next stage comes behind the products of digits 0 to 2 of A,
// after which digits 3 to 5 of B are free; 2 to 0 follow as their last products
// are issued, and the products of one digit of A run from the last digit of B
// down, so the fragment read last is needed last.
// Against stages restarted for every pair, with all reads ahead of the MFMAs
// (MI355X): the two products of the chi = 4096 U(1) network 410 -> 346 us,
// 4096^3 1.26 -> 1.08 ms, 1000^3 28.5 -> 22.3 us, 300^3 11 -> 7.8 us, 2000 x 64 x
// 2000 17 -> 15.3 us. 4096^3 is bound by power like the complex kernel (2.7
// POP/s in both); the U(1) blocks by the start and the end of their short
// tiles.
template <int S>
__global__ void __launch_bounds__(kThreads, 2)
    split_gemm_real_kernel(const SplitPair* __restrict__ pairs,
                           const GemmGroup* __restrict__ groups,
                           const GemmTile* __restrict__ tiles, const int8_t* __restrict__ planesA,
                           const int8_t* __restrict__ planesB, const int32_t* __restrict__ expA,
                           const int32_t* __restrict__ expB, double* __restrict__ Cg, double ga,
                           double beta) {
  using Fill = StageFill<S, 1>;
  constexpr int NLD = Fill::kLoads, NL = S;
  constexpr int NP = S * (S + 1) / 2;  // digit products of a step
  constexpr int kOpen = digit_first<S>(3) - 1;  // the next stage opens behind this MFMA
  static_assert(S % 2 == 0 && S + NLD - 1 <= kOpen, "reads and fills fit before the barrier");
  __shared__ v4i lds[kRing * Fill::kStage];

  const GemmTile& tt = tiles[blockIdx.x];
  if (tt.g < 0) return;
  const GemmGroup grp = groups[tt.g];
  const int m0 = tt.m0, n0 = tt.n0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave & 1) * 32, wn0 = (wave >> 1) * 32;
  const int l32 = lane & 31, lh = lane >> 5;
  Fill fill(pairs, grp, planesA, planesB, m0, n0, lane, wave);

  double acc[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0;

  auto frag = [&](const v4i* op, int i, int w0) { return op[(i * 2 + lh) * kBT + w0 + l32]; };

  v4i a[S], b[S];
  int st = 0;
  if (grp.p0 < grp.p1) {
    fill.begin(lds);
    a[0] = frag(lds, 0, wm0);
#pragma unroll
    for (int j = 0; j < S; ++j) b[j] = frag(lds + Fill::kOperand, j, wn0);
  }

  for (int p = grp.p0; p < grp.p1; ++p) {
    const __attribute__((address_space(4))) SplitPair& pr = fill.pairs[p];
    const int kpad = pr.kpad;
    v16i lev[NL];
#pragma unroll
    for (int L = 0; L < NL; ++L) lev[L] = v16i{0};
    const int32_t *xa = expA + pr.a_exp, *xb = expB + pr.b_exp;
    const int ea = xa[(uint32_t)min(m0 + wm0 + l32, grp.M - 1)];
    int eb[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      eb[r] = xb[(uint32_t)min(n0 + wn0 + (r & 3) + 8 * (r >> 2) + 4 * lh, grp.N - 1)];

    for (int k0 = 0; k0 < kpad; k0 += BKB) {
      const v4i* sA = lds + st * Fill::kStage;
      fill.stage(lds + (st == 0 ? kRing - 1 : st - 1) * Fill::kStage);
      if (++st == kRing) st = 0;
      const v4i* nA = lds + st * Fill::kStage;
      const v4i* nB = nA + Fill::kOperand;
      static_for([&](auto n) __attribute__((always_inline)) {
        // digit j descending: the digits of B freed first are read first
        constexpr int i = digit_row<S>(n), j = S - 1 - i - (n - digit_first<S>(i));
        lev[i + j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[j], a[i], lev[i + j], 0, 0, 0);
        if constexpr (n < S - 1) a[n + 1] = frag(sA, n + 1, wm0);
        if constexpr (n >= S - 1 && n < S - 1 + NLD) fill.load(n - (S - 1));
        if constexpr (n == kOpen) {
          fill.next();
          wait_vmcnt<NLD>();
          stage_barrier();
          a[0] = frag(nA, 0, wm0);
#pragma unroll
          for (int q = S - 1; q >= S - 3; --q) b[q] = frag(nB, q, wn0);
        }
        if constexpr (i >= 3 && n == digit_first<S>(i + 1) - 1) {
          constexpr int q = S - 1 - i;  // no later product uses it
          b[q] = frag(nB, q, wn0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }, std::make_integer_sequence<int, NP>{});
    }

#pragma unroll
    for (int r = 0; r < 16; ++r) {
      double h = (double)lev[NL - 1][r];
#pragma unroll
      for (int L = NL - 2; L >= 0; --L) h = fma(h, kInvRadix, (double)lev[L][r]);
      double v = ldexp(h * kInvLead2, ea + eb[r]);
      if (ea == kNonFinite || eb[r] == kNonFinite) v = __builtin_nan("");
      acc[r] = fma(ga * pr.alpha, v, acc[r]);
    }
  }
  wait_vmcnt<0>();  // no fill outlives the workgroup

  const int gm = m0 + wm0 + l32;
  if (gm >= grp.M) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int gn = n0 + wn0 + (r & 3) + 8 * (r >> 2) + 4 * lh;
    if (gn >= grp.N) continue;
    const int64_t o = grp.off_c + gm + (int64_t)gn * grp.ldc;
    double out = acc[r];
    if (beta != 0.0) out = fma(beta, Cg[o], out);
    Cg[o] = out;
  }
}

}  // namespace

int split_slices(int prec) { return prec == 2 ? kSliceCount : 0; }

hipError_t launch_slice(hipStream_t s, int prec, int cplx, const SliceBlock* blocks,
                        const SliceGrid& grid, const SliceOperands& ops) {
  if (prec != 2) return hipErrorNotSupported;
  hipError_t e;
  if (grid.n_once > 0) {
    ITG_LAUNCH((slice_once_kernel<kSliceCount>), dim3((unsigned)grid.n_once), dim3(kOnceThreads),
               0, s, blocks, grid.once, ops);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (grid.n_two == 0) return hipSuccess;
  const dim3 g((unsigned)grid.n_two), blk(kThreads);
  if (cplx) {
    ITG_LAUNCH((slice_max_kernel<1>), g, blk, 0, s, blocks, grid.two, ops);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    ITG_LAUNCH((slice_kernel<kSliceCount, 1>), g, blk, 0, s, blocks, grid.two, ops);
  } else {
    ITG_LAUNCH((slice_max_kernel<0>), g, blk, 0, s, blocks, grid.two, ops);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    ITG_LAUNCH((slice_kernel<kSliceCount, 0>), g, blk, 0, s, blocks, grid.two, ops);
  }
  return hipGetLastError();
}

int32_t slice_once_rows(int32_t rows, int32_t kpad) {
  if (rows <= 0 || kpad <= 0) return 0;
  const int32_t cap = kOnceChunks / (kpad / 16) / kOnceRowsMin * kOnceRowsMin;
  if (cap == 0) return 0;
  // as few row tiles as hold the rows, of even size
  const int32_t tiles = (rows + cap - 1) / cap, even = (rows + tiles - 1) / tiles;
  return (even + kOnceRowsMin - 1) / kOnceRowsMin * kOnceRowsMin;
}

int64_t slice_block_wgs(int32_t rows, int32_t kparts) {
  return (int64_t)((rows + kSliceRows - 1) / kSliceRows) * kparts;
}

hipError_t launch_split_gemm(hipStream_t s, int prec, const SplitPair* pairs,
                             const GemmGroup* groups, const GemmTile* tiles, int64_t grid,
                             const void* planesA, const void* planesB, const void* expA,
                             const void* expB, void* C, double ga, double beta) {
  if (grid == 0) return hipSuccess;
  if (prec != 2) return hipErrorNotSupported;
  ITG_LAUNCH((split_gemm_real_kernel<kSliceCount>), dim3((unsigned)grid), dim3(kThreads), 0, s,
             pairs, groups, tiles, (const int8_t*)planesA, (const int8_t*)planesB,
             (const int32_t*)expA, (const int32_t*)expB, (double*)C, ga, beta);
  return hipGetLastError();
}

hipError_t launch_split_gemm_cplx(hipStream_t s, int prec, bool conja, bool conjb,
                                  const SplitPair* pairs, const GemmGroup* groups,
                                  const GemmTile* tiles, int64_t grid, const void* planesA,
                                  const void* planesB, const void* expA, const void* expB,
                                  void* C, double ga, double beta, int aim) {
  if (grid == 0) return hipSuccess;
  if (prec != 2) return hipErrorNotSupported;
#define ITG_LAUNCH_CPLX(DIFF)                                                                 \
  ITG_LAUNCH((split_gemm_cplx_kernel<kSliceCount, DIFF>), dim3((unsigned)grid), dim3(kThreads), \
             0, s, pairs, groups, tiles, (const int8_t*)planesA, (const int8_t*)planesB,      \
             (const int32_t*)expA, (const int32_t*)expB, (double2*)C, ga, beta, (int)conjb,   \
             aim)
  if (conja != conjb)
    ITG_LAUNCH_CPLX(true);
  else
    ITG_LAUNCH_CPLX(false);
#undef ITG_LAUNCH_CPLX
  return hipGetLastError();
}

}  // namespace itg
