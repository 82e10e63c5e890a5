// Grouped FP64 GEMM on CDNA4 matrix cores (v_mfma_f64_16x16x4_f64).
//
// One launch covers every output block ("group") of a contraction plan: a
// dense contraction is one group with one pair; a QN block-sparse step has
// one group per output block and one pair per allowed (block1, block2).
// A workgroup owns one BM x BN tile of one group and walks the group's pairs
// in plan order, accumulating in registers, then writes the tile once:
//
//   C_g = beta*C_g (dense entry only) + sum_{p in g} alpha_p * op(A_p) op(B_p)
//
// so every output element has exactly one writer and a fixed summation
// order (deterministic, no atomics).
//
// Scheduling: the host builds a tile table in which workgroup w runs on XCD
// w % 8 (the hardware's round-robin dispatch). Each XCD receives whole groups
// (or large chunks of a big group) so the A and B panels of a group are
// fetched once into that XCD's L2 and shared by its tiles; chunks are spread
// over the XCDs largest-first to balance the work.
//
// Tiles: 256 threads = 4 wave64s in a 2x2 grid; each wave owns a
// (BM/2) x (BN/2) sub-tile as (BM/32) x (BN/32) MFMA 16x16 blocks of FP64
// accumulators and multiplies only the blocks that hold outputs. The MFMA is
// issued as D = B^T A^T so that each lane's accumulators run down a column
// of C, which makes the column-major epilogue stores contiguous.
//
// K loop: the slices (16 real or 8 complex values of k) of all pairs form one
// sequence. Slice s is multiplied from one LDS buffer while slice s + 1 goes
// from registers to the other, slice s + 2 is in registers and slice s + 3 is
// loaded, one barrier per slice; the fragments of each half slice are read
// while the other half's MFMAs run. What bounds it: the FP64 matrix pipe (76
// TF/s measured with MFMAs alone; one instruction takes 64 cycles) and, with
// it, every vector instruction, which FP64 MFMAs do not overlap (about 8 per
// slice and wave, in 16-byte loads and LDS accesses). A slice's MFMAs take 0.5
// us on a CU with one workgroup, less than a load that misses L2: with one
// slice in registers (four waves per SIMD) instead of two (three waves),
// 4096^3 took 2.08 instead of 1.95 ms, 3001 x 1777 x 2049 432 instead of 418 us,
// 4800 x 495 x 2100 218 instead of 206, the chi = 1024 dense network's two
// products (5120 x 4096 x 1024) 1.365 instead of 1.307 ms; complex products,
// the chi = 4096 U(1) network's (0.60 ms for both) and small ones are level.
//
// Complex data (interleaved re/im) uses the 4-real-product form on the same
// tiles, with conj(A)/conj(B) folded into the sign of the imaginary parts.
// Replaces BLAS dgemm/zgemm behind mul!! (NDTensors/src/abstractarray/mul.jl:1-12,
// NDTensors/src/array/mul.jl:1-4) and the per-pair loop of
// NDTensors/src/blocksparse/contract_generic.jl:78-129.
#include <algorithm>
#include <type_traits>

#include "itg_internal.h"

namespace itg {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kTile = 64;  // tile side
// A K slice of a tile holds 8 chunks of 16 bytes along K: 16 real or 8
// complex values.
constexpr int kChunksK = 8;

// 16 bytes at an address that need only be aligned to the element (NDTensors'
// block offsets put Float64 blocks on 8-byte boundaries).
struct __attribute__((aligned(8))) Chunk {
  double x, y;
};

// One operand of the tile: kTile rows (of M or N) by one K slice, moved from
// global memory to LDS in 16-byte chunks (two real values along the
// operand's contiguous mode, or one complex value). KC: the values of a row
// are contiguous along K (A stored K x M, B stored K x N), else along the rows.
//
// FP64 MFMAs and vector-ALU instructions do not overlap on a SIMD (a slice's
// cycles add up to MFMA busy + 4 per VALU instruction), so the steady state
// is kept free of the latter: a uniform base that advances per slice plus
// fixed 32-bit offsets for the loads, fixed LDS addresses, and every special
// case (conj, alpha, partial slices) behind a uniform branch.
template <int CPLX, int KC>
struct Operand {
  static constexpr int R = kTile;
  static constexpr int CE = CPLX ? 1 : 2;          // elements per chunk
  static constexpr int ES = CPLX ? 16 : 8;         // bytes per element
  static constexpr int BK = kChunksK * CE;         // contracted values per slice
  static constexpr int NCH = R * kChunksK / kThreads;  // chunks per thread
  static constexpr int RC = R / CE;                // chunks along the rows (KC = 0)
  static constexpr bool kLines = !CPLX && !KC;     // LDS rows of one k, else of one chunk of k
  // padded so that the lanes of a fragment read (kLines) or of a chunk write
  // fall on different banks
  static constexpr int kRowBytes = kLines ? (R + 8) * 8 : (R + 1) * 16;
  // 16 bytes in front: a chunk moved back by one row may start at row -1
  static constexpr int kBytes = 16 + (kLines ? BK : kChunksK) * kRowBytes;
  // LDS distance of a thread's consecutive chunks
  static constexpr int kStep = KC ? kThreads / kChunksK * 16 : kThreads / RC * kRowBytes;

  double2 v[2][NCH];  // the slices in flight
  const char* base;   // uniform: the next fast slice's first element
  uint32_t off[NCH];  // byte offsets of this thread's chunks from base
  uint32_t mask[2];   // masked slices: bits 2 r, 2 r + 1 for the halves of chunk r
  int wr, rd;         // LDS offsets: first chunk written, first fragment read

  // chunk r of this thread: first row / first k inside the tile
  static __device__ __forceinline__ int row(int tid, int r) {
    const int idx = tid + r * kThreads;
    return KC ? idx / kChunksK : (idx % RC) * CE;
  }
  static __device__ __forceinline__ int kofs(int tid, int r) {
    const int idx = tid + r * kThreads;
    return KC ? (idx % kChunksK) * CE : idx / RC;
  }
  // LDS offset of (row, k)
  static __device__ __forceinline__ int at(int row_, int k) {
    return 16 + (kLines ? k * kRowBytes + row_ * 8 : (k / CE) * kRowBytes + row_ * 16);
  }
  // Rows past the end re-read the last ones: they only feed outputs that are
  // not stored. A real chunk along the rows moves back by one when its second
  // row is past the end, in global memory and in LDS alike.
  static __device__ __forceinline__ int clamp_row(int g, int rows) {
    return min(g, rows - (KC ? 1 : CE));
  }
  __device__ __forceinline__ void init(int r0, int rows, int w0, int l16, int lk, int tid) {
    wr = at(kLines ? clamp_row(r0 + row(tid, 0), rows) - r0 : row(tid, 0), kofs(tid, 0));
    rd = 16 + (kLines ? 2 * lk * kRowBytes + (w0 + l16) * 8 : lk * kRowBytes + (w0 + l16) * 16);
  }
  // whether the byte offsets of a slice fit 32 bits (with room to spare)
  static __device__ __forceinline__ bool fits(int ld, int r0, int rows) {
    return (int64_t)ld * (KC ? min(R, rows - r0) : BK) <= (INT64_C(1) << 31) / ES;
  }
  // first slice of a pair's block: rows r0.. of `rows`, leading dimension ld
  __device__ __forceinline__ void start(const double* __restrict__ X, int64_t block, int64_t ld,
                                        int r0, int rows, int tid) {
    const int rb = max(clamp_row(r0, rows), 0);
    base = reinterpret_cast<const char*>(X) + (block + (KC ? rb * ld : rb)) * ES;
#pragma unroll
    for (int r = 0; r < NCH; ++r) {
      const uint32_t dr = (uint32_t)(clamp_row(r0 + row(tid, r), rows) - rb);
      const uint32_t k = (uint32_t)kofs(tid, r);
      off[r] = (KC ? dr * (uint32_t)ld + k : k * (uint32_t)ld + dr) * ES;
    }
  }
  // Buffer loads: a scalar base and a 32-bit lane offset, with no address
  // arithmetic on the vector ALU.
  template <int B>
  __device__ __forceinline__ void load_fast(int64_t ld) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, 0xffffffffu, 0x00027000);
#pragma unroll
    for (int r = 0; r < NCH; ++r)
      v[B][r] = __builtin_bit_cast(
          double2, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off[r], 0, 0));
    base += (KC ? 1 : ld) * (BK * ES);
  }
  // The last, partial slice of a pair (krem < BK values of k left, K >= 2):
  // chunks past the end re-read values of the slice (KC: the last two before
  // the end, which may start one value before the slice), and mask says
  // which elements count.
  template <int B>
  __device__ __forceinline__ void load_tail(int64_t ld, int krem, int tid) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(base) - ES, 0, 0xffffffffu, 0x00027000);
    mask[B] = 0u;
#pragma unroll
    for (int r = 0; r < NCH; ++r) {
      const int k = kofs(tid, r);
      const int back = max(k - (krem - (KC ? CE : 1)), 0);
      if (k < krem) mask[B] |= 1u << (2 * r);
      if (k + (KC ? CE - 1 : 0) < krem) mask[B] |= 2u << (2 * r);
      v[B][r] = __builtin_bit_cast(
          double2, __builtin_amdgcn_raw_buffer_load_b128(
                       rs, (int)(off[r] + ES - (uint32_t)back * (KC ? 1u : (uint32_t)ld) * ES), 0,
                       0));
    }
  }
  // any slice of a pair without fast loads (a block of one row, one
  // contracted value, or one that does not fit): element by element from
  // clamped addresses
  template <int B>
  __device__ __forceinline__ void load_slow(const double* __restrict__ X, int64_t block,
                                            int64_t ld, int r0, int rows, int k0, int K,
                                            int tid) {
    mask[B] = 0u;
#pragma unroll
    for (int r = 0; r < NCH; ++r) {
#pragma unroll
      for (int e = 0; e < CE; ++e) {
        const int g = r0 + row(tid, r) + (KC ? 0 : e), k = k0 + kofs(tid, r) + (KC ? e : 0);
        if (g < rows && k < K) mask[B] |= (CPLX ? 3u : 1u << e) << (2 * r);
        const int64_t gc = min(g, rows - 1), kc = min(k, K - 1);
        const int64_t o = block + (KC ? gc * ld + kc : kc * ld + gc);
        if (CPLX)
          v[B][r] = reinterpret_cast<const double2*>(X)[o];
        else if (e == 0)
          v[B][r].x = X[o];
        else
          v[B][r].y = X[o];
      }
    }
  }
  template <int B>
  __device__ __forceinline__ void store_fast(char* S) const {
#pragma unroll
    for (int r = 0; r < NCH; ++r) {
      Chunk c;
      c.x = v[B][r].x;
      c.y = v[B][r].y;
      *reinterpret_cast<Chunk*>(S + wr + r * kStep) = c;
    }
  }
  // slow: load_slow's, at the chunks' unmoved places; else load_tail's, where
  // the last value of an odd end is the second of the chunk that was re-read
  template <int B>
  __device__ __forceinline__ void store_masked(char* S, int tid, bool slow) const {
#pragma unroll
    for (int r = 0; r < NCH; ++r) {
      const bool in0 = mask[B] >> (2 * r) & 1u, in1 = mask[B] >> (2 * r + 1) & 1u;
      Chunk c;
      c.x = !CPLX && KC && !slow && !in1 ? v[B][r].y : v[B][r].x;
      c.x = in0 ? c.x : 0.0;
      c.y = in1 ? v[B][r].y : 0.0;
      char* d = !CPLX && !KC && slow ? S + at(row(tid, r), kofs(tid, r)) : S + wr + r * kStep;
      *reinterpret_cast<Chunk*>(d) = c;
    }
  }
  template <int B>
  __device__ __forceinline__ void conj() {
#pragma unroll
    for (int r = 0; r < NCH; ++r) v[B][r].y = -v[B][r].y;
  }
  template <int B>
  __device__ __forceinline__ void scale(double re, double im) {
#pragma unroll
    for (int r = 0; r < NCH; ++r)
      v[B][r] = CPLX ? make_double2(re * v[B][r].x - im * v[B][r].y, re * v[B][r].y + im * v[B][r].x)
                  : make_double2(re * v[B][r].x, re * v[B][r].y);
  }
  // The fragments of one wave for half a slice (Q = 0, 1), two values per
  // row: f[h][i], row w0 + 16 i + l16. Real: the MFMA steps h = 0, 1 take
  // k = 8 Q + 2 lk + h in lane group lk, the same map for both operands and
  // both storage orders; complex: h = real, imaginary part of k = 4 Q + lk.
  template <int F>
  __device__ __forceinline__ void frags(const char* S, int Q, double (&f)[2][F]) const {
#pragma unroll
    for (int i = 0; i < F; ++i) {
      if (kLines) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          f[h][i] = *reinterpret_cast<const double*>(S + rd + (8 * Q + h) * kRowBytes + i * 128);
      } else {
        const double2 c =
            *reinterpret_cast<const double2*>(S + rd + 4 * Q * kRowBytes + i * 256);
        f[0][i] = c.x;
        f[1][i] = c.y;
      }
    }
  }
};

// A workgroup barrier that waits for LDS accesses only (the global loads of
// the next slice stay in flight).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xF | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The tables are never written while a launch runs: scalar loads.
typedef const __attribute__((address_space(4))) GemmPair* PairTable;
typedef const __attribute__((address_space(4))) GemmGroup* GroupTable;
typedef const __attribute__((address_space(4))) GemmTile* TileTable;

template <int CPLX, int TA, int TB>
__global__ void __launch_bounds__(kThreads, 3)  // waves per SIMD
    gemm_f64_kernel(const GemmPair* __restrict__ pairs, const GemmGroup* __restrict__ groups,
                    const GemmTile* __restrict__ tiles, int quarters,
                    const double* __restrict__ Ag, const double* __restrict__ Bg,
                    double* __restrict__ Call, double* __restrict__ Pall, unsigned flags,
                    double ga_re, double ga_im,
                    double beta_re, double beta_im) {
  constexpr int NPLANE = CPLX ? 2 : 1;
  using OpA = Operand<CPLX, TA ? 1 : 0>;
  using OpB = Operand<CPLX, TB ? 0 : 1>;
  constexpr int BK = OpA::BK;

  __shared__ __attribute__((aligned(16))) char smem[2][OpA::kBytes + OpB::kBytes];

  // the four quarters of an entry run on the entry's XCD
  int entry = blockIdx.x, side = kTile, quarter = 0;
  if (quarters) {
    quarter = entry >> 3 & 3;
    entry = (entry >> 5) * 8 + (entry & 7);
    side = kTile / 2;
  }
  const TileTable tile = (TileTable)(uintptr_t)(tiles + entry);
  if (tile->g < 0) return;  // padding slot of the XCD-balanced table
  const GroupTable grp = (GroupTable)(uintptr_t)(groups + tile->g);
  const int ldc = grp->ldc;
  double* const Cg = grp->part ? Pall : Call;
  const bool use_beta = !grp->part && (beta_re != 0.0 || beta_im != 0.0);
  const int m0 = tile->m0 + (quarter & 1) * side, n0 = tile->n0 + (quarter >> 1) * side;
  if (m0 >= grp->M || n0 >= grp->N) return;
  // rows and columns of this workgroup: [m0, M) x [n0, N)
  const int M = min(grp->M, m0 + side), N = min(grp->N, n0 + side);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;

  // a chunk of two rows needs two rows
  const bool wide = CPLX || ((TA || M >= 2) && (!TB || N >= 2));

  // The slices of all pairs form one sequence: slice s is multiplied from LDS
  // buffer s % 2 while slices s + 1 and s + 2 are in registers, on their way
  // there, in the sets of the same parity.
  OpA a;
  OpB b;
  const PairTable ptab = (PairTable)(uintptr_t)pairs;
  // of the slice loaded last
  int p = grp->pf, k0 = 0, K = grp->K;
  int64_t off_a = grp->off_a, off_b = grp->off_b;
  int lda = grp->lda, ldb = grp->ldb;
  // of the slice in each set
  bool masked[2], fast[2];  // fast: of its pair
  bool special[2];          // conj or alpha to apply
  double al_re[2], al_im[2];
  auto same_pair = [&](auto set) __attribute__((always_inline)) {  // as the other set's
    constexpr int B = decltype(set)::value;
    fast[B] = fast[B ^ 1];
    special[B] = special[B ^ 1];
    al_re[B] = al_re[B ^ 1];
    al_im[B] = al_im[B ^ 1];
  };
  auto load = [&](auto set) __attribute__((always_inline)) {
    constexpr int B = decltype(set)::value;
    masked[B] = !fast[B] || k0 + BK > K;
    if (!masked[B]) {
      a.template load_fast<B>(lda);
      b.template load_fast<B>(ldb);
    } else if (fast[B]) {
      a.template load_tail<B>(lda, K - k0, tid);
      b.template load_tail<B>(ldb, K - k0, tid);
    } else {
      a.template load_slow<B>(Ag, off_a, lda, m0, M, k0, K, tid);
      b.template load_slow<B>(Bg, off_b, ldb, n0, N, k0, K, tid);
    }
  };
  // the first slice of pair p
  auto load_first = [&](auto set) __attribute__((always_inline)) {
    constexpr int B = decltype(set)::value;
    k0 = 0;
    fast[B] = wide && K >= 2 && OpA::fits(lda, m0, M) && OpB::fits(ldb, n0, N);
    if (fast[B]) {
      a.start(Ag, off_a, lda, m0, M, tid);
      b.start(Bg, off_b, ldb, n0, N, tid);
    }
    load(set);
    const double are = ptab[p].alpha_re, aim = ptab[p].alpha_im;
    al_re[B] = ga_re * are - ga_im * aim;
    al_im[B] = ga_re * aim + ga_im * are;
    special[B] = al_re[B] != 1.0 || (CPLX && (al_im[B] != 0.0 || (flags & 3u)));
  };
  // issue the loads of the slice after the last one into a set; false when
  // there is none
  auto load_next = [&](auto set) __attribute__((always_inline)) -> bool {
    k0 += BK;
    if (k0 < K) {
      same_pair(set);
      load(set);
      return true;
    }
    do {
      if (++p >= grp->p1) return false;
      K = ptab[p].K;
    } while (K <= 0);
    off_a = ptab[p].off_a;
    off_b = ptab[p].off_b;
    lda = ptab[p].lda;
    ldb = ptab[p].ldb;
    load_first(set);
    return true;
  };
  auto adjust = [&](auto set) __attribute__((always_inline)) {
    constexpr int B = decltype(set)::value;
    if (special[B]) {
      asm volatile("; conj, alpha");  // stays a branch: it is almost never taken
      if (CPLX && (flags & 1u)) a.template conj<B>();
      if (CPLX && (flags & 2u)) b.template conj<B>();
      if (al_re[B] != 1.0 || (CPLX && al_im[B] != 0.0))
        a.template scale<B>(al_re[B], al_im[B]);
    }
  };
  auto store_any = [&](auto set) __attribute__((always_inline)) {
    constexpr int B = decltype(set)::value;
    char* S = smem[B];
    adjust(set);
    if (!masked[B]) {
      a.template store_fast<B>(S);
      b.template store_fast<B>(S + OpA::kBytes);
    } else {
      a.template store_masked<B>(S, tid, !fast[B]);
      b.template store_masked<B>(S + OpA::kBytes, tid, !fast[B]);
    }
  };

  // The tile's product and its store, for a wave with NM x NN blocks of
  // 16 x 16 from (w_m, w_n) on (0 x 0: only its share of the loads). Every
  // wave of the workgroup passes the same barriers, whichever form it runs.
  auto run = [&](auto nm, auto nn, int w_m, int w_n) __attribute__((always_inline)) {
    constexpr int NM = decltype(nm)::value, NN = decltype(nn)::value;
    constexpr bool LIVE = NM > 0 && NN > 0;
    a.init(m0, M, w_m, l16, lk, tid);
    b.init(n0, N, w_n, l16, lk, tid);
    v4d acc[NPLANE][LIVE ? NM : 1][LIVE ? NN : 1];
#pragma unroll
    for (int c = 0; c < NPLANE; ++c)
#pragma unroll
      for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NN; ++j) acc[c][i][j] = v4d{0.0, 0.0, 0.0, 0.0};
    double fa[2][2][LIVE ? NM : 1], fb[2][2][LIVE ? NN : 1];  // [half slice][h][block]
    auto frags = [&](int Q, const char* S) __attribute__((always_inline)) {
      if constexpr (LIVE) {
        a.template frags<NM>(S, Q, fa[Q]);
        b.template frags<NN>(S + OpA::kBytes, Q, fb[Q]);
      }
    };
    auto mfmas = [&](int Q) __attribute__((always_inline)) {
      if constexpr (LIVE) {
#pragma unroll
        for (int h = 0; h < (CPLX ? 1 : 2); ++h)
#pragma unroll
          for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int j = 0; j < NN; ++j) {
              if (CPLX) {
                // re += Bre*Are - Bim*Aim ; im += Bre*Aim + Bim*Are
                acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[Q][0][j], fa[Q][0][i],
                                                                    acc[0][i][j], 0, 0, 0);
                acc[NPLANE - 1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    fb[Q][0][j], fa[Q][1][i], acc[NPLANE - 1][i][j], 0, 0, 0);
                acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-fb[Q][1][j], fa[Q][1][i],
                                                                    acc[0][i][j], 0, 0, 0);
                acc[NPLANE - 1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    fb[Q][1][j], fa[Q][0][i], acc[NPLANE - 1][i][j], 0, 0, 0);
              } else {
                acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[Q][h][j], fa[Q][h][i],
                                                                    acc[0][i][j], 0, 0, 0);
              }
            }
      }
    };
    // Slice s from its buffer: slice s + 1 (full) goes from its registers to
    // the other buffer and slice s + 3, a full one of the pair loaded last, is
    // loaded into them. The halves of a slice are read one half ahead of their
    // MFMAs; the other buffer was last read before the previous barrier.
    auto steady = [&](auto buf) __attribute__((always_inline)) {
      constexpr int B = decltype(buf)::value;
      adjust(std::integral_constant<int, B ^ 1>{});
      a.template store_fast<B ^ 1>(smem[B ^ 1]);
      b.template store_fast<B ^ 1>(smem[B ^ 1] + OpA::kBytes);
      frags(1, smem[B]);
      __builtin_amdgcn_sched_barrier(0);
      a.template load_fast<B ^ 1>(lda);
      b.template load_fast<B ^ 1>(ldb);
      mfmas(0);
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
      frags(0, smem[B ^ 1]);
      __builtin_amdgcn_sched_barrier(0);
      mfmas(1);
      __builtin_amdgcn_sched_barrier(0);
    };
    // the same for any slices s + 1 (there is one) and s + 3: have_after says
    // whether there is a slice s + 2, have_next then whether there is s + 3
    auto any = [&](auto buf, bool& have_next, bool& have_after) __attribute__((always_inline)) {
      constexpr int B = decltype(buf)::value;
      const std::integral_constant<int, B ^ 1> next{};
      store_any(next);
      frags(1, smem[B]);
      __builtin_amdgcn_sched_barrier(0);
      mfmas(0);
      have_next = have_after && load_next(next);
      lds_barrier();
      frags(0, smem[B ^ 1]);
      __builtin_amdgcn_sched_barrier(0);
      mfmas(1);
    };
    if (K > 0) {
      const std::integral_constant<int, 0> even{};
      const std::integral_constant<int, 1> odd{};
      load_first(even);
      bool have1 = load_next(odd), have0 = false;  // the sets hold slices to come
      store_any(even);
      if (have1) have0 = load_next(even);
      lds_barrier();
      frags(0, smem[0]);
      int buf = 0;
      for (;;) {
        // buffer 0 is next. Slices whose third successors are full slices of
        // the pair loaded last, two by two, while neither set is masked.
        if (have0 && !masked[0] && !masked[1]) {
          int n = (K - k0) / BK - 1;
          if (n >= 2) {
            n &= ~1;
            k0 += n * BK;
            do {
              steady(even);
              same_pair(odd);  // set 1 may have held the pair before
              steady(odd);
              n -= 2;
            } while (n);
          }
        }
        if (!have1) break;
        any(even, have1, have0);
        buf = 1;
        if (!have0) break;
        any(odd, have0, have1);
        buf = 0;
      }
      frags(1, smem[buf]);
      __builtin_amdgcn_sched_barrier(0);
      mfmas(0);
      mfmas(1);
    }
    // v_mfma_f64_16x16x4_f64 leaves D[i][j] in lane j + 16*(i%4), register
    // i/4 (rows interleaved across the four lane groups), so with D = (A B)^T
    // this lane holds C[m = l16][n = lk + 4*r] of each 16x16 block.
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      const int gm = m0 + w_m + i * 16 + l16;
      if (gm >= M) continue;
#pragma unroll
      for (int j = 0; j < NN; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gn = n0 + w_n + j * 16 + lk + 4 * r;
          if (gn >= N) continue;
          const int64_t o = grp->off_c + gm + (int64_t)gn * ldc;
          if (CPLX) {
            double2 out = make_double2(acc[0][i][j][r], acc[NPLANE - 1][i][j][r]);
            if (use_beta) {
              const double2 c = reinterpret_cast<double2*>(Cg)[o];
              out.x += beta_re * c.x - beta_im * c.y;
              out.y += beta_re * c.y + beta_im * c.x;
            }
            reinterpret_cast<double2*>(Cg)[o] = out;
          } else {
            double out = acc[0][i][j][r];
            if (use_beta) out = fma(beta_re, Cg[o], out);
            Cg[o] = out;
          }
        }
      }
    }
  };

  // Spread the live blocks (rm x rn of 4 x 4) over the waves: halves of both
  // sides, or, where fewer then fall to the busiest wave (an odd number of
  // blocks along a side), one block row or column each. Wave w of every
  // workgroup runs on the same SIMD, so work left with two waves of an edge
  // tile would leave the other SIMDs idle (27 % of the tiles at chi = 4096
  // U(1): 0.309 -> 0.302 ms per product; chi = 1500 complex 0.121 -> 0.115).
  const int rm = (M - m0 + 15) / 16, rn = (N - n0 + 15) / 16;
  const int hm = (rm + 1) / 2, hn = (rn + 1) / 2;
  int qm = hm, qn = hn;                              // blocks per wave
  int b_m = (wave & 1) * hm, b_n = (wave >> 1) * hn;  // this wave's first
  if (rm < hm * hn && rm <= rn) {
    qm = rm, qn = 1;
    b_m = 0, b_n = wave;
  } else if (rn < hm * hn) {
    qm = 1, qn = rn;
    b_m = wave, b_n = 0;
  }
  const std::integral_constant<int, 0> c0{};
  const std::integral_constant<int, 1> c1{};
  const std::integral_constant<int, 2> c2{};
  const std::integral_constant<int, 3> c3{};
  const int w_m = b_m * 16, w_n = b_n * 16;
  if (b_m >= rm || b_n >= rn)
    run(c0, c0, 0, 0);
  else if (qm == 2 && qn == 2)
    run(c2, c2, w_m, w_n);
  else if (qm == 3)
    run(c3, c1, w_m, w_n);
  else if (qn == 3)
    run(c1, c3, w_m, w_n);
  else if (qm == 2)
    run(c2, c1, w_m, w_n);
  else if (qn == 2)
    run(c1, c2, w_m, w_n);
  else
    run(c1, c1, w_m, w_n);
}

// C of the tiles computed in parts along K: four workgroups per tile, each
// thread up to four elements of it, every part's value added in order. Beta is
// applied as the GEMM's epilogue does.
template <int CPLX>
__global__ void __launch_bounds__(kThreads)
    gemm_join_kernel(const GemmJoin* __restrict__ joins, const double* __restrict__ P,
                     double* __restrict__ C, double beta_re, double beta_im) {
  const GemmJoin J = joins[blockIdx.x >> 2];
  const bool use_beta = (beta_re != 0.0 || beta_im != 0.0);
  const int mn = J.M * J.N;
  for (int e = (int)(blockIdx.x & 3) * kThreads + (int)threadIdx.x; e < mn; e += 4 * kThreads) {
    const int n = e / J.M, m = e - n * J.M;
    const int64_t o = J.off_c + m + (int64_t)n * J.ldc;
    if (CPLX) {
      const double2* p = reinterpret_cast<const double2*>(P) + J.poff + e;
      double2 v = p[0];
#pragma unroll 4
      for (int q = 1; q < J.S; ++q) {
        const double2 w = p[(int64_t)q * mn];
        v.x += w.x;
        v.y += w.y;
      }
      if (use_beta) {
        const double2 c = reinterpret_cast<double2*>(C)[o];
        v.x += beta_re * c.x - beta_im * c.y;
        v.y += beta_re * c.y + beta_im * c.x;
      }
      reinterpret_cast<double2*>(C)[o] = v;
    } else {
      const double* p = P + J.poff + e;
      double v = p[0];
#pragma unroll 4
      for (int q = 1; q < J.S; ++q) v += p[(int64_t)q * mn];
      if (use_beta) v = fma(beta_re, C[o], v);
      C[o] = v;
    }
  }
}

// The block of output element e, found by binary search over the blocks'
// first elements (a split-K plan has few blocks).
__device__ inline int ksplit_block(const KsReduce* red, int nred, int64_t e) {
  int lo = 0, hi = nred - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (red[mid].e0 <= e)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// WIDE = false: one thread per output element, adding the partials in slice
// order. WIDE = true (many slices, few elements: inner products, small
// cotangents): one wave per output element, lane l adding slices l, l + 64,
// ... in order, then a butterfly over the lanes -- a fixed order for a given
// slice count, so the result is deterministic. Beta is applied as the
// GEMM's epilogue does.
template <int CPLX, bool WIDE>
__global__ void __launch_bounds__(kThreads)
    ksplit_reduce_kernel(const KsReduce* __restrict__ red, int nred, int64_t total,
                         const double* __restrict__ P, double* __restrict__ C, double beta_re,
                         double beta_im) {
  const bool use_beta = (beta_re != 0.0 || beta_im != 0.0);
  constexpr int kPer = WIDE ? 64 : 1;  // threads per element
  const int lane = WIDE ? (int)(threadIdx.x & 63) : 0;
  const int64_t stride = (int64_t)gridDim.x * (kThreads / kPer);
  for (int64_t e = (int64_t)blockIdx.x * (kThreads / kPer) + threadIdx.x / kPer; e < total;
       e += stride) {
    const KsReduce r = red[ksplit_block(red, nred, e)];
    const int64_t loc = e - r.e0, mn = (int64_t)r.M * r.N;
    double vr = 0.0, vi = 0.0;
    // unrolled so that the loads of several slices are in flight at once
#pragma unroll 8
    for (int q = lane; q < r.S; q += kPer) {
      if (CPLX) {
        const double2 w = reinterpret_cast<const double2*>(P)[r.poff + q * mn + loc];
        vr = q == lane ? w.x : vr + w.x;
        vi = q == lane ? w.y : vi + w.y;
      } else {
        const double w = P[r.poff + q * mn + loc];
        vr = q == lane ? w : vr + w;
      }
    }
    if (WIDE) {
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) {
        vr += __shfl_xor(vr, m);
        if (CPLX) vi += __shfl_xor(vi, m);
      }
      if (lane != 0) continue;
    }
    const int64_t n = loc / r.M, m = loc - n * r.M;
    const int64_t o = r.off_c + m + n * r.ldc;
    if (CPLX) {
      double2 v = make_double2(vr, vi);
      if (use_beta) {
        const double2 c = reinterpret_cast<double2*>(C)[o];
        v.x += beta_re * c.x - beta_im * c.y;
        v.y += beta_re * c.y + beta_im * c.x;
      }
      reinterpret_cast<double2*>(C)[o] = v;
    } else {
      double v = vr;
      if (use_beta) v = fma(beta_re, C[o], v);
      C[o] = v;
    }
  }
}

// Split-K partial blocks of dot-like plans (every output block has at most
// kKsDotMN elements: inner products, norms): one workgroup per (block,
// slice) entry of the split tables streams its sub-pairs' operands once on
// the vector ALUs (a 64 x 64 MFMA tile would compute 4096 products per
// useful one), each thread summing every kThreads-th contracted value into
// M x N accumulators (MNC = 1: one output, four values in flight per thread;
// MNC = kKsDotMN: up to that many outputs); the workgroup then adds its
// threads' sums (a fixed tree) and writes the partial block. Per pair, the
// sum is scaled by that pair's factor times the global one, as the GEMM
// scales its A operand.
template <int CPLX, int MNC>
__global__ void __launch_bounds__(kThreads)
    ksplit_dot_kernel(const GemmPair* __restrict__ pairs, const GemmGroup* __restrict__ groups,
                      const double* __restrict__ Ag, const double* __restrict__ Bg,
                      double* __restrict__ P, int ta, int tb, unsigned flags, double ga_re,
                      double ga_im) {
  constexpr int NP = CPLX ? 2 : 1;
  constexpr int U = MNC == 1 ? 4 : 1;  // contracted values per thread in flight
  __shared__ double red[kThreads / 64][MNC * NP];
  const GemmGroup grp = groups[blockIdx.x];
  const int M = grp.M, MN = MNC == 1 ? 1 : grp.M * grp.N;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double sa = (flags & 1u) ? -1.0 : 1.0;  // conj(A): negate Im(A)
  const double sb = (flags & 2u) ? -1.0 : 1.0;
  double tot[MNC][NP];
#pragma unroll
  for (int i = 0; i < MNC; ++i)
#pragma unroll
    for (int c = 0; c < NP; ++c) tot[i][c] = 0.0;
  for (int p = grp.p0; p < grp.p1; ++p) {
    const GemmPair pr = pairs[p];
    double acc[MNC][NP];
#pragma unroll
    for (int i = 0; i < MNC; ++i)
#pragma unroll
      for (int c = 0; c < NP; ++c) acc[i][c] = 0.0;
    for (int k0 = tid; k0 < pr.K; k0 += U * kThreads) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * kThreads;
        if (U > 1 && k >= pr.K) break;
#pragma unroll
        for (int i = 0; i < MNC; ++i) {
          if (MNC > 1 && i >= MN) continue;
          const int m = i % M, n = i / M;
          const int64_t oa =
              pr.off_a + (ta ? (int64_t)m * pr.lda + k : (int64_t)k * pr.lda + m);
          const int64_t ob =
              pr.off_b + (tb ? (int64_t)k * pr.ldb + n : (int64_t)n * pr.ldb + k);
          if (CPLX) {
            const double2 a = reinterpret_cast<const double2*>(Ag)[oa];
            const double2 b = reinterpret_cast<const double2*>(Bg)[ob];
            const double ai = sa * a.y, bi = sb * b.y;
            acc[i][0] = fma(a.x, b.x, fma(-ai, bi, acc[i][0]));
            acc[i][NP - 1] = fma(a.x, bi, fma(ai, b.x, acc[i][NP - 1]));
          } else {
            acc[i][0] = fma(Ag[oa], Bg[ob], acc[i][0]);
          }
        }
      }
    }
    const double al_re = ga_re * pr.alpha_re - ga_im * pr.alpha_im;
    const double al_im = ga_re * pr.alpha_im + ga_im * pr.alpha_re;
#pragma unroll
    for (int i = 0; i < MNC; ++i) {
      if (CPLX) {
        tot[i][0] += al_re * acc[i][0] - al_im * acc[i][NP - 1];
        tot[i][NP - 1] += al_re * acc[i][NP - 1] + al_im * acc[i][0];
      } else {
        tot[i][0] += al_re * acc[i][0];
      }
    }
  }
  // threads -> waves (butterfly), waves -> one thread per output (wave order)
#pragma unroll
  for (int i = 0; i < MNC; ++i)
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      double v = tot[i][c];
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
      if (lane == 0) red[wave][i * NP + c] = v;
    }
  __syncthreads();
  if (tid < MN) {
    double v[NP];
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      v[c] = red[0][tid * NP + c];
      for (int w = 1; w < kThreads / 64; ++w) v[c] += red[w][tid * NP + c];
    }
    const int m = tid % M, n = tid / M;
    const int64_t o = grp.off_c + m + (int64_t)n * grp.ldc;
    if (CPLX)
      reinterpret_cast<double2*>(P)[o] = make_double2(v[0], v[NP - 1]);
    else
      P[o] = v[0];
  }
}

// Split-K partial blocks of skinny plans (every output block has one side of
// at most kKsSkinny: matrix times vector or a few vectors). Workgroup w
// takes consecutive rows of the long side of entry rows[w].x of the split
// tables, starting at rows[w].y, and writes those rows of the partial
// block. KC = 0 (the long side's rows run along the long side in memory):
// 256 rows, a thread owns one and walks the entry's contracted values in
// order, four in flight, so a wave's loads are 64 consecutive rows. KC = 1
// (each row is contiguous along the contracted values): 16 rows, a wave
// takes four of them with its lanes striding along the contracted values,
// then adds each row's lane sums with a butterfly. The short side's values
// are the same for every row (they come from the caches). Per pair the sums
// are scaled by that pair's factor times the global one.
template <int CPLX, int KC>
__global__ void __launch_bounds__(kThreads)
    ksplit_skinny_kernel(const GemmPair* __restrict__ pairs, const GemmGroup* __restrict__ groups,
                         const int2* __restrict__ rows, const double* __restrict__ Ag,
                         const double* __restrict__ Bg, double* __restrict__ P, int ta, int tb,
                         unsigned flags, double ga_re, double ga_im) {
  constexpr int NP = CPLX ? 2 : 1;
  constexpr int CS = kKsSkinny;
  constexpr int NR = KC ? 4 : 1;  // rows per thread (KC = 1: per wave)
  const int2 t = rows[blockIdx.x];
  const GemmGroup grp = groups[t.x];
  const bool mrows = grp.N <= CS;  // the long side is M (A's rows), else N
  const int R = mrows ? grp.M : grp.N, C = mrows ? grp.N : grp.M;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = KC ? t.y + wave * NR : t.y + (int)threadIdx.x;
  if (r0 >= R) return;  // KC = 1: the whole wave (r0 is the same on every lane)
  const double sa = (flags & 1u) ? -1.0 : 1.0;  // conj(A): negate Im(A)
  const double sb = (flags & 2u) ? -1.0 : 1.0;
  double tot[NR][CS][NP];
#pragma unroll
  for (int j = 0; j < NR; ++j)
#pragma unroll
    for (int c = 0; c < CS; ++c)
#pragma unroll
      for (int q = 0; q < NP; ++q) tot[j][c][q] = 0.0;
  for (int p = grp.p0; p < grp.p1; ++p) {
    const GemmPair pr = pairs[p];
    // element (m, k) of A and (n, k) of B, as the GEMM kernel indexes them
    auto aoff = [&](int m, int k) {
      return pr.off_a + (ta ? (int64_t)m * pr.lda + k : (int64_t)k * pr.lda + m);
    };
    auto boff = [&](int n, int k) {
      return pr.off_b + (tb ? (int64_t)k * pr.ldb + n : (int64_t)n * pr.ldb + k);
    };
    double acc[NR][CS][NP];
#pragma unroll
    for (int j = 0; j < NR; ++j)
#pragma unroll
      for (int c = 0; c < CS; ++c)
#pragma unroll
        for (int q = 0; q < NP; ++q) acc[j][c][q] = 0.0;
    // KC = 0: k = 0, 1, ... four at a time; KC = 1: k = lane, lane + 64, ...
    constexpr int U = KC ? 1 : 4;
    for (int k0 = KC ? lane : 0; k0 < pr.K; k0 += KC ? 64 : U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u;
        if (!KC && k >= pr.K) break;
#pragma unroll
        for (int j = 0; j < NR; ++j) {
          const int rr = min(r0 + j, R - 1);  // rows past R: computed, not stored
          const int64_t ox = mrows ? aoff(rr, k) : boff(rr, k);
          if (CPLX) {
            double2 x = reinterpret_cast<const double2*>(mrows ? Ag : Bg)[ox];
            x.y *= mrows ? sa : sb;
#pragma unroll
            for (int c = 0; c < CS; ++c) {
              if (c >= C) break;
              double2 y = reinterpret_cast<const double2*>(mrows ? Bg : Ag)[mrows ? boff(c, k)
                                                                                  : aoff(c, k)];
              y.y *= mrows ? sb : sa;
              acc[j][c][0] = fma(x.x, y.x, fma(-x.y, y.y, acc[j][c][0]));
              acc[j][c][NP - 1] = fma(x.x, y.y, fma(x.y, y.x, acc[j][c][NP - 1]));
            }
          } else {
            const double x = (mrows ? Ag : Bg)[ox];
#pragma unroll
            for (int c = 0; c < CS; ++c) {
              if (c >= C) break;
              const double y = (mrows ? Bg : Ag)[mrows ? boff(c, k) : aoff(c, k)];
              acc[j][c][0] = fma(x, y, acc[j][c][0]);
            }
          }
        }
      }
    }
    const double al_re = ga_re * pr.alpha_re - ga_im * pr.alpha_im;
    const double al_im = ga_re * pr.alpha_im + ga_im * pr.alpha_re;
#pragma unroll
    for (int j = 0; j < NR; ++j)
#pragma unroll
      for (int c = 0; c < CS; ++c) {
        double ar = acc[j][c][0], ai = acc[j][c][NP - 1];
        if (KC) {  // the row's sum over the wave's lanes (a fixed tree)
#pragma unroll
          for (int m = 32; m >= 1; m >>= 1) {
            ar += __shfl_xor(ar, m);
            if (CPLX) ai += __shfl_xor(ai, m);
          }
        }
        if (CPLX) {
          tot[j][c][0] += al_re * ar - al_im * ai;
          tot[j][c][NP - 1] += al_re * ai + al_im * ar;
        } else {
          tot[j][c][0] += al_re * ar;
        }
      }
  }
  if (KC && lane != 0) return;
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    if (r0 + j >= R) break;
#pragma unroll
    for (int c = 0; c < CS; ++c) {
      if (c >= C) break;
      const int m = mrows ? r0 + j : c, n = mrows ? c : r0 + j;
      const int64_t o = grp.off_c + m + (int64_t)n * grp.ldc;
      if (CPLX)
        reinterpret_cast<double2*>(P)[o] = make_double2(tot[j][c][0], tot[j][c][NP - 1]);
      else
        P[o] = tot[j][c][0];
    }
  }
}

}  // namespace

hipError_t launch_ksplit_reduce(hipStream_t s, int cplx, const KsReduce* red, int nred,
                                int64_t total, int max_slices, const void* P, void* C,
                                double beta_re, double beta_im) {
  if (total <= 0) return hipSuccess;
  if (nred <= 0) return hipErrorInvalidValue;
  const bool wide = max_slices >= 64;
  const int64_t per_block = wide ? kThreads / 64 : kThreads;
  const int64_t blocks = std::min<int64_t>((total + per_block - 1) / per_block, 4096);
#define ITG_KS_LAUNCH(c, w)                                                                  \
  ITG_LAUNCH((ksplit_reduce_kernel<c, w>), dim3((unsigned)blocks), dim3(kThreads), 0, s, red, \
             nred, total, (const double*)P, (double*)C, beta_re, beta_im)
  if (cplx && wide)
    ITG_KS_LAUNCH(1, true);
  else if (cplx)
    ITG_KS_LAUNCH(1, false);
  else if (wide)
    ITG_KS_LAUNCH(0, true);
  else
    ITG_KS_LAUNCH(0, false);
#undef ITG_KS_LAUNCH
  return hipGetLastError();
}

hipError_t launch_ksplit_dot(hipStream_t s, int cplx, int one, int ta, int tb,
                             const GemmPair* pairs, const GemmGroup* groups, int64_t ngroups,
                             const void* A, const void* B, void* P, unsigned flags,
                             double ga_re, double ga_im) {
  if (ngroups <= 0) return hipSuccess;
#define ITG_DOT_LAUNCH(c, mn)                                                                  \
  ITG_LAUNCH((ksplit_dot_kernel<c, mn>), dim3((unsigned)ngroups), dim3(kThreads), 0, s, pairs, \
             groups, (const double*)A, (const double*)B, (double*)P, ta, tb, flags, ga_re,     \
             ga_im)
  if (cplx && one)
    ITG_DOT_LAUNCH(1, 1);
  else if (cplx)
    ITG_DOT_LAUNCH(1, kKsDotMN);
  else if (one)
    ITG_DOT_LAUNCH(0, 1);
  else
    ITG_DOT_LAUNCH(0, kKsDotMN);
#undef ITG_DOT_LAUNCH
  return hipGetLastError();
}

hipError_t launch_ksplit_skinny(hipStream_t s, int cplx, int kc, int ta, int tb,
                                const GemmPair* pairs, const GemmGroup* groups, const int2* rows,
                                int64_t nrows, const void* A, const void* B, void* P,
                                unsigned flags, double ga_re, double ga_im) {
  if (nrows <= 0) return hipSuccess;
#define ITG_SK_LAUNCH(c, k)                                                                    \
  ITG_LAUNCH((ksplit_skinny_kernel<c, k>), dim3((unsigned)nrows), dim3(kThreads), 0, s, pairs, \
             groups, rows, (const double*)A, (const double*)B, (double*)P, ta, tb, flags,      \
             ga_re, ga_im)
  if (cplx && kc)
    ITG_SK_LAUNCH(1, 1);
  else if (cplx)
    ITG_SK_LAUNCH(1, 0);
  else if (kc)
    ITG_SK_LAUNCH(0, 1);
  else
    ITG_SK_LAUNCH(0, 0);
#undef ITG_SK_LAUNCH
  return hipGetLastError();
}

hipError_t launch_gemm_join(hipStream_t s, int cplx, const GemmJoin* joins, int64_t n,
                            const void* P, void* C, double beta_re, double beta_im) {
  if (n == 0) return hipSuccess;
  if (n > INT32_MAX / 4) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(4 * n));
  if (cplx)
    ITG_LAUNCH((gemm_join_kernel<1>), grid, dim3(kThreads), 0, s, joins, (const double*)P,
               (double*)C, beta_re, beta_im);
  else
    ITG_LAUNCH((gemm_join_kernel<0>), grid, dim3(kThreads), 0, s, joins, (const double*)P,
               (double*)C, beta_re, beta_im);
  return hipGetLastError();
}

hipError_t launch_gemm_f64(hipStream_t s, int cplx, int ta, int tb, const GemmPair* pairs,
                           const GemmGroup* groups, const GemmTile* tiles, int64_t entries,
                           bool quarters, const void* A, const void* B, void* C, void* P,
                           unsigned flags, double ga_re, double ga_im, double beta_re,
                           double beta_im) {
  const int64_t grid = quarters ? 4 * entries : entries;
  if (grid == 0) return hipSuccess;
  if (entries % 8 || grid > INT32_MAX) return hipErrorInvalidValue;
#define ITG_GEMM_CASE(c, a, b)                                                                   \
  if ((cplx != 0) == c && (ta != 0) == a && (tb != 0) == b) {                                    \
    ITG_LAUNCH((gemm_f64_kernel<c, a, b>), dim3((unsigned)grid), dim3(kThreads), 0, s, pairs,    \
               groups, tiles, (int)quarters, (const double*)A, (const double*)B, (double*)C,     \
               (double*)P, flags, ga_re, ga_im, beta_re, beta_im);                               \
    return hipGetLastError();                                                                    \
  }
  ITG_GEMM_CASE(0, 0, 0)
  ITG_GEMM_CASE(0, 0, 1)
  ITG_GEMM_CASE(0, 1, 0)
  ITG_GEMM_CASE(0, 1, 1)
  ITG_GEMM_CASE(1, 0, 0)
  ITG_GEMM_CASE(1, 0, 1)
  ITG_GEMM_CASE(1, 1, 0)
  ITG_GEMM_CASE(1, 1, 1)
#undef ITG_GEMM_CASE
  return hipErrorInvalidValue;
}

}  // namespace itg
