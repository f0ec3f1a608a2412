// Float32 tile engine on the matrix cores, shared by the covariance (SYRK) and
// preconditioning (GEMM) kernels; the convolution kernels use its tile shapes, accumulator
// layout and epilogues with main loops of their own, the inverse its split of operands.
//
// A workgroup of 256 threads (4 waves, 2 x 2) computes a (64*WM) x (64*WN)
// tile of  D[i][j] = sum_k Aop(i, k) * Bop(j, k);  each wave owns WM x WN
// accumulator blocks of 32 x 32.  Operand panels (rows x 32 k-values) are
// staged through LDS by "loaders" that know how an operand is laid out in
// memory:
//
//   LoaderKC  k is the contiguous index:  (sample, row, l) tensors such as an
//             NCHW activation viewed as rows = channel, k = (sample, pixel),
//             and plain row-major matrices used as the k-contiguous operand.
//   LoaderKS  row is the contiguous index: a row-major (k, row) matrix, e.g.
//             the (batch, features) input of a Linear layer or the right-hand
//             operand of an NN product; an optional extra row supplies the
//             bias column (a second array).
//   LoaderIM  implicit im2col: row = (c, kh, kw), k = (sample, y, x);
//             the patch matrix is gathered straight from the NCHW tensor.
//
// The float32 product.  The matrix cores multiply float32 at 256 flop per cycle
// and CU and bfloat16 at 4096.  A float32 number (of the range at note_least below; a
// tile with others takes the float32 instruction) is the exact sum of three
// bfloat16 numbers (8 significand bits each: 24 in all), x = hi + mid + lo, each
// the rounded rest of the one before, so a product of two float32 numbers is nine
// products of bfloat16 numbers, every one exact in float32.  The three smallest
// (mid*lo, lo*mid, lo*lo: at most 2^-23 of the product together, of either sign) are
// left out; the other six are accumulated in float32.  hi*hi has an accumulator of its
// own: it is rounded once per instruction, every sixteen k-values, where the float32
// instruction is rounded every two; the five small products add up in a second one,
// whose roundings are 2^-8 as large, and the two are added at the end.  (All six in one
// accumulator round it six times per sixteen k-values, also where half of the operands
// are zeros and the float32 sum is not rounded at all: 1.05 to 1.8 times the float32
// instruction's error for rectified operands.)  The error against float64, root mean
// square relative to sum |a||b|, over that of the float32 instruction: signed operands
// 0.68 at 4 k-values, 0.43 at 16, 0.32 at 128, 0.5 at 8192; rectified ones 0.96, 0.73,
// 0.51, 0.96 (one in six nonzero: 1.02, 0.99, 0.78, 0.99); magnitudes spread over e^6
// 0.84, 0.63, 0.41, 0.49.  The split is the published one of Henry, Tang and
// Heinecke (2019).  Six products of bfloat16 at the rate a large library product
// reaches here (1370 TFLOP/s at the clock the power budget leaves) are 228 TFLOP/s
// of float32, against 157 that the float32 instructions could reach at best.  With the
// float32 instruction and with split products: the covariance of 2048 rows of 4096 364 and
// 264 us, a layer of 512 x 4609 preconditioned 299 and 239 us.
//
// An LDS panel holds one row of the operand after the other: 32 k-values of hi
// (64 bytes), of mid, of lo, and 16 bytes that spread the rows over the banks.  A
// lane's operand of v_mfma_f32_32x32x16_bf16 is eight consecutive k-values of a
// plane, one 16-byte chunk; the chunks of a row are stored at their index xor
// (row / 16) mod 4, so that the writes of every loader below (rows four apart in
// LoaderKS) and the 16-byte reads all spread over the 64 banks.  One LDS buffer:
// the next panel is prefetched into registers while the current one feeds the
// matrix cores, and split when it is stored.
#pragma once

#include <hip/hip_runtime.h>

namespace kfac {
namespace mma {

constexpr int KT = 32;        // k-values per LDS panel
constexpr int THREADS = 256;  // 4 waves
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

// Loads from global memory at a wave-uniform base plus a 32-bit byte offset per
// lane: the form of the load instruction that takes the base from scalar
// registers, so that no 64-bit address is formed per lane and per load.  The
// tensors read this way are smaller than 4 GiB (checked on the host).
typedef float floatx4 __attribute__((ext_vector_type(4), aligned(4)));
#define KFAC_GLOBAL_AS __attribute__((address_space(1)))
__device__ __forceinline__ float4 gload4(const float *base, unsigned byte_off) {
  const floatx4 t = *(const KFAC_GLOBAL_AS floatx4 *)((const KFAC_GLOBAL_AS char *)base + byte_off);
  return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ float gload1(const float *base, unsigned byte_off) {
  return *(const KFAC_GLOBAL_AS float *)((const KFAC_GLOBAL_AS char *)base + byte_off);
}

// Thread index inside a team of THREADS threads.  The workgroups of this engine
// have THREADS threads, except those of the macro-tile covariance kernel, whose
// four teams each stage and multiply like one such workgroup.
__device__ __forceinline__ int team_tid() { return (int)(threadIdx.x & (THREADS - 1)); }

// Two float32 numbers as three packed pairs of bfloat16 numbers (first number in the low
// half), a = hi + mid + lo exactly (inside the range below).  11 vector instructions: three v_cvt_pk_bf16_f32 (round
// to nearest even) and the two rests of either number.
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  const floatx2 t = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(t, bf16x2));
}
__device__ __forceinline__ void split_pair(float a, float b, unsigned &hi, unsigned &mid, unsigned &lo) {
  hi = pack_bf16(a, b);
  const float a1 = a - __uint_as_float(hi << 16), b1 = b - __uint_as_float(hi & 0xffff0000u);
  mid = pack_bf16(a1, b1);
  const float a2 = a1 - __uint_as_float(mid << 16), b2 = b1 - __uint_as_float(mid & 0xffff0000u);
  lo = pack_bf16(a2, b2);
}
// The six plane pairs of a product (0 = hi, 1 = mid, 2 = lo), the leading one last.
constexpr int kSplitTerms = 6;
constexpr int kSplitA[kSplitTerms] = {2, 0, 1, 1, 0, 0};
constexpr int kSplitB[kSplitTerms] = {0, 2, 1, 0, 1, 0};

// How a product is formed: kSplit as six bfloat16 products of split operands, kF32 by the
// float32 instruction.  A kF32 panel is row-major with a stride of 33 floats (loaders with k
// contiguous) or k-major with a stride of rows + 4 (LoaderKS); either gives operand reads
// without bank conflicts.  It fits the memory of a kSplit panel of as many rows.
enum Format { kF32, kSplit };

template <int ROWS, Format F>
struct Panel {
  static constexpr int kPlaneBytes = KT * 2;
  static constexpr int kRowBytes = 3 * kPlaneBytes + 16;
  static constexpr int kFloats = ROWS * kRowBytes / 4;
};
template <int ROWS>
struct Panel<ROWS, kF32> {
  static constexpr int kRowKStride = KT + 1;
  static constexpr int kKRowStride = ROWS + 4;
  static constexpr int kFloats = ROWS * kRowKStride > KT * kKRowStride ? ROWS * kRowKStride : KT * kKRowStride;
};
// Byte offset of 16-byte chunk `chunk` (k-values 8 chunk ..) of a row inside a plane of the row.
__device__ __forceinline__ int panel_chunk(int row, int chunk) { return ((chunk ^ (row >> 4)) & 3) * 16; }

// Range of the split.  Below 2^-110 the lowest bit of a float32 number is less than the least
// bfloat16 number, and the planes hold fewer than 24 bits; from 0x1.ffp127 on hi rounds to infinity,
// and the rests of an infinity are NaN.  Threads note the least nonzero magnitude that they split
// (twice the bits without the sign, minus one: zero becomes the largest), and the main loop repeats a
// tile with the float32 instruction if that is below 2^-110 or a sum came out as infinity or NaN, as
// it does wherever an operand above the range takes part.
constexpr unsigned kNothingSplit = 0xffffffffu;
constexpr unsigned kLeastSplit = (17u << 24) - 1u;   // of 2^-110
__device__ __forceinline__ void note_least(float a, float b, unsigned &least) {
  const unsigned ka = (__float_as_uint(a) << 1) - 1u, kb = (__float_as_uint(b) << 1) - 1u;
  least = min(least, min(ka, kb));
}

// Store the planes of two or four consecutive k-values at their place in a row.
__device__ __forceinline__ void panel_store2(char *p, float a, float b, unsigned &least) {
  unsigned h, m, l;
  note_least(a, b, least);
  split_pair(a, b, h, m, l);
  *reinterpret_cast<unsigned *>(p) = h;
  *reinterpret_cast<unsigned *>(p + KT * 2) = m;
  *reinterpret_cast<unsigned *>(p + KT * 4) = l;
}
__device__ __forceinline__ void panel_store4(char *p, float a, float b, float c, float d, unsigned &least) {
  unsigned h0, m0, l0, h1, m1, l1;
  note_least(a, b, least);
  note_least(c, d, least);
  split_pair(a, b, h0, m0, l0);
  split_pair(c, d, h1, m1, l1);
  *reinterpret_cast<uintx2 *>(p) = uintx2{h0, h1};
  *reinterpret_cast<uintx2 *>(p + KT * 2) = uintx2{m0, m1};
  *reinterpret_cast<uintx2 *>(p + KT * 4) = uintx2{l0, l1};
}

// E consecutive k-values t of panel row r0 + RPP i, the lane's part `pr` of the row's 32
// (the scalar loaders with k contiguous).
template <int ROWS, Format FMT, bool SUM, int RPP, int E>
__device__ __forceinline__ void store_row(float *lds, int r0, int pr, int i, const float (&t)[E], float *sum,
                                          unsigned &least) {
  if constexpr (FMT == kF32) {
    float *p = lds + (r0 + RPP * i) * Panel<ROWS, kF32>::kRowKStride + pr * E;
#pragma unroll
    for (int e = 0; e < E; ++e) p[e] = t[e];
  } else {
    static_assert(E == 2 && RPP == 16, "pairs of k-values, sixteen rows per pass");
    if (SUM) sum[i] += t[0] + t[1];
    char *p = reinterpret_cast<char *>(lds) + r0 * Panel<ROWS, kSplit>::kRowBytes + (pr & 3) * 4;
    panel_store2(p + 16 * i * Panel<ROWS, kSplit>::kRowBytes + panel_chunk(16 * i, pr >> 2), t[0], t[1], least);
  }
}

// Loader protocol: init() fixes the panel (first row) and precomputes what
// does not change along k (row offsets, row validity); load() issues the
// global loads of one panel; store() writes it to LDS.  Interior panels (all
// rows and all k valid: a workgroup-uniform test) take a path without any
// per-element selects; edge panels load from clamped (always valid) addresses
// and apply validity masks when storing.  Nothing between load() and store()
// touches the loaded registers, so the loads stay in flight while the matrix
// cores work on the previous panel.  Offsets are 32-bit element offsets from
// the tensor base (tensors hold fewer than 2^30 elements, 4 GiB; checked on the host).
// F is the format that a loader's thread layout is made for (two consecutive k-values per thread
// and row where the planes are written in pairs, one where float32 is written), FMT the one that
// store() writes: F, or kF32 from the layout of kSplit.
// With kSplit, store() notes the least magnitude it split; with SUM it also adds what it stores to the thread's row sums: slot i of `sum` belongs
// to panel row sum_row(i), and the kSumParts threads with sum_part() = 0 .. kSumParts - 1 hold
// the parts of a row (add_row_sums below).

// ---------------------------------------------------------------------------
// LoaderKC: element (row, kg) at base + (kg / L) * sample_stride
//                                     + row * row_stride + (kg % L)
// rows >= rows_valid read as 0.
// ---------------------------------------------------------------------------
// VEC: 16-byte loads of four consecutive k-values of a row; for tensors whose
// rows start on 16-byte boundaries (base, row and sample strides multiples of 4
// floats: misaligned 16-byte loads work but were measured slower than the
// scalar variant below).  A quad that is cut by the end of the range, or that
// runs from one sample into the next, is loaded element by element by the
// lanes concerned, so the reduction length is free.  A compile-time choice so
// that this common case carries no code or registers of the scalar variant.
// The primary template is this one.
template <int ROWS, bool VEC, Format F>
struct LoaderKC {
  static_assert(VEC, "the scalar variant is the specialisation below");
  static constexpr Format kFormat = F;
  static constexpr bool kKRow = false;
  static constexpr int NV = ROWS / 32;
  struct Regs {
    float4 v[NV];
    unsigned kmask;  // bit e: k-value e of this thread's quad is inside the range
    bool fast;       // interior panel: no masks needed
  };
  const float *base;
  unsigned sample_stride;
  unsigned row_stride;
  unsigned L;      // k-values per sample
  int rows_valid;
  // per-thread panel state
  unsigned rowoff[NV];
  unsigned rowvalid;  // bit i: row i of this thread is a data row
  bool full_rows;

  __device__ __forceinline__ void init(float *, int row0) {
    const int rr = team_tid() >> 3;
    rowvalid = 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int row = row0 + rr + 32 * i;
      const bool ok = row < rows_valid;
      rowoff[i] = (ok ? (unsigned)row : 0u) * row_stride;
      if (ok) rowvalid |= 1u << i;
    }
    full_rows = row0 + ROWS <= rows_valid;
  }

  __device__ __forceinline__ void load(Regs &r, int, long long k0, long long k_end) const {
    const unsigned kq = (team_tid() & 7) * 4;
    const long long kgl = k0 + kq;
    const bool full_k = k0 + KT <= k_end;
    r.fast = full_rows && full_k;
    const bool whole = full_k || kgl + 3 < k_end;
    const long long left = k_end - kgl;   // valid k-values from kg on
    r.kmask = whole ? 0xfu : (left > 0 ? (1u << (int)left) - 1u : 0u);
    const unsigned kc = left > 0 ? (unsigned)kgl : 0u;
    unsigned koff = kc, rem = kc;
    if (L < (unsigned)k_end) {  // more than one sample
      const unsigned s = kc / L;
      rem = kc - s * L;
      koff = s * sample_stride + rem;
    }
    if (whole && rem + 3 < L) {
#pragma unroll
      for (int i = 0; i < NV; ++i) r.v[i] = gload4(base, (koff + rowoff[i]) * 4u);
    } else {
      // element by element: k-values past the range read k = 0 of the row (masked when
      // stored), k-values past the end of the sample continue in the next sample
      unsigned off[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = (r.kmask >> e) & 1u;
        off[e] = in ? koff + e + (rem + e >= L ? sample_stride - L : 0u) : 0u;
      }
#pragma unroll
      for (int i = 0; i < NV; ++i)
        r.v[i] = make_float4(gload1(base, (off[0] + rowoff[i]) * 4u), gload1(base, (off[1] + rowoff[i]) * 4u),
                             gload1(base, (off[2] + rowoff[i]) * 4u), gload1(base, (off[3] + rowoff[i]) * 4u));
    }
  }

  static constexpr int kSumSlots = NV, kSumParts = 8;
  __device__ __forceinline__ static int sum_row(int i) { return (team_tid() >> 3) + 32 * i; }
  __device__ __forceinline__ static int sum_part() { return team_tid() & 7; }

  template <Format FMT, bool SUM>
  __device__ __forceinline__ void store(const Regs &r, float *lds, float *sum, unsigned &least) const {
    const int rr = team_tid() >> 3;
    if constexpr (FMT == kF32) {
      float *q = lds + rr * Panel<ROWS, kF32>::kRowKStride + (team_tid() & 7) * 4;
      if (r.fast) {
#pragma unroll
        for (int i = 0; i < NV; ++i, q += 32 * Panel<ROWS, kF32>::kRowKStride) {
          q[0] = r.v[i].x;
          q[1] = r.v[i].y;
          q[2] = r.v[i].z;
          q[3] = r.v[i].w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < NV; ++i, q += 32 * Panel<ROWS, kF32>::kRowKStride) {
          const float t[4] = {r.v[i].x, r.v[i].y, r.v[i].z, r.v[i].w};
          const bool rv = (rowvalid >> i) & 1u;
#pragma unroll
          for (int e = 0; e < 4; ++e) q[e] = (((r.kmask >> e) & 1u) && rv) ? t[e] : 0.f;
        }
      }
      return;
    }
    char *p = reinterpret_cast<char *>(lds) + rr * Panel<ROWS, kSplit>::kRowBytes + (team_tid() & 1) * 8;
    const int chunk = panel_chunk(rr, (team_tid() & 7) >> 1);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float t[4] = {r.v[i].x, r.v[i].y, r.v[i].z, r.v[i].w};
      if (!r.fast) {
        const bool rv = (rowvalid >> i) & 1u;
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = (rv && ((r.kmask >> e) & 1u)) ? t[e] : 0.f;
      }
      if (SUM) sum[i] += (t[0] + t[1]) + (t[2] + t[3]);
      // rows 32 apart: the chunk index differs in bit 1
      panel_store4(p + 32 * i * Panel<ROWS, kSplit>::kRowBytes + ((i & 1) ? chunk ^ 32 : chunk), t[0], t[1], t[2], t[3],
                   least);
    }
  }
};

// Scalar variant: dword loads, a thread takes E consecutive k-values of a row and
// KT / E lanes the 32 of a panel.  It is the one that can subsample (line_len > 0).
template <int ROWS, Format F>
struct LoaderKC<ROWS, false, F> {
  static constexpr Format kFormat = F;
  static constexpr bool kKRow = false;
  static constexpr int E = F == kSplit ? 2 : 1;
  static constexpr int LPR = KT / E;          // lanes per row
  static constexpr int RPP = THREADS / LPR;   // rows per pass
  static constexpr int NR = ROWS / RPP;       // rows per thread
  struct Regs {
    float v[NR][E];
    bool kvalid[E];   // k-value e of this thread is inside the range
  };
  const float *base;
  unsigned sample_stride;
  unsigned row_stride;
  unsigned L;      // k-values per sample
  int rows_valid;
  // Subsampled rows (a strided 1x1 convolution reads every sx-th pixel of every
  // sy-th image line): k-value p of a sample is pixel (p / line_len) *
  // line_stride + (p % line_len) * px_stride of the row.  line_len = 0: k-values
  // are consecutive elements.
  unsigned line_len = 0, line_stride = 0, px_stride = 1;
  // per-thread panel state: row i of the thread is first_row + RPP i; rows past
  // the end load from the last data row (masked when stored)
  int first_row;
  unsigned last_off;

  __device__ __forceinline__ void init(float *, int row0) {
    first_row = row0 + team_tid() / LPR;
    last_off = (unsigned)(rows_valid > 0 ? rows_valid - 1 : 0) * row_stride;
  }

  __device__ __forceinline__ void load(Regs &r, int, long long k0, long long k_end) const {
    const long long kg = k0 + team_tid() % LPR * E;
    unsigned koff[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      r.kvalid[e] = kg + e < k_end;
      const unsigned kc = r.kvalid[e] ? (unsigned)kg + e : 0u;
      koff[e] = kc;
      if (L < (unsigned)k_end || line_len) {  // more than one sample, or subsampled rows
        const unsigned s = kc / L;
        unsigned pix = kc - s * L;
        if (line_len) {
          const unsigned line = pix / line_len;
          pix = line * line_stride + (pix - line * line_len) * px_stride;
        }
        koff[e] = s * sample_stride + pix;
      }
    }
    // The row offsets are cheap to recompute and expensive to keep: hide the
    // row from the optimiser so that it does not hoist NR offsets per operand
    // out of the k loop (which spills under a 3-workgroup register budget).
    int fr = first_row;
    asm volatile("" : "+v"(fr));
    const unsigned off0 = (unsigned)fr * row_stride;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const unsigned off = off0 + (unsigned)(RPP * i) * row_stride;
      const unsigned ro = off < last_off ? off : last_off;
#pragma unroll
      for (int e = 0; e < E; ++e) r.v[i][e] = gload1(base, (koff[e] + ro) * 4u);
    }
  }

  static constexpr int kSumSlots = NR, kSumParts = LPR;
  __device__ __forceinline__ static int sum_row(int i) { return team_tid() / LPR + RPP * i; }
  __device__ __forceinline__ static int sum_part() { return team_tid() % LPR; }

  template <Format FMT, bool SUM>
  __device__ __forceinline__ void store(const Regs &r, float *lds, float *sum, unsigned &least) const {
    const int pr = team_tid() % LPR;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const bool rv = first_row + RPP * i < rows_valid;
      float t[E];
#pragma unroll
      for (int e = 0; e < E; ++e) t[e] = (r.kvalid[e] && rv) ? r.v[i][e] : 0.f;
      store_row<ROWS, FMT, SUM, RPP>(lds, team_tid() / LPR, pr, i, t, sum, least);
    }
  }
};

// ---------------------------------------------------------------------------
// LoaderKS: element (row, kg) at base + kg * ld + row for row < rows_valid;
// with EXTRA row == rows_valid reads extra[kg], unless that is null.
// ---------------------------------------------------------------------------
template <int ROWS, bool VEC, Format F, bool EXTRA = false>
struct LoaderKS {
  static constexpr Format kFormat = F;
  static constexpr bool kKRow = true;
  static constexpr int RQ = ROWS / 4;          // row quads per k
  static constexpr int KPP = THREADS / RQ;     // threads per row quad
  static constexpr int NV = KT / KPP;          // k-values of a thread: 4 or 2
  struct Regs {
    float4 v[NV];
    unsigned kmask;  // bit i: k-value i of this thread is inside the range
    bool fast;
  };
  const float *base;
  const float *extra;
  unsigned ld;
  int rows_valid;
  // per-thread panel state
  int row;          // first of this thread's four rows
  bool quad_ok;     // all four rows are data rows and float4 loads are allowed
  bool full_rows;

  __device__ __forceinline__ void init(float *, int row0) {
    row = row0 + (team_tid() % RQ) * 4;
    quad_ok = VEC && row + 3 < rows_valid;
    full_rows = VEC && row0 + ROWS <= rows_valid;
  }

  __device__ __forceinline__ bool is_row(int r) const { return r < rows_valid || (EXTRA && r == rows_valid && extra); }

  // k-value i of this thread in a panel: consecutive ones, or KPP apart where rows are stored whole
  __device__ __forceinline__ static int k_of(int i) {
    return F == kSplit ? team_tid() / RQ * NV + i : team_tid() / RQ + KPP * i;
  }

  __device__ __forceinline__ void load(Regs &r, int, long long k0, long long k_end) const {
    const bool full_k = k0 + KT <= k_end;
    r.fast = full_rows && full_k;
    r.kmask = 0;
    if (quad_ok) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const long long kg = k0 + k_of(i);
        const bool kok = full_k || kg < k_end;
        if (kok) r.kmask |= 1u << i;
        r.v[i] = gload4(base, ((unsigned)(kok ? kg : 0) * ld + (unsigned)row) * 4u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const long long kg = k0 + k_of(i);
        const bool kok = kg < k_end;
        if (kok) r.kmask |= 1u << i;
        const unsigned kc = (unsigned)(kok ? kg : 0);
        float t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int re = row + e;
          const unsigned at = kc * ld + (unsigned)(re < rows_valid ? re : 0);
          if constexpr (EXTRA)
            t[e] = *(re == rows_valid && extra ? extra + kc : base + at);
          else
            t[e] = gload1(base, at * 4u);
        }
        r.v[i] = make_float4(t[0], t[1], t[2], t[3]);
      }
    }
  }

  static constexpr int kSumSlots = 4, kSumParts = KPP;
  __device__ __forceinline__ static int sum_row(int i) { return (team_tid() % RQ) * 4 + i; }
  __device__ __forceinline__ static int sum_part() { return team_tid() / RQ; }

  template <Format FMT, bool SUM>
  __device__ __forceinline__ void store(const Regs &r, float *lds, float *sum, unsigned &least) const {
    const int rq = team_tid() % RQ;
    if constexpr (FMT == kF32) {
      float *q = lds + rq * 4;
      if (r.fast) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
          *reinterpret_cast<float4 *>(q + k_of(i) * Panel<ROWS, kF32>::kKRowStride) = r.v[i];
      } else {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const float t[4] = {r.v[i].x, r.v[i].y, r.v[i].z, r.v[i].w};
          const bool kv = (r.kmask >> i) & 1u;
          float o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = kv && is_row(row + e) ? t[e] : 0.f;
          *reinterpret_cast<float4 *>(q + k_of(i) * Panel<ROWS, kF32>::kKRowStride) = make_float4(o[0], o[1], o[2], o[3]);
        }
      }
      return;
    }
    const int kk = k_of(0);
    char *p = reinterpret_cast<char *>(lds) + rq * 4 * Panel<ROWS, kSplit>::kRowBytes +
              panel_chunk(rq * 4, kk >> 3) + (kk & 7) * 2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int re = row + e;
      float t[NV];
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        t[i] = e == 0 ? r.v[i].x : e == 1 ? r.v[i].y : e == 2 ? r.v[i].z : r.v[i].w;
        if (!r.fast) {
          t[i] = ((r.kmask >> i) & 1u) && is_row(re) ? t[i] : 0.f;
        }
        if (SUM) sum[e] += t[i];
      }
      if (NV == 4)
        panel_store4(p + e * Panel<ROWS, kSplit>::kRowBytes, t[0], t[1], t[NV - 2], t[NV - 1], least);
      else
        panel_store2(p + e * Panel<ROWS, kSplit>::kRowBytes, t[0], t[1], least);
    }
  }
};

// ---------------------------------------------------------------------------
// LoaderIM: implicit im2col over an NCHW tensor.
//   row = (c * kh + i) * kw + j  for row < d_patch (rows past it read as 0);
//   kg = (sample * ho + oy) * wo + ox.
// ---------------------------------------------------------------------------
template <int ROWS, Format F>
struct LoaderIM {
  static constexpr Format kFormat = F;
  static constexpr bool kKRow = false;
  static constexpr int E = F == kSplit ? 2 : 1;   // consecutive k-values of a thread
  static constexpr int LPR = KT / E;              // lanes per row
  static constexpr int RPP = THREADS / LPR;       // rows per pass
  static constexpr int NV = ROWS / RPP;
  struct Regs {
    float v[NV][E];
    unsigned use;   // bit E i + e: value e of row i lies inside the image
  };
  const float *base;
  int C, H, W, kh, kw, sy, sx, ph, pw, ho, wo;
  int d_patch;
  int2 *table;  // LDS, ROWS entries: {offset inside a sample, (i << 16) | j}; y = -1: row past the end

  // Build the per-row table for panel rows [row0, row0 + ROWS).
  __device__ __forceinline__ void init(float *lds_table, int row0) {
    table = reinterpret_cast<int2 *>(lds_table);
    for (int t = team_tid(); t < ROWS; t += THREADS) {
      const int row = row0 + t;
      int2 e;
      if (row < d_patch) {
        const int c = row / (kh * kw);
        const int rem = row - c * (kh * kw);
        const int i = rem / kw;
        const int j = rem - i * kw;
        e.x = (c * H + i) * W + j;
        e.y = (i << 16) | j;
      } else {
        e.x = 0;
        e.y = -1;
      }
      table[t] = e;
    }
  }

  // k-value kg of the reduction: its patch's corner in the image, and the corner's offset from base
  struct Corner {
    bool kok;
    int iy, ix;
    long long idx;
  };
  __device__ __forceinline__ Corner corner(long long kg, long long k_end) const {
    Corner o;
    o.kok = kg < k_end;
    const unsigned kc = o.kok ? (unsigned)kg : 0u;
    const unsigned howo = (unsigned)(ho * wo);
    const unsigned s = kc / howo;
    const unsigned rem = kc - s * howo;
    const int oy = (int)(rem / (unsigned)wo);
    const int ox = (int)rem - oy * wo;
    o.iy = oy * sy - ph;
    o.ix = ox * sx - pw;
    o.idx = ((long long)s * C * H + o.iy) * (long long)W + o.ix;
    return o;
  }

  __device__ __forceinline__ void load(Regs &r, int, long long k0, long long k_end) const {
    const long long kg = k0 + team_tid() % LPR * E;
    r.use = 0;
    if constexpr (E == 1) {
      // (without the arrays of the pair below, which cost this variant 2 .. 8 %)
      const Corner o = corner(kg, k_end);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int2 t = table[team_tid() / LPR + RPP * i];
        const int iy = o.iy + (t.y >> 16);
        const int ix = o.ix + (t.y & 0xffff);
        const bool ok = o.kok && t.y >= 0 && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
        r.v[i][0] = base[ok ? o.idx + t.x : 0];
        if (ok) r.use |= 1u << i;
      }
      return;
    }
    Corner o[E];
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = corner(kg + e, k_end);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int2 t = table[team_tid() / LPR + RPP * i];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int iy = o[e].iy + (t.y >> 16);
        const int ix = o[e].ix + (t.y & 0xffff);
        const bool ok = o[e].kok && t.y >= 0 && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
        r.v[i][e] = base[ok ? o[e].idx + t.x : 0];
        if (ok) r.use |= 1u << (E * i + e);
      }
    }
  }

  static constexpr int kSumSlots = NV, kSumParts = LPR;
  __device__ __forceinline__ static int sum_row(int i) { return team_tid() / LPR + RPP * i; }
  __device__ __forceinline__ static int sum_part() { return team_tid() % LPR; }

  template <Format FMT, bool SUM>
  __device__ __forceinline__ void store(const Regs &r, float *lds, float *sum, unsigned &least) const {
    const int pr = team_tid() % LPR;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float t[E];
#pragma unroll
      for (int e = 0; e < E; ++e) t[e] = ((r.use >> (E * i + e)) & 1u) ? r.v[i][e] : 0.f;
      store_row<ROWS, FMT, SUM, RPP>(lds, team_tid() / LPR, pr, i, t, sum, least);
    }
  }
};

template <int WM, int WN>
__device__ __forceinline__ void zero_acc(floatx16 (&acc)[WM][WN]) {
#pragma unroll
  for (int im = 0; im < WM; ++im)
#pragma unroll
    for (int in = 0; in < WN; ++in)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[im][in][v] = 0.f;
}

// Operand of v_mfma_f32_32x32x2_f32 from a kF32 panel: lane l supplies element (row = l % 32, k = l / 32).
template <int ROWS, bool KROW>
__device__ __forceinline__ float fetch(const float *lds, int row, int k) {
  return KROW ? lds[k * Panel<ROWS, kF32>::kKRowStride + row] : lds[row * Panel<ROWS, kF32>::kRowKStride + k];
}

// The MFMAs of one kF32 panel.  With RS the lane also sums the A operand values it feeds to the
// matrix cores: rs[im] ends as the sum over this lane's k-values (k = lane / 32 mod 2) of row
// (wave_m * WM + im) * 32 + lane % 32, i.e. half of that row's sum.
template <int WM, int WN, bool KROWA, bool KROWB, unsigned MASK = 0xffffffffu>
__device__ __forceinline__ void mma_panel_f32(const float *pa, const float *pb, int wm, int wn,
                                              floatx16 (&acc)[WM][WN], bool RS, float *rs) {
  const int lane = threadIdx.x & 63;
  const int lrow = lane & 31, lk = lane >> 5;
#pragma unroll
  for (int kk = 0; kk < KT / 2; ++kk) {
    float a[WM], b[WN];
#pragma unroll
    for (int im = 0; im < WM; ++im) a[im] = fetch<64 * WM, KROWA>(pa, (wm * WM + im) * 32 + lrow, 2 * kk + lk);
    if (RS) {
#pragma unroll
      for (int im = 0; im < WM; ++im) rs[im] += a[im];
    }
#pragma unroll
    for (int in = 0; in < WN; ++in) b[in] = fetch<64 * WN, KROWB>(pb, (wn * WN + in) * 32 + lrow, 2 * kk + lk);
#pragma unroll
    for (int im = 0; im < WM; ++im)
#pragma unroll
      for (int in = 0; in < WN; ++in)
        if (MASK & (1u << (im * WN + in)))
          acc[im][in] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[im], b[in], acc[im][in], 0, 0, 0);
  }
}

// The MFMAs of one kSplit panel: this wave's WM x WN blocks from the LDS panels pa and pb (the same
// array for the diagonal tile of a SYRK), 6 per block and 16 k-values.  Lane l supplies row
// l % 32 and k-values 8 (l / 32) .. + 7 of a 16-k step.  hi * hi goes to acc, the other five to low.
// MASK: bit im * WN + in set = this wave computes block (im, in) (compile time, so that a wave
// that owns fewer blocks carries no test per MFMA).
template <int WM, int WN, unsigned MASK = 0xffffffffu>
__device__ __forceinline__ void mma_panel(const float *pa, const float *pb, int wm, int wn,
                                          floatx16 (&acc)[WM][WN], floatx16 (&low)[WM][WN]) {
  constexpr int RB = Panel<64, kSplit>::kRowBytes;
  const int lane = threadIdx.x & 63;
  const int lrow = lane & 31, lk = lane >> 5;
  // 32-row block b keeps chunk c of its lower / upper 16 rows at c ^ (2 b) / c ^ (2 b + 1) (mod 4)
  const int lane_off = lrow * RB + ((lk ^ (lrow >> 4)) & 1) * 16;
  const char *a0 = reinterpret_cast<const char *>(pa) + wm * WM * 32 * RB + lane_off;
  const char *b0 = reinterpret_cast<const char *>(pb) + wn * WN * 32 * RB + lane_off;
  const int pm = WM == 1 ? (wm & 1) * 32 : 0, pn = WN == 1 ? (wn & 1) * 32 : 0;
#pragma unroll
  for (int s = 0; s < KT / 16; ++s) {
    bf16x8 fa[WM][3], fb[WN][3];
#pragma unroll
    for (int im = 0; im < WM; ++im) {
      const char *p = a0 + im * 32 * RB + ((((s ^ im) & 1) * 32) ^ pm);
#pragma unroll
      for (int q = 0; q < 3; ++q) fa[im][q] = *reinterpret_cast<const bf16x8 *>(p + q * (KT * 2));
    }
#pragma unroll
    for (int in = 0; in < WN; ++in) {
      const char *p = b0 + in * 32 * RB + ((((s ^ in) & 1) * 32) ^ pn);
#pragma unroll
      for (int q = 0; q < 3; ++q) fb[in][q] = *reinterpret_cast<const bf16x8 *>(p + q * (KT * 2));
    }
#pragma unroll
    for (int t = 0; t < kSplitTerms; ++t)
#pragma unroll
      for (int im = 0; im < WM; ++im)
#pragma unroll
        for (int in = 0; in < WN; ++in)
          if (MASK & (1u << (im * WN + in))) {
            floatx16 &sum = t == kSplitTerms - 1 ? acc[im][in] : low[im][in];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[im][kSplitA[t]], fb[in][kSplitB[t]], sum, 0, 0, 0);
          }
  }
}

// The row sums of a panel from the parts that its threads added up while storing it (SUM in the
// loaders), in a fixed order: the sum of panel row t in the team's thread t < ROWS.  `lds`: a
// panel's memory of this team, free to overwrite.  Every thread of the workgroup calls it.
template <int ROWS, class Loader>
__device__ __forceinline__ float add_row_sums(const float *sum, float *lds) {
  static_assert(Loader::kSumParts * ROWS <= Panel<ROWS, kSplit>::kFloats, "the parts must fit a panel");
  __syncthreads();
#pragma unroll
  for (int i = 0; i < Loader::kSumSlots; ++i) lds[Loader::sum_part() * ROWS + Loader::sum_row(i)] = sum[i];
  __syncthreads();
  float total = 0.f;
  if (team_tid() < ROWS) {
#pragma unroll
    for (int p = 0; p < Loader::kSumParts; ++p) total += lds[p * ROWS + team_tid()];
  }
  __syncthreads();
  return total;
}

// Whether `mine` holds in any thread of the workgroup (of THREADS threads, all of which call it, once).
__device__ __forceinline__ bool any_in_workgroup(bool mine) {
  __shared__ int flag[THREADS / 64];
  const bool any = __any(mine);
  if ((threadIdx.x & 63) == 0) flag[threadIdx.x >> 6] = any;
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(flag[0] | flag[1] | flag[2] | flag[3]) != 0;
}

// Main loop of the float32 instruction.  acc[im][in] accumulates the 32x32 block at rows
// (wave_m * WM + im) * 32 of the A panel and (wave_n * WN + in) * 32 of the B
// panel.  With SAME the B operand is read from the A panel (diagonal tile of a
// SYRK) and lb is not used.  ldsA / ldsB hold Panel<64*WM> / Panel<64*WN>
// floats.
// With RS rs[im] ends as half of a row's sum (mma_panel_f32).
// A wave with `active` false stages panels like the others but feeds nothing to
// the matrix cores (its block of the tile is not needed: above the diagonal of a
// symmetric product, or past the end of the matrix); its accumulators stay as
// they are.
template <int WM, int WN, bool SAME, bool RS, class LA, class LB, unsigned MASK = 0xffffffffu>
__device__ __forceinline__ void mainloop_f32(const LA &la, const LB &lb, int rowA0, int rowB0,
                                             long long kbeg, long long kend, float *ldsA, float *ldsB,
                                             floatx16 (&acc)[WM][WN], float *rs, bool active,
                                             int wave = threadIdx.x >> 6) {
  const int wm = wave >> 1, wn = wave & 1;
  unsigned unused = kNothingSplit;
  typename LA::Regs ra;
  typename LB::Regs rb;
  if (kbeg < kend) {
    la.load(ra, rowA0, kbeg, kend);
    if (!SAME) lb.load(rb, rowB0, kbeg, kend);
  }
  for (long long k0 = kbeg; k0 < kend; k0 += KT) {
    la.template store<kF32, false>(ra, ldsA, nullptr, unused);
    if (!SAME) lb.template store<kF32, false>(rb, ldsB, nullptr, unused);
    __syncthreads();
    if (k0 + KT < kend) {
      la.load(ra, rowA0, k0 + KT, kend);
      if (!SAME) lb.load(rb, rowB0, k0 + KT, kend);
    }
    if (active)
      mma_panel_f32<WM, WN, LA::kKRow, SAME ? LA::kKRow : LB::kKRow, MASK>(ldsA, SAME ? ldsA : ldsB, wm, wn, acc, RS,
                                                                          rs);
    __syncthreads();
  }
}

// Main loop of split products, arguments as above; acc comes as zeros.  With RS the sums over k of the
// A operand's rows are formed on the side, from the float32 values: *rowsum is that of row threadIdx.x
// of the tile (threads below 64*WM).
template <int WM, int WN, bool SAME, bool RS, class LA, class LB, unsigned MASK = 0xffffffffu>
__device__ __forceinline__ void mainloop_impl(const LA &la, const LB &lb, int rowA0, int rowB0,
                                              long long kbeg, long long kend, float *ldsA,
                                              float *ldsB, floatx16 (&acc)[WM][WN], float *rowsum,
                                              bool active = true, int wave = threadIdx.x >> 6) {
  const int wm = wave >> 1, wn = wave & 1;
  typename LA::Regs ra;
  typename LB::Regs rb;
  float sum[LA::kSumSlots];
#pragma unroll
  for (int i = 0; i < LA::kSumSlots; ++i) sum[i] = 0.f;
  unsigned least = kNothingSplit;
  floatx16 low[WM][WN];
  zero_acc<WM, WN>(low);
  if (kbeg < kend) {
    la.load(ra, rowA0, kbeg, kend);
    if (!SAME) lb.load(rb, rowB0, kbeg, kend);
  }
  for (long long k0 = kbeg; k0 < kend; k0 += KT) {
    la.template store<kSplit, RS>(ra, ldsA, sum, least);
    if (!SAME) lb.template store<kSplit, false>(rb, ldsB, nullptr, least);
    __syncthreads();
    if (k0 + KT < kend) {
      la.load(ra, rowA0, k0 + KT, kend);
      if (!SAME) lb.load(rb, rowB0, k0 + KT, kend);
    }
    if (active) mma_panel<WM, WN, MASK>(ldsA, SAME ? ldsA : ldsB, wm, wn, acc, low);
    __syncthreads();
  }
  float nonfinite = 0.f;   // NaN as soon as a sum is infinite or NaN
#pragma unroll
  for (int im = 0; im < WM; ++im)
#pragma unroll
    for (int in = 0; in < WN; ++in) {
      acc[im][in] += low[im][in];
#pragma unroll
      for (int v = 0; v < 16; ++v) nonfinite = __builtin_fmaf(acc[im][in][v], 0.f, nonfinite);
    }
  if (RS) *rowsum = add_row_sums<64 * WM, LA>(sum, ldsA);
  if (__builtin_expect(any_in_workgroup(least < kLeastSplit || nonfinite != 0.f), 0)) {
    zero_acc<WM, WN>(acc);
    mainloop_f32<WM, WN, SAME, false, LA, LB, MASK>(la, lb, rowA0, rowB0, kbeg, kend, ldsA, ldsB, acc, nullptr, active,
                                                    wave);
  }
}

template <int WM, int WN, bool SAME, class LA, class LB>
__device__ __forceinline__ void mainloop(const LA &la, const LB &lb, int rowA0, int rowB0,
                                         long long kbeg, long long kend, float *ldsA,
                                         float *ldsB, floatx16 (&acc)[WM][WN], bool active = true,
                                         int wave = threadIdx.x >> 6) {
  mainloop_impl<WM, WN, SAME, false>(la, lb, rowA0, rowB0, kbeg, kend, ldsA, ldsB, acc, nullptr,
                                     active, wave);
}

template <int WM, int WN, bool SAME, class LA, class LB>
__device__ __forceinline__ void mainloop_rowsum(const LA &la, const LB &lb, int rowA0, int rowB0,
                                                long long kbeg, long long kend, float *ldsA,
                                                float *ldsB, floatx16 (&acc)[WM][WN],
                                                float &rowsum, bool active = true,
                                                int wave = threadIdx.x >> 6) {
  mainloop_impl<WM, WN, SAME, true>(la, lb, rowA0, rowB0, kbeg, kend, ldsA, ldsB, acc, &rowsum, active,
                                    wave);
}

// Whether this wave's block of a symmetric product's tile (first rows row0A /
// row0B, dt rows in all) is needed: it is not when it lies entirely above the
// diagonal (the epilogues take those entries from the mirrored block) or past
// the end of the matrix.
template <int WM>
__device__ __forceinline__ bool syrk_wave_active(int row0A, int row0B, int dt,
                                                 int wave = threadIdx.x >> 6) {
  const int ra = row0A + (wave >> 1) * WM * 32, rb = row0B + (wave & 1) * WM * 32;
  return ra + WM * 32 > rb && ra < dt && rb < dt;
}

// The diagonal 128-tile of a symmetric product needs 10 of its 16 blocks of 32 x
// 32 (the lower triangle).  Dealt by 64 x 64 quadrant, three waves compute four
// blocks each (two of them above the diagonal) and the fourth wave nothing; here
// the wave of the unused quadrant takes over the lower block row of quadrant
// (1, 0) and the diagonal quadrants skip their upper block: 3, 2, 2 and 3 blocks,
// three quarters of the time.
//   role     the wave index (2 x 2 layout) whose accumulator coordinates this wave uses
//   compute  bit im * 2 + in: block (im, in) is multiplied out
//   store    bit im * 2 + in: block (im, in) is this wave's to write (a block that
//            is not computed but stored holds zeros)
struct DiagRole {
  int role;
  unsigned compute, store;
};
__device__ __forceinline__ DiagRole diag_tile_role(int wave) {
  switch (wave) {
    case 0: return DiagRole{0, 0xdu, 0xfu};    // quadrant (0,0): blocks (0,0) (1,0) (1,1)
    case 3: return DiagRole{3, 0xdu, 0xfu};    // quadrant (1,1)
    case 2: return DiagRole{2, 0x3u, 0x3u};    // quadrant (1,0), upper block row
    default: return DiagRole{2, 0xcu, 0xcu};   // the wave of quadrant (0,1): quadrant (1,0), lower block row
  }
}

// Visit every accumulator element of this lane: f(row, col, value) with row /
// col relative to the workgroup tile.
template <int WM, int WN, class F>
__device__ __forceinline__ void for_each_acc(floatx16 (&acc)[WM][WN], F f,
                                             int wave = threadIdx.x >> 6) {
  const int lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
#pragma unroll
  for (int im = 0; im < WM; ++im)
#pragma unroll
    for (int in = 0; in < WN; ++in)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = (wm * WM + im) * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const int col = (wn * WN + in) * 32 + (lane & 31);
        f(row, col, acc[im][in][v]);
      }
}

// for_each_acc over the blocks whose bit (im * WN + in) is set in `mask`
template <int WM, int WN, class F>
__device__ __forceinline__ void for_each_acc_masked(floatx16 (&acc)[WM][WN], unsigned mask, F f, int wave) {
  const int lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
#pragma unroll
  for (int im = 0; im < WM; ++im)
#pragma unroll
    for (int in = 0; in < WN; ++in) {
      if (!(mask & (1u << (im * WN + in)))) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = (wm * WM + im) * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const int col = (wn * WN + in) * 32 + (lane & 31);
        f(row, col, acc[im][in][v]);
      }
    }
}

// Writes the finished tile: C[I,J] = alpha*acc + beta*C[I,J] and its mirror
// image C[J,I], 64x64 quadrant by quadrant through an LDS transpose so that
// every global access is a contiguous row segment.  Only entries on or below
// the diagonal of C are taken from the accumulators: a quadrant above the
// diagonal of a diagonal tile is skipped (it is the mirror of the one below),
// and a quadrant on the diagonal writes its upper triangle from its lower one.
// Rows and columns below dt (the tiled part); d is the leading dimension of C.
// `store`: the blocks of this wave's 2 x 2 that are its to write (see DiagRole).
template <int WM>
__device__ __forceinline__ void write_tile(floatx16 (&acc)[WM][WM], float *lds, int I, int J,
                                           int dt, int d, float alpha, float beta,
                                           float *__restrict__ C, int wave = threadIdx.x >> 6,
                                           unsigned store = 0xffffffffu) {
  constexpr int BM = 64 * WM;
  float(*t)[65] = reinterpret_cast<float(*)[65]>(lds);
  const int lc = threadIdx.x & 63, lr0 = threadIdx.x >> 6;
  for (int q = 0; q < WM * WM; ++q) {
    const int qm = q / WM, qn = q % WM;
    if (I == J && qm < qn) continue;
    const bool diag = I == J && qm == qn;
    __syncthreads();
    for_each_acc_masked<WM, WM>(acc, store, [&](int r, int c, float v) {
      if (r / 64 == qm && c / 64 == qn) t[r % 64][c % 64] = v;
    }, wave);
    __syncthreads();
    const int r0 = I * BM + qm * 64, c0 = J * BM + qn * 64;
#pragma unroll 4
    for (int p = 0; p < 16; ++p) {
      const int lr = lr0 + 4 * p;
      const int r = r0 + lr, c = c0 + lc;
      float v = alpha * t[lr][lc];
      const bool ok = r < dt && c < dt && (!diag || lc <= lr);
      if (ok) {
        if (beta != 0.f) v += beta * C[(long long)r * d + c];
        C[(long long)r * d + c] = v;
      }
      if (beta != 0.f) t[lr][lc] = v;   // the mirror gets the same value
    }
    if (beta != 0.f) __syncthreads();
#pragma unroll 4
    for (int p = 0; p < 16; ++p) {
      const int lr = lr0 + 4 * p;
      const float v = (beta != 0.f) ? t[lc][lr] : alpha * t[lc][lr];
      if (diag) {
        const int r = r0 + lr, c = c0 + lc;     // upper triangle of the quadrant itself
        if (lc > lr && r < dt && c < dt) C[(long long)r * d + c] = v;
      } else {
        const int mr = c0 + lr, mc = r0 + lc;   // row of the mirrored quadrant = column here
        if (mr < dt && mc < dt) C[(long long)mr * d + mc] = v;
      }
    }
  }
}

}  // namespace mma
}  // namespace kfac
