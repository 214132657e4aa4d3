// Convolution products in fp32 accuracy on the bf16 matrix pipe.  Part of conv_igemm.hip
// (inside its namespace), which defines the argument block, the gather modes and the
// common end of a tile.

// Both operands are multiplied by 2^24 before they are split, the sums by 2^-48 after the K
// loop.  bf16 has float's exponents, so the third term of a value, 2^-17 of it and less, would
// fall below bf16's smallest normal number for values under 2^-109 and be lost; times
// 2^24 every float, down to the smallest subnormal, keeps all its bits in normal
// bf16 numbers.  The price is at the other end: operands from 2^103 and sums from 2^80 on are not
// finite in the accumulators and take the fp32 products below.
constexpr float kSplitScale = 0x1p24f;
constexpr float kSplitUnscale = 0x1p-48f;

// x * 2^24 = h + m + l in bf16 (round to nearest even at every step): 8 + 8 + 8 significand
// bits hold every bit of a float.  Two values at a time: each returned word holds the
// terms of a (low half) and b (high half).
__device__ __forceinline__ void split_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l) {
  a *= kSplitScale;
  b *= kSplitScale;
  const bf16x2 hv = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  h = __builtin_bit_cast(unsigned, hv);
  a -= __builtin_bit_cast(float, h << 16);
  b -= __builtin_bit_cast(float, h & 0xFFFF0000u);
  const bf16x2 mv = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  m = __builtin_bit_cast(unsigned, mv);
  a -= __builtin_bit_cast(float, m << 16);
  b -= __builtin_bit_cast(float, m & 0xFFFF0000u);
  const bf16x2 lv = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  l = __builtin_bit_cast(unsigned, lv);
}

__device__ __forceinline__ float bf16_value(unsigned bits) { return __builtin_bit_cast(float, bits << 16); }

// First term of a filter value whose terms cannot hold it: a NaN, which sends every sum it
// enters to the fp32 products.  The other two terms are the upper and the lower half of the value.
constexpr unsigned kNotSplit = 0x7FFFu;

// The filter value of packed terms, exactly.
__device__ __forceinline__ float filter_value(unsigned h, unsigned m, unsigned l) {
  const float sum = ((bf16_value(h) + bf16_value(m)) + bf16_value(l)) * (1.f / kSplitScale);
  return h == kNotSplit ? __builtin_bit_cast(float, m << 16 | l) : sum;
}

// The end of a tile.  `arrived`: an int of LDS that no wavefront needs any more after a barrier.
template <int BM, int BN, int TM, int TN>
__device__ __forceinline__ void finish_split_tile(const IgemmArgs& a, int slices, int kslice, int g, int mt,
                                                  int nt, int wm0, int wn0, acc16 (&acc)[TM][TN],
                                                  const float2* factors, int* arrived_lds,
                                                  const float* scale_ptr, const float* shift_ptr,
                                                  float* __restrict__ yout) {
  const int tid = threadIdx.x;
  const int l32 = tid & 31, lhi = (tid & 63) >> 5;
  constexpr int sub_index = 0;  // a Convolution is one sub-problem
#define MC_FACTORS(row) (factors + (row))
#define MC_ARRIVED arrived_lds
#define MC_SLICES slices
#define MC_AHEAD (TM * TN == 1 ? 4 : (TM * TN == 2 ? 2 : 1))
#define MC_PLAIN false
#include "igemm_finish.h"
}

// The products run on the bf16 matrix pipe, which multiplies sixteen times as many values per
// cycle as the fp32 one, without giving up fp32 accuracy: both operands are split
// into three bf16 terms (split_pair; the filters once, when they are packed, the bottom's
// values by the thread that brings them to LDS), every product of two terms is exact in
// fp32, and of the nine products of x = h + m + l with w = h' + m' + l' the six largest are
// summed (h h', h m', m h', m m', h l', l h'; the other three come to at most 2^-24 of the
// product, 2^-27.4 on the average of random operands.  Summing m l' and l m' as well costs 10 to
// 18 % of a launch; instead sums of a few products, which round too seldom to hide the
// difference, stay with the fp32 kernel, see short_sums).
// The sums run in fp32 accumulators: h h' in one or two, the five small ones in another, added
// once after the K loop, so the large accumulator rounds a few times per sixteen K rows
// where the fp32 instruction rounds eight: over one chain of additions the error against a
// 64-bit sum is 0.32 to 0.48 of the fp32 instruction's (512 -> 2048 on 64 x 7x7, five
// distributions of operands; all six products in one accumulator: up to 1.17 of it).  How many
// chains a launch needs beside that: least_chains.
// Unlike fp32 products, which keep the vector ALU of every co-resident wavefront waiting,
// bf16 products overlap with it: six VALU instructions per product cost nothing measurable
// with four wavefronts per SIMD.
//
// What bounds it: the matrix pipe at the clock the chip holds under this load:
// 1024 -> 1024 1x1 over 16 384 pixels 174 us, 197 TFLOP/s (fp32 products: 261 us); small K on
// large maps: HBM (64 -> 256 1x1 on 64 x 56x56: 77 -> 67 us, 3.8 TB/s); single
// images: the latency of a slice's loads (512 -> 512 3x3 on one 7x7 map: 21 -> 16 us).
// The two multiplications by 2^24 per pair of bottom values cost 2 % of a full launch.
//
// Values the split cannot hold (infinities, NaN, magnitudes of 2^103 and above) and sums of
// 2^80 and above leave an accumulator non-finite.  A wavefront that finds one after the K loop
// forms its block again with fp32 products straight from memory (below).
//
// OCC = wavefronts per SIMD the register allocation must leave room for.
// MODE selects how the K loop finds and guards the elements it gathers:
//   kModeMasks     tap table + one "outside the image" bit mask per tap row and
//                  per tap column (any kernel up to 31 x 31 taps);
//   kModeOneMask   one mask with a bit per (row, column) tap pair, the taps' offsets from
//                  the scalar unit, for kernels with at most 31 taps (3x3, 5x5) and a channel
//                  count that is a multiple of 4: the K rows are then ordered
//                  (channel block of 4, tap, channel in block), so four
//                  consecutive rows share one tap and one validity test;
//   kModePointwise every row k of the gather is channel k of the bottom blob at
//                  the thread's own pixel (1x1 kernel, no padding): no table, no mask.
template <int BM, int BN, int WM, int WN, int OCC, int MODE, int KS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void igemm_split_kernel(
    const IgemmBatch batch) {
  static_assert(WM * WN == 4, "four wavefronts per workgroup");
  const int kslice = blockIdx.z;
  const IgemmArgs& a = batch.sub[0];  // a Convolution is one sub-problem
  static_assert(BN >= 64 && 256 % BN == 0, "BN must be 64, 128 or 256");
  constexpr int TM = BM / WM / 32;
  constexpr int TN = BN / WN / 32;
  static_assert(TM >= 1 && TN >= 1, "wave tile must hold a 32x32 block");
  constexpr int BE = BN * BK / 256;           // consecutive K rows of its pixel a thread gathers per K tile
  constexpr int A_CHUNKS = 6 * BM;            // 16-byte pieces of an A tile: plane, K half, row
  constexpr int A_VEC = (A_CHUNKS + 255) / 256;

  // Operands in LDS: [plane h, m, l][K half][row][8 K rows].  Lane l of the 32x32x16
  // product supplies row l % 32 and K rows 8 (l / 32) .. + 7 of either operand: one
  // ds_read_b128 per plane, 512 contiguous bytes per half-wave, no bank conflicts; a
  // gathering thread stores the rows it holds of a plane with one instruction, too.
  // KS 16-row K tiles form one stage (one barrier per stage).
  __shared__ __attribute__((aligned(16))) uint16_t As[2][KS][3][2][BM][8];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[2][KS][3][2][BN][8];
  __shared__ float2 factors[BM];  // (scale, shift) of the tile's rows

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int g = blockIdx.y;

  // XCD-aware tile order: workgroup ids are dealt round-robin to the 8 XCDs, so
  // give each XCD a contiguous run of logical tiles (m fastest): the tiles that
  // share one pixel tile, and neighbouring pixel tiles, then hit the same L2.
  int mt, nt;
  {
    const int total = a.MT * a.NT;
    const int bid = blockIdx.x;
    const int q = total / kNumXcd, r = total % kNumXcd;
    const int xcd = bid % kNumXcd, local = bid / kNumXcd;
    const int logical = xcd * q + (xcd < r ? xcd : r) + local;
    nt = fast_div(logical, a.div_mt_mul, a.div_mt_shift);
    mt = logical - nt * a.MT;
  }

  // The loop does its addressing on the scalar unit and in the memory instructions
  // themselves:
  //  * the bottom is read through a buffer descriptor: scalar base, scalar offset per
  //    K row, one fixed VGPR offset per thread, and an out-of-range VGPR offset
  //    returns 0 without a branch or a select.
  //    The bottom is kept below 2 GiB and "no element" is offset bit 31.  The
  //    descriptor starts far enough before the blob that the sum of a
  //    pixel origin and a tap offset is never negative, so a flagged offset lies
  //    in [2^31, 2^32 - 16) and offset + access size cannot wrap around 2^32
  //    (an access that carries into bit 32 would leave the checked range);
  //  * per thread, bit b of row_bad / col_bad says that row (column) tap b
  //    falls outside the image for the thread's pixel, so an element costs two
  //    bit-field extracts and two shift-ors (one extract and one shift-or per four
  //    elements with one mask, nothing at all when pointwise);
  //  * the loop is unrolled over the two LDS buffers so every LDS address is
  //    a base register plus an immediate.
  const __amdgpu_buffer_rsrc_t xres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x), 0, a.x_bytes, kBufferFlags);
  constexpr bool PW = MODE == kModePointwise;

  // Byte offset of pixel p's origin from the descriptor base (never negative) and its
  // masks.  A column past the last pixel gets kNoElement and full masks.
  auto pixel_setup = [&](int p, unsigned& voff, unsigned& row_bad, unsigned& col_bad) {
    // (the divisions are prepared for every column of the last tile, also those past the
    // last pixel: the pointwise mode computes first and picks afterwards, without a branch)
    const int n = fast_div(p, a.div_hw_mul, a.div_hw_shift);
    const int rem = p - n * a.HqWq;
    const int qh = fast_div(rem, a.div_w_mul, a.div_w_shift);
    const int qw = rem - qh * a.Wq;
    const int hi0 = qh * a.q_sh + a.in_oh;
    const int wi0 = qw * a.q_sw + a.in_ow;
    const unsigned origin = static_cast<unsigned>(
        ((n * a.x_nstride + g * a.x_gstride + (hi0 * a.W + wi0)) << 2) + a.pix_shift);
    voff = PW ? (p < a.P ? origin : kNoElement) : 0u;
    row_bad = col_bad = 0xFFFFFFFFu;
    if (!PW && p < a.P) {
      voff = origin;
      row_bad = 0x80000000u;  // bit 31: the tap of K padding rows, never valid
      col_bad = 0u;
      for (int b = 0; b < a.n_dh; ++b)
        row_bad |= static_cast<unsigned>(static_cast<unsigned>(hi0 + a.tap_dh[b]) >=
                                         static_cast<unsigned>(a.H))
                   << b;
      for (int b = 0; b < a.n_dw; ++b)
        col_bad |= static_cast<unsigned>(static_cast<unsigned>(wi0 + a.tap_dw[b]) >=
                                         static_cast<unsigned>(a.W))
                   << b;
      if constexpr (MODE == kModeOneMask) {
        // bit i*n_dw + j = row tap i or column tap j outside; the result replaces row_bad
        const unsigned all_cols = (1u << a.n_dw) - 1u;
        unsigned pair_bad = 0x80000000u;
        for (int b = 0; b < a.n_dh; ++b)
          pair_bad |= (((row_bad >> b) & 1u) ? all_cols : col_bad) << (b * a.n_dw);
        row_bad = pair_bad;
      }
    }
  };
  // The pixel this thread gathers for the B tile (fixed over the K loop).
  const int pj = tid % BN;
  const int prow = tid / BN;  // wave-uniform because BN >= 64
  unsigned xvoff, row_bad, col_bad;
  pixel_setup(nt * BN + pj, xvoff, row_bad, col_bad);
  const int KT = a.Kpad / (BK * KS);  // stages
  // Split-K: slice z multiplies K stages [kt_begin, kt_end); its partial sums go
  // to the workspace the last workgroup of the tile adds up (IgemmArgs::partial)
  // or, for a launch with two tops, into its own copy of the top blob.
  const int kt_begin = kslice * a.kt_per_split;
  const int kt_end = min(KT, kt_begin + a.kt_per_split);
  float* __restrict__ yout = a.y + (size_t)kslice * a.split_stride;

  // Packed filter: [g][K tile][plane][K half][m][8 k]: piece c of an A tile is row
  // c % BM of (plane, half) c / BM, and goes to the same place in LDS.
  unsigned avoff[A_VEC];
#pragma unroll
  for (int i = 0; i < A_VEC; ++i) {
    const int c = tid + 256 * i;
    avoff[i] = static_cast<unsigned>(((c / BM) * a.Mpad + mt * BM + c % BM) * 16);
  }
  const size_t wt_kt_bytes = static_cast<size_t>(a.Mpad) * (6 * 16);
  const char* const wt_g =
      reinterpret_cast<const char*>(a.wt_split) + static_cast<size_t>(g) * (a.Kpad / BK) * wt_kt_bytes;
  const unsigned x_cbytes = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a.x_cstride) * 4);
  const int kmax = a.K - 1;
  const int n_taps = a.n_dh * a.n_dw, quads = a.K / 4;  // (kModeOneMask: K is a multiple of 4)
  int quad_tap[(BE + 3) / 4];
  unsigned quad_off[(BE + 3) / 4];

  // two sets: tile t waits in set t % 2
  u32x4 areg[2][KS][A_VEC];
  float breg[2][KS][BE];

#define MC_LOADF(res, voff, soff) \
  __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(res, voff, soff, 0))
#define MC_GATHER1(dst, t)                                                                   \
  {                                                                                          \
    /* The tap's byte offset rides in the scalar offset of the load; the VGPR                \
       offset is the pixel origin, with bit 31 set when the tap is outside the               \
       image.  Origin + tap offset stays below 2^31, so a flagged sum cannot wrap            \
       whether or not the hardware adds the scalar offset before its range check. */        \
    const unsigned rb = __builtin_amdgcn_ubfe(row_bad, (t).y, 1);                            \
    const unsigned cb = __builtin_amdgcn_ubfe(col_bad, (t).z, 1);                            \
    dst = MC_LOADF(xres, (cb << 31) | ((rb << 31) | xvoff), (t).x);                          \
  }
  // Piece i of the A tile `kt16` / element e of the thread's B rows, fetched into set `set`.
#define MC_LOAD_A(set, ks, kt16, i)                                                          \
  if (A_CHUNKS % 256 == 0 || tid + 256 * (i) < A_CHUNKS)                                     \
    areg[set][ks][i] = *reinterpret_cast<const u32x4*>(                                      \
        wt_g + static_cast<size_t>(kt16) * wt_kt_bytes + avoff[i]);
#define MC_LOAD_B(set, ks, kt16, e)                                                          \
  {                                                                                          \
    const int krow = __builtin_amdgcn_readfirstlane((kt16)*BK + prow * BE);                  \
    if constexpr (PW) {                                                                      \
      /* padding rows re-read the last channel; their filter rows are zero (an infinity there \
         makes NaN of it, and the sum is formed again below, without padding rows) */        \
      breg[set][ks][e] = MC_LOADF(xres, xvoff, static_cast<unsigned>(min(krow + (e), kmax)) * x_cbytes); \
    } else if constexpr (MODE == kModeOneMask) {                                             \
      const unsigned pb = __builtin_amdgcn_ubfe(row_bad, quad_tap[(e) / 4], 1);              \
      breg[set][ks][e] = MC_LOADF(xres, (pb << 31) | xvoff, quad_off[(e) / 4] + (e) % 4 * x_cbytes); \
    } else {                                                                                 \
      const int4 tap = a.ktab[krow + (e)];                                                   \
      MC_GATHER1(breg[set][ks][e], tap);                                                     \
    }                                                                                        \
  }
  // One mask: rows 4 q .. 4 q + 3 are four channels (block q / taps) at tap q % taps.
  // Computed on the scalar unit: a table would be fetched through the scalar cache, whose
  // answers arrive in no order among the LDS reads, and the first product of every stage would
  // wait for it.  Padding rows get tap 31, which is outside the image for every pixel.
#define MC_QUADS(kt16)                                                                       \
  if constexpr (MODE == kModeOneMask) {                                                      \
    _Pragma("unroll") for (int q = 0; q < BE / 4; ++q) {                                     \
      const int row = __builtin_amdgcn_readfirstlane((kt16)*BK + prow * BE) / 4 + q;         \
      const int block = fast_div(row, batch.div_taps_mul, batch.div_taps_shift);                     \
      const int tap = row - block * n_taps;                                                  \
      const int ti = (tap * batch.div_kw_mul) >> 16;                                             \
      const unsigned off = static_cast<unsigned>(block) * 4u * x_cbytes +                    \
                           static_cast<unsigned>(ti * batch.tap_h4 + (tap - ti * a.n_dw) * batch.tap_w4); \
      quad_tap[q] = row < quads ? tap : 31;                                                  \
      quad_off[q] = row < quads ? off : 0u;                                                  \
    }                                                                                        \
  }
#define MC_STORE_A(set, ks, i)                                                               \
  if (A_CHUNKS % 256 == 0 || tid + 256 * (i) < A_CHUNKS)                                     \
    reinterpret_cast<u32x4*>(&As[set][ks][0][0][0][0])[tid + 256 * (i)] = areg[set][ks][i];
#define MC_SPLIT_B(set, ks, q) \
  split_pair(breg[set][ks][2 * (q)], breg[set][ks][2 * (q) + 1], bt[0][q], bt[1][q], bt[2][q]);
#define MC_STORE_B(set, ks)                                                                  \
  _Pragma("unroll") for (int pl = 0; pl < 3; ++pl) {                                         \
    if constexpr (BE == 4) {                                                                 \
      *reinterpret_cast<u32x2*>(&Bs[set][ks][pl][prow >> 1][pj][(prow & 1) * 4]) =           \
          u32x2{bt[pl][0], bt[pl][1]};                                                       \
    } else {                                                                                 \
      _Pragma("unroll") for (int q = 0; q < BE / 8; ++q)                                     \
        *reinterpret_cast<u32x4*>(&Bs[set][ks][pl][prow + q][pj][0]) =                       \
            u32x4{bt[pl][4 * q], bt[pl][4 * q + 1], bt[pl][4 * q + 2], bt[pl][4 * q + 3]};   \
    }                                                                                        \
  }
#define MC_LOAD_TILES(set, kt)                                                               \
  _Pragma("unroll") for (int ks = 0; ks < KS; ++ks) {                                        \
    _Pragma("unroll") for (int i = 0; i < A_VEC; ++i) MC_LOAD_A(set, ks, (kt)*KS + ks, i)    \
    MC_QUADS((kt)*KS + ks)                                                                   \
    _Pragma("unroll") for (int e = 0; e < BE; ++e) MC_LOAD_B(set, ks, (kt)*KS + ks, e)       \
  }
#define MC_STORE_TILES(set)                                                                  \
  _Pragma("unroll") for (int ks = 0; ks < KS; ++ks) {                                        \
    unsigned bt[3][BE / 2];                                                                  \
    _Pragma("unroll") for (int i = 0; i < A_VEC; ++i) MC_STORE_A(set, ks, i)                 \
    _Pragma("unroll") for (int q = 0; q < BE / 2; ++q) MC_SPLIT_B(set, ks, q)                \
    MC_STORE_B(set, ks)                                                                      \
  }
#define MC_READ_A(buf, ks, q)                                                                \
  _Pragma("unroll") for (int i = 0; i < TM; ++i) av[q][i] =                                  \
      *reinterpret_cast<const bf16x8*>(&As[buf][ks][q][lhi][wm0 + i * 32 + l32][0]);
#define MC_READ_B(buf, ks, q)                                                                \
  _Pragma("unroll") for (int j = 0; j < TN; ++j) bv[q][j] =                                  \
      *reinterpret_cast<const bf16x8*>(&Bs[buf][ks][q][lhi][wn0 + j * 32 + l32][0]);
  // The products of tile `buf` with, if asked for, the loads of stage `next` and the stores of
  // the other buffer.  The order is pinned one product at a time (the barriers are for the
  // compiler's scheduler only): a product occupies the matrix pipe for 32 cycles, in which
  // the wavefront issues the side work placed behind it.  First half of the
  // products: the remaining operand reads and the global loads; second half: the splitting of
  // the tile that has arrived meanwhile and its LDS stores.
#define MC_STAGE(buf, load, store, next)                                                     \
  _Pragma("unroll") for (int ks = 0; ks < KS; ++ks) {                                        \
    constexpr int P = TM * TN;          /* products per pair of terms */                     \
    constexpr int L = A_VEC + BE;       /* loads, over the first 3 P products */             \
    constexpr int NP = BE / 2;          /* pairs to split, over all but one of the others */ \
    constexpr int S = 3 * P - 1;                                                             \
    bf16x8 av[3][TM], bv[3][TN];                                                             \
    unsigned bt[3][BE / 2];                                                                  \
    const int kt16 = (next)*KS + ks;                                                         \
    __builtin_amdgcn_sched_barrier(0);                                                       \
    MC_READ_A(buf, ks, 0)                                                                    \
    MC_READ_B(buf, ks, 0)                                                                    \
    if constexpr (P == 1) {                                                                  \
      MC_READ_B(buf, ks, 1)                                                                  \
      MC_READ_A(buf, ks, 1)                                                                  \
    }                                                                                        \
    __builtin_amdgcn_sched_barrier(0);                                                       \
    _Pragma("unroll") for (int s = 0; s < 6 * P; ++s) {                                      \
      const int i = s % P / TN, j = s % P % TN;                                              \
      if (P == 1 && s == 0 && (buf) == 1)                                                    \
        odd = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[0][0], bv[0][0], odd, 0, 0, 0);     \
      else if (s < P)                                                                        \
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[0][i], bv[0][j], acc[i][j], 0, 0, 0); \
      else                                                                                   \
        accs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                                \
            av[s / P == 2 || s / P == 3 ? 1 : (s / P == 5 ? 2 : 0)][i],                      \
            bv[s / P == 1 || s / P == 3 ? 1 : (s / P == 4 ? 2 : 0)][j], accs[i][j], 0, 0, 0);\
      if (load && s == 0) {                                                                  \
        MC_QUADS(kt16)                                                                       \
      }                                                                                      \
      if (P > 1 && s == 0) MC_READ_B(buf, ks, 1)                                             \
      if (P > 1 && s == 1) MC_READ_A(buf, ks, 1)                                             \
      if (s == P) MC_READ_B(buf, ks, 2)                                                      \
      if (s == P + (P > 1)) MC_READ_A(buf, ks, 2)                                            \
      if (load) {                                                                            \
        _Pragma("unroll") for (int u = 0; u < L; ++u) {                                      \
          if (s >= 3 * P || u < s * L / (3 * P) || u >= (s + 1) * L / (3 * P)) continue;     \
          if (u < A_VEC) {                                                                   \
            MC_LOAD_A(buf, ks, kt16, u)                                                      \
          } else {                                                                           \
            MC_LOAD_B(buf, ks, kt16, (u < A_VEC ? 0 : u - A_VEC))                            \
          }                                                                                  \
        }                                                                                    \
      }                                                                                      \
      if (store) {                                                                           \
        _Pragma("unroll") for (int i2 = 0; i2 < A_VEC; ++i2)                                 \
          if (s == 3 * P + i2 % (3 * P)) MC_STORE_A(1 - (buf), ks, i2)                       \
        _Pragma("unroll") for (int q = 0; q < NP; ++q) {                                     \
          if (s < 3 * P || s == 6 * P - 1 || q < (s - 3 * P) * NP / S ||                     \
              q >= (s - 3 * P + 1) * NP / S)                                                 \
            continue;                                                                        \
          MC_SPLIT_B(1 - (buf), ks, q)                                                       \
        }                                                                                    \
        if (s == 6 * P - 2) MC_STORE_B(1 - (buf), ks)                                        \
      }                                                                                      \
      __builtin_amdgcn_sched_barrier(0);                                                     \
    }                                                                                        \
  }

  acc16 acc[TM][TN], accs[TM][TN];  // h h', and the five small products
  // A wavefront of one block has registers left for two chains of h h', of the even and of
  // the odd stages: half the error of one chain, as two K slices would leave (kChains).
  acc16 odd;
#pragma unroll
  for (int r = 0; r < 16; ++r) odd[r] = 0.f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = accs[i][j][r] = 0.f;

  const int wm0 = (wave % WM) * (BM / WM);
  const int wn0 = (wave / WM) * (BN / WN);
  const int l32 = lane & 31;
  const int lhi = lane >> 5;

  // Per-channel factors of the epilogue: thread t < BM fetches scale and shift of row t
  // of this tile before the K loop; the first barrier of the loop publishes them, and
  // after the last product a wavefront reads the (scale, shift) pairs of its rows
  // without another barrier.
  float2 ep_val = make_float2(1.f, 0.f);
  const float* scale_ptr = a.scale;
  const float* shift_ptr = a.shift;
  if (tid < BM && mt * BM + tid < a.M) {
    if (scale_ptr != nullptr) ep_val.x = scale_ptr[g * a.M + mt * BM + tid];
    if (shift_ptr != nullptr) ep_val.y = shift_ptr[g * a.M + mt * BM + tid];
  }
  if (kt_end > kt_begin) {
    // Tile kt_begin + t sits in LDS buffer t % 2.  Stage t requests tile t + 2, multiplies
    // tile t and stores tile t + 1, which was requested a stage ago: a load has more than a
    // stage to arrive.  (In the loop a request past the end asks for the last tile again;
    // nobody waits for it.)
    const int nk = kt_end - kt_begin;
    const int kt_last = kt_end - 1;
    MC_LOAD_TILES(0, kt_begin);
    MC_LOAD_TILES(1, min(kt_begin + 1, kt_last));
    MC_STORE_TILES(0);
    if (tid < BM) factors[tid] = ep_val;
    __syncthreads();
    int t = 0;
    if constexpr (TM * TN == 1) {
      // short launches end on the latency of what they wait for: the last stages request
      // and store nothing (64 -> 256 1x1 on one 56x56 map: 6.2 us with, 5.0 without)
      for (; t + 2 < nk; t += 2) {
        MC_STAGE(0, true, true, kt_begin + t + 2)
        __syncthreads();
        MC_STAGE(1, true, true, min(kt_begin + t + 3, kt_last))
        __syncthreads();
      }
      if (t + 1 < nk) {
        MC_STAGE(0, false, true, 0)
        __syncthreads();
        MC_STAGE(1, false, false, 0)
      } else {
        MC_STAGE(0, false, false, 0)
      }
    } else {
      // more copies of the stage than these three do not fit the registers of the larger tiles
      for (; t + 1 < nk; t += 2) {
        MC_STAGE(0, true, true, min(kt_begin + t + 2, kt_last))
        __syncthreads();
        MC_STAGE(1, true, true, min(kt_begin + t + 3, kt_last))
        __syncthreads();
      }
      if (t < nk) MC_STAGE(0, false, false, 0)
    }
  } else {
    // (a slice past the last K tile of a short sub-problem: zeros, but it may be the one
    // that sums the slices and runs the epilogue)
    if (tid < BM) factors[tid] = ep_val;
    __syncthreads();
  }
#undef MC_GATHER1
#undef MC_LOAD_A
#undef MC_LOAD_B
#undef MC_QUADS
#undef MC_STORE_A
#undef MC_SPLIT_B
#undef MC_STORE_B
#undef MC_LOAD_TILES
#undef MC_STORE_TILES
#undef MC_READ_A
#undef MC_READ_B
#undef MC_STAGE

  float probe = 0.f;  // NaN as soon as one sum of this lane is not finite
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if constexpr (TM * TN == 1) acc[i][j][r] += odd[r];
        acc[i][j][r] = (acc[i][j][r] + accs[i][j][r]) * kSplitUnscale;
        probe = __builtin_fmaf(acc[i][j][r], 0.f, probe);
      }
  if (__any(probe != 0.f)) {
    // Rare: an operand is infinite, NaN or of 2^103 and above, or a sum is of 2^80 and
    // above.  The wavefront forms its blocks again from fp32 values: its lanes read
    // their filter rows and the bottom straight from memory, eight K rows each, and
    // multiply with the fp32 instruction.  No LDS and no barrier: the other wavefronts
    // do not take part.
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      unsigned voff, rbad, cbad;
      pixel_setup(nt * BN + wn0 + j * 32 + l32, voff, rbad, cbad);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        acc16 sum;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = 0.f;
        const uint16_t* wrow = a.wt_split + ((static_cast<size_t>(g) * (a.Kpad / BK) * 6 + lhi) * a.Mpad +
                                       mt * BM + wm0 + i * 32 + l32) * 8;
        for (int kt16 = kt_begin * KS; kt16 < kt_end * KS; ++kt16) {
          const uint16_t* w = wrow + static_cast<size_t>(kt16) * a.Mpad * 48;
          const size_t plane = static_cast<size_t>(a.Mpad) * 16;
#pragma unroll 2
          for (int e = 0; e < 8; ++e) {
            const int k = kt16 * BK + 8 * lhi + e;
            unsigned off;
            if constexpr (PW) {
              // (a padding row is no element: an infinity of the last channel times zero is NaN)
              off = voff == kNoElement || k > kmax ? kNoElement : voff + static_cast<unsigned>(k) * x_cbytes;
            } else {
              const int4 tap = a.ktab[k];
              const unsigned bad = MODE == kModeOneMask
                                       ? (rbad >> tap.w) & 1u
                                       : ((rbad >> tap.y) | (cbad >> tap.z)) & 1u;
              off = bad ? kNoElement : voff + static_cast<unsigned>(tap.x);
            }
            const float wv = filter_value(w[e], w[plane + e], w[2 * plane + e]);
            sum = __builtin_amdgcn_mfma_f32_32x32x2f32(wv, MC_LOADF(xres, off, 0), sum, 0, 0, 0);
          }
        }
        acc[i][j] = sum;
      }
    }
  }
#undef MC_LOADF

  finish_split_tile<BM, BN, TM, TN>(a, batch.slices, kslice, g, mt, nt, wm0, wn0, acc, factors,
                                    reinterpret_cast<int*>(&As[0][0][0][0][0][0]), scale_ptr, shift_ptr, yout);
}

// Packed filter wt[g][kt][plane][kl / 8][m][kl % 8] = the bf16 terms of
// w[g*wg_stride + wk_off[k] + m*wm_stride] with k = kt*16 + kl, zero where k >= K or
// m >= M.  filter_value() of the terms is the weight, for every weight.
__global__ void pack_split_kernel(const float* __restrict__ w, uint16_t* __restrict__ wt,
                                  const int* __restrict__ wk_off, int G, int K, int Kpad, int M, int Mpad, int wm_stride, int wg_stride) {
  const long total = (long)G * Kpad * Mpad;
  const int KT = Kpad / BK;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total;
       i += (long)gridDim.x * blockDim.x) {
    const int kl = static_cast<int>(i % BK);
    long t = i / BK;
    const int m = static_cast<int>(t % Mpad);
    t /= Mpad;
    const int kt = static_cast<int>(t % KT);
    const int g = static_cast<int>(t / KT);
    const int k = kt * BK + kl;
    float v = 0.f;
    if (k < K && m < M) v = w[(long)g * wg_stride + wk_off[k] + (long)m * wm_stride];
    const unsigned bits = __builtin_bit_cast(unsigned, v);
    v *= kSplitScale;
    const float h = static_cast<float>(static_cast<__bf16>(v));
    const float mid = static_cast<float>(static_cast<__bf16>(v - h));
    const float low = static_cast<float>(static_cast<__bf16>(v - h - mid));
    const bool fits = __builtin_isfinite(h);
    uint16_t* out = wt + (((static_cast<size_t>(g) * KT + kt) * 6 + kl / 8) * Mpad + m) * 8 + kl % 8;
    const size_t plane = static_cast<size_t>(Mpad) * 16;
    out[0] = static_cast<uint16_t>(fits ? __builtin_bit_cast(unsigned, h) >> 16 : kNotSplit);
    out[plane] = static_cast<uint16_t>(fits ? __builtin_bit_cast(unsigned, mid) >> 16 : bits >> 16);
    out[2 * plane] = static_cast<uint16_t>(fits ? __builtin_bit_cast(unsigned, low) >> 16 : bits & 0xFFFFu);
  }
}

#include "igemm_small.h"

struct SplitConfig {
  int bm, bn;
  int ks;   // 16-row K tiles per stage
  int occ;  // workgroups per CU the kernel is built for
  int chains;  // accumulators h h' alternates between (small: two per run, the second of a third of it)
  // measured on full launches: a CU's time per 16-row K tile and per tile (prologue and
  // epilogue); 0 = taken on request only
  float stage_us, fixed_us;
  const char* name;
  void (*kernel[3])(const IgemmBatch);  // indexed by mode
  // igemm_small_kernel, whose tiles are taken for small launches: wavefronts that share K and the
  // kernels for taps, for pointwise launches, and for those whose last K tiles hold padding
  // (0 and null: igemm_split_kernel)
  int waves;
  void (*small[3])(const SmallArgs);
};

#define MC_CONFIG(BM, BN, WM, WN, OCC, KS, STAGE, FIXED, NAME)                \
  {BM, BN, KS, OCC, BM / WM * (BN / WN) == 32 * 32 ? 2 : 1, STAGE, FIXED, NAME,                                       \
   {igemm_split_kernel<BM, BN, WM, WN, OCC, kModeMasks, KS>,                  \
    igemm_split_kernel<BM, BN, WM, WN, OCC, kModeOneMask, KS>,                \
    igemm_split_kernel<BM, BN, WM, WN, OCC, kModePointwise, KS>}, 0, {nullptr, nullptr, nullptr}}
#define MC_SMALL(NW, NAME)                                                   \
  {32, 32, 1, 16 / NW, 3 * NW / 2, 0.f, 0.f, NAME, {nullptr, nullptr, nullptr}, NW,  \
   {igemm_small_kernel<NW, kModeOneMask, false>, igemm_small_kernel<NW, kModePointwise, false>, \
    igemm_small_kernel<NW, kModePointwise, true>}}
const SplitConfig kSplitConfigs[] = {
    MC_CONFIG(128, 128, 2, 2, 2, 1, 0.56f, 3.3f, "igemm_split_128x128"),
    MC_CONFIG(128, 64, 2, 2, 3, 1, 0.363f, 0.9f, "igemm_split_128x64"),
    MC_CONFIG(64, 128, 2, 2, 3, 1, 0.377f, 1.2f, "igemm_split_64x128"),
    // (3, 5 and 6, taken on request only, are other places' tiles: each instance is many
    // seconds of compilation, and none of their own shapes was the best of any layer measured)
    MC_CONFIG(64, 64, 2, 2, 3, 2, 0.f, 0.f, "igemm_split_64x64x32"),
    MC_CONFIG(32, 128, 1, 4, 4, 1, 0.215f, 0.6f, "igemm_split_32x128"),
    MC_CONFIG(32, 128, 1, 4, 4, 1, 0.f, 0.f, "igemm_split_32x128"),
    MC_CONFIG(64, 128, 2, 2, 3, 1, 0.f, 0.f, "igemm_split_64x128"),
    MC_CONFIG(64, 64, 2, 2, 3, 2, 0.21f, 0.8f, "igemm_split_64x64x32"),
    MC_SMALL(4, "igemm_split_32x32_k4"),
    MC_SMALL(8, "igemm_split_32x32_k8"),
};
#undef MC_CONFIG
#undef MC_SMALL
constexpr int kNumSplitConfigs = sizeof(kSplitConfigs) / sizeof(kSplitConfigs[0]);

