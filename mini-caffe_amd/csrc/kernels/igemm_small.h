// Convolutions of few output tiles: the products of igemm_split.h with K spread over the
// wavefronts of a workgroup.  Part of conv_igemm.hip (inside its namespace).

// A launch of a few dozen 64x64 tiles (a single image through a classifier, a detector's heads)
// is a chain of latencies: a K stage's loads, its barrier, and above all the sum of the many
// slices it takes to occupy the chip, 16 KB of partial sums per slice that the last workgroup
// of a tile fetches a few slices at a time.  Here a tile is 32 channels x 32 pixels and
// each of the NW wavefronts of its workgroup multiplies a run of K tiles of its own: operands
// go from memory to the registers that the matrix instruction reads, without LDS, without a
// barrier, DEPTH K tiles ahead; the NW blocks of sums then meet in LDS.  Four times as many
// tiles and NW runs each occupy the chip with a quarter or less of the slices, and what a
// slice leaves in memory is 4 KB.  The price is that every operand is fetched and split
// by each wavefront that multiplies it, and a 32x32 tile multiplies each value it fetches half as
// often as a 64x64 tile (64 values for 1024 products, 128 for 4096: twice the traffic and twice the
// splitting), which larger launches do not earn back: see pick_split_launch.
//
// What bounds it: on one image the fixed 3 us of a launch (dispatch, arguments, first loads, the
// meeting of the wavefronts), 0.33 us per K tile of a wavefront, and 2 us where slices are summed.
// us per launch, 64x64 tiles / this, launches of one layer one behind the other: 64 -> 64 3x3 on one 56x56 map
// 10.2 / 7.0, 128 -> 128 @28 11.9 / 8.8, 256 -> 256 @14 13.8 / 9.3, 512 -> 512 @7 16.0 / 10.1, 256 -> 1024 1x1
// @14 8.1 / 5.0, 1024 -> 256 10.2 / 7.2, 512 -> 2048 @7 8.5 / 5.8, 2048 -> 512 11.4 / 7.8, 512 -> 24 3x3 @10
// 15.6 / 8.0.  In the trace of a network's forward, where the filters come from memory, medians 0.6 to 0.8 us above these.
// Sixteen wavefronts to a workgroup instead of slices: 13.6 us where four slices take 10.3.
//
// Lane l of the 32x32x16 product holds K rows 8 (l / 32) .. + 7 of filter row / pixel l % 32: of
// the packed filter 16 contiguous bytes per plane, of the bottom eight dwords, each
// 128 contiguous bytes per half-wave.
struct SmallArgs {
  const float* x;            // the descriptor's base: pix_shift bytes and the taps' reach before the blob
  const uint16_t* wt;        // pack_split_kernel
  float* y;
  const float* scale;
  const float* shift;
  const float* residual;
  float* partial;            // [slice][tile][value][thread]
  int* counters;
  unsigned x_bytes;
  int pix_shift, P, HqWq, Wq;
  unsigned div_hw_mul, div_hw_shift, div_w_mul, div_w_shift;
  int H, W, q_sh, q_sw, in_oh, in_ow;
  int x_cbytes, x_nstride, x_gstride;
  int K, KT;                 // rows of the gather, 16-row tiles of them
  int kt_per_slice, slices;
  int M, Mpad, MT, NT;
  // The one-dimensional grid holds the tiles with this index fastest, then the other, then the
  // groups, then the slices.
  int pixels_fastest, groups;
  unsigned div_inner_mul, div_inner_shift, div_outer_mul, div_outer_shift, div_group_mul, div_group_shift;
  int y_cstride, y_nstride, partial_tiles, act;
  float slope;
  // taps (kModeOneMask): row / taps, tap / columns (times 2^-16), bytes and pixels between neighbours
  int n_dh, n_dw, div_kw_mul, tap_h4, tap_w4, dil_h, dil_w;
  unsigned div_taps_mul, div_taps_shift;
  int c_first;
  float* y_second;           // two tops: channels [c_first, ..) go here, or null
  const int4* ktab;
};

// TAIL: a pointwise launch whose K is not a multiple of 32, so that the last K tiles hold rows of padding.
template <int NW, int MODE, bool TAIL>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 4))) void igemm_small_kernel(
    const SmallArgs a) {
  static_assert(MODE == kModeOneMask || MODE == kModePointwise, "no tap table here");
  static_assert(MODE == kModePointwise || !TAIL, "taps: padding rows have a tap that no pixel has");
  constexpr bool PW = MODE == kModePointwise;
  constexpr int BN = 32;                    // pixels of a tile (64 measured no better anywhere)
  constexpr int EPT = 32 * BN / (NW * 64);  // sums a thread finishes: consecutive rows of a pixel
  constexpr int DEPTH = 3;                  // K tiles on their way
  __shared__ float sums[NW][32][BN];
  __shared__ int arrived;
  extern __shared__ int4 taps[][2];  // [K tile of the slice][K half] {offset, tap} of its two quads
  // The arguments are six cache lines, each a trip to memory the first time a CU reads it.
  // One word of each is wanted here, so the trips are made together; fetched where they are
  // first used, in four or five batches, they cost a launch 0.5 us and more.
  asm volatile("" ::"s"(a.x), "s"(a.x_bytes), "s"(a.in_ow), "s"(a.div_inner_mul), "s"(a.n_dw), "s"(a.ktab));
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lhi = lane >> 5;
  // Workgroup ids are dealt round-robin to the 8 XCDs; each gets a contiguous run of tiles,
  // ordered so that the run's tiles share the larger operand: a launch this small reads
  // little more than its operands once, and every XCD that reads one fetches it into an L2
  // of its own (512 -> 1024 1x1/2 on one 28x28 map, 3.1 MB of filters: 8.5
  // us with the channels' tiles next to each other, 7.0 with the pixels').
  int mt, nt, g, kslice;
  {
    const int total = gridDim.x;
    const int bid = blockIdx.x;
    const int q = total / kNumXcd, r = total % kNumXcd;
    const int xcd = bid % kNumXcd, local = bid / kNumXcd;
    const int logical = xcd * q + (xcd < r ? xcd : r) + local;
    const int inner = a.pixels_fastest ? a.NT : a.MT, outer = a.pixels_fastest ? a.MT : a.NT;
    const int o = fast_div(logical, a.div_inner_mul, a.div_inner_shift);
    const int i = logical - o * inner;
    const int z = fast_div(o, a.div_outer_mul, a.div_outer_shift);
    const int t = o - z * outer;
    mt = a.pixels_fastest ? t : i;
    nt = a.pixels_fastest ? i : t;
    kslice = fast_div(z, a.div_group_mul, a.div_group_shift);
    g = z - kslice * a.groups;
  }
  const int m0 = mt * 32;

  // This thread's outputs: EPT rows of pixel `ep`, and what the epilogue needs of them,
  // requested before the K loop.
  const int ep = nt * BN + tid % BN;
  const int erow = tid / BN * EPT;
  const int en = fast_div(ep, a.div_hw_mul, a.div_hw_shift);
  const int epix = ep - en * a.HqWq;  // (a Convolution: pixel p of an image is element p of its top plane)
  const int ebase = en * a.y_nstride + epix;
  float fscale[EPT], fshift[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) fscale[i] = 1.f, fshift[i] = 0.f;
  if (a.scale != nullptr) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) fscale[i] = a.scale[g * a.M + min(m0 + erow + i, a.M - 1)];
  }
  if (a.shift != nullptr) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) fshift[i] = a.shift[g * a.M + min(m0 + erow + i, a.M - 1)];
  }

  float fres[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) fres[i] = 0.f;
  if (a.residual != nullptr && a.slices == 1 && ep < a.P) {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      fres[i] = a.residual[ebase + (g * a.M + min(m0 + erow + i, a.M - 1)) * a.y_cstride];
  }

  // K tiles of this slice, and of them this wavefront's run
  const int KT = a.KT;
  const int kt_begin = kslice * a.kt_per_slice;
  const int kt_end = min(KT, kt_begin + a.kt_per_slice);
  const int per_wave = (a.kt_per_slice + NW - 1) / NW;
  const int w_begin = min(kt_begin + wave * per_wave, kt_end);
  const int w_end = min(w_begin + per_wave, kt_end);

  const __amdgpu_buffer_rsrc_t xres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x), 0, a.x_bytes, kBufferFlags);
  const unsigned x_cbytes = static_cast<unsigned>(a.x_cbytes);
  if constexpr (!PW) {
    // rows 4 q .. 4 q + 3 are four channels (block q / taps) at tap q % taps; padding rows get
    // tap 31, which is outside the image for every pixel
    const int n_taps = a.n_dh * a.n_dw, quads = a.K / 4;  // (one mask: K is a multiple of 4)
    for (int i = tid; i < (kt_end - kt_begin) * 4; i += NW * 64) {
      const int row = kt_begin * 4 + i;
      const int block = fast_div(row, a.div_taps_mul, a.div_taps_shift);
      const int t = row - block * n_taps;
      const int ti = (t * a.div_kw_mul) >> 16;
      const unsigned off = static_cast<unsigned>(block) * 4u * x_cbytes +
                           static_cast<unsigned>(ti * a.tap_h4 + (t - ti * a.n_dw) * a.tap_w4);
      reinterpret_cast<int2*>(taps)[i] = row < quads ? make_int2(static_cast<int>(off), t) : make_int2(0, 31);
    }
  }
  const int n_dw = a.n_dw;
  // byte offset of the pixel's origin, and (3x3 and the like) a bit per tap outside the image;
  // a column past the last pixel has no elements
  unsigned voff, bad = 0xFFFFFFFFu;
  {
    const int p = nt * BN + l32;
    const int n = fast_div(p, a.div_hw_mul, a.div_hw_shift);
    const int rem = p - n * a.HqWq;
    const int qh = fast_div(rem, a.div_w_mul, a.div_w_shift);
    const int qw = rem - qh * a.Wq;
    const int hi0 = qh * a.q_sh + a.in_oh;
    const int wi0 = qw * a.q_sw + a.in_ow;
    const unsigned origin = static_cast<unsigned>(
        ((n * a.x_nstride + g * a.x_gstride + (hi0 * a.W + wi0)) << 2) + a.pix_shift);
    voff = p < a.P ? origin : kNoElement;
    if constexpr (PW) {
      voff += static_cast<unsigned>(lhi) * 8u * x_cbytes;
    } else if (p < a.P) {
      unsigned col_bad = 0u;
      for (int b = 0; b < n_dw; ++b)
        col_bad |= static_cast<unsigned>(static_cast<unsigned>(wi0 + b * a.dil_w) >= static_cast<unsigned>(a.W)) << b;
      const unsigned all_cols = (1u << n_dw) - 1u;
      bad = 0x80000000u;  // bit 31: the tap of K padding rows, never valid
      for (int b = 0; b < a.n_dh; ++b) {
        const bool row_bad = static_cast<unsigned>(hi0 + b * a.dil_h) >= static_cast<unsigned>(a.H);
        bad |= (row_bad ? all_cols : col_bad) << (b * n_dw);
      }
    }
  }

  // (a group's packed filter is below 2 GiB, see fits_small)
  const unsigned wt_kt_bytes = static_cast<unsigned>(a.Mpad) * (6 * 16);
  const char* const wt_g =
      reinterpret_cast<const char*>(a.wt) + static_cast<size_t>(g) * KT * wt_kt_bytes;
  const __amdgpu_buffer_rsrc_t wres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(wt_g), 0, KT * wt_kt_bytes, kBufferFlags);
  const unsigned a_plane = static_cast<unsigned>(a.Mpad) * 32;
  const unsigned avoff = static_cast<unsigned>((lhi * a.Mpad + m0 + l32) * 16);

  if constexpr (!PW) __syncthreads();  // the taps

  u32x4 areg[DEPTH][3];
  float breg[DEPTH][8];
#define MC_LOADF(voff, soff) \
  __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xres, voff, soff, 0))
  // Rows past K (TAIL): their filter rows are zero.  They read what follows the last channel,
  // nothing past the blob's end (small_rows.h); an infinity there makes NaN of a sum, which is
  // then formed again below, without padding rows.
#define MC_LOAD(set, kt)                                                                      \
  {                                                                                           \
    const int kt_ = (kt);                                                                     \
    _Pragma("unroll") for (int q = 0; q < 3; ++q) areg[set][q] = __builtin_bit_cast(u32x4,    \
        __builtin_amdgcn_raw_buffer_load_b128(wres, avoff, static_cast<unsigned>(kt_) * wt_kt_bytes + q * a_plane, 0)); \
    if constexpr (PW) {                                                                       \
      _Pragma("unroll") for (int e = 0; e < 8; ++e) breg[set][e] =                            \
          MC_LOADF(small_lane_offset<TAIL>(voff, kt_, e, x_cbytes),                           \
                   small_scalar_offset<TAIL>(kt_, e, x_cbytes));                              \
    } else {                                                                                  \
      const int4 two = taps[kt_ - kt_begin][lhi];                                             \
      _Pragma("unroll") for (int h = 0; h < 2; ++h) {                                         \
        const unsigned v = ((__builtin_amdgcn_ubfe(bad, h ? two.w : two.y, 1) << 31) | voff) + \
                           static_cast<unsigned>(h ? two.z : two.x);                          \
        _Pragma("unroll") for (int e = 0; e < 4; ++e)                                         \
          breg[set][4 * h + e] = MC_LOADF(v, e * x_cbytes);                                   \
      }                                                                                       \
    }                                                                                         \
  }
  // h h' in two accumulators in turn, the five small products of terms in another
  // (igemm_split_kernel).  A sum that starts in the matrix instruction is rounded less than one that goes
  // on there, so the last tiles of an unfinished turn take one accumulator each: a run of up to two
  // tiles has no sum that goes on.
#define MC_MULTIPLY(set, chain)                                                               \
  {                                                                                           \
    unsigned bt[3][4];                                                                        \
    _Pragma("unroll") for (int q = 0; q < 4; ++q)                                             \
      split_pair(breg[set][2 * q], breg[set][2 * q + 1], bt[0][q], bt[1][q], bt[2][q]);       \
    bf16x8 av[3], bv[3];                                                                      \
    _Pragma("unroll") for (int q = 0; q < 3; ++q) {                                           \
      av[q] = __builtin_bit_cast(bf16x8, areg[set][q]);                                       \
      bv[q] = __builtin_bit_cast(bf16x8, u32x4{bt[q][0], bt[q][1], bt[q][2], bt[q][3]});      \
    }                                                                                         \
    chain = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[0], bv[0], chain, 0, 0, 0);            \
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[0], bv[1], small, 0, 0, 0);            \
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[1], bv[0], small, 0, 0, 0);            \
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[1], bv[1], small, 0, 0, 0);            \
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[0], bv[2], small, 0, 0, 0);            \
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[2], bv[0], small, 0, 0, 0);            \
  }

  acc16 acc, odd, small;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = odd[r] = small[r] = 0.f;

  if (w_end > w_begin) {
    // (a request past the run's end asks for its last tile again; nobody waits for it)
    const int last = w_end - 1;
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      MC_LOAD(d, min(w_begin + d, last))
      __builtin_amdgcn_sched_barrier(0);
    }
    int kt = w_begin;
    for (; kt + DEPTH <= w_end; kt += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        // (the barriers are for the compiler's scheduler, which would gather the loads of all
        // sets at the end of the loop)
        if (d % 2) MC_MULTIPLY(d, odd) else MC_MULTIPLY(d, acc)
        __builtin_amdgcn_sched_barrier(0);
        MC_LOAD(d, min(kt + d + DEPTH, last))
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    static_assert(DEPTH == 3, "at most two tiles are left");
    if (kt < w_end) MC_MULTIPLY(0, acc)
    if (kt + 1 < w_end) MC_MULTIPLY(1, odd)
  }
#undef MC_LOAD
#undef MC_MULTIPLY

  float probe = 0.f;  // NaN as soon as one sum of this lane is not finite
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    acc[r] = (acc[r] + (odd[r] + small[r])) * kSplitUnscale;
    probe = __builtin_fmaf(acc[r], 0.f, probe);
  }
  if (__any(probe != 0.f)) {
    // Rare, see igemm_split_kernel: the run again from fp32 values.
    acc16 sum;
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[r] = 0.f;
    for (int kt = w_begin; kt < w_end; ++kt) {
      const uint16_t* w = reinterpret_cast<const uint16_t*>(wt_g + static_cast<size_t>(kt) * wt_kt_bytes + avoff);
#pragma unroll 2
      for (int e = 0; e < 8; ++e) {
        const int k = kt * BK + 8 * lhi + e;
        unsigned off;
        if constexpr (PW) {
          off = k < a.K && !(voff & kNoElement) ? voff + static_cast<unsigned>(kt * BK + e) * x_cbytes : kNoElement;
        } else {
          const int4 tap = a.ktab[k];
          off = (bad >> tap.w) & 1u ? kNoElement : voff + static_cast<unsigned>(tap.x);
        }
        const float wv = filter_value(w[e], w[a_plane / 2 + e], w[a_plane + e]);
        sum = __builtin_amdgcn_mfma_f32_32x32x2f32(wv, MC_LOADF(off, 0), sum, 0, 0, 0);
      }
    }
    acc = sum;
  }
#undef MC_LOADF

#pragma unroll
  for (int r = 0; r < 16; ++r) sums[wave][8 * (r / 4) + 4 * lhi + r % 4][l32] = acc[r];
  __syncthreads();
  float v[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    // (In 64 bits: one rounding instead of one per addition.  With this and the chains above the
    // error is below that of 64x64 tiles for every K; in the norm, ReLU'd operands: 64 -> 256 1x1
    // @14 3.9e-8 (in 32 bits 4.8, tiles 4.0), 128 -> 512 @28 4.3 (5.1, 4.8), 96 -> 100 5x5 6.7
    // (8.0, 8.5).  0.0 to 0.1 us of a launch.)
    double sum = sums[0][erow + i][tid % BN];
#pragma unroll
    for (int w = 1; w < NW; ++w) sum += sums[w][erow + i][tid % BN];
    v[i] = static_cast<float>(sum);
  }

  if (a.counters != nullptr) {
    // Slices: left in memory and added by the last workgroup of the tile, in slice order; what
    // the accesses rest on is written down in igemm_finish.h.
    const int tile_id = (g * a.NT + nt) * a.MT + mt;
    constexpr int kThreads = NW * 64;
    float* mine = a.partial + (static_cast<size_t>(kslice) * a.partial_tiles + tile_id) * (32 * BN) + tid;
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      __hip_atomic_store(mine + i * kThreads, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial sums have arrived
    __syncthreads();                                  // ... and every thread's
    if (tid == 0)
      arrived = __hip_atomic_fetch_add(&a.counters[tile_id], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != a.slices - 1) return;  // uniform over the workgroup
    if (tid == 0) __hip_atomic_store(&a.counters[tile_id], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const float* part = a.partial + static_cast<size_t>(tile_id) * (32 * BN) + tid;
    const size_t slice_elems = static_cast<size_t>(a.partial_tiles) * (32 * BN);
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      v[i] = __hip_atomic_load(part + i * kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr int AHEAD = 32 / EPT;  // slices fetched together
    for (int z = 1; z < a.slices; z += AHEAD) {
      float s[AHEAD][EPT];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        // (a slice past the last one is read as the last one and not added)
        const float* from = part + min(z + u, a.slices - 1) * slice_elems;
#pragma unroll
        for (int i = 0; i < EPT; ++i)
          s[u][i] = __hip_atomic_load(from + i * kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int u = 0; u < AHEAD; ++u)
        if (z + u < a.slices) {
#pragma unroll
          for (int i = 0; i < EPT; ++i) v[i] += s[u][i];
        }
    }
  }

  if (ep >= a.P) return;
  if (a.residual != nullptr && a.slices > 1) {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      fres[i] = a.residual[ebase + (g * a.M + min(m0 + erow + i, a.M - 1)) * a.y_cstride];
  }
  // (NaN and -infinity under ReLU as in igemm_finish.h, by whole blocks of 32 channels)
  const bool relu = a.act == MC_ACT_RELU && a.slope == 0.f && m0 + 32 <= a.M;
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int m = m0 + erow + i;
    if (m >= a.M) continue;
    const int c = g * a.M + m;
    float* y = a.y + (ebase + c * a.y_cstride);
    if (a.y_second != nullptr) {
      // two tops: channels [0, c_first) and the others
      const int second = a.groups * a.M - a.c_first;
      y = c < a.c_first ? a.y + ((en * a.c_first + c) * a.y_cstride + epix)
                        : a.y_second + ((en * second + c - a.c_first) * a.y_cstride + epix);
    }
    const float out = v[i] * fscale[i] + fshift[i] + fres[i];
    *y = relu ? fmaxf(out, 0.f) : apply_act(out, a.act, a.slope);
  }
}
