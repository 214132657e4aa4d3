// What follows the K loop of igemm_kernel and igemm_split_kernel: the sum over K slices inside
// the launch, then the layer's epilogue and the store.  The text of a block and not a function:
// igemm_kernel includes it in its own body, because through a function's parameters the
// compiler fetches what the block reads from the kernel arguments before the K loop and spills
// it (1 -> 1006 3x3 on 3 x 100x100 35.0 us, as a function 37.4; 848 -> 8 on 4 x 21x21 in 24
// slices 35.3 and 39.2).  igemm_split_kernel has the registers and is 2 % faster with the
// function (finish_split_tile).
//
// Names it uses: batch, a, sub_index, kslice, g, mt, nt, wm0, wn0, acc, scale_ptr, shift_ptr, yout,
// tid, l32, lhi.  The includer defines
//   MC_FACTORS(row)  address in LDS of the (scale, shift) pair of tile row `row`
//   MC_ARRIVED       address of an int of LDS that no wavefront needs any more after a barrier
//   MC_SLICES        number of K slices
//   MC_AHEAD         K slices whose partial sums are fetched together
//   MC_PLAIN         pixel p of an image is element p of its top plane (the pixel-quad mode)
  // What the epilogue reads from the argument block is fetched here in one batch:
  // fetched where it is first used, the fields cost the wavefront four or five
  // scalar-memory round trips after the last MFMA, one after the other.  (Before the K
  // loop they would not fit the scalar registers the loop needs.)
  struct {
    int* counters;
    const float* residual;
    unsigned y_bytes, div_hw_mul, div_hw_shift, div_w_mul, div_w_shift;
    int y_cstride, y_nstride, Wo, out_sh, out_sw, out_oh, out_ow, M, P, HqWq, Wq, act;
    float slope;
  } e = {a.counters, a.residual, a.y_bytes, a.div_hw_mul, a.div_hw_shift, a.div_w_mul, a.div_w_shift,
         a.y_cstride, a.y_nstride, a.Wo, a.out_sh, a.out_sw, a.out_oh, a.out_ow, a.M, a.P, a.HqWq, a.Wq,
         a.act, a.slope};
  asm volatile("" ::"s"(e.counters), "s"(e.residual), "s"(e.y_bytes), "s"(e.div_hw_mul), "s"(e.div_hw_shift),
               "s"(e.div_w_mul), "s"(e.div_w_shift), "s"(e.y_cstride), "s"(e.y_nstride), "s"(e.Wo),
               "s"(e.out_sh), "s"(e.out_sw), "s"(e.out_oh), "s"(e.out_ow), "s"(e.M), "s"(e.P), "s"(e.HqWq),
               "s"(e.Wq), "s"(e.act), "s"(e.slope));

  if (e.counters != nullptr) {
    // K slices summed here: see IgemmArgs::partial.  The partial sums and the
    // counter are accessed with device-scope atomic operations only (relaxed
    // stores and loads that go past the per-XCD L2, which is not coherent with
    // the other seven), so no cache write-back or invalidation is needed: a
    // workgroup waits until its own stores have completed and then counts.
    // What this rests on is particular to the parts it is built for: a store with
    // device scope (sc1) is written through to the memory side, where all XCDs meet,
    // and vmcnt counts it down only when that write has been acknowledged; an
    // atomic on the counter issued after the wait is therefore ordered behind the
    // partial sums at the one place every later device-scope load reads from.  The
    // language's memory model promises none of this for relaxed accesses.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx942__) && !defined(__gfx950__)
#error "the in-launch sum of K slices relies on gfx942 / gfx950 device-scope write-through"
#endif
    const int tile_id = (sub_index * gridDim.y + g) * gridDim.x + blockIdx.x;
    constexpr int kRegs = TM * TN * 16;  // accumulator registers per thread
    float* mine = a.partial +
                  (static_cast<size_t>(kslice) * a.partial_tiles + tile_id) * (kRegs * 256) + tid;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          __hip_atomic_store(mine + ((i * TN + j) * 16 + r) * 256, acc[i][j][r], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial sums have arrived
    __syncthreads();  // ... every thread's, and every wave is done with the tiles in LDS
    int* arrived = MC_ARRIVED;
    if (tid == 0)
      arrived[0] = __hip_atomic_fetch_add(&e.counters[tile_id], 1, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived[0] != MC_SLICES - 1) return;  // uniform over the workgroup
    // the next launch on this stream starts from zero
    if (tid == 0)
      __hip_atomic_store(&e.counters[tile_id], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // Slices are added in slice order, the loads of MC_AHEAD of them together (as many as the
    // registers hold): one at a time each costs a round trip to memory (2048 -> 512 1x1
    // on one 7x7 map, eight slices: 12.9 us, four at a time 11.8).
    const float* part = a.partial + static_cast<size_t>(tile_id) * (kRegs * 256) + tid;
    const size_t slice_elems = static_cast<size_t>(a.partial_tiles) * (kRegs * 256);
#pragma unroll
    for (int r = 0; r < kRegs; ++r)
      acc[r / 16 / TN][r / 16 % TN][r % 16] =
          __hip_atomic_load(part + r * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if constexpr (MC_AHEAD == 1) {
      for (int z = 1; z < MC_SLICES; ++z) {
        part += slice_elems;
#pragma unroll
        for (int r = 0; r < kRegs; ++r)
          acc[r / 16 / TN][r / 16 % TN][r % 16] +=
              __hip_atomic_load(part + r * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else {
      for (int z = 1; z < MC_SLICES; z += MC_AHEAD) {
        float v[MC_AHEAD][kRegs];
#pragma unroll
        for (int u = 0; u < MC_AHEAD; ++u) {
          // (a slice past the last one is read as the last one and not added)
          const float* from = part + min(z + u, MC_SLICES - 1) * slice_elems;
#pragma unroll
          for (int r = 0; r < kRegs; ++r)
            v[u][r] = __hip_atomic_load(from + r * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int u = 0; u < MC_AHEAD; ++u)
          if (z + u < MC_SLICES) {
#pragma unroll
            for (int r = 0; r < kRegs; ++r) acc[r / 16 / TN][r / 16 % TN][r % 16] += v[u][r];
          }
      }
    }
  }

  // Epilogue.  Accumulator register r of lane l holds row 8*(r/4)+4*(l/32)+r%4,
  // column l%32 of its 32x32 block; a half-wave therefore stores 32 consecutive
  // pixels of one output channel.  Like the K loop it addresses through buffer
  // descriptors: one VGPR offset per lane (bit 31 set for a column past the last
  // pixel, which drops its stores), the row as a scalar offset.  Per-channel
  // factors and residual values are fetched eight rows at a time, all loads of
  // a batch issued before the first use.
  const bool has_scale = scale_ptr != nullptr;
  const bool has_shift = shift_ptr != nullptr;
  const bool has_res = e.residual != nullptr;
  const __amdgpu_buffer_rsrc_t yres =
      __builtin_amdgcn_make_buffer_rsrc(yout, 0, e.y_bytes, kBufferFlags);
  const __amdgpu_buffer_rsrc_t rres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(e.residual), 0, has_res ? e.y_bytes : 0, kBufferFlags);
  // 0: none, 1: ReLU (max with 0), 2: leaky ReLU, 3: TanH / Sigmoid
  const int act_mode = e.act == MC_ACT_NONE ? 0
                       : e.act == MC_ACT_RELU ? (e.slope == 0.f ? 1 : 2)
                                              : 3;
  const unsigned cs4 = static_cast<unsigned>(e.y_cstride) * 4;
#define MC_ROW(r) (8 * ((r) / 4) + ((r) % 4))
#define MC_LOADF(res, voff, soff) \
  __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(res, voff, soff, 0))
#define MC_STORE_ROWS(EXPR)                                                                  \
  _Pragma("unroll") for (int q = 0; q < 8; ++q) {                                            \
    const float v = acc[i][j][half * 8 + q];                                                 \
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (EXPR)), yres, y_voff,\
                                          MC_ROW(half * 8 + q) * cs4, 0);                    \
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int p = nt * BN + wn0 + j * 32 + l32;
    const int n = fast_div(p, e.div_hw_mul, e.div_hw_shift);
    const int rem = p - n * e.HqWq;
    int ybase;
    if constexpr (MC_PLAIN) {
      ybase = n * e.y_nstride + rem;
    } else {
      const int qh = fast_div(rem, e.div_w_mul, e.div_w_shift);
      const int qw = rem - qh * e.Wq;
      ybase = n * e.y_nstride + (qh * e.out_sh + e.out_oh) * e.Wo + qw * e.out_sw + e.out_ow;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int mblock = mt * BM + wm0 + i * 32;  // wave-uniform
      const int m0 = mblock + 4 * lhi;
      if (mblock + 32 <= e.M) {
        // All 32 rows are real channels.
        const unsigned c0 = g * e.M + m0;
        const unsigned y_voff =
            p < e.P ? static_cast<unsigned>(ybase + c0 * e.y_cstride) * 4 : kNoElement;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          if (has_scale | has_shift) {
            float sc[8], sh[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const int lrow = wm0 + i * 32 + 4 * lhi + MC_ROW(half * 8 + q);
              const float2 f = *reinterpret_cast<const float2*>(MC_FACTORS(lrow));
              sc[q] = f.x;
              sh[q] = f.y;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
              acc[i][j][half * 8 + q] = acc[i][j][half * 8 + q] * sc[q] + sh[q];
          }
          if (has_res) {
            float rs[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) rs[q] = MC_LOADF(rres, y_voff, MC_ROW(half * 8 + q) * cs4);
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[i][j][half * 8 + q] += rs[q];
          }
          if (act_mode == 0) {
            MC_STORE_ROWS(v)
          } else if (act_mode == 1) {
            MC_STORE_ROWS(fmaxf(v, 0.f))
          } else if (act_mode == 2) {
            MC_STORE_ROWS(v > 0.f ? v : v * e.slope)
          } else {
            MC_STORE_ROWS(apply_act(v, e.act, e.slope))
          }
        }
      } else if (p < e.P) {
        // Block straddles the last channel: row by row, skipping rows >= M.
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + MC_ROW(r);
          if (m < e.M) {
            const int c = g * e.M + m;
            float v = acc[i][j][r];
            if (has_scale) v *= a.scale[c];
            if (has_shift) v += a.shift[c];
            const int yo = ybase + c * e.y_cstride;
            if (has_res) v += e.residual[yo];
            yout[yo] = apply_act(v, e.act, e.slope);
          }
        }
      }
    }
  }
#undef MC_ROW
#undef MC_LOADF
#undef MC_STORE_ROWS
#undef MC_FACTORS
#undef MC_ARRIVED
#undef MC_SLICES
#undef MC_AHEAD
#undef MC_PLAIN
