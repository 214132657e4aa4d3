// Offsets of the pointwise loads of igemm_small_kernel.  Plain arithmetic, so that a host program
// can check them for every K.
#ifndef MCHIP_SMALL_ROWS_H_
#define MCHIP_SMALL_ROWS_H_

#ifdef __HIPCC__
#define MC_SMALL_ROWS_FN __host__ __device__ constexpr
#else
#define MC_SMALL_ROWS_FN constexpr
#endif

namespace mchip {

// A buffer load is told its address in two parts, the lane's offset and a scalar one, and only the
// lane's is sure to be compared with the buffer's end.  Half-wave h takes rows 16 kt + 8 h + e, e =
// 0 .. 7, of K tile kt; `own` is the offset of the lane's pixel in row 8 h.  Where every row exists
// the rest goes into the scalar offset, which costs nothing.  With TAIL, for a K that leaves rows
// of padding in the last tiles (the filter has a multiple of 32), it goes into the lane's, so that
// a row past the end of the blob is seen to be there.  That is an addition per load (1x1 @14, 528
// -> 160 5.28 us beside 5.31 for 544 -> 160 without; a comparison and a selection per load 5.99).
template <bool TAIL>
MC_SMALL_ROWS_FN unsigned small_lane_offset(unsigned own, int kt, int e, unsigned plane_bytes) {
  return TAIL ? own + static_cast<unsigned>(16 * kt + e) * plane_bytes : own;
}
template <bool TAIL>
MC_SMALL_ROWS_FN unsigned small_scalar_offset(int kt, int e, unsigned plane_bytes) {
  return TAIL ? 0u : static_cast<unsigned>(16 * kt + e) * plane_bytes;
}
MC_SMALL_ROWS_FN bool small_needs_tail(int K, int Kpad) { return K != Kpad; }

}  // namespace mchip

#undef MC_SMALL_ROWS_FN

#endif  // MCHIP_SMALL_ROWS_H_
