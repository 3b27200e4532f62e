// The fused beam step for rows whose addresses are not all multiples of 16 bytes: lengths that are no multiple of 4, or
// tables that start elsewhere.  The shapes of beam.hip, without the sketch (which such rows do not have).  Read element by
// element, one row at a time, 37 queries at 20,011 x 50 took 4,558 us; several rows in flight, 16 bytes a load: 1,284 us.
#include "beam_kernels.h"

namespace {

template <RowForm FORM>
void launch_long(const StepArgs &s, int threads, size_t smem, hipStream_t st) {
    const int nchunks = s.nchunks;
    if (nchunks <= 128) launch_step<2, 64, 4, FORM>(s, threads, smem, st);
    else if (nchunks <= 192) launch_step<3, 64, 2, FORM>(s, threads, smem, st);
    else if (nchunks <= 256) launch_step<4, 64, 2, FORM>(s, threads, smem, st);
    else if (nchunks <= 320) launch_step<5, 64, 2, FORM>(s, threads, smem, st);
    else if (nchunks <= 384) launch_step<6, 64, 2, FORM>(s, threads, smem, st);
    else if (nchunks <= 448) launch_step<7, 64, 2, FORM>(s, threads, smem, st);
    else launch_step<8, 64, 2, FORM>(s, threads, smem, st);
}

}  // namespace

void vl_launch_step_unaligned(const StepArgs &s, int threads, size_t smem, hipStream_t st) {
    const int nchunks = s.nchunks;
    // From 385 columns on batches of up to twelve rows per compute unit turn their sums into distances together, larger ones, which
    // wait on bytes, right away: 300 / 1,500 / 2,300 / 10,000 queries at 30,000 x 390 right away 3.51 / 6.48 / 8.17 / 31.9 ms,
    // together 3.16 / 5.81 / 7.65 / 33.1, at 30,000 x 902 4.24 / 9.96 / 14.8 / 63.0 and 3.28 / 9.90 / 15.2 / 65.2, at 30,000 x 1,282
    // 4.61 / 13.5 / 24.7 / 88.1 and 3.75 / 13.9 / 23.1 / 90.6.  The shape for 769 to 1,024 columns leaves five wavefronts per SIMD,
    // ten rows of 128 threads per compute unit, and with one row in flight instead of two seven; eleven and twelve rows would
    // wait for a second round (2,800 at 30,000 x 902 22.0 and 18.7 ms; 2,400, ten rows, 15.6 and 16.4).
    const int64_t rows_per_cu = (s.m.n_rows + kComputeUnits - 1) / kComputeUnits;
    // Rows in flight of the short shapes: where many rows share a compute unit, as many as leave eight wavefronts per SIMD (59
    // and 62 registers).  With twice as many (84 and 82) five fit, ten rows of 128 threads, and those beyond ran in a round of
    // their own: 2,400 / 2,800 / 10,000 queries at 20,011 x 50 1,562 -> 1,599, 2,352 -> 1,636 and 5,299 -> 4,817 us, at
    // 30,000 x 126 1,920 -> 1,930, 2,947 -> 2,065 and 6,555 -> 6,478.  A few rows want the loads: 37 queries at 20,011 x 50
    // 941 us with eight, 958 with four.
    if (nchunks <= 16 && threads == 128) launch_step<1, 16, 4, kRowUnalignedSums>(s, threads, smem, st);
    else if (nchunks <= 16) launch_step<1, 16, 8, kRowUnalignedSums>(s, threads, smem, st);
    else if (nchunks <= 32 && threads == 128) launch_step<2, 16, 2, kRowUnalignedSums>(s, threads, smem, st);
    else if (nchunks <= 32) launch_step<2, 16, 4, kRowUnalignedSums>(s, threads, smem, st);
    // (four rows in flight: eight take registers that leave five wavefronts per SIMD instead of seven; builds of 34,111 x 130 150.2 ->
    // 133.1 ms, 20,696 x 130 109.2 -> 97.7, 30,000 x 250 163.1 -> 154.7, searches the same)
    else if (nchunks <= 64) launch_step<1, 64, 4, kRowUnalignedSums>(s, threads, smem, st);
    else if (nchunks <= 96) launch_step<3, 32, 2, kRowUnalignedSums>(s, threads, smem, st);
    else if (rows_per_cu > 12) launch_long<kRowUnaligned>(s, threads, smem, st);
    else if (rows_per_cu > 10 && nchunks > 192 && nchunks <= 256) launch_step<4, 64, 1, kRowUnalignedSums>(s, threads, smem, st);
    else launch_long<kRowUnalignedSums>(s, threads, smem, st);
}
