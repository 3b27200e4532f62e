// The fused beam step for rows whose addresses are not all multiples of 16 bytes: lengths that are no multiple of 4, or
// tables that start elsewhere.  The shapes of beam.hip, without the sketch (which such rows do not have).  Read element by
// element, one row at a time, 37 queries at 20,011 x 50 took 4,558 us; several rows in flight, 16 bytes a load: 1,284 us.
#include "beam_kernels.h"

void vl_launch_step_unaligned(const StepArgs &s, int threads, size_t smem, hipStream_t st) {
    const int nchunks = s.nchunks;
    // Two longer shapes leave five wavefronts per SIMD, ten rows of 128 threads per compute unit, and half as many rows in flight
    // six and more.  Ten rows and many want the loads, eleven and twelve would wait for a second round: 2,400 / 2,800 /
    // 10,000 queries at 30,000 x 390 8.4 and 8.4, 13.1 and 9.6, 31.9 and 33.9 ms, at 30,000 x 902 15.6 and 16.4, 22.0 and
    // 18.7, 63.2 and 65.4.
    const int64_t rows_per_cu = (s.m.n_rows + kComputeUnits - 1) / kComputeUnits;
    const bool one_round = rows_per_cu == 11 || rows_per_cu == 12;
    // Rows in flight of the short shapes: where many rows share a compute unit, as many as leave eight wavefronts per SIMD (59
    // and 62 registers).  With twice as many (84 and 82) five fit, ten rows of 128 threads, and those beyond ran in a round of
    // their own: 2,400 / 2,800 / 10,000 queries at 20,011 x 50 1,562 -> 1,599, 2,352 -> 1,636 and 5,299 -> 4,817 us, at
    // 30,000 x 126 1,920 -> 1,930, 2,947 -> 2,065 and 6,555 -> 6,478.  A few rows want the loads: 37 queries at 20,011 x 50
    // 941 us with eight, 958 with four.
    if (nchunks <= 16 && threads == 128) launch_step<1, 16, 4, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 16) launch_step<1, 16, 8, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 32 && threads == 128) launch_step<2, 16, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 32) launch_step<2, 16, 4, kRowUnaligned>(s, threads, smem, st);
    // (four rows in flight: eight take registers that leave five wavefronts per SIMD instead of seven; builds of 34,111 x 130 150.2 ->
    // 133.1 ms, 20,696 x 130 109.2 -> 97.7, 30,000 x 250 163.1 -> 154.7, searches the same)
    else if (nchunks <= 64) launch_step<1, 64, 4, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 96) launch_step<3, 32, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 128 && one_round) launch_step<2, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 128) launch_step<2, 64, 4, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 192) launch_step<3, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 256 && one_round) launch_step<4, 64, 1, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 256) launch_step<4, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 320) launch_step<5, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 384) launch_step<6, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 448) launch_step<7, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else launch_step<8, 64, 2, kRowUnaligned>(s, threads, smem, st);
}
