// The fused beam step for rows whose addresses are not all multiples of 16 bytes: lengths that are no multiple of 4, or
// tables that start elsewhere.  The shapes of beam.hip, without the sketch (which such rows do not have).  Read element by
// element, one row at a time, 37 queries at 20,011 x 50 took 4,558 us; several rows in flight, 16 bytes a load: 1,284 us.
#include "beam_kernels.h"

void vl_launch_step_unaligned(const StepArgs &s, int threads, size_t smem, hipStream_t st) {
    const int nchunks = s.nchunks;
    if (nchunks <= 16) launch_step<1, 16, 8, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 32) launch_step<2, 16, 4, kRowUnaligned>(s, threads, smem, st);
    // (four rows in flight: eight take registers that leave five wavefronts per SIMD instead of seven; builds of 34,111 x 130 150.2 ->
    // 133.1 ms, 20,696 x 130 109.2 -> 97.7, 30,000 x 250 163.1 -> 154.7, searches the same)
    else if (nchunks <= 64) launch_step<1, 64, 4, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 96) launch_step<3, 32, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 128) launch_step<2, 64, 4, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 192) launch_step<3, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 256) launch_step<4, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 320) launch_step<5, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 384) launch_step<6, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else if (nchunks <= 448) launch_step<7, 64, 2, kRowUnaligned>(s, threads, smem, st);
    else launch_step<8, 64, 2, kRowUnaligned>(s, threads, smem, st);
}
