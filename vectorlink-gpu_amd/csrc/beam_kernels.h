// The kernels of the fused beam step and their launches; which shape serves which rows is decided in beam.hip and
// beam_unaligned.hip.
#pragma once
#include "beam_row.h"

namespace {

// ---- the fused step: one launch per iteration, or per window of iterations ------
// The expand phase (memory bound) and the merge phase (LDS / latency bound) of one
// row run in the same workgroup, so on every CU some workgroups stream candidate
// rows while others merge: the merge time hides behind the memory traffic, the
// candidate ids and distances never leave LDS, and an iteration is one launch.
template <int CPL, int LPR, int U, RowForm FORM, int THREADS>
__global__ __launch_bounds__(THREADS) void beam_step_kernel(StepArgs s) {
    beam_row<CPL, LPR, U, FORM, THREADS>(s);
}
// The same kernel built to leave room for WPP wavefronts per SIMD.  Its vector registers would allow that anyway;
// what does not is its scalar registers (more than 96 of them mean seven wavefronts instead of eight), which the
// compiler keeps within bounds when asked, at the price of a few moves to and from lanes of a vector register.
template <int CPL, int LPR, int U, int THREADS, int WPP>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPP)))
void beam_step_kernel_w(StepArgs s) {
    beam_row<CPL, LPR, U, kRowAligned, THREADS>(s);
}
template <int CPL, int LPR, int U, RowForm FORM, int THREADS, int WPP>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPP))) void beam_window_kernel(StepArgs s) {
    beam_row<CPL, LPR, U, FORM, THREADS, 0, 64, 1, true>(s);
}
template <int CPL, int LPR, int U, int THREADS, int SCPL, int SLPR, int SU, int WPE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPE))) void beam_window_sketch_kernel(StepArgs s) {
    beam_row<CPL, LPR, U, kRowAligned, THREADS, SCPL, SLPR, SU, true>(s);
}
// ... and with the products of all queries and vectors at hand (near_products.h); it keeps no query row for the sketch.  An
// iteration of 10,000 rows at 1M x 768 takes 0.16 ms (through the sketch 0.58): a launch of five moves 3.9 GB past L2, most of it rows
// that the bounds leave, 4.9 TB/s of the 6.0 that gathered rows reach, with vector instructions issuing in 62 % of cycles.  Rows in
// flight and room for wavefronts per SIMD are the fastest of those tried (of the chosen ones those for 384, 768 and 1,536 columns keep
// three or four vector registers in scratch memory, for 1,792 25, for 2,048 57, the others none).  First-loop batches of 10,000 (ms), 1M x 768 /
// 500,000 x 1,024 / 500,000 x 1,536 / 1M x 384: one row and six wavefronts 59.2 / 57.6 / 93.3 / 35.9, two and six 57.8 / 66.5 / 93.1 / 36.0,
// one and five 59.4 / 57.7 / 82.9 / 36.0, two and five 62.5 / 61.0 / 99.7 / 38.6, two and four 62.7 / 60.8 / 86.4 / 38.4, four and six 76.6 /
// 135.6 / 305.9 / 47.7.  With 128 threads a row 76.0 and 96.6 instead of 59.9 and 84.7 (768 and 1,536 columns).
template <int CPL, int LPR, int U, int THREADS, int SCPL, int WPE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPE))) void beam_window_near_kernel(StepArgs s) {
    beam_row<CPL, LPR, U, kRowAligned, THREADS, SCPL, 64, 1, true, true>(s);
}

// The same step for rows that may use the sketch.  WPE: wavefronts per SIMD the compiler is asked to leave room
// for.  The sketch's copy of the query row takes 16 registers per chunk and lane, and a row's phases (sketch
// pass, two rounds of exact rows, merge) each wait on memory, so residency is worth a few spilled registers:
// measured at 768 and 384 columns, five wavefronts per SIMD with two loads in flight beat three wavefronts
// with four (0.84 -> 0.75 ms and 0.61 -> 0.43 ms per launch).  Residency is what a launch that is not bound by
// memory traffic responds to (768 columns, state of the second optimisation loop, workgroups per compute unit
// limited through LDS: 4 / 5 / 6 -> 0.53 / 0.46 / 0.42 ms per launch; 8 with one load in flight and 62 registers:
// 0.415), which is also why the step's LDS arrays are overlaid where their lifetimes allow.
template <int CPL, int LPR, int U, int THREADS, int SCPL, int SLPR, int SU, int WPE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPE)))
void beam_step_sketch_kernel(StepArgs s) {
    beam_row<CPL, LPR, U, kRowAligned, THREADS, SCPL, SLPR, SU>(s);
}

template <class Kernel>
void launch_rows(Kernel kernel, int threads, const StepArgs &s, size_t smem, hipStream_t st) {
    if (vl_allow_lds(kernel, smem) != hipSuccess) return;  // seen by the launch check
    hipLaunchKernelGGL(kernel, dim3((unsigned)s.m.n_rows), dim3((unsigned)threads), smem, st, s);
}

template <int THREADS, int CPL, int LPR, int U, RowForm FORM, int SCPL, int SLPR, int SU, int WPE, int UX, int WPP, int WPW>
void launch_step_threads(const StepArgs &s, size_t smem, hipStream_t st) {
    if constexpr (SCPL > 0) {
        if (s.sketch) {
            if (s.window > 0 && s.near_values) launch_rows(beam_window_near_kernel<CPL, LPR, (CPL <= 3 ? 2 : 1), THREADS, SCPL, (CPL <= 3 ? 6 : 5)>, THREADS, s, smem, st);
            else if (s.window > 0) launch_rows(beam_window_sketch_kernel<CPL, LPR, UX, THREADS, SCPL, SLPR, SU, (WPE < 6 ? WPE : 6)>, THREADS, s, smem, st);
            else launch_rows(beam_step_sketch_kernel<CPL, LPR, UX, THREADS, SCPL, SLPR, SU, WPE>, THREADS, s, smem, st);
            return;
        }
    }
    if (s.window > 0) launch_rows(beam_window_kernel<CPL, LPR, U, FORM, THREADS, WPW>, THREADS, s, smem, st);
    else if constexpr (WPP > 0 && FORM == kRowAligned) launch_rows(beam_step_kernel_w<CPL, LPR, U, THREADS, WPP>, THREADS, s, smem, st);
    else launch_rows(beam_step_kernel<CPL, LPR, U, FORM, THREADS>, THREADS, s, smem, st);
}

template <int CPL, int LPR, int U, RowForm FORM, int SCPL = 0, int SLPR = 64, int SU = 1, int WPE = 4, int UX = U, int WPP = 0, int WPW = (WPP > 0 ? 6 : 1)>
void launch_step(const StepArgs &s, int threads, size_t smem, hipStream_t st) {
    if (threads == 128) launch_step_threads<128, CPL, LPR, U, FORM, SCPL, SLPR, SU, WPE, UX, WPP, WPW>(s, smem, st);
    else launch_step_threads<256, CPL, LPR, U, FORM, SCPL, SLPR, SU, WPE, UX, WPP, WPW>(s, smem, st);
}

}  // namespace

// Rows whose addresses are not all multiples of 16 bytes, of 4 to 2,048 elements (beam_unaligned.hip).
void vl_launch_step_unaligned(const StepArgs &s, int threads, size_t smem, hipStream_t st);
