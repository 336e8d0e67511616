// Compiled solver variants: X(id, slots per thread R, largest workgroup,
// waves-per-SIMD hint).  The hint caps the registers per lane at 512 / hint;
// the host picks a variant whose R * W covers the plan's slots.
#pragma once

// Two shapes gave wrong results that no other variant showed, deterministic
// and with no cause found in the kernel: (4, 256, 1), once entry 6, on the
// full n=39 plan, and (12, 256, 1) and (12, 256, 2), once entry 10, on the
// restricted n=72 plan (12 slots per lane, one wave, about 1,300 spilled
// VGPRs).  Neither is compiled; every entry is checked bitwise against the
// default launch on the n=72 plan.
#define LB_CONFIGS(X)                                                                            \
  X(0, 1, 1024, 4) X(1, 2, 512, 4) X(2, 2, 512, 2) X(3, 3, 1024, 4) X(4, 4, 256, 4)                \
  X(5, 4, 256, 2) X(6, 3, 512, 2) X(7, 6, 512, 2) X(8, 6, 512, 1) X(9, 8, 128, 2) X(10, 6, 256, 2)

// Single-wave variants for plans of at most 64 elements (one slot per lane, 64
// threads): Y(id, waves-per-SIMD hint).  Ids 13 and 14 are other names of 12
// (A(id, of)), once shapes that held their rows in registers.  Whatever the
// rows, one wave is the better form: 4,096 trajectories of a dense system of 55
// elements and 18 rows 2.58 ms against 2.99 ms in the best multi-wave shape.
#define LB_WAVE_CONFIGS(Y) Y(11, 4) Y(12, 2)
#define LB_WAVE_ALIASES(A) A(13, 12) A(14, 12)

// Paired variants for plans of at most 32 elements: two trajectories per wave
// (one per 32-lane half); Q(id, coupling rows in registers, waves-per-SIMD
// hint).  Only for persistent calls that push at every accepted step with a
// given initial step (no trace, save plan or replay; a tape may be recorded);
// the forms compiled per plan cover more (lb_host.cpp).  Variant 15 runs plans
// of at most four rows in a shape of their own, which needs fewer registers
// (two-level scan 2.37 against 3.04 ms, n=39 grid 2.70 against 2.96).
#define LB_PAIR_CONFIGS(Q) Q(15, 8, 2) Q(16, 12, 2)
#define LB_PAIR_NARROW(Q) Q(17, 4, 2)

// Fixed-step kernel variants (fixed_dopri5 / fixed_rk2 / fixed_rk4):
// F(id, slots per thread R, largest workgroup, waves-per-SIMD hint).
#define LB_FIXED_CONFIGS(F) F(0, 1, 1024, 2) F(1, 2, 512, 2) F(2, 4, 256, 2) F(3, 8, 256, 2)
// Stop-event forms (adaptive and fixed-step, compiled apart so the event code
// leaves the other kernels' register allocation alone): one slot per lane up
// to 1024 slots, six per lane up to 3072.
#define LB_EVENT_CONFIGS(E) E(0, 1, 1024, 4) E(1, 6, 512, 1)
// Effective-Hamiltonian integrator: rows of the real state per lane, largest
// workgroup, waves-per-SIMD hint, trajectories (seats) per workgroup.  Seats are
// built for up to 512 rows (16 levels), the sizes they were measured at; a trial
// of two seats for up to 1,024 rows took 20.9 ms against 33.2 with one (20
// levels, 1,024 trajectories).
#define LB_EFF_CONFIGS(E) \
  E(0, 1, 512, 2, 4) E(1, 1, 512, 2, 2) E(2, 1, 512, 2, 1) E(3, 1, 1024, 4, 1) E(4, 4, 512, 2, 1) E(5, 8, 512, 1, 1)

// Adjoint kernel variants over gather tables: Z(id, slots per thread R, largest
// workgroup, waves-per-SIMD hint).
#define LB_ADJ_CONFIGS(Z) Z(0, 1, 1024, 2) Z(1, 2, 512, 2) Z(2, 4, 256, 2) Z(3, 8, 256, 2)

// Single-block adjoint variants for plans of one 64-slot block (lane = slot,
// several waves per trajectory): V(id, gather rows held in registers by
// the recomputation, waves-per-SIMD hint), in increasing rows (the host takes
// the first that covers the plan).
#define LB_ADJ_WAVE_CONFIGS(V) V(4, 12, 2) V(5, 16, 2)

// Multi-wave adjoint over couplings: B(id, slots per thread R, largest
// workgroup, waves-per-SIMD hint), in increasing slots (the host takes the
// first that covers the plan).  Two waves a SIMD: with 128 registers (one
// slot a lane, 1024 threads) three times as many values spilled.
#define LB_ADJ_BLOCK_CONFIGS(B) B(6, 1, 512, 2) B(7, 2, 512, 2) B(8, 4, 512, 2)

#define LB_NPARTS_BUILT 8
