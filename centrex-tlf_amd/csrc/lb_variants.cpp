// Host view of the variant table and of the kernels compiled in the parts of
// lb_kernels.hip (one part per object file, LB_NPARTS_BUILT in total).
#include "lb_variants.h"

extern "C" void* lb_dev_solve_kernel_p0(int, int);
extern "C" void* lb_dev_solve_kernel_p1(int, int);
extern "C" void* lb_dev_solve_kernel_p2(int, int);
extern "C" void* lb_dev_solve_kernel_p3(int, int);
extern "C" void* lb_dev_solve_kernel_p4(int, int);
extern "C" void* lb_dev_solve_kernel_p5(int, int);
extern "C" void* lb_dev_solve_kernel_p6(int, int);
extern "C" void* lb_dev_solve_kernel_p7(int, int);
extern "C" void* lb_dev_lean_kernel_p0(int, int);
extern "C" void* lb_dev_lean_kernel_p1(int, int);
extern "C" void* lb_dev_lean_kernel_p2(int, int);
extern "C" void* lb_dev_lean_kernel_p3(int, int);
extern "C" void* lb_dev_lean_kernel_p4(int, int);
extern "C" void* lb_dev_lean_kernel_p5(int, int);
extern "C" void* lb_dev_lean_kernel_p6(int, int);
extern "C" void* lb_dev_lean_kernel_p7(int, int);
extern "C" void* lb_dev_fixed_kernel_p0(int, int);
extern "C" void* lb_dev_fixed_kernel_p1(int, int);
extern "C" void* lb_dev_fixed_kernel_p2(int, int);
extern "C" void* lb_dev_fixed_kernel_p3(int, int);
extern "C" void* lb_dev_fixed_kernel_p4(int, int);
extern "C" void* lb_dev_fixed_kernel_p5(int, int);
extern "C" void* lb_dev_fixed_kernel_p6(int, int);
extern "C" void* lb_dev_fixed_kernel_p7(int, int);
extern "C" void* lb_dev_event_kernel_p0(int, int);
extern "C" void* lb_dev_event_kernel_p1(int, int);
extern "C" void* lb_dev_event_kernel_p2(int, int);
extern "C" void* lb_dev_event_kernel_p3(int, int);
extern "C" void* lb_dev_event_kernel_p4(int, int);
extern "C" void* lb_dev_event_kernel_p5(int, int);
extern "C" void* lb_dev_event_kernel_p6(int, int);
extern "C" void* lb_dev_event_kernel_p7(int, int);
extern "C" void* lb_dev_adjoint_kernel_p0(int, int);
extern "C" void* lb_dev_adjoint_kernel_p1(int, int);
extern "C" void* lb_dev_adjoint_kernel_p2(int, int);
extern "C" void* lb_dev_adjoint_kernel_p3(int, int);
extern "C" void* lb_dev_adjoint_kernel_p4(int, int);
extern "C" void* lb_dev_adjoint_kernel_p5(int, int);
extern "C" void* lb_dev_adjoint_kernel_p6(int, int);
extern "C" void* lb_dev_adjoint_kernel_p7(int, int);
extern "C" void* lb_dev_rhs_kernel_p0(int);
extern "C" void* lb_dev_rhs_kernel_p1(int);
extern "C" void* lb_dev_rhs_kernel_p2(int);
extern "C" void* lb_dev_rhs_kernel_p3(int);
extern "C" void* lb_dev_rhs_kernel_p4(int);
extern "C" void* lb_dev_rhs_kernel_p5(int);
extern "C" void* lb_dev_rhs_kernel_p6(int);
extern "C" void* lb_dev_rhs_kernel_p7(int);

static_assert(LB_NPARTS_BUILT == 8, "lb_variants.cpp lists eight kernel parts");

extern "C" int lb_dev_variant_count(void) {
  int n = 0;
#define X(i, r, w, v) ++n;
  LB_CONFIGS(X)
#undef X
#define Y(i, v) ++n;
  LB_WAVE_CONFIGS(Y)
#undef Y
#define A(i, of) ++n;
  LB_WAVE_ALIASES(A)
#undef A
#define Q(i, g, v) ++n;
  LB_PAIR_CONFIGS(Q)
#undef Q
  return n;
}

// The id that variant `id` is another name of, or itself.
extern "C" int lb_dev_variant_of(int id) {
#define A(i, of) \
  if (id == i) return of;
  LB_WAVE_ALIASES(A)
#undef A
  return id;
}

extern "C" int lb_dev_variant(int id, int* R, int* maxw, int* waves) {
  id = lb_dev_variant_of(id);
#define X(i, r, w, v)                                                                           \
  if (id == i) { *R = r; *maxw = w; *waves = v; return 1; }
  LB_CONFIGS(X)
#undef X
#define Y(i, v)                                                                                 \
  if (id == i) { *R = 1; *maxw = 64; *waves = v; return 1; }
  LB_WAVE_CONFIGS(Y)
#undef Y
#define Q(i, g, v)                                                                              \
  if (id == i) { *R = 1; *maxw = 64; *waves = v; return 1; }
  LB_PAIR_CONFIGS(Q)
#undef Q
  return 0;
}

// 1 for the single-wave (one trajectory per wave) variants.
extern "C" int lb_dev_variant_wave(int id) {
  id = lb_dev_variant_of(id);
#define Y(i, v) \
  if (id == i) return 1;
  LB_WAVE_CONFIGS(Y)
#undef Y
  return 0;
}

// Coupling rows a paired variant holds in registers (0: not a paired variant).
extern "C" int lb_dev_variant_rows(int id) {
#define Q(i, g, v) \
  if (id == i) return g;
  LB_PAIR_CONFIGS(Q)
#undef Q
  return 0;
}

// The shape that runs variant `id` on a plan of `rows` coupling rows.
extern "C" int lb_dev_variant_shape(int id, int rows) {
#define Q(i, g, v) \
  if (id == 15 && rows <= g) return i;
  LB_PAIR_NARROW(Q)
#undef Q
  return id;
}

extern "C" void* lb_dev_solve_kernel(int id, int solver) {
  void* (*parts[])(int, int) = {lb_dev_solve_kernel_p0, lb_dev_solve_kernel_p1, lb_dev_solve_kernel_p2, lb_dev_solve_kernel_p3, lb_dev_solve_kernel_p4, lb_dev_solve_kernel_p5, lb_dev_solve_kernel_p6, lb_dev_solve_kernel_p7};
  return id < 0 ? nullptr : parts[id % LB_NPARTS_BUILT](id, solver);
}

// The lean form of a single- or multi-wave variant (lb_solve_kernel); null for the others.
extern "C" void* lb_dev_lean_kernel(int id, int solver) {
  void* (*parts[])(int, int) = {lb_dev_lean_kernel_p0, lb_dev_lean_kernel_p1, lb_dev_lean_kernel_p2, lb_dev_lean_kernel_p3, lb_dev_lean_kernel_p4, lb_dev_lean_kernel_p5, lb_dev_lean_kernel_p6, lb_dev_lean_kernel_p7};
  return id < 0 ? nullptr : parts[id % LB_NPARTS_BUILT](id, solver);
}

extern "C" void* lb_dev_rhs_kernel(int id) {
  void* (*parts[])(int) = {lb_dev_rhs_kernel_p0, lb_dev_rhs_kernel_p1, lb_dev_rhs_kernel_p2, lb_dev_rhs_kernel_p3, lb_dev_rhs_kernel_p4, lb_dev_rhs_kernel_p5, lb_dev_rhs_kernel_p6, lb_dev_rhs_kernel_p7};
  return id < 0 ? nullptr : parts[id % LB_NPARTS_BUILT](id);
}

// Adjoint variants: Z(id, R, largest workgroup, waves hint), then the
// single-wave V(id, gather rows, waves hint) with *rows = gather rows (0 for
// the multi-wave form).
// rows > 0: a single-block variant; block: a multi-wave one over couplings.
extern "C" int lb_dev_adjoint_variant(int id, int* R, int* maxw, int* rows, int* block) {
#define Z(i, r, w, v)                                                                           \
  if (id == i) { *R = r; *maxw = w; *rows = 0; *block = 0; return 1; }
  LB_ADJ_CONFIGS(Z)
#undef Z
#define V(i, g, v)                                                                              \
  if (id == i) { *R = 1; *maxw = 64; *rows = g; *block = 0; return 1; }
  LB_ADJ_WAVE_CONFIGS(V)
#undef V
#define B(i, r, w, v)                                                                           \
  if (id == i) { *R = r; *maxw = w; *rows = 0; *block = 1; return 1; }
  LB_ADJ_BLOCK_CONFIGS(B)
#undef B
  return 0;
}

extern "C" void* lb_dev_adjoint_kernel(int id, int solver) {
  void* (*parts[])(int, int) = {lb_dev_adjoint_kernel_p0, lb_dev_adjoint_kernel_p1, lb_dev_adjoint_kernel_p2, lb_dev_adjoint_kernel_p3, lb_dev_adjoint_kernel_p4, lb_dev_adjoint_kernel_p5, lb_dev_adjoint_kernel_p6, lb_dev_adjoint_kernel_p7};
  return id < 0 ? nullptr : parts[id % LB_NPARTS_BUILT](id, solver);
}

// Fixed-step variants: F(id, R, largest workgroup, waves hint).
extern "C" int lb_dev_fixed_variant(int id, int* R, int* maxw) {
#define F(i, r, w, v)                                                                           \
  if (id == i) { *R = r; *maxw = w; return 1; }
  LB_FIXED_CONFIGS(F)
#undef F
  return 0;
}

extern "C" int lb_dev_eff_variant(int id, int* R, int* maxw, int* seats) {
#define E(i, r, w, v, t)                                                                        \
  if (id == i) { *R = r; *maxw = w; *seats = t; return 1; }
  LB_EFF_CONFIGS(E)
#undef E
  return 0;
}

extern "C" int lb_dev_event_variant(int id, int* R, int* maxw) {
#define E(i, r, w, v)                                                                           \
  if (id == i) { *R = r; *maxw = w; return 1; }
  LB_EVENT_CONFIGS(E)
#undef E
  return 0;
}

extern "C" void* lb_dev_event_kernel(int id, int solver) {
  void* (*parts[])(int, int) = {lb_dev_event_kernel_p0, lb_dev_event_kernel_p1, lb_dev_event_kernel_p2, lb_dev_event_kernel_p3, lb_dev_event_kernel_p4, lb_dev_event_kernel_p5, lb_dev_event_kernel_p6, lb_dev_event_kernel_p7};
  return id < 0 ? nullptr : parts[id % LB_NPARTS_BUILT](id, solver);
}

extern "C" void* lb_dev_fixed_kernel(int id, int solver) {
  void* (*parts[])(int, int) = {lb_dev_fixed_kernel_p0, lb_dev_fixed_kernel_p1, lb_dev_fixed_kernel_p2, lb_dev_fixed_kernel_p3, lb_dev_fixed_kernel_p4, lb_dev_fixed_kernel_p5, lb_dev_fixed_kernel_p6, lb_dev_fixed_kernel_p7};
  return id < 0 ? nullptr : parts[id % LB_NPARTS_BUILT](id, solver);
}
