// Plan-specialised kernels: the time-dependent coefficient program emitted as
// straight-line device code and compiled with the paired integrator at run
// time (hiprtc), so the per-step coefficient evaluation runs without the
// expression machine's dispatch, LDS stack and instruction fetches.
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <string>
#include <vector>

#include "lb_program.h"

// The device function lb_gen_coef(sl, cf, t) for the time-dependent programs
// of `prog` (expressions e with expr_dyn[e], compounds first, then the K
// coefficients), or an empty string with `why` set when an instruction has no
// generated form.
std::string lb_rtc_coef_source(const LbProgram& prog, const std::vector<int32_t>& expr_dyn, int K,
                               std::string& why);

// Compiles the kernel sources with `coef_source` for gfx950 and loads the
// kernel named by `name_expr` (a template-id such as
// "lb_solve_pair_kernel<0, 8, 2>") from the resulting code object.
// Plans of one program on one device share the loaded module; the plans that
// use it hold it, and the last few stay loaded for the next plan.  Returns 0,
// or -1 with `why` holding the compiler log or the runtime error.
struct LbModule {
  hipModule_t module = nullptr;
  hipFunction_t function = nullptr;
  ~LbModule() {
    if (module) (void)hipModuleUnload(module);
  }
};
int lb_rtc_compile(const std::string& coef_source, const std::string& name_expr, std::shared_ptr<LbModule>* out,
                   std::string& why);
// Counts a call (as `calls` of them) that would take the kernel: whether `after`
// have come in the process, or it holds the kernel already.
bool lb_rtc_ready(const std::string& coef_source, const std::string& name_expr, int64_t calls, int after);
