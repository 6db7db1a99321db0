// Independent pointwise and short-stencil dispatches side by side in one
// launch (te_batch_part).
#include "pointwise.hpp"
#include "te_kernels.hpp"

namespace te {

TE_DEV void turb_km_kh_body(uint32_t* M, const KArg& a, const Blk& b) { turb_km_kh_at<false>(M, a, b); }
TE_DEV void turb_km_kh_xy_body(uint32_t* M, const KArg& a, const Blk& b) { turb_km_kh_at<true>(M, a, b); }

enum {
#define TE_ID(n) kPoint_##n,
  TE_POINT_LIST(TE_ID)
#undef TE_ID
};

// All bodies in one kernel: 55 VGPRs in all, 8 waves per SIMD, so the widest
// body does not cost the others waves, and a launch brings in the code of its own
// dispatches only.  What it saves is the drain and start between them, 2 to 4
// us each: a stage's diagnostics, tendency reset, mass fluxes and pressure
// tendency, and the end of a step, are 3 to 5 launches of 3.5-6 us each at
// 64 x 64 x 40.  Workgroups are lines of 256 threads.
__global__ __launch_bounds__(256) void k_point_batch(uint32_t* M, KBatch) {
  const BatchPart p = te_batch_part();
  if (!p.in) return;
  bool in;
  const Blk b = p.line_blk(in);
  if (!in) return;
  // (a switch: the compiler's tree of compares; one after the other they cost
  // the last bodies 20% of their time)
#define TE_CASE(n) \
  case kPoint_##n: n##_body(M, p.a, b); return;
  switch (p.body) { TE_POINT_LIST(TE_CASE) }
#undef TE_CASE
}

int point_body(const char* name) {
#define TE_NAME(n) \
  if (__builtin_strcmp(name, #n) == 0) return kPoint_##n;
  TE_POINT_LIST(TE_NAME)
#undef TE_NAME
  return -1;
}

}  // namespace te
