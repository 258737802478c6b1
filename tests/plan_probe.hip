// The launch planner's choice for a call, for tests on the host: compiled with the planner's source, linked to the library for the rest.
#include "../vllm_amd/csrc/gemm.hip"

extern "C" int plan_probe(const w4a16_gemm_args* a, int more_scratch, int32_t* out) {
  using namespace w4a16;
  if (int rc = validate(a)) return rc;
  Plan pl;
  if (int rc = make_plan(a, pl, more_scratch != 0)) return rc;
  Plan first;  // what the planner starts from
  if (int rc = make_plan_16bit(a, first)) return rc;
  const auto kib = [](int64_t bytes) { return (int32_t)((bytes + 1023) / 1024); };
  const int32_t v[] = {pl.kind, pl.mb, pl.tn, pl.splits, pl.kps, pl.ks, pl.tail_strips, pl.tail_kind, pl.tail_mb, pl.xcd_map,
                       kib(plan_scratch(pl)), kib(plan_scratch(first)), first.kind};
  for (int i = 0; i < (int)(sizeof(v) / sizeof(v[0])); ++i) out[i] = v[i];
  return 0;
}
