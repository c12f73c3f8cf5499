// Host program around the rule that chooses an expert call's GEMMs (afd_rows_rule.h): reads lines
//   weight_fmt inter topk expert_lo num_local tile_walk n pairs groups active
// and prints, for each, the plan's form, rows of a group, and the router's choice for those counts.
#include <cstdio>

#include "../sgl-afd-plugin_amd/csrc/afd_rows_rule.h"

int main() {
  long long n;
  int pairs, groups, active;
  afd_moe_cfg cfg = {};
  cfg.hidden = 4096;
  while (std::scanf("%d %d %d %d %d %d %lld %d %d %d", &cfg.weight_fmt, &cfg.inter, &cfg.topk, &cfg.expert_lo,
                    &cfg.num_local, &cfg.tile_walk, &n, &pairs, &groups, &active) == 10) {
    const afd::RowsPlan p = afd::rows_plan(cfg, n);
    std::printf("%d %d %d\n", p.form, 1 << p.group_shift, static_cast<int>(afd::rows_few(p, pairs, groups, active)));
  }
  return 0;
}
