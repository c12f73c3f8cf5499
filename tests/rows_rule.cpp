// Host program around the rule that chooses an expert call's GEMMs (afd_rows_rule.h): reads lines
//   weight_fmt inter topk expert_lo num_local tile_walk n capacity pairs groups active
// and prints, for each, the plan's form, rows of a group, the router's choice for those counts and the
// row groups the few-rows GEMMs are launched for.
#include <cstdio>

#include "../sgl-afd-plugin_amd/csrc/afd_rows_rule.h"

int main() {
  long long n;
  int capacity, pairs, groups, active;
  afd_moe_cfg cfg = {};
  cfg.hidden = 4096;
  while (std::scanf("%d %d %d %d %d %d %lld %d %d %d %d", &cfg.weight_fmt, &cfg.inter, &cfg.topk, &cfg.expert_lo,
                    &cfg.num_local, &cfg.tile_walk, &n, &capacity, &pairs, &groups, &active) == 11) {
    const afd::RowsPlan p = afd::rows_plan(cfg, n, capacity != 0);
    std::printf("%d %d %d %d\n", p.form, 1 << p.group_shift,
                static_cast<int>(afd::rows_few(p, pairs, groups, active)), p.grid_groups);
  }
  return 0;
}
