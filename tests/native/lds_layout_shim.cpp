// C entry points over hc_lds_plan.h for the CPU test of the layout a launch takes
// (tests/test_lds_layout.py builds this file with g++).
#include <cstdint>

#include "../../hemocell_amd/csrc/hc_lds_plan.h"

extern "C" {

// out: ok, staged, fixed, region, lists, dyn, box_nodes
void layout(int model, int nv, int visc, int64_t psize, int64_t box_bytes, int64_t lds_device, int64_t st, int pos,
            int64_t* out) {
  const hcg::CellLdsPlan p =
      hcg::cell_lds_layout(model, nv, visc != 0, (size_t)psize, (size_t)box_bytes, (size_t)lds_device, (size_t)st,
                           (size_t)st, (size_t)st, (hcg::CellPositions)pos);
  const int64_t v[7] = {p.ok, p.staged, (int64_t)p.fixed, (int64_t)p.region, (int64_t)p.lists, (int64_t)p.dyn,
                        p.box_nodes};
  for (int k = 0; k < 7; ++k) out[k] = v[k];
}

int64_t mech_bytes(int model, int nv, int64_t psize) { return (int64_t)hcg::cell_mech_bytes(model, nv, (size_t)psize); }
int64_t edge_bytes(int nv, int64_t psize) { return (int64_t)hcg::platelet_edge_bytes(nv, (size_t)psize); }
}
