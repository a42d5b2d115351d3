// C entry points over hc_wrap.h for the CPU test of periodic node coordinates
// (tests/test_wrap.py builds this file with g++).
#include "../../hemocell_amd/csrc/hc_wrap.h"

extern "C" {
int wrap_node(double fl, int n) { return hcg::wrap_node(fl, n); }
int wrap_far(double fl, int n) { return hcg::wrap_far(fl, n); }
}
