// split_rules.cpp -- the rules of jne_segments.h and jne_forms.h by which the
// moment passes choose a form, built for the host (test_split_rules.py).
#include "jne_forms.h"
#include "jne_segments.h"

extern "C" unsigned long long split_doubles(unsigned waves, unsigned steps) {
  return jne::segment_split_doubles(waves, steps);
}
extern "C" unsigned chunks(unsigned steps) { return jne::split_chunks(steps); }
extern "C" int turn_lanes(int dim, unsigned walks) { return jne::fp64_turn_lanes(dim, walks); }
extern "C" unsigned turns(int dim, unsigned steps, unsigned walks) { return jne::fp64_turns(dim, steps, walks); }
// 0: a wave per block, 1: a lane per component, 2: the dim's own lane group
extern "C" int form(int dim, unsigned steps, unsigned walks) { return (int)jne::split_form(dim, steps, walks); }
