// split_rules.cpp -- the rule of jne_segments.h by which a small mixed batch is
// split over its walks' segments, built for the host (test_split_rules.py).
#include "jne_segments.h"

extern "C" unsigned long long split_doubles(unsigned waves, unsigned steps) {
  return jne::segment_split_doubles(waves, steps);
}
extern "C" unsigned chunks(unsigned steps) { return jne::split_chunks(steps); }
