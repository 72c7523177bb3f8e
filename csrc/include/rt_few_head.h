// What lies ahead of the rows that workgroups of encoder_few.hip hand to one another; the launch ahead of it (the embedding) writes it.
#pragma once

namespace rt {

struct FewHead {
  unsigned next;      // the next task
  unsigned gap[15];
  unsigned lost;      // somebody gave up; on a line of its own
  unsigned tries;     // askings after which one does
  unsigned* report;   // a word of host memory that says so
  unsigned rest[44];
};
static_assert(sizeof(FewHead) == 256, "rows lie 256 bytes behind");

}  // namespace rt
