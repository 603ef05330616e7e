// calendar_groups.h -- device layout of a large calendar's logs (laq_calendar_groups.cuh).
#pragma once

#include "gpq_device.h"

namespace gpq {
namespace cal {

constexpr int kUnit = 512;               // LPs per unit: a commit workgroup's threads
constexpr uint32_t kUnitLog2 = 9;

constexpr uint32_t kMaxGroups = 256;     // a workgroup of the filing launch per CU

struct Groups {
  Event* wlog;                           // [units][B][log_cap]
  uint32_t* wlog_n;                      // [units][B]
  Event* out;                            // [units][passes][kUnitPass]
  uint32_t* parts;                       // [units][passes][kMaxGroups]
  uint32_t* npass;                       // [units]
  Event* over;                           // [groups][over_cap]
  uint32_t* over_n;                      // [groups], 16 words apart
  uint32_t units, groups, group_shift, log_cap, passes, over_cap;
};

}  // namespace cal
}  // namespace gpq
