// calendar_groups.h -- device layout of a large calendar's logs (laq_calendar_groups.cuh).
#pragma once

#include "gpq_device.h"

namespace gpq {
namespace cal {

constexpr int kUnit = 512;               // LPs per unit: a commit workgroup's threads
constexpr uint32_t kUnitLog2 = 9;

constexpr uint32_t kMaxGroups = 256;     // a workgroup of the filing launch per CU

// A group's words: its events beyond the calendar, its part of the shared records (first and number),
// and whether that part is its own yet.
enum OverWord : uint32_t { kOverN = 0, kOverFrom = 1, kOverMore = 2, kOverShared = 3 };
constexpr uint32_t kOverWords = 16;

struct Groups {
  Event* wlog;                           // [units][B][log_cap]
  uint32_t* wlog_n;                      // [units][B]
  Event* out;                            // [units][passes][kUnitPass]
  uint32_t* parts;                       // [units][passes][kMaxGroups]
  uint32_t* npass;                       // [units]
  Event* over;                           // [groups][own_cap], then as many records shared by the groups
  uint32_t* over_n;                      // [groups], kOverWords apart: see OverWord
  uint32_t* spill_n;                     // before the start: initial events in the shared records
  uint32_t units, groups, group_shift, log_cap, passes, own_cap;
};

}  // namespace cal
}  // namespace gpq
