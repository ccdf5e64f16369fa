// plan_layout.hpp -- where the parts of a SIR plan's one device buffer lie.
#pragma once

#include <cstddef>

namespace dream {

// Descriptors (from 0) | status blocks | counters | tables, each a whole line
// of 128 bytes or more from the next: the descriptors and tables are read by
// every work-group, the status and counters written by atomics, and reads of
// a line wait for the atomics on it (512 elements of 0.3 x 0.3 mm by 4096
// points, half of it out of range: 0.60 ms, in one line 1.3).
struct PlanLayout {
  size_t status, counter, tables, bytes;
};

inline PlanLayout plan_layout(size_t descriptor_bytes, size_t status_bytes, size_t counter_bytes,
                              size_t table_bytes)
{
  auto apart = [](size_t n) { return (n + 255) / 128 * 128; };
  PlanLayout l;
  l.status = apart(descriptor_bytes);
  l.counter = apart(l.status + status_bytes);
  l.tables = apart(l.counter + counter_bytes);
  l.bytes = l.tables + table_bytes;
  return l;
}

} // namespace dream
