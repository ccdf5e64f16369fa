// Lays out SIR plans of many sizes (plan_layout.hpp) and prints how many have
// two parts in one line of 128 bytes, and how many are not 8-byte aligned.
#include <cstdio>
#include <initializer_list>

#include "plan_layout.hpp"

int main()
{
  long shared = 0, misaligned = 0;
  for (size_t probs = 1; probs < 70; probs++)
    for (size_t descriptor : {8, 256, 408, 472, 512})
      for (size_t table : {8, 1000, 4096}) {
        const dream::PlanLayout l = dream::plan_layout(probs * descriptor, probs * 16, 16, table * 8);
        shared += (probs * descriptor - 1) / 128 >= l.status / 128;
        shared += (l.status + probs * 16 - 1) / 128 >= l.counter / 128;
        shared += (l.counter + 16 - 1) / 128 >= l.tables / 128;
        misaligned += l.status % 8 || l.counter % 8 || l.tables % 8 || l.bytes != l.tables + table * 8;
      }
  std::printf("%ld %ld\n", shared, misaligned);
  return 0;
}
