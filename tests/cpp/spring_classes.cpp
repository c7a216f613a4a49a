// The spring chains' class rules (csrc/de_spring_classes.h) on the host.  Reads lines
// "dopri5 n size count size count ..." and prints the set of classes that a launch of
// those systems uses; "shape masses lanes" prints the lanes and masses per lane of
// DE_MAP_GROUP with that group_size.
#include <stdio.h>

#include <sstream>
#include <iostream>
#include <string>
#include <vector>

#include "../../differential-equations_amd/csrc/de_spring_classes.h"

using namespace de::parity;

int main() {
  for (std::string line; std::getline(std::cin, line);) {
    std::istringstream in(line);
    if (line.rfind("shape", 0) == 0) {
      std::string word;
      int masses = 0, lanes = 0;
      in >> word >> masses >> lanes;
      const ClassSet cs = class_set(true);
      const LaneShape sh = group_shape(cs.caps[class_index(cs, masses)], lanes);
      printf("%d %d\n", sh.g, sh.c);
      continue;
    }
    int dopri5 = 0, size = 0;
    long long n = 0;
    in >> dopri5;
    const ClassSet cs = class_set(dopri5 != 0);
    std::vector<int64_t> count(cs.n, 0);
    while (in >> size >> n) count[class_index(cs, size)] += n;
    static const char* names[] = {"all", "mid", "few"};
    printf("%s\n", names[merge_of(dopri5 != 0, count.data())]);
  }
}
