// The spring chains' class rules (csrc/de_spring_classes.h) on the host.  Reads lines
// "dopri5 n size count size count ..." and prints the set of classes that a launch of
// those systems uses.
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
