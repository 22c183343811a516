// Prints max_layers of a mesh given as records of 12 floats per face (stdin) and the
// smallest number of faces of a part.
//
// usage: layers_check <min_faces> < records

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../ugu_amd/csrc/bvh_build.h"

int main(int argc, char** argv) {
  std::vector<float> rec;
  float buf[12];
  while (std::fread(buf, 4, 12, stdin) == 12) rec.insert(rec.end(), buf, buf + 12);
  ugu_hip::BvhBuild b;
  if (argc != 2 || ugu_hip::build_bvh(rec.data(), int(rec.size() / 12), 31, &b) != 0) return 1;
  std::printf("%.6f\n", ugu_hip::max_layers(b, std::atoi(argv[1])));
  return 0;
}
