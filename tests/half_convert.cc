// fp32 -> fp16 bits (half.h): floats on standard input, halfs on standard output.
#include <cstdio>

#include "half.h"

int main() {
  float f;
  while (std::fread(&f, 4, 1, stdin) == 1) {
    const uint16_t h = arthip::f32_to_f16(f);
    std::fwrite(&h, 2, 1, stdout);
  }
  return 0;
}
