// Prints what the library's host-side dispatch rules say: one command a line on stdin, one answer a line.
#include <iostream>
#include <string>

#include "moe_gemm_device.h"
#include "moe_token.h"

int main() {
  std::string what;
  while (std::cin >> what) {
    if (what == "depth") {   // gate/up or down, list of short tiles only, row tiles, work items, rows
      int mode, short_only, tiles, items, rows;
      std::cin >> mode >> short_only >> tiles >> items >> rows;
      std::cout << moe_stream_depth(mode, short_only, tiles, items, rows) << "\n";
    } else {
      return 1;
    }
  }
}
