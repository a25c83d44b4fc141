// Prints what the library's host-side dispatch rules say: one command a line on stdin, one answer a line.
#include <iostream>
#include <string>
#include <vector>

#include "moe_gemm_device.h"
#include "moe_small.h"
#include "moe_token.h"

int main() {
  std::string what;
  while (std::cin >> what) {
    if (what == "depth") {   // gate/up or down, list of short tiles only, row tiles, work items, rows
      int mode, short_only, tiles, items, rows;
      std::cin >> mode >> short_only >> tiles >> items >> rows;
      std::cout << moe_stream_depth(mode, short_only, tiles, items, rows) << "\n";
    } else if (what == "tile_rows") {   // rows, groups, most rows of a group; column blocks, K steps of gate/up and down; dense rows and column blocks
      TileShape t;
      std::cin >> t.R >> t.E >> t.max_rows >> t.ncb[0] >> t.ncb[1] >> t.kb[0] >> t.kb[1] >> t.dense_rows >> t.dense_ncb[0] >> t.dense_ncb[1];
      std::cout << moe_gemm_tile_rows(t) << "\n";
    } else if (what == "down_list") {   // tokens, D, experts, k, I, SI: rows of a full tile of the lists, gate/up's and the down GEMM's own (or 0)
      int M, D, E, k, I, SI;
      std::cin >> M >> D >> E >> k >> I >> SI;
      const TileShape t{M * k, E, M, {I / 128, (D + 255) / 256}, {D / 128, I / 128}, SI ? M : 0, {SI / 128, (D + 255) / 256}};
      std::cout << moe_gemm_tile_rows(t) << " " << moe_gemm_down_tile_rows(t, moe_gemm_tile_rows(t)) << "\n";
    } else if (what == "scales") {   // tokens, D, experts, k, I, forked: whether gate/up's activation scales are gathered, and by the placing launch
      int M, D, E, k, I, forked;
      std::cin >> M >> D >> E >> k >> I >> forked;
      const ScalePlan p = moe_scale_plan(M * k, E, D, I, forked);
      std::cout << p.gathered << " " << p.placed << "\n";
    } else if (what == "scan") {   // tokens, D, experts, k, I, SI: rows of a full tile where the GEMMs read the selection, or 0
      int M, D, E, k, I, SI;
      std::cin >> M >> D >> E >> k >> I >> SI;
      const TileShape t{M * k, E, M, {I / 128, (D + 255) / 256}, {D / 128, I / 128}, SI ? M : 0, {SI / 128, (D + 255) / 256}};
      std::cout << moe_gemm_scan_rows(t, moe_gemm_from_memory(((long long)E * I + SI) * D)) << "\n";
    } else if (what == "small") {   // tokens, D, experts, k, I, SI: selections a lane of a small layer's down launch holds, or 0
      int M, D, E, k, I, SI;
      std::cin >> M >> D >> E >> k >> I >> SI;
      std::cout << moe_small_down_lanes(M, D, E, k, I, SI) << "\n";
    } else if (what == "token") {   // tokens, D, experts, k, I, SI
      int M, D, E, k, I, SI;
      std::cin >> M >> D >> E >> k >> I >> SI;
      std::cout << moe_token_takes(M, D, E, k, I, SI) << "\n";
    } else if (what == "token_routes" || what == "token_selected") {   // tokens, D, experts, k, I, SI: whether the first launch routes ready logits, or takes a selection
      int M, D, E, k, I, SI;
      std::cin >> M >> D >> E >> k >> I >> SI;
      std::cout << moe_token_routes(M, D, E, k, I, SI, what == "token_selected") << "\n";
    } else if (what == "token_chain") {   // the same of ready logits by the steps of their selection: routing, groups, kept groups
      int M, D, E, k, I, SI, routing, n_group, topk_group;
      std::cin >> M >> D >> E >> k >> I >> SI >> routing >> n_group >> topk_group;
      std::cout << moe_token_routes(M, D, E, k, I, SI, false, moe_token_chain(routing, E, k, n_group, topk_group)) << "\n";
    } else if (what == "token_fronts") {   // tokens, D, experts, k, I, SI, norm: whether it takes a small router too
      int M, D, E, k, I, SI, norm;
      std::cin >> M >> D >> E >> k >> I >> SI >> norm;
      std::cout << moe_token_fronts(M, k, I, SI, norm, moe_gemm_from_memory(((long long)E * I + SI) * D)) << "\n";
    } else if (what == "token_router") {   // the same of that router, with a column for the shared expert's gate
      int M, D, E, k, I, SI, norm;
      std::cin >> M >> D >> E >> k >> I >> SI >> norm;
      std::cout << moe_token_fronts(M, k, I, SI, norm, moe_gemm_from_memory(((long long)E * I + SI) * D), (E + (SI > 0)) * D) << "\n";
    } else if (what == "stages") {   // tokens, D, experts, k, I, SI: K steps of a stage in the two launches of single tokens
      int M, D, E, k, I, SI;
      std::cin >> M >> D >> E >> k >> I >> SI;
      const TokenStages st = moe_token_stages(M, D, k, I, SI, moe_gemm_from_memory(((long long)E * I + SI) * D));
      std::cout << st.gateup << " " << st.down << "\n";
    } else if (what == "down") {   // tokens, D, k, I, SI: tiles and waves of a workgroup, and whether LDS sets the waves
      int M, D, k, I, SI;
      std::cin >> M >> D >> k >> I >> SI;
      const TokenDownPlan p = moe_token_down_plan(M, D, k, I, SI);
      std::cout << p.tiles << " " << p.waves << " " << (p.waves < 16 && p.waves < k + (SI > 0)) << "\n";
    } else if (what == "memory") {   // experts, D, I, SI of a layer
      long long E, D, I, SI;
      std::cin >> E >> D >> I >> SI;
      std::cout << moe_gemm_from_memory((E * I + SI) * D) << "\n";
    } else if (what == "voted") {   // rows of a full tile of a list that may have tall ones: groups, then the rows of each
      int E, R = 0, votes = 0;
      std::cin >> E;
      std::vector<int> rows(E);
      for (int& r : rows) std::cin >> r, R += r;
      for (int r : rows) votes += moe_tall_vote(r, moe_tall_tiles(R, E));
      std::cout << moe_tile_rows_voted(kTallTileRows, votes) << "\n";
    } else if (what == "both") {   // routed rows without a list beside a dense group: refused before any GPU call
      alignas(256) static unsigned char memory[1 << 16];
      const float* f = (const float*)memory;
      const GemmOperands op{memory, f, nullptr, memory, f, memory, f, 256, 256, memory, (float*)memory, moe_row_major_scales(256, 256)};
      const RoutedGemm routed{op, (const int32_t*)memory, 8, 64, memory, sizeof memory, 0, 0};
      const DenseGemm dense{op, 64};
      std::cout << moe_gemm_gateup_impl(&routed, &dense, nullptr) << " " << moe_gemm_down_impl(&routed, &dense, nullptr) << " " << moe_last_error() << "\n";
    } else if (what == "front") {   // tokens, D, experts, columns, whether a norm, f32 input, a sort
      int M, D, E, N;
      bool norm, x_f32, sorted;
      std::cin >> M >> D >> E >> N >> norm >> x_f32 >> sorted;
      std::cout << moe_front_takes(M, D, E, N, norm, x_f32, sorted) << "\n";
    } else if (what == "routing") {   // tokens, D, experts: what moe_routing refuses before any GPU call
      int M, D, E;
      std::cin >> M >> D >> E;
      alignas(256) static unsigned char memory[256];
      std::cout << moe_routing(memory, M, D, memory, E, 1, 1, (int32_t*)memory, (float*)memory, memory, ~(size_t)0, nullptr) << " " << moe_last_error() << "\n";
    } else {
      return 1;
    }
  }
}
