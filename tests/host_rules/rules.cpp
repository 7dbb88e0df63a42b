// Prints what the launch rules choose: one question a line on stdin, one answer a line on stdout.
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "launch_rules.hpp"

int main() {
  std::string line;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    std::string rule;
    in >> rule;
    if (rule == "pieces") {
      int64_t rows, threads;
      in >> rows >> threads;
      fo::for_row_pieces(rows, threads, [](int64_t first, int64_t count) { std::printf("%lld+%lld ", (long long)first, (long long)count); });
      std::printf("\n");
    } else if (rule == "attention") {
      int64_t heads, seq;
      int causal;
      in >> heads >> seq >> causal;
      const char* names[] = {"2x4", "4x2", "256"};
      std::printf("%s\n", names[(int)fo::attention_form(heads, seq, causal != 0)]);
    } else if (rule == "gemm") {
      std::string type;
      int64_t batch, m, n, k;
      in >> type >> batch >> m >> n >> k;
      std::printf("%d\n", (int)fo::gemm_tile(m, n, k, batch, type == "bf16" ? 2 : 1, type == "f8"));
    } else if (rule == "gemm_any") {
      std::string type;
      int64_t batch, m, n, k;
      in >> type >> batch >> m >> n >> k;
      std::printf("%d\n", fo::gemm_any_tile(m, n, k, batch, type == "i8"));
    } else if (rule == "mlp") {
      int64_t batch, in_f, hidden, out_f;
      int split;
      in >> batch >> in_f >> hidden >> out_f >> split;
      const char* names[] = {"thread", "split", "rows"};
      std::printf("%s\n", names[(int)fo::mlp_form(batch, in_f, hidden, out_f, split != 0)]);
    } else if (rule == "gemv") {
      int64_t n, k;
      in >> n >> k;
      std::printf("%d\n", fo::gemv_cells(n, k));
    } else if (rule == "norm") {
      int64_t rows, cols;
      in >> rows >> cols;
      std::printf("%s\n", fo::norm_dma(rows, cols) ? "dma" : "row");
    } else {
      return 1;
    }
  }
  return 0;
}
