// The dispatch rules of the row kernels (credit_amd/csrc/row_rules.hpp) as
// tests/test_row_rules.py asks for them; built with g++.
#include "../../credit_amd/csrc/row_rules.hpp"

using namespace credit::rows;

// op: 0 LayerNorm and quantisation, 1 softmax forward, 2 its backward, 3 the
// logits backward.
extern "C" int row_rules_stream_threads(int op, int64_t rows, int64_t cols) {
  const StreamRule* rules[] = {&kStream, &kSoftmaxFwdStream, &kSoftmaxBwdStream, &kLogitsStream};
  return stream_threads(*rules[op], rows, cols);
}
