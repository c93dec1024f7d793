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

// The entry that rows_pick takes from the softmax tables' ladder: lanes * 100 +
// vectors a lane.
extern "C" int row_rules_pick(int64_t rows, int64_t cols) {
  static const RowsPick<int> ladder[] = {
      {6401, 64, 256, true},    {12801, 128, 512, true}, {25601, 256, 1024, true},
      {25602, 256, 2048, true}, {6404, 64, 1024},        {12804, 128, 2048},
      {25604, 256, 4096}};
  const RowsPick<int>* p = rows_pick(ladder, rows, cols);
  return p == nullptr ? 0 : p->fn;
}

// op: 0 softmax forward and logits backward, 1 softmax backward, 2 LayerNorm
// backward fp32, 3 and 4 bf16 LayerNorm of even and odd width.
extern "C" int row_rules_narrow(int op, int64_t rows, int64_t cols) {
  const NarrowRule* rules[] = {&kSoftmaxNarrow, &kSoftmaxBwdNarrow, &kLnBwdNarrow, &kLnHalfNarrow,
                               &kLnHalfOddNarrow};
  return narrow(*rules[op], rows, cols);
}

// op: 0 softmax forward, 1 its backward, 2 the logits backward, 3 quantisation,
// 4 LayerNorm forward, 5 and 6 its backward in fp32 and bf16.
extern "C" int row_rules_wide(int op, int64_t rows, int64_t cols, int vec) {
  const WideRule* rules[] = {&kSoftmaxFwdWide, &kSoftmaxBwdWide, &kLogitsWide, &kQuantWide,
                             &kLnFwdWide,      &kLnBwdWide,      &kLnBwdHalfWide};
  return wide(*rules[op], rows, cols, vec != 0);
}
