// Dispatch rules of the row kernels that take any width (rows.hpp and the READ
// variants).  Host arithmetic alone, so that the CPU tests build it with g++
// (tests/cpp/row_rules_query.cpp).
#pragma once

#include <stdint.h>

namespace credit {
namespace rows {

// READ streams a row with one workgroup, of 256 lanes or, where `StreamRule`
// says so, of 1024: from `one` columns on with at most 256 rows (a row per CU),
// `two` with at most 512, `three` below 1024.  A narrower row leaves most of
// 1024 lanes idle and every reduction goes over 16 waves in place of 4; with
// more rows four small workgroups share a CU (LayerNorm backward 1023 x 1000:
// 5.8 us on 256 lanes, 12.3 on 1024; 700 x 6000: 24 and 18; 128 x 16384: 39 and
// 17).  The softmaxes, whose passes are longer, gain later (forward 700 x
// 12288: 17.8 and 18.7; backward 400 x 16384: 19.1 and 20.4, so never above 256
// rows).
struct StreamRule {
  int64_t one, two, three;
};
constexpr int64_t kNever = INT64_MAX;
constexpr StreamRule kStream{2048, 6144, 6144};
constexpr StreamRule kSoftmaxFwdStream{6144, 6144, 16384};
constexpr StreamRule kSoftmaxBwdStream{6144, kNever, kNever};
constexpr StreamRule kLogitsStream{2048, 4096, 6144};
inline int stream_threads(const StreamRule& rule, int64_t rows, int64_t cols) {
  const int64_t from = rows <= 256 ? rule.one : rows <= 512 ? rule.two
                                   : rows < 1024 ? rule.three : kNever;
  return cols >= from ? 1024 : 256;
}

}  // namespace rows
}  // namespace credit
