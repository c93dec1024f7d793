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
//
// A row without the 16-byte layout moves in vectors (at 4-byte addresses, its
// last elements by themselves) from `vectors` columns on, below that in single
// elements: a vector leaves three lanes of four idle there and the last
// elements take a step of their own (softmax forward 3000 x 257: 6.9 us in
// elements, 7.4 in vectors; backward 3000 x 1002: 7.6, 9.6).
struct StreamRule {
  int64_t one, two, three, vectors;
};
constexpr int64_t kNever = INT64_MAX;
constexpr StreamRule kStream{2048, 6144, 6144, 512};
constexpr StreamRule kSoftmaxFwdStream{6144, 6144, 16384, 512};
constexpr StreamRule kSoftmaxBwdStream{6144, kNever, kNever, 3072};
constexpr StreamRule kLogitsStream{2048, 4096, 6144, 512};
inline int stream_threads(const StreamRule& rule, int64_t rows, int64_t cols) {
  const int64_t from = rows <= 256 ? rule.one : rows <= 512 ? rule.two
                                   : rows < 1024 ? rule.three : kNever;
  return cols >= from ? 1024 : 256;
}

// Rows narrow enough, and few enough, that AUTO runs READ where it could hold
// them in registers: both corners' columns are exclusive, rows inclusive.  A
// row of a few elements shares its cache lines with other workgroups' rows, to
// which READ's plain stores do less harm than nontemporal ones, and 256 lanes
// take one element each without a loop (softmax backward 3000 x 3: 2.7 us, 3.6
// held; 1500 x 257: 2.7, 2.9; 8000 x 62: 4.7, 4.1; LayerNorm forward 300 x 7:
// 2.6, 3.3; 300 x 201: 2.7, 2.9; 3000 x 7: 5.2, 4.6).
struct NarrowRule {
  int64_t cols1, rows1, cols2, rows2;
};
constexpr NarrowRule kSoftmaxNarrow{8, 2048, 0, 0};  // forward and logits backward
constexpr NarrowRule kSoftmaxBwdNarrow{16, 12288, 512, 4096};
constexpr NarrowRule kLnBwdNarrow{8, 1024, 0, 0};       // fp32
constexpr NarrowRule kLnHalfNarrow{16, 2048, 64, 512};  // bf16, both directions
constexpr NarrowRule kLnHalfOddNarrow{16, 2048, 256, 512};
inline bool narrow(const NarrowRule& rule, int64_t rows, int64_t cols) {
  return (cols < rule.cols1 && rows <= rule.rows1) || (cols < rule.cols2 && rows <= rule.rows2);
}

// Few wide rows in two launches of chunks (widerows.hip), columns exclusive:
// ragged rows past `few` columns with up to kFewWide rows and past `many` with
// more, rows of whole 16-byte vectors past `vec`.
//
// Ragged rows of up to kFewWide rows leave most of the chip idle on a workgroup
// each: from 16384 columns on (8195: the same or 0.4 us slower; quantisation,
// one pass of a narrow output, from 32768; bf16 LayerNorm forward 16 x 16386 7.1
// us, 7.6 in chunks, 64 x 16387 9.6, 8.5).  More rows fill it, and the kernels
// that hold a row in registers read it once (softmax logits backward 256 x
// 40003: 30 us, 33.5 in chunks); past `many` columns they stream it more than
// once, or so few rows fit that latency shows (LayerNorm backward 384 x 40003:
// 76 us, 49).
//
// Rows of whole vectors have faster kernels, SPLIT among them: at most 32 rows,
// wide ones and little data (softmax logits backward 64 x 131072: 22 us, 27 in
// chunks).  One workgroup that holds the row is sooner done than two launches:
// softmax forward and logits backward up to 24576 columns (8 x 24584: 7.5 and
// 7.8 us, 6.1 and 6.2 in chunks), softmax backward up to 32768 (8 x 24584: 4.9, 6.0;
// 8 x 36864, SPLIT: 8.1, 6.0), quantisation up to 65536 (16 x 65536: 6.4, 7.0;
// 16 x 65544, SPLIT: 7.8, 5.9), LayerNorm forward up to 57344 (24 x 49160: 6.6,
// 7.2; 16 x 65536: 7.2, 7.1), its bf16 backward up to 49152.  16 x 262144 would
// gain too (softmax forward 13.4, 9.9) but AUTO is known to run SPLIT there
// (credit_last_split_shape).
struct WideRule {
  int64_t few, many, vec;
};
constexpr int64_t kWideMaxRows = 2048;
constexpr int64_t kFewWide = 128;
constexpr WideRule kSoftmaxFwdWide{16384, 32768, 24576};
constexpr WideRule kSoftmaxBwdWide{16384, 53248, 32768};
constexpr WideRule kLogitsWide{16384, 53248, 24576};
constexpr WideRule kLnBwdWide{16384, 32768, 24576};
constexpr WideRule kLnBwdHalfWide{16384, 32768, 49152};
constexpr WideRule kLnFwdWide{20480, 32768, 57344};
constexpr WideRule kQuantWide{32768, 65536, 65536};
inline bool wide(const WideRule& rule, int64_t rows, int64_t cols, bool vec) {
  if (rows > kWideMaxRows) return false;
  if (vec) return rows <= 32 && cols > rule.vec && rows * cols <= int64_t{1} << 21;
  return cols > (rows <= kFewWide ? rule.few : rule.many);
}

// A kernel that holds a ragged row in one workgroup's registers (rows.hpp).
template <class Fn>
struct RowsPick {
  Fn fn;
  int threads;
  int64_t capacity;  // elements
  bool few = false;  // for at most kFewRows rows, unless it is one wave
};

// The first entry that holds `cols`; nullptr: none.  A lone row's time is its
// lanes' serial work, so the tables open with narrow rows spread over many
// lanes, taken up to kFewRows rows (softmax logits backward 1 x 1134: 4.5 ->
// 3.4 us a call); with more, fewer lanes of more vectors keep more rows in
// flight (softmax forward 16384 x 770: 20.6 us on 64 lanes, 25.2 on 256).  One
// wave of one vector a lane is the least there is: rows that fit it take it at
// any number (20000 x 62, us a call, against four vectors a lane: softmax
// forward 17.8 -> 11.1, backward 12.9 -> 6.4, LayerNorm forward 23.3 -> 11.3).
constexpr int64_t kFewRows = 2048;
constexpr int kWaveLanes = 64;
template <class Fn, int N>
const RowsPick<Fn>* rows_pick(const RowsPick<Fn> (&table)[N], int64_t rows, int64_t cols) {
  for (const RowsPick<Fn>& p : table)
    if (cols <= p.capacity && (rows <= kFewRows || !p.few || p.threads == kWaveLanes)) return &p;
  return nullptr;
}

}  // namespace rows
}  // namespace credit
