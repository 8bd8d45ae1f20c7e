// rnpx_cqr_layout.hpp -- what lies where in the outer-block kernel's scratch
// (rnpx_cqr.hip), in doubles.  Plain constants: a CPU test compiles this file.
#pragma once

namespace rnpx {
namespace blk {

constexpr int kHalf = 64 * 64;                     // a 64 x 64 block
constexpr int kPasses = 4;                         // Cholesky passes at most (and one first-order pass)
// R11, R12, R22 of each pass (workgroup 2)
constexpr int kR = 0, kRSize = 3 * kHalf * (kPasses + 1);
// the blocks that one workgroup publishes to the others
constexpr int kU1i = kR + kRSize, kU12 = kU1i + kHalf, kT1 = kU12 + kHalf, kU2i = kT1 + kHalf, kD1 = kU2i + kHalf,
              kD2 = kD1 + 64, kPublishedEnd = kD2 + 64;
// The column-wise refactorization's Gram and T (workgroup 0): a region of
// their own, since nothing orders them after workgroup 2's stores into kR -- a
// line of those that its cache writes back late would land on them.
constexpr int kGram = kPublishedEnd, kTFactor = kGram + 128 * 128;
// a column's row of the block on its way to every workgroup, two parities
constexpr int kRow = kTFactor + 128 * 128;
constexpr int kScratch = kRow + 2 * 128;

static_assert(kR + kRSize <= kU1i && kPublishedEnd <= kGram && kGram + 128 * 128 <= kTFactor &&
                  kTFactor + 128 * 128 <= kRow,
              "block scratch regions overlap");

}  // namespace blk
}  // namespace rnpx
