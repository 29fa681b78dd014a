// Sizes of the photon grid's buffers.  Plain host arithmetic, so that it can be checked at its
// limits without a device.
#pragma once

#include <cstddef>

namespace imba {

constexpr int kGridMaxPhotons = 1 << 29;

// Buckets of a build: max(previous size, 2 * count) (rangesearch/rangesearch.h:33-34).
constexpr int grid_table_size(int previous, int photons) { return previous > 2 * photons ? previous : 2 * photons; }

// 32-bit words of the buckets' boxes, six each (2^30 buckets: more than an int counts).
constexpr size_t grid_box_words(int table) { return 6 * (size_t)table; }

}  // namespace imba
