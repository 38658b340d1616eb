// Launch arithmetic of the kernels, plain C++.
#pragma once

#include <algorithm>
#include <cstdint>

namespace pxh {

// Blocks of a launch over `items`, `perBlock` of them a block, at most `most` (the
// kernel strides over the rest). The items are a buffer's capacity, up to 2^31 - 1,
// so nothing is multiplied, and the sum is made in 64 bits.
inline int strideBlocks(int64_t items, int perBlock, int most)
{
	return int(std::min<int64_t>((items + perBlock - 1) / perBlock, most));
}

}  // namespace pxh
