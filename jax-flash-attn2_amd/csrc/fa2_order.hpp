// Order of the workgroups of a causal grid whose workgroups are all resident at once: which of them share a compute unit.
// (Plain C++: the host tests compile it as it is.)
#pragma once

#ifdef __HIP__
#define FA2_HD __host__ __device__ inline
#else
#define FA2_HD inline
#endif

namespace fa2 {

constexpr int kNumCULog2 = 8, kNumCU = 1 << kNumCULog2;  // compute units of the MI355X

// n workgroups, the longest first, on 1 << log2_width compute units: the position in that order of the workgroup that arrives as the i-th.  The first
// 1 << log2_width arrivals take the first place of every unit, the next as many the second place in the same order of units, and so on; what counts is the
// sum over the places of a unit.  Units that get nothing of a last layer that is not full hold the longest workgroups, and the order of units starts from them.  The first
// half of the layers follows it, the second half is visited backwards, so that the unit with the longest tiles of the first half gets the shortest of the second; of
// three layers the middle one is turned by half its width, and a third one that is full takes what makes the sum the same everywhere.
FA2_HD int resident_position(int i, int n, int log2_width) {
	const int width = 1 << log2_width, layer = i >> log2_width, layers = (n + width - 1) >> log2_width;
	const int base = layer << log2_width, last = n - ((layers - 1) << log2_width);
	int r = (i & (width - 1)) + width - last;
	if (r >= width) r -= width;
	if (layers == 3 && layer == 1) return base + ((r + width / 2) & (width - 1));
	if (layers == 3 && layer == 2 && last == width) return base + (r < width / 2 ? width - 1 - 2 * r : 2 * width - 2 - 2 * r);
	return base + (2 * layer < layers ? r : width - 1 - r);
}

}  // namespace fa2
