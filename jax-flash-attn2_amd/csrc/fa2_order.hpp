// Order of the workgroups of a grid.  (Plain C++: the host tests compile it as it is.)
#pragma once
#include <cstdint>

#ifdef __HIP__
#define FA2_HD __host__ __device__ inline
#else
#define FA2_HD inline
#endif

namespace fa2 {

constexpr int kNumCULog2 = 8, kNumCU = 1 << kNumCULog2;  // compute units of the MI355X

// A causal grid whose workgroups are all resident at once: which of them share a compute unit.
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

// The i-th of the workgroups of `groups` groups of `heads` heads with `tiles` row tiles each, where `together` groups advance through their row tiles
// together (the last ones may be fewer): its group, its place in the order of row tiles and its head.
struct Place {
	int group, tile, head;
};
FA2_HD Place place_of(int i, int groups, int heads, int tiles, int together) {
	const int first = i / (together * tiles * heads) * together, e = groups - first < together ? groups - first : together;
	const int rem = i - first * tiles * heads, in_tile = rem % (e * heads);
	return {first + in_tile / heads, rem / (e * heads), in_tile % heads};
}

// Groups that advance together on a causal grid of `wgs` workgroups of head dim 64, four waves a SIMD, that are not all resident.  Group by group the longest row tiles
// of the later groups start late, and the launch waits for them: the more workgroups share a CU, the longer, so that grids of four to eight a CU were slower than with two.
// Up to eight a CU all groups (of the XCD, where they are placed by XCD) advance together, as long as the K and V of those of an XCD are
// within four times its L2; beyond, the tail is short, and it is enough that as many do as a round of the chip holds.  Two a CU / group by group / now:
// B2 Hq32 Hkv8 S3000 100 / 111 / 87 us, B4 Hq32 Hkv8 S2000 98 / 103 / 80, B2 H24 S3000 95 / 100 / 77, B8 H16 S1200 with dropout 82 / 90 / 59; groups not by XCD, B1 Hq36 Hkv12
// S5000 197 / 190 / 136.  Larger grids, group by group / 4 / 8 / 16 / all of an XCD: B16 H16 S4096 644 / 620 / 611 / 623 / 668, B64 H16 S1024 227 / 209 / 208 / 210 / 255,
// B8 H16 S8192 1193 / 1143 / 1174 / 1198 / 1204; not by XCD, 4 / 16 / 64 / all: B65 H12 S1024 234 / 194 / 166 / 162 / 177, B17 H12 S4096 696 / 540 / 506 / 506 / 527,
// B9 Hq28 Hkv7 S4096 657 / 614 / 606 / 651 / 651.
inline int groups_together(int groups, int heads, bool by_xcd, int64_t wgs, int64_t kv_bytes) {
	if (wgs <= 8 * kNumCU && (!by_xcd || groups * kv_bytes <= (16 << 20))) return groups;
	const int most = by_xcd ? (kv_bytes <= (1 << 20) ? 8 : 4) : heads < 16 ? 64 / heads : 4;
	const int parts = (groups + most - 1) / most;
	return (groups + parts - 1) / parts;
}

}  // namespace fa2
