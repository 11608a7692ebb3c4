// Which form of workgroup the forward takes at head dim 64 without bias, by the sizes of the call.  (Plain C++: the host tests compile it as it is.)
#pragma once
#include <cstdint>

#include "fa2_order.hpp"

namespace fa2 {

// Keys that a tile of 128 rows looks at, at most.
inline int64_t fwd_seen_keys(int Sk, int win_left, int win_right) {
	const int64_t w = (int64_t)win_left + win_right + 128;
	return win_left >= 0 && win_right >= 0 && w < Sk ? w : Sk;
}

// A window that hides no key, or less than a third of them, leaves the row tiles about as uneven as no window.  Such grids are laid out and split like those without
// one: causal, B4 H16 S892 in a window of 1728 keys 24.2 -> 20.5 us, B3 Hq32 Hkv8 S1063 of 4444 39.2 -> 30.4, B2 Hq24 Hkv12 S2409 of 1815 66.8 -> 53.5.
inline bool window_is_open(int Sk, int win_left) { return win_left < 0 || 3 * (int64_t)win_left >= 2 * (int64_t)Sk; }

struct FwdForm {
	int groups;  // of four waves in a workgroup, which take its key tiles in turn
	int waves;   // a SIMD (the launch bound)
};

// Head dim 64 without bias, workgroups of 128 rows, block by block.
inline FwdForm fwd_form_64(int B, int Hq, int Hkv, int Sq, int Sk, bool causal, int win_left, int win_right, bool drop) {
	const int64_t wgs = ((int64_t)Sq + 127) / 128 * B * Hq, seen = fwd_seen_keys(Sk, win_left, win_right);
	// At most one a CU: two groups from four tiles on (B2 Hq16 Hkv4 S512 causal 10.8 -> 10.0 us, S256 of B4 8.2 -> 8.0), three from seventeen (B1 Hq16 Hkv4 S2000
	// 29.9 -> 28.4; at S1024 and below 1 to 6 % slower than two).  Four take 128 registers a wave and spill.
	if (wgs <= kNumCU) {
		if (seen > 16 * 64) return {3, 3};
		if (seen > 3 * 64) return {2, 2};
		return {1, 4};
	}
	// Four waves a SIMD: four such workgroups a CU, or two of two groups each where the grid has no more than that (over
	// ten tiles and more; B4 Hq16 Hkv4 S1000 29.3 -> 28.4 us against 30.2 with one group, causal 23.9 -> 21.6 against 24.9; at S400 14.0 -> 12.8 with one, 15.0
	// with two) or seventeen of a window (B1 Hq16 Hkv4 S4000, 1024 keys a row 29.3 -> 28.4 against 29.5, 512 keys 20.3 -> 21.5 against 20.0).
	const bool open = window_is_open(Sk, win_left);
	if (wgs <= 2 * kNumCU && Sk > 9 * 64 && (open || seen > 16 * 64)) return {2, 4};
	// ... and where a causal grid would wait for its longest tiles, of more than 32 tiles of keys, which two groups go through in half the steps.  Two of one group a CU (the tile
	// body) / four of one group / two of two groups: B1 Hq32 Hkv8 S2200 45.5 / 47.3 / 37.9 us, S3000 61 / 67 / 53, B1 Hq16 Hkv8 S7000 140 / 158 / 122, B2 Hq16 Hkv4 S3700 76 / 87 / 72,
	// B1 Hq24 Hkv12 S4328 121 / 97 / 77, B1 Hq16 Hkv4 S6000 141 / 128 / 100; at four a CU B1 Hq32 Hkv16 S3973 88 / 97 / 83, B1 Hq32 Hkv8 S4096 90 / 83 / 85.  With dropout four of one
	// group are faster up to there (S3973 152 / 127 / 133).  Up to five and a half a CU more than 64 tiles: B1 Hq32 Hkv8 S4200 94 / 105 / 89, B1 Hq16 Hkv8 S9000 200 / 224 / 189, with
	// dropout 350 / 355 / 315, S11000 281 / 290 / 273, B1 Hq32 Hkv8 S5700 (5.6 a CU) 157 / 155 / 156, S6000 170 / 166 / 170; but B2 H24 S3200 89 / 75 / 81, B4 H16 S2400 67 / 57 / 65.
	const bool chain = causal && open && 8 * (int64_t)Sq >= 7 * (int64_t)Sk;
	if (chain && wgs <= 4 * kNumCU && Sk > 2048 && !drop) return {2, 4};
	if (chain && wgs > 4 * kNumCU && 2 * wgs <= 11 * kNumCU && Sk > 4096) return {2, 4};
	return {1, 4};
}

}  // namespace fa2
