"""The orders of a grid's workgroups (csrc/fa2_order.hpp), compiled for the host.  Of a causal grid whose workgroups are all resident at once: every workgroup is
visited once, and no compute unit has much more work than the best split of the same workgroups over as many places.  Of groups that advance together: each
workgroup once, the longest first, and as many groups at a time as the rule says."""

import ctypes
import heapq
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-flash-attn2_amd", "csrc")


SRC = """
#include "fa2_order.hpp"
extern "C" int position(int i, int n, int w) { return fa2::resident_position(i, n, w); }
extern "C" void place(int i, int groups, int heads, int tiles, int together, int* out) {
	const fa2::Place p = fa2::place_of(i, groups, heads, tiles, together);
	out[0] = p.group, out[1] = p.tile, out[2] = p.head;
}
extern "C" int together(int groups, int heads, int by_xcd, long long wgs, long long kv_bytes) { return fa2::groups_together(groups, heads, by_xcd, wgs, kv_bytes); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
	d = tmp_path_factory.mktemp("order")
	src, out = d / "order.cc", d / "order.so"
	src.write_text(SRC)
	subprocess.check_call([os.environ.get("CXX", "c++"), "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(out), str(src)])
	return ctypes.CDLL(str(out))


@pytest.fixture(scope="module")
def position(lib):
	f = lib.position
	f.argtypes, f.restype = [ctypes.c_int] * 3, ctypes.c_int
	return f


@pytest.mark.parametrize("log2_width", [5, 8])
def test_every_workgroup_once(position, log2_width):
	width = 1 << log2_width
	for n in range(width + 1, 4 * width + 1):
		assert sorted(position(i, n, log2_width) for i in range(n)) == list(range(n))


def _loads(position, B, Hq, Hkv, S):
	"""Tiles of 64 keys per compute unit (and one for a workgroup's start and end): ours, and the longest workgroup to the idlest unit that has a place left."""
	mtiles = (S + 127) // 128
	n, width, log2_width = mtiles * B * Hq, 256, 8
	if B * Hkv % 8 == 0:  # an XCD's share
		n, width, log2_width = n // 8, 32, 5
	work = [(min(128 * (mtiles - j // (n // mtiles)), S) + 63) // 64 + 1 for j in range(n)]
	ours = [0] * width
	for i in range(n):
		ours[i % width] += work[position(i, n, log2_width)]
	places = (n + width - 1) // width
	heap, best = [(0, 0)] * width, []
	for x in work:
		load, used = heapq.heappop(heap)
		best.append(load + x)
		if used + 1 < places:
			heapq.heappush(heap, (load + x, used + 1))
	return max(ours), max(best), sum(work) / width


@pytest.mark.parametrize(
	"B,Hq,Hkv,S",
	[(1, 16, 4, 6000), (1, 16, 4, 5000), (3, 16, 4, 2000), (1, 36, 12, 3000), (3, 16, 16, 1500), (2, 24, 24, 1500), (1, 24, 12, 4328), (6, 8, 8, 1322), (9, 3, 3, 2348)]
	+ [(B, Hkv * r, Hkv, S) for Hkv in (4, 8, 12, 16) for r in (1, 4) for S in (257, 700, 1500, 4000) for B in (1, 2, 3, 5, 8, 13, 21) if 256 < (S + 127) // 128 * B * Hkv * r <= 1024],
)
def test_no_unit_has_much_more_than_its_share(position, B, Hq, Hkv, S):
	ours, best, mean = _loads(position, B, Hq, Hkv, S)
	# (mean: where it is beyond any split, the longest workgroups alone are; three places of which the last is taken by a few are the worst of the rule)
	assert ours <= 1.2 * max(best, mean), (ours, best, mean)


@pytest.mark.parametrize("groups,heads,tiles,together", [(1, 1, 1, 1), (5, 1, 7, 1), (5, 3, 7, 2), (7, 4, 3, 7), (135, 1, 2, 8), (17, 2, 9, 6), (8, 8, 5, 3)])
def test_groups_that_advance_together(lib, groups, heads, tiles, together):
	out, seen, last = (ctypes.c_int * 3)(), set(), (0, 0)
	for i in range(groups * heads * tiles):
		lib.place(i, groups, heads, tiles, together, out)
		group, tile, head = out
		assert 0 <= group < groups and 0 <= tile < tiles and 0 <= head < heads
		seen.add((group, tile, head))
		at = (group // together, tile)  # each block of groups from its longest tiles down
		assert at >= last
		last = at
	assert len(seen) == groups * heads * tiles


def test_how_many_advance_together(lib):
	def f(groups, heads, by_xcd, wgs, kv_bytes):
		return lib.together(groups, heads, int(by_xcd), ctypes.c_longlong(wgs), ctypes.c_longlong(kv_bytes))

	# up to eight workgroups a CU: all, of an XCD as long as their K and V are within 16 MiB
	assert f(780, 1, False, 2048, 1 << 22) == 780 and f(16, 1, True, 2048, 1 << 20) == 16 and f(16, 1, True, 2048, (1 << 20) + 1) == 4
	# beyond: evened out
	assert f(780, 1, False, 2049, 1 << 18) == 60 and f(9, 1, True, 2049, 1 << 20) == 5 and f(9, 1, True, 2049, 2 << 20) == 3 and f(63, 4, False, 8000, 1 << 20) == 16
	for groups in range(1, 200):
		for heads in (1, 2, 4, 8, 16, 64):
			for by_xcd in (False, True):
				for wgs in (300, 2048, 2049, 1 << 20):
					assert 1 <= f(groups, heads, by_xcd, wgs, 3 << 19) <= groups
