"""The order of a causal grid whose workgroups are all resident at once (csrc/fa2_order.hpp), compiled for the host: every workgroup is
visited once, and no compute unit has much more work than the best split of the same workgroups over as many places."""

import ctypes
import heapq
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-flash-attn2_amd", "csrc")


@pytest.fixture(scope="module")
def position(tmp_path_factory):
	d = tmp_path_factory.mktemp("order")
	src, out = d / "order.cc", d / "order.so"
	src.write_text('#include "fa2_order.hpp"\nextern "C" int position(int i, int n, int w) { return fa2::resident_position(i, n, w); }\n')
	subprocess.check_call([os.environ.get("CXX", "c++"), "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(out), str(src)])
	f = ctypes.CDLL(str(out)).position
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
