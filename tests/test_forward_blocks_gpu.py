"""The forward block by block (head dim 64, and rows of 72 to 96 columns), three and four workgroups a CU: grids whose workgroups are all resident at
once and whose parts are visited backwards, two and three groups of waves on the keys of a row tile, ragged blocks of keys."""

import ctypes

import pytest
import torch

from jax_flash_attn2 import _hip_op as op
from jax_flash_attn2 import _lib
import fa2_oracle as O
from _cases import check_forward, f64, make_inputs

pytestmark = pytest.mark.gpu
BF, FP = torch.bfloat16, torch.float16


def _check(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, window, p, ranges=None, qk_scale=None):
	"""ranges: into how many parts the keys of a row tile are meant to be cut (0: the call is meant to run unsplit)."""
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq + Sk, qk_scale=qk_scale)
	kw = dict(causal=causal, kv_lens=lens, window=window, p_drop=p, seed=5)
	q_, k_, v_ = q.cuda(), k.cuda(), v.cuda()
	kl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda:0")
	if ranges is not None:
		n = _lib.load().fa2_fwd_scratch_bytes(ctypes.byref(op._block(D, q_, k_, v_, None, None, 1.0, p, causal, 5, kl, window)))
		assert n == (ranges * B * Hq * Sq * (D + 1) * 4 + 255) // 256 * 256
	o, lse = op.fwd(q_, k_, v_, None, None, None, p, causal, 5, kl, window)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), None, **kw)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} qk_scale={qk_scale} {kw}")


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,lens,window,p",
	[
		# causal grids that are all resident: 264 workgroups (two layers), 768 (three whole ones, twice), 700 and 610 (the last one short), 1024 (four); by XCD and not
		(2, 300, 300, 44, 11, 64, BF, True, None, None, 0.0),
		(8, 130, 130, 48, 6, 64, FP, True, None, None, 0.0),
		(8, 257, 257, 32, 4, 64, BF, True, None, None, 0.0),
		(5, 600, 600, 28, 7, 64, BF, True, None, None, 0.0),
		(4, 250, 300, 128, 8, 64, BF, True, None, None, 0.0),
		(6, 250, 250, 64, 16, 80, FP, True, None, None, 0.0),
		(5, 129, 129, 61, 61, 96, BF, True, None, None, 0.0),
		# ... in a window that hides less than a third of the keys, or none
		(5, 600, 600, 28, 7, 64, FP, True, None, (400, 0), 0.0),
		(5, 257, 257, 40, 8, 64, BF, True, None, (1000, 0), 0.1),
		(5, 250, 300, 64, 16, 88, BF, True, None, (200, 0), 0.0),
		# causal grids that are not: all groups advance together (by XCD and not), or as many as leave the last ones fewer
		(8, 600, 600, 32, 8, 64, FP, True, None, None, 0.0),
		(9, 600, 600, 28, 7, 64, BF, True, None, None, 0.1),
		(9, 600, 600, 28, 7, 64, BF, True, None, (500, 0), 0.0),
		(36, 130, 130, 30, 30, 64, BF, True, None, None, 0.0),
		(35, 130, 140, 30, 30, 64, FP, True, None, None, 0.0),
		(63, 130, 130, 20, 5, 64, BF, True, None, None, 0.0),
		# two groups of waves a workgroup, two workgroups a CU: ten tiles and more
		(2, 600, 590, 30, 10, 64, FP, True, None, None, 0.0),
		(2, 300, 640, 48, 16, 64, BF, False, [640, 65], None, 0.1),
		# ... and causal grids of up to four a CU over more than 32 tiles: the shortest, more keys than rows, four a CU
		(1, 2049, 2049, 32, 8, 64, BF, True, None, None, 0.0),
		(1, 2100, 2200, 56, 8, 64, FP, True, None, None, 0.0),
		(1, 4033, 4033, 32, 16, 64, BF, True, None, None, 0.0),
		# more than two workgroups a CU: blocks of keys that only some rows see, lengths, a window, rows without keys, one key
		(9, 257, 257, 20, 20, 80, FP, False, None, None, 0.0),
		(9, 200, 97, 32, 8, 72, BF, True, [97, 96, 64, 33, 32, 31, 1, 0, 97], None, 0.0),
		(9, 300, 300, 20, 5, 88, FP, True, None, (70, 0), 0.0),
		(9, 300, 300, 20, 5, 64, BF, True, None, (33, 0), 0.0),
		(70, 33, 1, 16, 2, 64, FP, False, None, None, 0.0),
		(40, 65, 129, 30, 6, 64, BF, False, None, None, 0.2),
	],
)
def test_blocks(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, window, p):
	_check(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, window, p)


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,dtype,causal,lens,window,p",
	[
		# head dim 64, at most one workgroup a CU, keys in one range: one group of waves (three tiles), two (four, five, sixteen), three (seventeen and more)
		(1, 130, 192, 3, 1, BF, False, None, None, 0.0),
		(1, 130, 193, 3, 1, BF, False, None, None, 0.0),
		(2, 300, 257, 2, 2, FP, True, None, None, 0.0),
		(2, 900, 1024, 14, 7, BF, True, None, None, 0.0),
		(2, 900, 1025, 14, 7, FP, True, None, None, 0.0),
		(1, 2000, 2000, 16, 4, BF, True, None, None, 0.0),
		# ... the same without a causal mask, with dropout
		(2, 900, 1025, 14, 7, BF, False, None, None, 0.0),
		(1, 1100, 1024, 16, 16, FP, True, None, None, 0.1),
		(1, 1100, 1025, 16, 16, FP, True, None, None, 0.1),
		(1, 1100, 1150, 16, 16, BF, False, None, None, 0.2),
		# ... rows without keys; lengths that leave the second, or the third, of three groups without a tile
		(2, 1200, 1200, 12, 4, BF, True, [1200, 0], None, 0.0),
		(2, 900, 1025, 14, 7, FP, False, [64, 65], None, 0.0),
		(2, 900, 1025, 14, 7, BF, False, [128, 129], None, 0.1),
		# ... windows of which a row tile sees three, four, sixteen and seventeen tiles' keys, and one that begins in the middle
		(2, 450, 450, 2, 1, BF, True, None, (64, 0), 0.0),
		(2, 450, 450, 2, 1, BF, True, None, (65, 0), 0.0),
		(2, 1300, 1300, 2, 1, FP, True, None, (896, 0), 0.0),
		(2, 1300, 1300, 2, 1, FP, True, None, (897, 0), 0.0),
	],
)
def test_groups_of_waves_on_a_range_of_keys(B, Sq, Sk, Hq, Hkv, dtype, causal, lens, window, p):
	assert (Sq + 127) // 128 * B * Hq <= 256
	_check(B, Sq, Sk, Hq, Hkv, 64, dtype, causal, lens, window, p, ranges=0)


@pytest.mark.parametrize(
	"Sq,Sk,Hq,Hkv,D,dtype,causal,ranges",
	[
		# head dim 64: workgroups that share a CU
		(700, 5000, 16, 4, 64, BF, True, 5),
		# head dim 128, four waves a workgroup and two workgroups a CU (these are 384 to 512 in all): two ranges, three, of which the last ends with one key in its last
		# tile, and five, of which the first rows see no key of the last
		(1000, 5700, 24, 8, 128, BF, True, 2),
		(600, 2945, 32, 8, 128, FP, False, 3),
		(1500, 6200, 8, 2, 128, BF, True, 5),
		(1100, 4097, 10, 5, 128, FP, True, 5),
		# ... and of eight waves, one a CU
		(1500, 1601, 8, 2, 128, BF, True, 2),
	],
)
def test_ranges_of_keys(Sq, Sk, Hq, Hkv, D, dtype, causal, ranges):
	_check(1, Sq, Sk, Hq, Hkv, D, dtype, causal, None, None, 0.0, ranges)


@pytest.mark.parametrize("qk_scale", [2.1, 4.2])
@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,lens,p",
	[
		# block by block: a later block raises the reference of a row that has one.  Rows of 72 to 96 columns; one group of waves (four a SIMD, few tiles), two
		# (two and four waves a SIMD), three; with dropout
		(9, 257, 257, 20, 20, 80, FP, False, None, 0.0),
		(9, 257, 300, 20, 5, 72, BF, True, None, 0.0),
		(9, 257, 257, 20, 20, 96, BF, False, [257, 1, 33, 64, 65, 0, 200, 256, 97], 0.0),
		(8, 257, 257, 32, 4, 64, BF, True, None, 0.0),
		(9, 257, 257, 20, 20, 64, FP, False, None, 0.1),
		(1, 130, 192, 3, 1, 64, FP, False, None, 0.1),
		(2, 200, 520, 2, 2, 64, BF, False, None, 0.1),
		(2, 600, 700, 30, 10, 64, FP, True, None, 0.1),
		(2, 900, 1100, 14, 7, 64, BF, False, None, 0.0),
		(1, 1100, 1100, 16, 16, 64, FP, True, None, 0.2),
		# on key ranges of two workgroups a CU
		(1, 700, 5000, 16, 4, 64, FP, True, None, 0.0),
		(1, 600, 2945, 32, 8, 128, BF, False, None, 0.0),
	],
)
def test_large_scores(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, p, qk_scale):
	"""Scores within about +-20 and +-80 at qk_scale 2.1 and 4.2."""
	_check(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, None, p, qk_scale=qk_scale)


def test_256_row_workgroups_beyond_the_l2():
	q, k, v, _, _ = make_inputs(1, 200, 16500, 264, 1, 64, BF, seed=3)
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), None, None, None, 0.0, True, 0)
	heads = [0, 131, 263]
	o_ref, lse_ref = O.attention_fwd(f64(q[:, :, heads]), f64(k), f64(v), None, causal=True)
	check_forward(o[:, :, heads], lse[:, heads], o_ref, lse_ref, BF)


@pytest.mark.parametrize("S,Hq,Hkv", [(4100, 32, 16), (2300, 36, 12), (4100, 33, 3)])
def test_two_groups_of_waves_on_grids_that_are_not_resident(S, Hq, Hkv):
	q, k, v, _, _ = make_inputs(1, S, S, Hq, Hkv, 64, BF, seed=S + Hq)
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), None, None, None, 0.0, True, 0)
	r = Hq // Hkv
	for j in (0, Hkv // 2, Hkv - 1):
		heads = slice(j * r, j * r + min(r, 3))
		o_ref, lse_ref = O.attention_fwd(f64(q[:, :, heads]), f64(k[:, :, j : j + 1]), f64(v[:, :, j : j + 1]), None, causal=True)
		check_forward(o[:, :, heads], lse[:, heads], o_ref, lse_ref, BF, f"S{S} Hq{Hq} Hkv{Hkv} group {j}")
