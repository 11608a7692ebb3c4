"""The forward block by block (head dim 64, and rows of 72 to 96 columns), three and four workgroups a CU: grids whose workgroups are all resident at
once and whose parts are visited backwards, two and three groups of waves on the keys of a row tile, ragged blocks of keys."""

import pytest
import torch

from jax_flash_attn2 import _hip_op as op
import fa2_oracle as O
from _cases import check_forward, f64, make_inputs

pytestmark = pytest.mark.gpu
BF, FP = torch.bfloat16, torch.float16


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,lens,window,p",
	[
		# causal grids that are all resident: 264 workgroups (two layers), 768 (three whole ones), 640, 700 (the last one short), 1024 (four); by XCD and not
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
		# two groups of waves a workgroup, two workgroups a CU: ten tiles and more
		(2, 600, 590, 30, 10, 64, FP, True, None, None, 0.0),
		(2, 300, 640, 48, 16, 64, BF, False, [640, 65], None, 0.1),
		# ... and causal grids of up to four a CU over more than 32 tiles: the shortest, more keys than rows, four a CU
		(1, 2049, 2049, 32, 8, 64, BF, True, None, None, 0.0),
		(1, 2100, 2200, 56, 8, 64, FP, True, None, None, 0.0),
		(1, 4033, 4033, 32, 16, 64, BF, True, None, None, 0.0),
		# one to three groups on a grid below the CU count: four, five, sixteen, seventeen tiles; the last group without a tile
		(1, 130, 193, 3, 1, 64, BF, False, None, None, 0.0),
		(2, 300, 257, 2, 2, 64, FP, True, None, None, 0.0),
		(1, 1100, 1024, 2, 2, 64, BF, True, None, None, 0.0),
		(1, 1100, 1025, 2, 2, 64, FP, True, None, None, 0.1),
		(2, 1200, 1200, 2, 1, 64, BF, True, [1200, 0], None, 0.0),
		(1, 1300, 1300, 2, 1, 64, FP, True, None, (900, 0), 0.0),
		# more than two workgroups a CU: blocks of keys that only some rows see, lengths, a window, rows without keys, one key
		(9, 257, 257, 20, 20, 80, FP, False, None, None, 0.0),
		(9, 200, 97, 32, 8, 72, BF, True, [97, 96, 64, 33, 32, 31, 1, 0, 97], None, 0.0),
		(9, 300, 300, 20, 5, 88, FP, True, None, (70, 0), 0.0),
		(9, 300, 300, 20, 5, 64, BF, True, None, (33, 0), 0.0),
		(70, 33, 1, 16, 2, 64, FP, False, None, None, 0.0),
		(40, 65, 129, 30, 6, 64, BF, False, None, None, 0.2),
		# key ranges of workgroups that share a CU
		(1, 700, 5000, 16, 4, 64, BF, True, None, None, 0.0),
		# head dim 128, four waves a workgroup and two workgroups a CU: two ranges, three, five; rows that end before the last, a range of one tile with one key
		(1, 1000, 5700, 24, 8, 128, BF, True, None, None, 0.0),
		(1, 600, 2945, 32, 8, 128, FP, False, None, None, 0.0),
		(1, 1500, 1601, 8, 2, 128, BF, True, None, None, 0.0),
		(2, 1500, 1400, 6, 6, 128, FP, True, None, None, 0.0),
	],
)
def test_blocks(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, window, p):
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq + Sk)
	kw = dict(causal=causal, kv_lens=lens, window=window, p_drop=p, seed=5)
	kl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda:0")
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), None, None, None, p, causal, 5, kl, window)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), None, **kw)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} {kw}")


def test_256_row_workgroups_beyond_the_l2():
	q, k, v, _, _ = make_inputs(1, 200, 16500, 264, 1, 64, BF, seed=3)
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), None, None, None, 0.0, True, 0)
	heads = [0, 131, 263]
	o_ref, lse_ref = O.attention_fwd(f64(q[:, :, heads]), f64(k), f64(v), None, causal=True)
	check_forward(o[:, :, heads], lse[:, heads], o_ref, lse_ref, BF)
