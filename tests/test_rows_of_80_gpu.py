"""Rows of 72 and 80 columns on larger grids: products over 80 columns where longer rows take 96, dQ with two and three workgroups a CU (the
latter in tiles of one block of 32 keys), dK/dV with two slots of a block that hold no product of its scores."""

import pytest
import torch

from jax_flash_attn2 import _hip_op as op
import fa2_oracle as O
from _cases import check_forward, check_grads, f64, make_inputs

pytestmark = pytest.mark.gpu
BF, FP = torch.bfloat16, torch.float16


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,kv_lens,window",
	[
		# more than two workgroups of 128 rows a CU, 512 key tiles and more: one key, one beyond a block, whole blocks, one row tile and a row
		(70, 33, 1, 16, 16, 80, FP, False, None, None),
		(33, 65, 33, 16, 16, 72, BF, False, None, None),
		(20, 128, 96, 32, 32, 80, BF, True, None, None),
		(9, 257, 257, 20, 20, 80, FP, False, None, None),
		(8, 300, 300, 32, 32, 80, FP, True, None, None),
		# lengths (a row without keys among them), rows that see no key, a window whose two edges meet in a block
		(9, 200, 97, 32, 8, 72, BF, True, [97, 96, 64, 33, 32, 31, 1, 0, 31], None),
		(9, 300, 300, 24, 24, 80, FP, True, None, (17, 0)),
		# two workgroups a CU: fewer of them, and the causal grids that wait for their longest tile
		(3, 500, 700, 24, 8, 80, BF, False, None, None),
		(2, 1100, 1100, 44, 11, 72, FP, True, None, None),
		(1, 2100, 2100, 36, 36, 80, BF, True, None, None),
		# three layers of workgroups that are all resident
		(6, 250, 250, 64, 16, 80, BF, True, None, None),
		(6, 250, 250, 64, 16, 80, FP, True, None, (170, 0)),
	],
)
def test_against_the_oracle(B, Sq, Sk, Hq, Hkv, D, dtype, causal, kv_lens, window):
	q, k, v, do, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=D + Sq)
	kl = None if kv_lens is None else torch.tensor(kv_lens, dtype=torch.int32, device="cuda:0")
	args = (None, None, None, 0.0, causal, None, kl, window)
	q_, k_, v_, do_ = (x.cuda() for x in (q, k, v, do))
	o, lse = op.fwd(q_, k_, v_, *args)
	grads = op.bwd(q_, k_, v_, o, lse, do_, *args)
	# (the first and the last KV group of the last batch row are enough for the oracle)
	bs = slice(B - 1, B)
	for j in {0, Hkv - 1}:
		hs, kv = slice(j * (Hq // Hkv), (j + 1) * (Hq // Hkv)), slice(j, j + 1)
		ref = dict(causal=causal, kv_lens=None if kv_lens is None else kv_lens[bs], window=window)
		a = [f64(x) for x in (q[bs, :, hs], k[bs, :, kv], v[bs, :, kv], do[bs, :, hs])]
		name = f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} {ref} group {j}"
		check_forward(o[bs, :, hs], lse[bs, hs], *O.attention_fwd(*a[:3], **ref), dtype, name)
		check_grads([x[bs, :, y] for x, y in zip(grads, (hs, kv, kv))], O.attention_bwd(*a, **ref), name)
