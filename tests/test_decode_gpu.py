"""The forward for a handful of query rows (fwd_decode_kernel): the key tiles of all (batch, kv-head) units are one sequence cut
into equal shares, one per wave; checked where shares, tiles and units meet."""

import numpy as np
import pytest
import torch

import fa2_oracle as O
from _cases import check_forward, f64, make_inputs
from jax_flash_attn2 import _hip_op as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,lens",
	[
		# a tile of 32 keys (64 at head dim 64): less than one, one, one key more; up to 256 keys a unit is one wave's
		(1, 1, 1, 4, 1, 128, torch.bfloat16, False, None),
		(2, 1, 32, 4, 2, 128, torch.float16, True, None),
		(3, 2, 33, 4, 4, 256, torch.bfloat16, True, [33, 0, 1]),
		(2, 3, 65, 5, 1, 64, torch.float16, True, [65, 64]),
		(1, 1, 256, 8, 2, 128, torch.bfloat16, False, None),
		# from 257 keys on units are cut and merged: uneven lengths, one of them 0, all of them 0
		(1, 1, 257, 8, 2, 128, torch.bfloat16, False, None),
		(5, 1, 700, 8, 2, 128, torch.bfloat16, False, [700, 0, 31, 384, 1]),
		(2, 1, 300, 4, 4, 64, torch.bfloat16, False, [0, 0]),
		# sixteen rows of a unit (causal rows that see different keys), the most this kernel takes, and seventeen, one more
		(2, 4, 1000, 8, 2, 128, torch.float16, True, [1000, 3]),
		(2, 16, 500, 2, 2, 64, torch.bfloat16, True, None),
		(2, 17, 700, 2, 2, 64, torch.bfloat16, True, None),
		(1, 8, 900, 4, 2, 256, torch.float16, True, [517]),
		# more rows of Q than keys: rows without a key
		(1, 12, 5, 1, 1, 128, torch.bfloat16, True, None),
		# more than 64 batch rows (lengths are added up 64 at a time), shares that span many units, more tiles than waves
		(70, 1, 330, 4, 2, 64, torch.bfloat16, False, "ramp"),
		(150, 1, 300, 12, 12, 64, torch.float16, False, "ramp"),
		(3, 1, 9001, 12, 12, 128, torch.bfloat16, False, "ramp"),
		# whole units over more than 256 keys: half a round of waves, more than a round
		(64, 1, 600, 8, 8, 128, torch.bfloat16, False, "ramp"),
		(70, 4, 290, 16, 16, 64, torch.float16, True, None),
		# sixteen rows over four and six tiles of 32 keys, and over a few hundred keys: left to the general kernel
		(2, 16, 128, 4, 4, 128, torch.bfloat16, True, None),
		(2, 4, 190, 8, 2, 256, torch.float16, True, [190, 0]),
		(24, 16, 270, 8, 8, 128, torch.bfloat16, True, "ramp"),
		# from 2048 units on every unit is one wave's
		(130, 1, 270, 16, 16, 64, torch.bfloat16, False, "ramp"),
	],
)
def test_few_rows_over_many_keys(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens):
	if lens == "ramp":
		lens = [int(x) for x in np.linspace(0, Sk, B)]
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=B + Sk)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), causal=causal, kv_lens=lens)
	kl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda:0")
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal, kv_lens=kl)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} causal={causal} lens={lens}")
