"""The forward for a handful of query rows (fwd_decode_kernel): the key tiles of all (batch, kv-head) units are one sequence cut
into equal shares, one per wave, or every unit is one wave's; checked where shares, tiles and units meet."""

import ctypes

import numpy as np
import pytest
import torch

import fa2_oracle as O
from _cases import check_forward, f64, make_inputs
from jax_flash_attn2 import _hip_op as op
from jax_flash_attn2 import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,lens,cut",
	[
		# a tile of 32 keys (64 at head dim 64): less than one, one, one key more; up to six tiles a unit is one wave's, eight are the general kernel's
		(1, 1, 1, 4, 1, 128, torch.bfloat16, False, None, False),
		(2, 1, 32, 4, 2, 128, torch.float16, True, None, False),
		(3, 2, 33, 4, 4, 256, torch.bfloat16, True, [33, 0, 1], False),
		(2, 3, 65, 5, 1, 64, torch.float16, True, [65, 64], False),
		(1, 1, 256, 8, 2, 128, torch.bfloat16, False, None, False),
		# from 257 keys on units are cut and merged: uneven lengths, one of them 0, all of them 0 (units that are few; see below)
		(1, 1, 257, 8, 2, 128, torch.bfloat16, False, None, True),
		(5, 1, 700, 8, 2, 128, torch.bfloat16, False, [700, 0, 31, 384, 1], True),
		(2, 1, 300, 4, 4, 64, torch.bfloat16, False, [0, 0], True),
		# sixteen rows of a unit (causal rows that see different keys), the most this kernel takes, and seventeen, one more
		(2, 4, 1000, 8, 2, 128, torch.float16, True, [1000, 3], True),
		(2, 16, 500, 2, 2, 64, torch.bfloat16, True, None, True),
		(2, 17, 700, 2, 2, 64, torch.bfloat16, True, None, True),
		(1, 8, 900, 4, 2, 256, torch.float16, True, [517], True),
		# more rows of Q than keys: rows without a key
		(1, 12, 5, 1, 1, 128, torch.bfloat16, True, None, False),
		# more than 64 batch rows (lengths are added up 64 at a time), shares that span several units, more tiles than waves
		(110, 1, 330, 10, 10, 64, torch.float16, False, "ramp", True),
		(70, 4, 290, 16, 16, 64, torch.float16, True, None, True),
		(3, 1, 9001, 12, 12, 128, torch.bfloat16, False, "ramp", True),
		# whole units over more than 256 keys: a part of a round of waves, more than a round, more than two
		(70, 1, 330, 4, 2, 64, torch.bfloat16, False, "ramp", False),
		(64, 1, 600, 8, 8, 128, torch.bfloat16, False, "ramp", False),
		(150, 1, 300, 12, 12, 64, torch.float16, False, "ramp", False),
		(130, 1, 270, 16, 16, 64, torch.bfloat16, False, "ramp", False),
		# sixteen rows over four and six tiles of 32 keys, and over a few hundred keys: left to the general kernel
		(2, 16, 128, 4, 4, 128, torch.bfloat16, True, None, False),
		(2, 4, 190, 8, 2, 256, torch.float16, True, [190, 0], False),
		(24, 16, 270, 8, 8, 128, torch.bfloat16, True, "ramp", False),
	],
)
def test_few_rows_over_many_keys(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, cut):
	# cut: the key tiles are shared by the waves, the pieces merged in scratch
	if lens == "ramp":
		lens = [int(x) for x in np.linspace(0, Sk, B)]
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=B + Sk)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), causal=causal, kv_lens=lens)
	kl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda:0")
	q, k, v = q.cuda(), k.cuda(), v.cuda()
	block = op._block(D, q, k, v, None, None, 1.0, 0.0, causal, None, kl)
	assert bool(_lib.load().fa2_fwd_scratch_bytes(ctypes.byref(block))) == cut, "not the way through the kernel that this case is for"
	o, lse = op.fwd(q, k, v, causal=causal, kv_lens=kl)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} causal={causal} lens={lens}")
