"""NaN and infinity through the forwards that work on pieces of a key range (the split kernels and the decoding kernel): a row that
sees a non-finite value must come out non-finite whatever the keys were cut into, and a value that no row may see - a slot of
the cache beyond its row's length - must not come out at all."""

import ctypes

import numpy as np
import pytest
import torch

import fa2_oracle as O
from _cases import check_forward, f64, make_inputs
from jax_flash_attn2 import _hip_op as op
from jax_flash_attn2 import _lib

pytestmark = pytest.mark.gpu


def _scratch(q, k, v, causal=False, kv_lens=None):
	return _lib.load().fa2_fwd_scratch_bytes(ctypes.byref(op._block(q.shape[3], q, k, v, None, None, 1.0, 0.0, causal, None, kv_lens)))


# (B, Sq, Sk, Hq, Hkv, D, causal): 128-row workgroups on several ranges, and of four waves, two a CU, on five; ranges of the 64-row kernel with the q-heads packed; head
# dim 256, which takes that kernel unpacked; the decoding kernel with units of several waves, and of few keys (257 .. 448)
_PIECES = [
	(1, 100, 2000, 8, 2, 128, True),
	(1, 300, 1500, 4, 4, 64, False),
	(1, 1500, 6200, 8, 2, 128, True),
	(1, 8, 4000, 8, 2, 128, False),
	(1, 65, 2048, 2, 2, 256, True),
	(1, 1, 1029, 32, 8, 128, False),
	(2, 2, 300, 4, 2, 64, True),
	(2, 1, 400, 4, 4, 256, False),
]


@pytest.mark.parametrize("B,Sq,Sk,Hq,Hkv,D,causal", _PIECES)
@pytest.mark.parametrize("what", ["nan in one key", "infinity in one key", "nan in a query row", "infinity in a query row"])
def test_non_finite_rows_stay_non_finite(B, Sq, Sk, Hq, Hkv, D, causal, what):
	dtype = torch.bfloat16
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq + Sk)
	bad = float("nan") if "nan" in what else float("inf")
	key, row = Sk - 40, Sq // 2
	if "key" in what:
		q[..., 3] = q[..., 3].abs() + 0.1  # (of infinity: every row that sees the key scores +inf, whose softmax is NaN)
		k[:, key, Hkv - 1, 3] = bad
	else:
		q[:, row, Hq - 1, 3] = bad
		k[..., 3] = k[..., 3].abs() + 0.1
	assert _scratch(q, k, v, causal) > 0, "this shape is meant to be cut into pieces"
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal)
	o = o.float().cpu()
	hit = torch.zeros(B, Sq, Hq, dtype=torch.bool)
	if "key" in what:
		first = max(0, key - (Sk - Sq)) if causal else 0
		hit[:, first:, Hq - Hq // Hkv :] = True
	else:
		hit[:, row, Hq - 1] = True
	assert torch.isnan(o[hit]).all(), f"{int((~torch.isnan(o[hit])).sum())} finite values in rows that see {what}"
	# and nothing else changed
	for x in (q, k):
		x[~torch.isfinite(x)] = 0.0
	o_ref, _ = O.attention_fwd(f64(q), f64(k), f64(v), causal=causal)
	assert np.abs(o[~hit].numpy() - torch.from_numpy(o_ref)[~hit].numpy()).max() <= 2e-2


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,lens,cut",
	[
		# one wave a unit: few keys, and from 2048 units on
		(3, 1, 200, 8, 2, 64, [0, 200, 7], False),
		(2, 2, 192, 4, 2, 128, [0, 33], False),
		(2, 1, 100, 4, 4, 256, [64, 0], False),
		(128, 1, 300, 16, 16, 64, None, None),
		# units of several waves; 128-row workgroups, unsplit and split
		(4, 1, 700, 8, 2, 128, [700, 0, 31, 384], True),
		(2, 130, 200, 2, 1, 128, [0, 70], False),
		(2, 150, 1500, 4, 4, 128, [0, 40], True),
	],
)
def test_slots_beyond_the_length_are_not_looked_at(B, Sq, Sk, Hq, Hkv, D, lens, cut):
	dtype = torch.bfloat16
	if lens is None:
		lens = [int(x) for x in np.linspace(0, Sk, B)]
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=B + Sk)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), kv_lens=lens)
	for b, n in enumerate(lens):
		k[b, n:] = float("nan")
		v[b, n:] = float("nan")
	kl = torch.tensor(lens, dtype=torch.int32, device="cuda:0")
	if cut is not None:
		assert bool(_scratch(q, k, v, kv_lens=kl)) == cut
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), kv_lens=kl)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} lens={lens}")
	for b, n in enumerate(lens):
		if n == 0:
			assert not o[b].any() and torch.isneginf(lse[b]).all()
