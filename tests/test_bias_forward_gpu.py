"""The operator with a bias: biases that leave the reference of a row alone, that raise it now and then or on every tile, and references
that no exponent may be formed against."""

import numpy as np
import pytest
import torch

from jax_flash_attn2 import _hip_op as op
import fa2_oracle as O
from _cases import check_forward, check_grads, f64, make_inputs

pytestmark = pytest.mark.gpu


def _bias(kind, dtype, B, H, Sq, Sk):
	"""[B, H, Sq, Sk] in float64"""
	i, j = np.arange(Sq)[:, None], np.arange(Sk)[None, :]
	lowest = torch.finfo(dtype).min
	if kind == "flat":
		x = 1.0 / (1.0 + abs(i - j))
	elif kind == "steep":  # every tile raises the maximum by 32
		x = 0.5 * (j - i)
	elif kind == "one late key":  # far above the reference
		x = np.where(j == Sk - 9, 30.0, 0.0) + 0.0 * i
	elif kind == "first tiles hidden":  # the reference of the first tiles is the lowest finite value
		x = np.where(j < min(Sk - 8, 150), lowest, 0.5) + 0.0 * i
	elif kind == "rows hidden":  # uniform over all keys, in half of the rows of a wave; nothing in the other half is hidden
		x = np.where(i % 2 == 0, lowest, 0.25) + 0.0 * j
	else:
		assert kind == "infinite"
		x = np.where((i + j) % 3 == 0, -np.inf, 0.0)
	return torch.from_numpy(np.broadcast_to(x, (B, H, Sq, Sk)).copy()).to(dtype)


@pytest.mark.parametrize("kind", ["flat", "steep", "one late key", "first tiles hidden", "rows hidden", "infinite"])
@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,p",
	[
		(1, 200, 448, 2, 1, 64, torch.bfloat16, False, 0.0),  # two groups of waves
		(1, 328, 328, 2, 2, 64, torch.float16, True, 0.1),
		(300, 40, 136, 1, 1, 64, torch.bfloat16, False, 0.0),  # one group, a last tile of eight keys
		(1, 130, 264, 2, 2, 128, torch.float16, False, 0.0),
		(1, 200, 264, 2, 2, 256, torch.bfloat16, True, 0.0),
		(1, 100, 320, 2, 1, 256, torch.float16, False, 0.2),
		(1, 8, 1024, 2, 2, 64, torch.bfloat16, False, 0.0),  # several ranges of keys, equal ones (a hidden row weighs them by their number)
	],
)
def test_bias_that_rises_falls_and_hides(B, Sq, Sk, Hq, Hkv, D, dtype, causal, p, kind):
	q, k, v, _, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq + D)
	bias = _bias(kind, dtype, B, 1, Sq, Sk)
	if kind == "infinite":
		bias[..., 1] = 0.0  # (every row keeps a key)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), f64(bias), causal=causal, p_drop=p, seed=5)
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), bias.cuda(), dropout_prob=p, causal=causal, dropout_seed=5)
	if kind == "rows hidden":  # (their logsumexp is the lowest finite value in the 24 bits of fp32: -3.39e38 to a part in 1e7)
		hidden = lse_ref < -6e4
		assert np.allclose(lse.float().cpu().numpy()[hidden], lse_ref[hidden], rtol=1e-6)
		lse_ref = np.where(hidden, 0.0, lse_ref)
		lse = torch.where(torch.from_numpy(hidden).cuda(), torch.zeros_like(lse), lse)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"{kind} B{B} Sq{Sq} Sk{Sk} D{D} causal={causal} p={p}")


@pytest.mark.parametrize("D", [64, 128, 256])
def test_values_near_the_largest_number(D):
	"""A late key far above the reference, and values of V of 2^93 (bfloat16 has the range of fp32): no product of the two may pass
	the fp32 range on the way to a result that is within it."""
	B, Sq, Sk, H, dtype = 1, 72, 320, 2, torch.bfloat16
	q, k, v, _, _ = make_inputs(B, Sq, Sk, H, H, D, dtype, seed=D)
	bias = _bias("flat", dtype, B, 1, Sq, Sk)
	bias[..., Sk - 9] = 25.0
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), f64(bias))
	o, lse = op.fwd(q.cuda(), k.cuda(), (v * 2.0**93).cuda(), bias.cuda())
	check_forward(o.float() * 2.0**-93, lse, o_ref, lse_ref, dtype, f"D{D}")


# Masks that are spelt as a large negative number: beyond about 1e6 the product of a reference and log2(e) is rounded by more than an
# exponent bears, from the lowest value / log2(e) on it leaves the fp32 range.
_FILLS = [-1e6, -1e9, -1e10, -1e12, -1e30, None]  # (None: the lowest finite value)


def _masked(fill, bias_dtype, Sq, Sk):
	"""Two heads: in the first the keys of the first tiles are hidden, in the second all keys of every other row (their q is zero, so
	that the oracle weighs these keys alike too; fp32 does so whatever q is, the bias absorbs the score)."""
	fill = torch.finfo(bias_dtype).min if fill is None else fill
	bias = _bias("flat", torch.float32, 1, 2, Sq, Sk)
	bias[0, 0, :, :150] = fill
	bias[0, 1, ::2] = fill
	return bias.to(bias_dtype)


def _masked_inputs(Sq, Sk, D, dtype):
	q, k, v, do, _ = make_inputs(1, Sq, Sk, 2, 2, D, dtype, seed=D)
	q[:, ::2, 1] = 0
	return q, k, v, do


_MASKED = [
	(torch.bfloat16, torch.bfloat16, 320),  # tiles of bias in LDS
	(torch.bfloat16, torch.bfloat16, 321),  # bias read value by value
	(torch.float16, torch.float32, 320),
]


@pytest.mark.parametrize("fill", _FILLS)
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype,bias_dtype,Sk", _MASKED)
def test_large_negative_bias_as_a_mask(dtype, bias_dtype, Sk, D, fill):
	Sq = 72
	q, k, v, _ = _masked_inputs(Sq, Sk, D, dtype)
	bias = _masked(fill, bias_dtype, Sq, Sk)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), f64(bias))
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), bias.cuda())
	# (the logsumexp of a hidden row is the bias to the 24 bits of fp32)
	assert np.allclose(lse[0, 1, ::2].cpu().numpy(), lse_ref[0, 1, ::2], rtol=1e-6)
	lse[0, 1, ::2] = 0
	lse_ref[0, 1, ::2] = 0
	check_forward(o, lse, o_ref, lse_ref, dtype, f"D{D} {fill}")


@pytest.mark.parametrize("fill", [f for f in _FILLS if f != -1e6])
@pytest.mark.parametrize("D,softcap", [(64, 0.0), (128, 0.0), (256, 0.0), (64, 20.0)])
@pytest.mark.parametrize("dtype,bias_dtype,Sk", _MASKED)
def test_gradients_of_a_large_negative_bias_as_a_mask(dtype, bias_dtype, Sk, D, softcap, fill):
	"""A row whose keys are all hidden has a logsumexp that holds nothing of the sum any more: it passes no gradient on, whatever
	gradient arrives at it, and it leaves the gradients of K and V to the other rows."""
	Sq = 72
	q, k, v, do = _masked_inputs(Sq, Sk, D, dtype)
	bias = _masked(fill, bias_dtype, Sq, Sk)
	a = [x.cuda() for x in (q, k, v)]
	args = (bias.cuda(), None, None, 0.0, False, None, None, None, softcap)
	o, lse = op.fwd(*a, *args)
	got = op.bwd(*a, o, lse, do.cuda(), *args)
	with_dbias = op.bwd(*a, o, lse, do.cuda(), *args, need_dbias=True)
	do[:, ::2, 1] = 0
	want = O.attention_bwd(f64(q), f64(k), f64(v), f64(do), f64(bias), softcap=softcap, return_dbias=True)
	check_grads(got, want[:3], f"D{D} {fill}")
	check_grads(with_dbias[:3], want[:3], f"D{D} {fill} with the gradient of the bias")
	dbias = with_dbias[3].cpu().numpy()
	assert np.isfinite(dbias).all() and O.rel_l2(dbias, want[3]) <= 1e-2
