"""Which forwards ask for scratch and which rows of fewer columns are taken as they are: decided on the host, no kernel is launched."""

import ctypes

import pytest
import torch

from jax_flash_attn2 import _hip_op as op, _lib


def _call(B, Sq, Sk, Hq, Hkv, rows, lens=False):
	q = torch.empty(B, Sq, Hq, rows, dtype=torch.bfloat16)
	k, o, lse = torch.empty(B, Sk, Hkv, rows, dtype=torch.bfloat16), torch.empty_like(q), torch.empty(B, Hq, Sq)
	kl = torch.full((B,), Sk, dtype=torch.int32) if lens else None
	return op._block(128, q, k, k, None, None, 0.1, 0.0, True, 0, kl, None, 0.0, op._t4(o), lse), (q, k, o, lse, kl)


@pytest.mark.parametrize(
	"shape,lens,ranges",
	[
		((1, 1000, 9000, 32, 8), False, 2),
		((1, 600, 3000, 32, 8), False, 3),
		((1, 1000, 3000, 32, 8), False, 0),  # one range of workgroups of eight waves
		((1, 1100, 9000, 32, 8), False, 0),  # more workgroups than CUs
		((1, 1000, 9000, 32, 8), True, 0),  # ranges beyond a length would be empty
	],
)
def test_two_workgroups_a_cu_over_many_keys(shape, lens, ranges):
	lib = _lib.load()
	B, Sq, Sk, Hq, Hkv = shape
	p, _keep = _call(*shape, 128, lens)
	n = lib.fa2_fwd_scratch_bytes(ctypes.byref(p))
	assert n == (ranges * B * Hq * Sq * (128 + 1) * 4 + 255) // 256 * 256
	# rows of fewer columns have no such form: they are taken as they were, not refused for it
	p, _keep = _call(*shape, 80, lens)
	assert lib.fa2_validate(ctypes.byref(p), 0) == 0
