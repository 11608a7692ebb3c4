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


@pytest.mark.parametrize(
	"shape,ranges",
	[
		# two ranges of four waves only where rows do not fill their last wave
		((1, 1000, 9000, 32, 8), 2),
		((1, 1024, 9000, 32, 8), 0),
		((1, 500, 9000, 48, 16), 2),
		((1, 512, 9000, 48, 16), 0),
		((2, 370, 7500, 32, 16), 0),
		((3, 409, 7033, 16, 8), 2),
		# ... and, over up to 10000 keys, groups are placed by XCD
		((1, 1000, 9000, 25, 5), 0),
		((1, 1000, 13000, 25, 5), 2),
		((4, 512, 3000, 12, 12), 0),
		# three, and five, where they do; five not over few keys, where groups are not placed by XCD up to 10000 keys (two of eight waves)
		((1, 512, 4000, 40, 8), 3),
		((1, 512, 7500, 24, 8), 5),
		((1, 640, 4000, 20, 5), 2),
		((1, 896, 7500, 14, 14), 2),
		((1, 896, 13000, 14, 14), 5),
	],
)
def test_rows_that_fill_their_last_wave(shape, ranges):
	B, Sq, _, Hq, _ = shape
	p, _keep = _call(*shape, 128)
	assert _lib.load().fa2_fwd_scratch_bytes(ctypes.byref(p)) == (ranges * B * Hq * Sq * (128 + 1) * 4 + 255) // 256 * 256
