"""Lengths of a 2-D validity mask: row lengths around the 16-byte pieces and the workgroup, rows at every alignment, mask types."""

import pytest
import torch

from jax_flash_attn2 import _hip_op as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 15, 16, 17, 31, 255, 511, 4096, 4113, 70001])
def test_lengths_of_a_mask(S):
	q = torch.empty(1, device="cuda:0")
	n = torch.tensor([0, 1, S // 2, S - 1, S], device="cuda:0").clamp(0, S)
	mask = torch.arange(S, device="cuda:0")[None, :] < n[:, None]
	for m in (mask, mask.int(), mask.half(), mask.cpu(), mask.t().contiguous().t()):
		got = op._seqlens_from_mask(m, q)
		assert got.dtype == torch.int32 and got.is_contiguous() and got.cpu().tolist() == n.tolist()
	for off in range(1, 17):  # (a slice of wider rows: its first byte anywhere, what surrounds it set)
		wide = torch.ones((5, S + 21), dtype=torch.bool, device="cuda:0")
		wide[:, off : off + S] = mask
		assert op._seqlens_from_mask(wide[:, off : off + S], q).cpu().tolist() == n.tolist()
	assert op._seqlens_from_mask(mask[:1].expand(3, S), q).cpu().tolist() == [0, 0, 0]
