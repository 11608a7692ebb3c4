"""The dK/dV kernel where a sequence ends within a tile: key tiles of which one or two blocks of 32 keys are left (the waves of the
workgroup share them), query tiles of which one or two blocks of rows are left, and the sizes around both."""

import pytest
import torch

from jax_flash_attn2 import _hip_op as op
import fa2_oracle as O
from _cases import check_forward, check_grads, f64, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (80, torch.bfloat16), (128, torch.bfloat16)])
@pytest.mark.parametrize(
	"Sq,Sk,Hq,Hkv,causal,kv_lens,window",
	[
		(257, 257, 1, 1, False, None, None),   # one key, one row left
		(1, 1, 2, 1, False, None, None),
		(130, 32, 2, 1, False, None, None),    # a whole block of keys
		(320, 161, 2, 1, False, None, None),   # two blocks with one key in the second; two blocks of rows
		(65, 193, 1, 1, False, None, None),    # three blocks: no sharing
		(289, 192, 4, 2, True, None, None),    # rows without keys, groups of heads
		(290, 290, 2, 1, True, None, None),
		(200, 384, 1, 1, False, [130, 300], None),   # lengths that end in the second tile: keys beyond them get zeros
		(384, 384, 1, 1, True, [5, 384], None),
		(420, 420, 2, 2, True, None, (70, 0)),
		(33, 33, 2, 2, False, None, None),     # keys that waves would share, but only the first of them has rows; one row more
		(64, 64, 2, 1, True, None, None),
		(32, 20, 1, 1, False, None, None),
		(33, 20, 2, 1, False, None, None),
		(2100, 40, 16, 1, False, None, None),  # the steps of the one key tile split over workgroups
		# more than four row tiles (or heads times row tiles): only there do waves share the keys, and only if more than one has rows
		(641, 257, 1, 1, False, None, None),   # one block of keys
		(600, 150, 2, 1, True, None, None),
		(650, 192, 4, 2, False, [192, 140], None),   # two blocks; a row of the batch with one block
		(769, 35, 1, 1, False, None, (300, 500)),
		(130, 20, 6, 1, False, None, None),
		(33, 20, 6, 1, True, None, None),      # rows 13 to 32 see keys: in two shares of 32 rows
		(33, 1, 6, 1, True, None, None),       # one row does
		(645, 645, 6, 1, True, None, None),    # five rows and keys in the last tiles
	],
)
def test_ends_of_sequences(Sq, Sk, Hq, Hkv, causal, kv_lens, window, D, dtype):
	B = 2 if kv_lens else 1
	q, k, v, do, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq + Sk + D)
	ref = dict(causal=causal, kv_lens=kv_lens, window=window)
	a = [f64(x) for x in (q, k, v, do)]
	kl = None if kv_lens is None else torch.tensor(kv_lens, dtype=torch.int32, device="cuda:0")
	args = (None, None, None, 0.0, causal, None, kl, window)
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), *args)
	g = op.bwd(q.cuda(), k.cuda(), v.cuda(), o, lse, do.cuda(), *args)
	name = f"Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} {ref}"
	check_forward(o, lse, *O.attention_fwd(*a[:3], **ref), dtype, name)
	check_grads(g, O.attention_bwd(*a, **ref), name, O.attention_bwd(*a, o_stored=f64(o.cpu()), **ref))
	for y, n in ((x[b, kv_lens[b] :], kv_lens[b]) for x in g[1:] for b in range(B) if kv_lens):
		assert not y.any(), f"{name}: gradients of keys from {n} on"
