"""The forward on grids that leave compute units idle: workgroups whose groups of waves share the keys of their rows, alone and on
several key ranges per row tile; checked where tiles, groups and ranges meet."""

import pytest
import torch

from jax_flash_attn2 import _hip_op as op
import fa2_oracle as O
from _cases import check_forward, f64, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,lens,window,p,bias",
	[
		# one to five tiles of 64 keys: two groups take them in turn from four tiles on, the second may have one fewer or none
		(1, 130, 192, 2, 1, 128, torch.bfloat16, False, None, None, 0.0, False),
		(1, 130, 193, 2, 1, 128, torch.bfloat16, False, None, None, 0.0, False),
		(2, 257, 257, 2, 2, 64, torch.float16, True, None, None, 0.0, False),
		(1, 300, 320, 2, 2, 64, torch.bfloat16, True, None, None, 0.2, True),
		(2, 200, 260, 2, 1, 128, torch.float16, True, None, None, 0.1, False),
		# rows without keys, in one group or in both; a window that begins in the middle
		(2, 290, 290, 4, 2, 64, torch.bfloat16, False, [0, 70], None, 0.0, True),
		(1, 400, 200, 2, 2, 128, torch.bfloat16, True, None, None, 0.0, False),
		(1, 600, 600, 2, 1, 128, torch.bfloat16, True, None, (100, 0), 0.0, False),
		# several key ranges of 128-row workgroups: causal rows that end before a range, lengths that end inside the first
		(1, 100, 2000, 8, 2, 128, torch.bfloat16, True, None, None, 0.0, False),
		(1, 1030, 1030, 2, 1, 64, torch.float16, True, None, None, 0.0, False),
		(2, 150, 1500, 4, 4, 128, torch.float16, False, [40, 1500], None, 0.0, False),
		(1, 17, 1100, 4, 4, 64, torch.bfloat16, True, None, None, 0.0, False),
		# up to 64 rows over many keys: ranges of the 64-row kernel (head dim 64; head dim 128 with few heads, and with lengths)
		(1, 40, 4200, 4, 4, 64, torch.bfloat16, True, None, None, 0.0, False),
		(2, 64, 1100, 32, 32, 64, torch.float16, False, [1100, 30], None, 0.0, False),
		(1, 33, 8200, 2, 2, 128, torch.bfloat16, True, None, None, 0.0, False),
		(4, 20, 3100, 8, 8, 128, torch.float16, False, [3100, 0, 1, 2000], None, 0.0, False),
		# head dim 64 without bias: two groups from four tiles on; a window of which a row tile sees three tiles' keys, and one more
		(2, 192, 192, 2, 2, 64, torch.float16, True, None, None, 0.0, False),
		(2, 193, 193, 2, 2, 64, torch.float16, True, None, None, 0.0, False),
		(2, 320, 320, 2, 2, 64, torch.float16, True, None, None, 0.0, False),
		(2, 321, 321, 2, 2, 64, torch.float16, True, None, None, 0.0, False),
		(2, 450, 450, 2, 1, 64, torch.bfloat16, True, None, (64, 0), 0.0, False),
		(2, 450, 450, 2, 1, 64, torch.bfloat16, True, None, (65, 0), 0.0, False),
		(2, 450, 450, 2, 1, 64, torch.bfloat16, True, None, (192, 0), 0.0, False),
		(2, 450, 450, 2, 1, 64, torch.bfloat16, True, None, (193, 0), 0.0, False),
		# head dim 128 under a causal mask: from five tiles on; rows without keys, a window that begins in the middle
		(1, 500, 256, 2, 2, 128, torch.bfloat16, True, None, None, 0.0, False),
		(1, 500, 257, 2, 2, 128, torch.bfloat16, True, None, None, 0.0, False),
		(1, 600, 600, 2, 1, 128, torch.bfloat16, True, None, (200, 0), 0.0, False),
	],
)
def test_groups_and_ranges_of_keys(B, Sq, Sk, Hq, Hkv, D, dtype, causal, lens, window, p, bias):
	q, k, v, _, bs = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq + Sk, bias_shape=(B, 1, Sq, Sk) if bias else None)
	kw = dict(causal=causal, kv_lens=lens, window=window, p_drop=p, seed=9)
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k), f64(v), f64(bs), **kw)
	kl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda:0")
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), None if bs is None else bs.cuda(), None, None, p, causal, 9, kl, window)
	check_forward(o, lse, o_ref, lse_ref, dtype, f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} {kw}")
