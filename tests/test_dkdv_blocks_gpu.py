"""The dK/dV kernel of head dim 64 on grids of at least two workgroups per CU, which goes through its tiles block by block: every operand
it takes, row counts around the blocks and tiles, checked on the first and the last KV group."""

import pytest
import torch

from jax_flash_attn2 import _hip_op as op
import fa2_oracle as O
from _cases import check_grads, f64, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
	"Sq,Sk,kw",
	[
		(520, 520, {}),
		(417, 520, dict(p=0.2)),
		(545, 545, dict(causal=True)),
		(545, 545, dict(causal=True, p=0.1)),
		(200, 600, dict(causal=True, kv_lens=[600, 301])),
		(640, 640, dict(window=(99, 0), causal=True)),
		(512, 512, dict(bias="shared")),              # whole pieces: bias tiles in LDS
		(300, 520, dict(bias="head", p=0.1)),
		(33, 513, dict(bias="head")),                 # unaligned rows: value by value
		(97, 640, dict(bias="mask", causal=True)),
		(160, 560, dict(softcap=2.0)),
	],
)
def test_block_by_block(Sq, Sk, kw, dtype):
	B, Hq, Hkv, D = 2, 64, 64, 64
	bias, p, kv_lens = kw.get("bias"), kw.get("p", 0.0), kw.get("kv_lens")
	assert B * Hkv * ((Sk + 127) // 128) >= 512
	q, k, v, do, bs = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=Sq, bias_shape={None: None, "shared": (B, 1, Sq, Sk)}.get(bias, (1, Hq, Sq, Sk)))
	dev_bias, ref_bias = bs, bs
	if bias == "mask":
		dev_bias = bs > -1.0
		ref_bias = torch.where(dev_bias, 0.0, float(torch.finfo(dtype).min)).double()
	kl = None if kv_lens is None else torch.tensor(kv_lens, dtype=torch.int32, device="cuda:0")
	args = (None if dev_bias is None else dev_bias.cuda(), None, None, p, kw.get("causal", False), 7, kl, kw.get("window"), kw.get("softcap", 0.0))
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), *args)
	g = op.bwd(q.cuda(), k.cuda(), v.cuda(), o, lse, do.cuda(), *args)
	for b, h in ((0, 0), (B - 1, Hq - 1)):
		bs_, hs = slice(b, b + 1), slice(h, h + 1)
		rb = None if ref_bias is None else f64(ref_bias[(bs_ if bias == "shared" else slice(None)), (slice(None) if bias == "shared" else hs)])
		want = O.attention_bwd(*[f64(x[bs_, :, hs]) for x in (q, k, v, do)], rb, causal=kw.get("causal", False), window=kw.get("window"),
		                       kv_lens=None if kv_lens is None else kv_lens[bs_], softcap=kw.get("softcap", 0.0), p_drop=p, seed=7, pos_offset=(b, h, 0))
		check_grads([x[bs_, :, hs] for x in g], want, f"Sq{Sq} Sk{Sk} {kw} b{b} h{h}")
