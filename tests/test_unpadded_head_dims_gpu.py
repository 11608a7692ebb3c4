"""Head dims that run in the tiles of head dim 128 without padded copies of the operands: shortest and longest rows, query and key
counts around the tiles, strided operands, and what surrounds the rows in memory (never read into a result, never written)."""

import ctypes

import pytest
import torch

from jax_flash_attn2 import _hip_op as op, _lib
import fa2_oracle as O
from _cases import check_forward, check_grads, f64, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
	"B,Sq,Sk,Hq,Hkv,D,dtype,causal,kv_lens,window",
	[
		(2, 257, 257, 2, 2, 80, torch.float16, False, None, None),   # one row and one key beyond the tiles
		(1, 33, 31, 2, 1, 72, torch.bfloat16, False, None, None),    # a single ragged tile
		(1, 128, 128, 4, 2, 96, torch.bfloat16, True, None, None),   # whole tiles
		(2, 300, 430, 4, 1, 88, torch.float16, True, [430, 70], None),
		(1, 700, 700, 2, 2, 72, torch.bfloat16, True, None, (100, 0)),
		(3, 1030, 1030, 32, 8, 80, torch.bfloat16, True, None, None),   # grids of more than one workgroup per CU
		(8, 520, 5600, 16, 16, 96, torch.float16, False, None, None),   # keys of a head beyond what the smaller workgroups are for
		(1, 2050, 2050, 64, 64, 88, torch.bfloat16, True, None, None),  # a bit more than two workgroups per CU
	],
)
def test_short_rows_against_the_oracle(B, Sq, Sk, Hq, Hkv, D, dtype, causal, kv_lens, window):
	q, k, v, do, _ = make_inputs(B, Sq, Sk, Hq, Hkv, D, dtype, seed=D + Sq)
	kl = None if kv_lens is None else torch.tensor(kv_lens, dtype=torch.int32, device="cuda:0")

	def inside(x):
		# a slice of wider rows whose other columns are NaN: the kernels must not look at them
		wide = torch.full((*x.shape[:3], D + 16), float("nan"), dtype=dtype, device="cuda:0")
		wide[..., 8 : D + 8] = x.cuda()
		return wide[..., 8 : D + 8]

	q_, k_, v_, do_ = (inside(x) for x in (q, k, v, do))
	args = (None, None, None, 0.0, causal, None, kl, window)
	o, lse = op.fwd(q_, k_, v_, *args)
	grads = op.bwd(q_, k_, v_, o, lse, do_, *args)
	# (the last KV group of the last batch row is enough for the oracle)
	bs, hs, kv = slice(B - 1, B), slice(Hq - Hq // Hkv, Hq), slice(Hkv - 1, Hkv)
	ref = dict(causal=causal, kv_lens=None if kv_lens is None else kv_lens[bs], window=window)
	a = [f64(x) for x in (q[bs, :, hs], k[bs, :, kv], v[bs, :, kv], do[bs, :, hs])]
	name = f"B{B} Sq{Sq} Sk{Sk} Hq{Hq} Hkv{Hkv} D{D} {ref}"
	check_forward(o[bs, :, hs], lse[bs, hs], *O.attention_fwd(*a[:3], **ref), dtype, name)
	check_grads([x[bs, :, y] for x, y in zip(grads, (hs, kv, kv))], O.attention_bwd(*a, **ref), name)


def test_infinite_last_column():
	"""A key whose last column is -inf scores -inf for a positive query (probability 0); the columns that are not there add nothing to it."""
	q, k, v, _, _ = make_inputs(1, 64, 100, 1, 1, 72, torch.bfloat16, seed=3)
	q[..., -1] = q[..., -1].abs() + 0.1
	k[:, 5, :, -1] = float("-inf")
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda())
	keep = [j for j in range(100) if j != 5]
	o_ref, lse_ref = O.attention_fwd(f64(q), f64(k[:, keep]), f64(v[:, keep]))
	check_forward(o, lse, o_ref, lse_ref, torch.bfloat16, "key of -inf")


@pytest.mark.parametrize("how", ["two bytes into a buffer", "odd batch stride", "rows too far apart"])
def test_short_rows_in_any_memory(how):
	"""Tensors that are contiguous and yet not aligned, or whose rows lie further apart than the kernels address: padded rows were
	copies in order, rows taken as they are have to be brought in order."""
	B, S, H, D, dtype = 1, 300, 2, 80, torch.float16
	q, k, v, do, _ = make_inputs(B, S, S, H, H, D, dtype, seed=4)

	def placed(x):
		x = x.cuda()
		if how == "two bytes into a buffer":
			return torch.nn.functional.pad(x.flatten(), (1, 0))[1:].view(x.shape)
		if how == "odd batch stride":
			return x.as_strided(x.shape, (x.numel() + 1, *x.stride()[1:]))
		far = 0x7FFFFFFF // 256 + 8 - (0x7FFFFFFF // 256) % 8  # the first multiple of 8 beyond the limit
		wide = torch.empty((S - 1) * far + H * D, dtype=dtype, device="cuda:0")
		y = wide.as_strided(x.shape, (S * far, far, D, 1))
		y.copy_(x)
		return y

	args = [placed(x) for x in (q, k, v, do)]
	o, lse = op.fwd(*args[:3], causal=True)
	grads = op.bwd(*args[:3], o, lse, args[3], causal=True)
	a = [f64(x) for x in (q, k, v, do)]
	check_forward(o, lse, *O.attention_fwd(*a[:3], causal=True), dtype, how)
	check_grads(grads, O.attention_bwd(*a, causal=True), how)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 72), (torch.float16, 80), (torch.bfloat16, 96), (torch.float16, 88)])
@pytest.mark.parametrize(
	"Sq,Sk,kw",
	[
		(257, 257, {}),                                       # a row beyond the fourth tile, a key beyond the second key tile
		(31, 513, {}),                                        # one block of rows
		(96, 520, dict(causal=True)),                         # rows that see no key of the last key tile's end; a tile of one block
		(545, 545, dict(causal=True, kv_lens=[545, 129])),
		(640, 640, dict(causal=True, window=(99, 0))),
	],
)
def test_short_rows_block_by_block(Sq, Sk, kw, dtype, D):
	"""dK/dV on grids of at least two workgroups per CU: block by block in tiles of 64 rows."""
	B, H = 2, 128
	assert B * H * ((Sk + 127) // 128) >= 512
	q, k, v, do, _ = make_inputs(B, Sq, Sk, H, H, D, dtype, seed=Sq + D)
	kv_lens = kw.get("kv_lens")
	kl = None if kv_lens is None else torch.tensor(kv_lens, dtype=torch.int32, device="cuda:0")
	args = (None, None, None, 0.0, kw.get("causal", False), None, kl, kw.get("window"))
	o, lse = op.fwd(q.cuda(), k.cuda(), v.cuda(), *args)
	g = op.bwd(q.cuda(), k.cuda(), v.cuda(), o, lse, do.cuda(), *args)
	for b, h in ((0, 0), (B - 1, H - 1)):
		bs, hs = slice(b, b + 1), slice(h, h + 1)
		want = O.attention_bwd(*[f64(x[bs, :, hs]) for x in (q, k, v, do)], causal=kw.get("causal", False), window=kw.get("window"),
		                       kv_lens=None if kv_lens is None else kv_lens[bs])
		check_grads([x[bs, :, hs] for x in g], want, f"Sq{Sq} Sk{Sk} D{D} {kw} b{b} h{h}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
	"how,B,S,Hq,Hkv,D,window",
	[
		("split", 1, 2048, 32, 8, 80, None),                 # the steps of a key tile over several workgroups that leave partial sums
		("split, blocks", 1, 2048, 32, 8, 80, (700, 0)),     # ... block by block
		("split, blocks", 1, 2001, 32, 8, 96, (1000, 0)),    # ... a last key tile and a last row tile that are not whole
		("blocks", 3, 1030, 40, 20, 72, None),               # block by block, two q-heads a kv-head
		("one round", 4, 1024, 32, 16, 88, None),            # 512 workgroups of a causal mask: not block by block
		("paired", 1, 2048, 32, 32, 88, None),               # two key tiles a workgroup
		("paired", 1, 2030, 64, 32, 96, None),
	],
)
def test_short_rows_by_the_plan_of_dkdv(how, B, S, Hq, Hkv, D, window, dtype):
	q, k, v, do, _ = make_inputs(B, S, S, Hq, Hkv, D, dtype, seed=S + D)
	qd, kd, vd, dod = (x.cuda() for x in (q, k, v, do))
	# (the launcher's choice, from the sizes)
	p, lib = op._block(128, q, k, v, None, None, 0.1, 0.0, True, None), _lib.load()
	least, split = lib.fa2_bwd_scratch_bytes(ctypes.byref(p)), lib.fa2_bwd_split_scratch_bytes(ctypes.byref(p))
	parts = (split - least) // (B * Hkv * S * 2 * 128 * 4) if split else 1
	tiles = (S + 127) // 128
	pairs, grid = (tiles + 1) // 2 * B * Hkv, B * Hkv * tiles * parts
	assert (parts > 1) == ("split" in how)
	assert (parts == 1 and window is None and tiles >= 16 and (pairs % 256 == 0 or pairs >= 2048)) == (how == "paired")
	assert how == "paired" or (grid >= (512 if window else 640 if parts > 1 else 513)) == ("blocks" in how)
	o, lse = op.fwd(qd, kd, vd, causal=True, window=window)
	grads = op.bwd(qd, kd, vd, o, lse, dod, causal=True, window=window)
	for b, hk in ((0, 0), (B - 1, Hkv - 1)):
		r = Hq // Hkv
		bs, hs, kv = slice(b, b + 1), slice(hk * r, hk * r + r), slice(hk, hk + 1)
		a = [f64(x) for x in (q[bs, :, hs], k[bs, :, kv], v[bs, :, kv], do[bs, :, hs])]
		check_grads([x[bs, :, y] for x, y in zip(grads, (hs, kv, kv))], O.attention_bwd(*a, causal=True, window=window), f"{how} S{S} D{D} b{b} hk{hk}")
