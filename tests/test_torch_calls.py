"""The extension that makes the torch operator's calls fills the parameter block the Python code fills, for every form of a call that it
takes, and leaves the others - and every error of an argument's form - to the Python code."""

import ctypes
import itertools
import math
import os
import subprocess
import sys

import pytest
import torch

from jax_flash_attn2 import _fa2_torch, _hip_op as op, _lib
from jax_flash_attn2._checks import check_shapes

_CALL = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.POINTER(_lib.Fa2Params), ctypes.c_void_p)


class _Recorder:
	"""Stands in for the two launching entry points; the others are the library's own."""

	def __init__(self, rc=0):
		self.rc, self.seen = rc, []
		self.keep = _CALL(self._call)
		lib = _lib.load()
		at = ctypes.cast(self.keep, ctypes.c_void_p).value
		rest = ("fa2_validate", "fa2_fwd_scratch_bytes", "fa2_bwd_scratch_bytes", "fa2_bwd_split_scratch_bytes")
		self.bound = _fa2_torch.bind(at, at, *(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in rest))

	def _call(self, p, stream):
		self.seen.append((_lib.Fa2Params.from_buffer_copy(p.contents), stream))
		return self.rc


def _x(*shape, dtype=torch.bfloat16, form="plain"):
	B, S, H, D = shape
	if form == "plain":
		return torch.zeros(shape, dtype=dtype)
	if form == "heads first":  # [B, H, S, D] in memory
		return torch.zeros((B, H, S, D), dtype=dtype).transpose(1, 2)
	if form == "slice":  # of fused rows, 16-byte aligned
		return torch.zeros((B, S, H, 3 * D), dtype=dtype)[..., D : 2 * D]
	if form == "one batch row":
		return torch.zeros((1, S, H, D), dtype=dtype).expand(B, S, H, D)
	if form == "reversed axes":
		return torch.zeros((D, H, S, B), dtype=dtype).permute(3, 2, 1, 0)
	if form == "far rows":  # beyond what the kernels address short rows by
		far = 0x7FFFFFFF // 256 // 8 * 8 + 8
		return torch.empty((S - 1) * far + H * D, dtype=dtype).as_strided(shape, (S * far, far, D, 1))
	assert form == "odd address"
	n = B * S * H * D
	return torch.zeros(n + 8, dtype=dtype)[1 : n + 1].view(shape)


def _fields(p):
	out = {}
	for name, t in _lib.Fa2Params._fields_:
		v = getattr(p, name)
		out[name] = (v.ptr, v.stride_b, v.stride_s, v.stride_h) if t is _lib.Fa2Tensor else v
	return out


def _same(p, want, *own):
	a, b = _fields(p), _fields(want)
	for n in ("scratch", "scratch_bytes", *own):
		a.pop(n), b.pop(n)
	assert a == b


def _scale(q, s):
	return 1.0 / math.sqrt(q.shape[-1]) if s is None else s


_SIZES = [(2, 5, 9, 4, 2, 64), (1, 1, 1029, 32, 8, 128), (2, 130, 130, 2, 2, 256), (1, 257, 257, 2, 1, 80), (1, 40, 40, 1, 1, 96)]
_FORMS = ["plain", "heads first", "slice", "one batch row", "odd address"]


def _in_order(x, short):
	"""Whether the kernels take the tensor as it lies (`short`: rows of fewer columns than theirs)."""
	sb, ss, sh, sd = x.stride()
	return sd == 1 and not (sb | ss | sh) % 8 and not x.data_ptr() % 16 and not (short and ss > 0x7FFFFFFF // 256)


def _check_forward(rec, q, k, v):
	B, Sq, Hq, D = q.shape
	call = (None, None, None, 0.0, True, None, None, None, 0.0)
	Dk, lib, launched = op._kernel_head_dim(D), _lib.load(), len(rec.seen)
	res = _fa2_torch.forward(rec.bound, q, k, v, *call, 77)
	want = (None, None, _scale(q, None), 0.0, True, None, None, None, 0.0)
	served = all(_in_order(x, D < Dk) for x in (q, k, v)) and (D == Dk or op._runs_unpadded(lib, 0, Dk, q, k, v, *want))
	assert (res is not None) == served and len(rec.seen) == launched + served
	if not served:
		return False
	out, lse = res
	assert out.shape == q.shape and out.is_contiguous() and out.dtype == q.dtype and lse.shape == (B, Hq, Sq) and lse.dtype == torch.float32
	p, stream = rec.seen[-1]
	assert stream == 77
	_same(p, op._block(Dk, q, k, v, *want, op._t4(out), lse))
	assert (p.scratch_bytes or 0) == lib.fa2_fwd_scratch_bytes(ctypes.byref(p))
	assert bool(p.scratch) == bool(p.scratch_bytes)
	return True


def _check_backward(rec, q, k, v, out, dout):
	B, Sq, Hq, D = q.shape
	call = (None, None, None, 0.0, True, None, None, None, 0.0)
	Dk, lib, launched = op._kernel_head_dim(D), _lib.load(), len(rec.seen)
	lse = torch.zeros((B, Hq, Sq))
	res = _fa2_torch.backward(rec.bound, q, k, v, *call, out, lse, dout, 5)
	want = (None, None, _scale(q, None), 0.0, True, None, None, None, 0.0)
	served = all(_in_order(x, D < Dk) for x in (q, k, v, out, dout)) and (D == Dk or op._runs_unpadded(lib, 1, Dk, q, k, v, *want))
	assert (res is not None) == served and len(rec.seen) == launched + served
	if not served:
		return False
	dq, dk, dv = res
	p, stream = rec.seen[-1]
	assert stream == 5 and dq.shape == q.shape and dk.shape == k.shape and dv.shape == v.shape
	assert dq.is_contiguous() and dk.is_contiguous() and dv.is_contiguous()
	_same(p, op._block(Dk, q, k, v, *want, op._t4(out), lse, (op._t4(dout), op._t4(dq), op._t4(dk), op._t4(dv))))
	assert p.scratch and p.scratch_bytes == max(256, lib.fa2_bwd_scratch_bytes(ctypes.byref(p)), lib.fa2_bwd_split_scratch_bytes(ctypes.byref(p)))
	return True


@pytest.mark.parametrize("B,Sq,Sk,Hq,Hkv,D", _SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_blocks_over_strides(B, Sq, Sk, Hq, Hkv, D, dtype):
	rec, served = _Recorder(), []
	for fq, fk in itertools.product(_FORMS, _FORMS):
		q, k, v = _x(B, Sq, Hq, D, dtype=dtype, form=fq), _x(B, Sk, Hkv, D, dtype=dtype, form=fk), _x(B, Sk, Hkv, D, dtype=dtype)
		served.append(_check_forward(rec, q, k, v))
		served.append(_check_forward(rec, q, v, k))
		for fo in _FORMS:
			o, do = _x(B, Sq, Hq, D, dtype=dtype), _x(B, Sq, Hq, D, dtype=dtype, form=fo)
			served.append(_check_backward(rec, q, k, v, o, do))
			served.append(_check_backward(rec, q, v, k, do, o))
	assert any(served) and not all(served)


@pytest.mark.parametrize("D", [64, 80])
def test_blocks_of_rows_far_apart(D):
	rec = _Recorder()
	near, far = _x(1, 2, 1, D), _x(1, 2, 1, D, form="far rows")
	for i in range(3):
		assert _check_forward(rec, *(far if i == j else near for j in range(3))) == (D == 64)
	for i in range(5):
		assert _check_backward(rec, *(far if i == j else near for j in range(5))) == (D == 64)


def _biases(B, Hq, Hkv, Sq, Sk):
	for b, h in itertools.product((1, B), (1, Hkv, Hq)):
		for dt in (torch.float16, torch.bfloat16, torch.float32, torch.uint8, torch.bool):
			yield torch.zeros((b, h, Sq, Sk), dtype=dt)
	yield torch.zeros((B, Hq, Sq, Sk + 5))[..., :Sk]
	yield torch.zeros((1, 1, 1, Sk)).expand(B, Hq, Sq, Sk)


def test_blocks_over_options():
	rec = _Recorder()
	B, Sq, Sk, Hq, Hkv, D = 2, 6, 10, 4, 2, 64
	q, k, v = _x(B, Sq, Hq, D), _x(B, Sk, Hkv, D), _x(B, Sk, Hkv, D)
	lens, seed = torch.full((B,), 3, dtype=torch.int32), torch.tensor([5])
	full = dict(bias=None, seqlens=None, scale=None, p=0.0, causal=False, seed=None, kv_lens=None, window=None, softcap=0.0)
	calls = [dict(full, bias=b) for b in _biases(B, Hq, Hkv, Sq, Sk)]
	calls += [dict(full, seqlens=lens), dict(full, kv_lens=lens), dict(full, scale=0.3), dict(full, scale=2), dict(full, causal=True)]
	calls += [dict(full, p=0.2, seed=s) for s in (None, 0, 7, -3, 1 << 63, (1 << 70) + 9, seed)]
	calls += [dict(full, p=0), dict(full, softcap=30.0), dict(full, softcap=None), dict(full, softcap=5)]
	calls += [dict(full, window=w) for w in ((3, 0), (-1, -1), (-7, 2), (1 << 40, -(1 << 70)), (1 << 70, 0))]
	for c in calls:
		res = _fa2_torch.forward(rec.bound, q, k, v, *c.values(), 0)
		assert res is not None, c
		want = dict(c, scale=_scale(q, c["scale"]), bias=op._prep_bias(c["bias"]))
		_same(rec.seen[-1][0], op._block(D, q, k, v, *want.values(), op._t4(res[0]), res[1]))


def test_what_is_left_to_the_python_code():
	rec = _Recorder()
	q = _x(1, 4, 2, 64)
	plain = [None, None, None, 0.0, False, None, None, None, 0.0]

	def served(*qkv, **change):
		call = list(plain)
		for i, x in change.values():
			call[i] = x
		return _fa2_torch.forward(rec.bound, *qkv, *call, 0) is not None

	assert served(q, q, q)
	assert not served(q, _x(1, 4, 2, 64, form="odd address"), q)
	assert not served(_x(1, 4, 2, 64, form="reversed axes"), q, q)
	for D in (32, 50, 72 + 4, 104, 200):
		assert not served(*(_x(1, 4, 2, D) for _ in range(3)))
	assert not served(*(x.float() for x in (q, q, q)))
	assert not served(*(x.as_subclass(type("Other", (torch.Tensor,), {})) for x in (q, q, q)))
	for i, x in [(0, torch.zeros(1, 1, 4, 4, dtype=torch.float64)), (0, torch.zeros(1, 1, 4, 4).mT), (0, torch.zeros(4, 4)), (2, torch.tensor(0.1)), (2, 1e300),
	             (4, 1), (4, None), (5, 2.0), (5, True), (5, torch.tensor([1, 2])), (6, torch.tensor([4])), (6, torch.zeros(2, dtype=torch.int32)), (7, [1, 0]), (7, (1, 0, 0)),
	             (7, (1.0, 0)), (8, True)]:
		assert not served(q, q, q, change=(i, x)), (i, x)
	assert len(rec.seen) == 1
	# the code of an error comes back as a number
	assert _fa2_torch.forward(_Recorder(rc=-12).bound, q, q, q, *plain, 0) == -12


def _takes(*args):
	try:
		check_shapes(*args)
	except Exception:
		return False
	return True


def test_checks():
	"""What the extension passes is what check_shapes() passes; a call that differentiates keeps its autograd function."""
	z = torch.zeros
	q = z(2, 4, 4, 64, dtype=torch.float16)
	others = [q, z(2, 6, 2, 64, dtype=torch.float16), z(2, 4, 3, 64, dtype=torch.float16), z(1, 4, 4, 64, dtype=torch.float16), z(2, 4, 4, 32, dtype=torch.float16), z(2, 4, 4, 64),
	          z(2, 4, 4, 64, dtype=torch.bfloat16)]
	biases = [None, z(2, 4, 4, 4), z(1, 1, 4, 4), z(2, 2, 4, 6), z(3, 1, 4, 4), z(2, 3, 4, 4), z(2, 4, 4, 5)]
	masks = [None, z(2, 4, dtype=torch.bool)]
	for k, v, bias, mask in itertools.product(others, others, biases, masks):
		assert bool(_fa2_torch.checked(q, k, v, bias, mask)) == _takes(q, k, v, bias, mask)
	k = q.clone()
	assert _fa2_torch.checked(q, k, q, None, None) == 3
	k.requires_grad_()
	assert _fa2_torch.checked(q, k, q, None, None) == 1
	with torch.no_grad():
		assert _fa2_torch.checked(q, k, q, None, None) == 3
	bias = z(1, 1, 4, 4, requires_grad=True)
	assert _fa2_torch.checked(q, q, q, bias, None) == 1
	with torch.autograd.forward_ad.dual_level(), torch.no_grad():
		dual = torch.autograd.forward_ad.make_dual(q, q.clone())
		assert _fa2_torch.checked(q, dual, q, None, None) == 1
	seen = []
	torch.func.vmap(lambda x: (seen.append(_fa2_torch.checked(x, x, x, None, None)), x)[1])(z(3, 2, 4, 4, 64, dtype=torch.float16))
	torch.jit.trace(lambda x: (seen.append(_fa2_torch.checked(x, x, x, None, None)), x * 1)[1], (q,), check_trace=False)
	assert seen and all(not f & 2 for f in seen), seen


def test_operands_in_other_memory_are_refused():
	"""An operand that is not where q is, lengths or a logsumexp of another type: nothing is launched, the Python code names it."""
	rec = _Recorder()
	q = _x(2, 4, 2, 64)
	out, lse = torch.empty_like(q), torch.zeros(2, 2, 4)
	lens = torch.full((2,), 3, dtype=torch.int32)
	sound = dict(k=q, v=q, bias=torch.zeros(1, 1, 4, 4), seqlens=None, kv_lens=lens, out=out, lse=lse, dout=q)
	cases = [(n, x.to("meta")) for n, x in sound.items() if x is not None] + [("seqlens", lens.to("meta"))]
	cases += [("seqlens", lens.long()), ("seqlens", lens[:1]), ("kv_lens", lens.long()), ("lse", lse.double()), ("lse", lse.mT), ("lse", lse[:1])]

	def block(d):
		return (q, d["k"], d["v"], d["bias"], d["seqlens"], None, 0.0, False, None, d["kv_lens"], None, 0.0)

	residuals = ("out", "lse", "dout")
	assert _fa2_torch.forward(rec.bound, *block(sound), 0) is not None
	assert _fa2_torch.backward(rec.bound, *block(sound), *(sound[n] for n in residuals), 0) is not None
	assert len(rec.seen) == 2
	for name, x in cases:
		d = dict(sound, **{name: x})
		if name not in residuals:
			assert _fa2_torch.forward(rec.bound, *block(d), 0) is None, name
			with pytest.raises(ValueError, match=name):
				op.fwd(*block(d))
		assert _fa2_torch.backward(rec.bound, *block(d), *(d[n] for n in residuals), 0) is None, name
		b = block(d)
		with pytest.raises(ValueError, match=name):
			op.bwd(*b[:3], *(d[n] for n in residuals), *b[3:])
	assert len(rec.seen) == 2


def test_other_threads_run_while_a_call_allocates_and_launches():
	held = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value  # (1 where the calling thread holds the interpreter's lock)
	rec = _Recorder()
	at = ctypes.cast(rec.keep, ctypes.c_void_p).value
	q = _x(1, 4, 2, 64)
	call = (q, q, q, None, None, None, 0.0, False, None, None, None, 0.0)
	# the size of the scratch is asked for between the allocation of the outputs and that of the scratch
	out, lse = _fa2_torch.forward(_fa2_torch.bind(at, at, held, held, held, held), *call, 0)
	assert not rec.seen[0][0].scratch
	for entry, args in ((_fa2_torch.forward, (0,)), (_fa2_torch.backward, (out, lse, q, 0))):
		assert isinstance(entry(_fa2_torch.bind(*[held] * 6), *call, *args), tuple)  # (an error code of 1 otherwise)


@pytest.mark.parametrize("how", ["missing", "of another torch"])
def test_without_the_extension(how):
	"""Python makes every call, says so once and refuses what it did."""
	code = """
import sys, types, warnings
import torch
import jax_flash_attn2
if sys.argv[1] == "missing":
	sys.modules["jax_flash_attn2._fa2_torch"] = None
else:
	other = sys.modules["jax_flash_attn2._fa2_torch"] = jax_flash_attn2._fa2_torch = types.ModuleType("other")
	other.built_for = "1.0 2.7"
with warnings.catch_warnings(record=True) as seen:
	warnings.simplefilter("always")
	from jax_flash_attn2 import _hip_op as op
assert op._fa2_torch is None
assert [w.category for w in seen if "_fa2_torch" in str(w.message)] == [RuntimeWarning]
q = torch.zeros(1, 4, 2, 64, dtype=torch.bfloat16)
for args, error in (((q, q, q), ValueError), ((q, q[:, :, :, :8], q), AssertionError)):
	try:
		op.flash_attention(*args)
	except error as e:
		print(type(e).__name__, e)
"""
	env = dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(op.__file__)))
	r = subprocess.run([sys.executable, "-c", code, how], env=env, capture_output=True, text=True, timeout=300)
	assert r.returncode == 0, r.stderr
	assert "ValueError Expected a cuda device" in r.stdout and "AssertionError key shape" in r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 80, 40])
def test_the_python_code_makes_the_same_calls(monkeypatch, D):
	g = torch.Generator(device="cuda").manual_seed(D)
	q, do = (torch.empty(2, 130, 4, D, dtype=torch.float16, device="cuda").normal_(generator=g) for _ in range(2))
	k, v = (torch.empty(2, 130, 2, D, dtype=torch.float16, device="cuda").normal_(generator=g) for _ in range(2))
	for x in (q, k, v):
		x.requires_grad_()
	got = []
	for ext in (_fa2_torch, None):
		monkeypatch.setattr(op, "_fa2_torch", ext)
		out = op.flash_attention(q, k, v, causal=True)
		with torch.no_grad():
			got.append((out, *torch.autograd.grad(out, (q, k, v), do), op.flash_attention(q, k, v, causal=True)))
	for a, b in zip(*got):
		assert torch.equal(a, b)


@pytest.mark.parametrize("which", ["softmax_scale", "dropout_prob", "softcap"])
def test_a_number_that_requires_a_gradient_keeps_the_autograd_function(monkeypatch, which):
	"""(The operator returns none for it, but its result is part of the graph.)"""
	monkeypatch.setattr(op, "fwd", lambda q, *a: (torch.zeros_like(q), torch.zeros(1)))
	q = _x(1, 4, 2, 64)
	x = torch.tensor(0.5, requires_grad=True)
	assert op.flash_attention(q, q, q, **{which: x}).requires_grad
	assert not op.flash_attention(q, q, q, **{which: x.detach()}).requires_grad
	with torch.no_grad():
		assert not op.flash_attention(q, q, q, **{which: x}).requires_grad
