"""The HIP attention operator: forward / backward calls into libfa2_hip.so and
the differentiation rule that ties them together.

Takes the place of the reference's per-platform operator
`jax_flash_attn2/flash_attention_triton/_flash_attention.py:27-157`
(`_jax_fwd_attention_call`, `_jax_bwd_attention_call`, `flash_attention_call`,
`flash_attention`): same argument list, same residuals (q, k, v, bias, mask,
out, lse, seed), gradients for q, k, v only.

Arrays here are torch tensors on a ROCm device - torch is used for device
memory and the stream handle only; every number is produced by the C ABI.  The
same two entry points are what the XLA-FFI handlers in csrc/fa2_xla_ffi.cc
forward to when the caller is JAX.
"""

from __future__ import annotations

import ctypes
import math
import sys
import typing as tp
import warnings

import torch

from . import _lib
from ._checks import check_shapes  # noqa: F401  (re-exported)
from ._lib import FA2_BF16, FA2_FP16, FA2_FP32, FA2_MASK_U8


def _load_extension():
	"""The extension that makes ordinary calls (csrc/fa2_torch.cpp), or None: the Python code below serves every call too, it only takes
	longer about it.  It is built for one torch and one Python."""
	here = f"{torch.__version__} {sys.version_info[0]}.{sys.version_info[1]}"
	try:
		from . import _fa2_torch as ext

		built_for = getattr(ext, "built_for", None)
		if built_for == here:
			return ext
		why = f"built for torch and Python {built_for}, not {here}"
	except ImportError as e:
		why = str(e)
	warnings.warn(f"the extension _fa2_torch is not used ({why}): calls spend more time on the host; `make -C csrc` builds it", RuntimeWarning, stacklevel=3)
	return None


_fa2_torch = _load_extension()

_DTYPES = {torch.float16: FA2_FP16, torch.bfloat16: FA2_BF16}
# (a uint8 / bool `bias` is a boolean mask, one byte per position: see fa2_params.bias_dtype)
_BIAS_DTYPES = {torch.float16: FA2_FP16, torch.bfloat16: FA2_BF16, torch.float32: FA2_FP32, torch.uint8: FA2_MASK_U8}


def _stream_ptr(device) -> int:
	# (what torch.cuda.current_stream(device).cuda_stream gives, without building the stream object)
	index = device.index
	if index is None:  # (a tensor in host memory)
		raise ValueError(f"Expected a cuda device, but got: {device}")
	return torch._C._cuda_getCurrentRawStream(index)


_NONE4 = (0, 0, 0, 0)  # an absent tensor


def _t4(x) -> tuple:
	"""[B, S, H, D] tensor -> pointer + element strides (D stride must be 1): the fields of an fa2_tensor."""
	return (x.data_ptr(), *x.stride()[:3])


# Head dims the kernels are built for.  Any other head dim up to 256 is zero-padded to the next
# one, as the reference pads to the next power of two (_forward_triton.py:525-526): zero
# columns of q / k leave the scores unchanged, zero columns of v and dO give zero columns of
# O, dV and dQ / dK, which are cut off again.  The softmax scale keeps using the true head dim.
# Where the kernels have a variant for the shorter rows (fa2_params.head_dim) nothing is padded.
HEAD_DIMS = (64, 128, 256)


def _kernel_head_dim(D: int) -> int:
	for d in HEAD_DIMS:
		if D <= d:
			return d
	raise ValueError(f"head dim {D} is not supported (at most {HEAD_DIMS[-1]})")


def _pad_d(x: torch.Tensor, Dp: int) -> torch.Tensor:
	return x if x.shape[-1] == Dp else torch.nn.functional.pad(x, (0, Dp - x.shape[-1]))


def _runs_unpadded(lib, which, D, q, k, v, *call) -> bool:
	"""Whether the library runs this forward (which = 0) / backward (1) on rows that are shorter than its head dim D."""
	return lib.fa2_validate(ctypes.byref(_block(D, q, k, v, *call)), which) != _lib.FA2_EUNSUPPORTED


def _usable(x: torch.Tensor) -> torch.Tensor:
	"""Kernels read 16 bytes at a time along D: unit D stride, 16-byte aligned rows."""
	sb, ss, sh, sd = x.stride()
	if sd != 1 or (sb | ss | sh) & 7 or x.data_ptr() & 15:
		return x.contiguous()
	return x


def _usable_short(x: torch.Tensor) -> torch.Tensor:
	"""The same for rows that are shorter than the kernels' head dim.  A padded copy of such rows would be in order whatever the
	tensor is, so what the library refuses of it is copied too: a contiguous tensor that is not aligned, rows too far apart."""
	sb, ss, sh, sd = x.stride()
	if sd != 1 or (sb | ss | sh) & 7 or x.data_ptr() & 15 or ss > 0x7FFFFFFF // 256:
		return x.clone(memory_format=torch.contiguous_format)
	return x


def _block(D, q, k, v, bias, seqlens, scale, p_drop, causal, seed, kv_lens=None, window=None, softcap=0.0, o=_NONE4, lse=None,
           backward=(_NONE4, _NONE4, _NONE4, _NONE4)):
	"""The parameter block of a call on rows of q.shape[3] columns in the kernels of head dim D.  `o` and `backward` (dO, dq, dk, dv)
	as _t4() gives them; scratch and the bias gradient are the caller's to add."""
	B, Sq, Hq, rows = q.shape
	_, Sk, Hkv, _ = k.shape
	seed, seed_dev = _seed_fields(seed, q.device)
	b = (0, 0, 0, 0, 0, 0)
	if bias is not None:
		b_b, b_h = bias.shape[:2]
		# broadcast rules of calc_bias_strides (_utils.py:169-190): size-1 axes get stride 0.
		# a bias with Hkv heads is read per KV group instead of being repeated to Hq heads
		# (the facade materialises that repeat, flash_attention.py:161-164)
		b = (bias.data_ptr(), _BIAS_DTYPES[bias.dtype], 1 if (b_h == Hkv and Hkv != Hq and b_h != 1) else 0,
		     0 if b_b == 1 else bias.stride(0), 0 if b_h == 1 else bias.stride(1), bias.stride(2))
	if kv_lens is not None and (kv_lens.dtype != torch.int32 or kv_lens.numel() != B or not kv_lens.is_contiguous()):
		raise ValueError("kv_lens must be a contiguous int32 tensor with one entry per batch row")
	# (a bound beyond 2^30 is none at all; kept within the 32 bits of the field)
	left, right = (0, 0) if window is None else (max(-1, min(int(w), 1 << 30)) for w in window)
	dout, dq, dk, dv = backward
	# (in the order of include/fa2.h)
	return _lib.Fa2Params.from_buffer_copy(_lib.PACKED.pack(
		_lib.PACKED.size, _DTYPES[q.dtype], B, Sq, Sk, Hq, Hkv, D, 1 if causal else 0, float(scale), float(p_drop), seed,
		*_t4(q), *_t4(k), *_t4(v), *o, 0 if lse is None else lse.data_ptr(),
		*b, 0 if seqlens is None else seqlens.data_ptr(),
		*dout, *dq, *dk, *dv, 0, 0,  # (scratch)
		seed_dev, 0 if kv_lens is None else kv_lens.data_ptr(),
		0 if window is None else 1, left, right, float(softcap or 0.0),
		0, 0, 0, 0,  # (dbias)
		rows))


def _seed_fields(seed, device):
	"""The dropout seed is a Python int (copied into the parameter block) or a one-element int64 tensor on the device,
	which the kernels read there: a seed that is itself the result of device work - as a traced `dropout_seed` is in
	the reference, an operand of the custom call (_forward_triton.py:553) - needs no host round trip."""
	if isinstance(seed, torch.Tensor):
		if seed.dtype != torch.int64 or seed.numel() != 1 or seed.device != device:
			raise ValueError("a tensor dropout_seed must be a one-element int64 tensor on the device of q")
		return 0, seed.data_ptr()
	return int(seed or 0) & 0xFFFFFFFFFFFFFFFF, 0


def _check_memory(q, seqlens=None, lse=None, **operands):
	"""The kernels are given bare addresses: an operand in host memory or on another GPU would be a memory fault there, one of another
	type wrong numbers.  (Pinned host memory has an address the GPU can read.)"""
	B, Sq, Hq = q.shape[:3]
	for name, x, dtype, n in (("seqlens", seqlens, torch.int32, B), ("lse", lse, torch.float32, B * Hq * Sq)):
		if x is not None and (x.dtype != dtype or x.numel() < n or not x.is_contiguous()):
			raise ValueError(f"{name} must be a contiguous {dtype} tensor with {n} entries")
	for name, x in (*operands.items(), ("seqlens", seqlens), ("lse", lse)):
		if x is not None and x.device != q.device and not (q.is_cuda and x.device.type == "cpu" and x.is_pinned()):
			raise ValueError(f"{name} is on {x.device}, q on {q.device}")


def _prep_bias(bias):
	if bias is None:
		return None
	if bias.dtype == torch.bool:
		bias = bias.view(torch.uint8)  # same bytes: 0 = masked
	if bias.dtype not in _BIAS_DTYPES:
		bias = bias.to(torch.float32)
	if bias.stride(3) != 1:
		bias = bias.contiguous()
	return bias


def _mask_operand(mask, q):
	"""A 4-D boolean mask [B|1, H|1, Sq, Sk] is handed to the kernels as it is, one byte per position.  They add the
	lowest finite value of q's dtype at masked positions, i.e. they compute what the reference's documentation
	spells as the bias where(mask, 0, finfo(dtype).min) (README.md:188) without that bias ever being built.
	(The reference's GPU path itself only takes the 2-D mask.)"""
	m = mask.to(device=q.device)
	m = m if m.dtype == torch.bool else m.ne(0)
	return m.contiguous() if m.stride(3) != 1 else m


def _seqlens_from_mask(attention_mask, q):
	"""The reference's GPU path takes a right-padded 2-D validity mask [B, S] and
	packs the valid tokens (_forward_triton.py:499-510).  Here the mask is reduced
	to one length per batch row which the kernels consume directly."""
	if attention_mask is None:
		return None
	if attention_mask.dim() != 2:
		raise ValueError("attention_mask must be a 2-D [batch, seq] right-padded validity mask; use bias for general masks")
	m = attention_mask.to(device=q.device)
	if m.dtype != torch.bool:
		m = m.ne(0)
	if not q.is_cuda or m.numel() == 0 or m.stride(1) != 1:
		return m.sum(dim=1, dtype=torch.int32).contiguous()
	lens = torch.empty((m.shape[0],), dtype=torch.int32, device=q.device)
	_lib.check(_lib.load().fa2_mask_lengths(m.data_ptr(), m.stride(0), m.shape[0], m.shape[1], lens.data_ptr(), _stream_ptr(q.device)))
	return lens


_bound = None


def _entry_points():
	"""The entry points of libfa2_hip.so as the extension module takes them."""
	global _bound
	lib = _lib.load()
	if _bound is None:
		names = ("fa2_fwd", "fa2_bwd", "fa2_validate", "fa2_fwd_scratch_bytes", "fa2_bwd_scratch_bytes", "fa2_bwd_split_scratch_bytes")
		_bound = _fa2_torch.bind(*(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in names))
	return _bound


def fwd(q, k, v, bias=None, seqlens=None, softmax_scale=None, dropout_prob=0.0, causal=False, dropout_seed=None, kv_lens=None,
        window=None, softcap=0.0):
	"""Returns (out [B,Sq,Hq,D] in q.dtype, lse [B,Hq,Sq] fp32 natural log)."""
	if _fa2_torch is not None and q.is_cuda:
		# an ordinary call: plain tensors in order for the kernels (anything else: None, and what follows copies, pads or refuses)
		res = _fa2_torch.forward(_entry_points(), q, k, v, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens, window,
		                         softcap, _stream_ptr(q.device))
		if res.__class__ is int:
			_lib.check(res)
		elif res is not None:
			return res
	_check_memory(q, seqlens, k=k, v=v, bias=bias, kv_lens=kv_lens)
	lib = _lib.load()
	D0 = q.shape[-1]
	D = _kernel_head_dim(D0)
	bias = _prep_bias(bias)
	scale = 1.0 / math.sqrt(D0) if softmax_scale is None else softmax_scale
	call = (bias, seqlens, scale, dropout_prob, causal, dropout_seed, kv_lens, window, softcap)
	rows = D0 if D0 != D and _runs_unpadded(lib, 0, D, q, k, v, *call) else D  # columns of the rows the library is given
	if rows == D:
		q, k, v = _usable(_pad_d(q, D)), _usable(_pad_d(k, D)), _usable(_pad_d(v, D))
	else:
		q, k, v = _usable_short(q), _usable_short(k), _usable_short(v)
	out = torch.empty_like(q, memory_format=torch.contiguous_format)
	lse = torch.empty((q.shape[0], q.shape[2], q.shape[1]), dtype=torch.float32, device=q.device)
	p = _block(D, q, k, v, *call, _t4(out), lse)
	ref = ctypes.byref(p)
	# short query over many keys: scratch lets the library split the keys over workgroups
	need = lib.fa2_fwd_scratch_bytes(ref)
	if need:
		scratch = torch.empty((need,), dtype=torch.uint8, device=q.device)
		p.scratch = scratch.data_ptr()
		p.scratch_bytes = need
	_lib.check(lib.fa2_fwd(ref, _stream_ptr(q.device)))
	return (out if rows == D0 else out[..., :D0]), lse


def bwd(q, k, v, out, lse, dout, bias=None, seqlens=None, softmax_scale=None, dropout_prob=0.0, causal=False,
        dropout_seed=None, kv_lens=None, window=None, softcap=0.0, need_dbias=False):
	"""Returns (dq, dk, dv) in the dtypes of q, k, v; dk/dv summed over each KV group.  With `need_dbias` a fourth
	result: the gradient of the additive bias, fp32, in the shape of `bias` (summed over the axes it is broadcast on;
	those sums are atomic adds in the dQ kernel - see fa2_params.dbias - so the buffer is as small as the bias)."""
	if _fa2_torch is not None and q.is_cuda and not need_dbias:
		res = _fa2_torch.backward(_entry_points(), q, k, v, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens, window,
		                          softcap, out, lse, dout, _stream_ptr(q.device))
		if res.__class__ is int:
			_lib.check(res)
		elif res is not None:
			return res
	_check_memory(q, seqlens, lse, k=k, v=v, bias=bias, kv_lens=kv_lens, out=out, dout=dout)
	lib = _lib.load()
	D0 = q.shape[-1]
	D = _kernel_head_dim(D0)
	bias = _prep_bias(bias)
	scale = 1.0 / math.sqrt(D0) if softmax_scale is None else softmax_scale
	call = (bias, seqlens, scale, dropout_prob, causal, dropout_seed, kv_lens, window, softcap)
	rows = D0 if D0 != D and _runs_unpadded(lib, 1, D, q, k, v, *call) else D
	q, k, v, out, dout = (_usable(_pad_d(x, D)) if rows == D else _usable_short(x) for x in (q, k, v, out, dout))
	Sq = q.shape[1]
	dq = torch.empty_like(q, memory_format=torch.contiguous_format)
	dk = torch.empty_like(k, memory_format=torch.contiguous_format)
	dv = torch.empty_like(v, memory_format=torch.contiguous_format)
	p = _block(D, q, k, v, *call, _t4(out), lse, (_t4(dout), _t4(dq), _t4(dk), _t4(dv)))
	# (the larger size, where it applies, lets the dK/dV kernel of a small grid split the q-heads of a group over workgroups)
	need = max(lib.fa2_bwd_scratch_bytes(ctypes.byref(p)), lib.fa2_bwd_split_scratch_bytes(ctypes.byref(p)))
	scratch = torch.empty((max(need, 256),), dtype=torch.uint8, device=q.device)
	p.scratch = scratch.data_ptr()
	p.scratch_bytes = scratch.numel()
	dbias = None
	if need_dbias:
		if bias is None or bias.dtype == torch.uint8:
			raise ValueError("the bias gradient needs a floating-point bias")
		# fp32, zero-filled (the kernel leaves skipped key tiles alone), in the SHAPE OF THE BIAS: on the axes the bias is
		# broadcast on (size-1 batch / head axis, Hkv heads) the dQ kernel accumulates with atomic adds, so the memory is
		# that of the bias itself and not B * Hq * Sq * Sk * 4 bytes.  Rows start on 16 bytes.
		Skp = (k.shape[1] + 3) // 4 * 4
		dbias = torch.zeros((bias.shape[0], bias.shape[1], Sq, Skp), dtype=torch.float32, device=q.device)[..., : k.shape[1]]
		p.dbias = dbias.data_ptr()
		p.dbias_stride_b = 0 if bias.shape[0] == 1 else dbias.stride(0)
		p.dbias_stride_h = 0 if bias.shape[1] == 1 else dbias.stride(1)
		p.dbias_stride_m = dbias.stride(2)
	_lib.check(lib.fa2_bwd(ctypes.byref(p), _stream_ptr(q.device)))
	if rows != D0:
		dq, dk, dv = dq[..., :D0], dk[..., :D0], dv[..., :D0]
	if need_dbias:
		return dq, dk, dv, dbias
	return dq, dk, dv


def dropout_mask(B, H, Sq, Sk, dropout_prob, dropout_seed, device) -> torch.Tensor:
	"""keep[b,h,i,j] (uint8) exactly as the kernels regenerate it."""
	lib = _lib.load()
	keep = torch.empty((B, H, Sq, Sk), dtype=torch.uint8, device=device)
	p = _lib.new_params()
	p.B, p.Hq, p.Hkv, p.Sq, p.Sk, p.D = B, H, H, Sq, Sk, 64
	p.p_drop = float(dropout_prob)
	p.seed, p.seed_dev = _seed_fields(dropout_seed, torch.device(device))
	_lib.check(lib.fa2_dropout_mask(ctypes.byref(p), keep.data_ptr(), _stream_ptr(keep.device)))
	return keep


class Plan:
	"""A filled parameter block with its output buffers, for callers that repeat
	the same call (benchmarks, graph capture): `forward()` / `backward()` only
	enqueue kernels, nothing is allocated per call."""

	def __init__(self, q, k, v, dout=None, bias=None, seqlens=None, softmax_scale=None, dropout_prob=0.0, causal=False,
	             dropout_seed=None, kv_lens=None, window=None, softcap=0.0):
		_check_memory(q, seqlens, k=k, v=v, bias=bias, kv_lens=kv_lens, dout=dout)
		self.lib = _lib.load()
		self.q, self.k, self.v = _usable(q), _usable(k), _usable(v)
		self.bias = _prep_bias(bias)
		self.seqlens = seqlens
		B, Sq, Hq, D = q.shape
		scale = 1.0 / math.sqrt(D) if softmax_scale is None else softmax_scale
		self.out = torch.empty((B, Sq, Hq, D), dtype=q.dtype, device=q.device)
		self.lse = torch.empty((B, Hq, Sq), dtype=torch.float32, device=q.device)
		self.kv_lens = kv_lens
		self.seed = dropout_seed  # (a device-resident seed must outlive the plan's calls)
		self.device = q.device
		backward = (_NONE4, _NONE4, _NONE4, _NONE4)
		if dout is not None:
			self.dout = _usable(dout)
			self.dq = torch.empty_like(self.q, memory_format=torch.contiguous_format)
			self.dk = torch.empty_like(self.k, memory_format=torch.contiguous_format)
			self.dv = torch.empty_like(self.v, memory_format=torch.contiguous_format)
			backward = (_t4(self.dout), _t4(self.dq), _t4(self.dk), _t4(self.dv))
		p = self.params = _block(D, self.q, self.k, self.v, self.bias, seqlens, scale, dropout_prob, causal, dropout_seed, kv_lens, window, softcap,
		                         _t4(self.out), self.lse, backward)
		if dout is not None:
			need = max(self.lib.fa2_bwd_scratch_bytes(ctypes.byref(p)), self.lib.fa2_bwd_split_scratch_bytes(ctypes.byref(p)))
		else:
			need = 0
		# one buffer serves both calls: the backward needs its scratch, the forward uses scratch when it splits a
		# short query over key ranges (the partial results do not outlive the forward call)
		need = max(need, self.lib.fa2_fwd_scratch_bytes(ctypes.byref(p)))
		if need:
			self.scratch = torch.empty((max(need, 256),), dtype=torch.uint8, device=q.device)
			p.scratch = self.scratch.data_ptr()
			p.scratch_bytes = self.scratch.numel()

	def forward(self):
		_lib.check(self.lib.fa2_fwd(ctypes.byref(self.params), _stream_ptr(self.device)))
		return self.out, self.lse

	def backward(self, stages: int = 7):
		_lib.check(self.lib.fa2_bwd_stages(ctypes.byref(self.params), _stream_ptr(self.device), stages))
		return self.dq, self.dk, self.dv


class _FlashAttentionFn(torch.autograd.Function):
	"""Differentiation rule; the torch spelling of the reference's
	`flash_attention_call.defvjp(_jax_fwd_attention_call, _jax_bwd_attention_call)`
	(_flash_attention.py:119-122).  Returns (dq, dk, dv) and None for everything else, as the reference does
	(_flash_attention.py:88) - unless the caller asked for the gradient of the bias (`bias_grad=True`)."""

	@staticmethod
	def forward(ctx, q, k, v, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens=None, window=None, softcap=0.0,
	            bias_grad=False):
		out, lse = fwd(q, k, v, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens, window, softcap)
		ctx.save_for_backward(q, k, v, bias, seqlens, out, lse, kv_lens)
		ctx.cfg = (softmax_scale, dropout_prob, causal, dropout_seed, window, softcap, bias_grad)
		return out

	@staticmethod
	def backward(ctx, dout):
		q, k, v, bias, seqlens, out, lse, kv_lens = ctx.saved_tensors
		softmax_scale, dropout_prob, causal, dropout_seed, window, softcap, bias_grad = ctx.cfg
		need_dbias = bool(bias_grad) and bias is not None and ctx.needs_input_grad[3]
		res = bwd(q, k, v, out, lse, dout, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens, window, softcap,
		          need_dbias=need_dbias)
		dbias = res[3].to(bias.dtype) if need_dbias else None
		return res[0], res[1], res[2], dbias, None, None, None, None, None, None, None, None, None


def flash_attention(
	q,
	k,
	v,
	attention_mask=None,
	bias=None,
	softmax_scale: tp.Optional[float] = None,
	dropout_prob: float = 0.0,
	causal: bool = False,
	dropout_seed: tp.Optional[int] = None,
	varlen_mode: bool = True,
	*,
	kv_lens=None,
	window_size=None,
	softcap: float = 0.0,
	bias_grad: bool = False,
):
	"""Same signature as the reference's `triton_flash_attention`
	(_flash_attention.py:125-157).  `varlen_mode` is accepted for source
	compatibility; padded batches are always handled in-kernel from per-row
	lengths, never by packing.  `kv_lens` (keyword only, not in the reference):
	int32 [B] number of valid keys per batch row - key padding that may be combined
	with a bias and with Sq != Sk, which the 2-D attention_mask may not.  `window_size` =
	(left, right) (keyword only): the sliding window of the reference's naive attention
	(refrence_call.py:32,55-75); a negative bound is none, causal sets right = 0.  `softcap` > 0
	(keyword only): scores become softcap * tanh(score / softcap) before bias and masks
	(refrence_call.py:33,48-51).  `bias_grad` (keyword only): also differentiate with respect to a floating-point
	`bias` that requires a gradient - off by default, as the reference returns no gradient for its bias
	(_flash_attention.py:88); costs a zero-filled fp32 buffer in the shape of the bias and, where the bias is
	broadcast over batch or heads, atomic adds in the dQ kernel (summation order not fixed)."""
	del varlen_mode
	if bias_grad and attention_mask is not None and attention_mask.dim() == 4:
		raise ValueError("bias_grad needs a floating-point bias, not a boolean mask")
	if attention_mask is not None and attention_mask.dim() == 4:
		assert bias is None, "Attention mask is not supported along with attention bias. Just use bias instead."
		bias, attention_mask = _mask_operand(attention_mask, q), None
	flags = 0 if _fa2_torch is None else _fa2_torch.checked(q, k, v, bias, attention_mask, softmax_scale, dropout_prob, softcap)
	if not flags:
		check_shapes(q, k, v, bias, attention_mask)
	seqlens = _seqlens_from_mask(attention_mask, q)
	if flags & 2:  # (nothing differentiates, batches or traces this call)
		return fwd(q, k, v, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens, window_size, softcap)[0]
	return _FlashAttentionFn.apply(q, k, v, bias, seqlens, softmax_scale, dropout_prob, causal, dropout_seed, kv_lens, window_size, softcap,
	                               bias_grad)
