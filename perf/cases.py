"""Performance cases of the attention operator: what a user of this package has it do, from one token of decoding to training
over 32768 tokens, through its public entry points (`FlashAttention.__call__`, and `hip_flash_attention` for the operands that
the facade has no argument for: key lengths and the sliding window) with torch's autograd for the gradients.

A case is a dict of plain values:
  B, Sq, Sk, Hq, Hkv, D   q is [B, Sq, Hq, D]; k and v are [B, Sk, Hkv, D]
  dtype                   "bf16" | "fp16"
  causal                  bottom-right aligned causal mask
  bias                    "" | "shared" ([B, 1, Sq, Sk], padded keys folded in) | "head" ([B, Hq, Sq, Sk])
  mask                    2-D right-padded attention_mask [B, S]
  kv_lens                 number of valid keys per batch row (a cache that is filled to different lengths)
  window                  0, or how many keys a row sees to its left (causal sliding window)
  p                       dropout probability
  train                   forward and backward (gradients of q, k, v), else forward only
"""

import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "jax-flash-attn2_amd")
if _PACKAGE not in sys.path:
	sys.path.insert(0, _PACKAGE)

from jax_flash_attn2 import AttentionConfig, Backend, FlashAttention, Platform, hip_flash_attention  # noqa: E402

_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(B, Sq, Sk, Hq, Hkv, D, dtype="bf16", causal=False, bias="", mask=False, kv_lens=False, window=0, p=0.0, train=False):
	return dict(B=B, Sq=Sq, Sk=Sk, Hq=Hq, Hkv=Hkv, D=D, dtype=dtype, causal=causal, bias=bias, mask=mask, kv_lens=kv_lens, window=window, p=p,
	            train=train)


def listed():
	cases = {
		# one sequence generates a token from a short cache: the smallest call, all latency
		"decode_one_sequence": _case(1, 1, 1029, 32, 8, 128),
		# a serving batch generates a token each, from caches of 8192 slots that are filled to different lengths: K and V stream
		"decode_batch": _case(8, 1, 8192, 32, 8, 128, kv_lens=True),
		# the example of the project's documentation: a short causal prompt in half precision
		"short_prompt": _case(2, 512, 512, 16, 4, 64, "fp16", causal=True),
		# a long prompt is taken in pieces: a ragged piece of new queries over everything cached so far
		"prompt_chunk": _case(1, 1000, 9000, 32, 8, 128, causal=True),
		# training of an image encoder: many short sequences of odd length, a head dim between the kernels' own
		"image_encoder_train": _case(64, 257, 257, 16, 16, 80, "fp16", train=True),
		# training of a text encoder on padded sentences (2-D attention mask)
		"padded_text_train": _case(32, 511, 511, 12, 12, 64, "fp16", mask=True, train=True),
		# training step of an 8-billion-parameter decoder's attention at 4096 tokens (the benchmark's default workload)
		"decoder_train": _case(4, 4096, 4096, 32, 8, 128, causal=True, train=True),
		# padded multi-head attention with a bias that all heads share (the benchmark's padded workload)
		"shared_bias_train": _case(8, 2048, 2048, 16, 16, 64, bias="shared", train=True),
		# attention with a learned bias per head, forward (a shape of the benchmark's grid)
		"head_bias_forward": _case(2, 4096, 4096, 32, 16, 128, bias="head"),
		# wide heads with dropout in training (the benchmark's dropout workload)
		"wide_dropout_train": _case(8, 2048, 2048, 16, 16, 256, causal=True, p=0.1, train=True),
		# a sliding window over a long sequence of odd length, training
		"window_train": _case(1, 8191, 8191, 32, 8, 128, causal=True, window=1023, train=True),
		# long-context training (the benchmark's 32768-token workload): the largest call
		"long_context_train": _case(1, 32768, 32768, 64, 8, 128, causal=True, train=True),
	}
	return [dict(c, name=name) for name, c in cases.items()]


def _log_int(rng, lo, hi):
	"""An integer spread over the logarithm of [lo, hi]."""
	return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
	Hkv = rng.choice([4, 8, 12, 16])
	return Hkv * rng.choice([1, 1, 2, 4]), Hkv


def draw(rng):
	"""One more case of the same kinds of use: decoding, a prompt or a piece of one, an encoder, a padded batch, a decoder, a bias,
	dropout, a window - sizes over the whole range of the listed cases, ragged ones included."""
	kind = rng.choice(["decode", "prompt", "encoder", "padded", "decoder", "shared_bias", "head_bias", "dropout", "window"])
	dtype = rng.choice(["bf16", "bf16", "fp16"])
	Hq, Hkv = _heads(rng)
	if kind == "decode":
		B, Sk = _log_int(rng, 1, 64), _log_int(rng, 512, 16384)
		return _case(B, 1, Sk, Hq, Hkv, rng.choice([64, 128, 128]), dtype, kv_lens=B > 1)
	if kind == "prompt":
		Sq = _log_int(rng, 64, 4096)
		return _case(_log_int(rng, 1, 4), Sq, Sq + rng.choice([0, _log_int(rng, 128, 8192)]), Hq, Hkv, rng.choice([64, 128, 256]), dtype, causal=True)
	if kind == "encoder":
		S, H = _log_int(rng, 100, 1100), rng.choice([12, 16])
		return _case(_log_int(rng, 4, 64), S, S, H, H, rng.choice([64, 80, 96]), dtype, train=True)
	if kind == "padded":
		S, H = _log_int(rng, 128, 2048), rng.choice([12, 16])
		return _case(_log_int(rng, 2, 32), S, S, H, H, rng.choice([64, 128]), dtype, causal=rng.random() < 0.3, mask=True, train=True)
	S = _log_int(rng, 512, 8192)
	# (as many batch rows as a step of about 8192 tokens has)
	B = _log_int(rng, 1, max(1, 8192 // S))
	if kind == "decoder":
		return _case(B, S, S, Hq, Hkv, rng.choice([64, 128, 128, 256]), dtype, causal=True, train=True)
	if kind == "shared_bias":
		S = min(S, 4096) // 8 * 8
		return _case(8192 // S, S, S, Hkv, Hkv, rng.choice([64, 128]), dtype, bias="shared", train=True)
	if kind == "head_bias":
		return _case(B, S // 8 * 8, S // 8 * 8, Hq, Hkv, rng.choice([64, 128, 256]), dtype, bias="head")
	if kind == "dropout":
		return _case(B, S, S, Hq, Hkv, rng.choice([64, 128, 256]), dtype, causal=rng.random() < 0.7, p=rng.choice([0.1, 0.2]), train=True)
	return _case(B, S, S, Hq, Hkv, rng.choice([64, 128]), dtype, causal=True, window=_log_int(rng, 128, 2048) - 1, train=True)


def _lengths(seed, B, S):
	"""How far each row of a batch is filled: between half and all of S, the same on every machine."""
	return np.random.default_rng(seed).integers((S + 1) // 2, S + 1, B)


def prepare(case, seed):
	"""The operator object and its inputs on the GPU: normally distributed activations (scores of standard deviation 1), the mask
	or the lengths of the batch, the bias, and in training the gradient that arrives from behind."""
	dev, dt = torch.device("cuda"), _DTYPE[case["dtype"]]
	B, Sq, Sk, Hq, Hkv, D = (case[n] for n in ("B", "Sq", "Sk", "Hq", "Hkv", "D"))
	gen = torch.Generator(device=dev).manual_seed(seed)

	def normal(*shape):
		return torch.empty(shape, dtype=dt, device=dev).normal_(generator=gen)

	state = dict(q=normal(B, Sq, Hq, D), k=normal(B, Sk, Hkv, D), v=normal(B, Sk, Hkv, D))
	if case["train"]:
		for x in state.values():
			x.requires_grad_()
		state["dout"] = normal(B, Sq, Hq, D)
	kw = dict(causal=case["causal"])
	if case["bias"] == "head":
		kw["bias"] = normal(B, Hq, Sq, Sk)
	elif case["bias"] == "shared":
		# a bias that falls off with the distance; keys beyond a row's length get the lowest finite value
		i, j = torch.arange(Sq, device=dev), torch.arange(Sk, device=dev)
		near = 1.0 / (1.0 + (i[:, None] - j[None, :]).abs().float())
		valid = j[None, :] < torch.from_numpy(_lengths(seed, B, Sk)).to(dev)[:, None]
		kw["bias"] = torch.where(valid[:, None, None, :], near, torch.finfo(dt).min).to(dt)
	if case["mask"]:
		valid = torch.from_numpy(_lengths(seed, B, Sk)).to(dev)
		kw["attention_mask"] = torch.arange(Sk, device=dev)[None, :] < valid[:, None]
	if case["p"] > 0:
		kw.update(dropout_prob=case["p"], dropout_seed=seed)
	if case["kv_lens"]:
		kw["kv_lens"] = torch.from_numpy(_lengths(seed, B, Sk)).to(device=dev, dtype=torch.int32)
	if case["window"]:
		kw["window_size"] = (case["window"], 0)
	if case["kv_lens"] or case["window"]:
		state["attend"] = hip_flash_attention
	else:
		state["attend"] = FlashAttention(AttentionConfig(backend=Backend.GPU, platform=Platform.HIP))
	state["kw"] = kw
	return state


def run(state):
	q, k, v = state["q"], state["k"], state["v"]
	if "dout" not in state:
		with torch.no_grad():
			return state["attend"](q, k, v, **state["kw"])
	out = state["attend"](q, k, v, **state["kw"])
	dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
	return {"out": out, "dq": dq, "dk": dk, "dv": dv}


def _pairs(case):
	"""(row, key) pairs that a head of a batch row has to look at, on average over the lengths."""
	Sq, Sk = case["Sq"], case["Sk"]
	if case["causal"]:
		last = np.arange(Sq, dtype=np.int64) + Sk - Sq
		first = np.maximum(last - case["window"], 0) if case["window"] else 0
		n = float(np.maximum(last + 1 - first, 0).sum())
	else:
		n = float(Sq) * Sk
	if case["mask"]:
		n *= 7 / 12  # mean square of a length between a half and one
	elif case["kv_lens"]:
		n *= 3 / 4
	return n


def work(case):
	"""Matrix products: 2 in the forward, 5 in the backward (scores, dP, dV, dK, dQ); bytes: q, k, v, the bias and the incoming
	gradient once, the output and the gradients once.  What a mask or length leaves out is not counted, on average over the seeds;
	keys that a bias hides are, since only the bias says so."""
	B, Sq, Sk, Hq, Hkv, D = (case[n] for n in ("B", "Sq", "Sk", "Hq", "Hkv", "D"))
	flops = 4.0 * B * Hq * D * _pairs(case) * (3.5 if case["train"] else 1.0)
	rows, keys = float(B * Sq * Hq * D), float(B * Sk * Hkv * D)
	if case["kv_lens"] or case["mask"]:
		keys *= 3 / 4
	if case["mask"]:
		rows *= 3 / 4
	elements = 2 * rows + 2 * keys
	if case["train"]:
		elements += 2 * rows + 2 * keys
	if case["bias"]:
		elements += float(B) * (Hq if case["bias"] == "head" else 1) * Sq * Sk
	return {"bytes": 2 * elements, "flops": flops}


def tolerance(case):
	"""Four times what the results are off by from an evaluation in 64 bits of the same inputs: in the 2-norm 0.0026 in bfloat16 and
	0.0003 in half precision, whatever the size; the largest single difference, over the root mean square of the result, is 0.016 and
	0.0018 - and under a causal mask, where the first rows are an order of magnitude larger than the last, 0.24 at 32768 tokens in
	bfloat16 (half precision resolves eight times finer)."""
	half = case["dtype"] == "fp16"
	if case["causal"]:
		return {"rel": 0.0012 if half else 0.0105, "max": 0.12 if half else 0.95}
	return {"rel": 0.0012 if half else 0.0105, "max": 0.0075 if half else 0.07}
