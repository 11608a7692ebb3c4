"""Which form the forward takes at head dim 64 without bias (csrc/fa2_fwd_form.hpp), compiled for the host: (groups of waves, waves a SIMD)."""

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-flash-attn2_amd", "csrc")
SRC = """
#include "fa2_fwd_form.hpp"
extern "C" int form(int B, int Hq, int Hkv, int Sq, int Sk, int causal, int wl, int wr, int drop) {
	const fa2::FwdForm f = fa2::fwd_form_64(B, Hq, Hkv, Sq, Sk, causal, wl, wr, drop);
	return f.groups * 10 + f.waves;
}
extern "C" int is_open(int Sk, int wl) { return fa2::window_is_open(Sk, wl); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
	d = tmp_path_factory.mktemp("form")
	src, out = d / "form.cc", d / "form.so"
	src.write_text(SRC)
	subprocess.check_call([os.environ.get("CXX", "c++"), "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(out), str(src)])
	return ctypes.CDLL(str(out))


def _form(lib, B, Hq, Hkv, S, causal=True, window=(-1, 0), drop=False, Sk=None):
	return divmod(lib.form(B, Hq, Hkv, S, Sk or S, causal, *(window if causal else (window[0], window[1] or -1)), drop), 10)


@pytest.mark.parametrize("drop", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv", [(1, 1, 1), (2, 8, 2), (4, 16, 16), (7, 12, 3), (3, 32, 8)])
@pytest.mark.parametrize("S", [100, 193, 577, 892, 1063, 2049, 4000])
def test_a_window_that_hides_nothing_is_none(lib, B, Hq, Hkv, S, drop):
	for w in (S, 2 * S, 1 << 30):
		assert lib.is_open(S, w)
		assert _form(lib, B, Hq, Hkv, S, window=(w, 0), drop=drop) == _form(lib, B, Hq, Hkv, S, drop=drop)


def test_windows(lib):
	assert lib.is_open(900, 600) and not lib.is_open(900, 599) and lib.is_open(900, -1) and not lib.is_open(900, 0)
	# at most one workgroup a CU: by the keys that a row tile looks at, however long the window
	assert _form(lib, 2, 8, 8, 892, window=(1727, 0)) == (2, 2)
	assert _form(lib, 2, 4, 4, 4000, window=(896, 0)) == (2, 2) and _form(lib, 2, 4, 4, 4000, window=(897, 0)) == (3, 3)
	assert _form(lib, 2, 4, 4, 1000, window=(64, 0)) == (1, 4) and _form(lib, 2, 4, 4, 1000, window=(65, 0)) == (2, 2)
	# up to two: seventeen tiles of a window that hides keys
	assert _form(lib, 1, 16, 4, 4000, window=(896, 0)) == (1, 4) and _form(lib, 1, 16, 4, 4000, window=(897, 0)) == (2, 4)
	assert _form(lib, 4, 16, 16, 892, window=(500, 0)) == (1, 4) and _form(lib, 4, 16, 16, 892, window=(600, 0)) == (2, 4)
	assert _form(lib, 1, 16, 4, 4000, causal=False, window=(448, 449)) == (2, 4) and _form(lib, 1, 16, 4, 4000, causal=False, window=(448, 448)) == (1, 4)


def test_tiles_of_keys(lib):
	for n, form in ((192, (1, 4)), (193, (2, 2)), (1024, (2, 2)), (1025, (3, 3))):
		assert _form(lib, 2, 4, 2, 130, causal=False, Sk=n) == form
	for n, form in ((576, (1, 4)), (577, (2, 4))):
		assert _form(lib, 2, 100, 100, 130, causal=False, Sk=n) == form


def test_causal_grids_that_wait_for_their_longest_tiles(lib):
	one, two = (1, 4), (2, 4)
	# up to four workgroups a CU over more than 2048 keys, without dropout; groups placed by XCD or not
	for B, Hq, Hkv in ((1, 40, 8), (1, 36, 9)):
		assert _form(lib, B, Hq, Hkv, 2048) == one and _form(lib, B, Hq, Hkv, 2049) == two and _form(lib, B, Hq, Hkv, 2049, drop=True) == one
	assert _form(lib, 1, 32, 8, 4096) == two and _form(lib, 1, 32, 8, 4096, drop=True) == one and _form(lib, 1, 36, 9, 4096) == one
	# up to five and a half over more than 4096
	for drop in (False, True):
		assert _form(lib, 1, 32, 8, 4097, drop=drop) == two and _form(lib, 1, 32, 8, 5632, drop=drop) == two and _form(lib, 1, 32, 8, 5633, drop=drop) == one
	assert _form(lib, 2, 24, 24, 3200) == one
	# not where rows see about as many keys each
	assert _form(lib, 1, 32, 8, 3500, Sk=4000) == two and _form(lib, 1, 32, 8, 3499, Sk=4000) == one and _form(lib, 1, 32, 8, 3000, causal=False) == one
