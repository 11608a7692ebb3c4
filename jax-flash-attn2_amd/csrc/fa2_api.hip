// C ABI of libfa2_hip.so: argument validation and kernel dispatch.
// Declarations and the reference call sites they replace: include/fa2.h.
#include "../../include/fa2.h"

#include <math.h>
#include <string.h>

#include <mutex>

#include "fa2_kernels.hpp"

// Scratch of fa2_bwd_static(): one copy per GPU the library runs on, held until the process
// ends.  In host code this name is only a handle for hipGetSymbolAddress(), never an address.
static __device__ __align__(256) unsigned char scratch[FA2_STATIC_SCRATCH_BYTES];

namespace {

using fa2::KArgs;
using fa2::KTensor;

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Parameter blocks of earlier versions of the header are shorter (struct_size says which): they are
// completed with zeros.  Returns NULL for a NULL block or one shorter than the first version.
const fa2_params* complete(const fa2_params* p, fa2_params& local) {
	if (!p || p->struct_size < FA2_PARAMS_SIZE_V1) return nullptr;
	if (p->struct_size >= sizeof(fa2_params)) return p;
	memset(&local, 0, sizeof(local));
	memcpy(&local, p, p->struct_size);
	local.struct_size = sizeof(fa2_params);
	return &local;
}

int check_tensor(const fa2_tensor& t, bool required) {
	if (!t.ptr) return required ? FA2_EINVAL_PTR : FA2_OK;
	if (!aligned16(t.ptr)) return FA2_EINVAL_PTR;
	// 16-byte vector access along D needs every row start 16-byte aligned
	if (t.stride_b % 8 || t.stride_s % 8 || t.stride_h % 8) return FA2_EINVAL_STRIDE;
	// the tile copies address the rows of a tile (up to 128) with 32-bit byte offsets
	if (t.stride_s < 0 || t.stride_s > (int64_t)0x7fffffff / (2 * 128)) return FA2_EINVAL_STRIDE;
	return FA2_OK;
}

int esize(int dtype) { return dtype == FA2_FP32 ? 4 : dtype == FA2_MASK_U8 ? 1 : 2; }

KTensor conv(const fa2_tensor& t) {
	KTensor k;
	k.ptr = (char*)t.ptr;
	k.sb = t.stride_b * 2;
	k.ss = t.stride_s * 2;
	k.sh = t.stride_h * 2;
	return k;
}

// delta [B, Hq, Sq] fp32, rounded up to 256 bytes (p: a completed block)
size_t bwd_scratch_bytes(const fa2_params* p) {
	if (p->B <= 0 || p->Hq <= 0 || p->Sq <= 0) return 0;
	size_t n = (size_t)p->B * (size_t)p->Hq * (size_t)p->Sq * sizeof(float);
	return (n + 255) & ~(size_t)255;
}

// rows of fewer columns than the head dim of the tiles
bool short_rows(const fa2_params* p) { return p->head_dim > 0 && p->head_dim != p->D; }
bool fwd_takes_ranges(const fa2_params* p);

// own_scratch: the backward brings its scratch itself (fa2_bwd_static), p->scratch is not looked at
int validate(const fa2_params* p, int which, bool own_scratch = false) {
	if (!p) return FA2_EINVAL_STRUCT;
	if (p->seed_dev && ((uintptr_t)p->seed_dev & 7)) return FA2_EINVAL_PTR;
	if (p->dtype != FA2_FP16 && p->dtype != FA2_BF16) return FA2_EINVAL_DTYPE;
	if (p->B <= 0 || p->Sq <= 0 || p->Sk <= 0 || p->Hq <= 0 || p->Hkv <= 0 || p->D <= 0) return FA2_EINVAL_SHAPE;
	if (p->Hq % p->Hkv) return FA2_EINVAL_HEADS;
	if (p->D != 64 && p->D != 128 && p->D != 256) return FA2_EUNSUPPORTED;
	if (short_rows(p)) {
		// (up to 64 columns the tiles of head dim 64 would do, from 104 on there is too little to leave out)
		if (p->D != 128 || p->head_dim <= 64 || p->head_dim > 96 || p->head_dim % 8) return FA2_EUNSUPPORTED;
		if (p->bias || p->softcap > 0.f || p->p_drop > 0.f) return FA2_EUNSUPPORTED;
		// a forward for which the kernels of few query rows or the key ranges are the better ones runs on padded rows
		if (which == 0 && fwd_takes_ranges(p)) return FA2_EUNSUPPORTED;
	}
	if (!(p->p_drop >= 0.f && p->p_drop < 1.f)) return FA2_EINVAL_DROPOUT;
	if (!isfinite(p->scale) || !(p->scale > 0.f)) return FA2_EINVAL_SHAPE;
	if (!isfinite(p->softcap) || p->softcap < 0.f) return FA2_EINVAL_SHAPE;
	int rc;
	if ((rc = check_tensor(p->q, true))) return rc;
	if ((rc = check_tensor(p->k, true))) return rc;
	if ((rc = check_tensor(p->v, true))) return rc;
	if ((rc = check_tensor(p->o, true))) return rc;
	if (!p->lse || ((uintptr_t)p->lse & 3)) return FA2_EINVAL_PTR;
	if (p->bias) {
		if (p->bias_dtype != FA2_FP16 && p->bias_dtype != FA2_BF16 && p->bias_dtype != FA2_FP32 && p->bias_dtype != FA2_MASK_U8)
			return FA2_EINVAL_BIAS;
		if (((uintptr_t)p->bias % esize(p->bias_dtype)) != 0) return FA2_EINVAL_BIAS;
		if (p->bias_stride_b < 0 || p->bias_stride_h < 0 || p->bias_stride_m < p->Sk) return FA2_EINVAL_BIAS;
	}
	if (p->seqlens) {
		if (p->bias || p->Sq != p->Sk) return FA2_EINVAL_MASK;
		if ((uintptr_t)p->seqlens & 3) return FA2_EINVAL_PTR;
	}
	if (p->kv_lens && ((uintptr_t)p->kv_lens & 3)) return FA2_EINVAL_PTR;
	if (which == 1) {
		if ((rc = check_tensor(p->dout, true))) return rc;
		if ((rc = check_tensor(p->dq, true))) return rc;
		if ((rc = check_tensor(p->dk, true))) return rc;
		if ((rc = check_tensor(p->dv, true))) return rc;
		if (p->dbias) {
			if (!p->bias && !(p->softcap > 0.f)) return FA2_EINVAL_BIAS;
			if (!aligned16(p->dbias)) return FA2_EINVAL_BIAS;
			if (p->dbias_stride_b < 0 || p->dbias_stride_h < 0 || p->dbias_stride_m < p->Sk) return FA2_EINVAL_BIAS;
			if (p->dbias_stride_b % 4 || p->dbias_stride_h % 4 || p->dbias_stride_m % 4) return FA2_EINVAL_BIAS;
		}
		size_t need = bwd_scratch_bytes(p);
		if (own_scratch) {
			if (need > FA2_STATIC_SCRATCH_BYTES) return FA2_ESCRATCH_STATIC;
		} else if (!p->scratch || ((uintptr_t)p->scratch & 255) || p->scratch_bytes < need) {
			return FA2_ESCRATCH;
		}
	}
	return FA2_OK;
}

// an element is kept iff its 16-bit value is >= this
uint32_t drop_threshold(float p) {
	double t = floor((double)p * 65536.0);
	return t >= 65535.0 ? 0xFFFFu : (uint32_t)t;
}

void fill(const fa2_params* p, KArgs& a) {
	memset(&a, 0, sizeof(a));
	a.q = conv(p->q);
	a.k = conv(p->k);
	a.v = conv(p->v);
	a.o = conv(p->o);
	a.lse = p->lse;
	a.bias = (const char*)p->bias;
	if (p->bias) {
		int es = esize(p->bias_dtype);
		a.bias_sb = p->bias_stride_b * es;
		a.bias_sh = p->bias_stride_h * es;
		a.bias_sm = p->bias_stride_m * es;
		a.bias_dtype = p->bias_dtype;
		a.bias_group = p->bias_group ? 1 : 0;
		int valign = es == 4 ? 16 : es == 2 ? 8 : 4;
		// a masked position of a boolean mask adds the lowest finite value of the element type, which is what
		// where(mask, 0, finfo(dtype).min) passed as a bias would add
		a.mask_fill = p->dtype == FA2_BF16 ? -3.38953139e38f : -65504.f;
		a.bias_vec4 = (((uintptr_t)p->bias % valign) == 0 && a.bias_sb % valign == 0 && a.bias_sh % valign == 0 &&
		               a.bias_sm % valign == 0)
		                  ? 1
		                  : 0;
		// tiles of bias can be copied to LDS like K / V tiles: element type of q, 16-byte aligned
		// rows of whole 16-byte pieces (8 keys), row stride within the 32-bit offsets of the tile copies
		a.bias_lds = (p->bias_dtype == p->dtype && ((uintptr_t)p->bias % 16) == 0 && a.bias_sb % 16 == 0 && a.bias_sh % 16 == 0 &&
		              a.bias_sm % 16 == 0 && a.bias_sm >= 0 && a.bias_sm <= 0x7fffffff / 256 && p->Sk % 8 == 0)
		                 ? 1
		                 : 0;
	}
	a.seqlens = p->seqlens;
	a.kv_lens = p->kv_lens;
	a.hd = short_rows(p) ? p->head_dim : p->D;
	a.B = p->B;
	a.Sq = p->Sq;
	a.Sk = p->Sk;
	a.Hq = p->Hq;
	a.Hkv = p->Hkv;
	a.group_heads = p->Hq / p->Hkv;
	a.causal = p->causal ? 1 : 0;
	// causal caps the right bound at 0, as the reference does (refrence_call.py:36-37)
	a.win_left = p->has_window && p->window_left >= 0 ? p->window_left : -1;
	a.win_right = p->causal ? 0 : (p->has_window && p->window_right >= 0 ? p->window_right : -1);
	a.scale = p->scale;
	a.softcap = p->softcap;
	a.cap_k1 = p->softcap > 0.f ? p->scale / p->softcap : 0.f;
	a.drop_k0 = (uint32_t)(p->seed & 0xFFFFFFFFull);
	a.drop_k1 = (uint32_t)(p->seed >> 32);
	a.seed_dev = (const uint32_t*)p->seed_dev;  // little-endian: low word first
	a.drop_thr = drop_threshold(p->p_drop);
	// kept values are scaled by the reciprocal of the probability the 16-bit threshold really gives,
	// (65536 - thr) / 65536, so that the expectation of the output is exact for every p
	a.drop_inv_keep = 65536.0f / (float)(65536u - a.drop_thr);
}

}  // namespace

namespace fa2 {

hipError_t launch_fwd(int dtype, int D, bool bias, bool drop, KArgs& a, hipStream_t s) {
	if (a.hd != D) return dtype == FA2_BF16 ? launch_fwd_bf16_96(bias, drop, a, s) : launch_fwd_fp16_96(bias, drop, a, s);
	if (dtype == FA2_BF16) {
		if (D == 64) return launch_fwd_bf16_64(bias, drop, a, s);
		if (D == 128) return launch_fwd_bf16_128(bias, drop, a, s);
		return launch_fwd_bf16_256(bias, drop, a, s);
	}
	if (D == 64) return launch_fwd_fp16_64(bias, drop, a, s);
	if (D == 128) return launch_fwd_fp16_128(bias, drop, a, s);
	return launch_fwd_fp16_256(bias, drop, a, s);
}

hipError_t launch_bwd(int dtype, int D, bool bias, bool drop, KArgs& a, hipStream_t s) {
	if (a.hd != D) return dtype == FA2_BF16 ? launch_bwd_bf16_96(bias, drop, a, s) : launch_bwd_fp16_96(bias, drop, a, s);
	if (dtype == FA2_BF16) {
		if (D == 64) return launch_bwd_bf16_64(bias, drop, a, s);
		if (D == 128) return launch_bwd_bf16_128(bias, drop, a, s);
		return launch_bwd_bf16_256(bias, drop, a, s);
	}
	if (D == 64) return launch_bwd_fp16_64(bias, drop, a, s);
	if (D == 128) return launch_bwd_fp16_128(bias, drop, a, s);
	return launch_bwd_fp16_256(bias, drop, a, s);
}

}  // namespace fa2

extern "C" {

int fa2_validate(const fa2_params* p, int which) {
	fa2_params lp;
	return validate(complete(p, lp), which ? 1 : 0);
}

size_t fa2_bwd_scratch_bytes(const fa2_params* p) {
	fa2_params lp;
	p = complete(p, lp);
	return p ? bwd_scratch_bytes(p) : 0;
}

// dK/dV on a small grid: B * Hkv * ceil(Sk / 128) workgroups that leave at least half of the chip idle - the steps a
// key tile streams (the q-heads of its KV group x the query tiles) are then split over up to 8 workgroups whose fp32
// partial dK / dV a reduce kernel sums.  Returns the number of parts (1 = no split).
static int bwd_step_split(const fa2_params* p) {
	if (p->Hkv <= 0 || p->Hq % p->Hkv) return 1;
	long wgs = (long)p->B * p->Hkv * ((p->Sk + 127) / 128);
	long steps = (long)(p->Hq / p->Hkv) * ((p->Sq + 127) / 128);  // of the longest key tile, in units of 128 rows
	long parts = wgs > 0 ? 256 / wgs : 1;  // fill the chip
	if (p->causal && wgs < 512) {
		// Causal key tiles differ in length (the first has all the steps, the last one row block's), and with one
		// workgroup per CU the longest sets the time.  Measured (D = 128, dK/dV kernel): up to 128 workgroups do best in
		// 8 parts, one per XCD, down to 16 steps a part (B4 Hq32 Hkv1 S4096 3.00 ms unsplit, 1.58 in 2, 1.07 in 8;
		// B2 Hq8 Hkv2 S4096 0.209 ms in 2, 0.172 in 8); above that about 1024 workgroups of at least 64 steps - up to
		// 256 workgroups at least 2 parts (B4 Hq32 Hkv2 S4096 1.56 ms unsplit, 1.06 in 2 or 4; B1 Hq32 Hkv8 S4096 0.39 /
		// 0.27 in 2 / 0.29 in 4; B1 H8 S4096, 32 steps, 0.103 / 0.090 in 2; B3 Hq32 Hkv4, 384 workgroups, 1.53 / 1.05
		// in 2 / 0.98 in 3; B1 H8 S6144, 384 of 48 steps, 0.163 / 0.185 in 2); from 512 on the launch order packs them
		// unsplit.
		long bal;
		if (wgs <= 128) {
			bal = steps / 16;
		} else if (wgs <= 256) {
			bal = steps / 64 > 2 ? steps / 64 : 2;
			if (bal > 4) bal = 4;
			if (bal > steps / 16) bal = steps / 16;
		} else {
			bal = (1024 + wgs / 2) / wgs;
			if (bal > steps / 64) bal = steps / 64;
		}
		if (bal > 8) bal = 8;
		if (bal > parts) parts = bal;
	}
	if (parts > 8) parts = 8;
	// (the partial sums and their reduction have a fixed cost - about 5 us: measured, a key tile of fewer than 8 such steps
	// is faster unsplit, and a part should have at least two)
	if (steps < 8) return 1;
	if (parts > steps / 2) parts = steps / 2;
	return parts >= 2 ? (int)parts : 1;
}

static size_t bwd_split_part_bytes(const fa2_params* p, int hs) {
	return (size_t)hs * (size_t)p->B * (size_t)p->Hkv * (size_t)p->Sk * 2 * (size_t)p->D * sizeof(float);
}

size_t fa2_bwd_split_scratch_bytes(const fa2_params* p) {
	fa2_params lp;
	p = complete(p, lp);
	if (!p) return 0;
	size_t base = bwd_scratch_bytes(p);
	if (!base || p->Sk <= 0 || p->D <= 0) return 0;
	int hs = bwd_step_split(p);
	return hs > 1 ? base + bwd_split_part_bytes(p, hs) : 0;
}

// the rows of all q-heads of a kv-head fit one row tile: they share one workgroup (and one pass over K, V)
static bool fwd_pack_gqa(const fa2_params* p) {
	return p->Hkv > 0 && p->Hq % p->Hkv == 0 && p->Hq > p->Hkv && (long)(p->Hq / p->Hkv) * p->Sq <= 64;
}

// The most scratch a forward asks for.  It binds the ranges of grids of 128-row workgroups that are more than half full over very many keys
// (0.2 % of shapes spread over the logarithm of their sizes; 1 % longer on average there, 4 % at most by the plan's own estimate).
constexpr size_t kFwdScratchMax = 128u << 20;

// Scratch of fwd_decode_kernel for this many waves: the pieces (at most one per wave and one more per (batch, kv-head)), O and lse of a
// unit's rows; where they are, per unit.
static size_t fwd_decode_scratch(const fa2_params* p, int64_t waves) {
	const size_t units = (size_t)p->B * (size_t)p->Hkv, rows = ((size_t)waves + units) * (size_t)(p->Hq / p->Hkv) * (size_t)p->Sq;
	return (rows * ((size_t)p->D + 1) * sizeof(float) + units * 8 + 255) & ~(size_t)255;
}

// Few query rows in all, nothing but masks by position and key lengths: fwd_decode_kernel.  Returns the number of waves that
// share the key tiles (0 = not this kernel); *whole: one (batch, kv-head) per wave, no scratch.
static int fwd_decode_waves(const fa2_params* p, int* whole) {
	if (p->Hkv <= 0 || p->Hq % p->Hkv || p->bias || p->p_drop > 0.f || p->softcap > 0.f || p->has_window || p->seqlens) return 0;
	const int64_t r = p->Hq / p->Hkv, units = (int64_t)p->B * p->Hkv;
	if (r * p->Sq > 16) return 0;  // (the columns of a 16 x 16 product)
	// the query rows of a unit are addressed with 32-bit byte offsets from its first, the tiles are counted in 32 bits
	if (p->q.stride_h < 0 || ((r - 1) * p->q.stride_h + (p->Sq - 1) * p->q.stride_s) * 2 > 0x7fff0000) return 0;
	const int kt = p->D == 64 ? 64 : 32;
	const int64_t tiles = (p->Sk + kt - 1) / kt, total = units * tiles;
	if (total > 0x3fffffff) return 0;
	const int64_t resident = p->D == 256 ? 512 : 1024;  // waves that run at once
	const int64_t heads = (int64_t)p->B * p->Hq;        // workgroups of the general kernel, of which 512 run at once (256 at D = 256)
	const int64_t rows = r * p->Sq;
	if (p->Sk <= 256) {
		// A wave takes about a microsecond per tile, so units of up to six tiles are left whole.  Six tiles, or four under more than eight
		// rows, are whole tiles of the general kernel too, which is then as fast or faster unless the units are many: 8 kv-heads, D128, 16 rows,
		// here and there, B8 Sk192 10.2 and 9.2 us, Sk160 9.1 and 9.3, Sk128 8.1 and 7.6, B64 Sk192 11.3 and 13.2; D256 B8 Sk192 14.3 and 13.2.
		if (tiles > 6) return 0;
		const bool many = heads > resident / 2 || units >= resident / 2;
		if (!many && p->D != 64 && (tiles == 6 || (tiles == 4 && rows > 8))) return 0;
		*whole = 1;
		return (int)units;
	}
	// A few hundred keys under many rows: the general kernel runs all its workgroups at once (B40 H8 D128, 16 rows over 300 keys: 16.9 us;
	// 18.5 here with whole units, 21.7 in shares).
	if (p->D == 128 && rows > 8 && p->Sk <= 512 && units >= 192 && heads <= 512) return 0;
	// Whole units or equal shares?  Whole units leave the last round of waves to less than the full stream of memory, unless it is nearly full:
	// that costs so many us a tile, and a quarter of a tile's time where rows of different length may end early.  Shares cost the
	// second launch, the partial results written and read, and with lengths the search for a wave's first tile.  From 2989
	// calls (8 to 2560 units of 257 to 4000 keys, caches not in L2; us whole / shares): H8 D128 B64 Sk500 27.3 / 29.7, Sk2048 98.6 / 93.6;
	// B96 Sk700 47.4 / 54.0; B192 Sk2048 271 / 271; D64 B64, 16 rows over 700 keys 21.3 / 28.8; D256 B80 Sk1000 144 / 116.
	// The rule is within 0.6 % of the better of the two on average; what it replaced, shares below 2048 units, lost up to a third
	// to the general kernel where these are many and the keys few (D64 B64 H8, 16 rows over 257 keys: 17.8 us against 12.1; whole 11.6).
	const int64_t rem = units % resident;
	double idle = rem == 0 ? 0.0 : p->D == 256 ? 2.0 - 0.0056 * rem : 1.25 - 0.0022 * rem;
	idle = (idle > 0 ? idle : 0) + (p->kv_lens ? 0.25 : 0.0);
	int64_t waves = resident < total ? resident : total;
	const double merge = 3.4 + (p->kv_lens ? 3.7 : 0.0) + (waves + (units < waves ? units : waves)) * rows * p->D * 8 / 3.1e6;
	// as many waves as are resident at once, down to a tile each (B1 Hkv8 Sk1029: 8.5 us, two tiles each 10.0), at most 63 a unit
	if (waves > 63 * units) waves = 63 * units;
	*whole = idle * tiles < merge || fwd_decode_scratch(p, waves) > kFwdScratchMax;
	return (int)(*whole ? units : waves);
}

// Key ranges for a split forward: too few workgroups to fill the chip, many keys.  Returns the number of ranges (1 = no split) of
// *split_len keys; *tall: in workgroups of 128 rows (1: of eight waves, one a CU; 2: of four, two a CU).
static int fwd_split_plan(const fa2_params* p, int* split_len, int* tall) {
	*split_len = 0;
	*tall = 0;
	const int tiles = (p->Sk + 63) / 64;
	// Up to 64 rows a q-head fill half of a 128-row workgroup at most.  Over many keys the two-wave workgroups of the 64-row kernel, four of them a
	// CU, have more of the memory's and the chip's time, and ranges beyond a row's length cost them little (here and in 128 rows): D64 B18 H8,
	// 19 rows over 1880 keys 22 and 34 us, B8 Hq16 Hkv4, 60 over 14088 64 and 101; D128 B1 H4, 39 over 15090 17.4 and 26.1, with lengths
	// B3 Hq64 Hkv32, 62 over 10371 134 and 180; but D128 B12 H1, 55 over 15914 without lengths 58 and 31.  Over 700 calls the
	// rule is 0.8 % (D64) and 0.5 % (D128) from the better of the two on average; always 128 rows 10.7 and 1.9, always 64 rows 2.6 and 11.8.
	// Above 256 workgroups of 128 rows the alternative is the unsplit kernel, at D128 over K / V beyond an XCD's L2 in workgroups of 256 rows
	// (B18 Hq16 Hkv8, 55 over 5126: 139 and 232 us), and an odd number of 64-row tiles can leave fewer than 512 of these (D64 B17 H8, 176 over
	// 5979 with lengths: 68 and 112; unsplit up to 64 % longer and never shorter in the 14 such calls of 500).
	const int64_t heads = (int64_t)p->B * p->Hq, wide = heads * ((p->Sq + 127) / 128), narrow = heads * ((p->Sq + 63) / 64);
	bool few_rows;
	if (p->Sq > 64)
		few_rows = p->D == 64 && tiles >= 32 && wide > 256 && narrow < 512;
	else if (p->D == 64)
		few_rows = tiles >= (heads < 32 ? 64 : heads < 64 ? 24 : 16);
	else
		few_rows = (tiles >= 128 && heads < 16) || (p->kv_lens && tiles >= 48 && heads >= 32) ||
		           (heads > 256 && (int64_t)p->Sk * p->D * 4 > (p->causal ? 4 << 20 : 2 << 20));
	if (p->D <= 128 && !p->bias && !(p->p_drop > 0.f) && !fwd_pack_gqa(p) && !few_rows) {
		// Workgroups of 128 rows whose eight waves share the keys, one per CU: as many key ranges as make the estimate smallest - whole
		// rounds of the longest workgroup (less where a causal mask makes them unequal and they even out over
		// several rounds), plus 3 us for the second launch and the partial results written and read.  Figures measured: a tile
		// takes such a workgroup 1.07 us (0.8 at D = 64), partial results move at 2.8 TB/s; without ranges and with more than 256 workgroups
		// the 128-row kernel runs two workgroups a CU and needs 1.46 to 2.2 us a tile (1.05 to 1.8 at D = 64).  B1 Hq32 Hkv8 D128, 100 rows over
		// 4000 keys: 71 us in one range, 44 in 2, 30 in 4, 24 in 8, 35 in 12 (16 ranges of the 64-row kernel: 36); B1 H4 S4096 D128
		// causal: 61 / 42 / 54 us in 1 / 2 / 4; B2 Hq16 300 rows over 3000 keys: 55 / 36 / 44 us in 1 / 2 / 4; B2 H12 D64, 2048 rows over
		// 3048 keys (384 workgroups): 63 / 72 / 89 in 1 / 2 / 4.
		const int64_t base = wide;
		if (base >= 512) return 1;
		// (eight tiles of D = 64 are too little for a second launch: B1 H8, 64 rows over 512 keys 10.3 us in one range, 10.9 in 2, 11.7 in 4)
		if (p->D == 64 && tiles <= 8) return 1;
		const double mean = p->causal && p->Sq <= p->Sk ? (p->Sk - 0.5 * p->Sq) / 64 : tiles;
		const bool even = mean > 0.75 * tiles;
		const double tile_us = p->D == 64 ? 0.8 : 1.07;
		const double part_us = (double)p->B * p->Hq * p->Sq * p->D * 8 / 2.8e6 * (mean / tiles);
		int best = 1;
		double best_us = tiles * (base <= 256 ? tile_us : ((p->D == 64 ? 1.05 : 1.46) + (base - 256) / 256.0 * 0.7) * (even ? 1.0 : 0.6));
		const size_t range_bytes = (size_t)p->B * (size_t)p->Hq * (size_t)p->Sq * ((size_t)p->D + 1) * sizeof(float);
		for (int n = 2; n <= 16 && n <= tiles / 2 && n * range_bytes <= kFwdScratchMax; ++n) {
			const int64_t rounds = (base * n + 255) / 256;
			const double us = rounds * ((tiles + n - 1) / n) * (even || rounds == 1 ? 1.0 : 0.85) * tile_us + 3 + n * part_us;
			if (us < best_us) {
				best = n;
				best_us = us;
			}
		}
		*tall = 1;
		if (p->D == 128 && !short_rows(p) && !p->kv_lens && !p->seqlens) {
			// Or workgroups of four waves, two a CU: no barrier holds one up for the other, but there are twice as many partial results. Fitted
			// to Hkv 8, 4200 to 14200 keys, of 384 to 512 such workgroups: a tile takes 0.67 us and 1.24 more with the share of the places that are
			// taken, partial results 0.57 of the above. B1 Hq32 Hkv8, 1000 causal rows over 9000 / 14200 keys 174 / 261 -> 155 / 227 us in two ranges, 700 rows over
			// 8200 140 -> 120, 600 rows over 3000 / 10200 in three 56 / 126 -> 45 / 112; B1 Hq8 Hkv2, 1500 over 6200 in five 64 -> 51. Workgroups of eight waves in one
			// range take 6 % more than their estimate over many keys (1000 rows over 6200: 104 and 117); from three ranges on a tenth has to be gained (four,
			// estimated as even: B1 H4 S4096 over 6200 57 and 61, B1 Hq16 Hkv4, 1000 over 3000 41 and 45).
			// All this with rows that do not fill their last wave, whose tiles all take the masked path: a workgroup of eight waves alone on its CU waits for that wave.
			// Where rows are a multiple of 32 it takes 15 % less (B1 Hq64 Hkv16 over 3000 keys, 384 rows 47.5 us, 370 rows 55.8), workgroups that share a CU
			// nothing less. Two ranges then gain nothing (47.5 -> 54.5; 512 rows of B4 H12 48 -> 58, B1 Hq32 Hkv8, 1024 over 7500 123 -> 130, over 13000 206 -> 211), three do
			// (B1 Hq40 Hkv8, 512 over 4000 59.5 -> 55.4), more only over many keys (five, B1 Hq24 Hkv8, 512 over 7500 62.6 -> 59.2; four, B1 Hq20 Hkv5, 640 over 4000 40.9 -> 43.2), and
			// over more where groups are not placed by XCD and every range is read on all of them (five, B1 H14, 896 over 7500 64 -> 70, over 13000 115 -> 109). There two
			// ranges lose otherwise too (1000 rows of Hq25 Hkv5 over 3000 56 -> 62, of Hq30 Hkv10 over 7500 137 -> 141, over 13000 232 -> 230), and with more than three groups
			// an XCD (368 rows of B2 Hq32 Hkv16 over 3000 56 -> 60, over 11000 174 -> 183; three, 409 of B3 Hq16 Hkv8 over 7033 120 -> 97).
			// Fewer than 384 leave too many CUs with one: 288 of 96 x 3, 22.3 and 23.3, 72 x 4, 41 and 44; 320 of 80 x 4, 52.5 and 57, 160 x 2, 38.9 and 39.8; 352 of
			// 176 x 2, 36 and 41, 43.6 and 42.9.  Not with lengths: a range beyond a row's length is a place wasted (B3 Hq8 Hkv2, 1000 rows over
			// 3000 keys 51 and 60). (Rows of fewer columns run on the rows as they are.)
			int pairs = 0;
			double pairs_us = 0;
			for (int n = 2; n <= 16 && n <= tiles / 2 && base * n <= 512 && n * range_bytes <= kFwdScratchMax; ++n) {
				if (base * n < 384) continue;
				const double us = (tiles + n - 1) / n * (0.67 + 1.24 * (base * n) / 512) + 3.5 + 0.57 * n * part_us;
				if (!pairs || us < pairs_us) {
					pairs = n;
					pairs_us = us;
				}
			}
			const bool whole = p->Sq % 32 == 0;
			const bool by_xcd = (int64_t)p->B * p->Hkv % 8 == 0, far = tiles >= 160;
			const bool ok = pairs == 2 ? !whole && (by_xcd ? (int64_t)p->B * p->Hkv <= 24 : far) : pairs == 3 || !whole || far || (by_xcd && tiles >= 100);
			if (pairs && ok && pairs_us < best_us * (pairs == 2 ? 1.06 : 0.9)) {
				best = pairs;
				*tall = 2;
			}
		}
		const int per = (tiles + best - 1) / best;
		*split_len = per * 64;
		return (tiles + per - 1) / per;
	}
	// workgroups of an unsplit launch of this kernel variant (row tiles of 64)
	long base = fwd_pack_gqa(p) ? (long)p->B * p->Hkv : (long)narrow;
	// A query longer than one row tile (with bias or dropout, or at D = 256) runs unsplit on the 128-row kernel, which a quarter of the
	// chip's worth of units already keeps busy over a short key range: the second launch pays from 16 key tiles on up to 128 units
	// and from 32 above.
	int min_tiles = p->Sq <= 64 ? 8 : (base <= 128 ? 16 : 32);
	if (base >= 512 || tiles < min_tiles) return 1;
	long want = (1024 + base - 1) / base;
	if (want > tiles / 4) want = tiles / 4;
	if (want > 64) want = 64;
	if (want < 2) return 1;
	int per = (int)((tiles + want - 1) / want);
	*split_len = per * 64;
	return (tiles + per - 1) / per;
}

// p: a completed block.  The split forward knows no window and no soft-capping: such calls run unsplit and
// need no scratch (the same predicate decides the launch in fa2_fwd).
static size_t fwd_scratch_bytes(const fa2_params* p) {
	if (p->B <= 0 || p->Hq <= 0 || p->Sq <= 0 || p->Sk <= 0 || p->D <= 0) return 0;
	if (p->has_window || p->softcap > 0.f) return 0;
	int len;
	int whole;
	if (int waves = fwd_decode_waves(p, &whole)) return whole ? 0 : fwd_decode_scratch(p, waves);
	int tall, n = fwd_split_plan(p, &len, &tall);
	if (n <= 1) return 0;
	size_t rows = (size_t)n * (size_t)p->B * (size_t)p->Hq * (size_t)p->Sq;
	return (rows * ((size_t)p->D + 1) * sizeof(float) + 255) & ~(size_t)255;
}

}  // extern "C"

namespace {
// (of the padded rows, which are contiguous: whatever strides the short ones have, the answer is the same before and after
// the caller copies them for their alignment)
bool fwd_takes_ranges(const fa2_params* p) {
	fa2_params padded = *p;
	padded.q.stride_s = padded.q.stride_h = 0;
	int whole;
	return fwd_decode_waves(&padded, &whole) || fwd_scratch_bytes(&padded);
}
}  // namespace

extern "C" {

size_t fa2_fwd_scratch_bytes(const fa2_params* p) {
	fa2_params lp;
	p = complete(p, lp);
	return p && !short_rows(p) ? fwd_scratch_bytes(p) : 0;
}

int fa2_fwd(const fa2_params* p, void* hip_stream) {
	fa2_params lp;
	p = complete(p, lp);
	int rc = validate(p, 0);
	if (rc) return rc;
	KArgs a;
	fill(p, a);
	if (short_rows(p)) return fa2::launch_fwd(p->dtype, p->D, false, false, a, (hipStream_t)hip_stream) == hipSuccess ? FA2_OK : FA2_EHIP;
	// optional scratch: with enough of it a short query over many keys runs split over key ranges
	size_t need = fwd_scratch_bytes(p);
	const bool room = need && p->scratch && ((uintptr_t)p->scratch & 255) == 0 && p->scratch_bytes >= need;
	int whole = 0;
	const int waves = fwd_decode_waves(p, &whole);
	if (waves && (whole || room)) {
		a.decode_waves = waves;
		a.decode_whole = whole;
		size_t rows = (waves + (size_t)p->B * (size_t)p->Hkv) * (size_t)(p->Hq / p->Hkv) * (size_t)p->Sq;
		a.o_part = (float*)p->scratch;
		a.lse_part = a.o_part + rows * (size_t)p->D;
		a.decode_units = (int32_t*)(a.lse_part + rows);
	} else if (room && !waves) {
		a.nsplit = fwd_split_plan(p, &a.split_len, &a.tall_split);
		a.pack_gqa = fwd_pack_gqa(p) ? 1 : 0;
		size_t rows = (size_t)a.nsplit * (size_t)p->B * (size_t)p->Hq * (size_t)p->Sq;
		a.o_part = (float*)p->scratch;
		a.lse_part = a.o_part + rows * (size_t)p->D;
	}
	hipError_t e = fa2::launch_fwd(p->dtype, p->D, p->bias != nullptr || p->softcap > 0.f, p->p_drop > 0.f, a, (hipStream_t)hip_stream);
	return e == hipSuccess ? FA2_OK : FA2_EHIP;
}

int fa2_bwd(const fa2_params* p, void* hip_stream) { return fa2_bwd_stages(p, hip_stream, 7); }

static int bwd_launch(const fa2_params* p, void* hip_stream, int stages, void* scratch_ptr, size_t scratch_bytes) {
	KArgs a;
	fill(p, a);
	a.stages = stages & 7;
	// optional: with enough scratch behind delta the dK/dV kernel of a small grid runs split over the q-heads of a group
	a.kv_hsplit = 1;
	a.dkv_part = nullptr;
	{
		int hs = bwd_step_split(p);
		size_t base = bwd_scratch_bytes(p);
		if (hs > 1 && scratch_bytes >= base + bwd_split_part_bytes(p, hs)) {
			a.kv_hsplit = hs;
			a.dkv_part = (float*)((char*)scratch_ptr + base);
		}
	}
	a.dout = conv(p->dout);
	a.dq = conv(p->dq);
	a.dk = conv(p->dk);
	a.dv = conv(p->dv);
	a.delta = (float*)scratch_ptr;
	a.dbias = (char*)p->dbias;
	a.dbias_sb = p->dbias_stride_b * 4;
	a.dbias_sh = p->dbias_stride_h * 4;
	a.dbias_sm = p->dbias_stride_m * 4;
	a.dbias_atomic = p->dbias && ((p->dbias_stride_b == 0 && p->B > 1) || (p->dbias_stride_h == 0 && p->Hq > 1) ||
	                              (p->bias_group && p->Hq > p->Hkv))
	                     ? 1
	                     : 0;
	hipError_t e = fa2::launch_bwd(p->dtype, p->D, p->bias != nullptr || p->softcap > 0.f, p->p_drop > 0.f, a, (hipStream_t)hip_stream);
	return e == hipSuccess ? FA2_OK : FA2_EHIP;
}

int fa2_bwd_stages(const fa2_params* p, void* hip_stream, int stages) {
	fa2_params lp;
	p = complete(p, lp);
	int rc = validate(p, 1);
	if (rc) return rc;
	return bwd_launch(p, hip_stream, stages, p->scratch, (size_t)p->scratch_bytes);
}

// Device address of `scratch` on the current device, looked up once per device.
static int static_scratch_ptr(void** out) {
	constexpr int kMaxDevices = 64;
	static void* ptrs[kMaxDevices];
	static std::mutex mu;
	int dev = -1;
	if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FA2_EHIP;
	std::lock_guard<std::mutex> lock(mu);
	if (!ptrs[dev]) {
		void* ptr = nullptr;
		if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return FA2_EHIP;
		ptrs[dev] = ptr;
	}
	*out = ptrs[dev];
	return FA2_OK;
}

int fa2_bwd_static(const fa2_params* p, void* hip_stream) {
	fa2_params lp;
	p = complete(p, lp);
	int rc = validate(p, 1, /*own_scratch=*/true);
	if (rc) return rc;
	void* ptr = nullptr;
	if ((rc = static_scratch_ptr(&ptr))) return rc;
	// delta is written in full by the first kernel before the second reads it: nothing to clear
	return bwd_launch(p, hip_stream, 7, ptr, (size_t)FA2_STATIC_SCRATCH_BYTES);
}

int fa2_dropout_mask(const fa2_params* p, uint8_t* keep, void* hip_stream) {
	fa2_params lp;
	p = complete(p, lp);
	if (!p) return FA2_EINVAL_STRUCT;
	if (p->seed_dev && ((uintptr_t)p->seed_dev & 7)) return FA2_EINVAL_PTR;
	if (p->B <= 0 || p->Sq <= 0 || p->Sk <= 0 || p->Hq <= 0) return FA2_EINVAL_SHAPE;
	if (!(p->p_drop >= 0.f && p->p_drop < 1.f)) return FA2_EINVAL_DROPOUT;
	if (!keep) return FA2_EINVAL_PTR;
	hipError_t e = fa2::launch_dropout_mask(keep, p->B, p->Hq, p->Sq, p->Sk, (uint32_t)(p->seed & 0xFFFFFFFFull),
	                                        (uint32_t)(p->seed >> 32), drop_threshold(p->p_drop), (const uint32_t*)p->seed_dev,
	                                        (hipStream_t)hip_stream);
	return e == hipSuccess ? FA2_OK : FA2_EHIP;
}

int fa2_mask_lengths(const uint8_t* mask, int64_t stride, int32_t B, int32_t S, int32_t* lens, void* hip_stream) {
	if (B <= 0 || S <= 0) return FA2_EINVAL_SHAPE;
	if (!mask || !lens || ((uintptr_t)lens & 3)) return FA2_EINVAL_PTR;
	return fa2::launch_mask_lengths(mask, stride, B, S, lens, (hipStream_t)hip_stream) == hipSuccess ? FA2_OK : FA2_EHIP;
}

const char* fa2_strerror(int code) {
	switch (code) {
		case FA2_OK: return "ok";
		case FA2_EINVAL_STRUCT: return "params is NULL or struct_size is smaller than the first version of fa2_params";
		case FA2_EINVAL_DTYPE: return "Only support fp16 and bf16";
		case FA2_EINVAL_SHAPE: return "dimensions must be positive and the softmax scale finite and positive";
		case FA2_EINVAL_HEADS: return "query heads must be divisible by key/value heads";
		case FA2_EINVAL_PTR: return "required pointer is NULL or misaligned";
		case FA2_EINVAL_STRIDE: return "strides must be multiples of 8 elements and the sequence stride in [0, 2^31 / 256] elements";
		case FA2_EINVAL_DROPOUT: return "dropout probability must be in [0, 1)";
		case FA2_EINVAL_BIAS: return "bias dtype or strides invalid";
		case FA2_EINVAL_MASK: return "Attention mask is not supported along with attention bias or with QSeq != KSeq";
		case FA2_EUNSUPPORTED: return "head dim must be 64, 128 or 256 (and head_dim one the kernels of D have a variant for)";
		case FA2_ESCRATCH: return "backward scratch buffer missing, misaligned or too small";
		case FA2_EHIP: return "HIP launch failed";
		case FA2_ESCRATCH_STATIC: return "fa2_bwd_static: B * Hq * Sq * 4 bytes exceed the 16 MiB built-in scratch";
		default: return "unknown error";
	}
}

int fa2_version(void) { return 100; }

}  // extern "C"
