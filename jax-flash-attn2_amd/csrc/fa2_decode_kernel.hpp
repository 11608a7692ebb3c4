// Forward for a handful of query rows over many keys (decoding): the rows of all q-heads of a kv-head, at most sixteen in all,
// share one pass over K and V.  Same results as the split forward of fa2_fwd_kernel.hpp for these shapes
// (a single query row is the reference's decoding case, jax_flash_attn2/flash_attention.py:239-242).
//
// Bound: memory, so the kernel is built for bytes in flight and for equal shares.  The key tiles of all (batch, kv-head) units
// form one sequence, cut into equal shares, one per WAVE: rows of different length, or a number of units that does not divide
// over the chip, leave nobody waiting.  A wave streams its share through LDS tiles of its own, the next tile always on its
// way, across the ends of units too; there is no barrier in the kernel.  Four waves keep 64 KiB a CU in flight (a plain read of
// 150 MiB: 3.6 TB/s with 16 KiB a CU, 5.0 with 32, 5.5 with 64).  A unit that lies inside one share is stored directly, the
// pieces of the others go through scratch to fwd_decode_combine_kernel (3.4 us and more: where whole
// units leave little of the last round of waves idle, every unit is one wave's and there is no second launch, see fwd_decode_waves()).
// Measured against the split of fwd_kernel that these shapes took before (Hkv 8, D 128, half to all of the slots filled): B8 Hq32
// Sk8192 57 -> 44 us (201 MB: 5.3 TB/s without the combine), B64 Hq16 Sk8000 630 -> 274 us (5.7 TB/s), B2 Hq64 Sk16000 58 -> 27 us,
// B1 Hq32 Sk1029 16.4 -> 8.5 us.
// The products are 16 x 16 x 32 with the query rows as columns: the lane of a column owns its row, so P packs into the second
// product's operand without leaving the lane, and a tile of 32 keys costs a wave about 200 instructions (a form on the vector
// ALU, K and V in registers, took six times that and ran at 3.4 TB/s).
#pragma once
#include <type_traits>

#include "fa2_common.hpp"
#include "fa2_kernels.hpp"

namespace fa2 {

// D[16x16] += A[16x32] * B[32x16].  Lane l supplies A[row l%16][k 8*(l/16)..+7] and B[k 8*(l/16)..+7][col l%16]; it receives
// D[row 4*(l/16)+i][col l%16] in element i.
FA2_DEV f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
FA2_DEV f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// max / sum over the four lanes that hold the same column of such a product
FA2_DEV float column_max(float x) {
	auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
	return pair_max(__builtin_fmaxf(__builtin_bit_cast(float, (int)r[0]), __builtin_bit_cast(float, (int)r[1])));
}
FA2_DEV float column_sum(float x) {
	auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
	return pair_sum(__builtin_bit_cast(float, (int)r[0]) + __builtin_bit_cast(float, (int)r[1]));
}

template <int N>
FA2_DEV void wait_loads_but() {
	asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Keys per tile of a wave (16 KiB of K and V, 32 KiB at head dim 256) and waves per workgroup: one workgroup per CU.
template <int D>
struct DecodeCfg {
	static constexpr int KT = D == 64 ? 64 : 32;
	static constexpr int NW = D == 256 ? 2 : 4;
};

// Where the share of a wave begins, and what it needs to step from unit to unit.  All values are wave-uniform but `lens`.
struct DecodePos {
	int b, hk, t;     // batch row, kv-head, tile
	int len, tiles;   // of the batch row
};

FA2_DEV int decode_len(const KArgs& a, int b) {
	int len = a.Sk;
	if (a.kv_lens) {
		int x = a.kv_lens[b];
		x = x < 0 ? 0 : x;
		len = x < len ? x : len;
	}
	return len;
}

template <typename T, int D>
__global__ __launch_bounds__(DecodeCfg<D>::NW * 64) void fwd_decode_kernel(const KArgs a) {
	typedef typename T::V8 V8;
	constexpr int KT = DecodeCfg<D>::KT, NW = DecodeCfg<D>::NW;
	constexpr int KB = KT / 16;         // 16-key blocks of a tile
	constexpr int KS = D / 32, DB = D / 16;
	constexpr int TILE_BYTES = KT * D * 2, Q_BYTES = 16 * D * 2;
	constexpr int NIT = TILE_BYTES / 1024, NQ = Q_BYTES / 1024;  // load instructions of a tile / of the query rows
	__shared__ __attribute__((aligned(1024))) char smem[NW * (4 * TILE_BYTES + 2 * Q_BYTES)];

	const int r = a.Hq / a.Hkv, nrows = r * a.Sq;
	const int tid = threadIdx.x, lane = tid & 63;
	const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wid = (int)blockIdx.x * NW + w;
	const int g = lane >> 4, c = lane & 15;
	FA2_LDS char* const lds = (FA2_LDS char*)smem + w * (4 * TILE_BYTES);  // K[0] K[1] V[0] V[1] of this wave
	FA2_LDS char* const lds_q = (FA2_LDS char*)smem + NW * 4 * TILE_BYTES + w * 2 * Q_BYTES;  // Q[0] Q[1]: two units, in turn

	// this wave's share [f, f_end) of the tiles of all units, in the order (batch row, kv-head, tile)
	auto tiles_of = [](int len) { return (len + KT - 1) / KT; };
	int share, f, f_end;
	DecodePos pos;
	if (a.decode_whole) {
		// one unit per wave, which also stores the zeros of a unit without keys
		if (wid >= a.B * a.Hkv) return;
		pos.b = wid / a.Hkv;
		pos.hk = wid - pos.b * a.Hkv;
		pos.t = 0;
		pos.len = decode_len(a, pos.b);
		pos.tiles = pos.len > 0 ? tiles_of(pos.len) : 1;
		share = f_end = pos.tiles;
		f = 0;
	} else if (!a.kv_lens) {
		pos.len = a.Sk;
		pos.tiles = tiles_of(a.Sk);
		const int total = a.B * a.Hkv * pos.tiles;
		share = (total + a.decode_waves - 1) / a.decode_waves;
		f = wid * share;
		f_end = f + share < total ? f + share : total;
		const int unit = f / pos.tiles;
		pos.t = f - unit * pos.tiles;
		pos.b = unit / a.Hkv;
		pos.hk = unit - pos.b * a.Hkv;
	} else {
		// lanes add up the tiles of 64 batch rows at a time
		int total = 0;
		for (int b0 = 0; b0 < a.B; b0 += 64) {
			int x = b0 + lane < a.B ? tiles_of(decode_len(a, b0 + lane)) : 0;
#pragma unroll
			for (int d = 1; d < 64; d <<= 1) x += __shfl_xor(x, d, 64);
			total += x;
		}
		total = __builtin_amdgcn_readfirstlane(total) * a.Hkv;
		share = (total + a.decode_waves - 1) / a.decode_waves;
		f = wid * share;
		f_end = f + share < total ? f + share : total;
		int before = 0;  // tiles of the units of earlier batch rows
		pos.b = pos.hk = pos.t = pos.len = pos.tiles = 0;
		for (int b0 = 0; b0 < a.B && f < f_end; b0 += 64) {
			const int len = b0 + lane < a.B ? decode_len(a, b0 + lane) : 0;
			int x = tiles_of(len) * a.Hkv, sum = x;
#pragma unroll
			for (int d = 1; d < 64; d <<= 1) {
				int y = __shfl_up(sum, d, 64);
				sum += lane >= d ? y : 0;
			}
			const uint64_t hit = __builtin_amdgcn_ballot_w64(before + sum > f);
			if (hit) {
				const int l = __builtin_ctzll(hit);
				pos.b = b0 + l;
				pos.len = __builtin_amdgcn_readlane(len, l);
				pos.tiles = tiles_of(pos.len);
				const int rem = f - (before + __builtin_amdgcn_readlane(sum, l) - __builtin_amdgcn_readlane(x, l));
				pos.hk = rem / pos.tiles;
				pos.t = rem - pos.hk * pos.tiles;
				break;
			}
			before += __builtin_amdgcn_readlane(sum, 63);
		}
	}
	if (f >= f_end) return;

	TileLoader<D, KT, 64> kload, vload;
	kload.init(a.k.ss, lane);
	vload.init(a.v.ss, lane);
	// byte offsets of this lane's pieces of the unit's query rows (row n: position n % Sq of q-head n / Sq of the group; rows beyond
	// the last repeat it), swizzled like a tile
	uint32_t qoff[NQ];
#pragma unroll
	for (int it = 0; it < NQ; ++it) {
		const int slot = it * 64 + lane, row = slot / (D / 8), chunk = (slot % (D / 8)) ^ swz<D>(row);
		const int m = row < nrows ? row : nrows - 1, hh = m / a.Sq, i = m - hh * a.Sq;
		qoff[it] = (uint32_t)(hh * a.q.sh + i * a.q.ss) + (uint32_t)(chunk << 4);
	}
	auto issue = [&](const DecodePos& p, int buf, bool with_q, int qbuf) __attribute__((always_inline)) {
		const int n0 = p.t * KT;
		int rows = p.len - n0 < KT ? p.len - n0 : KT;
		rows = rows > 0 ? rows : 1;  // (a unit without keys: its only tile is masked as a whole)
		if (with_q) {
			const char* qb = TileLoader<D, KT, 64>::uniform(a.q.ptr + (int64_t)p.b * a.q.sb + (int64_t)(p.hk * r) * a.q.sh);
#pragma unroll
			for (int it = 0; it < NQ; ++it) lds_dma16_so(qoff[it], qb, lds_q + qbuf * Q_BYTES + it * 1024);
		}
		kload.load(lds + buf * TILE_BYTES, a.k.ptr + (int64_t)p.b * a.k.sb + (int64_t)p.hk * a.k.sh + (int64_t)n0 * a.k.ss, a.k.ss, rows, lane);
		vload.load(lds + (2 + buf) * TILE_BYTES, a.v.ptr + (int64_t)p.b * a.v.sb + (int64_t)p.hk * a.v.sh + (int64_t)n0 * a.v.ss, a.v.ss, rows, lane);
	};
	issue(pos, 0, true, 0);

	// per-lane LDS offsets (swizzle folded in).  K fragment (kb, ks): row 16 kb + c, chunk 4 ks + g (Q alike).  V fragment (kk, db),
	// its k-slots in the order in which a lane holds its scores: keys 32 kk + 4 g + j and 32 kk + 16 + 4 g + j, j = 0 .. 3, of
	// columns 16 db .. + 15 - two transposed reads.
	constexpr int KR = KS < 4 ? KS : 4, DR = DB < 8 ? DB : 8;
	int koff[KR], voff[DR];
#pragma unroll
	for (int ks = 0; ks < KR; ++ks) koff[ks] = tile_off<D>(c, 4 * ks + g);
#pragma unroll
	for (int db = 0; db < DR; ++db) {
		const int col = 16 * db + 4 * (c & 3);
		voff[db] = tile_off<D>(4 * g + (c >> 2), col >> 3) + ((col & 4) << 1) + 2 * TILE_BYTES;
	}

	V8 qf[KS] = {};
	f32x4 oacc[DB] = {};
	float m_run = -3.0e38f, l_run = 0.f;  // of the column, in the log2 domain / this lane's share of the sum
	const float c1 = a.scale * kLog2e;
	const int crow = c < nrows ? c : nrows - 1, chh = crow / a.Sq, ci = crow - chh * a.Sq;  // this lane's row of a unit

	auto body = [&](int n0, int jmax, int buf) __attribute__((always_inline)) {
		const FA2_LDS char* base = lds + buf * TILE_BYTES;
		f32x4 s[KB];
#pragma unroll
		for (int kb = 0; kb < KB; ++kb) s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for (int ks = 0; ks < KS; ++ks)
#pragma unroll
			for (int kb = 0; kb < KB; ++kb) {
				V8 kf = *(const FA2_LDS V8*)(base + koff[ks % KR] + (ks / KR) * 256 + kb * (16 * D * 2));
				s[kb] = mfma16(kf, qf[ks], s[kb]);
			}
		float mx = -INFINITY;
#pragma unroll
		for (int kb = 0; kb < KB; ++kb)
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				float x = n0 + 16 * kb + 4 * g + i <= jmax ? s[kb][i] * c1 : -INFINITY;
				s[kb][i] = x;
				mx = __builtin_fmaxf(mx, x);
			}
		mx = column_max(mx);
		if (__builtin_amdgcn_ballot_w64(mx > m_run) != 0) {
			const float mn = __builtin_fmaxf(m_run, mx), alpha = exp2_fast(m_run - mn);
			m_run = mn;
			l_run *= alpha;
#pragma unroll
			for (int db = 0; db < DB; ++db)
#pragma unroll
				for (int i = 0; i < 4; ++i) oacc[db][i] *= alpha;
		}
#pragma unroll
		for (int kb = 0; kb < KB; ++kb)
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				float p = exp2_fast(s[kb][i] - m_run);
				l_run += p;
				s[kb][i] = p;
			}
#pragma unroll
		for (int kk = 0; kk < KB / 2; ++kk) {
			const f32x4 &x = s[2 * kk], &y = s[2 * kk + 1];
			V8 pf = pack8<T>(x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]);
#pragma unroll
			for (int db = 0; db < DB; ++db) {
				const FA2_LDS char* vp = base + voff[db % DR] + (db / DR) * 256 + kk * (32 * D * 2);
				oacc[db] = mfma16(as_frag<T>(lds_tr_issue<0>(vp, vp + 16 * D * 2)), pf, oacc[db]);
			}
		}
	};
	// the columns' results: into O and lse when the unit lies inside this wave's share, else as a piece of it into scratch.  Pieces
	// are numbered wave + unit: both only grow along the sequence, and each piece begins with a new wave, a new unit or both.
	auto flush = [&](const DecodePos& p, bool whole) __attribute__((always_inline)) {
		if (p.len == 0) {
			// a unit without keys: the slot that was copied for it can hold anything, and 0 times NaN is NaN
#pragma unroll
			for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
		}
		const float l = column_sum(l_run);
		const float inv = l > 0.f ? 1.f / l : 0.f;
		const float lse = l > 0.f ? (m_run + log2_fast(l)) * kLn2 : -INFINITY;
		if (c >= nrows) return;
		if (whole) {
			const int h = p.hk * r + chh;
			char* rp = a.o.ptr + (int64_t)p.b * a.o.sb + (int64_t)h * a.o.sh + (int64_t)ci * a.o.ss + 8 * g;
#pragma unroll
			for (int db = 0; db < DB; ++db)
				*(u32x2*)(rp + 32 * db) = u32x2{pack2<typename T::V2>(oacc[db][0] * inv, oacc[db][1] * inv), pack2<typename T::V2>(oacc[db][2] * inv, oacc[db][3] * inv)};
			if (g == 0) a.lse[((int64_t)p.b * a.Hq + h) * a.Sq + ci] = lse;
		} else {
			const int64_t prow = (int64_t)(wid + p.b * a.Hkv + p.hk) * nrows + c;
			float* rp = a.o_part + prow * D + 4 * g;
#pragma unroll
			for (int db = 0; db < DB; ++db) *(f32x4*)(rp + 16 * db) = f32x4{oacc[db][0] * inv, oacc[db][1] * inv, oacc[db][2] * inv, oacc[db][3] * inv};
			if (g == 0) a.lse_part[prow] = l >= 0.f ? lse : INFINITY;  // (NaN: a weight of inf - inf in the combine kernel)
		}
	};

	int buf = 0, qbuf = 0, unit_f = f;  // where the piece of the current unit begins
	bool fresh = true;
	for (;; ++f) {
		DecodePos nxt = pos;
		bool next_unit = false;
		if (++nxt.t == pos.tiles) {
			nxt.t = 0;
			next_unit = true;
			if (++nxt.hk == a.Hkv) {
				nxt.hk = 0;
				do {
					++nxt.b;
					nxt.len = nxt.b < a.B ? __builtin_amdgcn_readfirstlane(decode_len(a, nxt.b)) : 1;
				} while (nxt.len == 0);
				nxt.tiles = tiles_of(nxt.len);
			}
		}
		__builtin_amdgcn_sched_barrier(0);
		asm volatile("" ::: "memory");
		// the next tile on its way, then wait for this one's copies - the older ones
		if (f + 1 < f_end) {
			issue(nxt, buf ^ 1, next_unit, qbuf ^ 1);
			if (next_unit)
				wait_loads_but<2 * NIT + NQ>();
			else
				wait_loads_but<2 * NIT>();
		} else {
			wait_async_loads();
		}
		__builtin_amdgcn_sched_barrier(0);
		if (fresh) {
			fresh = false;
#pragma unroll
			for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const FA2_LDS V8*)(lds_q + qbuf * Q_BYTES + koff[ks % KR] + (ks / KR) * 256);
#pragma unroll
			for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
			m_run = -3.0e38f;
			l_run = 0.f;
			if (pos.t == 0 && lane == 0 && !a.decode_whole) {
				// the unit's pieces, for the combine kernel: first wave and their number
				a.decode_units[2 * (pos.b * a.Hkv + pos.hk)] = wid;
				a.decode_units[2 * (pos.b * a.Hkv + pos.hk) + 1] = (f + pos.tiles - 1) / share - wid + 1;
			}
		}
		const int cmax = a.Sk - a.Sq + ci;  // causal alignment counts from the full key count
		body(pos.t * KT, a.win_right == 0 && cmax < pos.len - 1 ? cmax : pos.len - 1, buf);
		const bool ends = f + 1 == f_end;
		if (next_unit || ends) {
			const bool whole = next_unit && pos.t + 1 - (f + 1 - unit_f) == 0;
			flush(pos, whole);
			qbuf ^= 1;
			fresh = true;
			unit_f = f + 1;
		}
		if (ends) break;
		pos = nxt;
		buf ^= 1;
	}
}

// Merges the pieces of the units that several waves shared: O = sum_s exp(lse_s - lse) O_s.  A row is D / 8 threads wide and eight
// groups deep: the groups load every eighth piece each and meet in LDS.  Units of one piece are complete already; a unit
// without keys (length 0) gets its zeros here.
template <typename T, int D>
__global__ __launch_bounds__(256) void fwd_decode_combine_kernel(const KArgs a) {
	constexpr int TPR = D / 8, G = 8, RPB = 256 / (TPR * G);
	__shared__ __attribute__((aligned(16))) float sacc[RPB][G][D];
	__shared__ float smax[RPB][G], stot[RPB][G];
	const int r = a.Hq / a.Hkv, nrows = r * a.Sq;
	const int slot = threadIdx.x / (TPR * G), g = (threadIdx.x / TPR) % G, part = threadIdx.x % TPR;
	const int64_t row = (int64_t)blockIdx.x * RPB + slot;  // unit * nrows + row of the unit
	const bool live = row < (int64_t)a.B * a.Hkv * nrows;
	const int unit = live ? (int)(row / nrows) : 0, n = (int)(row - (int64_t)unit * nrows);
	const int b = unit / a.Hkv, hk = unit - b * a.Hkv;
	const bool empty = a.kv_lens && a.kv_lens[b] <= 0;
	const int w0 = a.decode_units[2 * unit], count = empty ? 0 : a.decode_units[2 * unit + 1];
	float m = -INFINITY, tot = 0.f;
	float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
	if (live && count > 1) {
#pragma unroll 4
		for (int s = g; s < count; s += G) {
			const int64_t prow = (int64_t)(w0 + s + unit) * nrows + n;
			const float lse = a.lse_part[prow];
			const float* op = a.o_part + prow * D + part * 8;
			f32x4 x0 = *(const f32x4*)op, x1 = *(const f32x4*)(op + 4);
			const float mn = __builtin_fmaxf(m, lse), ref = mn > -INFINITY ? mn : 0.f;
			const float old = exp2_fast((m - ref) * kLog2e), wgt = exp2_fast((lse - ref) * kLog2e);
			m = mn;
			tot = tot * old + wgt;
#pragma unroll
			for (int e = 0; e < 4; ++e) {
				acc[e] = acc[e] * old + wgt * x0[e];
				acc[4 + e] = acc[4 + e] * old + wgt * x1[e];
			}
		}
	}
	*(f32x4*)&sacc[slot][g][part * 8] = f32x4{acc[0], acc[1], acc[2], acc[3]};
	*(f32x4*)&sacc[slot][g][part * 8 + 4] = f32x4{acc[4], acc[5], acc[6], acc[7]};
	if (part == 0) {
		smax[slot][g] = m;
		stot[slot][g] = tot;
	}
	__syncthreads();
	if (!live || g != 0 || count == 1) return;
	m = -INFINITY;
#pragma unroll
	for (int x = 0; x < G; ++x) m = __builtin_fmaxf(m, smax[slot][x]);
	tot = 0.f;
#pragma unroll
	for (int e = 0; e < 8; ++e) acc[e] = 0.f;
	if (m > -INFINITY) {
#pragma unroll
		for (int x = 0; x < G; ++x) {
			const float wgt = exp2_fast((smax[slot][x] - m) * kLog2e);
			tot += wgt * stot[slot][x];
			f32x4 x0 = *(const f32x4*)&sacc[slot][x][part * 8], x1 = *(const f32x4*)&sacc[slot][x][part * 8 + 4];
#pragma unroll
			for (int e = 0; e < 4; ++e) {
				acc[e] += wgt * x0[e];
				acc[4 + e] += wgt * x1[e];
			}
		}
	}
	const int h = hk * r + n / a.Sq, i = n % a.Sq;
	const float inv = tot > 0.f ? 1.f / tot : 0.f;
	char* rp = a.o.ptr + (int64_t)b * a.o.sb + (int64_t)h * a.o.sh + (int64_t)i * a.o.ss + part * 16;
	*(typename T::V8*)rp = pack8<T>(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv, acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv);
	if (part == 0) a.lse[((int64_t)b * a.Hq + h) * a.Sq + i] = tot > 0.f ? m + log2_fast(tot) * kLn2 : -INFINITY;
}

template <typename T, int D>
hipError_t launch_fwd_decode_t(KArgs& a, hipStream_t s) {
	constexpr int NW = DecodeCfg<D>::NW;
	const int64_t rows = (int64_t)a.B * a.Hq * a.Sq;
	constexpr int RPB = 256 / (D / 8) / 8;
	hipLaunchKernelGGL((fwd_decode_kernel<T, D>), dim3((unsigned)((a.decode_waves + NW - 1) / NW)), dim3(NW * 64), 0, s, a);
	if (!a.decode_whole) hipLaunchKernelGGL((fwd_decode_combine_kernel<T, D>), dim3((unsigned)((rows + RPB - 1) / RPB)), dim3(256), 0, s, a);
	return hipGetLastError();
}

}  // namespace fa2
