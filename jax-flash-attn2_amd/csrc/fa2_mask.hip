// Lengths of a right-padded validity mask (the reference packs the valid tokens on the host side of its launcher,
// jax_flash_attn2/flash_attention_triton/_forward_triton.py:499-510).
#include "fa2_common.hpp"
#include "fa2_kernels.hpp"

namespace fa2 {

// non-zero bytes of a word: bit 7 of a byte of t is set where its low seven bits are not all zero
FA2_DEV int count_bytes(uint32_t x) {
	const uint32_t t = (x & 0x7f7f7f7fu) + 0x7f7f7f7fu;
	return __builtin_popcount((t | x) & 0x80808080u);
}

// One workgroup per batch row; 16 bytes per load from the first aligned one on.  A few KiB per row: what it costs is its launch, which
// is why it is one kernel and not a comparison, a conversion and a sum (B32 S511: 17 us as
// three kernels of the tensor library; a training step of that batch, H12 D64, 189 -> 179 us with this one).
__global__ __launch_bounds__(256) void mask_lengths_kernel(const uint8_t* mask, int64_t stride, int S, int32_t* lens) {
	__shared__ int part[4];
	const uint8_t* row = mask + (int64_t)blockIdx.x * stride;
	const int tid = threadIdx.x;
	int head = (int)(-(uintptr_t)row & 15);
	head = head < S ? head : S;
	const int n16 = (S - head) >> 4, tail = head + 16 * n16;
	int n = 0;
	if (tid < head) n += row[tid] != 0;
	for (int i = tid; i < n16; i += 256) {
		const u32x4 x = *(const u32x4*)(row + head + 16 * (int64_t)i);
		n += count_bytes(x[0]) + count_bytes(x[1]) + count_bytes(x[2]) + count_bytes(x[3]);
	}
	if (tid < S - tail) n += row[tail + tid] != 0;
#pragma unroll
	for (int sft = 32; sft >= 1; sft >>= 1) n += __shfl_xor(n, sft, 64);
	if ((tid & 63) == 0) part[tid >> 6] = n;
	__syncthreads();
	if (tid == 0) lens[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

hipError_t launch_mask_lengths(const uint8_t* mask, int64_t stride, int B, int S, int32_t* lens, hipStream_t s) {
	hipLaunchKernelGGL(mask_lengths_kernel, dim3((unsigned)B), dim3(256), 0, s, mask, stride, S, lens);
	return hipGetLastError();
}

}  // namespace fa2
