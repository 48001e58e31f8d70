// fp32 products too small for the 64 x 64 tiles to fill the chip: 32 x 32 tiles, K cut over the waves of a block.
//
// What bounds it: a serial chain, not a rate.  256 x 1024 x 512 is 64 tiles of 64 x 64, which leave 192 CUs idle while each of the
// others walks all of K behind barriers.  As 32 x 32 tiles they are 256 blocks, and the waves of a block take steps of 32 of K
// in turn, straight from memory into the operands of v_mfma_f32_32x32x2_f32 (no LDS, no barrier, two steps in flight), until
// their sums meet in LDS.  The summation index of an MFMA is a dummy index: lane half h takes k = 8 j + 4 h + e in MFMA (j, e), so
// that a lane reads four consecutive k of a k-contiguous operand with one 16-byte load; an n-contiguous right operand
// comes in whole 128-byte lines, a row of k per load and lane half.  Loads are aligned to elements, so any pitch is taken as it lies.
// 256 x 1024 x 512: 11.3 -> 6.5 us (41 TFLOP/s); from there on K costs 0.9 us per 128 (the L1's share of the operands' way, not MFMAs).
#include "device_utils.hpp"
#include "launch.hpp"
#include "anygpu_hip.h"

namespace anygpu {

namespace {

constexpr int kSmallTile = 32;                 // rows and columns of a block
constexpr int kSmallStep = 32;                 // of K
constexpr int kSmallWaves = 4;               // 8 and 16 move the same bytes and measured 0 - 25 % slower
constexpr int kSmallXcds = 8;

typedef float LooseFloat4 __attribute__((ext_vector_type(4), aligned(4)));

template <bool B_NK>
__global__ __launch_bounds__(64 * kSmallWaves) void gemm_f32_small_kernel(
	const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias, float* __restrict__ C,
	int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int tiles_m, int tiles, int tiles_per_xcd)
{
	__shared__ float sums[kSmallWaves][kSmallTile][kSmallTile];

	const int lane = threadIdx.x & (kWaveSize - 1);
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int i32 = lane & 31, h = lane >> 5;
	// consecutive blocks go to the eight XCDs in turn: an XCD takes neighbouring column tiles (all of their row tiles), so that
	// its L2 holds an eighth of B
	const int tile = (int)(blockIdx.x % kSmallXcds) * tiles_per_xcd + (int)(blockIdx.x / kSmallXcds);
	if (tile >= tiles) return;                  // the whole block
	const int m0 = tile % tiles_m * kSmallTile, n0 = tile / tiles_m * kSmallTile;
	// rows and columns past the end are replaced by the last one (their sums are never stored)
	const int m = m0 + i32 < M ? m0 + i32 : M - 1;
	const int n = n0 + i32 < N ? n0 + i32 : N - 1;
	const float* a_row = A + (int64_t)m * lda + 4 * h;
	const float* b_row = B_NK ? B + (int64_t)n * ldb + 4 * h : B + n + 4 * h * ldb;

	float16_t acc;
#pragma unroll
	for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
	float4_t a[2][4], b[2][4];
	auto load = [&](int d, int k) {             // k + kSmallStep <= K
#pragma unroll
		for (int j = 0; j < 4; ++j) a[d][j] = *reinterpret_cast<const LooseFloat4*>(a_row + k + 8 * j);
		if constexpr (B_NK)
		{
#pragma unroll
			for (int j = 0; j < 4; ++j) b[d][j] = *reinterpret_cast<const LooseFloat4*>(b_row + k + 8 * j);
		}
		else
		{
#pragma unroll
			for (int j = 0; j < 4; ++j)
#pragma unroll
				for (int e = 0; e < 4; ++e) b[d][j][e] = b_row[(int64_t)(k + 8 * j + e) * ldb];
		}
	};
	auto multiply = [&](int d) {
#pragma unroll
		for (int j = 0; j < 4; ++j)
#pragma unroll
			for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[d][j][e], b[d][j][e], acc, 0, 0, 0);
	};

	// whole steps wave, wave + kSmallWaves, ...  (conditions are the same for a whole wave)
	const int steps = K / kSmallStep;
	const int mine = steps > wave ? (steps - wave + kSmallWaves - 1) / kSmallWaves : 0;
	auto k_of = [&](int i) { return (wave + kSmallWaves * i) * kSmallStep; };
	int i = 0;
	if (mine >= 2)
	{
		load(0, k_of(0));
		load(1, k_of(1));
		for (; i + 4 <= mine; i += 2)
		{
			multiply(0);
			__builtin_amdgcn_sched_barrier(0);
			load(0, k_of(i + 2));
			__builtin_amdgcn_sched_barrier(0);
			multiply(1);
			__builtin_amdgcn_sched_barrier(0);
			load(1, k_of(i + 3));
			__builtin_amdgcn_sched_barrier(0);
		}
		multiply(0);
		__builtin_amdgcn_sched_barrier(0);
		if (i + 2 < mine) load(0, k_of(i + 2));
		__builtin_amdgcn_sched_barrier(0);
		multiply(1);
		if (i + 2 < mine) multiply(0);
	}
	else if (mine == 1)
	{
		load(0, k_of(0));
		multiply(0);
	}
	// the rest of K, element by element, by the wave whose turn it is
	if (steps % kSmallWaves == wave && steps * kSmallStep < K)
	{
#pragma unroll
		for (int j = 0; j < 4; ++j)
#pragma unroll
			for (int e = 0; e < 4; ++e)
			{
				const int k = steps * kSmallStep + 8 * j + e;              // of lane half 0
				const bool in = k + 4 * h < K;
				a[0][j][e] = in ? a_row[k] : 0.0f;
				b[0][j][e] = in ? (B_NK ? b_row[k] : b_row[(int64_t)k * ldb]) : 0.0f;
			}
		multiply(0);
	}

	// register r of a lane: row 8 (r / 4) + 4 h + r % 4, column i32
#pragma unroll
	for (int r = 0; r < 16; ++r) sums[wave][8 * (r / 4) + 4 * h + r % 4][i32] = acc[r];
	__syncthreads();
	for (int o = threadIdx.x; o < kSmallTile * kSmallTile; o += 64 * kSmallWaves)
	{
		const int r = o / kSmallTile, c = o % kSmallTile;
		if (m0 + r >= M || n0 + c >= N) continue;
		float sum = 0.0f;
#pragma unroll
		for (int w = 0; w < kSmallWaves; ++w) sum += sums[w][r][c];
		C[(int64_t)(m0 + r) * ldc + n0 + c] = sum + (bias ? bias[n0 + c] : 0.0f);
	}
}

template <bool B_NK>
hipError_t launch_small(const float* A, const float* B, const float* bias, float* C, int64_t M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc, hipStream_t stream)
{
	const int tiles_m = (int)((M + kSmallTile - 1) / kSmallTile);
	const int tiles = tiles_m * (int)((N + kSmallTile - 1) / kSmallTile);
	const int per_xcd = (tiles + kSmallXcds - 1) / kSmallXcds;
	discard_stale_error();
	gemm_f32_small_kernel<B_NK><<<dim3((unsigned)(per_xcd * kSmallXcds)), dim3(64 * kSmallWaves), 0, stream>>>(
		A, B, bias, C, (int)M, (int)N, (int)K, lda, ldb, ldc, tiles_m, tiles, per_xcd);
	return hipGetLastError();
}

}  // namespace

// Where it is ahead (us, before / here; right operand [K, N], [N, K] alike): whole slabs of K and aligned rows, which the 64 x 64
// tiles' four-wave kernel takes: up to a tile per CU and 768 of K (256 x 1024 x 512 11.3 / 6.5, 64 x 4096 x 256 7.2 / 4.7, 128^3 5.2 /
// 3.4; but 128 x 256 x 1024 9.3 / 9.6, 512 x 512 x 2048 15.6 / 17.3, where that kernel cuts K over blocks, and two tiles per CU: 512 x
// 1024 x 512 11.2 / 12.9).  Ragged operands cost the other kernels far more: up to 1536 of K (305 x 272 x 921 17.3 / 10.5, 150 x 1500
// x 333 15.5 / 5.7; 130 x 131 x 3000 21.1 / 23.0) and with two tiles per CU up to 768 (700^3 25.2 / 18.4; with four: 1000 x
// 1000 x 333 16.1 / 20.8).  Up to 16 rows the few-row kernels take all but ragged products of little K (12 x 777 x 333 15.5 / 5.2;
// 2 rows 2.9 / 5.4; 4 x 2304 x 750 6.9 / 7.5 with [K, N], 15.7 / 6.5 with [N, K]).
bool gemm_f32_small_applies(const float* A, const float* B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int b_layout)
{
	const int64_t cus = device_cu_count();
	if (M < 3 || K < 1 || K > 1536 || M > kSmallTile * 2 * cus || N > kSmallTile * 2 * cus) return false;
	const int64_t tiles = ((M + kSmallTile - 1) / kSmallTile) * ((N + kSmallTile - 1) / kSmallTile);
	const uintptr_t bits = reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B);
	const bool ragged = K % kSmallStep != 0 || lda % 4 != 0 || ldb % 4 != 0 || bits % 16 != 0;
	if (!ragged) return M > 16 && tiles <= cus && K <= 768;
	if (M <= 16) return tiles <= cus && K <= (M <= 4 && b_layout == ANYGPU_B_ROW_MAJOR ? 512 : 768);
	return tiles <= (K <= 768 ? 2 * cus : cus);
}

hipError_t launch_gemm_f32_small(const float* A, const float* B, const float* bias, float* C, int64_t M, int64_t N, int64_t K,
                                 int64_t lda, int64_t ldb, int64_t ldc, int b_layout, hipStream_t stream)
{
	if (b_layout == ANYGPU_B_COL_MAJOR) return launch_small<true>(A, B, bias, C, M, N, K, lda, ldb, ldc, stream);
	return launch_small<false>(A, B, bias, C, M, N, K, lda, ldb, ldc, stream);
}

}  // namespace anygpu
