// Products with up to 16 left-operand rows against k-contiguous weights (column-major B, [N, K]): K is cut over the waves of
// a block, so that a weight matrix of any number of columns is streamed by enough waves in ONE launch.
//
// What bounds it: the weights' way from memory.  The kernels this one replaces cut K over blocks: their partial sums went through
// memory and a second launch added them, and their blocks (128 columns, a band of A staged through LDS behind barriers) left
// one to two on a CU.  Here a block owns up to 32 weight rows (of each of its matrices) and its waves walk K in turn, a step of
// 128 bytes per weight row at a time, without LDS, barriers or partial sums in memory until their sums meet in LDS at the end.
//
// Eight rows on both sides of a 16 x 16 MFMA: slots 0 - 7 of either operand hold the rows' chunks 0, 2, 4, 6 of a step
// (a chunk: the 16 bytes of one lane), slots 8 - 15 the same rows' chunks 1, 3, 5, 7.  The two diagonal 8 x 8 blocks of the result
// are the two halves of the sums, the other two are dropped: the matrix cores have the time, and one load instruction
// reads whole 128-byte lines of eight rows.  The left operand is read the same way, straight from memory (it stays in the
// L2s); with 9 - 16 rows it has two such operands per weight vector.
//
// Rows per block: the fewest blocks that give every CU the same number of them (2304 columns: 256 blocks of 9 rows, 9216:
// 512 of 18), as a CU with one block more than the others is what the launch waits for (2304 columns in 288 blocks of 8: 18 us,
// in 256 of 9: 11.5), and few, as every block reads the whole left operand.  Two steps in flight per wave, eight waves to a block
// of up to 16 rows and four to a larger one (depths of 2, 3, 4 and 4, 8, 16 waves were measured).
// Measured, us before -> now, 8 rows, weights from memory (700 MB of them walked in turn), fp16: 2304 -> 9216 with the GELU of two matrices
// 30.7 -> 16.6, 9216 -> 2304 19.8 -> 12.3 (3.5 TB/s), 2304 -> 2048 10.4 -> 4.6, 4096 -> 4096 14.2 -> 8.3, 3584 -> 18944 35.5 -> 25.5 (5.3 TB/s).
// A matrix that the caches still hold from the product before is read at their rate by either kernel, where the one with a band
// of A in LDS can be a tenth ahead (9216 x 2304 10.0 / 11.2, 18944 x 3584 22.9 / 25.2; 2304 x 9216 14.2 / 12.9).
#include "gemm_band.hpp"
#include "anygpu_hip.h"

namespace anygpu {

using namespace band;

namespace {

constexpr int kKwaveRows = 8;                      // weight rows (output columns) per tile
constexpr int kKwaveMaxTiles = 4;
constexpr int kKwaveStepBytes = 128;               // bytes of a weight row per step

// C[m, n] = finish(sum_k A[m, k] B[n, k]), M <= 8 MB.  blockIdx.x: group of rows_per_block <= 8 * TILES
// output columns.  K a multiple of a step, with DEPTH or more steps for every wave.
template <typename T, int MB, int TILES, int WAVES, int DEPTH, int EPI>
__global__ __launch_bounds__(64 * WAVES) void gemm_kwave_kernel(
	const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ B2, const T* __restrict__ bias, T* __restrict__ C,
	int M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, float ep_param, int rows_per_block)
{
	constexpr bool DUAL = (EPI == kEpiGeluMul);
	constexpr int kMats = DUAL ? 2 : 1;
	constexpr int kW = kMats * TILES;                                  // weight vectors per lane and step
	constexpr int kStep = kKwaveStepBytes / (int)sizeof(T);
	constexpr int kChunk = 16 / (int)sizeof(T);
	__shared__ float sums[WAVES][kW][MB][2][8][kKwaveRows];            // [half][band row][weight row]

	const int lane = threadIdx.x & (kWaveSize - 1);
	const int wave = threadIdx.x >> 6;
	const int slot = lane & 15;
	const int row = slot & 7;
	const int half = slot >> 3;
	const int grp = lane >> 4;
	const int64_t n0 = (int64_t)blockIdx.x * rows_per_block;
	const int64_t n_last = n0 + rows_per_block < N ? n0 + rows_per_block - 1 : N - 1;
	const int64_t chunk_at = (int64_t)(2 * grp + half) * kChunk;

	// rows past the end are replaced by the last one (their sums are never stored)
	const T* wrow[kW];
#pragma unroll
	for (int t = 0; t < TILES; ++t)
	{
		int64_t n = n0 + 8 * t + row;
		n = n < n_last ? n : n_last;
		wrow[t] = B + n * ldb + chunk_at;
		if constexpr (DUAL) wrow[TILES + t] = B2 + n * ldb + chunk_at;
	}
	const T* arow[MB];
#pragma unroll
	for (int b = 0; b < MB; ++b) arow[b] = A + (int64_t)(8 * b + row < M ? 8 * b + row : M - 1) * lda + chunk_at;

	// steps wave, wave + WAVES, ...; walked from a start that differs from block to block (with weight rows a power of two
	// apart, equal offsets in all rows share their memory channel)
	const int steps = (int)(K / kStep);
	const int mine = steps > wave ? (steps - wave + WAVES - 1) / WAVES : 0;
	const int first = mine > 1 ? (int)((blockIdx.x * 2654435761u >> 8) % (unsigned)mine) : 0;
	auto k_at = [&](int i) {                                           // i < 2 * mine
		const int s = i + first;
		return (int64_t)(wave + WAVES * (s >= mine ? s - mine : s)) * kStep;
	};

	Vec w[DEPTH][kW], a[DEPTH][MB];
	auto issue = [&](int d, int i) {                                   // i < mine
		const int64_t k = k_at(i);
#pragma unroll
		for (int j = 0; j < kW; ++j) w[d][j] = __builtin_nontemporal_load(reinterpret_cast<const Vec*>(wrow[j] + k));
#pragma unroll
		for (int b = 0; b < MB; ++b) a[d][b] = *reinterpret_cast<const Vec*>(arow[b] + k);
	};

	float4_t acc[kW][MB];
#pragma unroll
	for (int j = 0; j < kW; ++j)
#pragma unroll
		for (int b = 0; b < MB; ++b) acc[j][b] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
	auto multiply = [&](int d) {
#pragma unroll
		for (int j = 0; j < kW; ++j)
#pragma unroll
			for (int b = 0; b < MB; ++b) BandMma<T, 16>::mma(w[d][j], a[d][b], acc[j][b]);
	};

	// (every condition here is the same for a whole wave; the launcher sees to it that every wave has DEPTH steps or more, so
	// that these loads are unconditional: with a condition around them the compiler waits for all of them at once)
#pragma unroll
	for (int d = 0; d < DEPTH; ++d) issue(d, d);
	int i = 0;
	for (; i + 2 * DEPTH <= mine; i += DEPTH)
	{
#pragma unroll
		for (int d = 0; d < DEPTH; ++d)
		{
			multiply(d);
			__builtin_amdgcn_sched_barrier(0);
			issue(d, i + DEPTH + d);
			__builtin_amdgcn_sched_barrier(0);
		}
	}
#pragma unroll
	for (int d = 0; d < DEPTH; ++d)
	{
		if (i + d < mine) multiply(d);
		if (i + DEPTH + d < mine) issue(d, i + DEPTH + d);
	}
#pragma unroll
	for (int d = 0; d < DEPTH; ++d)
		if (i + DEPTH + d < mine) multiply(d);

	// lane (slot, grp) holds the sums of band slot `slot` and weight slots 4 grp .. 4 grp + 3: of use where both are in
	// the same half
	if ((grp >> 1) == half)
	{
#pragma unroll
		for (int j = 0; j < kW; ++j)
#pragma unroll
			for (int b = 0; b < MB; ++b) *reinterpret_cast<float4_t*>(&sums[wave][j][b][half][row][4 * (grp & 1)]) = acc[j][b];
	}
	__syncthreads();
	// one output per thread: eight neighbouring columns of a row by eight neighbouring threads
	constexpr int kOutputs = TILES * MB * 64;
	for (int o = threadIdx.x; o < kOutputs; o += 64 * WAVES)
	{
		const int col = o & 7, m_in = (o >> 3) & 7, b = (o >> 6) % MB, t = (o >> 6) / MB;
		const int m = 8 * b + m_in;
		const int64_t n = n0 + 8 * t + col;
		if (m >= M || n > n_last) continue;
		float sum[kMats];
#pragma unroll
		for (int q = 0; q < kMats; ++q)
		{
			sum[q] = 0.0f;
#pragma unroll
			for (int v = 0; v < WAVES; ++v) sum[q] += sums[v][q * TILES + t][b][0][m_in][col] + sums[v][q * TILES + t][b][1][m_in][col];
		}
		const float bias_n = (EPI == kEpiBias && bias) ? (float)bias[n] : 0.0f;
		C[(int64_t)m * ldc + n] = (T)finish_sum<EPI>(sum[0], sum[kMats - 1], bias_n, ep_param);
	}
}

template <typename T, int MB, int TILES, int WAVES, int DEPTH, int EPI>
hipError_t launch_kwave(const T* A, const T* B, const T* B2, const T* bias, T* C, int M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc, float ep_param, int rows_per_block, hipStream_t stream)
{
	discard_stale_error();
	const unsigned blocks = (unsigned)((N + rows_per_block - 1) / rows_per_block);
	gemm_kwave_kernel<T, MB, TILES, WAVES, DEPTH, EPI><<<dim3(blocks), dim3(64 * WAVES), 0, stream>>>(
		A, B, B2, bias, C, M, N, K, lda, ldb, ldc, ep_param, rows_per_block);
	return hipGetLastError();
}

constexpr int kKwaveDepth = 2;
constexpr int kKwaveWavesFew = 8, kKwaveWavesMany = 4;      // waves of a block with up to two, with three or four tiles

// the same number of blocks for every CU, as few as the tiles of a block allow
int rows_per_block_for(int64_t N)
{
	const int64_t cus = device_cu_count();
	const int64_t per_cu = (N + cus * kKwaveRows * kKwaveMaxTiles - 1) / (cus * kKwaveRows * kKwaveMaxTiles);
	return (int)((N + cus * per_cu - 1) / (cus * per_cu));
}

template <typename T, int MB, int EPI>
hipError_t launch_kwave_tiles(const T* A, const T* B, const T* B2, const T* bias, T* C, int M, int64_t N, int64_t K,
                              int64_t lda, int64_t ldb, int64_t ldc, float ep_param, hipStream_t stream)
{
	const int rows = rows_per_block_for(N);
#define ANYGPU_KWAVE(TILES, WAVES) \
	return launch_kwave<T, MB, TILES, WAVES, kKwaveDepth, EPI>(A, B, B2, bias, C, M, N, K, lda, ldb, ldc, ep_param, rows, stream)
	if (rows <= kKwaveRows) ANYGPU_KWAVE(1, kKwaveWavesFew);
	if (rows <= 2 * kKwaveRows) ANYGPU_KWAVE(2, kKwaveWavesFew);
	if (rows <= 3 * kKwaveRows) ANYGPU_KWAVE(3, kKwaveWavesMany);
	ANYGPU_KWAVE(4, kKwaveWavesMany);
#undef ANYGPU_KWAVE
}

template <typename T, int EPI>
hipError_t launch_kwave_rows(const T* A, const T* B, const T* B2, const T* bias, T* C, int M, int64_t N, int64_t K,
                             int64_t lda, int64_t ldb, int64_t ldc, float ep_param, hipStream_t stream)
{
	if (M <= 8) return launch_kwave_tiles<T, 1, EPI>(A, B, B2, bias, C, M, N, K, lda, ldb, ldc, ep_param, stream);
	return launch_kwave_tiles<T, 2, EPI>(A, B, B2, bias, C, M, N, K, lda, ldb, ldc, ep_param, stream);
}

}  // namespace

// Rows of both operands at 16-byte boundaries and whole steps of 128 bytes of K, enough of them for every wave, and the row
// counts at which it is ahead of what took these products before (us, before / here):
// one matrix, up to 8 rows: from 2 rows in fp16 (weights from memory, 2 rows: 9216 x 2304 9.8 / 9.8, 2304 x 9216 11.6 / 10.0, 4096 x 4096
//   8.3 / 7.6, 14336 x 4096 22.8 / 21.2, 3000 x 1024 3.5 / 3.7; out of the caches 9.1 / 9.4, 10.9 / 11.2, 6.8 / 7.8, -, 3.1 / 3.6; 3 rows: 15.3 / 9.6) and
//   from 3 in fp32 (2 rows: 16.3 / 16.2; 3 rows: 25.3 / 17);
// one matrix, 9 - 16 rows, where the left operand's way through the L2s grows with the rows: small weight matrices only (fp16,
//   16 rows: 2048 x 2304 8.5 / 5.6, but 9216 x 2304 9.9 / 12.0; fp32: 2048 x 2048 9.8 / 8.0, 9216 x 2304 26.0 / 26.4);
// two matrices: in fp16 at all row counts (9216 x 2304: 1 row 22.5 / 15, 16 rows 29.8 / 18), in fp32 3 - 8 rows (46.8 / 31.4;
//   2 rows 30.4 / 30.3, 16 rows 47 / 52) and small matrices up to 16 (2048 x 2048, 16 rows 15.3 / 11.3).
template <typename T>
bool gemm_kwave_applies(const T* A, const T* B, const T* B2, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int b_layout, bool dual)
{
	constexpr bool HALF = sizeof(T) == 2;
	constexpr int64_t kChunk = 16 / (int64_t)sizeof(T), kStep = kKwaveStepBytes / (int64_t)sizeof(T);
	if (b_layout != ANYGPU_B_COL_MAJOR || N < 1 || K % kStep != 0 || K < kStep * kKwaveWavesFew * kKwaveDepth) return false;
	if (M < (HALF ? (dual ? 1 : 2) : 3) || M > 16) return false;
	if (M > 8 && !(HALF && dual) && (double)N * (double)K > 1.0e7) return false;
	if (N > (int64_t)0x7FFFFFFF || K / kStep > (int64_t)0x7FFFFFFF / 2) return false;
	return lda % kChunk == 0 && ldb % kChunk == 0 && aligned16(A) && aligned16(B) && (!dual || aligned16(B2));
}

template <typename T>
hipError_t launch_gemm_kwave(const T* A, const T* B, const T* B2, const T* bias, T* C, int64_t M, int64_t N, int64_t K,
                             int64_t lda, int64_t ldb, int64_t ldc, int epilogue, float ep_param, hipStream_t stream)
{
	if (epilogue == kEpiSoftcap) return launch_kwave_rows<T, kEpiSoftcap>(A, B, B2, bias, C, (int)M, N, K, lda, ldb, ldc, ep_param, stream);
	if (epilogue == kEpiGeluMul) return launch_kwave_rows<T, kEpiGeluMul>(A, B, B2, bias, C, (int)M, N, K, lda, ldb, ldc, ep_param, stream);
	return launch_kwave_rows<T, kEpiBias>(A, B, B2, bias, C, (int)M, N, K, lda, ldb, ldc, ep_param, stream);
}

template bool gemm_kwave_applies<float>(const float*, const float*, const float*, int64_t, int64_t, int64_t, int64_t, int64_t, int, bool);
template bool gemm_kwave_applies<half_t>(const half_t*, const half_t*, const half_t*, int64_t, int64_t, int64_t, int64_t, int64_t, int, bool);
template hipError_t launch_gemm_kwave<float>(const float*, const float*, const float*, const float*, float*, int64_t, int64_t, int64_t,
                                             int64_t, int64_t, int64_t, int, float, hipStream_t);
template hipError_t launch_gemm_kwave<half_t>(const half_t*, const half_t*, const half_t*, const half_t*, half_t*, int64_t, int64_t, int64_t,
                                              int64_t, int64_t, int64_t, int, float, hipStream_t);

}  // namespace anygpu
