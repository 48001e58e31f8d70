// Small fp16 products whose operands the tile kernels' 16-byte chunks cannot fetch (odd pitches, starts or K): 32 x 32 tiles, K cut over
// the waves of a block, one launch with the epilogue.
//
// What bounds it: a serial chain of launches and memory latencies, not a rate.  Such products went through copies of both operands and a tile
// kernel, or through an element-wise kernel that walks K behind barriers in 128 x 128 tiles (a handful of blocks).  Here the waves of a block take steps of
// 32 of K in turn, straight from memory into the operands of v_mfma_f32_32x32x16_f16 (no LDS, no barrier, four steps in flight), until their
// fp32 sums meet in LDS.  us, before / now: 301 x 214 x 311 16.8 / 6.5, 187 x 1116 x 422 with a bias 20.1 / 6.5, 76 x 68 x 1783 55.4 / 11.2, 103 x 349 x 166 11.8 /
// 5.9; from there on the L1's share of the operands' way (two lines per row and step) costs 5 us per tile of a CU and 1000 of K.
#include "device_utils.hpp"
#include "gemm_epilogue.hpp"
#include "launch.hpp"
#include "anygpu_hip.h"

namespace anygpu {

namespace {

constexpr int kSmallTile = 32;                 // rows and columns of a block
constexpr int kSmallWaves = 4;
constexpr int kSmallStep = 32;                 // of K
constexpr int kSmallAhead = 4;                 // steps in flight per wave
constexpr int kSmallXcds = 8;

typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
typedef uint4_t LooseUint4 __attribute__((aligned(4)));

// Sixteen halves of a row: eight whole 4-byte words, since a vector load at an odd half costs several times one at a word (330 x 192 x 175, [N, K], bias 10.7 us
// that way).  ODD: rows may start at an odd half; there the ninth word holds the last of them (otherwise it is the eighth once more).
template <bool ODD>
struct RowWords
{
	struct Piece
	{
		uint4_t four[2];
		unsigned ninth;
	};
	const unsigned* words;
	int last;               // 8 or 7
	unsigned shift;         // 16 or 0

	__device__ __forceinline__ explicit RowWords(const half_t* row)
	{
		const uintptr_t at = reinterpret_cast<uintptr_t>(row);
		words = reinterpret_cast<const unsigned*>(at & ~(uintptr_t)3);
		last = at & 2 ? 8 : 7;
		shift = at & 2 ? 16 : 0;
	}
	__device__ __forceinline__ void load(int k, Piece& p) const       // k: even
	{
		p.four[0] = *reinterpret_cast<const LooseUint4*>(words + k / 2);
		p.four[1] = *reinterpret_cast<const LooseUint4*>(words + k / 2 + 4);
		if constexpr (ODD) p.ninth = words[k / 2 + last];
	}
	__device__ __forceinline__ half8_t halves(const Piece& p, int j) const
	{
		uint4_t v = p.four[j];
		if constexpr (ODD)
		{
			const unsigned behind = j == 0 ? p.four[1][0] : p.ninth;
			v = uint4_t{__builtin_amdgcn_alignbit(v[1], v[0], shift), __builtin_amdgcn_alignbit(v[2], v[1], shift),
			            __builtin_amdgcn_alignbit(v[3], v[2], shift), __builtin_amdgcn_alignbit(behind, v[3], shift)};
		}
		return __builtin_bit_cast(half8_t, v);
	}
};

template <bool B_NK, bool ODD, int EPI>
__global__ __launch_bounds__(64 * kSmallWaves) void gemm_f16_small_kernel(
	const half_t* __restrict__ A, const half_t* __restrict__ B, const half_t* __restrict__ bias, half_t* __restrict__ C,
	int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, float ep_param, int tiles_m, int tiles, int tiles_per_xcd)
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
	const int m = min(m0 + i32, M - 1);
	const int n = min(n0 + i32, N - 1);
	// (the summation index of an MFMA is a dummy index: lane half h takes k = 16 h + 8 j + e of a step in MFMA j)
	const half_t* a_row = A + m * lda + 16 * h;
	const half_t* b_row = B_NK ? B + n * ldb + 16 * h : B + n + 16 * h * ldb;

	float16_t acc;
#pragma unroll
	for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
	const RowWords<ODD> a_words(a_row), b_words(b_row);
	typename RowWords<ODD>::Piece a[kSmallAhead], b[kSmallAhead];
	half8_t b_kn[kSmallAhead][2];
	auto load = [&](int d, int k) {             // k + kSmallStep <= K
		a_words.load(k, a[d]);
		if constexpr (B_NK) b_words.load(k, b[d]);
		else
		{
#pragma unroll
			for (int j = 0; j < 2; ++j)
#pragma unroll
				for (int e = 0; e < 8; ++e) b_kn[d][j][e] = b_row[(int64_t)(k + 8 * j + e) * ldb];
		}
	};
	auto multiply = [&](int d) {
#pragma unroll
		for (int j = 0; j < 2; ++j)
			acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_words.halves(a[d], j), B_NK ? b_words.halves(b[d], j) : b_kn[d][j], acc, 0, 0, 0);
	};

	// whole steps wave, wave + kSmallWaves, ...  (behind the last one: that one again, of no consequence)
	const int steps = K / kSmallStep;
	const int mine = steps > wave ? (steps - wave + kSmallWaves - 1) / kSmallWaves : 0;
	auto k_of = [&](int i) { return (wave + kSmallWaves * (i < mine ? i : mine - 1)) * kSmallStep; };
	if (mine > 0)
	{
#pragma unroll
		for (int d = 0; d < kSmallAhead; ++d) load(d, k_of(d));
		for (int i = 0; i < mine; i += kSmallAhead)
		{
#pragma unroll
			for (int d = 0; d < kSmallAhead; ++d)
			{
				if (i + d < mine) multiply(d);
				__builtin_amdgcn_sched_barrier(0);
				load(d, k_of(i + d + kSmallAhead));
				__builtin_amdgcn_sched_barrier(0);
			}
		}
	}
	// the rest of K, element by element (those past the end read the last one and count as zeros), by the wave whose turn it is
	if (steps % kSmallWaves == wave && steps * kSmallStep < K)
	{
		half8_t a_end[2], b_end[2];
#pragma unroll
		for (int j = 0; j < 2; ++j)
#pragma unroll
			for (int e = 0; e < 8; ++e)
			{
				const int k = steps * kSmallStep + 16 * h + 8 * j + e, at = min(k, K - 1) - 16 * h;
				const half_t x = a_row[at], y = B_NK ? b_row[at] : b_row[at * ldb];
				a_end[j][e] = k < K ? x : (half_t)0.0f;
				b_end[j][e] = k < K ? y : (half_t)0.0f;
			}
#pragma unroll
		for (int j = 0; j < 2; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_end[j], b_end[j], acc, 0, 0, 0);
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
		C[(m0 + r) * ldc + n0 + c] = (half_t)finish_sum<EPI, true>(sum, 0.0f, EPI == kEpiBias && bias ? (float)bias[n0 + c] : 0.0f, ep_param);
	}
}

template <bool B_NK, bool ODD, int EPI>
hipError_t launch_small(const half_t* A, const half_t* B, const half_t* bias, half_t* C, int64_t M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc, float ep_param, hipStream_t stream)
{
	const int tiles_m = (int)((M + kSmallTile - 1) / kSmallTile);
	const int tiles = tiles_m * (int)((N + kSmallTile - 1) / kSmallTile);
	const int per_xcd = (tiles + kSmallXcds - 1) / kSmallXcds;
	discard_stale_error();
	gemm_f16_small_kernel<B_NK, ODD, EPI><<<dim3((unsigned)(per_xcd * kSmallXcds)), dim3(64 * kSmallWaves), 0, stream>>>(
		A, B, bias, C, (int)M, (int)N, (int)K, lda, ldb, ldc, ep_param, tiles_m, tiles, per_xcd);
	return hipGetLastError();
}

}  // namespace

// Where it is ahead (us, the other kernels / here), for operands that the tile kernels' chunks do not fit:
//   * Few rows against [N, K] weights at any row count (1 x 1001 x 700 15.4 / 4.5, 16 x 2304 x 749 13.0 / 6.7; 8 x 700 x 2001 9.2 / 9.3, from where
//     few tiles walk longer rows the few-row kernels stay), [K, N] from three rows on (4 x 1001 x 700 8.5 / 6.6, 16 rows 23.6 / 6.9; 1 row 6.1 / 6.5).
//   * Against the element-wise kernel, and against copies of the operands and a tile kernel (two or three launches): up to one and a half tiles per CU and some
//     1600 of K at one (301 x 214 x 311 16.8 / 6.5, 352 x 536 x 2162 18.4 / 10.8, 48 x 3000 x 3001 24.0 / 16.0, 1535 x 178 x 551 13.7 / 11.0; but 353 x 693 x 2033
//     17.2 / 21.9, 1505 x 618 x 141 9.2 / 15.1), with an epilogue, which the copies do not take, up to two and a half (133 x 363 x 1342 56.7 / 10.0,
//     866 x 762 x 919 20.9 / 20.4, 516 x 1211 x 328 11.8 / 11.3; but 336 x 1757 x 3029 29.0 / 43.0).
bool gemm_f16_small_applies(int64_t M, int64_t N, int64_t K, int b_layout, bool with_epilogue)
{
	const int64_t cus = device_cu_count();
	if (K < 1 || K > 4096 || M > kSmallTile * 3 * cus || N > kSmallTile * 3 * cus) return false;
	if (b_layout == ANYGPU_B_ROW_MAJOR && M < 3) return false;
	const int64_t tiles = ((M + kSmallTile - 1) / kSmallTile) * ((N + kSmallTile - 1) / kSmallTile);
	if (M <= 16 && b_layout == ANYGPU_B_COL_MAJOR && 4 * tiles < cus && K > 1536) return false;
	if (with_epilogue) return 2 * tiles <= 5 * cus && tiles * K <= 2400 * cus;
	return 2 * tiles <= 3 * cus && tiles * K <= 1600 * cus;
}

hipError_t launch_gemm_f16_small(const void* A, const void* B, const void* bias, void* C, int64_t M, int64_t N, int64_t K,
                                 int64_t lda, int64_t ldb, int64_t ldc, int b_layout, int epilogue, float ep_param, hipStream_t stream)
{
	const half_t* a = static_cast<const half_t*>(A);
	const half_t* b = static_cast<const half_t*>(B);
	const half_t* bs = static_cast<const half_t*>(bias);
	half_t* c = static_cast<half_t*>(C);
	const bool nk = b_layout == ANYGPU_B_COL_MAJOR;
	const bool odd = lda % 2 != 0 || reinterpret_cast<uintptr_t>(A) % 4 != 0 || (nk && (ldb % 2 != 0 || reinterpret_cast<uintptr_t>(B) % 4 != 0));
#define ANYGPU_F16_SMALL(NK, EPI) \
	return odd ? launch_small<NK, true, EPI>(a, b, bs, c, M, N, K, lda, ldb, ldc, ep_param, stream) \
	           : launch_small<NK, false, EPI>(a, b, bs, c, M, N, K, lda, ldb, ldc, ep_param, stream)
	if (nk)
	{
		if (epilogue == kEpiSoftcap) ANYGPU_F16_SMALL(true, kEpiSoftcap);
		ANYGPU_F16_SMALL(true, kEpiBias);
	}
	if (epilogue == kEpiSoftcap) ANYGPU_F16_SMALL(false, kEpiSoftcap);
	ANYGPU_F16_SMALL(false, kEpiBias);
#undef ANYGPU_F16_SMALL
}

}  // namespace anygpu
