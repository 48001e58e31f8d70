// Equal shares of a masked attention launch: the set tiles of the visible-tile map, head after head and query block after query block, are cut
// into as many ranges of equal length as blocks are resident, and every block walks one range.
//
// Whole query blocks, or equal numbers of parts of each, leave the CUs unequal work where the mask leaves the query blocks unequal numbers
// of tiles, and every part pays for its start and its partial result; here a block starts a handful of query blocks, and only
// those that a range ends inside leave partial results, at most two per range.  A query block without a set tile counts as one tile: its
// rows are zeros that somebody has to write.
#pragma once

#include "attention_tile_map.hpp"
#include "device_utils.hpp"

#include <hip/hip_runtime.h>
#include <cstdint>

namespace anygpu {

struct AttnBalance
{
	int ranges;            // blocks of the launch
	int heads;
	int q_blocks;          // per head
	int words;             // 64-bit map words per query block
	int least;             // tiles of a range at least
};

// tiles that query block b counts for
__device__ __forceinline__ int balance_tiles(const unsigned long long* __restrict__ map, const AttnBalance& w, int b)
{
	int n = 0;
	for (int i = 0; i < w.words; ++i) n += __builtin_popcountll(map[(int64_t)b * w.words + i]);
	return n > 0 ? n : 1;
}

// Position of tiles in the order of the ranges.  All waves of a block compute the same (64 query blocks at a time, one per lane).
struct BalanceScan
{
	int per_head;          // tiles of one head
	int per;               // tiles of a range

	__device__ __forceinline__ BalanceScan(const unsigned long long* __restrict__ map, const AttnBalance& w)
	{
		const int lane = threadIdx.x & 63;
		int sum = 0;
		for (int b = lane; b < w.q_blocks; b += 64) sum += balance_tiles(map, w, b);
#pragma unroll
		for (int d = 1; d < 64; d <<= 1) sum += __shfl_xor(sum, d);
		per_head = __builtin_amdgcn_readfirstlane(sum);
		const int64_t total = (int64_t)per_head * w.heads;
		const int64_t even = (total + w.ranges - 1) / w.ranges;
		per = __builtin_amdgcn_readfirstlane((int)(even > w.least ? even : w.least));
	}
	// the query block that holds tile x of a head, and the first tile of it
	__device__ __forceinline__ void locate(const unsigned long long* __restrict__ map, const AttnBalance& w, int x, int& q_block, int& first) const
	{
		const int lane = threadIdx.x & 63;
		int before = 0;
		for (int c = 0; c < w.q_blocks; c += 64)
		{
			const int own = c + lane < w.q_blocks ? balance_tiles(map, w, c + lane) : 0;
			int upto = own;
#pragma unroll
			for (int d = 1; d < 64; d <<= 1)
			{
				const int other = __shfl_up(upto, d);
				upto += lane >= d ? other : 0;
			}
			const unsigned long long past = __builtin_amdgcn_ballot_w64(before + upto > x);
			if (past != 0)
			{
				const int at = __builtin_ctzll(past);
				q_block = c + at;
				first = before + __builtin_amdgcn_readlane(upto - own, at);
				return;
			}
			before += __builtin_amdgcn_readlane(upto, 63);
		}
		q_block = w.q_blocks;          // (not reached: x is below per_head)
		first = before;
	}
	// tiles of a head in front of query block b
	__device__ __forceinline__ int tiles_before(const unsigned long long* __restrict__ map, const AttnBalance& w, int b) const
	{
		const int lane = threadIdx.x & 63;
		int sum = 0;
		for (int i = lane; i < b; i += 64) sum += balance_tiles(map, w, i);
#pragma unroll
		for (int d = 1; d < 64; d <<= 1) sum += __shfl_xor(sum, d);
		return __builtin_amdgcn_readfirstlane(sum);
	}
};

// Index of the set bit number `nth` of a map row.
__device__ __forceinline__ int balance_nth_tile(const unsigned long long* __restrict__ map_row, int words, int nth)
{
	for (int i = 0; i < words; ++i)
	{
		unsigned long long bits = map_row[i];
		const int here = __builtin_popcountll(bits);
		if (nth >= here)
		{
			nth -= here;
			continue;
		}
		for (; nth > 0; --nth) bits &= bits - 1;
		return 64 * i + __builtin_ctzll(bits);
	}
	return 64 * words;
}

// Where a range's partial result of a query block lies: slot 2 i of range i holds the block the range starts inside (or with), 2 i + 1 any later
// one.  A query block of tiles [s, e) in ranges of `per`: parts s / per .. (e - 1) / per, one of them: it was stored whole.
__device__ __forceinline__ int64_t balance_slot(int64_t range, int64_t s, int per) { return 2 * range + (s > range * per ? 1 : 0); }

// y rows of the query blocks that several ranges share: one thread per four columns of a row, blocks of 256 threads, blockIdx.x over the
// block's rows and columns, blockIdx.y over the query blocks, blockIdx.z over the heads.
template <int D, typename OutT>
__global__ __launch_bounds__(256) void sdp_attention_merge_ranges_kernel(const float* __restrict__ partials, OutT* __restrict__ y, int n_q,
                                                                         int queries_per_block, const unsigned long long* __restrict__ map, AttnBalance w)
{
	constexpr int kQuads = D / 4;
	const int q_block = blockIdx.y, head = blockIdx.z;
	const BalanceScan scan(map, w);
	const int64_t s = (int64_t)head * scan.per_head + scan.tiles_before(map, w, q_block);
	const int64_t e = s + balance_tiles(map, w, q_block);
	const int64_t first = s / scan.per, last = (e - 1) / scan.per;
	if (first == last) return;
	const int item = blockIdx.x * 256 + threadIdx.x;
	const int quad = item % kQuads, r = item / kQuads;
	const int q_row = q_block * queries_per_block + r;
	if (q_row >= n_q) return;
	const int64_t rows = (int64_t)queries_per_block * (D + 2);
	const float* base = partials + (int64_t)r * (D + 2);
	float big = -INFINITY;
	for (int64_t i = first; i <= last; ++i) big = fmaxf(big, base[balance_slot(i, s, scan.per) * rows + D]);
	const float safe = big == -INFINITY ? 0.0f : big;
	float sum = 0.0f;
	float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
	for (int64_t i = first; i <= last; ++i)
	{
		const float* p = base + balance_slot(i, s, scan.per) * rows;
		const float weight = fast_exp2(p[D] - safe);
		sum += p[D + 1] * weight;
		acc += *reinterpret_cast<const WsFloat4*>(p + 4 * quad) * weight;
	}
	const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
	store_merged(y + ((int64_t)head * n_q + q_row) * D + 4 * quad, acc * inv);
}

}  // namespace anygpu
