// Fused attention, fp16, index rules, for launches with few query blocks: 16 rows per block, the key tiles shared out among the block's waves.
//
// The kernels with 128 queries per block leave most CUs idle on a prompt of a few hundred tokens, and the block that has the most keys walks them alone
// (8 heads x 394 x 256: 32 blocks, seven tiles of 64 keys at 2.7 us each).  Here every 16 rows are a block, and its four or eight waves take tiles of 32 keys in turn,
// each with its own running maximum, without a barrier; their results meet in LDS.  One launch, no workspace.
// What bounds it: a block's chain of queries, first tile, some tiles per wave and the meeting of the waves (matrix cores busy 3 - 6 %, 9 - 14 bytes fetched per clock and CU over the launch), and in
// it the rate at which a CU fetches, since every 16 rows read their keys again.  Rows of K and of the queries fetched straight in operand
// layout (16 rows x 64 bytes an instruction) come at 16 bytes per clock and CU, 1 KB of consecutive memory at 55 - 60 (all CUs at once, out of the L2s), so
// K passes through LDS like V, through the same wave-private tile, and the queries are fetched once per block (8 heads x 394 x 256 14.9 us with both
// in operand layout, 11.5 now).  A tile of K and V is requested while the one before is used.  Eight waves hide the latency where blocks are at most one to a CU; with more of
// them, four, of which two to three blocks fit a CU (64 / 8 heads x 163 x 746 x 128 22.5 us with eight, 17.1 with four).  Not kept: 32 rows per block (two
// groups of 16 per wave), which halves what is fetched but needs the chip full of blocks, where the 128-query kernels are better.
// Measured (us, kernels of 128 queries per block -> here): 8 / 4 heads x 96 x 256 10.9 -> 6.0, x 394 20.2 -> 11.4, x 700 26.2 -> 16.7; 16 x 200 x 128 8.7 -> 5.6, 16 x 163 x 746 x 128
// 15.1 -> 8.9, 16 x 500 x 64 12.0 -> 6.4, 32 x 250 x 1000 x 64 15.3 -> 9.5.
#pragma once

#include "attention_walk.hpp"
#include "attention_split.hpp"
#include "device_utils.hpp"

namespace anygpu {

namespace {

constexpr int kKeyWaveRows = 16;
constexpr int kKeyWaveTile = 32;                // keys of a tile: one MFMA step of the second product
// p is 2^15 for a score at the running maximum (attention_f16_q32.hpp)
constexpr float kKeyWaveHeadRoom = 15.0f;

// Whether that kernel takes a launch of `heads` x n_q queries, by its blocks of 16 queries, the tiles of the longest (t_last) and what all of them cost: a
// block's start and end are some five tiles.  us, 128 queries per block / here:
//   * Up to a block for each CU the longest one decides: head dimension 256 up to 48 tiles (8 heads x 100 x 1400 23.3 / 20.8; but 100 x 2000 24.3 / 27.7), 128 up to 100 (16 x
//     250 x 3000 27.4 / 21.2, 16 x 100 x 2500 21.3 / 18.0; but 16 x 100 x 5000 28.0 / 30.7), 64 up to 200 (16 x 100 x 5000 24.3 / 18.6).
//   * With more, what they fetch.  256, up to two and a quarter blocks for each CU: 8 x 700 26.2 / 16.7, 4 x 8 x 250 17.5 / 13.6, 8 x 1100 30.3 / 29.3; but 4 x 8 x
//     300 17.5 / 19.5, 8 x 949 without the causal rule 29.7 / 33.3.  128, up to three: 32 x 300 10.0 / 8.5, 32 x 250 x 1000 20.5 / 16.6, 64 x 160 7.7 / 7.2; but 64 x 200
//     9.0 / 9.5, 32 x 400 x 1000 23.8 / 26.0; up to four where the kernels of 128 queries would have half a block for each CU, which they cut into parts: 16 x 800 21.8 / 14.5, 16 x
//     1000 24.5 / 21.9.  64, up to four: 32 x 500 14.1 / 7.5, 64 x 250 7.3 / 5.9, 16 x 1000 without the causal rule 21.9 / 16.9; but 64 x 300 7.4 / 8.7.
//   * A mask tensor, whose hidden tiles are not known ahead: 8 x 400 x 256 24.8 / 12.6, 200 x 1500 25.9 / 24.1 (but 600 26.8 / 26.3, 100 x 3000 28.2 / 40.1), 16 x 600 x 128 21.2 / 16.9,
//     64 x 167 11.4 / 9.6 (but 32 x 422 17.1 / 18.4, 64 x 300 14.3 / 18.0, 64 x 200 x 1500 39.8 / 41.8), 16 x 1000 x 64 22.4 / 18.7, 32 x 100 x 3000 25.1 / 15.7 (but 32 x 1000 28.8 / 32.8).
//   * Not where blocks of 128 queries are many or have few tiles themselves: at 64 and 128 with a single tile of 64 keys (84 heads x 29 x 64 4.0 / 4.5, 7 x 4 x 34 x 128 4.7 / 5.2), at 256, and at 128
//     by a little, where estimated times say so (176 heads x 34 x 256 6.7 / 12.5, 10 x 8 x 81 x 242 x 256 14.7 / 25.9, 20 x 4 x 75 x 256 10.8 / 14.0, mask tensor 64 x 153 x 256 15.6 / 20.5, 31 x 8 x 68 x 128
//     6.5 / 8.1).  The constants are fitted to 2800 launches of 16 to 1600 queries; of the 1860 that the lines above give to this kernel 350 were slower by more than 4 %, 27 of the 1390 that are left.
inline bool attention_kwave_wanted(int head_dim, bool mask, int64_t heads, int n_q, int n_k, int causal, int diag, int window, int64_t cus)
{
	const int64_t groups = (n_q + kKeyWaveRows - 1) / kKeyWaveRows, blocks = heads * groups;
	if (blocks > 4 * cus) return false;
	const int64_t t_first = attention_block_tiles(0, n_q, n_k, causal, diag, window, kKeyWaveRows, kKeyWaveTile);
	const int64_t t_last = attention_block_tiles(groups - 1, n_q, n_k, causal, diag, window, kKeyWaveRows, kKeyWaveTile);
	const int64_t longest = std::max(t_first, t_last), q_blocks = (n_q + 127) / 128;
	if (!mask && head_dim != 256 && attention_block_tiles(0, n_q, n_k, causal, diag, window, 128, 64) <= 1 && attention_block_tiles(q_blocks - 1, n_q, n_k, causal, diag, window, 128, 64) <= 1) return false;
	if (head_dim == 256 || (head_dim == 128 && !mask))
	{
		const KeyWaveCost cost = head_dim == 128 ? KeyWaveCost{0.53, 0.21, 0.0, 1.38, 0.0, 1.65} : mask ? KeyWaveCost{3.13, 0.58, 2.2, 2.35, 0.85, 4.5} : KeyWaveCost{2.39, 0.59, 1.0, 2.46, 0.1, 4.2};
		if (!attention_kwave_ahead(cost, head_dim == 256, heads, n_q, n_k, causal, diag, window, kKeyWaveRows, kKeyWaveTile, cus)) return false;
	}
	if (blocks <= cus) return longest <= (head_dim == 256 ? 48 : head_dim == 128 ? 100 : 200);
	const int64_t cost = blocks * (t_first + t_last + 10) / 2;          // (tiles grow evenly from the first group to the last, but for a window)
	if (mask) return blocks <= (head_dim == 64 ? 4 : 3) * cus && cost <= (head_dim == 256 ? 26 : head_dim == 128 ? 110 : 200) * cus;
	if (head_dim == 256) return 4 * blocks <= 9 * cus && longest <= 48 && cost <= 56 * cus;
	if (head_dim == 128) return (blocks <= 3 * cus && cost <= 75 * cus) || (2 * heads * q_blocks <= cus && cost <= 90 * cus);
	return cost <= 160 * cus;
}

// Whether it takes a generation step of `blocks` groups of 16 rows that see `tiles` tiles (32 keys), which then needs no merge launch (us, split keys and merge /
// here): head dimension 64 up to 34 tiles (32 heads x 256 7.4 / 5.3, 4 x 32 x 2 queries x 1000 10.3 / 7.4, 32 x 1000 7.4 / 6.9; but 1500 7.8 / 8.4), 128 up to 20 (32 / 8 x 300
// 8.0 / 6.2, 600 8.2 / 7.6; but 1000 8.2 / 9.9), 256 up to 10 (8 / 4 x 256 9.8 / 8.3, x 300 10.3 / 9.2; but 400 10.1 / 10.4).
inline bool decode_kwave_wanted(int64_t head_dim, int64_t blocks, int64_t tiles, int64_t cus)
{
	return blocks <= cus && tiles <= (head_dim == 256 ? 10 : head_dim == 128 ? 20 : 34);
}

template <int D, int WAVES>
constexpr int kKeyWaveLdsBytes = (WAVES * kKeyWaveTile + kKeyWaveRows) * AttnLds<D>::kPitchV;

// `walk`: blocks of 16 rows of a "head" of `rows` rows; row r is query r % n_q (rows = n_q, or where the query heads of a key / value head are
// taken together, q_per_kv * n_q, at most kDecodeMaxRows).  MASK: an additive mask tensor instead of the index rules.
template <int D, bool SOFTCAP, bool MASK, int WAVES>
__global__ __launch_bounds__(64 * WAVES, D == 256 ? 2 : D == 128 ? 3 : 4) void sdp_attention_fwd_f16_kwave_kernel(const AttnArgs a, const AttnWalk walk, int rows)
{
	constexpr int ROWS = kKeyWaveRows, THREADS = 64 * WAVES;
	constexpr int kPitchV = AttnLds<D>::kPitchV;
	constexpr int KS = D / 32, DC = D / 16, VPR = D / 8, VPS = kKeyWaveTile * VPR / 64;
	constexpr int kPitchO = D + 4;              // floats of a row of the waves' results, where their V tiles were
	static_assert(16 * kPitchO * 4 <= kKeyWaveTile * kPitchV, "a wave's result fits its V tile");
	extern __shared__ __align__(16) char lds_all[];
	__shared__ float row_max[WAVES][ROWS], row_sum[WAVES][ROWS];

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 15, g = lane >> 4;
	char* const lds = lds_all + wave * (kKeyWaveTile * kPitchV);
	int head, group;
	if (!attn_walk_locate(walk, blockIdx.x, head, group)) return;      // the whole block
	const half_t* qp = a.q + (int64_t)head * rows * D;
	const half_t* kp = a.k + (int64_t)(head / walk.q_per_kv) * a.n_k * D;
	const half_t* vp = a.v + (int64_t)(head / walk.q_per_kv) * a.n_k * D;
	half_t* yp = a.y + (int64_t)head * rows * D;

	const int row0 = ROWS * group;
	// the visible keys of the block: of its first and last query, or of all queries where rows of several heads are together
	const bool one_head = rows == a.n_q;
	const int q_first = one_head ? row0 : 0, q_last = one_head && row0 + ROWS < a.n_q ? row0 + ROWS - 1 : a.n_q - 1;
	int key_hi = a.n_k - 1;
	if (a.causal && q_last + a.diag < key_hi) key_hi = q_last + a.diag;
	int key_lo = 0;
	if (a.window > 0 && q_first + a.diag - a.window + 1 > 0) key_lo = q_first + a.diag - a.window + 1;
	const int u_first = key_lo / kKeyWaveTile, u_last = key_hi >= 0 ? key_hi / kKeyWaveTile : -1;

	float4_t kr[VPS], vr[VPS];
	// a tile of K or V as it lies, 1 KB of consecutive memory per load (in operand layout, 16 rows x 64 bytes, a CU fetches a quarter of that
	// rate: 16 bytes per clock); rows past the last key come out as zeros (their scores are masked, their p is 0): for a buffer without a
	// stride the range check counts the scalar offset as well (a lane's offset against the buffer's bytes less the scalar one)
	auto fetch = [&](float4_t (&dst)[VPS], const half_t* src, int u) {
		const int keys = a.n_k - kKeyWaveTile * u;
		const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(src) + (int64_t)u * (kKeyWaveTile * D), 0, (keys < kKeyWaveTile ? keys : kKeyWaveTile) * (2 * D), 0x00020000);
#pragma unroll
		for (int i = 0; i < VPS; ++i) dst[i] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane * 16, i * 1024, 0));
	};
	auto put = [&](const float4_t (&src)[VPS]) {
#pragma unroll
		for (int i = 0; i < VPS; ++i)
		{
			const int idx = lane + 64 * i;
			*reinterpret_cast<float4_t*>(lds + (idx / VPR) * kPitchV + (idx % VPR) * 16) = src[i];
		}
	};
	const int q_idx = one_head ? row0 + n : (row0 + n) % a.n_q;
	// MASK: the values of this lane's scores of a tile, four consecutive halves of each half tile at any alignment; in the last tile keys
	// past the end read nothing (their scores are masked)
	half4_t mk[2] = {};
	const half_t* const mask_row = MASK ? a.mask + (int64_t)(q_idx < a.n_q ? q_idx : a.n_q - 1) * a.mask_stride : nullptr;
	auto fetch_mask = [&](int u) {
		typedef half4_t LooseHalf4 __attribute__((aligned(2)));
		const int key = kKeyWaveTile * u + 4 * g;
#pragma unroll
		for (int kb = 0; kb < 2; ++kb)
		{
			if ((u + 1) * kKeyWaveTile <= a.n_k) mk[kb] = *reinterpret_cast<const LooseHalf4*>(mask_row + key + 16 * kb);
			else
			{
#pragma unroll
				for (int r = 0; r < 4; ++r) mk[kb][r] = key + 16 * kb + r < a.n_k ? mask_row[key + 16 * kb + r] : (half_t)-INFINITY;
			}
		}
	};
	// the tile is this wave's alone: what it wrote is there, or what it reads has been read, once its counter says so
	auto wait_lds = [&]() {
		__builtin_amdgcn_s_waitcnt(0xC07F);               // lgkmcnt(0)
		__builtin_amdgcn_wave_barrier();
	};
	// the rows, once for all waves (padding rows repeat the last one)
	char* const q_lds = lds_all + WAVES * (kKeyWaveTile * kPitchV);
	constexpr int kQVecs = (ROWS * VPR + THREADS - 1) / THREADS;
	float4_t q_vec[kQVecs];
#pragma unroll
	for (int i = 0; i < kQVecs; ++i)
	{
		const int idx = tid + THREADS * i;
		if (idx < ROWS * VPR) q_vec[i] = *reinterpret_cast<const float4_t*>(qp + (int64_t)min(row0 + idx / VPR, rows - 1) * D + (idx % VPR) * 8);
	}
	__builtin_amdgcn_sched_barrier(0);
	int u = u_first + wave;
	if (u <= u_last)
	{
		fetch(kr, kp, u);
		if constexpr (MASK) fetch_mask(u);
		fetch(vr, vp, u);
	}
#pragma unroll
	for (int i = 0; i < kQVecs; ++i)
	{
		const int idx = tid + THREADS * i;
		if (idx < ROWS * VPR) *reinterpret_cast<float4_t*>(q_lds + (idx / VPR) * kPitchV + (idx % VPR) * 16) = q_vec[i];
	}
	const int vis_hi = a.causal && q_idx + a.diag < a.n_k - 1 ? q_idx + a.diag : a.n_k - 1;
	const int vis_lo = a.window > 0 ? q_idx + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;                // l_run: this lane's share of the row sum
	float4_t o[DC];
#pragma unroll
	for (int c = 0; c < DC; ++c) o[c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
	__syncthreads();
	for (; u <= u_last; u += WAVES)
	{
		const bool more = u + WAVES <= u_last;
		put(kr);
		const half4_t mask_now[2] = {mk[0], mk[1]};
		// a tile that the mask hides from every query of the block takes no part, whatever its keys and values hold
		bool visible = true;
		if constexpr (MASK)
		{
			bool any = false;
#pragma unroll
			for (int kb = 0; kb < 2; ++kb)
#pragma unroll
				for (int r = 0; r < 4; ++r) any |= mask_now[kb][r] > (half_t)(-INFINITY);
			visible = __builtin_amdgcn_ballot_w64(any) != 0;
		}
		if (more)
		{
			fetch(kr, kp, u + WAVES);
			if constexpr (MASK) fetch_mask(u + WAVES);
		}
		wait_lds();
		// ---- S^T = K Q^T ----
		float4_t s[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
		if (visible)
		{
#pragma unroll
			for (int st = 0; st < KS; ++st)
			{
				const half8_t qf = *reinterpret_cast<const half8_t*>(q_lds + n * kPitchV + (32 * st + 8 * g) * 2);
#pragma unroll
				for (int kb = 0; kb < 2; ++kb)
				{
					const half8_t kf = *reinterpret_cast<const half8_t*>(lds + (16 * kb + n) * kPitchV + (32 * st + 8 * g) * 2);
					s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf, s[kb], 0, 0, 0);
				}
			}
		}
		wait_lds();
		put(vr);
		if (more) fetch(vr, vp, u + WAVES);
		if (!visible) continue;

		// ---- online softmax ----
		float z[2][4];
		float mt = -INFINITY;
#pragma unroll
		for (int kb = 0; kb < 2; ++kb)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const int key = kKeyWaveTile * u + 16 * kb + 4 * g + r;
				const float zz = logit2<SOFTCAP>(s[kb][r], a.k_in, a.k_cap) + (MASK ? (float)mask_now[kb][r] * kLog2e : 0.0f);
				z[kb][r] = (key >= vis_lo && key <= vis_hi) ? zz : -INFINITY;
				mt = fmaxf(mt, z[kb][r]);
			}
		mt = max_over_lane_rows(mt);
		const float m_new = fmaxf(m_run, mt);
		const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;
		if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0)
		{
			const float corr = fast_exp2(m_run - m_safe);
			l_run *= corr;
#pragma unroll
			for (int c = 0; c < DC; ++c) o[c] *= corr;
		}
		m_run = m_new;
		half8_t pf;
#pragma unroll
		for (int kb = 0; kb < 2; ++kb)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const float p = fast_exp2((z[kb][r] - m_safe) + kKeyWaveHeadRoom);
				l_run += p;
				pf[4 * kb + r] = (half_t)p;
			}

		// ---- O^T += V^T P^T ----
		wait_lds();
#pragma unroll
		for (int c = 0; c < DC; ++c)
		{
			const char* src = lds + (4 * g + (n >> 2)) * kPitchV + (16 * c + 4 * (n & 3)) * 2;
			const half4_t lo = lds_read_tr_b64(src);
			const half4_t hi = lds_read_tr_b64(src + 16 * kPitchV);
			const half8_t vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
			o[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf, o[c], 0, 0, 0);
		}
		wait_lds();
	}

	// ---- the waves' results through LDS: lane (n, g) holds o[row n][16 c + 4 g .. + 3] ----
	const int waves = min(WAVES, max(u_last - u_first + 1, 1));      // those that had a tile
	float l = l_run;
	l += __shfl_xor(l, 16);
	l += __shfl_xor(l, 32);
	if (wave < waves)
	{
		float* const mine = reinterpret_cast<float*>(lds) + n * kPitchO + 4 * g;
#pragma unroll
		for (int c = 0; c < DC; ++c) *reinterpret_cast<float4_t*>(mine + 16 * c) = o[c];
		if (g == 0)
		{
			row_max[wave][n] = m_run;
			row_sum[wave][n] = l;
		}
	}
	__syncthreads();
	constexpr int kQuads = D / 4;
#pragma unroll
	for (int i = tid; i < ROWS * kQuads; i += THREADS)
	{
		const int r = i / kQuads, quad = i % kQuads;
		if (row0 + r >= rows) continue;
		float big = row_max[0][r];
		for (int w = 1; w < waves; ++w) big = fmaxf(big, row_max[w][r]);
		const float safe = big == -INFINITY ? 0.0f : big;
		float sum = 0.0f;
		float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
		for (int w = 0; w < waves; ++w)
		{
			const float weight = fast_exp2(row_max[w][r] - safe);
			sum += row_sum[w][r] * weight;
			acc += *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(lds_all + w * (kKeyWaveTile * kPitchV)) + r * kPitchO + 4 * quad) * weight;
		}
		store_merged(yp + (int64_t)(row0 + r) * D + 4 * quad, acc * (sum > 0.0f ? 1.0f / sum : 0.0f));
	}
}

}  // namespace

}  // namespace anygpu
