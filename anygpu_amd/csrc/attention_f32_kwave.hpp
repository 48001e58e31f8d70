// Fused attention, float32, for launches with few query blocks: 16 rows per block, tiles of 16 keys shared out among the block's waves
// (attention_f16_kwave.hpp has the manner), products on v_mfma_f32_16x16x4_f32.
//
// What bounds it: that instruction (128 of 32 cycles per tile and wave at head dimension 256), busy 0.28 - 0.45 of the time, and each block's chain of start, tiles and end; every SIMD is in use where the kernels with 64 and 128
// queries per block leave most of them idle and walk their tiles in sequence.  K passes through the wave's LDS tile, which a CU fills four times as fast
// as it fetches rows in operand layout; V comes straight into the registers of its products.  One launch, no workspace, no pass over a mask.
// Measured (us, former kernels -> here): 8 / 4 heads x 150 x 256 27.5 -> 12.9, x 500 36.3 -> 24.6, 16 x 300 x 128 28.1 -> 11.8, 16 x 500 x 64 18.7 -> 11.5; with a mask
// tensor 8 x 80 x 256 22.8 -> 10.7, 8 x 300 x 256 54.6 -> 24.6, 16 x 167 x 128 20.6 -> 8.9, 64 x 300 x 128 60.1 -> 41.9, 16 x 300 x 64 19.9 -> 11.0.
#pragma once

#include "attention_walk.hpp"
#include "attention_split.hpp"
#include "device_utils.hpp"

namespace anygpu {

namespace {

constexpr int kKeyWaveRows = 16;
constexpr int kKeyWaveTile = 16;

// Whether that kernel takes a launch of `heads` x n_q queries, by its blocks of 16 queries, the tiles (of 16 keys) of the longest and what all of them cost: a
// block's start and end are some six tiles.  us, former kernels / here:
//   * Up to a block for each CU the longest one decides: head dimension 256 up to 48 tiles (8 heads x 500 36.3 / 24.6; but 100 x 1000 34.9 / 40.4; with a mask tensor
//     up to 34: 400 57.4 / 31.7, but 600 58.2 / 77.7), 128 up to 80 (16 x 100 x 1000 27.2 / 23.3; but 100 x 3000 45.8 / 59.0; with a mask tensor up to 190: 100 x 3000 73.4 / 63.8),
//     64 up to 190 (16 x 100 x 3000 37.6 / 31.8, with a mask tensor 40.2 / 37.4).
//   * With more, all of them.  256: 8 x 800 47.8 / 36.2, 4 x 8 x 400 56.9 / 45.9, 8 x 1200 70.0 / 72.9.  128: 16 x 800 38.1 / 33.1, 64 x 350 36.4 / 31.1; but 32 x 200 x 1500 47.9 / 55.8; mask
//     tensor 16 x 600 57.4 / 39.2, 64 x 300 60.1 / 41.9; but 64 x 400 56.7 / 67.1.  64: 16 x 800 27.6 / 19.5, 64 x 350 22.4 / 16.9; but 32 x 200 x 1500 30.9 / 31.6; mask tensor
//     32 x 200 x 1500 41.7 / 38.1, 32 x 400 27.1 / 20.8; but 16 x 1000 44.3 / 44.4.
//   * Not at 256 where blocks of 128 queries are many or have few tiles themselves, by estimated times (240 heads x 105 31.5 / 52.6, 80 x 232 x 280 49.5 / 70.2, 32 x 783 window 51 39.8 / 57.0, mask tensor
//     99 x 93 25.5 / 33.7).  The constants are fitted to 1000 launches; of the 780 that the lines above give to this kernel 122 were slower by more than 4 %, 28 of the 630 that are left.
inline bool attention_kwave_wanted_f32(int head_dim, bool mask, int64_t heads, int n_q, int n_k, int causal, int diag, int window, int64_t cus)
{
	const int64_t groups = (n_q + kKeyWaveRows - 1) / kKeyWaveRows, blocks = heads * groups;
	if (blocks > 8 * cus) return false;
	const int64_t t_first = attention_block_tiles(0, n_q, n_k, causal, diag, window, kKeyWaveRows, kKeyWaveTile);
	const int64_t t_last = attention_block_tiles(groups - 1, n_q, n_k, causal, diag, window, kKeyWaveRows, kKeyWaveTile);
	const int64_t longest = std::max(t_first, t_last);
	if (head_dim == 256 && !attention_kwave_ahead(mask ? KeyWaveCost{3.95, 0.81, 2.4, 11.4, 1.2, 4.0} : KeyWaveCost{3.91, 0.71, 7.7, 5.5, 0.0, 13.3}, true, heads, n_q, n_k, causal, diag, window,
	                                              kKeyWaveRows, kKeyWaveTile, cus)) return false;
	if (blocks <= cus) return longest <= (head_dim == 256 ? (mask ? 34 : 48) : head_dim == 128 && !mask ? 80 : 190);
	const int64_t cost = blocks * (t_first + t_last + 12) / 2;          // (tiles grow evenly from the first group to the last, but for a window)
	if (head_dim == 256) return longest <= (mask ? 34 : 60) && cost <= (mask ? 40 : 80) * cus;
	if (head_dim == 128) return cost <= (mask ? 125 : 100) * cus;
	return cost <= (mask ? 180 : 130) * cus;
}

template <int D, int WAVES>
constexpr int kKeyWaveLdsBytes = (WAVES * kKeyWaveTile + kKeyWaveRows) * (D + 8) * 4;

// `walk`: blocks of 16 queries of a head.  MASK: an additive mask tensor instead of the index rules.
template <int D, bool SOFTCAP, bool MASK, int WAVES>
__global__ __launch_bounds__(64 * WAVES, D == 256 ? 2 : D == 128 ? 3 : 4) void sdp_attention_fwd_f32_kwave_kernel(const AttnArgsF32 a, const AttnWalk walk)
{
	constexpr int ROWS = kKeyWaveRows, THREADS = 64 * WAVES, KT = kKeyWaveTile;
	constexpr int kPitch = D + 8, kPitchO = D + 4;       // floats
	constexpr int KS = D / 16, DC = D / 64, VPR = D / 4, VPS = KT * VPR / 64;
	extern __shared__ __align__(16) char lds_raw[];
	__shared__ float row_max[WAVES][ROWS], row_sum[WAVES][ROWS];
	float* const lds_all = reinterpret_cast<float*>(lds_raw);

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 15, g = lane >> 4;
	float* const lds = lds_all + wave * (KT * kPitch);
	int head, group;
	if (!attn_walk_locate(walk, blockIdx.x, head, group)) return;      // the whole block
	const float* qp = a.q + (int64_t)head * a.n_q * D;
	const float* kp = a.k + (int64_t)(head / a.q_per_kv) * a.n_k * D;
	const float* vp = a.v + (int64_t)(head / a.q_per_kv) * a.n_k * D;
	float* yp = a.y + (int64_t)head * a.n_q * D;

	// the visible keys of the block: of its first and last query
	const int row0 = ROWS * group, q_last = row0 + ROWS < a.n_q ? row0 + ROWS - 1 : a.n_q - 1;
	int key_hi = a.n_k - 1;
	if (a.causal && q_last + a.diag < key_hi) key_hi = q_last + a.diag;
	int key_lo = 0;
	if (a.window > 0 && row0 + a.diag - a.window + 1 > 0) key_lo = row0 + a.diag - a.window + 1;
	const int u_first = key_lo / KT, u_last = key_hi >= 0 ? key_hi / KT : -1;

	// K passes through LDS (1 KB of consecutive memory per load), V is fetched as it is needed: four columns of four rows per lane, 256
	// consecutive bytes for sixteen lanes.  Rows past the last key come out as zeros (their scores are masked, their p is 0): for a buffer without
	// a stride the range check counts the scalar offset as well.  (All of it in the lane's offset takes 15 registers more at head dimension 256, 8 heads x 650 30.4 -> 31.5 us.)
	float4_t kr[VPS], vr[4][DC];
	const auto rsrc_of = [&](const float* src, int u) {
		const int keys = a.n_k - KT * u;
		return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src) + (int64_t)u * (KT * D), 0, (keys < KT ? keys : KT) * (4 * D), 0x00020000);
	};
	auto fetch_k = [&](int u) {
		const auto rsrc = rsrc_of(kp, u);
#pragma unroll
		for (int i = 0; i < VPS; ++i) kr[i] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane * 16, i * 1024, 0));
	};
	auto fetch_v = [&](int u) {
		const auto rsrc = rsrc_of(vp, u);
#pragma unroll
		for (int r = 0; r < 4; ++r)
#pragma unroll
			for (int c = 0; c < DC; ++c)
				vr[r][c] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, g * (16 * D) + n * 16, r * (4 * D) + c * 256, 0));
	};
	const int q_idx = row0 + n;
	// MASK: the values of this lane's scores of a tile, four consecutive floats at any alignment; in the last tile keys past the end read
	// nothing (their scores are masked)
	float4_t mk = {0.0f, 0.0f, 0.0f, 0.0f};
	const float* const mask_row = MASK ? a.mask + (int64_t)(q_idx < a.n_q ? q_idx : a.n_q - 1) * a.mask_stride : nullptr;
	auto fetch_mask = [&](int u) {
		typedef float4_t LooseF4 __attribute__((aligned(4)));
		const int key = KT * u + 4 * g;
		if ((u + 1) * KT <= a.n_k) mk = *reinterpret_cast<const LooseF4*>(mask_row + key);
		else
		{
#pragma unroll
			for (int r = 0; r < 4; ++r) mk[r] = key + r < a.n_k ? mask_row[key + r] : -INFINITY;
		}
	};
	// the tile is this wave's alone: what it wrote is there, or what it reads has been read, once its counter says so
	auto wait_lds = [&]() {
		__builtin_amdgcn_s_waitcnt(0xC07F);               // lgkmcnt(0)
		__builtin_amdgcn_wave_barrier();
	};
	// the rows, once for all waves (padding rows repeat the last one)
	float* const q_lds = lds_all + WAVES * (KT * kPitch);
	constexpr int kQVecs = (ROWS * VPR + THREADS - 1) / THREADS;
	float4_t q_vec[kQVecs];
#pragma unroll
	for (int i = 0; i < kQVecs; ++i)
	{
		const int idx = tid + THREADS * i;
		if (idx < ROWS * VPR) q_vec[i] = *reinterpret_cast<const float4_t*>(qp + (int64_t)min(row0 + idx / VPR, a.n_q - 1) * D + (idx % VPR) * 4);
	}
	__builtin_amdgcn_sched_barrier(0);
	int u = u_first + wave;
	if (u <= u_last)
	{
		fetch_k(u);
		if constexpr (MASK) fetch_mask(u);
		fetch_v(u);
	}
#pragma unroll
	for (int i = 0; i < kQVecs; ++i)
	{
		const int idx = tid + THREADS * i;
		if (idx < ROWS * VPR) *reinterpret_cast<float4_t*>(q_lds + (idx / VPR) * kPitch + (idx % VPR) * 4) = q_vec[i];
	}
	const int vis_hi = a.causal && q_idx + a.diag < a.n_k - 1 ? q_idx + a.diag : a.n_k - 1;
	const int vis_lo = a.window > 0 ? q_idx + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;                // l_run: this lane's share of the row sum
	float4_t o[DC][4];
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int e = 0; e < 4; ++e) o[c][e] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
	__syncthreads();
	for (; u <= u_last; u += WAVES)
	{
		const bool more = u + WAVES <= u_last;
#pragma unroll
		for (int i = 0; i < VPS; ++i)
		{
			const int idx = lane + 64 * i;
			*reinterpret_cast<float4_t*>(lds + (idx / VPR) * kPitch + (idx % VPR) * 4) = kr[i];
		}
		const float4_t mask_now = mk;
		// a tile that the mask hides from every query of the block (-inf, or the lowest float, which is -inf as a logit) takes no part, whatever its
		// keys and values hold
		bool visible = true;
		if constexpr (MASK)
		{
			bool any = false;
#pragma unroll
			for (int r = 0; r < 4; ++r) any |= mask_now[r] * kLog2e > -INFINITY;
			visible = __builtin_amdgcn_ballot_w64(any) != 0;
		}
		if (more)
		{
			fetch_k(u + WAVES);
			if constexpr (MASK) fetch_mask(u + WAVES);
		}
		wait_lds();
		// ---- S^T = K Q^T: even and odd elements in sums of their own ----
		float4_t s[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
		if (visible)
		{
#pragma unroll
			for (int st = 0; st < KS; ++st)
			{
				const float4_t kf = *reinterpret_cast<const float4_t*>(lds + n * kPitch + 16 * st + 4 * g);
				const float4_t qf = *reinterpret_cast<const float4_t*>(q_lds + n * kPitch + 16 * st + 4 * g);
#pragma unroll
				for (int e = 0; e < 4; ++e) s[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[e], s[e & 1], 0, 0, 0);
			}
			wait_lds();

			// ---- online softmax ----
			float z[4];
			float mt = -INFINITY;
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const int key = KT * u + 4 * g + r;
				const float zz = logit2<SOFTCAP>(s[0][r] + s[1][r], a.k_in, a.k_cap) + (MASK ? mask_now[r] * kLog2e : 0.0f);
				z[r] = (key >= vis_lo && key <= vis_hi) ? zz : -INFINITY;
				mt = fmaxf(mt, z[r]);
			}
			mt = max_over_lane_rows(mt);
			const float m_new = fmaxf(m_run, mt);
			const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;
			if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0)
			{
				const float corr = fast_exp2(m_run - m_safe);
				l_run *= corr;
#pragma unroll
				for (int c = 0; c < DC; ++c)
#pragma unroll
					for (int e = 0; e < 4; ++e) o[c][e] *= corr;
			}
			m_run = m_new;
			float p[4];
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				p[r] = fast_exp2(z[r] - m_safe);
				l_run += p[r];
			}

			// ---- O^T += V^T P^T ----
#pragma unroll
			for (int r = 0; r < 4; ++r)
#pragma unroll
				for (int c = 0; c < DC; ++c)
#pragma unroll
					for (int e = 0; e < 4; ++e) o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[r][c][e], p[r], o[c][e], 0, 0, 0);
		}
		if (more) fetch_v(u + WAVES);
	}

	// ---- the waves' results through LDS: register r of accumulator (c, e) is o[row n][64 c + 16 g + 4 r + e] ----
	const int waves = min(WAVES, max(u_last - u_first + 1, 1));      // those that had a tile
	float l = l_run;
	l += __shfl_xor(l, 16);
	l += __shfl_xor(l, 32);
	if (wave < waves)
	{
		float* const mine = lds + n * kPitchO + 16 * g;
#pragma unroll
		for (int c = 0; c < DC; ++c)
#pragma unroll
			for (int r = 0; r < 4; ++r) *reinterpret_cast<float4_t*>(mine + 64 * c + 4 * r) = float4_t{o[c][0][r], o[c][1][r], o[c][2][r], o[c][3][r]};
		if (g == 0)
		{
			row_max[wave][n] = m_run;
			row_sum[wave][n] = l;
		}
	}
	__syncthreads();
#pragma unroll
	for (int i = tid; i < ROWS * VPR; i += THREADS)
	{
		const int r = i / VPR, quad = i % VPR;
		if (row0 + r >= a.n_q) continue;
		float big = row_max[0][r];
		for (int w = 1; w < waves; ++w) big = fmaxf(big, row_max[w][r]);
		const float safe = big == -INFINITY ? 0.0f : big;
		float sum = 0.0f;
		float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
		for (int w = 0; w < waves; ++w)
		{
			const float weight = fast_exp2(row_max[w][r] - safe);
			sum += row_sum[w][r] * weight;
			acc += *reinterpret_cast<const float4_t*>(lds_all + w * (KT * kPitch) + r * kPitchO + 4 * quad) * weight;
		}
		store_merged(yp + (int64_t)(row0 + r) * D + 4 * quad, acc * (sum > 0.0f ? 1.0f / sum : 0.0f));
	}
}

}  // namespace

}  // namespace anygpu
