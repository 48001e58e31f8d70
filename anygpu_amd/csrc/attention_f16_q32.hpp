// Fused attention, fp16, head dimensions 64 and 128: 32 queries per wave.
//
// What bounds it.  Per tile of 64 keys a wave of 32 queries has 1024 (head dimension 64: 512) cycles of MFMAs, some 700 of vector
// instructions (22 clocks a score with two waves on a SIMD) and 32 (16) KB of fragments to read out of LDS.  With v_mfma_f32_32x32x16_f16 every
// fragment feeds 32 x 32 scores, so the LDS stays below half of its rate.  A block is FOUR waves with 128 queries, and two blocks (head dimension 64:
// three) share a CU without a barrier between them.  Scores sit 32 to a lane (S^T = K Q^T: a lane holds one query), so row maxima are in-lane
// but for one exchange of lane halves.  The two halves of a tile's work come from DIFFERENT tiles, so that a wave has vector instructions to issue
// behind every MFMA (a wave of such a mix and another like it on its SIMD keep the matrix cores busy, 33.7 clocks per MFMA of 32, where products and
// softmax in turn took 66): S(t + 1) = K(t + 1) Q^T beside p(t) = 2^(z(t) - m), then O^T += V(t)^T P(t)^T beside the rest of p(t) and the maximum of
// S(t + 1).  What is left is the power the part may draw: 16 heads x 8192 x 128 without the causal rule 548 us on operands of N(0, 1) and 345 (1.6
// PFLOP/s) on zeros, where the form with products and softmax in turn took 571 and 407; eight waves and 256 queries to a block, half of the tile
// loads, measured 540 there and up to a quarter slower where blocks are few.
// Sums are those of the fp32 p, and the maximum is exact in every tile, so that the largest p is
// a power of two, which rounds to a half without an error (a maximum that lags until it is outgrown by 2^8 and sums of the
// rounded p by v_dot2 measured 5 % faster, but up to a tenth further from 64-bit results: 16 heads x 4096 x 128, q of
// N(0, 4): 2.36e-4 against 2.17e-4 (2-norm), of which the result's own rounding is 2.1e-4).
// Measured, causal (us; products and softmax in turn -> here, the same bits): 16 x 4096 x 128 102.3 -> 91.7, 64 / 8 x 1000 x 128 32.0 -> 29.9, 16 x 8192 x
// 128 315 -> 299, 2 x 16 x 2280 x 128 63.3 -> 58.7, 32 / 8 x 3000 x 128 93.3 -> 91.4, 4096 166 -> 153, 32 x 2038 x 64 36.5 -> 32.8, 32 x 4000 x 64 window 500
// 36.9 -> 34.5; without the causal rule 32 / 8 x 3000 x 128 177 -> 159.  Blocks of some three tiles and fewer paid for its longer
// code (4 x 64 / 8 x 200 x 128 12.2 -> 13.7): they take products and softmax in turn (attention_q32_in_turn), with the same bits.
#pragma once

#include "attention_walk.hpp"
#include "attention_split.hpp"
#include "device_utils.hpp"

namespace anygpu {

namespace {

constexpr int kQ32Waves = 4;
constexpr int kQ32QueriesPerBlock = 32 * kQ32Waves;
// p, which the second product takes as halves, is 2^15 for a score at the running maximum: with all of the halves' exponents
// below it, p is a normal half (11 bits) down to 2^-29 of the maximum instead of 2^-14.  The factor is in the sums and the accumulators
// alike, also in those that pass through the workspace, and cancels.
constexpr float kQ32HeadRoom = 15.0f;

// Chunk (16 bytes) of row r that the tile keeps at position c is c ^ swizzle(r): the tile rows are 2 D bytes without padding,
// filled by direct loads whose lanes land on consecutive 16 bytes.  Both read patterns are free of bank conflicts with it
// (SQ_LDS_BANK_CONFLICT 0).
template <int D>
__device__ __forceinline__ constexpr int q32_k_swizzle(int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); }
template <int D>
__device__ __forceinline__ constexpr int q32_v_swizzle(int r) { return D == 128 ? (((r & 3) << 2) | (r & 2)) : ((r & 3) << 1); }

// Maximum of the two halves of a wave, lane by lane (v_permlane32_swap of two copies returns {lower, lower} and {upper, upper}).
__device__ __forceinline__ float max_over_lane_halves(float x)
{
	float a = x, b = x;
	asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
	return fmaxf(a, b);
}

// IN_TURN: the products and the softmax of a tile one after the other, for blocks of few tiles
template <int D, bool SOFTCAP, bool IN_TURN>
__global__ __launch_bounds__(64 * kQ32Waves, D == 64 && !IN_TURN ? 3 : 2) void sdp_attention_fwd_f16_q32_kernel(const AttnArgs a, const AttnWalk walk)
{
	constexpr int kRow = 2 * D;                              // bytes of a tile row
	constexpr int KT = kAttnKeysPerTile, KB = KT / 32;
	constexpr int kTile = KT * kRow;                         // bytes of a K or V tile
	constexpr int kStage = 2 * kTile;
	constexpr int KS = D / 16;                               // MFMA steps along the head dimension
	constexpr int DC = D / 32;                               // 32-wide column blocks of the output
	constexpr int kSlots = kTile / 1024 / kQ32Waves;         // direct loads of a tile per wave
	constexpr int kChunks = kRow / 16, kRowsPerLoad = 1024 / kRow;
	constexpr int kAhead = 4;                                // steps that a fragment is read ahead
	constexpr int kLoadSpacing = D == 128 ? 4 : 2;           // steps from one load of the next tiles to the next
	extern __shared__ __align__(16) char lds[];

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 31;                                 // query of the wave (second MFMA operand index)
	const int h = lane >> 5;                                 // lane half: k slots 8 h .. 8 h + 7 of an MFMA
	int bh, q_block, part, parts, split_slot;
	if (!attn_walk_locate_part(walk, blockIdx.x, bh, q_block, part, parts, split_slot)) return;
	const int q0 = q_block * kQ32QueriesPerBlock;
	const half_t* qp = a.q + (int64_t)bh * a.n_q * D;
	const half_t* kp = a.k + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	const half_t* vp = a.v + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	half_t* yp = a.y + (int64_t)bh * a.n_q * D;

	const int q_last = (q0 + kQ32QueriesPerBlock - 1 < a.n_q ? q0 + kQ32QueriesPerBlock - 1 : a.n_q - 1);
	int key_hi = a.n_k - 1;
	if (a.causal && q_last + a.diag < key_hi) key_hi = q_last + a.diag;
	int key_lo = 0;
	if (a.window > 0 && q0 + a.diag - a.window + 1 > 0) key_lo = q0 + a.diag - a.window + 1;
	int t_first = key_lo / KT;
	int t_last = key_hi >= 0 ? key_hi / KT : -1;
	if (parts > 1)
	{
		const int per = (t_last - t_first + parts) / parts;
		t_first += part * per;
		if (t_first + per - 1 < t_last) t_last = t_first + per - 1;
	}

	// A SIMD issues from the older of its two waves while that one can: blocks behind the first two rounds go first instead, whose partner is nearer to its end (us, causal: 32 /
	// 8 heads x 3000 x 128 91.2 -> 90.1, 3200 100.3 -> 98.4, window 1024 60.6 -> 58.7, 128 / 8 x 579 27.8 -> 26.9; three blocks on a CU, head dimension 64, are slower with it: 32 / 8 x 3000 55.0 / 57.9).
	if (D == 128 && walk.turn > 0 && (int)blockIdx.x >= 2 * kAttnXcds * walk.turn) __builtin_amdgcn_s_setprio(1);

	// this wave's queries as second operands: lane (n, h) holds q[row][16 s + 8 h .. + 7]
	const int wq0 = q0 + 32 * wave;
	const int q_row = wq0 + n;
	half8_t qf[KS];
	const float k_in = fabsf(a.k_in);
#pragma unroll
	for (int s = 0; s < KS; ++s)
	{
		half8_t val = {};
		if (q_row < a.n_q) val = *reinterpret_cast<const half8_t*>(qp + (int64_t)q_row * D + 16 * s + 8 * h);
		qf[s] = a.k_in < 0.0f ? -val : val;
	}
	int vis_hi = a.causal ? q_row + a.diag : a.n_k - 1;
	if (vis_hi > a.n_k - 1) vis_hi = a.n_k - 1;
	const int vis_lo = a.window > 0 ? q_row + a.diag - a.window + 1 : 0;
	// keys visible to every query of this wave: [all_lo, all_hi]; to any of them: [any_lo, any_hi]
	int any_hi = a.causal ? wq0 + 31 + a.diag : a.n_k - 1;
	if (any_hi > a.n_k - 1) any_hi = a.n_k - 1;
	if (wq0 >= a.n_q) any_hi = -1;
	const int any_lo = a.window > 0 ? wq0 + a.diag - a.window + 1 : 0;
	const int all_hi = a.causal ? (wq0 + a.diag < a.n_k - 1 ? wq0 + a.diag : a.n_k - 1) : a.n_k - 1;
	const int all_lo = a.window > 0 ? wq0 + 31 + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;                   // l_run: this lane's share of the row sum
	float16_t o[DC];
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;

	const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
	// Tiles go global -> LDS without staging registers: load i = wave + 4 j of a tile fills rows i kRowsPerLoad ..; the buffer's
	// range ends with the last key, so the rows behind it come out as zeros.  Written as assembly: the compiler would make
	// LDS reads wait for all outstanding direct loads of the wave.
	const int load_row = kRowsPerLoad * wave + lane / kChunks;
	int load_k[kSlots], load_v[kSlots];
#pragma unroll
	for (int j = 0; j < kSlots; ++j)
	{
		const int row = load_row + kRowsPerLoad * kQ32Waves * j;
		load_k[j] = row * kRow + ((lane % kChunks) ^ q32_k_swizzle<D>(row)) * 16;
		load_v[j] = row * kRow + ((lane % kChunks) ^ q32_v_swizzle<D>(row)) * 16;
	}
	typedef int int4_t __attribute__((ext_vector_type(4)));
	// load j of this wave's share (K: j < kSlots, V behind it) of the tile at `at` into a stage
	auto rsrc_of = [&](const half_t* src, int t) {
		const int bytes = min(KT, a.n_k - t * KT) * kRow;
		const uint64_t at = reinterpret_cast<uint64_t>(src) + (int64_t)t * kTile;
		return int4_t{(int)(uint32_t)at, (int)(uint32_t)(at >> 32), bytes, 0x00020000};
	};
	auto issue_k = [&](int4_t rsrc, int stage, int j) {
		const unsigned m0 = lds_base + stage * kStage + (wave + kQ32Waves * j) * 1024;
		asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(load_k[j]), "s"(rsrc), "s"(m0) : "m0");
	};
	auto issue_v = [&](int4_t rsrc, int stage, int j) {
		const unsigned m0 = lds_base + stage * kStage + kTile + (wave + kQ32Waves * j) * 1024;
		asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(load_v[j]), "s"(rsrc), "s"(m0) : "m0");
	};
	typedef __attribute__((address_space(3))) const half8_t* LdsHalf8;
	const unsigned k_addr = lds_base + n * kRow + ((h ^ q32_k_swizzle<D>(n)) * 16);          // ^ 32 st, + 32 kb rows
	// V: lane r of a group of 16 reads key row 16 u + 8 jj + 4 h + r / 4, chunk 4 c + 2 (group % 2) + (r % 4) / 2
	const int vr = (lane & 15) >> 2;
	const unsigned v_addr = lds_base + kTile + (4 * h + vr) * kRow +
	                        (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ q32_v_swizzle<D>(vr)) * 16) + (lane & 1) * 8;   // ^ 64 c

	// the tiles in which some query of this wave sees a key
	const int wt_first = any_lo > 0 && any_lo / KT > t_first ? any_lo / KT : t_first;
	const int wt_last = any_hi < 0 ? -1 : (any_hi / KT < t_last ? any_hi / KT : t_last);

	float mt = -INFINITY;                                    // maximum of the scores of the tile ahead (raw; with softcap logits)
	constexpr int kStepsA = KS * KB, kStepsB = 2 * KB * DC, kSteps = kStepsA + kStepsB;
	typedef float16_t Scores[KB];

	auto is_interior = [&](int t) { return t * KT >= all_lo && t * KT + KT - 1 <= all_hi; };      // wave-uniform
	auto max_pair = [&](const Scores& s, int y) {
		const float x0 = s[y / 8][2 * (y % 8)], x1 = s[y / 8][2 * (y % 8) + 1];
		mt = y == 0 ? fmaxf(x0, x1) : fmaxf(fmaxf(mt, x0), x1);
	};
	auto logits_of_pair = [&](Scores& s, int y) {
		if constexpr (SOFTCAP)
		{
			s[y / 8][2 * (y % 8)] = logit2<true>(s[y / 8][2 * (y % 8)], k_in, a.k_cap);
			s[y / 8][2 * (y % 8) + 1] = logit2<true>(s[y / 8][2 * (y % 8) + 1], k_in, a.k_cap);
		}
	};
	auto max_scores = [&](const Scores& s) {
#pragma unroll
		for (int y = 0; y < 8 * KB; ++y) max_pair(s, y);
	};
	auto mask_scores = [&](Scores& s, int t) {
		// (through an empty statement: the compiler would do without the branch around this and test every tile's scores)
		int lo = vis_lo - t * KT - 4 * h, hi = vis_hi - t * KT - 4 * h;
		asm volatile("" : "+v"(lo), "+v"(hi));
#pragma unroll
		for (int kb = 0; kb < KB; ++kb)
#pragma unroll
			for (int i = 0; i < 16; ++i)
			{
				const int key = 32 * kb + 8 * (i / 4) + i % 4;           // + 4 h
				s[kb][i] = (key >= lo && key <= hi) ? s[kb][i] : -INFINITY;
			}
	};
	// own loads have landed; behind the barrier everybody's have, and everybody is done with what the loads issued behind it overwrite:
	// at the turn of tile t K(t + 1) and V(t) are there, K(t) and V(t - 1) free
	auto tile_barrier = [&]() {
		__builtin_amdgcn_s_waitcnt(0x0F70);                  // vmcnt(0)
		__syncthreads();
	};
	auto issue_all = [&](int t) {
		const int stage = (t + 1 - t_first) & 1;
		if (t + 1 <= t_last && t >= t_first)
		{
			const int4_t rsrc = rsrc_of(vp, t + 1);
#pragma unroll
			for (int j = 0; j < kSlots; ++j) issue_v(rsrc, stage, j);
		}
		if (t + 2 <= t_last && t >= t_first)
		{
			const int4_t rsrc = rsrc_of(kp, t + 2);
#pragma unroll
			for (int j = 0; j < kSlots; ++j) issue_k(rsrc, stage ^ 1, j);
		}
	};
	// the maximum of tile t joins the running one
	float z_in = 1.0f, z_add = 0.0f;
	auto take_maximum = [&](Scores& cur) {
		float m_tile = max_over_lane_halves(mt);
		if constexpr (!SOFTCAP) m_tile *= k_in;
		// the running maximum settles after some tiles; while no query of the wave raises it, the pass over the accumulators is
		// left out
		if (__builtin_amdgcn_ballot_w64(m_tile > m_run) != 0)
		{
			const float m_new = fmaxf(m_run, m_tile);
			const float corr = fast_exp2(m_run - (m_new == -INFINITY ? 0.0f : m_new));
			m_run = m_new;
			l_run *= corr;
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int i = 0; i < 16; ++i) o[c][i] *= corr;
		}
		const float m_safe = m_run == -INFINITY ? 0.0f : m_run;
		// p = 2^(z_in s + z_add).  The maximum is a rounded product, which the fma does not see as such: from 2^20 on, before
		// the rounding can take p out of the halves' range, the difference is taken between rounded products
		z_in = SOFTCAP ? 1.0f : k_in;
		z_add = kQ32HeadRoom - m_safe;
		if (__builtin_amdgcn_ballot_w64(fabsf(m_safe) > 0x1p20f) != 0)
		{
#pragma clang fp contract(off)
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int i = 0; i < 16; ++i)
				{
					const float z = SOFTCAP ? cur[kb][i] : cur[kb][i] * k_in;
					cur[kb][i] = z - m_safe;
				}
			z_in = 1.0f;
			z_add = kQ32HeadRoom;
		}
	};
	auto p_of_score = [&](const Scores& s, int e) { return fast_exp2(fmaf(s[e / 16][e % 16], z_in, z_add)); };

	// fragment i (16-key step u = i / DC, columns 32 c ..) of the V tile at `va`: K slot (h, j) is key 16 u + 8 (j / 4) + 4 h + j % 4
	auto v_fragment = [&](unsigned va, int i) {
		const int u = i / DC, c = i % DC;
		const unsigned src = (va ^ (64 * c)) + 16 * u * kRow;
		const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)src);
		const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)(src + 8 * kRow));
		return __builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi), 0, 1, 2, 3, 4, 5, 6, 7);
	};

	// One tile: S(t + 1) = K(t + 1) Q^T (SCORES) beside p(t) = 2^(z(t) - m), then O^T += V(t)^T P(t)^T (OUTPUT) beside the
	// maximum of S(t + 1), as steps of one MFMA.
	auto tile = [&](auto scores_tag, auto output_tag, Scores& cur, Scores& next, int t) {
		constexpr bool SCORES = decltype(scores_tag)::value, OUTPUT = decltype(output_tag)::value, BOTH = SCORES && OUTPUT;
		constexpr int kFirst = SCORES ? 0 : kStepsA, kEnd = OUTPUT ? kSteps : kStepsA;
		const int stage = (t + 1 - t_first) & 1;
		const unsigned ka = k_addr + stage * kStage, va = v_addr + (stage ^ 1) * kStage;
		half8_t frag[kAhead];
		auto read_operand = [&](int i) {
			if (i < kStepsA)
			{
				const int st = i / KB, kb = i % KB;
				frag[i % kAhead] = *(LdsHalf8)(uintptr_t)((ka ^ (32 * st)) + kb * 32 * kRow);
				return;
			}
			frag[i % kAhead] = v_fragment(va, i - kStepsA);
		};
		const int4_t rsrc_v = rsrc_of(vp, t + 1), rsrc_k = rsrc_of(kp, t + 2 <= t_last ? t + 2 : t_last);
		half8_t pf[2 * KB];
		float psum[2] = {0.0f, 0.0f};
		float x[32];
		auto pair_into_p = [&](int y) {
			psum[0] += x[2 * y];
			psum[1] += x[2 * y + 1];
			pf[y / 4][2 * (y % 4)] = (half_t)x[2 * y];
			pf[y / 4][2 * (y % 4) + 1] = (half_t)x[2 * y + 1];
		};
		auto vector_work = [&](int i) {
#pragma unroll
			for (int y = 0; y < 8 * KB; ++y)
			{
				const int at = y * 3 * kSteps / 64;
				if (i == at)
				{
					x[2 * y] = p_of_score(cur, 2 * y);
					x[2 * y + 1] = p_of_score(cur, 2 * y + 1);
				}
				if (i == at + 1) pair_into_p(y);
				if (i == kStepsA + 2 + y * (kStepsB - 2) / (8 * KB))
				{
					logits_of_pair(next, y);
					max_pair(next, y);
				}
			}
		};
		float16_t zero;
#pragma unroll
		for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
		auto step = [&](auto step_tag) {
			constexpr int i = decltype(step_tag)::value;
			__builtin_amdgcn_sched_barrier(0);
			if constexpr (i < kStepsA)
				next[i % KB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[i % kAhead], qf[i / KB], i < KB ? zero : next[i % KB], 0, 0, 0);
			else
				o[(i - kStepsA) % DC] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[i % kAhead], pf[(i - kStepsA) / DC], o[(i - kStepsA) % DC], 0, 0, 0);
			if constexpr (i + kAhead < kEnd) read_operand(i + kAhead);
			// the next tiles' loads, spread over the steps (past the end: the last tile's K once more, into the free stage)
			if constexpr (BOTH && i % kLoadSpacing == 1 && i / kLoadSpacing < 2 * kSlots)
			{
				constexpr int m = i / kLoadSpacing;
				if constexpr (m < kSlots) issue_v(rsrc_v, stage, m);
				else issue_k(rsrc_k, stage ^ 1, m - kSlots);
			}
			if constexpr (BOTH) vector_work(i);
		};
#pragma unroll
		for (int i = kFirst; i < kFirst + kAhead; ++i) read_operand(i);
		if constexpr (!BOTH) issue_all(t);
		if constexpr (OUTPUT && !SCORES)
		{
#pragma unroll
			for (int y = 0; y < 8 * KB; ++y)
			{
				x[2 * y] = p_of_score(cur, 2 * y);
				x[2 * y + 1] = p_of_score(cur, 2 * y + 1);
				pair_into_p(y);
			}
		}
		[&]<int... I>(std::integer_sequence<int, I...>) { (step(std::integral_constant<int, kFirst + I>{}), ...); }(std::make_integer_sequence<int, kEnd - kFirst>{});
		__builtin_amdgcn_sched_barrier(0);
		if constexpr (OUTPUT) l_run += psum[0] + psum[1];
		// (uses here, or the compiler moves the sums and the maximum behind the branch that follows)
		if constexpr (BOTH) asm volatile("" : "+v"(l_run), "+v"(mt));
		if constexpr (SCORES)
		{
			if constexpr (!OUTPUT)
			{
#pragma unroll
				for (int y = 0; y < 8 * KB; ++y) logits_of_pair(next, y);
				max_scores(next);
			}
			if (!is_interior(t + 1))
			{
				mask_scores(next, t + 1);
				max_scores(next);
			}
		}
	};
	if (t_first > t_last) {}
	else if constexpr (IN_TURN)
	{
		auto issue_tile = [&](int t, int stage) {
			const int4_t rsrc_k = rsrc_of(kp, t), rsrc_v = rsrc_of(vp, t);
#pragma unroll
			for (int j = 0; j < kSlots; ++j)
			{
				issue_k(rsrc_k, stage, j);
				issue_v(rsrc_v, stage, j);
			}
		};
		constexpr int kVRing = 8;                            // V fragments in registers, read ahead of the softmax
		issue_tile(t_first, 0);
		for (int t = t_first; t <= t_last; ++t)
		{
			tile_barrier();
			const int stage = (t - t_first) & 1;
			const bool any_visible = t >= wt_first && t <= wt_last;        // wave-uniform
			const unsigned ka = k_addr + stage * kStage, va = v_addr + stage * kStage;
			// the first K fragments, on their way while the next tile's loads are issued
			half8_t kf[KS][KB];
			auto read_k = [&](int st) {
#pragma unroll
				for (int kb = 0; kb < KB; ++kb) kf[st][kb] = *(LdsHalf8)(uintptr_t)((ka ^ (32 * st)) + kb * 32 * kRow);
			};
			if (any_visible)
			{
#pragma unroll
				for (int st = 0; st < kAhead; ++st) read_k(st);
			}
			__builtin_amdgcn_sched_barrier(0);
			if (t < t_last) issue_tile(t + 1, stage ^ 1);
			if (!any_visible) continue;

			Scores s;
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int i = 0; i < 16; ++i) s[kb][i] = 0.0f;
			__builtin_amdgcn_s_setprio(1);
#pragma unroll
			for (int st = 0; st < KS; ++st)
			{
#pragma unroll
				for (int kb = 0; kb < KB; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[st][kb], qf[st], s[kb], 0, 0, 0);
				if (st + kAhead < KS) read_k(st + kAhead);
				__builtin_amdgcn_sched_barrier(0);
			}
			__builtin_amdgcn_s_setprio(0);
			half8_t vf[kVRing];
			auto read_v = [&](int i) { vf[i % kVRing] = v_fragment(va, i); };
#pragma unroll
			for (int i = 0; i < kVRing; ++i) read_v(i);
			__builtin_amdgcn_sched_barrier(0);

#pragma unroll
			for (int y = 0; y < 8 * KB; ++y) logits_of_pair(s, y);
			if (!is_interior(t)) mask_scores(s, t);
			max_scores(s);
			take_maximum(s);
			half8_t pf[2 * KB];
			float psum[2] = {0.0f, 0.0f};
#pragma unroll
			for (int y = 0; y < 8 * KB; ++y)
			{
				const float p0 = p_of_score(s, 2 * y), p1 = p_of_score(s, 2 * y + 1);
				psum[0] += p0;
				psum[1] += p1;
				pf[y / 4][2 * (y % 4)] = (half_t)p0;
				pf[y / 4][2 * (y % 4) + 1] = (half_t)p1;
			}
			l_run += psum[0] + psum[1];
			__builtin_amdgcn_sched_barrier(0);
			__builtin_amdgcn_s_setprio(1);
#pragma unroll
			for (int i = 0; i < kStepsB; ++i)
			{
				o[i % DC] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i % kVRing], pf[i / DC], o[i % DC], 0, 0, 0);
				if (i + kVRing < kStepsB) read_v(i + kVRing);
				__builtin_amdgcn_sched_barrier(0);
			}
			__builtin_amdgcn_s_setprio(0);
		}
	}
	else
	{
		// K of the first tile, then (the turn of the tile before the first has nothing else to load) its V and K of the second
		const int4_t rsrc_k = rsrc_of(kp, t_first), rsrc_v = rsrc_of(vp, t_first), rsrc_k2 = rsrc_of(kp, t_first < t_last ? t_first + 1 : t_first);
#pragma unroll
		for (int j = 0; j < kSlots; ++j) issue_k(rsrc_k, 0, j);
#pragma unroll
		for (int j = 0; j < kSlots; ++j) issue_v(rsrc_v, 0, j);
#pragma unroll
		for (int j = 0; j < kSlots; ++j) issue_k(rsrc_k2, 1, j);
		constexpr std::true_type yes{};
		constexpr std::false_type no{};
		const bool any = wt_first <= wt_last;
		int t = t_first - 1;
		__builtin_amdgcn_s_waitcnt(0x0F70 | (2 * kSlots));   // vmcnt: the first tile's K
		__syncthreads();
		for (const int until = any ? wt_first - 1 : t_last + 1; t < until;)
		{
			issue_all(t);
			++t;
			if (t <= t_last) tile_barrier();
		}
		if (any)
		{
			Scores s0, s1;
			tile(yes, no, s1, s0, t++);
			for (; t + 1 < wt_last; t += 2)
			{
				take_maximum(s0);
				tile_barrier();
				tile(yes, yes, s0, s1, t);
				take_maximum(s1);
				tile_barrier();
				tile(yes, yes, s1, s0, t + 1);
			}
			if (t < wt_last)
			{
				take_maximum(s0);
				tile_barrier();
				tile(yes, yes, s0, s1, t++);
#pragma unroll
				for (int kb = 0; kb < KB; ++kb) s0[kb] = s1[kb];
			}
			take_maximum(s0);
			tile_barrier();
			tile(no, yes, s0, s1, t++);
			for (; t <= t_last; ++t)
			{
				tile_barrier();
				issue_all(t);
			}
		}
	}

	// ---- normalise and store: lane (n, h) holds y[row][32 c + 8 (i / 4) + 4 h + i % 4] ----
	const float l = l_run + __shfl_xor(l_run, 32);
	if (q_row >= a.n_q) return;
	if (parts > 1)
	{
		float* dst = a.partials + ((((int64_t)bh * walk.n_split + split_slot) * parts + part) * kQ32QueriesPerBlock + (q_row - q0)) * (D + 2);
#pragma unroll
		for (int c = 0; c < DC; ++c)
#pragma unroll
			for (int r = 0; r < 4; ++r)
				*reinterpret_cast<WsFloat4*>(dst + 32 * c + 8 * r + 4 * h) = float4_t{o[c][4 * r], o[c][4 * r + 1], o[c][4 * r + 2], o[c][4 * r + 3]};
		if (h == 0)
		{
			dst[D] = m_run;
			dst[D + 1] = l;
		}
		return;
	}
	const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int r = 0; r < 4; ++r)
		{
			half4_t out;
#pragma unroll
			for (int i = 0; i < 4; ++i) out[i] = (half_t)(o[c][4 * r + i] * inv);
			*reinterpret_cast<half4_t*>(yp + (int64_t)q_row * D + 32 * c + 8 * r + 4 * h) = out;
		}
}

}  // namespace

}  // namespace anygpu
