// Fused attention, fp16, head dimensions 64 and 128: 32 queries per wave.
//
// What bounds it.  Per tile of 64 keys a wave of 32 queries has 1024 (head dimension 64: 512) cycles of MFMAs, about 900 (770) of
// vector instructions and 32 (16) KB of fragments to read out of LDS.  With v_mfma_f32_32x32x16_f16 every fragment feeds 32 x 32
// scores, so the LDS stays below half of its rate; the 16-queries-per-wave kernel this one replaces read twice the bytes
// per score, and its 8-wave blocks of 128 or 256 queries ran one to a CU in lockstep.  Here a block is FOUR waves with 128
// queries, and two blocks (head dimension 64: three) share a CU without a barrier between them, so that one block's
// softmax, loads and ends run beside the other's products, and causal launches of ordinary prompts have twice as many
// pieces to pack onto the CUs.  Scores sit 32 to a lane (S^T = K Q^T: a lane holds one query), so row maxima are in-lane
// but for one exchange of lane halves.  Sums are those of the fp32 p, and the maximum is exact in every tile, so that the largest p is
// a power of two, which rounds to a half without an error (a maximum that lags until it is outgrown by 2^8 and sums of the
// rounded p by v_dot2 measured 5 % faster, but up to a tenth further from 64-bit results: 16 heads x 4096 x 128, q of
// N(0, 4): 2.36e-4 against 2.17e-4 (2-norm), of which the result's own rounding is 2.1e-4).
// Measured, causal (us; 16-queries-per-wave kernels -> here): 32 / 8 heads x 3000 x 128 126.6 -> 94.9 (0.78 PFLOP/s), 16 x 4096 x 128 115.9 ->
// 101.4, 64 / 8 x 1000 x 128 45.1 -> 31.8, 16 x 8192 x 128 367 -> 313 (0.88 PFLOP/s; a kernel that overlaps the products and the softmax
// inside a wave ran at the same rate there, as the clock drops under the matrix units' power), 32 x 2038 x 64 41.9 -> 36.6; without the causal
// rule 32 / 8 x 3000 x 128 183 -> 172, but 16 x 8192 x 128 542 -> 570 (the former kernel's rounds are full there).
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

template <int D, bool SOFTCAP>
__global__ __launch_bounds__(64 * kQ32Waves, 2) void sdp_attention_fwd_f16_q32_kernel(const AttnArgs a, const AttnWalk walk)
{
	constexpr int kRow = 2 * D;                              // bytes of a tile row
	constexpr int KT = kAttnKeysPerTile, KB = KT / 32;
	constexpr int kTile = KT * kRow;                         // bytes of a K or V tile
	constexpr int kStage = 2 * kTile;
	constexpr int KS = D / 16;                               // MFMA steps along the head dimension
	constexpr int DC = D / 32;                               // 32-wide column blocks of the output
	constexpr int kSlots = kTile / 1024 / kQ32Waves;         // direct loads of a tile per wave
	constexpr int kChunks = kRow / 16, kRowsPerLoad = 1024 / kRow;
	constexpr int kAhead = 4;                                // steps that the K fragments are read ahead
	constexpr int kVRing = 8;                                // V fragments in registers, read ahead of the softmax
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
	auto issue_tile = [&](int t, int stage) {
		const int bytes = min(KT, a.n_k - t * KT) * kRow;
		const uint64_t at_k = reinterpret_cast<uint64_t>(kp) + (int64_t)t * kTile, at_v = reinterpret_cast<uint64_t>(vp) + (int64_t)t * kTile;
		const int4_t rsrc_k = {(int)(uint32_t)at_k, (int)(uint32_t)(at_k >> 32), bytes, 0x00020000};
		const int4_t rsrc_v = {(int)(uint32_t)at_v, (int)(uint32_t)(at_v >> 32), bytes, 0x00020000};
#pragma unroll
		for (int j = 0; j < kSlots; ++j)
		{
			const unsigned m0k = lds_base + stage * kStage + (wave + kQ32Waves * j) * 1024;
			const unsigned m0v = m0k + kTile;
			asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(load_k[j]), "s"(rsrc_k), "s"(m0k) : "memory", "m0");
			asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(load_v[j]), "s"(rsrc_v), "s"(m0v) : "memory", "m0");
		}
	};
	typedef __attribute__((address_space(3))) const half8_t* LdsHalf8;
	const unsigned k_addr = lds_base + n * kRow + ((h ^ q32_k_swizzle<D>(n)) * 16);          // ^ 32 st, + 32 kb rows
	// V: lane r of a group of 16 reads key row 16 u + 8 jj + 4 h + r / 4, chunk 4 c + 2 (group % 2) + (r % 4) / 2
	const int vr = (lane & 15) >> 2;
	const unsigned v_addr = lds_base + kTile + (4 * h + vr) * kRow +
	                        (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ q32_v_swizzle<D>(vr)) * 16) + (lane & 1) * 8;   // ^ 64 c
	if (t_first <= t_last) issue_tile(t_first, 0);
	for (int t = t_first; t <= t_last; ++t)
	{
		__builtin_amdgcn_s_waitcnt(0x0F70);                  // vmcnt(0)
		__syncthreads();
		const int stage = (t - t_first) & 1;
		const int key0 = t * KT;
		const bool any_visible = key0 <= any_hi && key0 + KT - 1 >= any_lo;        // wave-uniform
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

		// ---- S^T = K Q^T ----
		float16_t s[KB];
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
		// V^T fragments, the first of them on their way during the softmax.  K slot (h, j) of 16-key step u is key
		// 16 u + 8 (j / 4) + 4 h + j % 4
		half8_t vf[kVRing];
		auto read_v = [&](int i) {
			const int u = i / DC, c = i % DC;
			const unsigned src = (va ^ (64 * c)) + 16 * u * kRow;
			const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)src);
			const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)(src + 8 * kRow));
			vf[i % kVRing] = __builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi), 0, 1, 2, 3, 4, 5, 6, 7);
		};
#pragma unroll
		for (int i = 0; i < kVRing; ++i) read_v(i);
		__builtin_amdgcn_sched_barrier(0);

		// ---- online softmax ----
		if constexpr (SOFTCAP)
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int i = 0; i < 16; ++i) s[kb][i] = logit2<true>(s[kb][i], k_in, a.k_cap);
		}
		if (!(key0 >= all_lo && key0 + KT - 1 <= all_hi))
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int i = 0; i < 16; ++i)
				{
					const int key = key0 + 32 * kb + 8 * (i / 4) + 4 * h + i % 4;
					s[kb][i] = (key >= vis_lo && key <= vis_hi) ? s[kb][i] : -INFINITY;
				}
		}
		float mt = fmaxf(s[0][0], s[1][0]);
#pragma unroll
		for (int i = 1; i < 16; ++i) mt = fmaxf(fmaxf(mt, s[0][i]), s[1][i]);
		mt = max_over_lane_halves(mt);
		if constexpr (!SOFTCAP) mt *= k_in;
		// the running maximum settles after some tiles; while no query of the wave raises it, the pass over the accumulators is
		// left out
		if (__builtin_amdgcn_ballot_w64(mt > m_run) != 0)
		{
			const float m_new = fmaxf(m_run, mt);
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
		float z_in = SOFTCAP ? 1.0f : k_in, z_add = kQ32HeadRoom - m_safe;
		if (__builtin_amdgcn_ballot_w64(fabsf(m_safe) > 0x1p20f) != 0)
		{
#pragma clang fp contract(off)
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int i = 0; i < 16; ++i)
				{
					const float z = SOFTCAP ? s[kb][i] : s[kb][i] * k_in;
					s[kb][i] = z - m_safe;
				}
			z_in = 1.0f;
			z_add = kQ32HeadRoom;
		}
		half8_t pf[2 * KB];
		float psum[2] = {0.0f, 0.0f};
#pragma unroll
		for (int kb = 0; kb < KB; ++kb)
#pragma unroll
			for (int i = 0; i < 16; i += 2)
			{
				const float z0 = SOFTCAP ? s[kb][i] + z_add : fmaf(s[kb][i], z_in, z_add);
				const float z1 = SOFTCAP ? s[kb][i + 1] + z_add : fmaf(s[kb][i + 1], z_in, z_add);
				const float p0 = fast_exp2(z0), p1 = fast_exp2(z1);
				psum[0] += p0;
				psum[1] += p1;
				pf[2 * kb + i / 8][i % 8] = (half_t)p0;
				pf[2 * kb + i / 8][i % 8 + 1] = (half_t)p1;
			}
		l_run += psum[0] + psum[1];

		// ---- O^T += V^T P^T ----
		__builtin_amdgcn_sched_barrier(0);
		__builtin_amdgcn_s_setprio(1);
#pragma unroll
		for (int i = 0; i < 2 * KB * DC; ++i)
		{
			o[i % DC] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i % kVRing], pf[i / DC], o[i % DC], 0, 0, 0);
			if (i + kVRing < 2 * KB * DC) read_v(i + kVRing);
			__builtin_amdgcn_sched_barrier(0);
		}
		__builtin_amdgcn_s_setprio(0);
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
