// Fused attention, fp16, 32 queries per wave in two groups of waves that take turns: sdp_attention_fwd_f16_pair_kernel.
#pragma once

#include "attention_walk.hpp"
#include "attention_split.hpp"
#include "device_utils.hpp"

#include <type_traits>

namespace anygpu {

namespace {

constexpr int kPairWaves = 4;                               // per group
constexpr int kPairQueriesPerBlock = 32 * kPairWaves;

// Chunk (16 bytes) of row r that the tile keeps at position c is c ^ swizzle(r): the tile rows are 2 D bytes without padding,
// filled by direct loads whose lanes land on consecutive 16 bytes.
template <int D>
__device__ __forceinline__ constexpr int pair_k_swizzle(int r) { return D >= 128 ? (r & 15) : ((r >> 1) & 7); }
template <int D>
__device__ __forceinline__ constexpr int pair_v_swizzle(int r) { return D >= 128 ? (((r & 3) << 2) | (r & 2)) : ((r & 3) << 1); }
// keys per tile: at head dimension 256 the registers have room for the scores of 32 keys
template <int D> constexpr int pair_keys() { return D == 256 ? 32 : 64; }

__device__ __forceinline__ float max_over_lane_halves(float x)
{
	float a = x, b = x;
	asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
	return fmaxf(a, b);
}

template <int D, bool SOFTCAP>
__global__ __launch_bounds__(128 * kPairWaves, 2) void sdp_attention_fwd_f16_pair_kernel(const AttnArgs a, const AttnWalk walk)
{
	constexpr int kRow = 2 * D;                              // bytes of a tile row
	constexpr int KT = pair_keys<D>(), KB = KT / 32;
	constexpr int kTile = KT * kRow;                         // bytes of a K or V tile
	constexpr int KS = D / 16;                               // MFMA steps along the head dimension
	constexpr int DC = D / 32;                               // 32-wide column blocks of the output
	constexpr int kSlots = kTile / 1024 / kPairWaves;         // direct loads of a tile per wave
	constexpr int kChunks = kRow / 16, kRowsPerLoad = 1024 / kRow;
	constexpr int NS = KS * KB, NP = 2 * KB * DC;            // MFMAs of S = K Q^T and of O += V^T P^T (the same number)
	static_assert(NS == NP, "the two products of a tile are interleaved one to one");
	extern __shared__ __align__(16) char lds[];

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int group = __builtin_amdgcn_readfirstlane(tid >> 8), wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
	const int n = lane & 31;                                 // query of the wave (second MFMA operand index)
	const int h = lane >> 5;                                 // lane half: k slots 8 h .. 8 h + 7 of an MFMA
	int bh, q_block, part, parts, split_slot;
	if (!attn_walk_locate_part(walk, blockIdx.x, bh, q_block, part, parts, split_slot)) return;
	const int q0 = q_block * kPairQueriesPerBlock;
	const half_t* qp = a.q + (int64_t)bh * a.n_q * D;
	const half_t* kp = a.k + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	const half_t* vp = a.v + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	half_t* yp = a.y + (int64_t)bh * a.n_q * D;

	const int q_last = (q0 + kPairQueriesPerBlock - 1 < a.n_q ? q0 + kPairQueriesPerBlock - 1 : a.n_q - 1);
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
	const int any_lo = a.window > 0 ? max(0, wq0 + a.diag - a.window + 1) : 0;
	const int all_hi = a.causal ? (wq0 + a.diag < a.n_k - 1 ? wq0 + a.diag : a.n_k - 1) : a.n_k - 1;
	const int all_lo = a.window > 0 ? wq0 + 31 + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;                   // l_run: this lane's share of the row sum
	float16_t o[DC];
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;

	// This group's tiles: t_first + group, + 2, ...; turn i of the group works on tile(i)
	const int tiles = t_last - t_first + 1, turns = tiles > 0 ? (tiles + 1) / 2 : 0;
	auto tile_of = [&](int i) { return t_first + 2 * i + group; };

	// LDS: per group two stages of K, two of V.  Tiles go global -> LDS without staging registers: load j of a wave fills rows
	// (wave + 4 j) kRowsPerLoad ..; the buffer's range ends with the last key, so the rows behind it come out as zeros.  Written
	// as assembly: the compiler would make LDS reads wait for all outstanding direct loads of the wave.
	const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds + group * (4 * kTile);
	const int load_row = kRowsPerLoad * wave + lane / kChunks;
	int load_k[kSlots], load_v[kSlots];
#pragma unroll
	for (int j = 0; j < kSlots; ++j)
	{
		const int row = load_row + kRowsPerLoad * kPairWaves * j;
		load_k[j] = row * kRow + ((lane % kChunks) ^ pair_k_swizzle<D>(row)) * 16;
		load_v[j] = row * kRow + ((lane % kChunks) ^ pair_v_swizzle<D>(row)) * 16;
	}
	typedef int int4_t __attribute__((ext_vector_type(4)));
	auto issue = [&](const half_t* base, const int (&off)[kSlots], unsigned lds_at, int i) __attribute__((always_inline)) {
		const int t = tile_of(i);
		const int rows = t <= t_last ? min(KT, a.n_k - t * KT) : 0;              // (past the end: nothing is fetched, but the count stays)
		const uint64_t at = reinterpret_cast<uint64_t>(base) + (int64_t)t * kTile;
		const int4_t rsrc = {(int)(uint32_t)at, (int)(uint32_t)(at >> 32), rows * kRow, 0x00020000};
#pragma unroll
		for (int j = 0; j < kSlots; ++j)
		{
			const unsigned m0 = lds_at + (i & 1) * kTile + (wave + kPairWaves * j) * 1024;
			asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(off[j]), "s"(rsrc), "s"(m0) : "memory", "m0");
		}
	};
	auto issue_k = [&](int i) { issue(kp, load_k, lds_base, i); };
	auto issue_v = [&](int i) { issue(vp, load_v, lds_base + 2 * kTile, i); };

	typedef __attribute__((address_space(3))) const half8_t* LdsHalf8;
	typedef __attribute__((address_space(3))) short4_t* LdsShort4;
	const unsigned k_addr = lds_base + n * kRow + ((h ^ pair_k_swizzle<D>(n)) * 16);          // ^ 32 st, + 32 kb rows
	// V: lane r of a group of 16 reads key row 16 u + 8 jj + 4 h + r / 4, chunk 4 c + 2 (group % 2) + (r % 4) / 2
	const int vr = (lane & 15) >> 2;
	const unsigned v_addr = lds_base + 2 * kTile + (4 * h + vr) * kRow +
	                        (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ pair_v_swizzle<D>(vr)) * 16) + (lane & 1) * 8;   // ^ 64 c

	float16_t s[KB];
	half8_t pf[2 * KB];
	// The matrix half of a turn: S = K Q^T of tile i (WITH_S) and O^T += V^T P^T of tile i - 1 (WITH_P), one MFMA of each in turn, the
	// operands out of LDS kAhead MFMAs ahead.  K slot (h, j) of 16-key step u is key 16 u + 8 (j / 4) + 4 h + j % 4.
	auto multiply = [&](auto s_tag, auto p_tag, int i) __attribute__((always_inline)) {
		constexpr bool WITH_S = decltype(s_tag)::value, WITH_P = decltype(p_tag)::value;
		constexpr int kSteps = (WITH_S ? NS : 0) + (WITH_P ? NP : 0);
		constexpr int kAhead = D == 256 ? 4 : 6;
		const unsigned ka = k_addr + (i & 1) * kTile, va = v_addr + ((i & 1) ^ 1) * kTile;
		half8_t frag[kAhead];
		auto read_operand = [&](int step) {
			const bool is_s = WITH_S && (!WITH_P || step % 2 == 0);
			const int x = WITH_S && WITH_P ? step / 2 : step;
			if (is_s)
			{
				const int st = x / KB, kb = x % KB;
				return *(LdsHalf8)(uintptr_t)((ka ^ (32 * (st % 8))) + 256 * (st / 8) + kb * 32 * kRow);
			}
			const int u = x / DC, c = x % DC;
			const unsigned src = (va ^ (64 * (c % 4))) + 256 * (c / 4) + 16 * u * kRow;
			const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4)(uintptr_t)src);
			const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4)(uintptr_t)(src + 8 * kRow));
			return (half8_t)__builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi), 0, 1, 2, 3, 4, 5, 6, 7);
		};
		if constexpr (WITH_S)
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int e = 0; e < 16; ++e) s[kb][e] = 0.0f;
		}
#pragma unroll
		for (int step = 0; step < kAhead; ++step) frag[step] = read_operand(step);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int step = 0; step < kSteps; ++step)
		{
			const bool is_s = WITH_S && (!WITH_P || step % 2 == 0);
			const int x = WITH_S && WITH_P ? step / 2 : step;
			if (is_s) s[x % KB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[step % kAhead], qf[x / KB], s[x % KB], 0, 0, 0);
			else o[x % DC] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[step % kAhead], pf[x / DC], o[x % DC], 0, 0, 0);
			if (step + kAhead < kSteps) frag[step % kAhead] = read_operand(step + kAhead);
			__builtin_amdgcn_sched_barrier(0);
		}
	};
	// The vector half: softcap, mask, maximum, p = exp2(z - m) of tile i
	auto soften = [&](int i) __attribute__((always_inline)) {
		const int key0 = tile_of(i) * KT;
		if constexpr (SOFTCAP)
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int e = 0; e < 16; ++e) s[kb][e] = logit2<true>(s[kb][e], k_in, a.k_cap);
		}
		if (!(key0 >= all_lo && key0 + KT - 1 <= all_hi))
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					const int key = key0 + 32 * kb + 8 * (e / 4) + 4 * h + e % 4;
					s[kb][e] = (key >= vis_lo && key <= vis_hi) ? s[kb][e] : -INFINITY;
				}
		}
		float mt = fmaxf(s[0][0], s[KB - 1][15]);
#pragma unroll
		for (int e = 1; e < 16 * KB - 1; e += 2) mt = fmaxf(fmaxf(mt, s[e / 16][e % 16]), s[(e + 1) / 16][(e + 1) % 16]);
		mt = max_over_lane_halves(mt);
		if constexpr (!SOFTCAP) mt *= k_in;
		// The maximum is only moved when a query of the wave has outgrown it by 2^8: until then p runs up to 256, which
		// the halves hold with the same relative precision, and the pass over the accumulators is left out.
		if (__builtin_amdgcn_ballot_w64(mt > m_run + 8.0f) != 0)
		{
			const float m_new = fmaxf(m_run, mt);
			const float corr = fast_exp2(m_run - (m_new == -INFINITY ? 0.0f : m_new));
			m_run = m_new;
			l_run *= corr;
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int e = 0; e < 16; ++e) o[c][e] *= corr;
		}
		const float neg_m = m_run == -INFINITY ? 0.0f : -m_run;
		const half2_t ones = {(half_t)1.0f, (half_t)1.0f};
#pragma unroll
		for (int kb = 0; kb < KB; ++kb)
#pragma unroll
			for (int e = 0; e < 16; e += 2)
			{
				const float z0 = SOFTCAP ? s[kb][e] + neg_m : fmaf(s[kb][e], k_in, neg_m);
				const float z1 = SOFTCAP ? s[kb][e + 1] + neg_m : fmaf(s[kb][e + 1], k_in, neg_m);
				const half2_t pp = {(half_t)fast_exp2(z0), (half_t)fast_exp2(z1)};
				l_run = __builtin_amdgcn_fdot2(pp, ones, l_run, false);
				pf[2 * kb + e / 8][e % 8] = pp[0];
				pf[2 * kb + e / 8][e % 8 + 1] = pp[1];
			}
	};

	constexpr std::true_type yes{};
	constexpr std::false_type no{};
	if (turns > 0)
	{
		issue_k(0);
		issue_v(0);
		issue_k(1);
		// While one group multiplies, the other one does its vector work: a barrier between the halves of every turn, the second
		// group half a turn behind the first.
		if (group == 1) __syncthreads();
		int i = 0;
		const auto turn = [&](auto s_tag, auto p_tag) __attribute__((always_inline)) {
			constexpr bool WITH_S = decltype(s_tag)::value, WITH_P = decltype(p_tag)::value;
			// K(i) and V(i - 1) have landed (the loads of V(i) and K(i + 1) may be on their way)
			asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * kSlots) : "memory");
			__syncthreads();
			if constexpr (WITH_S || WITH_P)
			{
				__builtin_amdgcn_s_setprio(1);
				multiply(s_tag, p_tag, i);
				__builtin_amdgcn_s_setprio(0);
			}
			__syncthreads();
			// K(i) and V(i - 1) are free
			issue_v(i + 1);
			issue_k(i + 2);
			if constexpr (WITH_S) soften(i);
			++i;
		};
		// turns in front of this wave's first visible tile, its tiles, turns behind its last (turns + 1 of them in all)
		const int i_first = any_hi >= any_lo ? max(0, (any_lo / KT - t_first - group + 1) / 2) : turns;
		const int i_last = any_hi >= any_lo ? (min(t_last, any_hi / KT) - t_first - group + 2) / 2 - 1 : -1;
		if (i_first <= i_last)
		{
			while (i < i_first) turn(no, no);
			turn(yes, no);
			while (i <= i_last) turn(yes, yes);
			turn(no, yes);
		}
		while (i <= turns) turn(no, no);
		if (group == 0) __syncthreads();
		// nothing may be on its way into the LDS any more when the groups meet there
		asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
		__syncthreads();
		// the second group hands its accumulators, maximum and sum to the first, lane by lane
		constexpr int kHandLane = 16 * DC * 4;                 // bytes of accumulators per lane
		char* hand = lds + wave * (64 * kHandLane + 512);
		if (group == 1)
		{
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int r = 0; r < 4; ++r)
					*reinterpret_cast<float4_t*>(hand + ((4 * c + r) * 64 + lane) * 16) = float4_t{o[c][4 * r], o[c][4 * r + 1], o[c][4 * r + 2], o[c][4 * r + 3]};
			*reinterpret_cast<float2_t*>(hand + 64 * kHandLane + lane * 8) = float2_t{m_run, l_run};
		}
		__syncthreads();
		if (group == 1) return;
		const float2_t other = *reinterpret_cast<const float2_t*>(hand + 64 * kHandLane + lane * 8);
		const float m_new = fmaxf(m_run, other[0]), safe = m_new == -INFINITY ? 0.0f : m_new;
		const float mine = fast_exp2(m_run - safe), theirs = fast_exp2(other[0] - safe);
		m_run = m_new;
		l_run = l_run * mine + other[1] * theirs;
#pragma unroll
		for (int c = 0; c < DC; ++c)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const float4_t v = *reinterpret_cast<const float4_t*>(hand + ((4 * c + r) * 64 + lane) * 16);
#pragma unroll
				for (int e = 0; e < 4; ++e) o[c][4 * r + e] = o[c][4 * r + e] * mine + v[e] * theirs;
			}
	}
	else if (group == 1) return;

	// ---- normalise and store: lane (n, h) holds y[row][32 c + 8 (i / 4) + 4 h + i % 4] ----
	const float l = l_run + __shfl_xor(l_run, 32);
	if (q_row >= a.n_q) return;
	if (parts > 1)
	{
		float* dst = a.partials + ((((int64_t)bh * walk.n_split + split_slot) * parts + part) * kPairQueriesPerBlock + (q_row - q0)) * (D + 2);
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
