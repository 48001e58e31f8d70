// Fused scaled-dot-product attention, forward, float32 throughout, for gfx950:
//     y = softmax(mask(softcap(alpha * q k^T))) v        per (batch, head)
// in one kernel, with the true fp32 matrix instruction v_mfma_f32_16x16x4_f32.  The score matrix never
// reaches HBM (8 heads x 8192 x 8192 keys: 2 GiB of fp32 scores written and read twice by the three-launch form).
//
// The structure is the one of the half precision kernel: a wave owns 16 queries, the query of a lane is
// lane % 16 in every product, so row maxima and sums are in-lane loops plus two cross-lane steps, and the
// rescale of the running output is an in-lane multiply.  Per tile of 32 keys:
//   * S^T = K Q^T: first operand K, second operand Q (in registers for the whole kernel).  The summation index
//     of an MFMA is a dummy index: lane group g takes head-dimension elements 16 s + 4 g + e in step (s, e), so
//     that a lane reads its four K values of four consecutive MFMAs with one 16-byte LDS load and holds its Q
//     values as the matching vectors.  A lane ends up with the scores of keys 16 kb + 4 g + r of its query.
//   * scale / softcap / mask, online max / sum in the log2 domain, p = exp2(z - m), all fp32;
//   * O^T += V^T P^T: second operand the p values exactly as they sit in the lane (key slot (kb, r) of lane
//     group g <-> key 16 kb + 4 g + r), first operand V^T: lane (i, g) loads the four columns 64 c + 4 i .. + 3
//     of that key's V row with one 16-byte LDS load, and element e of the vector feeds its own MFMA and
//     accumulator, which therefore holds head-dimension elements 64 c + 4 i' + e: permuted between lanes and
//     accumulators, and un-permuted for free at the store, where the four accumulators of a lane hold four
//     consecutive elements.
// At 32 cycles per MFMA the matrix pipe is the bound by a wide margin (the softmax arithmetic of a tile is
// about 2 % of its MFMA time); the K and V tiles of the next step are in flight meanwhile.
//
// Most launches take a second form (attend_f32_split, attend_f32_split16; the rule: attention_split_wanted).  The fp32 instruction has a
// sixteenth of the bf16 one's rate, and a float is the sum of three bf16 exactly, so a product of floats is six bf16 products whose missing
// terms lie below 2^-24 of it, of either sign: 6 / 16 of the matrix time, summed in fp32 as before, in fewer roundings.  Error against float64 (2-norm),
// fp32 instruction / bf16 parts: q, k, v of N(0, 1) 24 heads x 800 x 64 5.9e-7 / 3.4e-7, 10 x 800 x 128 6.4e-7 / 3.6e-7, 3 x 800 x 256
// 5.9e-7 / 4.6e-7; all mantissas 0x00FFFF 6.2e-7 / 3.6e-7, 6.8e-7 / 4.6e-7, 5.1e-7 / 5.2e-7; all mantissas 0x007FC0, which lose the most, 5.6e-7 / 3.2e-7,
// 5.7e-7 / 4.1e-7, 3.3e-7 / 6.4e-7.
// K and V are cut into their parts on their way into LDS (three planes each, once per block), p in its registers.  Bound: the bf16 matrix rate (and
// the power that goes with it).  us, fp32 instruction / bf16 parts: 8 / 4 heads x 8192 x 256, softcap, window 4096 1711 / 1039 (198 TFLOP/s, so 1.19 PFLOP/s of bf16
// products), 16 x 2000 x 128 297 / 181, 32 / 8 x 3000 x 128 causal 654 / 430, 32 x 2000 x 64 causal 175 / 124, 8 x 1000 x 256 causal 82.8 / 59.2; with a mask
// tensor 8 x 3001 x 256 causal 394 / 265, dense bias 679 / 424, 64 x 1393 x 128 causal 556 / 232.
//
// Masks are index rules (causal with the diagonal at n_k - n_q, sliding window); tiles without a visible key
// are skipped.  A query without any visible key gets zeros.
#include "device_utils.hpp"
#include "attention_walk.hpp"
#include "attention_split.hpp"
#include "attention_tile_map.hpp"
#include "attention_balance.hpp"
#include "gemm_band.hpp"
#include "launch.hpp"

#include <atomic>
#include <optional>

namespace anygpu {

namespace {


struct AttnArgsF32
{
	const float* q;
	const float* k;
	const float* v;
	float* y;
	int n_q, n_k;
	int q_per_kv;          // query heads that share one k / v head
	int diag;              // key j is causally visible to query i iff j <= i + diag
	int causal;
	int window;            // 0: off; else key j is visible iff j > i + diag - window
	float k_in, k_cap;     // logit transform constants (see logit2)
	float* partials;       // key-split blocks leave their partial results here: [head][split slot][part][query][D + 2]
	const float* mask;     // MASK kernels: additive mask [n_q, n_k] shared by all heads (added behind scale and softcap)
	int64_t mask_stride;   // floats between its rows
	const unsigned long long* tile_map;   // MASK kernels: visible-tile words [query block][map_words] (attention_tile_map.hpp), or nullptr
	int map_words;
};

// log2(e) * softcap(alpha * s); without softcap k_in = alpha log2(e); with it
// cap log2(e) tanh(alpha s / cap) = k_cap - 2 k_cap / (1 + exp2(s k_in)), k_in = 2 log2(e) alpha / cap
template <bool SOFTCAP>
__device__ __forceinline__ float logit2(float s, float k_in, float k_cap)
{
	if constexpr (SOFTCAP)
	{
		const float t = fast_exp2(s * k_in);
		return fmaf(fast_rcp(1.0f + t), -2.0f * k_cap, k_cap);
	}
	return s * k_in;
}

template <int D, int KT>
struct AttnLdsF32
{
	static constexpr int kPitch = D + 8;                      // floats per tile row: 32 bytes of padding
	static constexpr int kStageFloats = 2 * KT * kPitch;      // a K tile and a V tile of KT keys
};

// Scheduling-group masks of __builtin_amdgcn_sched_group_barrier
constexpr int kSchedMfma = 0x008;
constexpr int kSchedDsRead = 0x100;

// vmcnt(0) with the other counters left alone (gfx9 encoding: vmcnt in [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8])
__device__ __forceinline__ void wait_vmem_all()
{
	__builtin_amdgcn_s_waitcnt(0x0F70);
}

// WAVES waves per block, 16 queries per wave, tiles of KT keys.
// DIRECT (head dimension 256, where a tile row is exactly the 1024 bytes one wave-wide load instruction moves): the
// tiles go from memory straight into LDS, into one of two stages, so no staging registers are held and a block of
// 8 waves (two per SIMD: one multiplies while the other does its softmax arithmetic) fits the register file.
// Otherwise the tiles pass through registers into a single stage.
// MASK: an additive mask tensor instead of (or on top of) the index rules: the four mask values of a lane's four scores
// of a key block are consecutive in memory; they are requested in front of the tile's first product and added behind
// scale and softcap.  A tile that the mask hides from every query of a wave costs the wave no products; a tile that the
// visible-tile map of the mask (attention_tile_map.hpp) has not set for the block is neither loaded nor waited for.
// x summed over the four groups of 16 lanes, in all of them (max_over_lane_rows has the manner)
__device__ __forceinline__ float sum_over_lane_rows(float x)
{
	float a = x, b = x;
	asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
	const float sum = a + b;
	a = sum;
	b = sum;
	asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
	return a + b;
}

// One query block over the tiles [t_first, t_last] (MASK: the set ones of map_row, if there is a map).  partial: NULL, or where the block's
// [query][D accumulators, maximum, sum] go instead of y.
template <int D, bool SOFTCAP, int WAVES, int KT, bool DIRECT, bool MASK>
__device__ __forceinline__ void attend_f32(const AttnArgsF32& a, float* const lds_base, int bh, int q_block, int t_first, int t_last,
                                           const unsigned long long* __restrict__ map_row, float* partial)
{
	constexpr int kKeysPerTile = KT;
	static_assert(!DIRECT || D == 256, "one load instruction per tile row");
	constexpr int kQueriesPerBlock = 16 * WAVES;
	constexpr int THREADS = 64 * WAVES;
	using L = AttnLdsF32<D, KT>;
	typedef __attribute__((address_space(3))) void lds_void;
	typedef const __attribute__((address_space(1))) void global_void;
	constexpr int KS = D / 16;                      // 16-element groups of the head dimension (q k^T: 4 MFMAs each)
	constexpr int DC = D / 64;                      // 64-wide column groups of the output (4 accumulators each)
	constexpr int KB = kKeysPerTile / 16;           // 16-key blocks per tile
	constexpr int VPR = D / 4;                      // 16-byte vectors per row
	constexpr int VPT = kKeysPerTile * VPR / THREADS;   // vectors per thread per tile and matrix
	static_assert(kKeysPerTile * VPR % THREADS == 0, "the tile divides over the threads");

	int tid = threadIdx.x;
	asm volatile("" : "+v"(tid));                   // (a caller's loop keeps nothing of a lane's addresses in registers)
	__builtin_assume(tid >= 0 && tid < 512);
	const int lane = tid & (kWaveSize - 1);
	const int wave = tid >> 6;
	const int n = lane & 15;                        // query inside the wave's block (second MFMA operand index)
	const int g = lane >> 4;                        // lane group: summation slot g of an MFMA
	const int q0 = q_block * kQueriesPerBlock;
	const float* qp = a.q + (int64_t)bh * a.n_q * D;
	const float* kp = a.k + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	const float* vp = a.v + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	float* yp = a.y + (int64_t)bh * a.n_q * D;

	// this lane's query as second operand: q[row][16 s + 4 g .. + 3]
	const int q_row = q0 + 16 * wave + n;
	float4_t qf[KS];
#pragma unroll
	for (int s = 0; s < KS; ++s)
	{
		float4_t val = {0.0f, 0.0f, 0.0f, 0.0f};
		if (q_row < a.n_q) val = *reinterpret_cast<const float4_t*>(qp + (int64_t)q_row * D + 16 * s + 4 * g);
		qf[s] = val;
	}
	int vis_hi = a.causal ? q_row + a.diag : a.n_k - 1;
	if (vis_hi > a.n_k - 1) vis_hi = a.n_k - 1;
	const int vis_lo = a.window > 0 ? q_row + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;         // l_run: this lane's share of the row sum
	float4_t o[DC][4];
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int e = 0; e < 4; ++e) o[c][e] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
	// keys visible to every query of this wave need no per-element test: [all_lo, all_hi]
	const int wq0 = q0 + 16 * wave, wq1 = wq0 + 15;
	const int all_hi = a.causal ? (wq0 + a.diag < a.n_k - 1 ? wq0 + a.diag : a.n_k - 1) : a.n_k - 1;
	const int all_lo = a.window > 0 ? wq1 + a.diag - a.window + 1 : 0;

	// DIRECT: wave w moves rows w, w + WAVES, ... of the K tile and of the V tile; rows past the last key are
	// replaced by the last one (their scores are masked, their p is 0)
	auto tile_direct = [&](int t, int stage) {
		float* k_dst = lds_base + stage * L::kStageFloats;
		float* v_dst = k_dst + kKeysPerTile * L::kPitch;
		const int w = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
		for (int i = 0; i < kKeysPerTile / WAVES; ++i)
		{
			const int row = w + WAVES * i;
			int key = t * kKeysPerTile + row;
			key = key < a.n_k ? key : a.n_k - 1;
			__builtin_amdgcn_global_load_lds((global_void*)(kp + (int64_t)key * D + 4 * lane), (lds_void*)(k_dst + row * L::kPitch), 16, 0, 0);
			__builtin_amdgcn_global_load_lds((global_void*)(vp + (int64_t)key * D + 4 * lane), (lds_void*)(v_dst + row * L::kPitch), 16, 0, 0);
		}
	};

	float4_t kr[DIRECT ? 1 : VPT], vr[DIRECT ? 1 : VPT];
	auto tile_load = [&](int t) {
#pragma unroll
		for (int i = 0; i < (DIRECT ? 0 : VPT); ++i)
		{
			const int idx = tid + THREADS * i;
			const int row = idx / VPR, col = idx % VPR;
			const int key = t * kKeysPerTile + row;
			float4_t kv = {0.0f, 0.0f, 0.0f, 0.0f}, vv = {0.0f, 0.0f, 0.0f, 0.0f};
			if (key < a.n_k)
			{
				kv = *reinterpret_cast<const float4_t*>(kp + (int64_t)key * D + col * 4);
				vv = *reinterpret_cast<const float4_t*>(vp + (int64_t)key * D + col * 4);
			}
			kr[i] = kv;
			vr[i] = vv;
		}
	};
	auto tile_store = [&]() {
		float* k_dst = lds_base;
		float* v_dst = k_dst + kKeysPerTile * L::kPitch;
#pragma unroll
		for (int i = 0; i < (DIRECT ? 0 : VPT); ++i)
		{
			const int idx = tid + THREADS * i;
			const int row = idx / VPR, col = idx % VPR;
			*reinterpret_cast<float4_t*>(k_dst + row * L::kPitch + col * 4) = kr[i];
			*reinterpret_cast<float4_t*>(v_dst + row * L::kPitch + col * 4) = vr[i];
		}
	};

	// MASK: the mask values of this lane's scores of tile t: four consecutive floats per key block, at any alignment.  They stay
	// as they come until the tile's turn (a product here would wait for them, and with them for the loads of the whole next
	// tile, on every tile: 8 heads x 3001 x 256 causal 422 -> 392 us, 64 x 1393 x 128 causal 694 -> 557).  In tiles that end inside the key range all lanes load, those of
	// rows past the last query the last row; in the last tile keys past the end read nothing (their scores are masked).
	float4_t mk_next[MASK ? KB : 1];
	const float* const mask_row = MASK ? a.mask + (int64_t)(q_row < a.n_q ? q_row : a.n_q - 1) * a.mask_stride : nullptr;
	auto load_mask = [&](float4_t (&dst)[MASK ? KB : 1], int t) {
		typedef float4_t LooseF4 __attribute__((aligned(4)));
		if ((t + 1) * kKeysPerTile <= a.n_k)
		{
#pragma unroll
			for (int kb = 0; kb < (MASK ? KB : 0); ++kb) dst[kb] = *reinterpret_cast<const LooseF4*>(mask_row + t * kKeysPerTile + 16 * kb + 4 * g);
			return;
		}
#pragma unroll
		for (int kb = 0; kb < (MASK ? KB : 0); ++kb)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const int key = t * kKeysPerTile + 16 * kb + 4 * g + r;
				dst[kb][r] = key < a.n_k ? mask_row[key] : -INFINITY;
			}
	};
	// MASK: the walk visits the tiles that the map has set (all of them without a map); t_next is the tile after t on
	// that walk, the stages alternate along it
	AttentionVisibleWalk visible{map_row};
	if constexpr (MASK) t_first = visible.next(t_first, t_last);
	if (t_first <= t_last)
	{
		if constexpr (MASK) load_mask(mk_next, t_first);
		if constexpr (DIRECT) tile_direct(t_first, 0);
		else tile_load(t_first);
	}
	int t_next = 0, stage_m = 0;
	for (int t = t_first; t <= t_last; t = MASK ? t_next : t + 1, stage_m ^= 1)
	{
		const float* k_lds = lds_base;
		const int stage = MASK ? stage_m : (t - t_first) & 1;
		if constexpr (MASK) t_next = visible.next(t + 1, t_last);
		else t_next = t + 1;
		if constexpr (DIRECT)
		{
			// own loads of tile t have landed; behind the barrier everybody's have, and everybody is done with the
			// stage of the tile before, which the loads of the next tile overwrite
			wait_vmem_all();
			__syncthreads();
			if (t_next <= t_last) tile_direct(t_next, stage ^ 1);
			k_lds = lds_base + stage * L::kStageFloats;
		}
		else
		{
			__syncthreads();                       // the previous tile has been read by everybody
			tile_store();
			__syncthreads();
			if (t_next <= t_last) tile_load(t_next);      // in flight while this tile is used
		}
		const float* v_lds = k_lds + kKeysPerTile * L::kPitch;

		// the mask values of this lane's scores of the tile (log2 domain) were requested a tile ahead; those of the next
		// tile go out now.  A tile in which the mask hides every key from every query of the wave costs the wave nothing
		// further (under a causal mask tensor that is half of the tiles).
		float4_t mk[MASK ? KB : 1];
		if constexpr (MASK)
		{
			bool any_visible = false;
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
			{
				mk[kb] = mk_next[kb] * kLog2e;
#pragma unroll
				for (int r = 0; r < 4; ++r) any_visible |= mk[kb][r] > -INFINITY && q_row < a.n_q;
			}
			if (t_next <= t_last) load_mask(mk_next, t_next);
			if (__builtin_amdgcn_ballot_w64(any_visible) == 0) continue;
		}

		// ---- S^T = K Q^T: s[kb][r] = score of key 16 kb + 4 g + r against this lane's query ----
		// The K vectors of step st + 1 are read from LDS before the MFMAs of step st are issued (the scheduling
		// groups pin that order: left alone the compiler puts every read right in front of its first use and the
		// matrix pipe drains while the wave waits for LDS).
		float4_t s[KB];
#pragma unroll
		for (int kb = 0; kb < KB; ++kb) s[kb] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
		float4_t kf[2][KB];
		auto read_k = [&](float4_t (&dst)[KB], int st) {
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
				dst[kb] = *reinterpret_cast<const float4_t*>(k_lds + (16 * kb + n) * L::kPitch + 16 * st + 4 * g);
		};
		read_k(kf[0], 0);
		__builtin_amdgcn_sched_group_barrier(kSchedDsRead, KB, 0);
#pragma unroll
		for (int st = 0; st < KS; ++st)
		{
			if (st + 1 < KS) read_k(kf[(st + 1) & 1], st + 1);
#pragma unroll
			for (int e = 0; e < 4; ++e)
#pragma unroll
				for (int kb = 0; kb < KB; ++kb)
					s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[st & 1][kb][e], qf[st][e], s[kb], 0, 0, 0);
			// the reads go out behind the step's first MFMA: the wait in front of that MFMA then covers exactly the
			// vectors it needs, not the ones just requested
			__builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
			if (st + 1 < KS) __builtin_amdgcn_sched_group_barrier(kSchedDsRead, KB, 0);
			__builtin_amdgcn_sched_group_barrier(kSchedMfma, 4 * KB - 1, 0);
		}

		// ---- online softmax ----
		const int tile_key0 = t * kKeysPerTile;
		const bool interior = tile_key0 >= all_lo && tile_key0 + kKeysPerTile - 1 <= all_hi;   // wave-uniform
		float z[KB][4];
		float mt = -INFINITY;
		if (interior && !MASK)
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int r = 0; r < 4; ++r)
				{
					z[kb][r] = logit2<SOFTCAP>(s[kb][r], a.k_in, a.k_cap);
					mt = fmaxf(mt, z[kb][r]);
				}
		}
		else
		{
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int r = 0; r < 4; ++r)
				{
					const int key = tile_key0 + 16 * kb + 4 * g + r;
					const float zz = logit2<SOFTCAP>(s[kb][r], a.k_in, a.k_cap) + (MASK ? mk[MASK ? kb : 0][r] : 0.0f);
					z[kb][r] = (key >= vis_lo && key <= vis_hi) ? zz : -INFINITY;
					mt = fmaxf(mt, z[kb][r]);
				}
		}
		mt = max_over_lane_rows(mt);
		const float m_new = fmaxf(m_run, mt);
		const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;   // nothing visible so far: every term is exp2(-inf) = 0
		float psum = 0.0f;
		float p[KB][4];
#pragma unroll
		for (int kb = 0; kb < KB; ++kb)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				p[kb][r] = fast_exp2(z[kb][r] - m_safe);
				psum += p[kb][r];
			}
		// the running maximum settles after a few tiles; when no query of the wave raised it, the rescale
		// factor is 1 everywhere and the pass over the accumulators is skipped
		if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0)
		{
			const float corr = fast_exp2(m_run - m_safe);
			l_run *= corr;
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int e = 0; e < 4; ++e) o[c][e] *= corr;
		}
		l_run += psum;
		m_run = m_new;

		// ---- O^T += V^T P^T, the V vectors of key slot i + 1 read before the MFMAs of slot i ----
		float4_t vf[2][DC];
		auto read_v = [&](float4_t (&dst)[DC], int slot) {
			const int kb = slot >> 2, r = slot & 3;
#pragma unroll
			for (int c = 0; c < DC; ++c)
				dst[c] = *reinterpret_cast<const float4_t*>(v_lds + (16 * kb + 4 * g + r) * L::kPitch + 64 * c + 4 * n);
		};
		read_v(vf[0], 0);
		__builtin_amdgcn_sched_group_barrier(kSchedDsRead, DC, 0);
#pragma unroll
		for (int slot = 0; slot < 4 * KB; ++slot)
		{
			if (slot + 1 < 4 * KB) read_v(vf[(slot + 1) & 1], slot + 1);
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int e = 0; e < 4; ++e)
					o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[slot & 1][c][e], p[slot >> 2][slot & 3], o[c][e], 0, 0, 0);
			__builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
			if (slot + 1 < 4 * KB) __builtin_amdgcn_sched_group_barrier(kSchedDsRead, DC, 0);
			__builtin_amdgcn_sched_group_barrier(kSchedMfma, 4 * DC - 1, 0);
		}
	}

	// ---- normalise and store: register r of accumulator (c, e) is y[row][64 c + 4 (4 g + r) + e] ----
	const float l = sum_over_lane_rows(l_run);
	if (partial != nullptr)
	{
		// unnormalised accumulators, running maximum and sum of this part of the keys
		if (q_row < a.n_q)
		{
			float* dst = partial + (int64_t)(q_row - q0) * (D + 2);
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int r = 0; r < 4; ++r)
					*reinterpret_cast<WsFloat4*>(dst + 64 * c + 16 * g + 4 * r) = float4_t{o[c][0][r], o[c][1][r], o[c][2][r], o[c][3][r]};
			if (g == 0)
			{
				dst[D] = m_run;
				dst[D + 1] = l;
			}
		}
		return;
	}
	const float inv = l > 0.0f ? 1.0f / l : 0.0f;
	if (q_row < a.n_q)
	{
#pragma unroll
		for (int c = 0; c < DC; ++c)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const float4_t out = {o[c][0][r] * inv, o[c][1][r] * inv, o[c][2][r] * inv, o[c][3][r] * inv};
				*reinterpret_cast<float4_t*>(yp + (int64_t)q_row * D + 64 * c + 16 * g + 4 * r) = out;
			}
	}
}

// The key tiles that some query of a block of QUERIES sees under the index rules: from the first key of its first query to the last of its last.
template <int QUERIES, int KT>
__device__ __forceinline__ void visible_tiles_f32(const AttnArgsF32& a, int q_block, int& t_first, int& t_last)
{
	const int q0 = q_block * QUERIES;
	const int q_last = (q0 + QUERIES - 1 < a.n_q ? q0 + QUERIES - 1 : a.n_q - 1);
	int key_hi = a.n_k - 1;
	if (a.causal && q_last + a.diag < key_hi) key_hi = q_last + a.diag;
	int key_lo = 0;
	if (a.window > 0 && q0 + a.diag - a.window + 1 > 0) key_lo = q0 + a.diag - a.window + 1;
	t_first = key_lo / KT;
	t_last = key_hi >= 0 ? key_hi / KT : -1;
}

// Which head and query block this block works on, the key tiles of it, and where a partial result goes (NULL: y).  False: a padding block.
template <int D, int QUERIES, int KT, bool MASK>
__device__ __forceinline__ bool attention_block_f32(const AttnArgsF32& a, const AttnWalk& walk, int& bh, int& q_block, int& t_first, int& t_last,
                                                    const unsigned long long*& map_row, float*& partial)
{
	int part, parts, split_slot;
	if (!attn_walk_locate_part(walk, blockIdx.x, bh, q_block, part, parts, split_slot)) return false;
	visible_tiles_f32<QUERIES, KT>(a, q_block, t_first, t_last);
	// MASK: the visible-tile map of the mask, where the launcher has made one: the words of this query block
	map_row = nullptr;
	if constexpr (MASK)
	{
		if (a.tile_map != nullptr) map_row = a.tile_map + (int64_t)q_block * a.map_words;
	}
	partial = nullptr;
	if (parts > 1)
	{
		// one part of the block's key tiles; the other parts are other blocks', a merge kernel combines them.  With a
		// map the parts divide the VISIBLE tiles among them, else the range
		if (MASK && map_row != nullptr) attention_visible_share(map_row, part, parts, t_first, t_last);
		else
		{
			const int per = (t_last - t_first + parts) / parts;
			t_first += part * per;
			if (t_first + per - 1 < t_last) t_last = t_first + per - 1;
		}
		partial = a.partials + (((int64_t)bh * walk.n_split + split_slot) * parts + part) * ((int64_t)QUERIES * (D + 2));
	}
	return true;
}

// The launch of the form above: every block finds its query block and the tiles of it.
template <int D, bool SOFTCAP, int WAVES, int KT, bool DIRECT, bool MASK>
__global__ __launch_bounds__(64 * WAVES) void sdp_attention_fwd_f32_kernel(const AttnArgsF32 a, const AttnWalk walk)
{
	extern __shared__ __align__(16) char lds_raw[];
	int bh, q_block, t_first, t_last;
	const unsigned long long* map_row;
	float* partial;
	if (!attention_block_f32<D, 16 * WAVES, KT, MASK>(a, walk, bh, q_block, t_first, t_last, map_row, partial)) return;
	attend_f32<D, SOFTCAP, WAVES, KT, DIRECT, MASK>(a, reinterpret_cast<float*>(lds_raw), bh, q_block, t_first, t_last, map_row, partial);
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));

// Two floats as sums of three bf16 each: the float rounded to nearest, what is left rounded likewise, and the rest, at most 2^-9, 2^-18 of the
// power of two below the float (8 bits each with their own signs, which together are all of its 24 bits).  Word p of w: part p of both, the
// first below.  Cut-off parts, twice as large and all of the float's sign, left 4.7e-7 of a product out of the six below, always
// towards zero; these 5.9e-8 (2^-24) at most and 5.3e-9 (root mean square over all mantissas) of either sign.
// Returned: what stands in the last part.  What lies below 2^-133 of it, the smallest bf16, is lost, of floats below 2^-110 (RestBits).
__device__ __forceinline__ float2_t split_pair(float lo, float hi, unsigned (&w)[3])
{
	typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
	for (int p = 0; p < 3; ++p)
	{
		w[p] = __builtin_bit_cast(unsigned, __builtin_convertvector(float2_t{lo, hi}, bf16x2_t));
		if (p == 2) break;
		lo -= __builtin_bit_cast(float, w[p] << 16);
		hi -= __builtin_bit_cast(float, w[p] & 0xFFFF0000u);
	}
	return float2_t{lo, hi};
}

// Whether parts have lost bits: the lower half of a last part's float is zero unless it has bits below the smallest bf16.
struct RestBits
{
	unsigned bits = 0;
	// (as an expression of its own it kept the last parts of a whole tile in registers)
	__device__ __forceinline__ void take(float2_t rest) { asm("v_or3_b32 %0, %1, %2, %0" : "+v"(bits) : "v"(rest[0]), "v"(rest[1])); }
	__device__ __forceinline__ bool lost() const { return (bits & 0xFFFFu) != 0; }
};

constexpr int kSplitQueries = 128, kSplitKeys = 32;
constexpr int64_t kSplitMaskStride = 1 << 22;   // mask rows at most this far apart: byte offsets in a query block fit 32 bits
// The form with 16 queries per wave, eight waves (the other: 32, four): where 32 leave no registers.
constexpr bool split_narrow(int head_dim, bool mask) { return head_dim == 256 || (head_dim == 128 && mask); }
constexpr int split_threads(int head_dim, bool mask) { return split_narrow(head_dim, mask) ? 512 : 256; }

template <int D, bool NARROW>
struct AttnLdsSplit
{
	// bytes of a row of a plane: both read patterns without bank conflicts (the lane groups that read V together are four keys apart
	// in the narrow form, else sixteen columns)
	static constexpr int kPitchK = 2 * D + 32, kPitchV = NARROW ? 2 * D + 32 : 2 * D + 64;
	static constexpr int kPlaneK = kSplitKeys * kPitchK, kPlaneV = kSplitKeys * kPitchV;
	static constexpr int kBytes = 3 * (kPlaneK + kPlaneV);
};

// Whether any thread of the block says so.  (Smaller than __syncthreads_or, whose lane numbers the compiler kept in registers through the
// key loop.)  The LDS may be in use before, and is free again behind the caller's next barrier.
template <int WAVES>
__device__ __forceinline__ bool any_of_block(bool said, char* const lds, int wave)
{
	int* const flags = reinterpret_cast<int*>(lds);
	const int of_wave = __builtin_amdgcn_ballot_w64(said) != 0;
	__syncthreads();
	flags[wave] = of_wave;
	__syncthreads();
	int any = 0;
#pragma unroll
	for (int i = 0; i < WAVES; ++i) any |= flags[i];
	return __builtin_amdgcn_readfirstlane(any) != 0;
}

// A query block of 128 with every product of floats as six products of bf16 parts on v_mfma_f32_32x32x16_bf16, accumulated in fp32:
// x y = x1 y1 + x1 y2 + x2 y1 + x2 y2 + x1 y3 + x3 y1; the terms left out are below 2^-24 of x y.
// False, with nothing stored, where a result is not finite (the parts of an infinity, and of the floats that round to one, are no numbers) or
// the parts of an operand have lost bits: the caller takes the form above.
template <int D, bool SOFTCAP, bool MASK>
__device__ __forceinline__ bool attend_f32_split(const AttnArgsF32& a, char* const lds, int bh, int q_block, int t_first, int t_last,
                                                 const unsigned long long* __restrict__ map_row, float* partial)
{
	constexpr int KT = kSplitKeys, THREADS = 256;
	using L = AttnLdsSplit<D, false>;
	constexpr int KS = D / 16;                      // MFMA steps along the head dimension
	constexpr int DC = D / 32;                      // 32-wide column blocks of the output
	constexpr int VPR = D / 4;                      // float4 per row
	constexpr int VPT = KT * VPR / THREADS;         // float4 per thread and tile

	int tid = threadIdx.x;
	asm volatile("" : "+v"(tid));                   // (a caller's loop keeps nothing of a lane's addresses in registers)
	__builtin_assume(tid >= 0 && tid < 512);
	const int lane = tid & (kWaveSize - 1);
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 31;                        // query of the wave (second MFMA operand index)
	const int h = lane >> 5;                        // lane half: k slots 8 h .. 8 h + 7 of an MFMA
	const int q0 = q_block * kSplitQueries;
	const float* qp = a.q + (int64_t)bh * a.n_q * D;
	const float* kp = a.k + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	const float* vp = a.v + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	float* yp = a.y + (int64_t)bh * a.n_q * D;

	// this lane's query as second operands: q[row][16 s + 8 h .. + 7] in three parts
	const int wq0 = q0 + 32 * wave;
	const int q_row = wq0 + n;
	bf16x8_t qf[3][KS];
	RestBits rest;                                  // of q, k and v (weights below 2^-110 of the row's largest may lose bits)
#pragma unroll
	for (int s = 0; s < KS; ++s)
	{
		float4_t x[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
		if (q_row < a.n_q)
		{
			x[0] = *reinterpret_cast<const float4_t*>(qp + (int64_t)q_row * D + 16 * s + 8 * h);
			x[1] = *reinterpret_cast<const float4_t*>(qp + (int64_t)q_row * D + 16 * s + 8 * h + 4);
		}
		uint4_t w[3];
#pragma unroll
		for (int e = 0; e < 8; e += 2)
		{
			unsigned parts[3];
			rest.take(split_pair(x[e / 4][e % 4], x[e / 4][e % 4 + 1], parts));
#pragma unroll
			for (int p = 0; p < 3; ++p) w[p][e / 2] = parts[p];
		}
#pragma unroll
		for (int p = 0; p < 3; ++p) qf[p][s] = __builtin_bit_cast(bf16x8_t, w[p]);
	}
	// keys visible to every query of this wave need no per-element test: [all_lo, all_hi]
	const int all_hi = a.causal ? (wq0 + a.diag < a.n_k - 1 ? wq0 + a.diag : a.n_k - 1) : a.n_k - 1;
	const int all_lo = a.window > 0 ? wq0 + 31 + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;          // l_run: this lane's share of the row sum
	float16_t o[DC];
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;

	// A tile goes through registers, where its floats are cut into their parts, into the planes: VPT pieces per thread.  Rows past the last
	// key repeat it (their scores are masked, their p is 0).
	float4_t staged[VPT];
	auto fetch = [&](const float* src, int t) {
		const char* base = reinterpret_cast<const char*>(src) + (int64_t)t * (KT * D * 4);
		const int last = a.n_k - 1 - t * KT;        // KT - 1 and more: a whole tile
#pragma unroll
		for (int i = 0; i < VPT; ++i)
		{
			const int idx = tid + THREADS * i;
			const int over = idx / VPR > last ? idx / VPR - last : 0;
			staged[i] = *reinterpret_cast<const float4_t*>(base + (unsigned)(idx * 16 - over * (D * 4)));
		}
	};
	auto put = [&](bool of_v, int i) {
		const int idx = tid + THREADS * i;
		const int pitch = of_v ? L::kPitchV : L::kPitchK, plane = of_v ? L::kPlaneV : L::kPlaneK;
		char* const dst = lds + (of_v ? 3 * L::kPlaneK : 0) + (idx / VPR) * pitch + (idx % VPR) * 8;
		unsigned parts[2][3];
		rest.take(split_pair(staged[i][0], staged[i][1], parts[0]));
		rest.take(split_pair(staged[i][2], staged[i][3], parts[1]));
#pragma unroll
		for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2_t*>(dst + p * plane) = uint2_t{parts[0][p], parts[1][p]};
	};

	// MASK: the mask values of this lane's scores, keys 8 j + 4 h .. + 3 of the tile: four consecutive floats at any alignment, as they come.
	// Keys past the end read nothing and count as hidden.
	float4_t mk[MASK ? 4 : 1];
	const char* const mask_block = MASK ? reinterpret_cast<const char*>(a.mask + q0 * a.mask_stride) : nullptr;
	const unsigned mask_at = MASK ? (unsigned)((q_row < a.n_q ? q_row : a.n_q - 1) - q0) * (unsigned)(a.mask_stride * 4) + 16u * h : 0u;   // (32 bits: kSplitMaskStride)
	auto load_mask = [&](int t) {
		typedef float4_t LooseF4 __attribute__((aligned(4)));
		const float* const at = reinterpret_cast<const float*>(mask_block + (int64_t)t * (KT * 4) + mask_at);
		if ((t + 1) * KT <= a.n_k)
		{
#pragma unroll
			for (int j = 0; j < (MASK ? 4 : 0); ++j) mk[j] = *reinterpret_cast<const LooseF4*>(at + 8 * j);
			return;
		}
#pragma unroll
		for (int j = 0; j < (MASK ? 4 : 0); ++j)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const int key = t * KT + 8 * j + 4 * h + r;
				mk[j][r] = key < a.n_k ? at[8 * j + r] : -INFINITY;
			}
	};
	AttentionVisibleWalk visible{map_row};
	if constexpr (MASK) t_first = visible.next(t_first, t_last);
	if (t_first <= t_last)
	{
		fetch(kp, t_first);
		if constexpr (MASK) load_mask(t_first);
		__syncthreads();                            // (the query block before has been read by everybody)
#pragma unroll
		for (int i = 0; i < VPT; ++i) put(false, i);
		fetch(vp, t_first);
	}
	// Each product is a sequence of steps: a fragment (of V: of two column blocks), the third, second and first part in turn, and its one, two
	// or three products; a step's fragments are read some steps ahead, and the tile that the other product needs next is cut into the
	// planes behind the steps of the second half, its loads having had the first.  Neighbouring MFMAs use different accumulators.
	constexpr int kStepsQ = 3 * KS, kAheadQ = 4, kStepsV = 3 * DC, kAheadV = 2;
	static_assert(DC % 2 == 0, "column blocks in pairs");
	bf16x8_t frag[4];
	auto read_k = [&](int f) {
		const int st = f / 3, p = 2 - f % 3;
		frag[f % kAheadQ] = *reinterpret_cast<const bf16x8_t*>(lds + p * L::kPlaneK + n * L::kPitchK + (16 * st + 8 * h) * 2);
	};
	// slot (h, j) of 16-key step u is key 16 u + 8 (j / 4) + 4 h + j % 4
	auto read_v = [&](int f) {
		const int pair = f / 3, p = 2 - f % 3, u = pair / (DC / 2), c = 2 * (pair % (DC / 2));
		typedef __attribute__((address_space(3))) short4_t* LdsShort4;
#pragma unroll
		for (int i = 0; i < 2; ++i)
		{
			const char* src = lds + 3 * L::kPlaneK + p * L::kPlaneV + (16 * u + 4 * h + ((lane & 15) >> 2)) * L::kPitchV +
			                  (32 * (c + i) + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
			const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4)(src));
			const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4)(src + 8 * L::kPitchV));
			frag[2 * (f % kAheadV) + i] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
		}
	};
	// piece of the staged tile that goes behind step f of `steps`, or -1
	auto piece_at = [](int f, int steps) {
		const int half = steps / 2, every = half / VPT;
		return f >= half && (f - half) % every == 0 && (f - half) / every < VPT ? (f - half) / every : -1;
	};
	static_assert(kStepsQ / 2 >= VPT && kStepsV / 2 >= VPT, "steps for the pieces");
	int t_next = 0;
	for (int t = t_first; t <= t_last; t = t_next)
	{
		if constexpr (MASK) t_next = visible.next(t + 1, t_last);
		else t_next = t + 1;
		__syncthreads();                            // K(t) is complete, V of the tile before has been read by everybody
		// ---- S^T = K Q^T ----
		float16_t s;
#pragma unroll
		for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
		for (int f = 0; f < kAheadQ; ++f) read_k(f);
		__builtin_amdgcn_sched_barrier(0);
		__builtin_amdgcn_s_setprio(1);              // (the SIMD's other block has its softmax in between: 1 - 4 %)
#pragma unroll
		for (int f = 0; f < kStepsQ; ++f)
		{
#pragma unroll
			for (int x = f % 3; x >= 0; --x) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[f % kAheadQ], qf[x][f / 3], s, 0, 0, 0);
			if (f + kAheadQ < kStepsQ) read_k(f + kAheadQ);
			if (piece_at(f, kStepsQ) >= 0) put(true, piece_at(f, kStepsQ));
			__builtin_amdgcn_sched_barrier(0);
		}
		__builtin_amdgcn_s_setprio(0);
		// ---- online softmax: score i of this lane is key 8 (i / 4) + 4 h + i % 4 ----
		const int tile_key0 = t * KT;
		const bool interior = tile_key0 >= all_lo && tile_key0 + KT - 1 <= all_hi;   // wave-uniform
#pragma unroll
		for (int i = 0; i < 16; ++i)
		{
			s[i] = logit2<SOFTCAP>(s[i], a.k_in, a.k_cap);
			if constexpr (MASK) s[i] += mk[MASK ? i / 4 : 0][i % 4] * kLog2e;
		}
		if (!MASK && !interior)                     // (a mask's values past the last key hide them)
		{
			int row = n;
			asm volatile("" : "+v"(row));           // (found anew at each such tile: two registers)
			row += wq0;
			const int vis_hi = a.causal && row + a.diag < a.n_k - 1 ? row + a.diag : a.n_k - 1;
			const int vis_lo = a.window > 0 ? row + a.diag - a.window + 1 : 0;
#pragma unroll
			for (int i = 0; i < 16; ++i)
			{
				const int key = tile_key0 + 8 * (i / 4) + 4 * h + i % 4;
				s[i] = (key >= vis_lo && key <= vis_hi) ? s[i] : -INFINITY;
			}
		}
		float mt = s[0];
#pragma unroll
		for (int i = 1; i < 16; ++i) mt = fmaxf(mt, s[i]);
		mt = fmaxf(mt, __shfl_xor(mt, 32));
		const float m_new = fmaxf(m_run, mt);
		const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;   // nothing visible so far: every term is exp2(-inf) = 0
		// the running maximum settles after a few tiles; when no query of the wave raised it, the
		// rescale factor is 1 everywhere and the pass over the accumulators is skipped
		if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0)
		{
			const float corr = fast_exp2(m_run - m_safe);
			l_run *= corr;
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int i = 0; i < 16; ++i) o[c][i] *= corr;
		}
		m_run = m_new;
		float psum[2] = {0.0f, 0.0f};
		bf16x8_t pf[3][2];
#pragma unroll
		for (int u = 0; u < 2; ++u)
		{
			uint4_t w[3];
#pragma unroll
			for (int j = 0; j < 8; j += 2)
			{
				const float p0 = fast_exp2(s[8 * u + j] - m_safe), p1 = fast_exp2(s[8 * u + j + 1] - m_safe);
				psum[0] += p0;
				psum[1] += p1;
				unsigned parts[3];
				split_pair(p0, p1, parts);
#pragma unroll
				for (int p = 0; p < 3; ++p) w[p][j / 2] = parts[p];
			}
#pragma unroll
			for (int p = 0; p < 3; ++p) pf[p][u] = __builtin_bit_cast(bf16x8_t, w[p]);
		}
		l_run += psum[0] + psum[1];
		// (behind the last tile: that tile once more, of no consequence)
		const int t_load = t_next <= t_last ? t_next : t;
		if constexpr (MASK) load_mask(t_load);
		fetch(kp, t_load);
		__syncthreads();                            // V(t) is complete, K(t) has been read by everybody
		// ---- O^T += V^T P^T ----
#pragma unroll
		for (int f = 0; f < kAheadV; ++f) read_v(f);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int f = 0; f < kStepsV; ++f)
		{
			const int pair = f / 3, u = pair / (DC / 2), c = 2 * (pair % (DC / 2));
#pragma unroll
			for (int x = f % 3; x >= 0; --x)
#pragma unroll
				for (int i = 0; i < 2; ++i) o[c + i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[2 * (f % kAheadV) + i], pf[x][u], o[c + i], 0, 0, 0);
			if (f + kAheadV < kStepsV) read_v(f + kAheadV);
			if (piece_at(f, kStepsV) >= 0) put(false, piece_at(f, kStepsV));
			__builtin_amdgcn_sched_barrier(0);
		}
		fetch(vp, t_load);
	}

	// ---- normalise and store: lane (n, h) holds y[row][32 c + 8 (i / 4) + 4 h + i % 4] ----
	const float l = l_run + __shfl_xor(l_run, 32);
	float all = l;                                  // not finite where anything that entered it is not
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int i = 0; i < 16; ++i) all = fmaf(o[c][i], 0.0f, all);
	if (any_of_block<THREADS / kWaveSize>(rest.lost() || !(fabsf(all) < INFINITY), lds, wave)) return false;
	if (q_row >= a.n_q) return true;
	if (partial != nullptr)
	{
		// unnormalised accumulators, running maximum and sum of this part of the keys
		float* dst = partial + (int64_t)(q_row - q0) * (D + 2);
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
		return true;
	}
	const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int r = 0; r < 4; ++r)
			*reinterpret_cast<float4_t*>(yp + (int64_t)q_row * D + 32 * c + 8 * r + 4 * h) =
				float4_t{o[c][4 * r] * inv, o[c][4 * r + 1] * inv, o[c][4 * r + 2] * inv, o[c][4 * r + 3] * inv};
	return true;
}

// The same for head dimension 256, where a wave of 32 queries has no registers left: eight waves of 16 queries, v_mfma_f32_16x16x32_bf16.
template <int D, bool SOFTCAP, bool MASK>
__device__ __forceinline__ bool attend_f32_split16(const AttnArgsF32& a, char* const lds, int bh, int q_block, int t_first, int t_last,
                                                 const unsigned long long* __restrict__ map_row, float* partial)
{
	constexpr int KT = kSplitKeys, THREADS = 512;
	using L = AttnLdsSplit<D, true>;
	constexpr int KS = D / 32;                      // MFMA steps along the head dimension
	constexpr int DC = D / 16;                      // 16-wide column blocks of the output
	constexpr int KB = KT / 16;                     // 16-key blocks per tile
	constexpr int VPR = D / 4;                      // float4 per row
	constexpr int VPT = KT * VPR / THREADS;         // float4 per thread and tile

	int tid = threadIdx.x;
	asm volatile("" : "+v"(tid));                   // (a caller's loop keeps nothing of a lane's addresses in registers)
	__builtin_assume(tid >= 0 && tid < 512);
	const int lane = tid & (kWaveSize - 1);
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 15;                        // query of the wave (second MFMA operand index)
	const int g = lane >> 4;                        // lane group: k slots 8 g .. 8 g + 7 of an MFMA
	const int q0 = q_block * kSplitQueries;
	const float* qp = a.q + (int64_t)bh * a.n_q * D;
	const float* kp = a.k + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	const float* vp = a.v + (int64_t)(bh / a.q_per_kv) * a.n_k * D;
	float* yp = a.y + (int64_t)bh * a.n_q * D;

	// this lane's query as second operands: q[row][32 s + 8 g .. + 7] in three parts
	const int wq0 = q0 + 16 * wave;
	const int q_row = wq0 + n;
	bf16x8_t qf[3][KS];
	RestBits rest;                                  // of q, k and v (weights below 2^-110 of the row's largest may lose bits)
#pragma unroll
	for (int s = 0; s < KS; ++s)
	{
		float4_t x[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
		if (q_row < a.n_q)
		{
			x[0] = *reinterpret_cast<const float4_t*>(qp + (int64_t)q_row * D + 32 * s + 8 * g);
			x[1] = *reinterpret_cast<const float4_t*>(qp + (int64_t)q_row * D + 32 * s + 8 * g + 4);
		}
		uint4_t w[3];
#pragma unroll
		for (int e = 0; e < 8; e += 2)
		{
			unsigned parts[3];
			rest.take(split_pair(x[e / 4][e % 4], x[e / 4][e % 4 + 1], parts));
#pragma unroll
			for (int p = 0; p < 3; ++p) w[p][e / 2] = parts[p];
		}
#pragma unroll
		for (int p = 0; p < 3; ++p) qf[p][s] = __builtin_bit_cast(bf16x8_t, w[p]);
	}
	// keys visible to every query of this wave need no per-element test: [all_lo, all_hi]
	const int all_hi = a.causal ? (wq0 + a.diag < a.n_k - 1 ? wq0 + a.diag : a.n_k - 1) : a.n_k - 1;
	const int all_lo = a.window > 0 ? wq0 + 15 + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;          // l_run: this lane's share of the row sum
	float4_t o[DC];
#pragma unroll
	for (int c = 0; c < DC; ++c) o[c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

	// A tile goes through registers, where its floats are cut into their parts, into the planes: VPT pieces per thread.  Rows past the last
	// key repeat it (their scores are masked, their p is 0).
	float4_t staged[VPT];
	auto fetch = [&](const float* src, int t) {
		const char* base = reinterpret_cast<const char*>(src) + (int64_t)t * (KT * D * 4);
		const int last = a.n_k - 1 - t * KT;        // KT - 1 and more: a whole tile
#pragma unroll
		for (int i = 0; i < VPT; ++i)
		{
			const int idx = tid + THREADS * i;
			const int over = idx / VPR > last ? idx / VPR - last : 0;
			staged[i] = *reinterpret_cast<const float4_t*>(base + (unsigned)(idx * 16 - over * (D * 4)));
		}
	};
	auto put = [&](bool of_v, int i) {
		const int idx = tid + THREADS * i;
		const int pitch = of_v ? L::kPitchV : L::kPitchK, plane = of_v ? L::kPlaneV : L::kPlaneK;
		char* const dst = lds + (of_v ? 3 * L::kPlaneK : 0) + (idx / VPR) * pitch + (idx % VPR) * 8;
		unsigned parts[2][3];
		rest.take(split_pair(staged[i][0], staged[i][1], parts[0]));
		rest.take(split_pair(staged[i][2], staged[i][3], parts[1]));
#pragma unroll
		for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2_t*>(dst + p * plane) = uint2_t{parts[0][p], parts[1][p]};
	};

	// MASK: the mask values of this lane's scores, keys 16 j + 4 g .. + 3 of the tile: four consecutive floats at any alignment, as they come.
	// Keys past the end read nothing and count as hidden.
	float4_t mk[MASK ? KB : 1];
	const char* const mask_block = MASK ? reinterpret_cast<const char*>(a.mask + q0 * a.mask_stride) : nullptr;
	const unsigned mask_at = MASK ? (unsigned)((q_row < a.n_q ? q_row : a.n_q - 1) - q0) * (unsigned)(a.mask_stride * 4) + 16u * g : 0u;   // (32 bits: kSplitMaskStride)
	auto load_mask = [&](int t) {
		typedef float4_t LooseF4 __attribute__((aligned(4)));
		const float* const at = reinterpret_cast<const float*>(mask_block + (int64_t)t * (KT * 4) + mask_at);
		if ((t + 1) * KT <= a.n_k)
		{
#pragma unroll
			for (int j = 0; j < (MASK ? KB : 0); ++j) mk[j] = *reinterpret_cast<const LooseF4*>(at + 16 * j);
			return;
		}
#pragma unroll
		for (int j = 0; j < (MASK ? KB : 0); ++j)
#pragma unroll
			for (int r = 0; r < 4; ++r)
			{
				const int key = t * KT + 16 * j + 4 * g + r;
				mk[j][r] = key < a.n_k ? at[16 * j + r] : -INFINITY;
			}
	};
	AttentionVisibleWalk visible{map_row};
	if constexpr (MASK) t_first = visible.next(t_first, t_last);
	if (t_first <= t_last)
	{
		fetch(kp, t_first);
		__syncthreads();                            // (the query block before has been read by everybody)
#pragma unroll
		for (int i = 0; i < VPT; ++i) put(false, i);
		fetch(vp, t_first);
	}
	// Each product is a sequence of steps: a fragment (of V: of two column blocks), the third, second and first part in turn, and its one, two
	// or three products; a step's fragments are read some steps ahead, and the tile that the other product needs next is cut into the
	// planes behind the steps of the second half, its loads having had the first.  Neighbouring MFMAs use different accumulators.
	constexpr int kStepsQ = 3 * KS * KB, kAheadQ = 4, kStepsV = 3 * DC / 2, kAheadV = 2;
	static_assert(DC % 2 == 0 && KB == 2, "column blocks in pairs; one 32-key step");
	bf16x8_t frag[4];
	auto read_k = [&](int f) {
		const int u = f / 3, p = 2 - f % 3, st = u / KB, kb = u % KB;
		frag[f % kAheadQ] = *reinterpret_cast<const bf16x8_t*>(lds + p * L::kPlaneK + (16 * kb + n) * L::kPitchK + (32 * st + 8 * g) * 2);
	};
	// slot (g, j) of the 32-key step is key 16 (j / 4) + 4 g + j % 4
	auto read_v = [&](int f) {
		const int c = 2 * (f / 3), p = 2 - f % 3;
		typedef __attribute__((address_space(3))) short4_t* LdsShort4;
#pragma unroll
		for (int i = 0; i < 2; ++i)
		{
			const char* src = lds + 3 * L::kPlaneK + p * L::kPlaneV + (4 * g + (n >> 2)) * L::kPitchV + (16 * (c + i) + 4 * (n & 3)) * 2;
			const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4)(src));
			const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4)(src + 16 * L::kPitchV));
			frag[2 * (f % kAheadV) + i] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
		}
	};
	// piece of the staged tile that goes behind step f of `steps`, or -1
	auto piece_at = [](int f, int steps) {
		const int half = steps / 2, every = half / VPT;
		return f >= half && (f - half) % every == 0 && (f - half) / every < VPT ? (f - half) / every : -1;
	};
	static_assert(kStepsQ / 2 >= VPT && kStepsV / 2 >= VPT, "steps for the pieces");
	int t_next = 0;
	for (int t = t_first; t <= t_last; t = t_next)
	{
		if constexpr (MASK) t_next = visible.next(t + 1, t_last);
		else t_next = t + 1;
		__syncthreads();                            // K(t) is complete, V of the tile before has been read by everybody
		if constexpr (MASK) load_mask(t);
		// ---- S^T = K Q^T ----
		float4_t s[KB];
#pragma unroll
		for (int kb = 0; kb < KB; ++kb) s[kb] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
		for (int f = 0; f < kAheadQ; ++f) read_k(f);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int f = 0; f < kStepsQ; ++f)
		{
			const int u = f / 3, st = u / KB, kb = u % KB;
#pragma unroll
			for (int x = f % 3; x >= 0; --x) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag[f % kAheadQ], qf[x][st], s[kb], 0, 0, 0);
			if (f + kAheadQ < kStepsQ) read_k(f + kAheadQ);
			if (piece_at(f, kStepsQ) >= 0) put(true, piece_at(f, kStepsQ));
			__builtin_amdgcn_sched_barrier(0);
		}
		// ---- online softmax: score (kb, r) of this lane is key 16 kb + 4 g + r ----
		const int tile_key0 = t * KT;
		const bool interior = tile_key0 >= all_lo && tile_key0 + KT - 1 <= all_hi;   // wave-uniform
		float z[4 * KB];
#pragma unroll
		for (int i = 0; i < 4 * KB; ++i)
		{
			z[i] = logit2<SOFTCAP>(s[i / 4][i % 4], a.k_in, a.k_cap);
			if constexpr (MASK) z[i] += mk[MASK ? i / 4 : 0][i % 4] * kLog2e;
		}
		if (!MASK && !interior)                     // (a mask's values past the last key hide them)
		{
			int row = n;
			asm volatile("" : "+v"(row));           // (found anew at each such tile: two registers)
			row += wq0;
			const int vis_hi = a.causal && row + a.diag < a.n_k - 1 ? row + a.diag : a.n_k - 1;
			const int vis_lo = a.window > 0 ? row + a.diag - a.window + 1 : 0;
#pragma unroll
			for (int i = 0; i < 4 * KB; ++i)
			{
				const int key = tile_key0 + 16 * (i / 4) + 4 * g + i % 4;
				z[i] = (key >= vis_lo && key <= vis_hi) ? z[i] : -INFINITY;
			}
		}
		float mt = z[0];
#pragma unroll
		for (int i = 1; i < 4 * KB; ++i) mt = fmaxf(mt, z[i]);
		mt = max_over_lane_rows(mt);
		const float m_new = fmaxf(m_run, mt);
		const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;   // nothing visible so far: every term is exp2(-inf) = 0
		// the running maximum settles after a few tiles; when no query of the wave raised it, the
		// rescale factor is 1 everywhere and the pass over the accumulators is skipped
		if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0)
		{
			const float corr = fast_exp2(m_run - m_safe);
			l_run *= corr;
#pragma unroll
			for (int c = 0; c < DC; ++c) o[c] *= corr;
		}
		m_run = m_new;
		float psum[2] = {0.0f, 0.0f};
		bf16x8_t pf[3];
		uint4_t w[3];
#pragma unroll
		for (int j = 0; j < 8; j += 2)
		{
			const float p0 = fast_exp2(z[j] - m_safe), p1 = fast_exp2(z[j + 1] - m_safe);
			psum[0] += p0;
			psum[1] += p1;
			unsigned parts[3];
			split_pair(p0, p1, parts);
#pragma unroll
			for (int p = 0; p < 3; ++p) w[p][j / 2] = parts[p];
		}
#pragma unroll
		for (int p = 0; p < 3; ++p) pf[p] = __builtin_bit_cast(bf16x8_t, w[p]);
		l_run += psum[0] + psum[1];
		// (behind the last tile: that tile once more, of no consequence)
		const int t_load = t_next <= t_last ? t_next : t;
		fetch(kp, t_load);
		__syncthreads();                            // V(t) is complete, K(t) has been read by everybody
		// ---- O^T += V^T P^T ----
#pragma unroll
		for (int f = 0; f < kAheadV; ++f) read_v(f);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int f = 0; f < kStepsV; ++f)
		{
			const int c = 2 * (f / 3);
#pragma unroll
			for (int x = f % 3; x >= 0; --x)
#pragma unroll
				for (int i = 0; i < 2; ++i) o[c + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag[2 * (f % kAheadV) + i], pf[x], o[c + i], 0, 0, 0);
			if (f + kAheadV < kStepsV) read_v(f + kAheadV);
			if (piece_at(f, kStepsV) >= 0) put(false, piece_at(f, kStepsV));
			__builtin_amdgcn_sched_barrier(0);
		}
		fetch(vp, t_load);
	}

	// ---- normalise and store: lane (n, g) holds y[row][16 c + 4 g .. + 3] ----
	const float l = sum_over_lane_rows(l_run);
	float all = l;                                  // not finite where anything that entered it is not
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int r = 0; r < 4; ++r) all = fmaf(o[c][r], 0.0f, all);
	if (any_of_block<THREADS / kWaveSize>(rest.lost() || !(fabsf(all) < INFINITY), lds, wave)) return false;
	if (q_row >= a.n_q) return true;
	if (partial != nullptr)
	{
		// unnormalised accumulators, running maximum and sum of this part of the keys
		float* dst = partial + (int64_t)(q_row - q0) * (D + 2);
#pragma unroll
		for (int c = 0; c < DC; ++c) *reinterpret_cast<WsFloat4*>(dst + 16 * c + 4 * g) = o[c];
		if (g == 0)
		{
			dst[D] = m_run;
			dst[D + 1] = l;
		}
		return true;
	}
	const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
	for (int c = 0; c < DC; ++c) *reinterpret_cast<float4_t*>(yp + (int64_t)q_row * D + 16 * c + 4 * g) = o[c] * inv;
	return true;
}

// The launch of that form: every block finds its query block and the tiles of it, or (BALANCED: MASK with a map) its range of the launch's
// set tiles (attention_balance.hpp), and walks it query block after query block.  One range per resident block: with two for each CU 16 heads x 2500 x 128 215 us, with one 199.
template <int D, bool SOFTCAP, bool MASK, bool BALANCED>
__global__ __launch_bounds__(split_threads(D, MASK), 2) void sdp_attention_fwd_f32_split_kernel(const AttnArgsF32 a, const AttnWalk walk, const AttnBalance balance)
{
	static_assert(!BALANCED || MASK, "ranges of a mask's set tiles");
	extern __shared__ __align__(16) char lds_raw[];
	const auto attend = [&](int bh, int q_block, int t_first, int t_last, const unsigned long long* map_row, float* partial) {
		if constexpr (split_narrow(D, MASK))
		{
			if (attend_f32_split16<D, SOFTCAP, MASK>(a, lds_raw, bh, q_block, t_first, t_last, map_row, partial)) return;
		}
		else if (attend_f32_split<D, SOFTCAP, MASK>(a, lds_raw, bh, q_block, t_first, t_last, map_row, partial)) return;
		// (16 queries to a wave: with four waves the block's queries in two halves)
		constexpr int kWaves = split_threads(D, MASK) / 64, kHalves = kSplitQueries / (16 * kWaves);
		for (int i = 0; i < kHalves; ++i)
		{
			__syncthreads();
			// (a value that is not finite reaches every query of a block whose tiles hold its key: those of each half, as where blocks have 64 queries)
			int first = t_first, last = t_last;
			if constexpr (kHalves > 1 && !MASK)
			{
				int of_half_first, of_half_last;
				visible_tiles_f32<16 * kWaves, kSplitKeys>(a, kHalves * q_block + i, of_half_first, of_half_last);
				first = max(first, of_half_first);
				last = min(last, of_half_last);
			}
			attend_f32<D, SOFTCAP, kWaves, kSplitKeys, D == 256, MASK>(a, reinterpret_cast<float*>(lds_raw), bh, kHalves * q_block + i, first, last, map_row,
			                                                           partial ? partial + i * (16 * kWaves) * (D + 2) : nullptr);
		}
	};
	if constexpr (!BALANCED)
	{
		int bh, q_block, t_first, t_last;
		const unsigned long long* map_row;
		float* partial;
		if (!attention_block_f32<D, kSplitQueries, kSplitKeys, MASK>(a, walk, bh, q_block, t_first, t_last, map_row, partial)) return;
		attend(bh, q_block, t_first, t_last, map_row, partial);
	}
	else
	{
		constexpr int64_t kPartialFloats = (int64_t)kSplitQueries * (D + 2);
		// (a run of ranges to each XCD: neighbours share a head's keys)
		const int64_t range = balance.ranges % 8 == 0 ? (int64_t)(blockIdx.x % 8) * (balance.ranges / 8) + blockIdx.x / 8 : blockIdx.x;
		const BalanceScan scan(a.tile_map, balance);
		int64_t at = range * scan.per;
		const int64_t range_end = min(at + scan.per, (int64_t)scan.per_head * balance.heads);
		if (at >= range_end) return;
		int bh = (int)(at / scan.per_head), q_block, first;
		const int x = (int)(at - (int64_t)bh * scan.per_head);
		scan.locate(a.tile_map, balance, x, q_block, first);
		q_block = __builtin_amdgcn_readfirstlane(q_block);
		int in_block = __builtin_amdgcn_readfirstlane(x - first);              // tiles of the query block in front of the range
		float* slot = a.partials + 2 * range * kPartialFloats;       // of the query block that the range starts inside; the next one's
		for (;;)
		{
			const unsigned long long* const map_row = a.tile_map + (int64_t)q_block * a.map_words;
			// (the same in every lane, which the compiler does not see by itself)
			const int count = __builtin_amdgcn_readfirstlane(balance_tiles(a.tile_map, balance, q_block));
			const int taken = __builtin_amdgcn_readfirstlane((int)min((int64_t)(count - in_block), range_end - at));
			const int t_first = __builtin_amdgcn_readfirstlane(balance_nth_tile(map_row, balance.words, in_block));
			int t_last = __builtin_amdgcn_readfirstlane(balance_nth_tile(map_row, balance.words, in_block + taken - 1));
			if (t_first > (a.n_k - 1) / kSplitKeys) t_last = t_first - 1;       // (no set tile at all: zeros)
			attend(bh, q_block, t_first, t_last, map_row, taken == count ? nullptr : slot);
			at += taken;
			if (at >= range_end) return;
			in_block = 0;
			slot = a.partials + (2 * range + 1) * kPartialFloats;
			if (++q_block == balance.q_blocks)
			{
				q_block = 0;
				++bh;
			}
		}
	}
}

template <int D, bool MASK>
constexpr int split_lds_bytes()
{
	constexpr int kPlainBytes = AttnLdsF32<D, kSplitKeys>::kStageFloats * 4 * (D == 256 ? 2 : 1);     // (the form that takes over from it)
	constexpr int kPlanes = AttnLdsSplit<D, split_narrow(D, MASK)>::kBytes;
	return kPlanes > kPlainBytes ? kPlanes : kPlainBytes;
}

}  // namespace

}  // namespace anygpu

#include "attention_f32_kwave.hpp"

namespace anygpu {

namespace {

// One launch over query blocks of QUERIES and tiles of KEYS, with the merge of whatever goes out in parts of its key range.  resident: as plan_attention_split
// takes it.
template <int D, int QUERIES, int KEYS, typename Launch>
hipError_t launch_blocks_f32(AttnArgsF32& args, int64_t batch_heads, hipStream_t stream, int resident, Launch launch)
{
	const int64_t q_blocks = (args.n_q + QUERIES - 1) / QUERIES;
	const AttnSplitPlan plan = plan_attention_split(args.n_q, args.n_k, args.causal, args.diag, args.window, batch_heads, QUERIES, KEYS, D,
	                                                band::workspace_capacity(stream), resident);
	// (or, with too few query blocks for the chip, every block in several parts of its key range)
	const int64_t parts_all = plan.n_split > 0 ? 1 : plan_attention_parts(args.n_q, args.n_k, args.causal, args.diag, batch_heads, QUERIES, KEYS, D,
	                                                                        band::workspace_capacity(stream));
	args.partials = nullptr;
	if (plan.n_split > 0 || parts_all > 1)
	{
		const hipError_t ws_err = band::workspace_acquire(stream, &args.partials);
		if (ws_err != hipSuccess) return ws_err;
	}
	const AttnWalk walk = make_attn_walk(q_blocks, batch_heads, args.q_per_kv, plan.n_split, plan.n_big, parts_all);
	if (attn_walk_blocks(walk) > 0x7FFFFFFFLL) return hipErrorInvalidValue;
	const hipError_t err = launch(walk);
	if (err != hipSuccess || walk.n_split == 0) return err;
	const int64_t items = batch_heads * walk.n_split * QUERIES * (D / 4);
	sdp_attention_merge_halves_kernel<D, float><<<dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream>>>(
		args.partials, args.y, args.n_q, (int)q_blocks, walk.n_split, QUERIES, parts_all > 1 ? (int)parts_all : 2);
	return hipGetLastError();
}

// blocks of the bf16 form that a CU holds (a mask tensor's have no lengths that are known ahead: 0)
template <int D, bool MASK>
constexpr int kSplitResident = MASK ? 0 : split_narrow(D, MASK) ? 1 : 2;

template <int D, bool SOFTCAP, bool MASK>
hipError_t launch_split_f32(AttnArgsF32& args, int64_t batch_heads, hipStream_t stream)
{
	return launch_blocks_f32<D, kSplitQueries, kSplitKeys>(args, batch_heads, stream, kSplitResident<D, MASK>, [&](const AttnWalk& walk) {
		auto kernel = sdp_attention_fwd_f32_split_kernel<D, SOFTCAP, MASK, false>;
		static std::atomic<uint64_t> configured_devices{0};
		const hipError_t err = grant_lds(kernel, split_lds_bytes<D, MASK>(), configured_devices);
		if (err != hipSuccess) return err;
		kernel<<<dim3((unsigned)attn_walk_blocks(walk)), dim3(split_threads(D, MASK)), split_lds_bytes<D, MASK>(), stream>>>(args, walk, AttnBalance{});
		return hipGetLastError();
	});
}

template <int D, bool SOFTCAP, bool MASK>
hipError_t launch_plain_f32(AttnArgsF32& args, int64_t batch_heads, hipStream_t stream)
{
	// head dimension 256: 8 waves (two per SIMD) on tiles of 32 keys in two stages, 130 KB, one block per CU.  Two
	// alternatives with two blocks of 4 waves per CU, for a better balance of long and short blocks under the causal
	// rule, measured 5 - 12 % slower: tiles of 16 keys, and one K and one V buffer refilled in turn.
	constexpr bool DIRECT = (D == 256);
	constexpr int WAVES = DIRECT ? 8 : 4;
	constexpr int KT = DIRECT ? 32 : 64;
	constexpr int kLdsBytes = AttnLdsF32<D, KT>::kStageFloats * 4 * (DIRECT ? 2 : 1);
	return launch_blocks_f32<D, 16 * WAVES, KT>(args, batch_heads, stream, 0, [&](const AttnWalk& walk) {
		auto kernel = sdp_attention_fwd_f32_kernel<D, SOFTCAP, WAVES, KT, DIRECT, MASK>;
		static std::atomic<uint64_t> configured_devices{0};
		const hipError_t err = grant_lds(kernel, kLdsBytes, configured_devices);
		if (err != hipSuccess) return err;
		kernel<<<dim3((unsigned)attn_walk_blocks(walk)), dim3(64 * WAVES), kLdsBytes, stream>>>(args, walk);
		return hipGetLastError();
	});
}

// Head dimensions 64 and 128, index rules: whether the blocks of 128 queries have enough tiles of 32 keys each (`longest`), which a short window
// does not leave them, nor a long key range that goes out in many parts (in tiles of 32 keys twice as many as in the other form's of 64).
// us, fp32 matrix instruction / bf16 parts, causal:
//   * Whole blocks under a window: 24 heads x 700 x 64, window 500 (20 tiles) 30.3 / 38.4, 16 / 8 x 1500, window 1000 (36 tiles) 64.3 / 44.6; with a block
//     for every CU from 5 tiles on (32 x 4000 x 64, window 30 50.8 / 38.8).
//   * In parts: 16 / 8 x 700 x 64, window 100 (8 tiles in 5 parts) 12.6 / 23.0, window 500 (20 in 5) 28.3 / 25.0, 4 x 300 x 3000 x 64 (94 in 23) 27.1 / 30.8, 2 x
//     300 x 6000 x 64 (188 in 47) 34.7 / 46.0, x 128 48.4 / 55.6, 16 / 8 x 700 x 128, window 100 21.1 / 30.2, window 300 (14 in 5) 35.5 / 32.2.
template <int D>
bool attention_split_fills(const AttnArgsF32& args, int64_t batch_heads)
{
	constexpr size_t kRoom = band::kBandPartialBytes;      // the library's own workspace, whatever the stream has: the form does not depend on it
	const int64_t q_blocks = (args.n_q + kSplitQueries - 1) / kSplitQueries;
	int64_t longest = 0;
	for (int64_t b = q_blocks - 1, step = q_blocks / 64 + 1; b >= 0; b = args.window > 0 ? b - step : -1)
		longest = std::max(longest, attention_block_tiles(b, args.n_q, args.n_k, args.causal, args.diag, args.window, kSplitQueries, kSplitKeys));
	const AttnSplitPlan plan = plan_attention_split(args.n_q, args.n_k, args.causal, args.diag, args.window, batch_heads, kSplitQueries, kSplitKeys, D, kRoom, 2);
	const int64_t parts = plan.n_split > 0 ? 1 : plan_attention_parts(args.n_q, args.n_k, args.causal, args.diag, batch_heads, kSplitQueries, kSplitKeys, D, kRoom);
	if (parts == 1) return args.window == 0 || longest >= 21 || (longest >= 5 && q_blocks * batch_heads >= device_cu_count());
	if (longest < 11) return false;
	if (D == 64) return longest >= 8 * parts || (parts <= 32 && 5 * longest >= 21 * parts);
	return longest > 4 * parts || (parts <= 16 && 2 * longest >= 5 * parts);
}

// Whether the launch takes the bf16 parts (us, fp32 matrix instruction / bf16 parts).
//   * Index rules: at head dimension 256 always (8 heads x 64 x 64 21.7 / 15.6, 8 / 4 x 8192, window 4096 1711 / 1039; 4 x 700, window 1 30.0 / 25.1);
//     at 64 and 128, where the other form has blocks of 64 queries, from some ten tiles on (attention_split_fills; 32 heads x 1000 x 128 153 /
//     109, 400 41.6 / 38.3, 64 heads x 400 x 64 causal 28.7 / 25.9; but 32 x 150 x 128 18.1 / 19.3, 64 x 250 x 64 15.2 / 19.9), at 64 for more than a
//     block of queries (8 x 64 x 4000 28.8 / 34.1, 32 x 100 x 1000 21.1 / 22.6).
//   * A mask tensor: with its visible-tile map, as there is no test of a tile by each wave.  The pass that makes the map and a range's start cost
//     20 - 30 us: head dimension 256 from 150 K mask values on (causal 8 heads x 250 x 600 58.8 / 57.2, 400 58.4 / 54.8, 2000 231 / 139); 128 from 6 M values
//     over all heads (8 x 100 x 8000 87.5 / 69.1, 8 x 1000 60.8 / 44.9; but 8 x 797 39.0 / 42.6, 32 x 250 x 600 39.5 / 43.7); 64 from 11 M in masks of
//     600 K (8 x 830 x 1800 51.3 / 48.3, 32 x 797 55.7 / 51.1; but 8 x 1000 33.1 / 37.8, 32 x 400 26.6 / 37.3).
template <int D, bool MASK>
bool attention_split_wanted(const AttnArgsF32& args, int64_t batch_heads)
{
	if constexpr (MASK)
	{
		const int64_t values = (int64_t)args.n_q * args.n_k;
		if (args.mask_stride > kSplitMaskStride) return false;
		if (D == 64) return values >= 600 * 1000 && batch_heads * values >= 11 * 1000 * 1000;
		return values >= 150 * 1000 && (D == 256 || batch_heads * values >= 6 * 1000 * 1000);
	}
	else return D == 256 || (args.n_k >= 350 && (D == 128 || args.n_q > 128) && attention_split_fills<D>(args, batch_heads));
}

template <int D, bool SOFTCAP, bool MASK, int WAVES>
hipError_t launch_kwave_variant_f32(const AttnArgsF32& args, int64_t batch_heads, hipStream_t stream)
{
	constexpr int kLdsBytes = kKeyWaveLdsBytes<D, WAVES>;
	const auto kernel = sdp_attention_fwd_f32_kwave_kernel<D, SOFTCAP, MASK, WAVES>;
	(void)hipGetLastError();
	static std::atomic<uint64_t> configured_devices{0};
	const hipError_t lds_err = grant_lds(kernel, kLdsBytes, configured_devices);
	if (lds_err != hipSuccess) return lds_err;
	const AttnWalk walk = make_attn_walk((args.n_q + kKeyWaveRows - 1) / kKeyWaveRows, batch_heads, args.q_per_kv);
	if (attn_walk_blocks(walk) > 0x7FFFFFFFLL) return hipErrorInvalidValue;
	kernel<<<dim3((unsigned)attn_walk_blocks(walk)), dim3(64 * WAVES), kLdsBytes, stream>>>(args, walk);
	return hipGetLastError();
}

template <int D, bool SOFTCAP, bool MASK>
hipError_t launch_kwave_f32(const AttnArgsF32& args, int64_t batch_heads, hipStream_t stream)
{
	if constexpr (D != 256)
	{
		if (batch_heads * ((args.n_q + kKeyWaveRows - 1) / kKeyWaveRows) > device_cu_count()) return launch_kwave_variant_f32<D, SOFTCAP, MASK, 4>(args, batch_heads, stream);
	}
	return launch_kwave_variant_f32<D, SOFTCAP, MASK, 8>(args, batch_heads, stream);
}

template <int D, bool SOFTCAP, bool MASK>
hipError_t launch_variant_f32(const AttnArgsF32& args_in, int64_t batch_heads, hipStream_t stream)
{
	(void)hipGetLastError();
	AttnArgsF32 args = args_in;
	args.tile_map = nullptr;
	args.map_words = 0;
	if (!(MASK && attention_mask_map_set()) &&
	    attention_kwave_wanted_f32(D, MASK, batch_heads, args.n_q, args.n_k, args.causal, args.diag, args.window, device_cu_count()))
		return launch_kwave_f32<D, SOFTCAP, MASK>(args, batch_heads, stream);
	const bool split = attention_split_wanted<D, MASK>(args, batch_heads);
	if constexpr (!MASK) return split ? launch_split_f32<D, SOFTCAP, false>(args, batch_heads, stream) : launch_plain_f32<D, SOFTCAP, false>(args, batch_heads, stream);
	else
	{
		// The visible-tile map of the mask, at the front of the stream's workspace (partial results go behind it), for large masks and long key
		// ranges (attention_mask_map_wanted), and left out where the stream has no workspace to offer (a capture without a
		// caller's workspace).
		const int queries = split || D == 256 ? kSplitQueries : 64, keys = split || D == 256 ? kSplitKeys : 64;
		const int64_t q_blocks = (args.n_q + queries - 1) / queries, words = attention_tile_map_words(args.n_k, keys);
		const size_t map_bytes = ((size_t)(q_blocks * words) * sizeof(unsigned long long) + 255) / 256 * 256;
		if (!attention_mask_map_wanted(args.n_q, args.n_k, split) || band::workspace_capacity(stream) < map_bytes + (1u << 16))
			return launch_plain_f32<D, SOFTCAP, true>(args, batch_heads, stream);
		// Up to four rounds of query blocks: the launch's set tiles in equal shares, whose partial results may need more than the library's own
		// workspace holds to begin with (it grows for them as it does for operand copies, eager launches only).
		const int64_t ranges = (split_narrow(D, true) ? 1 : 2) * (int64_t)device_cu_count();
		const size_t shares_bytes = map_bytes + (size_t)(2 * ranges) * kSplitQueries * (D + 2) * sizeof(float);
		const bool balanced = split && q_blocks * batch_heads < 4 * ranges && band::workspace_copy_capacity(stream) >= shares_bytes;
		float* front = nullptr;
		hipError_t e = band::workspace_acquire(stream, &front, balanced ? shares_bytes : 0);
		if (e != hipSuccess) return e;
		unsigned long long* map = reinterpret_cast<unsigned long long*>(front);
		e = launch_attention_mask_tile_map(args.mask, args.mask_stride, args.n_q, args.n_k, queries, keys, map, stream);
		if (e != hipSuccess) return e;
		args.tile_map = map;
		args.map_words = (int)words;
		if (!balanced)
		{
			const band::WorkspaceReserve map_hold(map_bytes);
			return split ? launch_split_f32<D, SOFTCAP, true>(args, batch_heads, stream) : launch_plain_f32<D, SOFTCAP, true>(args, batch_heads, stream);
		}
		args.partials = reinterpret_cast<float*>(reinterpret_cast<char*>(front) + map_bytes);
		const AttnBalance balance{(int)ranges, (int)batch_heads, (int)q_blocks, (int)words, 4};
		auto kernel = sdp_attention_fwd_f32_split_kernel<D, SOFTCAP, true, true>;
		static std::atomic<uint64_t> configured_devices{0};
		e = grant_lds(kernel, split_lds_bytes<D, MASK>(), configured_devices);
		if (e != hipSuccess) return e;
		kernel<<<dim3((unsigned)ranges), dim3(split_threads(D, MASK)), split_lds_bytes<D, MASK>(), stream>>>(args, AttnWalk{}, balance);
		e = hipGetLastError();
		if (e != hipSuccess) return e;
		sdp_attention_merge_ranges_kernel<D, float><<<dim3(kSplitQueries * (D / 4) / 256, (unsigned)q_blocks, (unsigned)batch_heads), dim3(256), 0, stream>>>(
			args.partials, args.y, args.n_q, kSplitQueries, map, balance);
		return hipGetLastError();
	}
}

// ---------------------------------------------------------------------------------------------
// Decode form: very few queries per head (a generation step), long key range: the KEYS are split.
//
// The q_per_kv query heads that share a key / value head, times the n_q queries of each, are the (at most 16)
// rows of one 16-query MFMA block, so K and V of a head are read once for all of them.  Pass 1: one wave per
// (key / value head, split of the visible key range) walks its keys in tiles of 16.  Both operands come straight
// from global memory in MFMA operand layout, no LDS: the K vectors as in the fused kernel, and the V vectors with
// the permuted accumulators described at the top (a lane loads four consecutive columns of a V row).  The wave
// leaves its running maximum, sum and unnormalised accumulators in the workspace.  Pass 2 merges the splits of a
// row: M = max m_i, y = sum o_i 2^(m_i - M) / sum l_i 2^(m_i - M).
// Workspace per (head, split, row): head_dim accumulators + maximum + sum, fp32.
// ---------------------------------------------------------------------------------------------
constexpr int kDecodeKeysPerTile = 16;

struct DecodeArgsF32
{
	AttnArgsF32 a;
	float* ws;              // [kv_heads][splits][rows][D + 2]
	int rows;               // q_per_kv * n_q
	int groups;             // of 16 rows: a wave each
	int splits;
	int tiles_per_split;
	int t_first, t_last;    // visible key tiles of the group
};

template <int D, bool SOFTCAP>
__global__ __launch_bounds__(64) void sdp_decode_partial_f32_kernel(const DecodeArgsF32 da)
{
	const AttnArgsF32& a = da.a;
	constexpr int KS = D / 16, DC = D / 64;
	const int lane = threadIdx.x;
	const int n = lane & 15, g = lane >> 4;
	int split, group;
	if (!decode_locate(da.groups, da.splits, split, group)) return;
	const int kvh = blockIdx.y;
	const float* qp = a.q + (int64_t)kvh * da.rows * D;  // the rows of a key / value head are contiguous: [q_per_kv][n_q][D]
	const int row = kDecodeRowsPerWave * group + n;        // this lane's row among them
	const float* kp = a.k + (int64_t)kvh * a.n_k * D;
	const float* vp = a.v + (int64_t)kvh * a.n_k * D;

	const bool row_ok = row < da.rows;
	const int q_idx = row_ok ? row % a.n_q : 0;             // position of this lane's row among the n_q queries
	float4_t qf[KS];
#pragma unroll
	for (int s = 0; s < KS; ++s)
	{
		float4_t val = {0.0f, 0.0f, 0.0f, 0.0f};
		if (row_ok) val = *reinterpret_cast<const float4_t*>(qp + (int64_t)row * D + 16 * s + 4 * g);
		qf[s] = val;
	}
	int vis_hi = a.causal ? q_idx + a.diag : a.n_k - 1;
	if (vis_hi > a.n_k - 1) vis_hi = a.n_k - 1;
	if (!row_ok) vis_hi = -1;                              // padding rows see nothing
	const int vis_lo = a.window > 0 ? q_idx + a.diag - a.window + 1 : 0;

	float m_run = -INFINITY, l_run = 0.0f;
	float4_t o[DC][4];
#pragma unroll
	for (int c = 0; c < DC; ++c)
#pragma unroll
		for (int e = 0; e < 4; ++e) o[c][e] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

	const int t0 = da.t_first + split * da.tiles_per_split;
	int t1 = t0 + da.tiles_per_split - 1;
	if (t1 > da.t_last) t1 = da.t_last;
	// All loads of a tile are issued before the first use; keys past the end are replaced by the last one (their
	// scores are masked).  A K load instruction covers half of each 128-byte line it touches, so it stays a plain
	// load (the other half is the next instruction's); a V load covers whole lines and is non-temporal.
	auto fetch = [&](float4_t (&kd)[KS], float4_t (&vd)[4][DC], int key0) {
		{
			int key = key0 + n;
			key = key < a.n_k ? key : a.n_k - 1;
#pragma unroll
			for (int st = 0; st < KS; ++st) kd[st] = *reinterpret_cast<const float4_t*>(kp + (int64_t)key * D + 16 * st + 4 * g);
		}
#pragma unroll
		for (int r = 0; r < 4; ++r)
		{
			int key = key0 + 4 * g + r;
			key = key < a.n_k ? key : a.n_k - 1;
#pragma unroll
			for (int c = 0; c < DC; ++c)
				vd[r][c] = __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(vp + (int64_t)key * D + 64 * c + 4 * n));
		}
	};
	auto consume = [&](const float4_t (&kd)[KS], const float4_t (&vd)[4][DC], int key0) {
		float4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
		for (int st = 0; st < KS; ++st)
#pragma unroll
			for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kd[st][e], qf[st][e], s, 0, 0, 0);

		float z[4];
		float mt = -INFINITY;
#pragma unroll
		for (int r = 0; r < 4; ++r)
		{
			const int key = key0 + 4 * g + r;
			const float zz = logit2<SOFTCAP>(s[r], a.k_in, a.k_cap);
			z[r] = (key >= vis_lo && key <= vis_hi) ? zz : -INFINITY;
			mt = fmaxf(mt, z[r]);
		}
		mt = max_over_lane_rows(mt);
		const float m_new = fmaxf(m_run, mt);
		const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;
		const float corr = fast_exp2(m_run - m_safe);
		float psum = 0.0f;
		float p[4];
#pragma unroll
		for (int r = 0; r < 4; ++r)
		{
			p[r] = fast_exp2(z[r] - m_safe);
			psum += p[r];
		}
		l_run = l_run * corr + psum;
		m_run = m_new;
#pragma unroll
		for (int c = 0; c < DC; ++c)
#pragma unroll
			for (int e = 0; e < 4; ++e) o[c][e] *= corr;
#pragma unroll
		for (int r = 0; r < 4; ++r)
#pragma unroll
			for (int c = 0; c < DC; ++c)
#pragma unroll
				for (int e = 0; e < 4; ++e) o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vd[r][c][e], p[r], o[c][e], 0, 0, 0);
	};
	if constexpr (D <= 128)
	{
		// two register buffers: the loads of tile t + 1 are in flight while tile t is multiplied (at head_dim 256 a
		// second buffer does not fit beside the accumulators)
		float4_t kf[2][KS], vf[2][4][DC];
		if (t0 <= t1) fetch(kf[0], vf[0], t0 * kDecodeKeysPerTile);
		for (int t = t0; t <= t1; t += 2)
		{
			if (t + 1 <= t1) fetch(kf[1], vf[1], (t + 1) * kDecodeKeysPerTile);
			__builtin_amdgcn_sched_barrier(0);
			consume(kf[0], vf[0], t * kDecodeKeysPerTile);
			if (t + 1 <= t1)
			{
				if (t + 2 <= t1) fetch(kf[0], vf[0], (t + 2) * kDecodeKeysPerTile);
				__builtin_amdgcn_sched_barrier(0);
				consume(kf[1], vf[1], (t + 1) * kDecodeKeysPerTile);
			}
		}
	}
	else
	{
		for (int t = t0; t <= t1; ++t)
		{
			float4_t kf[KS], vf[4][DC];
			fetch(kf, vf, t * kDecodeKeysPerTile);
			consume(kf, vf, t * kDecodeKeysPerTile);
		}
	}

	// partial result of this split: register r of accumulator (c, e) is o[row n][64 c + 16 g + 4 r + e]
	float l = l_run;
	l += __shfl_xor(l, 16);
	l += __shfl_xor(l, 32);
	if (row_ok)
	{
		float* dst = da.ws + (((int64_t)kvh * da.splits + split) * da.rows + row) * (D + 2);
#pragma unroll
		for (int c = 0; c < DC; ++c)
#pragma unroll
			for (int r = 0; r < 4; ++r)
				*reinterpret_cast<WsFloat4*>(dst + 64 * c + 16 * g + 4 * r) = float4_t{o[c][0][r], o[c][1][r], o[c][2][r], o[c][3][r]};
		if (g == 0)
		{
			dst[D] = m_run;
			dst[D + 1] = l;
		}
	}
}

template <int D, bool SOFTCAP>
hipError_t launch_decode_variant_f32(const DecodeArgsF32& da, int64_t kv_heads, hipStream_t stream)
{
	(void)hipGetLastError();
	sdp_decode_partial_f32_kernel<D, SOFTCAP><<<dim3(decode_blocks(da.groups, da.splits), (unsigned)kv_heads), dim3(64), 0, stream>>>(da);
	hipError_t e = hipGetLastError();
	if (e != hipSuccess) return e;
	sdp_decode_merge_kernel<D, float><<<dim3((unsigned)da.rows, (unsigned)kv_heads), dim3(256), 0, stream>>>(da.ws, da.a.y, da.rows, da.splits);
	return hipGetLastError();
}

}  // namespace

bool sdp_attention_fwd_f32_supports(int64_t head_dim)
{
	return head_dim == 64 || head_dim == 128 || head_dim == 256;
}

hipError_t launch_sdp_attention_fwd_f32(const float* q, const float* k, const float* v, float* y,
                                        int64_t batch_heads, int64_t q_per_kv, int64_t n_q, int64_t n_k, int64_t head_dim,
                                        float alpha, float softcap, int causal, int64_t window, hipStream_t stream,
                                        const float* mask, int64_t mask_stride)
{
	if (batch_heads == 0 || n_q == 0) return hipSuccess;
	AttnArgsF32 args;
	args.q = q;
	args.k = k;
	args.v = v;
	args.y = y;
	args.n_q = (int)n_q;
	args.n_k = (int)n_k;
	args.q_per_kv = (int)q_per_kv;
	args.diag = (int)(n_k - n_q);
	args.causal = causal ? 1 : 0;
	args.window = (int)window;
	const bool capped = softcap != 0.0f;
	args.k_in = capped ? 2.0f * kLog2e * alpha / softcap : alpha * kLog2e;
	args.k_cap = capped ? softcap * kLog2e : 0.0f;
	args.partials = nullptr;
	args.mask = mask;
	args.mask_stride = mask_stride;
#define ANYGPU_ATTN_F32_DIM(DIM) \
	if (mask != nullptr) \
		return capped ? launch_variant_f32<DIM, true, true>(args, batch_heads, stream) : launch_variant_f32<DIM, false, true>(args, batch_heads, stream); \
	return capped ? launch_variant_f32<DIM, true, false>(args, batch_heads, stream) : launch_variant_f32<DIM, false, false>(args, batch_heads, stream)
	switch (head_dim)
	{
	case 64: ANYGPU_ATTN_F32_DIM(64);
	case 128: ANYGPU_ATTN_F32_DIM(128);
	default: ANYGPU_ATTN_F32_DIM(256);
	}
#undef ANYGPU_ATTN_F32_DIM
}

bool sdp_attention_decode_f32_supports(int64_t q_per_kv, int64_t n_q, int64_t head_dim)
{
	return sdp_attention_fwd_f32_supports(head_dim) && q_per_kv >= 1 && n_q >= 1 && q_per_kv * n_q <= kDecodeMaxRows;
}

int64_t sdp_attention_decode_f32_workspace_bytes(int64_t batch_heads, int64_t q_per_kv, int64_t n_q, int64_t n_k, int64_t head_dim,
                                                 int causal, int64_t window)
{
	if (batch_heads == 0 || n_q == 0) return 0;
	const int64_t kv_heads = batch_heads / q_per_kv;
	const DecodePlan p = plan_decode(kv_heads * ((q_per_kv * n_q + kDecodeRowsPerWave - 1) / kDecodeRowsPerWave), n_q, n_k, causal, window, kDecodeKeysPerTile);
	return kv_heads * p.splits * (q_per_kv * n_q) * (head_dim + 2) * (int64_t)sizeof(float);
}

hipError_t launch_sdp_attention_decode_f32(const float* q, const float* k, const float* v, float* y, void* workspace,
                                           int64_t batch_heads, int64_t q_per_kv, int64_t n_q, int64_t n_k, int64_t head_dim,
                                           float alpha, float softcap, int causal, int64_t window, hipStream_t stream)
{
	if (batch_heads == 0 || n_q == 0) return hipSuccess;
	const int64_t kv_heads = batch_heads / q_per_kv;
	const DecodePlan p = plan_decode(kv_heads * ((q_per_kv * n_q + kDecodeRowsPerWave - 1) / kDecodeRowsPerWave), n_q, n_k, causal, window, kDecodeKeysPerTile);
	DecodeArgsF32 da;
	da.a.q = q;
	da.a.k = k;
	da.a.v = v;
	da.a.y = y;
	da.a.n_q = (int)n_q;
	da.a.n_k = (int)n_k;
	da.a.q_per_kv = (int)q_per_kv;
	da.a.diag = (int)(n_k - n_q);
	da.a.causal = causal ? 1 : 0;
	da.a.window = (int)window;
	const bool capped = softcap != 0.0f;
	da.a.k_in = capped ? 2.0f * kLog2e * alpha / softcap : alpha * kLog2e;
	da.a.k_cap = capped ? softcap * kLog2e : 0.0f;
	da.a.partials = nullptr;
	da.ws = static_cast<float*>(workspace);
	da.rows = (int)(q_per_kv * n_q);
	da.groups = (da.rows + kDecodeRowsPerWave - 1) / kDecodeRowsPerWave;
	da.splits = p.splits;
	da.tiles_per_split = p.tiles_per_split;
	da.t_first = p.t_first;
	da.t_last = p.t_last;
#define ANYGPU_DECODE_F32_DIM(DIM) \
	return capped ? launch_decode_variant_f32<DIM, true>(da, kv_heads, stream) : launch_decode_variant_f32<DIM, false>(da, kv_heads, stream)
	switch (head_dim)
	{
	case 64: ANYGPU_DECODE_F32_DIM(64);
	case 128: ANYGPU_DECODE_F32_DIM(128);
	default: ANYGPU_DECODE_F32_DIM(256);
	}
#undef ANYGPU_DECODE_F32_DIM
}

}  // namespace anygpu
