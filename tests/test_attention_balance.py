"""Equal shares of a masked attention launch (anygpu_amd/csrc/attention_balance.hpp): every set tile is walked once, by one range, and the
merge finds every partial result in the slot its range left it in.  The scalar helpers' text is compiled for the host; the walk over the
ranges is restated with plain prefix sums.  CPU only."""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <map>
#include <random>
#include <vector>
#define __device__
#define __forceinline__ inline
#define __restrict__
%s
int main()
{
	std::mt19937_64 rng(3);
	for (int iter = 0; iter < 3000; ++iter)
	{
		const int tiles = 1 + rng() %% 200, words = (tiles + 63) / 64, q_blocks = 1 + rng() %% 40, heads = 1 + rng() %% 5;
		const int ranges = 1 + rng() %% 64, least = 1 + rng() %% 6, density = rng() %% 5;
		std::vector<unsigned long long> map((size_t)q_blocks * words, 0);
		std::vector<std::vector<int>> set(q_blocks);
		std::vector<int> count(q_blocks), before(q_blocks + 1, 0);
		for (int b = 0; b < q_blocks; ++b)
		{
			const bool none = rng() %% 6 == 0;                    // a query block that sees nothing counts as one tile
			for (int t = 0; t < tiles; ++t)
				if (!none && (density == 4 || (int)(rng() %% 4) < density)) map[(size_t)b * words + t / 64] |= 1ull << (t %% 64), set[b].push_back(t);
			count[b] = std::max<int>(1, set[b].size());
			before[b + 1] = before[b] + count[b];
			for (int i = 0; i < (int)set[b].size(); ++i)
				if (balance_nth_tile(&map[(size_t)b * words], words, i) != set[b][i]) { std::printf("tile: mismatch\n"); return 1; }
			if (set[b].empty() && balance_nth_tile(&map[(size_t)b * words], words, 0) < tiles) { std::printf("no tile: mismatch\n"); return 1; }
		}
		const int64_t per_head = before[q_blocks], total = per_head * heads;
		const int per = (int)std::max<int64_t>((total + ranges - 1) / ranges, least);
		// the ranges as the kernel walks them: slot 2 i for the first query block, 2 i + 1 for any later one
		std::map<std::pair<int, int>, std::vector<std::pair<int64_t, int64_t>>> parts;      // (head, block): (range, slot)
		std::map<std::pair<int, int>, int> walked;
		std::map<int64_t, int> used;
		for (int64_t range = 0; range < ranges; ++range)
		{
			int64_t at = range * per;
			const int64_t end = std::min(at + per, total);
			bool first = true;
			while (at < end)
			{
				const int head = (int)(at / per_head), x = (int)(at %% per_head);
				const int b = (int)(std::upper_bound(before.begin(), before.end(), x) - before.begin()) - 1, in_block = x - before[b];
				const int taken = (int)std::min<int64_t>(count[b] - in_block, end - at);
				if (walked[{head, b}] != in_block) { std::printf("gap\n"); return 1; }
				walked[{head, b}] += taken;
				if (taken != count[b])
				{
					const int64_t slot = 2 * range + (first ? 0 : 1);
					if (used[slot]++) { std::printf("slot used twice\n"); return 1; }
					parts[{head, b}].push_back({range, slot});
				}
				first = false;
				at += taken;
			}
		}
		// ... and as the merge looks for them
		for (int head = 0; head < heads; ++head)
			for (int b = 0; b < q_blocks; ++b)
			{
				if (walked[{head, b}] != count[b]) { std::printf("not all tiles\n"); return 1; }
				const int64_t s = head * per_head + before[b], e = s + count[b], first = s / per, last = (e - 1) / per;
				const auto& got = parts[{head, b}];
				if (first == last ? !got.empty() : (int64_t)got.size() != last - first + 1) { std::printf("parts: mismatch\n"); return 1; }
				for (size_t i = 0; i < got.size(); ++i)
					if (got[i].first != first + (int64_t)i || got[i].second != balance_slot(got[i].first, s, per)) { std::printf("slot: mismatch\n"); return 1; }
			}
	}
	std::printf("ok\n");
	return 0;
}
"""


def test_equal_shares_cover_every_tile_once(tmp_path):
    text = (REPO / "anygpu_amd" / "csrc" / "attention_balance.hpp").read_text()
    body = []
    for start, end in (("__device__ __forceinline__ int balance_nth_tile", "\n}\n"), ("__device__ __forceinline__ int64_t balance_slot", "}\n")):
        begin = text.index(start)
        body.append(text[begin:text.index(end, begin) + len(end)])
    src, exe = tmp_path / "balance_check.cpp", tmp_path / "balance_check"
    src.write_text(HARNESS % "\n".join(body))
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout
