"""The block walk of the fused attention kernels (anygpu_amd/csrc/attention_walk.hpp), compiled for the host: every query block, half or part turns up
exactly once, and the second round is dispatched lightest first only where the launch has that many blocks, padding not counted.  CPU only."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "anygpu_amd" / "csrc"

HARNESS = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <tuple>
#define __device__
#define __forceinline__ inline
namespace anygpu {
%s
}
using namespace anygpu;
static void fail(const char* what, const AttnWalk& w) { std::printf("%%s: %%d query blocks, %%d groups of %%d, %%d in halves, %%d parts, turn %%d\n", what, w.real_q_blocks, w.groups, w.q_per_kv, w.n_split, w.parts_all, w.turn); std::exit(1); }
int main()
{
	long turned = 0, walks = 0;
	for (int q_per_kv : {1, 2, 3, 4, 5, 8, 16})
		for (int groups : {1, 2, 3, 7, 8, 14, 32, 56, 64})
			for (int q_blocks : {1, 2, 3, 4, 5, 7, 8, 13, 24, 33})
				for (int form = 0; form < 4; ++form)
				{
					const int n_split = form == 1 ? (q_blocks + 1) / 2 : 0, n_big = n_split > 0 ? q_blocks - n_split : 0, parts = form == 2 ? 3 : 1, turn = form == 3 ? 32 : 0;
					const int64_t heads = (int64_t)groups * q_per_kv;
					const AttnWalk w = make_attn_walk(q_blocks, heads, q_per_kv, n_split, n_big, parts, turn);
					std::map<std::tuple<int, int, int>, int> seen;
					for (int64_t block = 0; block < attn_walk_blocks(w); ++block)
					{
						int head, q_block, part, of, slot;
						if (!attn_walk_locate_part(w, (unsigned)block, head, q_block, part, of, slot)) continue;
						if (head < 0 || head >= heads || q_block < 0 || q_block >= q_blocks || part < 0 || part >= of) fail("outside", w);
						const bool cut = parts > 1 || q_block >= q_blocks - n_split;
						if (of != (parts > 1 ? parts : cut ? 2 : 1) || (cut && slot != q_blocks - 1 - q_block)) fail("part", w);
						if (++seen[{head, q_block, part}] > 1) fail("twice", w);
					}
					if ((int64_t)seen.size() != heads * (parts > 1 ? q_blocks * parts : q_blocks + n_split)) fail("missing", w);
					if (form == 3)
					{
						// at least seven eighths of two rounds of one block per CU (8 x 32), by the blocks that there are
						if ((w.turn > 0) != (8 * q_blocks * heads >= 7 * 2 * 32 * 8)) fail("turn", w);
						turned += w.turn > 0;
					}
					++walks;
				}
	std::printf("%%ld %%ld\n", walks, turned);
	return 0;
}
"""


def test_every_block_once_and_rounds_by_real_blocks(tmp_path):
    text = (CSRC / "attention_walk.hpp").read_text()
    body = text[text.index("constexpr int kAttnXcds"):text.rindex("}  // namespace anygpu")]
    source, program = tmp_path / "walk.cpp", tmp_path / "walk"
    source.write_text(HARNESS % body)
    subprocess.run(["g++", "-std=c++20", "-O2", "-o", str(program), str(source)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout
    walks, turned = map(int, done.stdout.split())
    assert walks == 7 * 9 * 10 * 4 and 100 < turned < 500
