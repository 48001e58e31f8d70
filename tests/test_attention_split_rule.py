"""The rule that gives a float32 attention its form (attention_split_wanted of anygpu_amd/csrc/attention_f32.hip), compiled for the host: calls whose
query blocks see few key tiles, or go out in many parts, stay on the fp32 matrix instruction, where they are faster.  CPU only."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "anygpu_amd" / "csrc"

HARNESS = r"""
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
inline int device_cu_count() { return 256; }
namespace band { constexpr size_t kBandPartialBytes = (size_t)64 << 20; }
constexpr int kSplitQueries = 128, kSplitKeys = 32;
constexpr int64_t kSplitMaskStride = 1 << 22;
struct AttnArgsF32 { int n_q, n_k, diag, causal, window; int64_t mask_stride; };
%s
int main(int argc, char** argv)
{
	for (int i = 1; i + 5 < argc; i += 6)
	{
		const int d = std::atoi(argv[i]), heads = std::atoi(argv[i + 1]), n_q = std::atoi(argv[i + 2]), n_k = std::atoi(argv[i + 3]);
		const AttnArgsF32 a{n_q, n_k, n_k - n_q, std::atoi(argv[i + 5]), std::atoi(argv[i + 4]), n_k};
		std::printf("%%d\n", (int)(d == 64 ? attention_split_wanted<64, false>(a, heads) : d == 128 ? attention_split_wanted<128, false>(a, heads) : attention_split_wanted<256, false>(a, heads)));
	}
	return 0;
}
"""

# head dimension, heads, queries, keys, window, causal: whether the bf16 parts are faster (both sides timed on the card)
CASES = [
    # short windows
    ((64, 16, 700, 700, 1, 1), 0), ((64, 16, 700, 700, 100, 1), 0), ((128, 16, 700, 700, 50, 1), 0), ((64, 24, 700, 700, 500, 1), 0), ((64, 16, 1500, 1500, 50, 1), 0),
    ((64, 32, 1500, 1500, 1, 1), 0), ((128, 32, 1500, 1500, 50, 1), 0), ((64, 16, 322, 658, 100, 1), 0), ((128, 16, 322, 658, 1, 1), 0), ((64, 8, 140, 700, 100, 0), 0),
    # many parts of a long key range
    ((64, 2, 300, 6000, 0, 1), 0), ((128, 2, 300, 6000, 0, 1), 0), ((64, 4, 300, 3000, 0, 0), 0), ((64, 4, 130, 6000, 4096, 1), 0), ((128, 2, 300, 6000, 2000, 1), 0), ((64, 1, 1000, 16000, 2000, 1), 0),
    # windows that leave enough, enough blocks
    ((64, 16, 4000, 4000, 100, 1), 1), ((128, 32, 4000, 4000, 30, 1), 1), ((64, 16, 1500, 1500, 1000, 1), 1), ((128, 16, 1500, 1500, 500, 1), 1), ((128, 16, 700, 700, 500, 1), 1),
    # no window: prompts, and a chunk against a cache
    ((64, 32, 2000, 2000, 0, 1), 1), ((128, 32, 3000, 3000, 0, 1), 1), ((128, 16, 2000, 2000, 0, 0), 1), ((128, 32, 400, 400, 0, 0), 1), ((64, 64, 400, 400, 0, 1), 1), ((64, 16, 700, 700, 0, 1), 1),
    ((128, 8, 350, 350, 0, 1), 1), ((64, 16, 300, 16000, 0, 1), 1), ((128, 16, 300, 16000, 0, 1), 1), ((64, 4, 140, 700, 0, 1), 1), ((128, 6, 300, 3000, 0, 1), 1),
    # few keys; few queries at 64; head dimension 256 always
    ((128, 32, 150, 150, 0, 0), 0), ((64, 64, 250, 250, 0, 0), 0), ((64, 8, 64, 4000, 0, 1), 0), ((256, 4, 700, 700, 1, 1), 1), ((256, 8, 64, 64, 0, 0), 1),
    # the largest index ranges that are taken: the rule's own time stays bounded
    ((64, 1, 1 << 29, 1 << 29, 4096, 1), 1), ((128, 1, 1 << 29, 1 << 29, 0, 1), 1),
]


def _function(text, start):
    begin = text.index(start)
    return text[begin:text.index("\n}", begin) + 3]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    split, f32 = (CSRC / "attention_split.hpp").read_text(), (CSRC / "attention_f32.hip").read_text()
    parts = [_function(split, "inline int64_t attention_block_tiles("), "struct AttnSplitPlan { int64_t n_split, n_big; };", _function(split, "inline AttnSplitPlan plan_attention_split("),
             _function(split, "inline int64_t plan_attention_parts("), _function(f32, "template <int D>\nbool attention_split_fills("), _function(f32, "template <int D, bool MASK>\nbool attention_split_wanted(")]
    where = tmp_path_factory.mktemp("rule")
    src, exe = where / "rule.cpp", where / "rule"
    src.write_text(HARNESS % "\n".join(parts))
    subprocess.run(["g++", "-O2", "-std=c++20", "-o", str(exe), str(src)], check=True)
    return exe


def test_float32_attention_takes_the_faster_form(rule):
    args = [str(v) for case, _ in CASES for v in case]
    got = subprocess.run([str(rule), *args], capture_output=True, text=True, check=True, timeout=5).stdout.split()
    assert [(case, int(g)) for (case, _), g in zip(CASES, got)] == CASES
