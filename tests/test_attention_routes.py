"""Which kernel a fused attention takes (the rules of attention.hip, attention_f16_kwave.hpp and attention_f32_kwave.hpp in anygpu_amd/csrc), compiled for the
host: launches that were timed on both sides go to the faster one, and the launches of the GPU tests to the kernels that these name.  CPU only."""
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
constexpr int kAttnKeysPerTile = 64, kQ32QueriesPerBlock = 128;
struct AttnArgs { int n_q, n_k, diag, causal, window; };
%s
namespace f16 { constexpr int kKeyWaveRows = 16, kKeyWaveTile = 32;
%s
}
namespace f32 { constexpr int kKeyWaveRows = 16, kKeyWaveTile = 16;
%s
}
template <int D> const char* f16_rules(const AttnArgs& a, int64_t heads, bool capped)
{
	if (f16::attention_kwave_wanted(D, false, heads, a.n_q, a.n_k, a.causal, a.diag, a.window, 256)) return 256 < heads * ((a.n_q + 15) / 16) && D != 256 ? "rows4" : "rows8";
	if constexpr (D == 256) return "skew";
	else
	{
		const int64_t blocks = heads * ((a.n_q + 127) / 128);
		if (!attention_q32_wanted<D>(a, blocks, true)) return "q16";
		return (capped ? attention_q32_in_turn<D, true>(a) : attention_q32_in_turn<D, false>(a)) ? "q32 in turn" : "q32";
	}
}
int main(int argc, char** argv)
{
	for (int i = 1; i + 8 < argc; i += 9)
	{
		const bool half = argv[i][1] == '1', mask = argv[i + 1][0] == '1', capped = argv[i + 7][0] == '1', decode = argv[i + 8][0] == '1';
		const int d = std::atoi(argv[i + 2]);
		const int64_t heads = std::atoi(argv[i + 3]);
		const int n_q = std::atoi(argv[i + 4]), n_k = std::atoi(argv[i + 5]), rule = std::atoi(argv[i + 6]);      // rule: -1 none, 0 causal, else a causal window
		const AttnArgs a{n_q, n_k, n_k - n_q, rule >= 0, rule > 0 ? rule : 0};
		const char* form = "";
		if (decode) form = f16::decode_kwave_wanted(d, heads, ((n_k + 31) / 32), 256) ? "rows8" : "splits";
		else if (half && !mask) form = d == 64 ? f16_rules<64>(a, heads, capped) : d == 128 ? f16_rules<128>(a, heads, capped) : f16_rules<256>(a, heads, capped);
		else
		{
			const bool rows = half ? f16::attention_kwave_wanted(d, true, heads, n_q, n_k, 0, a.diag, 0, 256)
			                       : f32::attention_kwave_wanted_f32(d, mask, heads, n_q, n_k, a.causal, a.diag, a.window, 256);
			form = !rows ? "blocks" : 256 < heads * ((n_q + 15) / 16) && d != 256 ? "rows4" : "rows8";
		}
		std::puts(form);
	}
	return 0;
}
"""

RULE, MASK = 0, 1
NONE, CAUSAL = -1, 0
# dtype, mask tensor, head dimension, heads, queries, keys, NONE / CAUSAL / a causal window, softcap, generation step: the kernel
TIMED = [
    # many heads with few tiles each: blocks of 128 queries
    (("f16", RULE, 256, 176, 34, 34, NONE, 0, 0), "skew"), (("f16", RULE, 256, 192, 33, 33, NONE, 0, 0), "skew"), (("f16", RULE, 256, 80, 81, 242, NONE, 0, 0), "skew"), (("f16", RULE, 256, 184, 36, 36, 20, 0, 0), "skew"),
    (("f16", RULE, 256, 80, 112, 112, NONE, 0, 0), "skew"), (("f16", MASK, 256, 64, 153, 153, NONE, 0, 0), "blocks"), (("f16", RULE, 128, 152, 68, 68, CAUSAL, 0, 0), "q16"), (("f16", RULE, 64, 84, 29, 29, NONE, 0, 0), "q16"),
    (("f32", RULE, 256, 224, 75, 91, NONE, 0, 0), "blocks"), (("f32", RULE, 256, 240, 105, 105, CAUSAL, 0, 0), "blocks"), (("f32", RULE, 256, 32, 783, 783, 51, 0, 0), "blocks"), (("f32", RULE, 256, 32, 813, 813, 99, 0, 0), "blocks"),
    # few heads, and windows over many keys: 16 rows per block
    (("f16", RULE, 256, 8, 96, 96, CAUSAL, 0, 0), "rows8"), (("f16", RULE, 256, 8, 394, 394, CAUSAL, 0, 0), "rows8"), (("f16", RULE, 256, 8, 700, 700, CAUSAL, 0, 0), "rows8"), (("f16", RULE, 128, 32, 300, 300, CAUSAL, 0, 0), "rows4"),
    (("f16", RULE, 64, 16, 500, 500, CAUSAL, 0, 0), "rows4"), (("f16", RULE, 64, 16, 309, 309, 33, 0, 0), "rows4"), (("f16", RULE, 128, 16, 772, 772, 23, 0, 0), "rows4"), (("f16", MASK, 256, 8, 400, 400, NONE, 0, 0), "rows8"),
    (("f32", RULE, 256, 8, 500, 500, CAUSAL, 0, 0), "rows8"), (("f32", RULE, 256, 8, 1824, 1824, 53, 0, 0), "rows8"), (("f32", RULE, 128, 16, 300, 300, CAUSAL, 0, 0), "rows4"), (("f32", MASK, 256, 8, 300, 300, NONE, 0, 0), "rows8"),
    # more than one block of 128 queries per CU: by the tiles of an average block
    (("f16", RULE, 128, 256, 200, 200, CAUSAL, 0, 0), "q32 in turn"), (("f16", RULE, 128, 192, 300, 300, CAUSAL, 0, 0), "q32 in turn"), (("f16", RULE, 128, 192, 300, 300, NONE, 0, 0), "q32"), (("f16", RULE, 128, 32, 3000, 3000, CAUSAL, 0, 0), "q32"),
    (("f16", RULE, 64, 256, 250, 250, CAUSAL, 0, 0), "q32 in turn"), (("f16", RULE, 64, 128, 600, 600, CAUSAL, 0, 0), "q32"), (("f16", RULE, 128, 288, 296, 296, CAUSAL, 1, 0), "q32 in turn"), (("f16", RULE, 128, 160, 596, 596, 236, 1, 0), "q32 in turn"), (("f16", RULE, 128, 128, 900, 900, CAUSAL, 1, 0), "q32"),
    # generation
    (("f16", RULE, 128, 8, 1, 600, CAUSAL, 0, 1), "rows8"), (("f16", RULE, 128, 8, 1, 1000, CAUSAL, 0, 1), "splits"), (("f16", RULE, 256, 4, 1, 400, CAUSAL, 0, 1), "splits"),
]


def _function(text, start):
    begin = text.index(start)
    return text[begin:text.index("\n}", begin) + 3]


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    split, f16, f32, host = ((CSRC / name).read_text() for name in ("attention_split.hpp", "attention_f16_kwave.hpp", "attention_f32_kwave.hpp", "attention.hip"))
    common = [_function(split, "inline int64_t attention_block_tiles("), split[split.index("template <typename TilesOf>"):split.index("struct KeyWaveCost")],
              split[split.index("struct KeyWaveCost"):split.index("};", split.index("struct KeyWaveCost")) + 2],
              _function(split, "inline bool attention_kwave_ahead("), _function(host, "template <int D>\nbool attention_q32_wanted("), _function(host, "template <int D, bool SOFTCAP>\nbool attention_q32_in_turn(")]
    where = tmp_path_factory.mktemp("routes")
    src, exe = where / "routes.cpp", where / "routes"
    src.write_text(HARNESS % ("\n".join(common), _function(f16, "inline bool attention_kwave_wanted(") + _function(f16, "inline bool decode_kwave_wanted("), _function(f32, "inline bool attention_kwave_wanted_f32(")))
    subprocess.run(["g++", "-O2", "-std=c++20", "-o", str(exe), str(src)], check=True)

    def run(cases):
        args = [str(v) for case in cases for v in case]
        return subprocess.run([str(exe), *args], capture_output=True, text=True, check=True, timeout=5).stdout.splitlines()
    return run


def test_timed_launches_take_the_faster_kernel(forms):
    assert [(case, got) for (case, _), got in zip(TIMED, forms([case for case, _ in TIMED]))] == TIMED
