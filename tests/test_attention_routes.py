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


def _launches(test_cases, dtype="f16", mask=RULE, dims=(64, 128), capped=0):
    """(heads, queries, keys, causal, window) of GPU tests as launches; a window without the causal rule as one with it, which sees fewer keys"""
    return [(dtype, mask, d, h, n_q, n_k, w if w else CAUSAL if causal else NONE, capped, 0) for h, n_q, n_k, causal, w in test_cases for d in dims]


def test_gpu_tests_reach_the_kernels_they_name(forms):
    def of(*launches, **more):
        return set(forms(_launches(launches, **more)))
    # 32 queries per wave, overlapped and in turn
    assert of((264, 1000, 1000, True, 0), (264, 897, 960, True, 0), (264, 1100, 1161, True, 600), (264, 130, 641, False, 0), (264, 97, 577, True, 0), (512, 900, 900, True, 0)) == {"q32"}
    assert of((528, 128, 192, True, 0), (528, 256, 256, True, 33), (512, 200, 200, True, 0)) == {"q32 in turn"}
    # 16 queries per wave
    sixteen = [(140, 31, 64, True, 0), (140, 127, 129, True, 0), (140, 128, 128, True, 0), (140, 113, 63, False, 0), (120, 129, 257, True, 70), (120, 160, 100, True, 0), (56, 300, 321, False, 0),
               (64, 257, 600, True, 1), (120, 130, 513, True, 0), (120, 130, 300, False, 0)]
    assert of(*sixteen) == {"q16"}
    # 16 rows per block with eight waves and four
    assert of((4, 40, 257, True, 0), (4, 31, 288, False, 0), (4, 100, 129, True, 33), (4, 130, 97, True, 0), (4, 33, 65, True, 0), (3, 16, 95, False, 0)) == {"rows8"}
    assert of((160, 40, 257, True, 0), (160, 31, 288, False, 0), (80, 70, 600, False, 0)) == {"rows4"}
    assert of((4, 17, 17, True, 0), (2, 33, 32, True, 0), (4, 60, 40, True, 0), dims=(256,)) == {"rows8"}
    assert of((160, 17, 17, True, 0), (160, 40, 257, True, 0), (160, 80, 150, True, 1), dtype="f32") == {"rows4"}
    # head dimension 256: blocks of 128 queries with many heads
    from test_gpu_parity import ATTN_D256_CASES
    many = [(h * (1030 // (h * ((n_q + 15) // 16)) + 1), n_q, n_k, causal, w) for h, _, n_q, n_k, _, _, _, causal, w in ATTN_D256_CASES if n_k < 1500]
    assert of(*many, (2, 129, 3000, True, 1800), dims=(256,)) == {"skew"}
    # mask tensors: what they hide, softcap and grouped heads
    for dtype in ("f16", "f32"):
        assert of((3, 40, 300, False, 0), (4, 40, 257, False, 0), (6, 17, 130, False, 0), (8, 100, 90, False, 0), dtype=dtype, mask=MASK, dims=(64, 128, 256)) == {"rows8"}
        assert of((100, 40, 300, False, 0), (160, 40, 300, False, 0), dtype=dtype, mask=MASK) == {"rows4"}
        assert of((700, 40, 300, False, 0), dtype=dtype, mask=MASK, dims=(64, 128, 256)) == {"blocks"}
    note = {"f16": [(64, 70, 300, 333), (64, 140, 130, 1500), (128, 48, 300, 300), (128, 96, 130, 700), (256, 26, 300, 301), (256, 30, 130, 1030)],
            "f32": [(64, 120, 300, 333), (64, 64, 200, 2100), (128, 80, 300, 300), (128, 40, 200, 1500), (256, 24, 300, 301), (256, 4, 150, 1100)]}
    for dtype, shapes in note.items():
        for d, *shape in shapes:
            assert of((*shape, False, 0), dtype=dtype, mask=MASK, dims=(d,)) == {"blocks"}, (dtype, d, shape)
