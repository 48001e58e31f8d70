"""The plan that cuts the key range of the fp16 decode attention into splits (anygpu_amd/csrc/attention_split.hpp), compiled for the
host (it uses nothing of the device) and swept over shapes: the size query, the least size that the entry points ask for and
the cut that a workspace gets agree with each other, and every cut covers the visible keys.  CPU only."""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <algorithm>
#include <cstdint>
#include <cstdio>
#define ANYGPU_DECODE_STATIC_SCRATCH_BYTES (8 * 1024 * 1024)
namespace anygpu {
%s
}
using namespace anygpu;
static long fails = 0, checks = 0, finer_needs_less = 0;
static void expect(bool ok, const char* what, long long units, long long rows, long long d, long long n_q, long long n_k, long long window)
{
	++checks;
	if (!ok && fails++ < 5) std::printf("%%s: %%lld key / value heads, %%lld rows, d %%lld, %%lld queries, %%lld keys, window %%lld\n", what, units, rows, d, n_q, n_k, window);
}
static void check(int64_t kv, int64_t per, int64_t n_q, int64_t n_k, int64_t d, int causal, int64_t window)
{
	const int64_t rows = per * n_q, split_bytes = kv * rows * (d + 2) * 4;
	const DecodePlansF16 p = plans_decode_f16(kv * per, per, n_q, n_k, d, causal, window);
	const int64_t query = p.query_bytes(), least = p.least_bytes();
	const auto ok = [&](bool c, const char* what) { expect(c, what, kv, rows, d, n_q, n_k, window); };
	ok(least <= query, "the entry points ask for more than the size query returns");
	ok(least <= p.pairs_bytes, "a workspace for the cut in 64 keys is refused");
	const int64_t static_bytes = ANYGPU_DECODE_STATIC_SCRATCH_BYTES;
	ok((least <= static_bytes) == (p.pairs_bytes <= static_bytes), "the fixed scratch takes other shapes than those whose cut in 64 keys fits it");
	if (least <= static_bytes) ok(p.within(static_bytes).splits == p.within(query).splits && p.within(static_bytes).tiles_per_split == p.within(query).tiles_per_split,
	                              "fixed scratch and queried workspace cut differently");
	finer_needs_less += p.take_fine && p.fine_bytes < p.pairs_bytes;
	for (int64_t room : {least, query, (least + query) / 2, query + 1000000})
	{
		const DecodePlan c = p.within(room);
		ok(c.splits * split_bytes <= room, "the cut does not fit the workspace");
		ok(c.splits >= 1 && c.splits <= kDecodeMaxSplits, "splits");
		const int64_t diag = n_k - n_q, key_hi = causal ? std::min(n_k - 1, n_q - 1 + diag) : n_k - 1;
		const int64_t key_lo = window > 0 ? std::max<int64_t>(0, diag - window + 1) : 0;
		ok(key_hi < key_lo || (c.t_first * 32 <= key_lo && (c.t_last + 1) * 32 > key_hi), "visible keys outside of the tiles");
		ok((int64_t)c.splits * c.tiles_per_split >= c.t_last - c.t_first + 1, "tiles outside of the splits");
	}
}
int main()
{
	for (int64_t kv = 1; kv <= 130; kv += kv < 84 ? 1 : 9)
		for (int64_t window : {0, 512, 1024, 2048, 4096, 8192})
			for (int64_t n_k : {1, 31, 32, 64, 65, 300, 511, 2016, 2080, 4127, 4128, 4129, 4192, 5001, 8224, 9000, 32768})
				for (int64_t n_q : {1, 3})
					for (int causal : {0, 1})
					{
						check(kv, 1, n_q, n_k, 256, causal, window);
						check(kv, 2, n_q, n_k, 256, causal, window);
						check(kv, 8, n_q, n_k, 128, causal, window);
						check(kv, 16, n_q, n_k, 128, causal, window);
					}
	for (int64_t n_k = 1; n_k < 9000; ++n_k) check(28, 2, 1, n_k, 256, 1, 4096);
	if (finer_needs_less == 0) { std::printf("no shape whose finer cut has fewer splits\n"); return 1; }
	if (fails) return 1;
	std::printf("ok %%ld\n", checks);
	return 0;
}
"""


def test_decode_plan_of_every_shape_fits_what_is_asked_for(tmp_path):
    text = (REPO / "anygpu_amd" / "csrc" / "attention_split.hpp").read_text()
    constants = text[text.index("constexpr int kDecodeRowsPerWave"):text.index("// a workspace row is")]
    plans = text[text.index("struct DecodePlan\n"):text.index("// Which split and which group of 16 rows")]
    src = tmp_path / "decode_plan_check.cpp"
    src.write_text(HARNESS % (constants + plans))
    exe = tmp_path / "decode_plan_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout.startswith("ok "), run.stdout
