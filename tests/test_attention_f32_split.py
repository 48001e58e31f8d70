"""The bf16 parts of floats in the float32 attention (split_pair of anygpu_amd/csrc/attention_f32.hip), the function's own text compiled for the
host: the parts add up to the float, and six of the nine products of parts miss at most 2^-24 of the product, without a bias.  CPU only."""
import subprocess
from pathlib import Path

from anygpu_amd import build

REPO = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#define __device__
#define __forceinline__ inline
typedef float float2_t __attribute__((ext_vector_type(2)));
%s
static std::mt19937_64 rng(1);
static float from_bits(uint32_t b) { return __builtin_bit_cast(float, b); }
static void parts_of(float x, double (&p)[3])
{
	unsigned w[3], v[3];
	split_pair(x, -x, w);
	split_pair(1.0f, x, v);
	for (int i = 0; i < 3; ++i)
	{
		p[i] = from_bits(w[i] << 16);
		if (p[i] != -from_bits(w[i] & 0xFFFF0000u) || p[i] != from_bits(v[i] & 0xFFFF0000u)) { std::printf("halves of a word\n"); std::exit(1); }
	}
}
int main()
{
	// every exponent from 2^-110 to the last below which rounding stays finite
	for (uint32_t e = 17; e <= 253; ++e)
		for (int i = 0; i < 2000; ++i)
		{
			const uint32_t m = i < 6 ? (const uint32_t[]){0, 1, 0x7FFFFF, 0x7FFF, 0x8000, 0xFFFF}[i] : (uint32_t)rng() & 0x7FFFFF;
			const float x = from_bits(e << 23 | m);
			double p[3];
			parts_of(x, p);
			if (p[0] + p[1] + p[2] != (double)x) { std::printf("parts of %%a\n", x); return 1; }
			if (std::fabs(p[1]) > std::ldexp(1.0, (int)e - 127 - 8) || std::fabs(p[2]) > std::ldexp(1.0, (int)e - 127 - 17)) { std::printf("size of the parts of %%a\n", x); return 1; }
		}
	double p[3];
	parts_of(0.0f, p);
	if (p[0] != 0 || p[1] != 0 || p[2] != 0) return 1;
	// products: all mantissas, mantissas around the rounding of the first and of the second part, and operands alike
	double worst = 0, sum = 0;
	long n = 0;
	const auto mantissa = [](int kind) -> uint32_t {
		const uint32_t near[] = {0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x7FC0, 0x7FBF, 0x7F80, 0x8040, 0x807F, 0x80FF};
		return kind %% 3 == 0 ? (uint32_t)rng() & 0x7FFFFF : kind %% 3 == 1 ? near[rng() %% 10] | ((uint32_t)rng() & 0x30000) : (uint32_t)rng() & 0x1FFFF;
	};
	for (long i = 0; i < 6000000; ++i)
	{
		const float x = from_bits(0x3F800000u | mantissa((int)(i / 2))), y = i & 1 ? x : from_bits(0x3F800000u | mantissa((int)(i / 6)));
		double a[3], b[3];
		parts_of(x, a);
		parts_of(y, b);
		const double exact = (double)x * y, off = (a[0] * b[0] + (a[0] * b[1] + a[1] * b[0]) + (a[1] * b[1] + (a[0] * b[2] + a[2] * b[0])) - exact) / exact;
		worst = std::fmax(worst, std::fabs(off));
		if (i / 2 %% 3 == 0 && !(i & 1)) { sum += off; ++n; }
	}
	if (worst > std::ldexp(1.0, -24)) { std::printf("worst product %%g\n", worst); return 1; }
	if (std::fabs(sum / n) > 1e-10) { std::printf("bias %%g\n", sum / n); return 1; }
	std::printf("ok\n");
	return 0;
}
"""


def test_bf16_parts_of_floats(tmp_path):
    text = (REPO / "anygpu_amd" / "csrc" / "attention_f32.hip").read_text()
    begin = text.index("__device__ __forceinline__ float2_t split_pair(")
    src, exe = tmp_path / "parts_check.cpp", tmp_path / "parts_check"
    src.write_text(HARNESS % text[begin:text.index("\n}\n", begin) + 3])
    subprocess.run([str(build.ROCM_DIR / "lib" / "llvm" / "bin" / "clang++"), "-O2", "-std=c++20", "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout
