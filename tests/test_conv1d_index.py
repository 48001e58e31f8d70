"""The division by a launch's number of channels and row length in the convolution over one run of vectors (divide and inverse_of of
anygpu_amd/csrc/conv1d.hip), compiled for the host: exact for every divisor from one on.  CPU only."""
import re
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#define __host__
#define __device__
#define __forceinline__ inline
inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((uint64_t)a * b) >> 32); }
%s
int main()
{
	const unsigned most = 0xFFFFFFFFu;
	long checked = 0;
	auto check = [&](unsigned n, unsigned d) {
		++checked;
		if (divide(n, d, inverse_of(d)) == n / d) return true;
		std::printf("%%u / %%u gives %%u\n", n, d, divide(n, d, inverse_of(d)));
		return false;
	};
	auto divisor = [&](unsigned d) {
		// the quotients' own steps, from both ends of the range, and numbers in between
		for (uint64_t k = 0; k < 40; ++k)
			for (uint64_t n : {k * d, k * d + d - 1, (most / d - k) * (uint64_t)d, (most / d - k) * (uint64_t)d + d - 1, (uint64_t)most - k, k, k * 107374183u + 12345u})
				if (n <= most && !check((unsigned)n, d)) return false;
		return true;
	};
	for (unsigned d = 1; d < 20000; ++d)
		if (!divisor(d)) return 1;
	for (int bit = 1; bit < 32; ++bit)
		for (int off = -2; off <= 2; ++off)
			if ((1u << bit) + off >= 1u && !divisor((1u << bit) + off)) return 1;
	for (unsigned d : {2147483647u, 2147483646u, 1431655765u, 4294967295u, 4294967294u})
		if (!divisor(d)) return 1;
	// one channel: any row number is channel 0
	for (unsigned n = 0; n < 100000; ++n)
		if (!check(n, 1) || n - divide(n, 1, inverse_of(1)) != 0) return 1;
	std::printf("%%ld\n", checked);
	return 0;
}
"""


def test_division_of_rows_and_channels(tmp_path):
    text = (REPO / "anygpu_amd" / "csrc" / "conv1d.hip").read_text()
    parts = re.findall(r"^__host__ __device__ __forceinline__ unsigned inverse_of\(.*\}\n", text, re.M) + \
        re.findall(r"^__device__ __forceinline__ unsigned divide\(.*?^\}\n", text, re.M | re.S)
    assert len(parts) == 2
    # the launcher takes its inverses from the function that is checked here
    assert "inverse_of((unsigned)chan), inverse_of((unsigned)seqlen)" in text
    source, program = tmp_path / "index.cpp", tmp_path / "index"
    source.write_text(HARNESS % "".join(parts))
    subprocess.run(["g++", "-std=c++20", "-O2", "-o", str(program), str(source)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout
    assert int(done.stdout) > 5000000
