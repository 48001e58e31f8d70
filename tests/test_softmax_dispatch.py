"""The rule that picks a row softmax's kernel (launch_softmax_rows of anygpu_amd/csrc/softmax.hip), compiled for the host with the kernels replaced
by checks: a kernel that reads a mask tensor is picked exactly where there is one, and the picked form holds every row.  CPU only."""
import re
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1;
inline hipError_t hipGetLastError() { return 0; }
inline void discard_stale_error() {}
struct half_t { unsigned short bits; };
constexpr int kWaveSize = 64;
constexpr float kLog2e = 1.44269504f;
#define __device__
#define __forceinline__ inline
using std::min;
using std::max;
inline int64_t min(int64_t a, int64_t b) { return a < b ? a : b; }
inline int64_t max(int64_t a, int64_t b) { return a > b ? a : b; }
%(args)s
enum : int { kCapNone, kCapShort, kCapFull };
constexpr float kCapShortMost = 64.0f;
static long picked[4] = {};
[[noreturn]] static void fail(const char* what, const SoftmaxArgs& a, int bytes, int vpl, int group)
{
	std::printf("%%s: %%lld x %%lld of %%d bytes, pitches %%lld %%lld, at %%llx %%llx, window %%lld, form %%d x %%d\n", what, (long long)a.rows, (long long)a.cols, bytes,
	            (long long)a.xs, (long long)a.ys, (unsigned long long)a.x, (unsigned long long)a.y, (long long)a.window, vpl, group);
	std::exit(1);
}
// the chunks that hold a row's visible part, as the kernel counts them
template <typename T, int VPL, int GROUP, %(cap)s>
void softmax_rows_kernel(const SoftmaxArgs& a)
{
	++picked[0];
	if (a.mask != nullptr) fail("mask", a, sizeof(T), VPL, GROUP);
	constexpr int EPV = 16 / (int)sizeof(T), kStart = GROUP == 16 ? EPV : 128 / (int)sizeof(T);
	for (int64_t row = 0; row < a.rows; row += row < 70 || row > a.rows - 70 ? 1 : 13)
	{
		const uintptr_t x = reinterpret_cast<uintptr_t>(a.x) + row * a.xs * sizeof(T), y = reinterpret_cast<uintptr_t>(a.y) + row * a.ys * sizeof(T);
		if (x %% 16 != y %% 16) fail("alignment", a, sizeof(T), VPL, GROUP);
		const int shift = (int)(y / sizeof(T) %% kStart);
		const RowSpan span = row_span(a, row);
		if (span.hi < span.lo) continue;
		// a vector that holds elements of the row: those of its elements that are loaded are the tensor's, and all of the row's are among them
		const RowNeighbours near = row_neighbours(a, row);
		const int end = shift + (int)a.cols;
		for (int v : {((int)span.lo + shift) / EPV, ((int)span.hi + shift) / EPV})
		{
			const int from = std::max(0, shift - v * EPV - near.before), to = std::min(EPV, end - v * EPV + near.behind);
			const int64_t at = row * a.xs - shift + (int64_t)v * EPV, tensor = (a.rows - 1) * a.xs + a.cols;
			if (at + from < 0 || at + to > tensor || from > std::max(0, shift - v * EPV) || to < std::min(EPV, end - v * EPV)) fail("outside", a, sizeof(T), VPL, GROUP);
		}
		const int c_lo = ((int)span.lo + shift) / EPV / GROUP, c_hi = ((int)span.hi + shift) / EPV / GROUP;
		if (c_hi - c_lo + 1 > VPL) fail("capacity", a, sizeof(T), VPL, GROUP);
	}
}
template <typename T, int VPL, bool LOOSE, int GROUP, bool MASK>
void softmax_rows_wave_kernel(const SoftmaxArgs& a)
{
	++picked[MASK ? 1 : 2];
	constexpr int EPV = 16 / (int)sizeof(T);
	if (MASK != (a.mask != nullptr)) fail("mask", a, sizeof(T), VPL, GROUP);
	if ((a.cols + EPV - 1) / EPV > (int64_t)VPL * GROUP) fail("capacity", a, sizeof(T), VPL, GROUP);
	if (!LOOSE && (a.cols %% EPV || a.xs %% EPV || a.ys %% EPV || (uintptr_t)a.x %% 16 || (uintptr_t)a.y %% 16 || (MASK && (a.mask_stride %% EPV || (uintptr_t)a.mask %% 16))))
		fail("alignment", a, sizeof(T), VPL, GROUP);
}
template <typename T> void softmax_rows_long_kernel(const SoftmaxArgs&) { ++picked[3]; }
%(rule)s
template <typename T>
void sweep()
{
	const uintptr_t base = 1 << 20;
	const int size = sizeof(T);
	for (int64_t cols = 1; cols <= 40000; cols += cols < 600 || (cols > 16200 && cols < 16500) || (cols > 32500 && cols < 32900) ? 1 : 7)
		for (int64_t rows : {5, 64, 300})
			for (int off : {0, 16, size})
				for (int pad : {0, 1, 8})
					for (int form = 0; form < 6; ++form)
					{
						// no window, a short one, about the row's width, shorter, without the causal rule; x and y an element apart
						const int64_t window = form == 0 || form == 5 ? 0 : form == 1 ? 100 : form == 2 ? std::max<int64_t>(1, cols - 3) : cols / 2 + 1;
						const void *x = (const void*)(base + off), *mask = (const void*)(base + (64 << 20) + off %% 16);
						void* y = (void*)(base + (32 << 20) + off + (form == 5 ? size : 0));
						for (float cap : {0.0f, 30.0f})
							if (launch_softmax_rows<T>(x, y, rows, cols, cols + pad, cols + pad, rows, cols - rows, 1.0f, cap, form != 4, window, nullptr, 0, nullptr) != 0)
							{
								std::printf("refused: %%lld x %%lld of %%d bytes\n", (long long)rows, (long long)cols, size);
								std::exit(1);
							}
						if (form == 0 && launch_softmax_rows<T>(x, y, rows, cols, cols + pad, cols + pad, rows, 0, 1.0f, 0.0f, 0, 0, mask, cols + pad, nullptr) != 0) std::exit(2);
					}
}
int main()
{
	sweep<half_t>();
	sweep<float>();
	for (long n : picked)
		if (n == 0) { std::printf("a form was never picked\n"); return 1; }
	std::printf("ok\n");
	return 0;
}
"""


def _between(text, start, end):
    begin = text.index(start)
    return text[begin:text.index(end, begin) + len(end)]


def test_softmax_kernels_are_picked_by_the_mask_and_hold_their_rows(tmp_path):
    text = (REPO / "anygpu_amd" / "csrc" / "softmax.hip").read_text()
    args = [_between(text, start, "\n}") + end for start, end in (("struct SoftmaxArgs", ";"), ("__device__ __forceinline__ int64_t query_of_row", ""),
                                                                  ("static inline unsigned blocks_for_rows", ""))]
    args += [_between(text, "struct RowNeighbours", ";") + " };", _between(text, "__device__ __forceinline__ RowNeighbours row_neighbours", "\n}")]
    args += [_between(text, "struct RowSpan", ";") + " };", _between(text, "__device__ __forceinline__ RowSpan row_span", "\n}")]
    rule = [_between(text, start, "\n}") for start in ("static bool rows_alike", "template <typename T, int VPL, int GROUP>\nstatic hipError_t launch_rows",
                                                       "template <typename T>\nstatic int64_t rows_vectors", "template <typename T, int VPL, bool LOOSE = false, int GROUP = 64>",
                                                       "template <typename T, bool LOOSE>\nstatic hipError_t launch_long_rows",
                                                       "template <typename T>\nhipError_t launch_softmax_rows")]
    rule = re.sub(r"<<<.*?>>>", "", "\n".join(rule))
    cap = _between(text, "template <typename T, int VPL, int GROUP, ", ">").rsplit(", ", 1)[1][:-1]
    src, exe = tmp_path / "dispatch_check.cpp", tmp_path / "dispatch_check"
    src.write_text(HARNESS % {"args": "\n".join(args), "rule": rule, "cap": cap})
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout
