"""The order of a launch's blocks over the XCDs, compiled for the host: every logical
block comes from one workgroup, and no XCD has more than its share and a sixteenth."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "tnl-lbm_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <vector>
#include "lbm_step.hpp"
namespace lbm {
int hip_check(hipError_t, const char*) { return 0; }
bool narrow_slots_allowed() { return true; }
}
int main()
{
	using namespace lbm;
	// arrays within half the last-level cache, within some times it, beyond
	const uint64_t bytes[] = {1ull << 20, 20ull << 20, 300ull << 20, 4000ull << 20};
	const uint32_t counts[] = {1, 7, 8, 9, 63, 64, 65, 128, 129, 1023, 1025, 2448, 2544, 4095, 4096, 4097, 20000, 32769, 131073};
	int bad = 0;
	for (uint64_t total : bytes)
		for (uint32_t n : counts)
			for (int even = 0; even < 2; even++)
				for (uint32_t most : {5u, 8u}) {
					StepArgs A;
					std::memset(&A, 0, sizeof A);
					A.plane_bytes = total / 27;
					A.nblocks = n;
					A.even = even;
					const uint32_t grid = padded_blocks(A, most);
					std::vector<int> seen(n, 0);
					uint32_t load[NXCD] = {};
					for (uint32_t b = 0; b < grid; b++) {
						const uint32_t L = block_of(b, A.group, A.span);
						if (L < n) {
							seen[L]++;
							load[b % NXCD]++;
						}
					}
					const uint32_t share = (n + NXCD - 1) / NXCD;
					bool ok = grid % NXCD == 0;
					for (int c : seen)
						ok = ok && c == 1;
					for (uint32_t l : load)
						ok = ok && l <= share + share / 16 + 1;
					if (! ok) {
						bad++;
						std::printf("bytes %llu blocks %u even %d most %u\n", (unsigned long long) total, n, even, most);
					}
				}
	return bad != 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_blocks_are_spread_over_the_xcds(tmp_path):
    (tmp_path / "order.hip").write_text(PROGRAM)
    exe = tmp_path / "order"
    subprocess.run([HIPCC, "-O0", "-std=c++17", "--offload-host-only", f"-I{CSRC}", f"-I{CSRC.parent.parent / 'include'}",
                    "-o", str(exe), str(tmp_path / "order.hip")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
