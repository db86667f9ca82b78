"""The kernels' index arithmetic on tile lists, compiled for the host and run at the limits
of its 32 bits, where no GPU buffer reaches: what a list of more rows than a call's, or of
almost 2^31 rows, makes of a GEMM's tiles."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """Compiles a main()'s body against bux_amd/csrc's headers and returns its lines of
    integers."""
    at = tmp_path_factory.mktemp("host")

    def go(body: str) -> list[list[int]]:
        src, exe = at / "main.hip", at / "main"
        src.write_text('#include "tiles.h"\n#include "mx_direct.h"\n#include <cstdio>\nusing namespace bux;\n'
                       f"int main() {{\n{body}\nreturn 0; }}\n")
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                        "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "bux_amd", "csrc"),
                        str(src), "-o", str(exe)], check=True, capture_output=True, text=True)
        out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]

    return go


@pytest.mark.parametrize("step", [32, 64])
def test_a_contracts_steps_stay_below_its_rows(run, step):
    """A group's K steps and its mask are those of its rows below m, whatever a list's
    starts say: the sums, and every offset, are those of starts capped at m."""
    starts = [0, 5, 64, 1000, 1024, 1025, 70000, 2**31 - 1, 2**31 - 1]
    for m in (0, 1, 64, 1000, 1024, 69999, 2**31 - 128):  # the most an MXFP8 contract takes
        lines = run(f"""
  const int32_t starts[] = {{{", ".join(map(str, starts))}}};
  const ContractTiles list{{starts, 300, 300, 1, 1, {step}, {m}}};
  for (int g = 0; g < {len(starts) - 1}; ++g) {{
    Job j{{}};
    list.job(g, j);
    printf("%d %d %d %d %d\\n", j.ks_begin, j.n, j.mlo, j.mhi, int(j.mask));
  }}""")
        for g, (first, n, lo, hi, mask) in enumerate(lines):
            want = min(starts[g], m), min(starts[g + 1], m)
            if want[1] > want[0]:
                assert (lo, hi) == want
                assert first == lo // step and first + n == -(-hi // step)
                assert bool(mask) == (lo % step != 0 or hi % step != 0)
            else:
                assert n == 0


def test_tiles_of_almost_2_31_rows(run):
    """A group's tiles cover its rows once each, in order, up to the last row that 32 bits
    hold; and the blocks of the last tile that reach past them stay past them."""
    top = 2**31 - 1
    cases = [(0, 0), (5, 4), (0, 1), (7, 263), (7, 264), (0, top), (top - 1, top), (top - 255, top),
             (top - 256, top), (top - 700, top), (2**31 - 256, top)]
    lines = run("\n".join(f"""
  {{
    const int64_t n = tile_count({lo}, {hi}), first = n > 4 ? n - 4 : 0;
    for (int64_t j = first; j < n; ++j) {{
      const Tile t = tile_at(3, {lo}, {hi}, j);
      printf("%d %lld %lld %d %d %d\\n", {i}, (long long)n, (long long)j, t.group, t.lo, t.hi);
    }}
  }}""" for i, (lo, hi) in enumerate(cases)))
    for i, (lo, hi) in enumerate(cases):
        got = [line[1:] for line in lines if line[0] == i]
        n = max(0, -(-(hi - lo) // 256))
        assert got == [[n, j, 3, lo + 256 * j, min(hi, lo + 256 * (j + 1))]
                       for j in range(max(0, n - 4), n)]
    rows = run(f"""
  for (uint32_t i = 0; i < 8; ++i) printf("%lld\\n", (long long)direct_row({top - 10}, i));""")
    assert rows == [[top - 10 + 32 * i] for i in range(8)]
