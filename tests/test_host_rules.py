"""Host-side rules of the kernels' launches and bookkeeping, compiled from the
sources for the CPU (hipcc, host code only) and checked there."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


def run_host(tmp_path, body, includes=("mdg_internal.h",)):
    """The integers that a host program with this main body prints, by line."""
    src = tmp_path / "rule.hip"
    src.write_text("".join(f'#include "{i}"\n' for i in includes) +
                   "#include <cstdio>\nint main()\n{\n" + body + "\n}\n")
    exe = tmp_path / "rule"
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-Wno-unused-result",
                    "-I" + os.path.join(ROOT, "mdbas_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout
    return [[int(v) for v in line.split()] for line in out.splitlines()]


def test_reference_list_partials_fit(tmp_path):
    """The pair loop's partial rows (six doubles a block) stay in their region of
    the partial-sum buffer at every atom count, and its groups cover every row."""
    sizes = [1, 33, 3000, 30000, 262144, 1398101, 1398102, 1400000, 4194304, 4300000, 33554432,
             100000000, 2000000000]
    rows = run_host(tmp_path, "".join(
        f'printf("%d %d %d %d\\n", {n}, mdg_ref64_group({n}), mdg_ref64_blocks({n}), PART_R);\n'
        for n in sizes))
    assert [r[0] for r in rows] == sizes
    for n, group, blocks, region in rows:
        assert group >= 4
        assert group * blocks >= n > group * (blocks - 1)
        assert blocks * 6 <= region, (n, blocks)


# Sweeps at which one replica's molecules of a wavefront are converged, while the
# wavefront sweeps on to the end for another replica; for a stop at sweep C, the
# latest state that part A kept.
@pytest.mark.parametrize("conv,end,stops", [
    (range(10, 41), 40, {9: -1, 10: 10, 11: 11, 12: 11, 25: 11, 40: 11}),
    ([3, 5, *range(9, 60)], 59, {2: -1, 3: 3, 4: 3, 5: 5, 9: 9, 10: 10, 50: 10}),
    ([10, 11, 12, *range(15, 30)], 29, {10: 10, 12: 11, 15: 11, 29: 11}),
    ([0, 1], 1, {0: 0, 1: 1}),
    ([1, 3, 5, 7, 9, 10], 10, {1: -1, 4: -1, 5: 5, 10: 10}),     # the ring holds four
])
def test_shake_states_for_a_replica(tmp_path, conv, end, stops):
    conv = set(conv)
    bits = ", ".join("1" if k in conv else "0" for k in range(end + 1))
    body = f"const int conv[] = {{{bits}}};\n" """
    TriRing r;
    int at[SHK_R] = {-1, -1, -1, -1};
    for (int k = 0; k < (int)(sizeof conv / sizeof *conv); k++) {
        if (!r.keep<true>(conv[k])) continue;
        at[r.slot()] = k;
        r.put(k);
    }
    """ + f"for (int c : {{{', '.join(map(str, stops))}}}) " """{
        int slot;
        const int s = tri_resume(r.saved, c, slot);
        printf("%d %d %d\\n", c, s, s < 0 ? -1 : at[slot]);
    }"""
    for c, s, kept in run_host(tmp_path, body, includes=("mdg_shake_tri.h",)):
        assert s == kept == stops[c], (c, s, kept)
