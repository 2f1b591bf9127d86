"""The prompt products without a GPU: the rule that chooses their workgroups, and
k_gemm_rs as compiled, read from the built library's gfx950 code object with
the LLVM tools that built it."""
import os
import re
import struct
import subprocess

import pytest

import phonemap_amd as pm

LLVM = "/opt/rocm/llvm/bin/"
LIB = os.path.join(os.path.dirname(pm.__file__), "libslipstream_hip.so")


def _tool(name, *args):
    if not os.path.exists(LLVM + name):
        pytest.skip("no " + name)
    return subprocess.run([LLVM + name, *args], check=True, stdout=subprocess.PIPE, text=True).stdout


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    """The device code of the translation unit that holds k_gemm_rs."""
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    blob = open(LIB, "rb").read()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob):
        at = m.start() + 32
        for _ in range(struct.unpack_from("<Q", blob, m.start() + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", blob, at)
            target, at = blob[at + 24:at + 24 + n], at + 24 + n
            part = blob[m.start() + off:m.start() + off + size]
            if b"gfx950" in target and b"k_gemm_rs" in part:
                path = tmp_path_factory.mktemp("co") / "gemm.co"
                path.write_bytes(part)
                return str(path)
    raise AssertionError("no k_gemm_rs in " + LIB)


def test_products_keep_their_sums_in_registers(code_object):
    """Two waves per SIMD have 256 registers each. A few addresses may be
    spilled (at most 16 bytes per lane), not the 32 accumulators of a wave."""
    notes = _tool("llvm-readelf", "--notes", code_object)
    seen = 0
    for k in notes.split(".name:")[1:]:
        name = k.split()[0]
        if "k_gemm_rs" not in name:
            continue
        seen += 1
        scratch = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", k).group(1))
        assert scratch <= 16, (name, scratch)
    assert seen >= 50   # ten block types, three epilogues, two shapes (two types: one)


def _rounds(rows, T, r, t, n_cu):
    return -(-(-(-rows // r) * -(-T // t)) // n_cu)


@pytest.mark.parametrize("n_cu", [64, 256, 304])
@pytest.mark.parametrize("two", [0, 1])
def test_the_shape_is_the_cheapest_one_the_type_has(n_cu, two):
    """At 4096 columns a round of workgroups takes 10 us with one row tile (18
    for two matrices), 24 with two, 38 with four; Q4_1 and Q5_1 have no four."""
    L, m = pm.lib(), 1 + two
    for qt, most in [(2, 4), (8, 4), (9, 4), (12, 4), (3, 2), (7, 2)]:
        for rows in (40, 1024, 2816, 4096, 4100, 11008, 14336):
            for T in (1, 33, 77, 128, 200, 324, 330, 340, 512):
                cost = {1: _rounds(rows, T, 32, 32, n_cu) * (18 if two else 10), 2: _rounds(rows, T, 64 // m, 64, n_cu) * 24,
                        4: _rounds(rows, T, 128 // m, 64, n_cu) * 38}
                got = L.ss_hip_gemm_shape(rows, T, two, 4096, qt, n_cu)
                assert got <= most and cost[got] == min(c for s, c in cost.items() if s <= most), (qt, rows, T, got, cost)


@pytest.mark.parametrize("cols", [32, 256, 288, 512])
def test_the_shape_with_few_columns(cols):
    """One unit of 256 columns: always one row tile, a wave per workgroup; two:
    four row tiles where the smaller workgroups would take two rounds."""
    L = pm.lib()
    for T in (1, 130, 330, 512):
        for rows in (512, 4100, 8192):
            waves = 4 * 256   # workgroups of a round, two units
            one = -(-(-(-rows // 32) * -(-T // 32)) // waves) == 1
            assert L.ss_hip_gemm_shape(rows, T, 0, cols, 8, 256) == (1 if cols <= 256 or one else 4)
            assert L.ss_hip_gemm_shape(rows, T, 0, cols, 3, 256) == 1
