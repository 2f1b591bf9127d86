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


# ---- k_gemm_rs's counted waits ------------------------------------------------
# x comes to LDS by direct loads, four per stage and wave; at a barrier of the
# loop at most the two youngest stages may still be in flight, outside it none.
VMEM = re.compile(r"(global|buffer|scratch|flat)_(load|store|atomic)")


def _instructions(text):
    """{kernel: [(address, instruction, branch target or None)]} of a disassembly."""
    out, cur = {}, None
    for line in text.splitlines():
        m = re.match(r"([0-9a-f]+) <(.*)>:", line)
        if m:
            base, cur = int(m.group(1), 16), out.setdefault(m.group(2), [])
        elif cur is not None and "//" in line:
            ins, rest = line.strip().split("//", 1)
            to = re.search(r"<[^>+]*(?:\+0x([0-9a-f]+))?>", rest)
            target = base + int(to.group(1) or "0", 16) if to and "branch" in ins else None
            cur.append((int(rest.split(":")[0], 16), ins.strip(), target))
    return out


def _in_flight(code):
    """[(address of a barrier, direct loads to LDS that may be in flight there,
    whether it is in the main loop)]. Forward data flow: each load with the
    least number of vector memory instructions after it on any path; a wait for
    all but N of them ends the loads with N or more."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    loops = [(code[at[t]][0], a) for a, _, t in code if t is not None and t <= a]
    main = max(loops, key=lambda l: sum("s_barrier" in i and l[0] <= a <= l[1] for a, i, _ in code))
    joins = {at[t] for _, _, t in code if t is not None}
    before, work, seen = {0: {}}, [0], {}
    while work:
        i = work.pop()
        state = dict(before[i])
        while True:
            a, ins, target = code[i]
            if VMEM.match(ins):
                state = {k: min(n + 1, 64) for k, n in state.items()}
                if "_lds_" in ins:   # an older one of the same instruction keeps its place
                    for g in (2, 1, 0):
                        if (a, g) in state:
                            state[(a, g + 1)] = state.pop((a, g))
                    state[(a, 0)] = 0
            m = re.match(r"s_waitcnt.*vmcnt\((\d+)\)", ins)
            if m:
                state = {k: n for k, n in state.items() if n < int(m.group(1))}
            if ins.startswith("s_barrier"):
                seen[a] = max(seen.get(a, 0), len(state))
            nxt = [] if ins.startswith(("s_endpgm", "s_branch")) else [i + 1]
            if target is None and nxt and i + 1 not in joins:
                i += 1
                continue
            for j in nxt + ([at[target]] if target is not None else []):
                old = before.get(j)
                new = dict(state) if old is None else {k: min(old.get(k, 99), state.get(k, 99)) for k in {**old, **state}}
                if new != old:
                    before[j] = new
                    work.append(j)
            break
    return [(a, n, main[0] <= a <= main[1]) for a, n in sorted(seen.items())]


def _too_many(code):
    return [(a, n) for a, n, loop in _in_flight(code) if n > (8 if loop else 0)]


@pytest.fixture(scope="module")
def products(code_object):
    text = _tool("llvm-objdump", "-d", "--no-show-raw-insn", code_object)
    return {k: v for k, v in _instructions(text).items() if "k_gemm_rs" in k}


def test_x_has_landed_at_every_barrier(products):
    assert len(products) >= 50
    for name, code in products.items():
        assert sum("_lds_" in i for _, i, _ in code) >= 32, name   # four stages before the loop, four in it
        assert not _too_many(code), (name, _too_many(code))


def test_a_missing_load_would_be_seen(products):
    """The same reading of a listing without the loop's code loads: the waits
    then count direct loads in their place."""
    for name, code in products.items():
        loop = [a for a, n, inside in _in_flight(code) if inside]
        fewer = [(a, "s_nop 0" if i.startswith("buffer_load") and a > loop[0] else i, t) for a, i, t in code]
        assert _too_many(fewer), name
