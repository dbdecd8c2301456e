"""Which kernels a call runs, and what it allocates, on a HIP runtime that runs
nothing (fake_hip/): the rules of the dispatch on the CPU."""
import json
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    from hypno_amd import _lib
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "fake_hip", "fake_hip.cpp")], check=True)

    def run(*steps):
        p = subprocess.run([sys.executable, os.path.join(HERE, "fake_hip", "calls.py"), so,
                            _lib.LIB_PATH, json.dumps(steps)], capture_output=True, text=True,
                           timeout=100)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout)

    return run


def _kernels(result):
    """Short names of a call's launches: mangled name -> identifier<int and bool
    template arguments>."""
    st, log = result
    assert st == 0, result
    out = []
    for line in log:
        if line.startswith("launch "):
            name = line.split()[1]
            # the last length-prefixed identifier before the template arguments
            ident = args = ""
            i = name.index("5hypno") + 6
            while i < len(name):
                if name.startswith("12_GLOBAL__N_1", i):
                    i += 14
                    continue
                g = re.match(r"(\d+)", name[i:])
                if not g:
                    break
                k = i + len(g.group(1))
                ident, i = name[k:k + int(g.group(1))], k + int(g.group(1))
            if name[i:i + 1] == "I":
                args = re.match(r"I((?:L[ib]\d+E)+)", name[i:])
                args = ",".join(re.findall(r"L[ib](\d+)E", args.group(1))) if args else ""
            out.append(f"{ident}<{args}>" if args else ident)
    return out


# Q4_0 prompts: 256 x 256 block tiles where they fill the chip evenly, the 16x16x32
# kernel elsewhere (us, that kernel and block tiles of 128 / 256 rows: 512 x 14336,
# K 4096 90 / 91 / 136; 2048 x 4096, K 4096 98 / 100 / 141; 2048 x 4096, K 14336
# 326 / 323 / 458; 1024 x 14336, K 4096 165 / 168 / 145; 2048 x 14336 332 / 340 / 290).
@pytest.mark.parametrize("tokens,n,m,block", [
    (512, 14336, 4096, False), (2048, 4096, 4096, False), (2048, 4096, 14336, False),
    (2048, 3072, 8192, False), (1024, 4096, 14336, False), (512, 8192, 3072, False),
    (512, 3072, 8192, False), (1500, 11008, 4096, False), (3000, 5632, 2048, False),
    (2048, 14336, 4096, True), (1024, 14336, 4096, True), (2048, 5632, 2048, True),
    (2048, 8192, 3072, True), (4096, 4096, 14336, True), (2048, 6144, 4096, True)])
def test_q4_0_prompt_tiles(calls, tokens, n, m, block):
    got = _kernels(calls(["q4_0", n, m, tokens])[0])
    assert ("gemm_block_kernel<0,8,0,1>" in got) == block, got
    assert any(k.startswith("q4_0_gemm_exact_kernel") for k in got) == (not block), got


# Calls that ran without a workspace, or with a smaller one, before the GEMMs that
# want one: with no device memory left, and under capture on a stream that holds
# too little, they still run.
@pytest.mark.parametrize("call,room,plain", [
    (["q4_0", 2400, 2080, 17], 0, "gemv_any_kernel<0,64>"),
    (["q8_0", 2880, 7200, 33], 0, "gemv_any_kernel<1,64>"),
    (["f16", 2880, 7200, 64], 0, "f16_gemv_fast_kernel"),
    # (the tile kernel's fp16 rows; the expanded fp16 weights and activations)
    (["q4_0", 640, 2880, 16], 128 * 2880 * 2 + 512, "gemm_kernel"),
    (["q8_0", 255, 8192, 127], 255 * 8192 * 2 + 128 * 8192 * 2 + (2 << 20), "f16_gemm")])
def test_no_room_for_a_workspace(calls, call, room, plain):
    full, first = calls(["room", room], call)[1], calls(call)[0]
    assert any(plain in k for k in _kernels(full)), full
    assert not any(plain in k for k in _kernels(first)), first
    # under capture, the stream holding what that plain run left
    steps = [["room", room], call, ["room", None], ["capture", 1], call, ["capture", 0], call]
    *_, captured, _, after = calls(*steps)
    assert any(plain in k for k in _kernels(captured)), captured
    assert not any(line.startswith(("malloc", "free")) for line in captured[1])
    assert _kernels(after) == _kernels(first)


def test_captured_workspace_is_kept(calls):
    """A workspace that went into a captured graph is not freed by a larger call;
    one that did not is, and each next one is at least twice as large as a kept
    one."""
    small, large, largest = (["q4_0", 2400, 2080, t] for t in (17, 300, 700))
    res = calls(small, ["capture", 1], small, ["capture", 0], large, largest)
    logs = [r[1] for r in res if r]
    assert all(r[0] == 0 for r in res if r)
    sizes = [[int(x.split()[1]) for x in log if x.startswith("malloc")] for log in logs]
    freed = [[int(x.split()[1]) for x in log if x.startswith("free")] for log in logs]
    assert [len(s) for s in sizes] == [1, 0, 1, 1]
    assert freed == [[], [], [], sizes[2]]
    assert sizes[2][0] >= 2 * sizes[0][0]


def _all_kernels(calls, steps):
    return {k for r in calls(*steps) for k in _kernels(r)}


def test_cases_reach_every_instantiation(calls):
    """The GPU tests' lists of shapes run every instantiation of the kernels that
    they are there for."""
    import test_any_shape
    import test_block_f16x
    import test_pair_gemm
    got = _all_kernels(calls, [[dt, n, m, t] for dt, t, n, m in test_any_shape.CASES])
    assert {k for k in got if k.startswith(("gemm_block", "gemv_any"))} >= {
        *(f"gemm_block_kernel<{f},{mt},{odd},3>" for f in (0, 1)
          for mt, odd in ((1, 0), (1, 1), (2, 1))),
        *(f"gemv_any_kernel<{f},{lanes}>" for f in (0, 1) for lanes in (8, 16, 32, 64))}
    assert "block_split_reduce_kernel" in got
    got = _all_kernels(calls, [[dt, n, m, t] for dt, t, n, m in test_block_f16x.CASES])
    assert {k for k in got if k.startswith("gemm_block")} == {
        *(f"gemm_block_kernel<1,{mt},0,1>" for mt in (2, 4, 8)), "gemm_block_kernel<0,8,0,1>"}
    odd = [["q8_0", n, m, t, {"w_off": 2}] for t, n, m in
           ((40, 129, 320), (64, 300, 1088), (130, 300, 1088), (300, 5000, 1088))]
    got = [_kernels(r) for r in calls(*odd)]
    assert all(k[0] == "q8_0_rows_to_f16_kernel" for k in got)
    assert [any("stream" in x for x in k) for k in got] == [True, True, False, False]
    for cases, kind, col in ((test_pair_gemm.COL_CASES, "q4_0_col", 1),
                             (test_pair_gemm.F16_CASES, "f16", 0)):
        got = calls(*([kind, c[1], c[2], c[0], {"extra": -c[3] if col else 0}] for c in cases))
        tiles = [[f"gemm_pair_kernel<{mt},{col}>" in _kernels(r) for mt in (1, 2)] for r in got]
        split = ["block_split_reduce_kernel" in _kernels(r) for r in got]
        assert {(t[1], s) for t, s in zip(tiles, split) if any(t)} == {
            (False, False), (False, True), (True, False), (True, True)}
