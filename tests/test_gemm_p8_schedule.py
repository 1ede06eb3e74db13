"""The 256 x 256 GEMM on the CPU: which launches take it, and the LDS hazards of its K loop, from the
order of its source.

The kernel's two wave rows run a barrier apart, so what one row's barrier stands for depends on
which one the other row meets.  Here both rows' programs are written out from the statements of
gemm_p8_kernel and numbered by the barriers passed; of two steps of different waves only those with
a barrier between them are in order.  A half-tile may be read once all of its loads have landed,
and loaded again once all of its reads have returned.
"""

import re
from pathlib import Path

import pytest

SOURCE = Path(__file__).parents[1] / "csrc" / "kernels" / "gemm.hip"
LOADS = 2  # LDS-DMA instructions a thread issues per half-tile


def statements(text):
    text = re.sub(r"//[^\n]*|#pragma unroll|LSD_STAMP\(\d\)|for \([^)]*\)", "", text)
    return [" ".join(s.split()) for s in re.split(r"[;{}]", text.replace("Int<", "(<").replace(">{}", ">)")) if s.strip()]


@pytest.fixture(scope="module")
def parts():
    body = SOURCE.read_text().split("void gemm_p8_kernel(")[1]
    cut = lambda a, b: body.split(a, 1)[1].split(b, 1)[0]  # noqa: E731
    loop = cut("if (T > 0) {", "LSD_STAMP(2)")
    return {"mma": statements(cut("auto mma = [&](auto vm, int mh, int nh, bf16x8 (&bf)[2][2]) {", "\n  };")),
            "tile": statements(cut("auto tile = [&](int t, int buf, bf16x8 (&bx)[2][2], bf16x8 (&by)[2][2]) {", "\n  };")),
            "start": statements(loop.split("int t = 0;")[0]), "end": statements(loop.split("if (t < T)")[1])}


def program(parts, wr, T):
    """(step, what) of a wave of row wr: load / read of (buffer, half) of a K-tile, uses of
    registers, waits, barriers."""
    out = []

    def step(s, env):
        at = lambda e: eval(e, {}, env)  # noqa: E731
        if m := re.fullmatch(r"stage\((.+), (.+), (.+)\)", s):
            t, buf, h = map(at, m.groups())
            out.append(("load", (buf, h), t))
        elif m := re.fullmatch(r"read_a\((.+), (.+)\)", s):
            out.append(("read", (at(m[1]), at(m[2])), "a"))
        elif m := re.fullmatch(r"read_b\((.+), (.+), (\w+)\)", s):
            out.append(("read", (at(m[1]), 2 + at(m[2])), env.get(m[3], m[3])))
        elif m := re.fullmatch(r"mma\(\(<(\d+)>\), \d, \d, (\w+)\)", s):
            for x in parts["mma"]:
                if "mfma16" in x:
                    out.append(("use", None, ("a", env[m[2]])))
                else:
                    step(x.replace("decltype(vm)::v", m[1]), env)
        elif m := re.fullmatch(r"__builtin_amdgcn_s_waitcnt\((?:vmcnt_imm\((\d+)\)|LGKM0)\)", s):
            out.append(("landed", None, int(m[1])) if m[1] else ("returned", None, None))
        elif m := re.fullmatch(r"(?:if \(wr == (\d)\) )?__builtin_amdgcn_s_barrier\(\)", s):
            if m[1] is None or int(m[1]) == wr:
                out.append(("barrier", None, None))
        else:
            assert re.fullmatch(r"tile\(.*\)|__builtin_amdgcn_(sched_barrier|s_setprio)\(\d\)", s), s

    for s in parts["start"]:
        step(s, {})
    for t in range(T):
        regs = ("b0", "b1") if t % 2 == 0 else ("b1", "b0")
        for s in parts["tile"]:
            step(s, {"t": t, "buf": t & 1, "bx": regs[0], "by": regs[1]})
    for s in parts["end"]:
        step(s, {})
    return out


def times(prog):
    """[(half, tile, barriers before the load, before it has landed)], [(half, barriers before the
    read, before it has returned)]"""
    n, loads, reads, queue, pending = 0, [], [], [], []
    for kind, half, x in prog:
        if kind == "barrier":
            n += 1
        elif kind == "load":
            loads.append([half, x, n, None])
            queue += [loads[-1]] * LOADS
        elif kind == "landed":
            while len(queue) > x:
                queue.pop(0)[3] = n
        elif kind == "read":
            reads.append([half, n, None])
            pending.append((x, reads[-1]))
        else:  # a register's use waits for its own reads
            for r in pending:
                if kind == "returned" or r[0] in x:
                    r[1][2] = n
            pending = [r for r in pending if r[1][2] is None]
    return loads, reads, n


@pytest.mark.parametrize("T", range(1, 8))
def test_reads_between_loads(parts, T):
    rows = [times(program(parts, wr, T)) for wr in (0, 1)]
    assert rows[0][2] == rows[1][2], "both rows pass as many barriers"
    for _, reads, _ in rows:
        seen = {}
        for half, asked, back in reads:
            tile = half[0] + 2 * seen.get(half, 0)
            if tile >= T:  # the next tile's B0 behind the last one: nobody uses it
                continue
            seen[half] = seen.get(half, 0) + 1
            for loads, _, _ in rows:
                (landed,) = [x[3] for x in loads if x[0] == half and x[1] == tile]
                assert landed is not None and landed < asked, (half, tile, "read before it has landed")
                again = [x[2] for x in loads if x[0] == half and x[1] > tile]
                assert not again or back < min(again), (half, tile, "loaded again before its reads have returned")
        assert sum(seen.values()) == 4 * T


# a round of the 128 x 128 tiles is two on each of 256 CUs
@pytest.mark.parametrize("M,N,K,S,big", [(1000, 8192, 192, 1, False), (1000, 8320, 192, 1, True), (256, 32768, 64, 1, False),
                                         (256, 32896, 64, 1, True), (255, 65536, 64, 1, False), (1000, 8320, 160, 1, False),
                                         (1000, 2048, 512, 4, False), (1000, 2176, 512, 4, True), (2000, 5120, 64, 1, True),
                                         (300, 20480, 64, 1, True), (300, 20224, 64, 1, False)])
def test_which_launches(M, N, K, S, big):
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    _C.gemm_set_big_min(160)
    try:
        assert _C.gemm_big_tiles(M, N, K, S) == big
        _C.gemm_set_big_min(1 << 16)  # never
        assert not _C.gemm_big_tiles(M, N, K, S)
        _C.gemm_set_big_min(1)  # wherever it can
        assert _C.gemm_big_tiles(M, N, K, S) == (M >= 256 and K % 64 == 0)
    finally:
        _C.gemm_set_big_min(160)
