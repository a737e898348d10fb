"""The rule that keeps an addition whose operands reach past 31-bit byte offsets away from
the blocked kernels: compared with every offset that the kernels form, for strides on
both sides of the limit (compiled for the host, no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
FIELDS = "kc kx1 kx2 cap m n cu_rs cu_cs cv_rs cv_cs lds xu_rs xu_cs xs_ld xv_rs xv_cs".split()
BASE = dict(kc=3, kx1=2, kx2=4, cap=8, m=64, n=48, cu_rs=1, cu_cs=64, cv_rs=48, cv_cs=1, lds=8, xu_rs=2, xu_cs=1,
            xs_ld=4, xv_rs=48, xv_cs=1)
LIMIT = 0x7fffff00


def reach(x, size):
    """The largest byte offset of an element that an addition reads or writes, or None below zero."""
    # the update writes as many columns as the rank it finds: at most the capacity and all columns of the sum
    k = max(x["kc"], min(x["cap"], x["kc"] + x["kx2"]))
    ends = [(x["m"], x["cu_rs"], k, x["cu_cs"]), (k, x["cv_rs"], x["n"], x["cv_cs"]), (k, x["lds"], k, 1),
            (x["m"], x["xu_rs"], x["kx1"], x["xu_cs"]), (x["kx1"], x["xs_ld"], x["kx2"], 1),
            (x["kx2"], x["xv_rs"], x["n"], x["xv_cs"])]
    ends = [(r, rs, c, cs) for r, rs, c, cs in ends if r > 0 and c > 0]
    if any(rs < 0 or cs < 0 for _, rs, _, cs in ends):
        return None
    return max((((r - 1) * rs + (c - 1) * cs) * size for r, rs, c, cs in ends), default=0)


@pytest.fixture(scope="module")
def near(tmp_path_factory):
    gxx = shutil.which("g++") or shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
    exe = tmp_path_factory.mktemp("near") / "near_test"
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{ROOT / 'frank_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cxx" / "near_test.cpp"), "-o", str(exe)], check=True)

    def run(cases):
        text = "\n".join(" ".join(str(x[f]) for f in FIELDS) for x in cases)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(bool(int(v)) for v in line.split()) for line in out.splitlines()]
    return run


def test_slots_as_they_are_laid_out(near):
    assert near([BASE]) == [(True, True)]


@pytest.mark.parametrize("field", ["cu_rs", "cu_cs", "cv_rs", "cv_cs", "xu_rs", "xu_cs", "xv_rs", "xv_cs", "lds", "xs_ld"])
@pytest.mark.parametrize("kc,kx2,cap", [(3, 4, 8), (1, 1, 2), (1, 8, 16), (8, 4, 8), (0, 4, 8), (1, 40, 128)])
def test_limit_of_every_stride(near, field, kc, kx2, cap):
    cases = []
    for p in range(20, 31):
        for d in (-1, 0, 1):
            x = dict(BASE, kc=kc, kx2=kx2, kx1=min(2, kx2), cap=cap)
            x[field] = (1 << p) // 3 + d
            cases.append(x)
            cases.append(dict(x, **{field: (1 << p) + d}))
    for x, got in zip(cases, near(cases)):
        for size, g in zip((8, 4), got):
            if g:  # taken: no offset past the limit
                r = reach(x, size)
                assert r is not None and r < LIMIT
            else:  # refused: only where an offset, or a stride by itself, reaches it
                used = [x[f] for f in FIELDS[6:]]
                assert reach(x, size) >= LIMIT - size or max(used) * size >= LIMIT - size


@pytest.mark.parametrize("field", ["cu_rs", "cu_cs", "cv_rs", "cv_cs", "xu_rs", "xu_cs", "xv_rs", "xv_cs"])
def test_negative_strides_are_refused(near, field):
    assert near([dict(BASE, **{field: -1})]) == [(False, False)]


def test_columns_that_the_update_adds_count(near):
    """One column is there, 30 more may be written: at 2^25 doubles apart they lie past 2^31 bytes."""
    x = dict(BASE, kc=1, kx2=40, cap=31, cu_cs=1 << 25)
    assert reach(x, 8) >= 1 << 31
    assert near([x]) == [(False, False)]
