"""LDS of the relaxation kernel as the planner asks for it: its arrays do not overlap, and
it keeps as many workgroups on a CU as rows without periodic copies would.

A CU has 160 KB, given out in units of 1280 B, static arrays included, and registers for
12 waves.  The sizes of the static arrays are the compiler's.
"""
import ctypes
import os

import numpy as np
import pytest

from firecore_amd import build as fb
from firecore_amd import native

FORMS = {"plain": 0, "constant": 1, "learned": 2}
MAXC = 4  # components


@pytest.fixture(scope="module")
def lib():
    L = native.lib()
    L.fc_relax_lds_bytes.restype = ctypes.c_int
    return L


@pytest.fixture(scope="module")
def static():
    if not os.path.exists(fb.RESOURCES):
        pytest.skip("library built elsewhere")
    res = fb.resources()

    def of(block, hb, form):
        tag = "relax_persistent_kernelILi%dELb%dELi%dE" % (block, hb, FORMS[form])
        return [r for k, r in res.items() if tag in k][0]["LDS Size"]
    return of


def per_cu(block, dynamic, static):
    units = -(-(dynamic + static) // 1280)
    return min(12 // (block // 64), 128 // units)


@pytest.mark.parametrize("nmax,mmax,block,want", [(256, 121, 256, (3, 3, 3)), (256, 128, 256, (3, 3, 3)),
                                                  (192, 100, 192, (4, 4, 4)), (128, 66, 128, (6, 6, 6)),
                                                  (64, 31, 64, (12, 12, 11))])
def test_resident_workgroups(lib, static, nmax, mmax, block, want):
    for hb in (0, 1):
        got = tuple(per_cu(block, lib.fc_relax_lds_bytes(nmax, mmax, block, int(f == "learned"), 0, hb),
                           static(block, hb, f)) for f in FORMS)
        assert got == want, (hb, got)


@pytest.mark.parametrize("block", [64, 128, 192, 256])
def test_residency_of_plain_rows(lib, static, block):
    """Rows without copies: 48 B an atom and 176 B a node, reaction rows of 64 + n/2
    entries, all exclusion words, activations over reactions to words, 16 floats per
    component for the rigid fit."""
    nw, less = block // 64, []
    for hb in (0, 1):
        for form in FORMS:
            learned = int(form == "learned")
            for n in range(1, block + 1):
                for m in range(1, min(n, 2 * block - n) + 1, 3):
                    facc = 48 * n + 16 * m
                    end = facc + 16 * nw * (64 + n // 2) + 160 * m + 4 * n * (n // 64 + 1)
                    if learned:
                        end = (max(end, facc + 136 * n) + 15) // 16 * 16 + (4 * (m + MAXC) + 15) // 16 * 16
                    st = static(block, hb, form)
                    plain = per_cu(block, end, st + (0 if form == "plain" else MAXC * (16 - 10) * 4))
                    have = per_cu(block, lib.fc_relax_lds_bytes(n, m, block, learned, 0, hb), st)
                    if have < plain:
                        less.append((form, hb, n, m, have, plain))
    assert not less, (len(less), less[:3])


@pytest.mark.gpu
@pytest.mark.parametrize("natoms,block", [(20, 64), (44, 64), (61, 64), (64, 64), (122, 128), (126, 128), (190, 192),
                                          (248, 256), (251, 256)])
def test_second_activation_buffer_costs_no_workgroup(static, natoms, block):
    lds = {}
    try:
        native.set_proposal_weights(np.load("firecore_amd/proposal_weights.npy"))
        for mode in (2, 1):
            native.set_learned_inkernel(mode)
            native.set_precond(2, 3.0, 127.0)
            native.init_workload(0, 1, 0, natoms, natoms, 0.1, None, 0.1)
            lds[mode], = [c["lds"] for c in native.class_info() if c["block"] == block]
    finally:
        native.set_learned_inkernel(2)
        native.set_precond(0)
    st = static(block, 0, "learned")
    assert per_cu(block, lds[1], st) >= per_cu(block, lds[2], st), lds


@pytest.mark.parametrize("learned,h2lds,hb", [(0, 0, 0), (0, 0, 1), (1, 0, 0), (1, 0, 1), (1, 1, 0), (1, 1, 1)])
def test_arrays_do_not_overlap(lib, learned, h2lds, hb):
    names = ["pos", "pi", "fnb", "re", "hb", "facc", "fself", "fng", "mask", "h", "nb", "gain", "h2", "end"]
    o = np.zeros(len(names), np.int32)
    for block in (64, 128, 192, 256):
        for n in list(range(1, 9)) + [31, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256]:
            if n > block:
                continue
            for m in sorted({1, n // 2 or 1, n}):
                lib.fc_relax_lds_offsets(n, m, block, learned, h2lds, hb, o.ctypes.data_as(ctypes.POINTER(ctypes.c_int)))
                at = dict(zip(names, o.tolist()))
                kn = (n // 2 & ~3) + 4  # offsets the pair loop computes; it reads two rows further ahead
                size = dict(pos=16 * (n - 1 + kn), pi=16 * m, fnb=16 * n, re=8 * (n - 1 + kn),
                            hb=4 * (n - 1 + kn) * hb, facc=16 * (block // 64) * (64 + n // 2), fself=16 * m,
                            fng=128 * m, mask=4 * n * (n // 2 // 32))
                if learned:
                    size.update(gain=4 * (m + MAXC), h2=136 * n * h2lds)
                seq = sorted((at[k], at[k] + s, k) for k, s in size.items() if s)
                for (_, e, k), (b, _, k2) in zip(seq, seq[1:]):
                    assert e <= b, (block, n, m, k, k2)
                assert seq[-1][1] <= at["end"] == lib.fc_relax_lds_bytes(n, m, block, learned, h2lds, hb)
                for k, row in (("pos", 16), ("re", 8)) + ((("hb", 4),) if hb else ()):
                    assert at[k] + row * (n + kn + 1) <= at["end"]  # rows read ahead
                for k in ("pos", "pi", "fnb", "facc", "fself", "fng", "h", "h2"):
                    assert at[k] % 16 == 0
                if learned:  # activations and neighbours lie on arrays that the step refills
                    assert at["fnb"] + 16 * n <= at["h"] and at["h"] + 136 * n <= at["nb"]
                    assert at["nb"] + 8 * n <= at["gain"] and at["nb"] % 8 == 0
                    assert at["mask"] + size["mask"] <= at["gain"]
