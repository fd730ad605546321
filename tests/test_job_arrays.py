"""The wf_job array that a batch hands to C holds every job's problem, flags,
symbols and lengths, whatever form the symbols come in."""
import ctypes as C

import numpy as np
import pytest

from gpumemefficient_amd import _lib
from gpumemefficient_amd.api import Job, Result, _JobArray


def _read_only(x):
    x = x.copy()
    x.flags.writeable = False
    return x


BASE = np.array([3, 0, 2, -7, 2 ** 31 - 1, 1], dtype=np.int32)
FORMS = {
    "int32": BASE,
    "read-only": _read_only(BASE),
    "strided": np.repeat(BASE, 3)[::3],
    "reversed": BASE[::-1].copy()[::-1],
    "matrix": BASE.reshape(2, 3),
    "fortran": np.asfortranarray(BASE.reshape(2, 3).T).T,
    "swapped": BASE.astype(">i4"),
    "int64": BASE.astype(np.int64),
    "list": BASE.tolist(),
    "tuple": tuple(BASE.tolist()),
    "offset": np.concatenate([[9], BASE]).astype(np.int32)[1:],
}


def test_job_array_of_all_forms():
    empty = np.zeros(0, np.int32)
    jobs = [Job(p, form, empty, ed_textbook=t, no_max=m)
            for form in FORMS.values() for p in ("LCS", "ed", 2) for t in (False, True) for m in (False, True)]
    ja = _JobArray(iter(jobs))
    assert ja.n == len(jobs) and len(ja.c) == len(jobs)
    for j, c in zip(jobs, ja.c):
        assert c.problem == {"LCS": _lib.WF_LCS, "ed": _lib.WF_ED, 2: _lib.WF_SW}[j.problem]
        assert c.flags == (_lib.WF_TILE_ED_TEXTBOOK * j.ed_textbook | _lib.WF_TILE_NO_MAX * j.no_max)
        assert (c.n1, c.n2) == (BASE.size, 0)
        assert [c.a[i] for i in range(c.n1)] == BASE.tolist()


def test_job_array_empty_and_refused():
    assert _JobArray([]).n == 0
    with pytest.raises(KeyError):
        _JobArray([Job("XYZ", BASE, BASE)])
    with pytest.raises(ValueError):
        _JobArray([Job(3, BASE, BASE)])


def test_no_copy_of_int32_symbols():
    c = _JobArray([Job("LCS", BASE, FORMS["read-only"])]).c[0]
    assert C.addressof(c.a.contents) == BASE.ctypes.data
    assert C.addressof(c.b.contents) == FORMS["read-only"].ctypes.data


def test_result_list_matches_each_structure():
    out = (_lib.wf_result * 5)()
    for i, r in enumerate(out):
        r.last, r.max_score, r.status, r.kernel_ms, r.cells = -i, 2 ** 31 - 1 - i, i, i / 3, 2 ** 63 + i
    got = Result._list(out)
    assert got == [Result._from(r) for r in out]
    assert [type(v) for v in vars(got[1]).values()] == [int, int, int, float, int]
