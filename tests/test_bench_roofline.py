"""The benchmark's roofline names the sweep kernel that ran and counts its bytes
by what the context says of its finest level, not by the size of the mesh."""
import types

import pytest

NNZB, NNOD = 5_600_000, 200_000
# bytes of a sweep as m3_profile counts them: blocks, row lengths, four vectors
FORMS = {("fp64", 391): NNZB * 74 + NNOD * 4 + NNOD * 12 * 8, ("fp64", 0): NNZB * 76 + NNOD * 4 + NNOD * 12 * 8,
         ("mixed", 391): NNZB * 22 + NNOD * 4 + NNOD * 12 * 4, ("mixed", 0): NNZB * 24 + NNOD * 4 + NNOD * 12 * 4}


@pytest.mark.parametrize("form,windows", list(FORMS))
def test_kernel_and_bytes_of_the_finest_level(form, windows):
    import bench
    nbytes = FORMS[form, windows]
    prof = dict(n_fp64=0, t_fp64=0.0, b_fp64=0.0, n_mixed=0, t_mixed=0.0, b_mixed=0.0, n_vcycle_other=1,
                t_vcycle_other=1e-3, b_vcycle_other=1e9)
    prof.update({f"n_{form}": 10, f"t_{form}": 1e-3, f"b_{form}": 10.0 * nbytes})
    api = types.SimpleNamespace(profile=lambda *a: None, profile_read=lambda c: prof, copy_rate=lambda *a: 6200.0)
    ctx = types.SimpleNamespace(stats=lambda: dict(nnzb=[NNZB], windows=[windows]))
    r = bench.roofline(ctx, types.SimpleNamespace(nnod=NNOD), api, lambda: None, form, "c1")
    assert r["bytes_per_launch"] == nbytes
    assert r["kernel"].startswith("k_sweep_win<" if windows else "k_sweep<")
