"""The scalars that the CG and pressure kernels share through device memory: a
launch of several workgroups that reads a value which one of its own workgroups
writes would race (some workgroups see the old value, some the new one, and a
flag that ends a workgroup early can split it at a barrier).  Read off the
source, because such a race need not show in a run."""
import os
import re

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "m3tet_sph_amd", "csrc",
                   "k_sparse.hip")
ONE_WORKGROUP = {"k_pcg_look"}


def _functions(kind):
    """Name, parameters and body of the file's functions of a kind, comments removed."""
    s = re.sub(r"//[^\n]*", "", open(SRC).read())
    out = {}
    for m in re.finditer(kind + r"\s+(\w+)\s*\(", s):
        i = s.index("{", m.end())
        depth, j = 1, i + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(s[j], 0)
            j += 1
        out[m.group(1)] = (s[m.end():i], s[i:j])
    return out


def _kernels():
    return _functions(r"__global__\s+(?:__launch_bounds__\((?:[^()]|\([^()]*\))*\)\s+)?void")


def _subscripts(body, name):
    """Subscripts that the body reads and writes of an array."""
    reads, writes = set(), set()
    for m in re.finditer(r"\b%s\[" % name, body):
        depth, j = 1, m.end()
        while depth:
            depth += {"[": 1, "]": -1}.get(body[j], 0)
            j += 1
        key = re.sub(r"\s", "", body[m.end():j - 1])
        (writes if re.match(r"\s*=[^=]", body[j:]) else reads).add(key)
    return reads, writes


CASES = [(k, a) for k, (params, _) in _kernels().items() for a in ("state", "scal")
         if re.search(r"\b%s\b" % a, params) and k not in ONE_WORKGROUP]


def test_the_kernels_are_found():
    names = {k for k, _ in CASES}
    assert {"k_pcg_dir", "k_pcg_q", "k_pcg_update", "k_cg_dir", "k_cg_update", "k_pp_dir", "k_pp_update"} <= names


@pytest.mark.parametrize("kernel,array", CASES)
def test_no_scalar_is_read_and_written_by_one_launch(kernel, array):
    body = _kernels()[kernel][1]
    for name, (params, inner) in _functions(r"__device__ inline void").items():
        if re.search(r"\b%s\(%s\b" % (name, array), body) and re.search(r"\b%s\b" % array, params):
            body += inner
    reads, writes = _subscripts(body, array)
    assert writes or kernel == "k_cg_dots" or kernel == "k_pp_update" or kernel == "k_pcg_Aq", kernel
    assert not reads & writes, (kernel, reads, writes)
