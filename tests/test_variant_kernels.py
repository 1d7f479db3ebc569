"""CPU: which variants of the static table run the same kernel. The autotuner times the
first of them only (trace_first_variant, called by its C++ name)."""
import ctypes as C

import pytest


@pytest.mark.parametrize("any_hit", [False, True])
def test_first_variant_of_each_kernel(rq, any_hit):
    first = rq.lib()._ZN2rq19trace_first_variantEib
    first.restype, first.argtypes = C.c_int, [C.c_int, C.c_bool]
    vs = [v for v in rq.Context.trace_variants() if not (any_hit and v["tstack"])]
    same = {v["index"]: first(v["index"], any_hit) for v in vs}
    assert same[17] == 14
    # kernels are told apart by block, stack depth, distances and node format
    shape = {v["index"]: (v["block"], v["lds_depth"], v["tstack"], v["wide"]) for v in vs}
    for a in same:
        assert same[a] <= a and first(same[a], any_hit) == same[a]
        for b in same:
            assert (shape[a] == shape[b]) == (same[a] == same[b]), (a, b)
