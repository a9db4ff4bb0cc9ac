"""The rules by which a step of single tokens takes its kernels: what they accept has to be what the kernels take, and a step padded to
more rows has to be decided as the step itself.  No GPU: the rules read sizes only."""
from types import SimpleNamespace

import pytest
import torch

from tempura_amd.kernels import ops


def _step(n, longest):
    return SimpleNamespace(num_tokens=n, num_requests=n, num_single=n, max_context_len=longest)


@pytest.mark.parametrize("what,takes", [("plain", True), ("odd state rows", False), ("odd place in the state", False), ("odd first column", False),
                                        ("odd state rows without a convolution", True), ("more requests than a grid has rows", False)])
def test_rows_at_odd_places_keep_the_separate_kernels(what, takes):
    """The kernel that takes a projection's rows reads pairs of floats, and has a request a row of its grid."""
    heads, kv, d, taps = 4, 2, 64, 4
    width = (heads + 2 * kv) * d
    n = 65536 if what.startswith("more") else 3
    rows = torch.empty((1, width + 8)).expand(n, -1)
    k = torch.empty((4, kv, 16, d), dtype=torch.bfloat16)
    state = torch.empty((n if n < 9 else 1, (taps - 1) * width + 10 + ("odd state rows" in what)))
    got = ops.attention_rows_ok(rows, _step(n, 300), heads, kv, d, d, k, 0 if "without" in what else taps, 0, 3 if "column" in what else 2, state,
                                5 if "place" in what else 4)
    assert got is takes


def _same_for_padded(rule):
    for n in [*range(1, 140), 200, 256, 300]:
        assert rule(n) == rule(ops.decode_rows_padded(n)), n


@pytest.mark.parametrize("longest", [30, 513, 1100, 5000])
@pytest.mark.parametrize("kvh,window,taps,step_heads", [(8, 1024, 0, 16), (4, 1024, 0, 8), (3, 0, 4, 5), (12, 0, 0, 24)])
def test_a_padded_step_runs_a_mixer_beside_the_attention_as_the_step_itself(longest, kvh, window, taps, step_heads):
    def rule(n):
        ctx = _step(n, longest)
        beside = ops.attention_beside_ok(ctx, 2 * kvh, kvh, window, taps, step_heads)
        return beside, ops._rows_splits(ctx, 2 * kvh, kvh, window, 0, 0, taps > 0, beside)
    _same_for_padded(rule)


@pytest.mark.parametrize("longest", [200, 1000, 3000])
@pytest.mark.parametrize("heads,kvh", [(8, 8), (24, 12), (6, 3), (80, 5), (32, 1)])
def test_a_padded_step_has_the_splits_and_waves_of_the_step_itself(longest, heads, kvh):
    def rule(n):
        splits = ops._decode_splits(n, heads, kvh, longest, 0, 0, 0, True)
        return splits, ops._decode_waves(n, heads, kvh, splits)
    _same_for_padded(rule)


@pytest.mark.parametrize("longest", [200, 800, 1500, 3000])
@pytest.mark.parametrize("kvh,dim,window", [(8, 128, 0), (8, 64, 0), (3, 128, 0), (8, 128, 1024), (1, 64, 0)])
def test_a_padded_step_takes_the_projections_rows_as_the_step_itself(longest, kvh, dim, window):
    _same_for_padded(lambda n: ops.attention_rows_pays(_step(n, longest), kvh, dim, window))


def test_few_blocks_or_short_streams_of_keys_take_the_projections_rows():
    pays = lambda n, longest, *rest: ops.attention_rows_pays(_step(n, longest), 8, *rest)
    assert pays(32, 100000, 128) and pays(64, 2000, 128) and not pays(64, 3000, 128) and pays(64, 3000, 64) and not pays(64, 5000, 64)
    assert pays(128, 500, 128) and not pays(128, 800, 128) and pays(128, 800, 64) and not pays(128, 1500, 64) and pays(64, 100000, 128, 1024)


def test_entry_points_are_called_as_they_are_declared():
    """Every call into the kernel library names an entry point of its sources and brings as many arguments as that has; a pointer, a size, a
    number and a flag of one of them are declared as such."""
    import ast
    import ctypes
    import inspect
    from tempura_amd.kernels import ops
    declared = ops.entry_points()
    calls = [c for c in ast.walk(ast.parse(inspect.getsource(ops))) if isinstance(c, ast.Call) and getattr(c.func, "id", "") == "_call"]
    names = [c.args[0].value for c in calls if isinstance(c.args[0], ast.Constant)]
    assert len(names) > 50 and set(names) <= set(declared)
    for c in calls:
        if isinstance(c.args[0], ast.Constant) and not any(isinstance(a, ast.Starred) for a in c.args):
            assert len(c.args) - 1 == len(declared[c.args[0].value][1]), c.args[0].value
    result, args = declared["tp_linear_fused"]
    assert result is ctypes.c_int and args[0] is args[-1] is ctypes.c_void_p and args[2] is ctypes.c_int
    assert args[11] is ctypes.c_size_t and args[14] is ctypes.c_float
    assert declared["tp_last_error"][0] is ctypes.c_char_p and declared["tp_linear_f32_scratch"][0] is ctypes.c_size_t


def test_every_argument_of_a_call_has_the_declared_type():
    """No definition in the sources is overlooked, and each argument whose kind shows in the call (an address, a float, a whole number), those that come
    as a row scale's or a split norm's three included, stands where one of that kind is declared."""
    import ast
    import ctypes
    import inspect
    import re
    from tempura_amd.csrc.build import sources
    from tempura_amd.kernels import ops
    declared = ops.entry_points()
    assert sum(len(re.findall(r'^extern "C"', open(p, encoding="utf-8").read(), re.M)) for p in sources()) == len(declared)
    address, number = {ctypes.c_void_p}, {ctypes.c_float, ctypes.c_double}
    whole = {ctypes.c_int, ctypes.c_uint, ctypes.c_size_t, ctypes.c_long, ctypes.c_longlong, ctypes.c_ulonglong}
    kinds = {"_ptr": address, "_stream": address, "at": address, "byref": address, "float": number, "c_float": number, "c_double": number, "int": whole,
             "len": whole, "max": whole, "min": whole, "_dt": whole, "_dtcode": whole, "c_size_t": whole, "c_longlong": whole, "c_ulonglong": whole}
    starred = {"pre": [address, whole, number], "post": [address, address, address]}

    def kind_of(arg):
        if "data_ptr" in ast.dump(arg):
            return address
        if isinstance(arg, ast.Constant) and arg.value is not None:
            return number if isinstance(arg.value, float) else whole
        return kinds.get(getattr(arg.func, "id", getattr(arg.func, "attr", ""))) if isinstance(arg, ast.Call) else None

    seen = 0
    for c in ast.walk(ast.parse(inspect.getsource(ops))):
        if not (isinstance(c, ast.Call) and getattr(c.func, "id", "") == "_call" and isinstance(c.args[0], ast.Constant)):
            continue
        name, got = c.args[0].value, []
        for a in c.args[1:]:
            got += starred[a.value.id] if isinstance(a, ast.Starred) else [kind_of(a)]
        types = declared[name][1]
        assert len(got) == len(types), name
        for i, (kind, want) in enumerate(zip(got, types)):
            assert kind is None or want in kind, (name, i, want)
            seen += kind is not None
    assert seen > 600
