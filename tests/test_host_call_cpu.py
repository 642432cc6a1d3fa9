"""How Python's arguments reach a C entry point (csrc/host_call.cpp): by a callback of a known signature, on the CPU."""
import ast
import ctypes
import re
import subprocess

import pytest
import torch

from tensorline_amd.ops import build, kernels


class Pair(ctypes.Structure):
    _fields_ = [("a", ctypes.c_void_p), ("b", ctypes.c_float)]


def enter(kinds, *args):
    """What a callee with parameters of ``kinds`` is given for ``args``, and the status that comes back."""
    seen = []
    c = ctypes.CFUNCTYPE(ctypes.c_int, *kinds)(lambda *a: (seen.extend(a), -7)[1])
    kernels._entry_point("tl_last_error")            # (loads the module)
    status = kernels._enter(ctypes.cast(c, ctypes.c_void_p).value, *args)
    return seen, status


def test_arguments_of_every_kind_in_any_order():
    t, pair = torch.arange(5.0), Pair(3, 0.25)
    i, q, f, p = ctypes.c_int, ctypes.c_longlong, ctypes.c_float, ctypes.c_void_p
    kinds = [p, f, q, i, p, f, i, i, q, f, ctypes.c_uint32, i, p, p, f, q, f]
    args = [t, 0.1, -(1 << 40), -3, None, 2.5, True, ctypes.c_int(-9), ctypes.c_longlong(1 << 50), ctypes.c_float(-1.5),
            ctypes.c_uint32(0xffffffff), 1 << 31, pair, ctypes.c_void_p(0x7fff12345678), 1e30, t[2:].data_ptr(), -0.0]
    seen, status = enter(kinds, *args)
    want = [t.data_ptr(), ctypes.c_float(0.1).value, -(1 << 40), -3, None, 2.5, 1, -9, 1 << 50, -1.5, 0xffffffff, -(1 << 31),
            ctypes.addressof(pair), 0x7fff12345678, ctypes.c_float(1e30).value, t.data_ptr() + 8, 0.0]
    assert seen == want and status == -7


def test_as_many_arguments_as_there_is_room_for():
    seen, _ = enter([ctypes.c_int] * 56 + [ctypes.c_float] * 8, *range(56), *[k + 0.5 for k in range(8)])
    assert seen == list(range(56)) + [k + 0.5 for k in range(8)]
    for args in ([0] * 57, [0.0] * 9):
        with pytest.raises(TypeError):
            enter([], *args)


@pytest.mark.parametrize("bad", ["text", b"", ctypes.c_double(1.0), [1], object(), (ctypes.c_int * 2)()])
def test_other_arguments_are_refused(bad):
    with pytest.raises((TypeError, AttributeError)):
        enter([ctypes.c_void_p], bad)


def test_the_same_without_the_module(monkeypatch):
    """Through ctypes: the same parameters are filled, the same arguments refused."""
    kernels._entry_point("tl_last_error")
    monkeypatch.setattr(kernels, "_enter", kernels._enter_by_ctypes)
    test_arguments_of_every_kind_in_any_order()
    seen, _ = enter([ctypes.c_int] * 56 + [ctypes.c_float] * 8, *range(56), *[k + 0.5 for k in range(8)])
    assert seen == list(range(56)) + [k + 0.5 for k in range(8)]
    for bad in ("text", b"", ctypes.c_double(1.0), [1], object(), (ctypes.c_int * 2)()):
        test_other_arguments_are_refused(bad)


def test_the_module_is_left_out_where_it_cannot_be_built(monkeypatch, tmp_path):
    """No headers of Python: the library is built without them and loads without Python's symbols, calls go through ctypes."""
    assert all(build.CALL_SOURCE != src for src in build.sources())
    symbols = subprocess.run(["nm", "-D", "--undefined-only", build.ensure_built()], capture_output=True, text=True, check=True).stdout
    assert "hipLaunchKernel" in symbols and not re.search(r"\b_?Py[A-Z_]", symbols)
    monkeypatch.setattr(build, "_candidate_dirs", lambda: [str(tmp_path)])
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path / "none")})
    assert build.find_call() is None and build.ensure_call(verbose=False) is None
    monkeypatch.setattr(kernels, "_enter", None)
    monkeypatch.setattr(build, "ensure_built", lambda: None)
    kernels._entry_point("tl_last_error")
    assert kernels._enter is kernels._enter_by_ctypes


def _signatures():
    """(name, a letter for each parameter: f float, w anything else) of the library's entry points that return a status."""
    out = {}
    for path in build.sources():
        with open(path, encoding="utf-8") as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        for name, params in re.findall(r'extern "C" int (tl_\w+)\(([^)]*)\)', text):
            kinds = []
            for p in params.split(","):
                assert "*" in p or "double" not in p, (name, p)
                kinds.append("f" if re.match(r"\s*(const\s+)?float\s+\w+\s*$", p) else "w")
            out[name] = "".join(kinds)
    return out


def _kinds(args, scope, returns):
    """The letters of a call's arguments: a float is a float literal, ``float(..)``, or a name that such a value was given to."""
    out = ""
    for a in args:
        if isinstance(a, ast.Starred):
            given = scope.get(a.value.id)
            assert isinstance(given, ast.Tuple), f"line {a.lineno}: what *{a.value.id} holds is not seen"
            out += _kinds(given.elts, scope, returns)
        else:
            if isinstance(a, ast.Name) and a.id in scope:
                a = scope[a.id]
            is_float = (isinstance(a, ast.Constant) and isinstance(a.value, float)) or (
                isinstance(a, ast.Call) and isinstance(a.func, ast.Name) and a.func.id == "float")
            out += "f" if is_float else "w"
    return out


def test_every_call_has_the_arguments_its_entry_point_takes():
    """Neither the module nor ctypes knows an entry point's parameters: the calls in kernels.py are held against the sources, number
    and kind of every argument."""
    signatures, seen = _signatures(), 0
    tree = ast.parse(open(kernels.__file__, encoding="utf-8").read())
    functions = [n for n in tree.body if isinstance(n, ast.FunctionDef)]
    returns = {f.name: [r.value for r in ast.walk(f) if isinstance(r, ast.Return) and r.value is not None] for f in functions}
    for f in functions:
        scope = {}                                       # names that hold a tuple or a float, in this function
        for n in ast.walk(f):
            if isinstance(n, ast.Assign):
                for target in n.targets:
                    if isinstance(target, ast.Name) and isinstance(n.value, (ast.Tuple, ast.Call)):
                        scope[target.id] = n.value
                    elif isinstance(target, ast.Tuple) and isinstance(n.value, ast.Call) and isinstance(n.value.func, ast.Name):
                        for i, name in enumerate(target.elts):
                            tuples = {ast.dump(ast.Tuple([ast.Constant(c) for c in _kinds(r.elts[i].elts, {}, returns)], ast.Load())): r.elts[i]
                                      for r in returns.get(n.value.func.id, []) if isinstance(r, ast.Tuple) and isinstance(r.elts[i], ast.Tuple)}
                            assert len(tuples) <= 1, f"line {n.lineno}: {name.id} holds arguments of several kinds"
                            for given in tuples.values():
                                scope[name.id] = given
        for n in ast.walk(f):
            if isinstance(n, ast.Call) and isinstance(n.func, ast.Name) and n.func.id == "_call" and isinstance(n.args[0], ast.Constant):
                got = _kinds(n.args[1:], scope, returns)
                assert got == signatures[n.args[0].value], f"kernels.py:{n.lineno}: {n.args[0].value} is given {got}"
                seen += 1
    assert seen > 50
    wrong = ast.parse("_call('tl_scale_cap', z, n, scale, float(cap), _stream())").body[0].value
    assert _kinds(wrong.args[1:], {}, returns) != signatures["tl_scale_cap"]
