"""CPU checks of the typed Python entry (csrc/call.cpp): conversions, what it refuses, and the tensor checks beside it."""
import copy
import ctypes as C
import os
import pickle
import subprocess
import sys

import numpy as np
import pytest
import torch

from pikv_amd import _native as N, dense, ops


def test_every_entry_point_is_there():
    for module in (N.entries(), N.entries().of_checked):
        assert set(N.SIGNATURES) - {"pikv_status_string"} <= set(dir(module))


def test_sizes_agree_with_ctypes():
    for name, args in (("pikv_router_workspace_bytes", (32768, 8, 2)), ("pikv_evict_workspace_bytes", (3, 70000)),
                       ("pikv_decode_attend_workspace_bytes", (4, 32, 128, 5000)), ("pikv_capacity_slots_static_max", ())):
        assert N.size(name, *args) == getattr(N.lib(), name)(*args)


@pytest.mark.parametrize("array", [[8, 16], (8, 16), np.array([8, 16], dtype=np.int32)])
def test_host_arrays_reach_the_library(array):
    """A bad layer width inside a host array is found by the library itself, whatever the array came as."""
    def call(widths):
        return N.entries().pikv_linear_group(64, 4, 128, 2, [64, 64], [64, 64], widths, [0, 1], 0, None, None, None, [64, 64],
                                             None, 0, None)
    assert call(array) == -3 and call([32, 0]) == -2     # widths that are no multiple of 32; no width at all


def test_refusals():
    f = N.entries()
    with pytest.raises(TypeError):
        f.pikv_evict_workspace_bytes(1)
    with pytest.raises(OverflowError):
        f.pikv_evict_workspace_bytes(1 << 40, 5)
    with pytest.raises(TypeError):
        f.pikv_evict_workspace_bytes(1.5, 5)
    with pytest.raises(AttributeError):
        f.pikv_h2o_budget(object(), 1, 0.1, 0.1, None, None, None)
    with pytest.raises(ValueError):
        f.pikv_linear_tiled(64, 4, 64, 1, [64] * 5000, [64], [4], [64], None)
    with pytest.raises(N.PiKVNativeError):
        N.call("pikv_h2o_budget", None, 1, 0.1, 0.1, None, None, None)


class _Tensor:
    def __init__(self, is_cuda):
        self.is_cuda, self.asked = is_cuda, 0

    def data_ptr(self):
        self.asked += 1
        return 64


@pytest.mark.parametrize("name", sorted(set(N.SIGNATURES) - {"pikv_status_string"}))
def test_pointer_parameters_take_what_they_are(name):
    """A pointer that a kernel reads never comes from host memory, a host array never from the GPU.  (No call here gets as far
    as the library.)"""
    _, types = N.SIGNATURES[name]
    plain = [0.0 if t in (C.c_float, C.c_double) else 0 if t is not C.c_void_p and not hasattr(t, "contents") else None
             for t in types]
    for i, t in enumerate(types):
        if t is C.c_void_p:
            wrong = [[64], (64,), np.zeros(4, np.float32), np.int64(64), (C.c_float * 4)(), b"abcd", bytearray(8),
                     torch.zeros(4), _Tensor(False)]
        elif hasattr(t, "contents"):
            numbers = t._type_ is not C.c_void_p
            wrong = [64, _Tensor(True), torch.zeros(4), np.zeros(4, np.float16), np.zeros((2, 2), np.int32), np.int64(64),
                     (C.c_double * 2)(), b"abcd", np.zeros(8, np.int64)[::2]]
            wrong += [C.c_void_p(64), [None], [_Tensor(True)], np.zeros(4, np.int32 if t._type_ is C.c_float else np.float32)] if numbers else [
                [torch.zeros(4)], [np.zeros(4)], [[64]], np.zeros(4, np.int32)]
        else:
            continue
        for w in wrong:
            # of callers that have checked their tensors everything but those is refused the same way
            forms = [N.entries()] if isinstance(w[0] if isinstance(w, list) else w, (torch.Tensor, _Tensor)) else [N.entries(), N.entries().of_checked]
            for f in forms:
                with pytest.raises((TypeError, ValueError)):       # (numpy: a strided array gives no plain buffer, a ValueError)
                    getattr(f, name)(*plain[:i], w, *plain[i + 1:])


def test_pointer_values():
    f = N.entries()
    # (n_caches = 0 is refused behind the null pointers: -1 null, -2 a bad size)
    for p, status in ((None, -1), (C.c_void_p(None), -1), (C.POINTER(C.c_int32)(), -1), (64, -2), (C.c_void_p(64), -2),
                      (C.cast(64, C.POINTER(C.c_int32)), -2), (_Tensor(True), -2)):
        assert f.pikv_h2o_budget(p, 0, 0.1, 0.1, 64, 64, None) == f.of_checked.pikv_h2o_budget(p, 0, 0.1, 0.1, 64, 64, None) == status, p
        if not isinstance(p, _Tensor):
            assert N.lib().pikv_h2o_budget(p, 0, 0.1, 0.1, 64, 64, None) == status
    # host arrays of ctypes, as the ctypes signatures take them: the width 0 is found behind them
    for widths in ((C.c_int32 * 2)(32, 0), C.cast((C.c_int32 * 2)(32, 0), C.POINTER(C.c_int32)), np.array([32, 0], np.int32)):
        w = (C.c_void_p * 2)(64, 64)
        assert f.pikv_linear_group(64, 4, 128, 2, w, w, widths, [0, 1], 0, None, None, None, w, None, 0, None) == -2
    assert f.pikv_linear_group(64, 4, 128, 1, [64], [64], C.byref(C.c_int32(0)), [0], 0, None, None, None, [64], None, 0, None) == -2


def test_need():
    t = torch.zeros(3, 4)
    assert ops._need(None, "x", optional=True) is None
    for args, kw, text in (((None, "x"), {}, "x is required"), ((5, "x"), {}, "must be a torch.Tensor"),
                           ((t, "x"), {"ndim": 2}, "must live on the GPU")):
        with pytest.raises(ValueError, match=text):
            ops._need(*args, **kw)
    for kw, text in (({"dtype": torch.int32}, "dtype"), ({"ndim": 3}, "dimensions")):
        with pytest.raises(ValueError, match=text):
            ops._refuse(type("T", (torch.Tensor,), {"is_cuda": True})(t), "x", kw.get("dtype"), kw.get("ndim"))
    with pytest.raises(TypeError):
        ops._need(t, "x", shape=3)


def test_ordinary_tensor():
    cpu = torch.device("cpu")
    t = torch.zeros(8, 4)
    assert dense.ordinary_tensor(t, cpu) and dense.ordinary_tensor(torch.nn.Parameter(t), cpu)
    assert not dense.ordinary_tensor(t.t(), cpu) and not dense.ordinary_tensor(t.double(), cpu)
    assert not dense.ordinary_tensor(t, torch.device("meta")) and not dense.ordinary_tensor(None, cpu)
    assert not dense.ordinary_tensor(t.view(-1)[1:], cpu) and dense.ordinary_tensor(t.view(-1)[1:], cpu, align=4)
    assert not dense.ordinary_tensor(t.as_subclass(type("S", (torch.Tensor,), {})), cpu)
    seen = []
    torch.func.vmap(lambda x: seen.append(dense.ordinary_tensor(x, cpu)) or x)(torch.zeros(2, 3))
    assert seen == [False]


def _host_pool():
    """The host side of a pool with four planes of rows."""
    pool = object.__new__(ops.CachePool)
    pool.k_codes, pool.k_scale, pool.acc, pool.ts = torch.zeros(4, 64, dtype=torch.int8), torch.zeros(4, 2), torch.zeros(4), torch.zeros(4)
    pool.k_zero = pool.v_codes = pool.v_scale = pool.v_zero = None
    pool.row_base = pool.keep_index = pool.new_len = pool.fill = None
    pool.n_caches, pool._row_bytes = 1, [64, 8, 4, 4]
    return pool


@pytest.mark.parametrize("kind", [list, tuple, iter])
def test_every_plane_of_a_compaction_has_its_row_bytes(monkeypatch, kind):
    """The library reads as many widths as there are planes, whatever the extra ones come in."""
    pool = _host_pool()
    seen = []
    monkeypatch.setattr(ops, "_need", lambda t, name: t)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(N, "launch", lambda name, *args: seen.append(args))
    pool.compact(extra_planes=kind([torch.zeros(4, 3), torch.zeros(4, dtype=torch.int64)]))
    planes, widths, n = seen[0][:3]
    assert len(planes) == len(widths) == n == 6 and widths == [64, 8, 4, 4, 12, 8]


@pytest.mark.parametrize("kind", [list, tuple, torch.stack, torch.nn.ParameterList])
def test_experts_factors_come_in_any_sequence(monkeypatch, kind):
    """What holds the experts' tensors becomes a host array of their addresses, not itself an address."""
    seen = []
    monkeypatch.setattr(ops, "_need", lambda t, name, **kw: t)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(N, "launch", lambda name, *args: seen.append((name, args)))
    a, b, d = ([torch.ones(s) for _ in range(3)] for s in ((8, 2), (2, 8), (5, 8)))
    t = [torch.ones(5, 2) for _ in range(3)]
    ops.value_lora(torch.ones(3, 8), kind(a), kind(b), [1.0] * 3)
    ops.expert_combine(kind(d), kind(d), [1.0] * 3, torch.ones(3, 8), torch.ones(5, 3))
    ops.expert_combine(kind(d), kind(t), [1.0] * 3, torch.ones(3, 8), torch.ones(5, 3), lora_b=kind(b))
    assert [name for name, _ in seen] == ["pikv_value_lora", "pikv_expert_combine", "pikv_expert_combine_factors"]
    for (_, args), arrays in zip(seen, ((4, 5), (0, 1), (0, 1, 2))):
        for i in arrays:
            assert type(args[i]) in (list, tuple) and [type(x) in (torch.Tensor, torch.nn.Parameter) for x in args[i]] == [True] * 3


_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _python(code):
    subprocess.run([sys.executable, "-c", code], check=True, cwd=_ROOT)


def test_tensor_check_before_any_operator():
    """dense alone sets up what its check needs."""
    _python("import torch\nfrom pikv_amd import dense\n"
            "assert dense.ordinary_tensor(torch.zeros(8), torch.device('cpu')) is True\n"
            "assert dense.ordinary_tensor(torch.zeros(8)[1:], torch.device('cpu')) is False")


def test_without_the_extension_every_way_in_says_so():
    _python("import sys, torch\nsys.modules['pikv_amd._call'] = None\n"
            "from pikv_amd import _native as N, dense, ops\n"
            "for f in (lambda: dense.ordinary_tensor(torch.zeros(8), torch.device('cpu')), lambda: ops._need(torch.zeros(8), 'x'),\n"
            "          lambda: N.call('pikv_abi_version'), lambda: N.launch('pikv_abi_version'), lambda: N.size('pikv_evict_workspace_bytes', 1, 5)):\n"
            "    try:\n        f()\n"
            "    except N.PiKVNativeError as e:\n"
            "        assert 'python -m pikv_amd.build' in str(e) and isinstance(e.__cause__, ImportError), e\n"
            "    else:\n        raise AssertionError('no error')")


@pytest.mark.parametrize("body", ["int pikv_abi_version(void) { return 1004; }", "int nothing;"])
def test_a_library_of_another_version_is_refused(monkeypatch, tmp_path, body):
    (tmp_path / "other.c").write_text(body)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "other.so"), str(tmp_path / "other.c")], check=True)
    monkeypatch.setattr(N, "LIB_PATH", str(tmp_path / "other.so"))
    monkeypatch.setattr(N, "_entries", None)
    with pytest.raises(N.PiKVNativeError, match="ABI version (1004|0)"):
        N.entries()
    monkeypatch.undo()
    assert N.size("pikv_abi_version") == N.lib().pikv_abi_version() >= 1005     # ... and the one in use stays


@pytest.mark.parametrize("again", [copy.copy, copy.deepcopy, lambda p: pickle.loads(pickle.dumps(p))])
def test_a_pool_of_another_version_makes_its_workspaces_anew(again):
    """One that another version of the package has pickled has that version's workspace sizes, and no row widths."""
    pool = _host_pool()
    del pool._row_bytes
    pool._decode_ws, pool._decode_ws_key, pool._evict_ws = torch.zeros(8), (32, 700), (torch.zeros(8), 32)
    new = again(pool)
    assert new._row_bytes == [64, 8, 4, 4] and torch.equal(new.k_codes, pool.k_codes) and new.n_caches == 1
    assert not {"_decode_ws", "_decode_ws_key", "_evict_ws"} & set(new.__dict__) and pool._decode_ws_key == (32, 700)
