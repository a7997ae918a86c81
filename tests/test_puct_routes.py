"""A PUCT launch on torch tensors goes through _puct_call where that is built and fits, else through Python: the same calls
are accepted with the same arguments, and the same refused with the same words; and the package builds without _puct_call."""
import collections
import ctypes

import numpy as np
import pytest

import puct_routes as pr
from mcts_numba_cuda_amd import build, puct

TREES, NODES, EDGES, WARPS, DEPTH = 2, 5, 4, 3, 7
SHAPES = dict(edge_child=(TREES, NODES, EDGES), edge_prior=(TREES, NODES, EDGES), edge_w=(TREES, NODES, EDGES), edge_n=(TREES, NODES, EDGES),
              edge_inflight=(TREES, NODES, EDGES), node_inflight=(TREES, NODES), node_expand_inflight=(TREES, NODES), node_expanded=(TREES, NODES),
              node_count=(TREES,), out_selected=(TREES, WARPS), out_path=(TREES, WARPS, DEPTH), out_len=(TREES, WARPS))
FLOATS = ("edge_prior", "edge_w", "values")
LAUNCHERS = {
    "select": lambda d, v: puct.launch_select(d, cpuct=1.25, c_pw=2, alpha_pw=np.float32(0.5), soft_winner=True),
    "node_preclaim": lambda d, v: puct.launch_node_select(d, cpuct=0.75, c_pw=0.0),
    "node_winner_recalc": lambda d, v: puct.launch_node_select(d, variant="winner_recalc"),
    "edge_backup": lambda d, v: puct.launch_edge_backup(d, v, virtual_loss=2),
    "edge_release": lambda d, v: puct.launch_edge_backup(d),
    "node_backup": lambda d, v: puct.launch_node_backup(d, v),
}


class Subclass(pr.Tensor):
    pass


def tensor(name, shape=None, dtype=None, cls=pr.Tensor, **kw):
    shape = SHAPES.get(name, (TREES, WARPS, DEPTH)) if shape is None else shape
    return cls(shape, dtype or (pr.FLOAT32 if name in FLOATS else pr.INT32), 0x100000000 + 0x1000 * (1 + sorted(SHAPES).index(name) if name in SHAPES else 0), **kw)


def arrays():
    return {name: tensor(name) for name in SHAPES}, tensor("values")


def spoilt():
    """(what, dictionary, values): one thing at a time that differs from the usual case."""
    yield "usual", *arrays()
    for name in list(SHAPES) + ["values"]:
        shape = SHAPES.get(name, (TREES, WARPS, DEPTH))
        changes = dict(longer=tensor(name, shape[:-1] + (shape[-1] + 1,)), trees=tensor(name, (TREES + 1,) + shape[1:]), flat=tensor(name, (int(np.prod(shape)),)),
                       deeper=tensor(name, shape + (1,)), type=tensor(name, dtype=pr.INT32 if name in FLOATS else pr.FLOAT32), host=tensor(name, is_cuda=False),
                       strided=tensor(name, contiguous=False), subclass=tensor(name, cls=Subclass), numpy=np.zeros(shape, np.int32), none=None)
        for what, t in changes.items():
            d, v = arrays()
            if name == "values":
                v = t
            else:
                d[name] = t
            yield f"{name} {what}", d, v
        if name != "values":
            d, v = arrays()
            del d[name]
            yield f"{name} missing", d, v
    d, v = arrays()
    yield "another mapping", collections.UserDict(d), v
    d, v = arrays()
    for name in ("out_selected", "out_path", "out_len"):
        d[name] = tensor(name, SHAPES[name][:1] + (0,) + SHAPES[name][2:])
    yield "no traversals", d, tensor("values", (TREES, 0, DEPTH))


@pytest.fixture
def library(monkeypatch):
    """Launchers that note what they are called with and return `code`."""
    calls, code = [], [0]
    vp, ci, cf = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    kinds = dict(puct_select_winner_recalc_launch=[cf] * 3 + [ci] + [vp] * 11 + [ci] * 5 + [vp], puct_edge_backup_launch=[ci] + [vp] * 9 + [ci] * 5 + [vp],
                 puct_node_select_preclaim_launch=[cf] * 3 + [vp] * 11 + [ci] * 5 + [vp], puct_node_select_winner_recalc_launch=[cf] * 3 + [vp] * 11 + [ci] * 5 + [vp],
                 puct_node_backup_launch=[ci] + [vp] * 10 + [ci] * 5 + [vp])

    def noting(name):
        def launcher(*args):
            calls.append((name, args))
            return code[0]
        return launcher

    class Library:
        pass
    lib = Library()
    for name, types in kinds.items():
        fn = ctypes.CFUNCTYPE(ci, *types)(noting(name))
        setattr(lib, name, fn)
    lib.puct_cpp_cuda_error_string = lambda c: b"error %d" % c
    monkeypatch.setattr(puct, "_LIB", lib)
    monkeypatch.setattr(puct, "_ENTRIES", {})
    lib.calls, lib.code = calls, code
    return lib


def outcome(library, launcher, d, v):
    del library.calls[:]
    try:
        LAUNCHERS[launcher](d, v)
    except Exception as e:
        return type(e), str(e), list(library.calls)
    return None, "", list(library.calls)


@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("launcher", LAUNCHERS)
def test_both_routes_take_and_refuse_the_same(library, monkeypatch, launcher, table):
    """table: the tensors are described by an exchange table, as torch's are, else by their attributes."""
    if table and not build.dlpack_flags():
        pytest.skip("_puct_call is built without torch's exchange table here")
    accepted = refused = asked = 0
    for code in (0, 700):
        library.code[0] = code
        for what, d, v in spoilt():
            described = [] if table else None
            with pr.routes(described=described) as call:
                if call is None:
                    pytest.skip("_puct_call is not built")
                by_c = outcome(library, launcher, d, v)
                puct._puct_call = None
                by_python = outcome(library, launcher, d, v)
            asked += len(described or ())
            assert by_c == by_python, what
            assert (by_c[0] is None) == (len(by_c[2]) == 1 and code == 0), what
            accepted, refused = accepted + len(by_c[2]), refused + (not by_c[2])
    assert accepted > 2 and refused > 2 and (not table or asked > 100)


@pytest.mark.parametrize("launcher", LAUNCHERS)
def test_the_usual_case_goes_through_c(library, monkeypatch, launcher):
    def python_route(*args):
        raise AssertionError("looked over in Python")
    with pr.routes() as call:
        if call is None:
            pytest.skip("_puct_call is not built")
        monkeypatch.setattr(puct, "_arguments", python_route)
        d, v = arrays()
        assert outcome(library, launcher, d, v)[0] is None
        assert library.calls[0][1][-1] == pr.STREAM and library.calls[0][1][-6:-1] == (TREES, NODES, EDGES, WARPS, DEPTH)
        assert outcome(library, launcher, collections.UserDict(d), v)[:2] == (AssertionError, "looked over in Python")


@pytest.mark.parametrize("route", ["c", "python"])
def test_what_is_refused_says_why(library, route):
    cases = [("edge_w longer", "edge_w must have shape [trees, nodes, edges]"), ("out_len trees", "out_selected / out_len must have shape [trees, warps]"),
             ("node_count longer", "node_count must have shape [trees]"), ("edge_w type", "edge_w: expected a contiguous torch.float32 tensor on the GPU"),
             ("edge_n host", "edge_n: expected a contiguous torch.int32 tensor on the GPU"), ("edge_inflight strided", "edge_inflight: expected a contiguous torch.int32 tensor on the GPU"),
             ("values longer", "path_edge_values must have shape [trees, warps, path_depth]"), ("node_inflight longer", "node_inflight must have shape [trees, nodes]")]
    every = {what: (d, v) for what, d, v in spoilt()}
    for what, text in cases:
        with pr.routes() as call:
            if route == "c" and call is None:
                pytest.skip("_puct_call is not built")
            if route == "python":
                puct._puct_call = None
            assert outcome(library, "edge_backup", *every[what]) == (ValueError, text, []), what


def test_package_builds_without_its_host_module(monkeypatch, tmp_path, capsys):
    """No C compiler, or no Python.h: the libraries are what matters, and a module of an earlier build does not stay."""
    monkeypatch.setattr(build, "LIBRARIES", {})
    no_headers = dict(build.sysconfig.get_paths(), include=str(tmp_path))
    for n, set_up in enumerate((lambda m: m.setenv("CC", "no-such-compiler"), lambda m: m.setattr(build.sysconfig, "get_paths", lambda: no_headers))):
        module = tmp_path / f"_puct_call{n}.so"
        module.write_bytes(b"old")
        with monkeypatch.context() as m:
            m.setattr(build, "HOST_MODULE", str(module))
            set_up(m)
            assert build.build() == build.LIB
            assert not module.exists() and "is not built" in capsys.readouterr().err
            with pytest.raises(RuntimeError, match="cannot be built"):
                build.build(only=str(module))


@pytest.mark.gpu
@pytest.mark.parametrize("route", ["c", "python"])
def test_both_routes_launch_on_the_gpu(route):
    """One traversal per tree, selection and backup in turn: every array equals the sequential oracle's."""
    import copy

    import puct_cases as pc
    from mcts_numba_cuda_amd.hipmem import DeviceArray, synchronize
    from oracle import puct_oracle as po
    rng = np.random.default_rng(11)
    for level in ("edge", "node"):
        h = pc.random_forest(rng, trees=16, nodes=120, actions=9, warps=1, path_depth=12)
        if level == "node":
            del h["edge_inflight"]
            h["node_inflight"] = np.zeros((16, 120), np.int32)
        held = {k: DeviceArray(v) for k, v in h.items()}
        d = {k: pr.Tensor(a.shape, pr.torch_type(a.dtype), a.data_ptr()) for k, a in held.items()}
        want = copy.deepcopy(h)
        for rnd in range(3):
            values = rng.uniform(-1, 1, h["out_path"].shape).astype(np.float32)
            on_gpu = DeviceArray(values)
            v = pr.Tensor(values.shape, pr.FLOAT32, on_gpu.data_ptr())
            with pr.routes(stream=0) as call:
                if route == "c":
                    assert call is not None, "_puct_call is not built"
                else:
                    puct._puct_call = None
                if level == "edge":
                    puct.launch_select(d, cpuct=1.5, c_pw=1.0)
                    puct.launch_edge_backup(d, v)
                else:
                    puct.launch_node_select(d, cpuct=1.5, c_pw=1.0, variant="winner_recalc")
                    puct.launch_node_backup(d, v)
            synchronize()
            if level == "edge":
                po.select(want, cpuct=1.5, c_pw=1.0)
                po.backup(want, values)
            else:
                po.node_select(want, cpuct=1.5, c_pw=1.0, variant="winner_recalc")
                po.backup(want, values, node_level=True)
            for k in want:
                assert np.array_equal(held[k].numpy(), want[k], equal_nan=True), (level, rnd, k)
