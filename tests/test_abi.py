"""CPU-side checks of the drop-in boundary: both libraries load, every symbol declared in
include/ is exported, the ctypes signature table covers every declared DIOPI function, and
the shim's tensor struct matches the header layout. No compute is launched."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INC = os.path.join(ROOT, "include")


def _declared(path, macro):
    text = open(path).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(macro + r"\s+[\w\s\*]+?\b(\w+)\s*\(", text)


def test_impl_exports_every_declared_function(pkg):
    lib = pkg._native.impl()
    names = _declared(os.path.join(INC, "diopi", "functions.h"), "DIOPI_API") + \
        _declared(os.path.join(INC, "diopi", "functions_ext.h"), "DIOPI_API")
    assert len(names) >= 40
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing
    unbound = [n for n in names if n != "diopiGetLastErrorString" and n not in pkg.diopi.SIGNATURES]
    assert not unbound, unbound


def test_runtime_exports_callbacks_and_facade(pkg):
    rt = pkg._native.runtime()
    cb = _declared(os.path.join(INC, "diopi", "diopirt.h"), "DIOPI_RT_API")
    assert "diopiRequireTensor" in cb and "diopiGetStream" in cb
    fac = _declared(os.path.join(INC, "dipu_amd", "runtime.h"), "DIPU_AMD_API")
    assert len(fac) >= 60
    missing = [n for n in cb + fac if not hasattr(rt, n)]
    assert not missing, missing


def test_impl_library_has_no_torch_dependency(pkg):
    # the boundary is plain C: the impl library must not link libtorch / libc10
    import subprocess
    out = subprocess.run(["ldd", pkg._native.IMPL_PATH], capture_output=True, text=True).stdout
    assert "libtorch" not in out and "libc10" not in out


def test_tensor_struct_layout_matches_header(pkg):
    d = pkg.diopi.dipuAmdTensor
    assert d.data.offset == 0 and d.ndim.offset == 8
    assert d.shape.offset == 16 and d.stride.offset == 16 + 64
    assert d.dtype.offset == 144 and d.device.offset == 148 and d.device_index.offset == 152
    assert d.storage_offset.offset == 160 and d.storage_ptr.offset == 168 and d.storage_nbytes.offset == 176
    assert ctypes.sizeof(d) == 184
    s = pkg.diopi.diopiScalar_t
    assert ctypes.sizeof(s) == 16 and s.u.offset == 8


def test_scalar_marshalling(pkg):
    # diopi_helper.cpp:74-97: bool/int -> int64 payload, float -> float64 payload
    s = pkg.diopi.scalar(3)
    assert (s.stype, s.ival) == (6, 3)
    s = pkg.diopi.scalar(True)
    assert (s.stype, s.ival) == (6, 1)
    s = pkg.diopi.scalar(0.5)
    assert (s.stype, s.fval) == (10, 0.5)
    with pytest.raises(TypeError):
        pkg.diopi.scalar("x")


def test_missing_library_fails_loudly(pkg, monkeypatch):
    monkeypatch.setattr(pkg._native, "_impl", None)
    monkeypatch.setattr(pkg._native, "IMPL_PATH", "/nonexistent/libdiopi_impl.so")
    with pytest.raises(pkg._native.NativeLibraryMissing):
        pkg._native.impl()


def test_version_and_error_string(pkg):
    rt = pkg._native.runtime()
    rt.diopiGetVersion.restype = ctypes.c_char_p
    assert rt.diopiGetVersion().startswith(b"DIOPI Version: ")
    assert isinstance(pkg.diopi.last_error(), str)


def test_profiler_hooks_count_ranges_only_while_enabled(pkg):
    """devapis::enableProfiler / disableProfiler and the diopiRecordStart/End pair
    (dipu/torch_dipu/csrc_dipu/runtime/device/profilerapis.h:12-14, diopirt/diopirt_impl.cpp:224-237):
    disabled -> null record, nothing counted; enabled -> one range started and ended per pair."""
    rt = pkg.runtime
    rt.disableProfiler()
    s0, e0, _ = rt.profilerCounts()
    rec = rt.recordStart("idle")
    assert not rec.value
    rt.recordEnd(rec)
    assert rt.profilerCounts()[:2] == (s0, e0)
    rt.enableProfiler("/tmp/unused")
    try:
        recs = [rt.recordStart(f"diopiOp{i}") for i in range(3)]
        assert all(r.value for r in recs)
        s1, e1, _ = rt.profilerCounts()
        assert (s1 - s0, e1 - e0) == (3, 0)
        for r in reversed(recs):
            rt.recordEnd(r)
            assert not r.value
        s2, e2, _ = rt.profilerCounts()
        assert (s2 - s0, e2 - e0) == (3, 3)
    finally:
        rt.disableProfiler()


def test_generator_state_round_trip(pkg):
    """The diopiGenerator* runtime callbacks with the CUDA vendor's state layout
    (dipu/torch_dipu/csrc_dipu/vendor/cuda/CudaGeneratorImpl.cpp:17-76; callbacks diopirt_impl.cpp:175-226): 16 host
    bytes = seed then Philox offset, an 8-byte state sets offset 0, offsets must be multiples of 4."""
    import struct
    import torch
    d = pkg.diopi
    g = d.Generator()
    try:
        assert g.seed_and_offset() == (67280421310721, 0)          # torch's default seed
        g.set_seed_and_offset(1234, 8)
        assert g.seed_and_offset() == (1234, 8)
        st = g.get_state()
        assert st.dtype == torch.uint8 and st.numel() == 16
        assert struct.unpack("<QQ", bytes(st.tolist())) == (1234, 8)
        h = d.Generator()
        h.set_state(st)
        assert h.seed_and_offset() == (1234, 8)
        h.set_state(torch.tensor(list(struct.pack("<Q", 99)), dtype=torch.uint8))   # seed only
        assert h.seed_and_offset() == (99, 0)
        with pytest.raises(d.DiopiError):
            g.set_seed_and_offset(1, 6)                               # offset not a multiple of 4
        with pytest.raises(d.DiopiError):
            h.set_state(torch.zeros(12, dtype=torch.uint8))           # wrong size
        h.close()
    finally:
        g.close()


def test_allocator_metrics_labels_events_and_histogram(pkg):
    """Label sets and event rules of dipu/torch_dipu/csrc_dipu/runtime/core/allocator/allocator_metrics.h:17-120, fed
    through the same call the allocators make (no device needed)."""
    rt = pkg.runtime
    assert rt.metricsEnable() is True                       # on by default (metrics/metrics.cpp:5-11)
    t, dev = "unit_test", 3
    key = lambda name, **kw: (name, frozenset({("type", t), ("device", str(dev))} | set(kw.items())))
    rt.metricsRecord(t, dev, 0x1000, 16)                    # <= 2^4: first bucket
    rt.metricsRecord(t, dev, 0x2000, 17)                    # second bucket
    rt.metricsRecord(t, dev, 0x3000, 1 << 31)               # last finite bucket
    rt.metricsRecord(t, dev, 0x4000, (1 << 31) + 1)         # +Inf
    rt.metricsRecord(t, dev, 0x5000, 0)                     # size 0: ignored
    rt.metricsRecord(t, dev, 0, 64)                         # null pointer
    rt.metricsRecord(t, dev, 0x1000, 32)                    # already live
    m = rt.metrics()
    assert m[key("allocator_event_count", method="allocate", event="nullptr")] == 1
    assert m[key("allocator_event_count", method="allocate", event="duplicated")] == 1
    assert m[key("allocator_size_bucket", method="allocate", le="16")] == 1
    assert m[key("allocator_size_bucket", method="allocate", le="32")] == 2
    assert m[key("allocator_size_bucket", method="allocate", le=str(1 << 30))] == 2
    assert m[key("allocator_size_bucket", method="allocate", le=str(1 << 31))] == 3
    assert m[key("allocator_size_bucket", method="allocate", le="+Inf")] == 4
    assert m[key("allocator_size_count", method="allocate")] == 4
    assert m[key("allocator_size_sum", method="allocate")] == 16 + 17 + (1 << 31) + (1 << 31) + 1
    rt.metricsRecord(t, dev, 0x2000, deallocate=True)       # records the size it was allocated with
    rt.metricsRecord(t, dev, 0x2000, deallocate=True)       # no longer live
    rt.metricsRecord(t, dev, 0, deallocate=True)
    m = rt.metrics()
    assert m[key("allocator_size_sum", method="deallocate")] == 17 and m[key("allocator_size_count", method="deallocate")] == 1
    assert m[key("allocator_event_count", method="deallocate", event="unexpected")] == 1
    assert m[key("allocator_event_count", method="deallocate", event="nullptr")] == 1
    # switched off nothing is recorded
    assert rt.metricsEnable(False) is False
    rt.metricsRecord(t, dev, 0x9000, 64)
    assert rt.metrics()[key("allocator_size_count", method="allocate")] == 4
    assert rt.metricsEnable(True) is True


def test_generated_gemm_loop_is_current(tmp_path):
    """The committed K loop of the 4-wave GEMM kernel is what its generator writes."""
    import subprocess
    import sys
    d = os.path.join(ROOT, "deeplink.framework_amd", "csrc", "diopi_impl")
    out = tmp_path / "loop.inc"
    subprocess.run([sys.executable, os.path.join(d, "gen_gemm_loop_4wave.py"), str(out)], check=True)
    assert out.read_text() == open(os.path.join(d, "gemm_loop_4wave.inc")).read()


def test_host_module_covers_the_signature_table_and_infers_like_torch(pkg):
    """The native half of the op adapter: a callable for every entry point the ctypes view knows, marshalling errors of the
    same class as that view's, and output inference equal to torch's own."""
    import torch
    h = pkg._native.host()
    assert all(hasattr(h, n) for n in pkg.diopi.SIGNATURES)
    for a, b in [((3, 1), (4,)), ((), (2, 3)), ((2, 0), (1, 1)), ((5,), (5,))]:
        for da in (torch.bfloat16, torch.float32, torch.int64, torch.bool):
            for db in (torch.float16, torch.float32, torch.uint8):
                x, y = torch.zeros(a, dtype=da), torch.zeros(b, dtype=db)
                o = h.broadcast_of(x, y, False)
                assert o.shape == torch.broadcast_shapes(a, b) and o.dtype == torch.result_type(x, y) and o.is_contiguous()
                assert h.broadcast_of(x, y, True).dtype == torch.bool
    for da in (torch.bfloat16, torch.int32, torch.bool):
        for v in (True, 2, 2.5):
            assert h.broadcast_of(torch.zeros(3, dtype=da), v, False).dtype == torch.result_type(torch.zeros(3, dtype=da), v)
    t = torch.zeros(2, 3, 4).transpose(0, 2)
    assert h.like(t).shape == t.shape and h.like(t).is_contiguous() and h.rows_of(t, 7).shape == (4, 3, 7)
    with pytest.raises(pkg.diopi.DiopiError, match="rank 9"):
        h.diopiSilu(1, torch.zeros([1] * 9), None)
    with pytest.raises(pkg.diopi.DiopiError, match="complex64"):
        h.diopiSilu(1, torch.zeros(1, dtype=torch.complex64), None)
    with pytest.raises(TypeError):
        h.diopiSilu(1, torch.zeros(1))
    with pytest.raises(RuntimeError, match="must match"):
        h.broadcast_of(torch.zeros(3), torch.zeros(4), False)


def test_ops_refuse_a_scope_that_was_closed(pkg):
    """An op inside `with scope:` after close(), of this scope or of the one around it, is an error and runs in no freed
    context; a scope nobody else holds lives as long as ops run in it."""
    import gc
    import torch
    ops, x = pkg.ops, torch.zeros(4)
    refused = lambda: pytest.raises(pkg.diopi.DiopiError, match="null diopiContext")
    outer, inner = ops.WorkspaceScope(stream=0), ops.WorkspaceScope(stream=0)
    with outer:
        with inner:
            outer.close()
            with pytest.raises(pkg.diopi.DiopiError, match="lives on the host"):     # the open scope's context got this far
                ops.silu(x)
            inner.close()
            with refused():
                ops.silu(x)
        with refused():
            ops.silu(x)
        with inner, refused():                                                        # entered after its close()
            ops.silu(x)
    ops.WorkspaceScope(stream=0).__enter__()
    gc.collect()
    with pytest.raises(pkg.diopi.DiopiError, match="lives on the host"):
        ops.silu(x)
    ops._ctx.close()
    with refused():
        ops.silu(x)
    ops._ctx = 0


def test_tensors_of_a_list_argument_live_for_the_call(pkg):
    """A sequence that makes its tensors as it is read: they are alive while the entry point runs (here: while its failure,
    a closed context, is reported)."""
    import weakref
    import torch
    h, made, alive = pkg._native.host(), [], []

    class Made:
        def __len__(self):
            return 2

        def __getitem__(self, i):
            if i > 1:
                raise IndexError
            t = torch.zeros(3)
            made.append(weakref.ref(t))
            return t

    def failure(name, ret):
        alive.extend(r() is not None for r in made)
        pkg.diopi.raise_failure(name, ret)

    ctx = pkg.diopi.Context(0)
    ctx.close()
    h.setup(pkg.diopi.DiopiError, failure)
    try:
        with pytest.raises(pkg.diopi.DiopiError, match="null diopiContext"):
            h.diopiCat(ctx, torch.zeros(6), Made(), 2, 0)
    finally:
        h.setup(pkg.diopi.DiopiError, pkg.diopi.raise_failure)
    assert alive == [True, True]


def test_integers_of_more_than_63_bits_marshal_as_the_ctypes_view_does(pkg):
    """A number that an int64 field reduces modulo 2^64 is taken (the call gets as far as the host tensor); output
    inference refuses what torch's promotion does."""
    import torch
    ops, d, x = pkg.ops, pkg.diopi, torch.zeros(3, dtype=torch.int64)
    assert d.scalar(2 ** 64 - 1).ival == -1
    with ops.WorkspaceScope(stream=0):
        for call in (lambda: ops.fill_(x, 2 ** 64 - 1), lambda: ops.masked_fill_(x, x == 0, 2 ** 70), lambda: ops.eq(x, 2 ** 64 - 1),
                     lambda: ops.add(x, 2 ** 63), lambda: ops.tril(x.view(1, 3), 2 ** 63)):
            with pytest.raises(d.DiopiError, match="lives on the host"):
                call()
        for v in (2 ** 64, -2 ** 63 - 1):
            with pytest.raises(OverflowError):
                torch.result_type(x, v)
            with pytest.raises(OverflowError):
                ops.add(x, v)


def test_native_descriptors_equal_the_ctypes_view_field_by_field(pkg, tmp_path):
    """What an entry point receives for a tensor: a stand-in for one, loaded before the library, keeps its descriptor."""
    import subprocess
    import sys
    (tmp_path / "probe.cpp").write_text('''
#include <dipu_amd/runtime.h>
extern "C" { dipuAmdTensor kept; int diopiSiluInp(void*, dipuAmdTensor* t) { kept = *t; return 0; } }
''')
    subprocess.run(["g++", "-shared", "-fPIC", f"-I{INC}", str(tmp_path / "probe.cpp"), "-o", str(tmp_path / "probe.so")], check=True)
    code = '''
import ctypes, sys
import torch
sys.path.insert(0, sys.argv[1])
from __graft_entry__ import load_package
pkg = load_package()
probe = ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
h, d = pkg._native.host(), pkg.diopi
kept = d.dipuAmdTensor.in_dll(probe, "kept")
base = torch.arange(48, dtype=torch.float32).view(2, 4, 6)
for t in [base, base[1:, 2], base[:, :, 3:3], base[2:], base.transpose(0, 2), torch.empty(0), torch.empty(3, 0, 2, dtype=torch.int64),
          torch.tensor(5, dtype=torch.uint8), base[1, 1, 1], base.to(torch.bfloat16)[1:], base[:, :1].expand(2, 4, 6)]:
    h.diopiSiluInp(1, t)
    want = d.Handle(t).desc
    for name, _ in d.dipuAmdTensor._fields_:
        a, b = getattr(kept, name), getattr(want, name)
        if hasattr(a, "__len__"):
            a, b = list(a)[:t.dim()], list(b)[:t.dim()]
        assert name == "reserved" or a == b, (tuple(t.shape), name, a, b)
'''
    r = subprocess.run([sys.executable, "-c", code, ROOT, str(tmp_path / "probe.so")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
