"""Host-side rules of cvcuda_amd.pyapi that need no GPU: the enumerations (names that share a value resolve to the
first name of the reference's headers, as its table of output formats does, python/mod_cvcuda/CvtColorUtil.cpp:30-42),
the output shapes and formats of cvtcolor (CvtColorUtil.cpp:244-330) and the argument checks the reference's bindings
make themselves."""
import ctypes as C
import importlib
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest


@pytest.fixture(scope="module")
def api(cv):
    return importlib.import_module("cvcuda_amd.pyapi")


@pytest.fixture(autouse=True)
def no_default_stream_is_followed(api, monkeypatch):
    monkeypatch.setattr(api, "_followed", {})


def test_enumerations(api, K):
    assert api.Interp.LINEAR == K.INTERP_LINEAR and api.Interp.WARP_INVERSE_MAP == K.WARP_INVERSE_MAP == 16
    assert api.Border.REFLECT101 == K.BORDER_REFLECT101 and api.ChannelManip.REVERSE == K.CHANNEL_REVERSE
    assert api.NormalizeFlags.SCALE_IS_STDDEV == 1
    assert api.Format.RGB8 == K.IMAGE_FORMAT_RGB8 and api.Type.F32 == K.DATA_TYPE_F32
    cc = api.ColorConversion
    assert cc.BGR2RGB == K.COLOR_BGR2RGB and cc.YUV2RGB_NV12 == K.COLOR_YUV2RGB_NV12
    assert all("SPEC" not in n and "XFER" not in n for n in cc.__members__)
    # one value, two names: the header's first name is the canonical one
    assert cc.RGB2RGBA is cc.BGR2BGRA and cc(0).name == "BGR2BGRA"
    assert cc.BGRA2RGB is cc.RGBA2BGR and cc(3).name == "RGBA2BGR"


@pytest.mark.parametrize("code,shape,want", [
    ("BGR2GRAY", (2, 8, 6, 3), (2, 8, 6, 1)), ("GRAY2BGR", (8, 6, 1), (8, 6, 3)), ("RGB2RGBA", (8, 6, 3), (8, 6, 4)),
    ("BGRA2RGB", (2, 8, 6, 4), (2, 8, 6, 3)), ("BGR2HSV", (4, 4, 3), (4, 4, 3)), ("BGR2YUV", (8, 6, 3), (8, 6, 3)),
    ("YUV2RGB_NV12", (2, 12, 6, 1), (2, 8, 6, 3)), ("YUV2BGRA_NV21", (60, 62, 1), (40, 62, 4)),
    ("BGR2YUV_NV21", (2, 40, 62, 3), (2, 60, 62, 1)), ("RGB2YUV_NV12", (8, 6, 3), (12, 6, 1)),
    ("YUV2BGR_YUY2", (4, 12, 1), (4, 6, 3)), ("YUV2BGR_YUY2", (4, 6, 2), (4, 6, 3)), ("YUV2GRAY_UYVY", (4, 12, 1), (4, 6, 1)),
])
def test_cvtcolor_output_shapes(api, code, shape, want):
    assert api._cvtcolor_shape(shape, api.ColorConversion[code]) == want


def test_cvtcolor_shape_and_format_errors(api):
    with pytest.raises(RuntimeError):
        api._cvtcolor_shape((8, 6), api.ColorConversion.BGR2RGB)
    F, cc = api.Format, api.ColorConversion
    assert api._cvtcolor_format(F.RGB8, cc.RGB2GRAY) == F.Y8_ER and api._cvtcolor_format(F.Y8, cc.GRAY2BGR) == F.BGR8
    assert api._cvtcolor_format(F.HSV8, cc.HSV2RGB) == F.RGB8 and api._cvtcolor_format(F.BGRA8, cc.BGRA2RGB) == F.BGR8
    assert api._cvtcolor_format(F.RGB8, cc.RGB2YUV_NV12) == F.Y8 and api._cvtcolor_format(F.BGRf32, cc.RGB2BGR) == F.RGBf32  # = BGR2RGB


def test_small_helpers(api):
    r = api.RectI(x=1, y=2, width=3, height=4)
    assert tuple(r) == (1, 2, 3, 4) and tuple(api.RectI(5, 6, 7, 8)) == (5, 6, 7, 8)
    assert api._border_value([]) == (0.0, 0.0, 0.0, 0.0) and api._border_value(3) == (3.0, 0.0, 0.0, 0.0)
    assert api._border_value([1, 2, 3, 4]) == (1.0, 2.0, 3.0, 4.0)
    with pytest.raises(RuntimeError):
        api._border_value([1, 2, 3, 4, 5])
    assert api._matrix([[1, 0, 2], [0, 1, 3]], 2) == [1.0, 0.0, 2.0, 0.0, 1.0, 3.0]
    with pytest.raises(RuntimeError):
        api._matrix([[1, 0, 2]], 2)
    assert api._image_axes("NHWC") == (2, 1) and api._image_axes("CHW") == (2, 1) and api._image_axes("NWC") == (1, None)
    with pytest.raises(ValueError):
        api._image_axes("NC")
    assert api._np_dtype(api.Type.F32) == np.float32 and api._np_dtype(np.uint8) == np.uint8


# ---- tests/nvcv_types/python/test_imgformat.py:20-45, test_datatype.py:21-54, test_rect.py:19-40 ------------------------
@pytest.mark.parametrize("format,gold_channels,gold_planes", [
    ("RGBA8", 4, 1), ("RGB8", 3, 1), ("_2S16", 2, 1), ("S8", 1, 1), ("NV12", 3, 2),
])
def test_imgformat_numchannels_and_planes(api, format, gold_channels, gold_planes):
    assert getattr(api.Format, format).channels == gold_channels and getattr(api.Format, format).planes == gold_planes


@pytest.mark.parametrize("type,dt", [
    ("U8", np.uint8), ("U8", np.dtype(np.uint8)), ("S8", np.int8), ("U16", np.uint16), ("S16", np.int16), ("U32", np.uint32),
    ("S32", np.int32), ("U64", np.uint64), ("S64", np.int64), ("F32", np.float32), ("F64", np.float64), ("C64", np.complex64),
    ("_2C64", np.dtype("2F")), ("C128", np.complex128), ("_2C128", np.dtype("2D")), ("_3S8", np.dtype("3i1")),
    ("_4S32", np.dtype("4i")),
])
def test_datatype_dtype(api, type, dt):
    type = getattr(api.Type, type)
    assert type == dt
    made = api.Type(dt)
    assert made == type and made == dt and made is type


@pytest.mark.parametrize("dt", [np.dtype([("f1", np.uint64), ("f2", np.int32)]), "invalid"])
def test_datatype_dtype_conv_error(api, dt):
    with pytest.raises(TypeError):
        api.Type(dt)


def test_recti(api):
    r = api.RectI()
    assert (r.x, r.y, r.width, r.height) == (0, 0, 0, 0)
    for x, y, w, h in ((0, 0, 0, 0), (10, -12, -45, 14)):
        for r in (api.RectI(x, y, w, h), api.RectI(y=y, width=w, height=h, x=x)):
            assert (r.x, r.y, r.width, r.height) == (x, y, w, h)


def test_reshape_of_wrapped_memory_keeps_its_owner_alive(api):
    # nvcvTensorReshape takes a reference on the source handle, but the owner of externally wrapped memory is held by the
    # Python wrapper of the source only: the reshaped tensor must hold it too (no GPU: the pointer is never followed)
    import gc
    import weakref

    class Owner:
        def __init__(self):
            self.__cuda_array_interface__ = {"shape": (8, 3, 3), "typestr": "|u1", "data": (0x7F0000001000, False),
                                             "version": 3, "strides": None}

    owner = Owner()
    alive = weakref.ref(owner)
    source = api.as_tensor(owner, "HWC")
    for view in (source.reshape((24, 3), "WC"), api.reshape(source, (72,), "W")):
        del source, owner
        gc.collect()
        assert alive() is not None, "the owner of the wrapped memory was collected while a reshaped tensor refers to it"
        assert view.cuda().__cuda_array_interface__["data"][0] == 0x7F0000001000
        owner = alive()
        source = api.as_tensor(owner, "HWC")
        del view
    del source, owner
    gc.collect()
    assert alive() is None


def test_submit_bookkeeping_under_parallel_readers(api, monkeypatch):
    # several threads record reads of one shared input on their own streams while another thread keeps writing it:
    # no read event may be lost (a later writer waits for every stream that read) and no iteration may trip over a
    # concurrent update. No GPU: streams and events are stand-ins that only record what was asked of them.
    import threading

    class FakeStream:
        def __init__(self, key):
            self.cuda_stream, self.waited = key, []

        def wait_event(self, event):
            self.waited.append(event)

    class FakeEvent:
        def record(self, stream):
            self.stream = stream.cuda_stream

    class Box:
        pass

    monkeypatch.setattr(api, "_torch_stream", lambda s: s)
    monkeypatch.setattr(api, "_new_event", FakeEvent)
    shared, errors = Box(), []

    def reader(key):
        try:
            out = Box()
            for _ in range(300):
                api._submit(FakeStream(key), [shared], [out], lambda s: None)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=reader, args=(100 + i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert sorted(shared._read) == [100 + i for i in range(8)]
    writer = FakeStream(7)
    api._submit(writer, [], [shared], lambda s: None)
    assert sorted(e.stream for e in writer.waited) == [100 + i for i in range(8)]
    assert shared._read == {} and shared._wrote[0] == 7


def test_submit_orders_the_default_stream_by_events_recorded_when_needed(api, monkeypatch):
    # the default stream's work leaves no event behind it; another stream that reads or overwrites its results waits
    # for one recorded on the default stream then, and the default stream waits for the other stream's own events.
    # No GPU: streams and events are stand-ins that only record what was asked of them.
    class FakeStream:
        def __init__(self, key):
            self.cuda_stream, self.waited = key, []

        def wait_event(self, event):
            self.waited.append(event.stream)

    made = []

    class FakeEvent:
        def __init__(self):
            made.append(self)

        def record(self, stream):
            self.stream = stream.cuda_stream

    class Box:
        pass

    default, side, other = FakeStream(0), FakeStream(7), FakeStream(9)
    monkeypatch.setattr(api, "_torch_stream", lambda s: s)
    monkeypatch.setattr(api, "_default_stream", lambda device: default)
    monkeypatch.setattr(api, "_new_event", FakeEvent)
    a, b, c = Box(), Box(), Box()
    handles = []
    for _ in range(3):
        api._submit(default, [a], [b], handles.append)
    assert handles == [0, 0, 0] and not made and not default.waited  # one stream: no events, no waits
    api._submit(side, [b], [c], lambda s: None)   # reads what the default stream wrote
    assert side.waited == [0] and [e.stream for e in made] == [0, 7]
    api._submit(other, [], [a], lambda s: None)   # overwrites what the default stream read
    assert other.waited == [0]
    api._submit(default, [c], [b], lambda s: None)  # reads what `side` wrote and overwrites what `side` read
    assert default.waited == [7, 7]
    api._submit(default, [b], [c], lambda s: None)  # its own result, and c, which only it has read since
    assert default.waited == [7, 7, 7]  # c was written by `side`


def test_a_stream_that_follows_the_default_one_waits_for_what_it_reads_alone(api, monkeypatch):
    # a program that prepares the next batch on the default stream while another stream works on the last one: from the
    # second wait on, the other stream waits for the write it reads and not for what the default stream was given since; a
    # program that stops doing so gets no events again. No GPU: a stand-in device that counts the default stream's work.
    class FakeStream:
        def __init__(self, key):
            self.cuda_stream, self.device_index, self.work, self.waited = key, 0, 0, []

        def wait_event(self, event):
            self.waited.append((event.stream.cuda_stream, event.at))

    class FakeEvent:
        made = 0

        def __init__(self):
            FakeEvent.made += 1

        def record(self, stream):
            self.stream, self.at = stream, stream.work

    class Box:
        pass

    default, side = FakeStream(0), FakeStream(7)
    monkeypatch.setattr(api, "_torch_stream", lambda s: s)
    monkeypatch.setattr(api, "_default_stream", lambda device: default)
    monkeypatch.setattr(api, "_new_event", FakeEvent)

    def launch(s):
        assert s == 0
        default.work += 1

    def one_batch():
        batch, other = Box(), Box()
        api._submit(default, [], [batch], launch)
        written = default.work
        for _ in range(5):
            api._submit(default, [other], [other], launch)
        api._submit(side, [batch], [], lambda s: None)
        return written

    assert one_batch() == 1 and side.waited == [(0, 6)]
    for _ in range(3):
        written = one_batch()
        assert side.waited[-1] == (0, written)
    other, before = Box(), FakeEvent.made
    for _ in range(2000):
        api._submit(default, [other], [other], launch)
    assert FakeEvent.made - before == api._FOLLOWED_CALLS < 2000


def test_planes_of_buffers_that_have_no_index(api, monkeypatch):
    import types

    import torch
    monkeypatch.setattr(api, "_native", types.SimpleNamespace(planes=lambda buffers: (3, b"planes")))
    frames = {"left": torch.zeros((4, 5, 3), dtype=torch.uint8), "right": torch.zeros((6, 5, 3), dtype=torch.uint8)}
    assert api._plane_list(frames.values(), None) == (int(api.Format.RGB8), b"planes")


def test_images_of_a_batch_asked_for_by_several_threads(api, monkeypatch):
    # a batch made in one call makes its Image objects when they are asked for: every thread gets all of them, the same
    # ones, and a failure loses no buffer (no GPU: the library's call is a stand-in that takes its time)
    import threading
    import time
    import types

    calls = []

    def get_images(handle, first, handles, n):
        calls.append(n)
        time.sleep(0.05)
        return status[0]

    monkeypatch.setattr(api, "_nv", types.SimpleNamespace(nvcvImageBatchVarShapeGetImages=get_images))
    batch = api.ImageBatchVarShape.__new__(api.ImageBatchVarShape)
    batch.handle, batch.images = None, []
    buffers = batch._buffers = [object() for _ in range(5)]
    status = [2]
    with pytest.raises(api.Error):
        batch.images
    assert batch._buffers is buffers and calls == [5]
    status = [0]
    got = []
    threads = [threading.Thread(target=lambda: got.append(list(batch.images))) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 8 and calls == [5, 5]
    assert [i._keep for i in got[0]] == [[b] for b in buffers] and batch._buffers is None
    assert all([id(i) for i in g] == [id(i) for i in got[0]] for g in got)


def test_results_come_back_only_from_the_default_stream_and_unseen(api, monkeypatch):
    # which of an operator's result tensors are handed out again (no GPU: the library's tensors are stand-ins)
    import gc

    class Raw:
        made = 0

        def __init__(self):
            Raw.made += 1
            self.handle = object()

        @classmethod
        def alloc(cls, shape, dtype, layout):
            raw = cls()
            raw.size = int(np.prod(shape)) * np.dtype(dtype).itemsize
            return raw

        def export(self):
            class D:
                rank, shape = 1, [1]

                class buffer:
                    strides = [self.size]
            return D

        def torch_view(self):
            return "view"

    monkeypatch.setattr(api, "_Tensor", Raw)
    monkeypatch.setattr(api.torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    outputs = api._Outputs()
    monkeypatch.setattr(api, "_outputs", outputs)

    def used(mark=(0, None), reads=()):
        t = outputs.get((2, 4), np.float32, "NC")
        t._wrote, t._read = mark, {k: None for k in reads}
        return t

    t = used()
    raw = t._t
    del t
    again = used(reads=[0])
    assert again._t is raw and Raw.made == 1
    other = outputs.get((2, 4), np.uint8, "NC")
    assert Raw.made == 2 and other._t is not raw
    del again
    fresh = outputs.get((2, 4), np.float32, "NC")
    assert fresh._t is raw and fresh._wrote == (0, None)  # a side stream's first use waits for the default stream
    for spoil in (lambda t: t.torch(), lambda t: t.handle, lambda t: setattr(t, "_wrote", (7, None)),
                  lambda t: t._read.update({7: None})):
        t = used()
        raw = t._t
        spoil(t)
        del t
        gc.collect()
        assert outputs.get((2, 4), np.float32, "NC")._t is not raw
    outputs.most_bytes = 4096
    keep = [outputs.get((256,), np.uint8, "N") for _ in range(40)]
    del keep
    assert outputs._bytes <= 4096 and outputs._count <= 16
    big = outputs.get((2048,), np.uint8, "N")
    raw = big._t
    del big
    assert outputs.get((2048,), np.uint8, "N")._t is not raw  # more than a quarter of the bound


def test_default_streams_of_two_devices_are_told_apart(api, monkeypatch):
    # a wait for work on the second device's default stream is for an event recorded there, whatever device is current
    class FakeStream:
        def __init__(self, key, device):
            self.cuda_stream, self.device_index, self.waited = key, device, []

        def wait_event(self, event):
            self.waited.append(event.stream)

    class FakeEvent:
        def record(self, stream):
            self.stream = (stream.cuda_stream, stream.device_index)

    class Box:
        pass

    default = [FakeStream(0, 0), FakeStream(0, 1)]
    monkeypatch.setattr(api, "_torch_stream", lambda s: s)
    monkeypatch.setattr(api, "_default_stream", lambda device: default[device])
    monkeypatch.setattr(api, "_new_event", FakeEvent)
    a, side = Box(), FakeStream(7, 0)
    api._submit(default[1], [], [a], lambda s: None)
    api._submit(side, [a], [], lambda s: None)
    assert side.waited == [(0, 1)]
    api._submit(default[1], [a], [], lambda s: None)
    assert not default[1].waited
    api._submit(default[0], [], [a], lambda s: None)
    assert default[0].waited == [(0, 1), (7, 0), (0, 1)]


def test_results_on_other_streams_are_always_new(api, monkeypatch):
    # a call on another stream (one that is being captured cannot wait for the default stream) takes no kept result
    class FakeStream:
        def __init__(self, key):
            self.cuda_stream, self.device_index = key, 0

    made = []
    monkeypatch.setattr(api, "Tensor", lambda *args: made.append(args) or "new")
    monkeypatch.setattr(api._outputs, "get", lambda *args: "kept")
    assert api._result([2, 3], np.uint8, "HW", FakeStream(7)) == "new" and made == [((2, 3), np.uint8, "HW")]
    assert api._result([2, 3], np.uint8, "HW", FakeStream(0)) == "kept"


def test_results_under_an_entered_default_stream_are_kept_ones(api, monkeypatch):
    # `with Stream.default:` is the default stream too
    class FakeStream:
        cuda_stream, device_index = 0, 0

    monkeypatch.setattr(api, "Tensor", lambda *args: "new")
    monkeypatch.setattr(api._outputs, "get", lambda *args: "kept")
    monkeypatch.setattr(api.Stream._tls, "stack", [FakeStream()], raising=False)
    assert api._result((2, 4), np.float32, "NC", None) == "kept"
    monkeypatch.setattr(FakeStream, "cuda_stream", 7)
    assert api._result((2, 4), np.float32, "NC", None) == "new"


def test_view_that_cannot_be_made_gives_its_owner_back(api, cv):
    # (memory of the host, which torch does not take for a device's)
    class Owner:
        pass

    memory, owner = np.zeros((2, 3), np.uint8), Owner()
    t = cv.Tensor.wrap(memory.ctypes.data, [2, 3], [3, 1], np.uint8, "HW", keep=memory)
    before = sys.getrefcount(owner)
    for _ in range(3):
        with pytest.raises(RuntimeError):
            api._native.torch_view(t.handle.value, 0, 0, owner)
    assert sys.getrefcount(owner) == before


def test_two_copies_of_the_package_in_one_process(api, monkeypatch):
    # what one copy's operators go through are that copy's names
    package = importlib.import_module(api.__package__)
    path = os.path.dirname(package.__file__)
    spec = importlib.util.spec_from_file_location("cvcuda_amd_twice", package.__file__, submodule_search_locations=[path])
    monkeypatch.setitem(sys.modules, "cvcuda_amd_twice", importlib.util.module_from_spec(spec))
    spec.loader.exec_module(sys.modules["cvcuda_amd_twice"])
    other = importlib.import_module("cvcuda_amd_twice.pyapi")
    for name in [m for m in sys.modules if m.startswith("cvcuda_amd_twice.")]:
        monkeypatch.setitem(sys.modules, name, sys.modules[name])
    for one in (api, other):
        monkeypatch.setattr(one, "_submit", lambda *args, one=one: one)
    assert api._run(None, [], [], None) is api and other._run(None, [], [], None) is other


def test_package_over_libraries_kept_elsewhere(api, tmp_path):
    # CVCUDA_AMD_LIBDIR names all that is needed: with the extension there pyapi as well, with the two C libraries alone the
    # ctypes layer, whose tensors are then made through it
    package = os.path.dirname(api.__file__)
    for whole in (False, True):
        root, libdir = tmp_path / str(whole), tmp_path / str(whole) / "elsewhere"
        shutil.copytree(package, root / "pkg", ignore=shutil.ignore_patterns("lib*", "build*", "csrc", "__pycache__"))
        libdir.mkdir()
        for so in ("libnvcv_types.so", "libcvcuda.so") + (("_cvcuda_native.so",) if whole else ()):
            os.symlink(os.path.join(package, "lib", so), libdir / so)
        code = ("import numpy as np, pkg\nassert (pkg.capi.native is None) != %s\n"
                "try:\n    pkg.Tensor.alloc([-1], np.uint8, 'N')\nexcept pkg.Error as e:\n    assert e.status == 2\n"
                "try:\n    import pkg.pyapi\nexcept ImportError as e:\n    assert '_cvcuda_native.so not found' in str(e)\n"
                "    print('no pyapi')\nelse:\n    print('pyapi')\n" % whole)
        r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, CVCUDA_AMD_LIBDIR=str(libdir), PYTHONPATH=str(root)),
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0 and r.stdout.strip() == ("pyapi" if whole else "no pyapi"), r.stdout + r.stderr


def test_extension_is_compiled_again_for_another_python(api, tmp_path, monkeypatch):
    spec = importlib.util.spec_from_file_location("_cvbuild_again", os.path.join(os.path.dirname(api.__file__), "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    src, obj, made = tmp_path / "Native.cpp", tmp_path / "Native.o", []
    src.write_text("")

    def run(cmd, **kw):
        made.append(cmd)
        obj.write_text("")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(build.subprocess, "run", run)
    for compiled, version in ((1, "one"), (1, "one"), (2, "two"), (2, "two")):
        monkeypatch.setattr(build.sys, "version", version)
        build._compile_native(str(src), str(obj), False, 0)
        assert len(made) == compiled


def test_kept_results_make_room_where_there_is_no_memory(api, monkeypatch):
    # an allocation that finds no memory is tried once more without the kept results, which it would otherwise never reach;
    # clear_cache() gives them and the library's blocks back (no GPU: the library's tensors are stand-ins)
    class Raw:
        alive, most = 0, 3

        def __init__(self):
            Raw.alive += 1

        def __del__(self):
            Raw.alive -= 1

        @classmethod
        def alloc(cls, shape, dtype=None, layout=None, row_align=0):
            if cls.alive >= cls.most:
                raise api.Error(7, "no memory")
            if shape == [0]:
                raise api.Error(2, "empty")
            return cls()

        for_images = alloc

        def export(self):
            class D:
                rank, shape = 1, [1]

                class buffer:
                    strides = [1]
            return D

    class Picture(api._Image):
        @staticmethod
        def alloc(size, fmt, row_align=0):
            made = Raw.alloc(size)
            made.handle = api.C.c_void_p()
            return made

    outputs = api._Outputs()
    monkeypatch.setattr(api, "_Tensor", Raw)
    monkeypatch.setattr(api, "_Image", Picture)
    monkeypatch.setattr(api, "_outputs", outputs)
    monkeypatch.setattr(api.torch._C, "_cuda_getDevice", lambda: 0, raising=False)

    def fill():
        kept = [outputs.get((n,), np.uint8, "N") for n in (1, 2, 3)]
        for t in kept:
            t._wrote = (0, None)
        del kept, t
        assert Raw.alive == outputs._count == 3

    for make in (lambda: outputs.get((9,), np.uint8, "N"), lambda: api.Tensor((4,), np.uint8, "N"),
                 lambda: api.Tensor(2, (4, 4), api.Format.U8), lambda: api.Image((4, 4), api.Format.U8)):
        fill()
        made = make()
        assert outputs._count == 0
        del made
        outputs.clear()
        assert Raw.alive == 0
    held = [api.Tensor((n,), np.uint8, "N") for n in (4, 5, 6)]
    with pytest.raises(api.Error) as e:  # nothing left to give back
        api.Tensor((7,), np.uint8, "N")
    assert e.value.status == 7
    del held, e
    fill()
    Raw.most = 9
    with pytest.raises(api.Error) as e:
        api.Tensor((0,), np.uint8, "N")
    assert e.value.status == 2 and outputs._count == 3  # another error than want of memory
    api.clear_cache()
    assert Raw.alive == outputs._count == outputs._bytes == 0


def test_a_copy_of_the_package_that_nobody_has_is_collected(api):
    # with the results that it kept, which belong to a table that holds the copy's names
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    program = """
import gc, importlib, importlib.util, sys, weakref
package = %r
spec = importlib.util.spec_from_file_location("pkg", package + "/__init__.py", submodule_search_locations=[package])
module = sys.modules["pkg"] = importlib.util.module_from_spec(spec)
spec.loader.exec_module(module)
api = importlib.import_module("pkg.pyapi")
class Raw:
    _nbytes = 1
    api = api
result = api.Tensor(_wrap=Raw())
result._key, result._wrote = ((1,), "u1", "N", 0), (0, None)
result = None
assert api._outputs._count == 1
gone = [weakref.ref(o) for o in (module, api, api._outputs, api.Tensor, Raw)]
for name in [n for n in sys.modules if n.split(".")[0] == "pkg"]:
    del sys.modules[name]
del spec, module, api, Raw
gc.collect()
assert [g() for g in gone] == [None] * 5, gone
""" % os.path.join(root, "cv-cuda_amd")
    r = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and not r.stderr, r.stderr
    empty = api._native.Outputs.__new__(api._native.Outputs)  # without tables: not a crash
    for call in (empty.clear, lambda: empty.get((1,), np.uint8, "N")):
        with pytest.raises(RuntimeError):
            call()
    empty.put(api.Tensor(_wrap=object()))


@pytest.mark.parametrize("handle", [None, C.c_void_p()])
def test_a_closed_image_batch_is_an_invalid_argument(api, handle):
    batch = api.ImageBatchVarShape.__new__(api.ImageBatchVarShape)
    batch.handle, batch._keep = handle, []
    for use in (lambda: len(batch), lambda: batch.uniqueformat,
                lambda: api.resize_crop_convert_reformat(batch, (4, 4), api.Interp.LINEAR, api.RectI(0, 0, 4, 4))):
        with pytest.raises(api.Error, match="NVCV_ERROR_INVALID_ARGUMENT"):
            use()


def test_results_alive_at_the_end_of_the_program_say_nothing():
    # a module's result tensors that outlive this package's module globals: nothing on stderr
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    program = """
import sys
sys.path.insert(0, %r)
from __graft_entry__ import load_package
load_package()
import cvcuda_amd.pyapi as api
class Raw:
    _nbytes = 1
result = api.Tensor(_wrap=Raw())
result._key, result._wrote = ((1,), "u1", "N", 0), (0, None)
api.kept = result
""" % root
    r = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "Exception ignored" not in r.stderr, r.stderr
