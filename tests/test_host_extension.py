"""The host extension's packing, allocation and entry calls (CPU): each refuses what does not fit."""

import ctypes
import threading
import time

import numpy as np
import pytest
import torch

from sonic_sampler import _native


class Example(ctypes.Structure):
    _fields_ = [("count", ctypes.c_int32), ("mask", ctypes.c_uint32), ("plane", ctypes.c_void_p),
                ("stride_plane", ctypes.c_int64), ("stride_step", ctypes.c_int64), ("seed", ctypes.c_uint64),
                ("row", ctypes.c_void_p), ("stride_row", ctypes.c_int64), ("one", ctypes.c_void_p)]


def gatherer():

    return _native.Gatherer(Example, dict(plane="U", row="S", one="T"), labels=dict(plane="the plane"))


@pytest.mark.parametrize("plane", [torch.zeros(3, 4, 5), torch.zeros(3, 5), torch.zeros(6, 4, 5)[::2, 1:], None])
def test_gathers_addresses_strides_and_scalars(plane):

    row = torch.zeros(7, 9).T
    g = gatherer()
    assert g.fields == ("count", "mask", "plane", "seed", "row", "one")
    got = Example.from_buffer_copy(g.gather(np.int64(-5), np.uint32(2 ** 32 - 1), plane, 2 ** 64 - 1, row, None))
    assert (got.count, got.mask, got.seed, got.one) == (-5, 2 ** 32 - 1, 2 ** 64 - 1, None)
    assert (got.row, got.stride_row) == (row.data_ptr(), 1)
    want = (None, 0, 0) if plane is None else (plane.data_ptr(), plane.stride(0), plane.stride(1) if plane.dim() == 3 else 0)
    assert (got.plane, got.stride_plane, got.stride_step) == want


@pytest.mark.parametrize("args,error,text", [
    ((2 ** 31, 0, None, 0, None, None), OverflowError, "count"),
    ((0, 2 ** 32, None, 0, None, None), OverflowError, "mask"),
    ((0, -1, None, 0, None, None), OverflowError, "negative"),
    ((0, 0, None, 0.5, None, None), TypeError, "integer"),
    ((0, 0, 7, 0, None, None), TypeError, "the plane"),
    ((0, 0, None, 0, None), TypeError, "arguments"),
])
def test_refuses_what_does_not_fit(args, error, text):

    with pytest.raises(error, match=text):

        gatherer().gather(*args)


def test_unit_strides_name_the_tensor():

    check = _native.unit_strides
    check(("a", "b", "c", "d"), torch.zeros(4, 4), None, torch.zeros(8, 2)[::2], torch.tensor(1.0))

    with pytest.raises(ValueError, match="`b` must be contiguous along its last dimension"):

        check(("a", "b"), torch.zeros(4, 4), torch.zeros(4, 4).T)

    with pytest.raises(ValueError, match="`a`"):

        check(("a",), torch.zeros(8)[::2])

    with pytest.raises(TypeError, match="`a` must be a tensor"):

        check(("a",), 7)

    with pytest.raises(TypeError):

        check(("a",), None, None)


@pytest.mark.parametrize("size,field,error", [
    (16, ("\0", 0, 0, 0, "x"), ValueError), (16, ("x", 0, 0, 0, "x"), ValueError), (16, ("\u0169", 0, 0, 0, "x"), ValueError),
    (16, ("q", 9, 0, 0, "x"), ValueError), (16, ("q", 2 ** 63 - 1, 0, 0, "x"), ValueError), (4, ("q", 0, 0, 0, "x"), ValueError),
    (16, ("S", 0, 16, 0, "x"), ValueError), (16, ("i", -1, 0, 0, "x"), ValueError), (16, ("i", 0), TypeError),
])
def test_layouts_refuse_fields_outside_the_struct(size, field, error):

    with pytest.raises(error):

        _native.host().make_layout(size, [field])


def test_empty_is_torch_empty():

    t = _native.empty(torch.device("cpu"), torch.bfloat16, 3, 0, 2)
    assert t.shape == (3, 0, 2) and t.dtype == torch.bfloat16 and t.device.type == "cpu" and not t.requires_grad

    with pytest.raises(RuntimeError):

        _native.empty(torch.device("cpu"), torch.int32, -3)

    with pytest.raises(TypeError):

        _native.host().empty("cpu", torch.int32, 3)


@pytest.mark.parametrize("device", ["cpu", torch.device("cpu"), None])
def test_output_containers_take_any_form_of_a_device(device, monkeypatch):
    """As torch.empty does; on the CPU without the host extension."""

    from sonic_sampler.base.sampler import LogProbabilities, TopTargets

    monkeypatch.setattr(_native, "host", lambda: pytest.fail("the host extension was asked for"))
    monkeypatch.setattr(_native, "_empty", None)

    for t in (LogProbabilities.empty_blocked(2, 3, 4, device=device), LogProbabilities.empty_varlen(6, 4, device=device)):

        assert t.selected.device.type == "cpu" and t.selected.dtype == torch.bfloat16
        assert t.top_k.tokens.dtype == torch.int32 and t.top_k.logprobs.numel() == 24

    assert TopTargets.empty_blocked(2, 4, device=device).tokens.shape == (2, 4)
    assert TopTargets.empty_varlen(6, 4, device=device).logprobs.shape == (6, 4)


@pytest.mark.parametrize("device", ["cuda", "cuda:0", 0])
def test_output_containers_name_a_gpu_as_torch_does(device, monkeypatch):
    """A GPU's name or index goes to torch.empty as it is."""

    from sonic_sampler.base.sampler import LogProbabilities

    seen = []
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: seen.append(kw["device"]))
    LogProbabilities.empty_varlen(6, device=device)
    assert seen == [device]


def test_outputs_are_of_their_source_class():
    """Token and offset buffers made for a tensor subclass are of that class, as new_empty and
    empty_like make them: the buffers' prefix-contiguous slices index differently."""

    from sonic_sampler.base.sampler import Verification
    from sonic_sampler.base.tensor import PrefixContiguousTensor, prefix_contiguous
    from sonic_sampler.interface.functional import multistep, singular

    drafted = prefix_contiguous(torch.zeros(4, 3, dtype=torch.int32))
    tokens = multistep.resolve_tokens(drafted, None)
    assert type(tokens) is PrefixContiguousTensor and tokens.shape == (4, 3) and tokens.dtype == torch.int32
    assert type(Verification.from_tokens(tokens, 4, 3).offsets) is PrefixContiguousTensor
    logits = prefix_contiguous(torch.zeros(4, 8, dtype=torch.bfloat16))
    assert type(singular.resolve_tokens(None, 4, logits)) is PrefixContiguousTensor
    assert type(multistep.resolve_tokens(drafted.as_subclass(torch.Tensor), None)) is torch.Tensor


def test_errors_are_those_of_torch():
    """A failed allocation and a stride that a tensor does not have raise what torch's own calls do."""

    call = _native.host().empty
    backend = torch.device("xla")

    with pytest.raises(Exception) as want:

        torch.empty(3, device=backend)

    with pytest.raises(type(want.value)) as got:

        call(backend, torch.float32, 3)

    assert type(want.value) is not RuntimeError and type(got.value) is type(want.value)

    with pytest.raises(IndexError):

        gatherer().gather(0, 0, None, 0, torch.tensor(1.0), None)


def test_allocation_lets_other_threads_run():
    """A second thread goes on while an allocation takes its time (here: the fill of deterministic
    mode), as it does beside torch.empty."""

    call, stamps, stop = _native.host().empty, [], threading.Event()

    def tick():

        while not stop.is_set():

            stamps.append(time.perf_counter())
            time.sleep(0.001)

    thread = threading.Thread(target=tick)
    torch.use_deterministic_algorithms(True)

    try:

        thread.start()
        start = time.perf_counter()
        kept = call(torch.device("cpu"), torch.float32, 2 ** 28)
        end = time.perf_counter()

    finally:

        stop.set()
        thread.join()
        torch.use_deterministic_algorithms(False)

    assert kept[0].isnan() and end - start > 0.02, "the fill was too short to tell"
    inside = [s for s in stamps if start + 0.2 * (end - start) < s < end - 0.2 * (end - start)]
    assert inside, "no other thread ran during the allocation"


@pytest.mark.gpu
def test_out_of_memory_is_torchs():
    """With the process held to a small share of the card, which the allocator checks itself."""

    device = torch.device("cuda:0")
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction(0.05, device)

    try:

        with pytest.raises(torch.OutOfMemoryError):

            _native.empty(device, torch.uint8, total // 10)

    finally:

        torch.cuda.set_per_process_memory_fraction(1.0, device)


def test_entries_take_bytes_only():

    call = _native.packed_entry("ss_topk")

    with pytest.raises(TypeError):

        call(None)

    # a struct that ends early would be read past its end
    for size in (0, ctypes.sizeof(_native.TopKArgs) - 1, ctypes.sizeof(_native.TopKArgs) + 8):

        with pytest.raises(ValueError, match="bytes"):

            call(bytes(size))

    with pytest.raises(ValueError):

        _native.host().entry(0, 8)

    assert call(bytes(ctypes.sizeof(_native.TopKArgs))) == 1  # no logits
