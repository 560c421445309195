"""The native host path (csrc/host_calls.cpp) against the general Python path behind it: the same bytes, and the same error
for every call that one of them refuses.  A tensor subclass takes the general path, whatever else the call looks like."""
import os
import shutil
import subprocess
import sys

import pytest
import torch

from monarch_amd import MhipError, Slice, fp8, staging
from monarch_amd import reduce as R
from monarch_amd._native import host
from monarch_amd.staging import RDMABuffer
from util import sync

DEV = "cuda:0"


class Sub(torch.Tensor):
    pass


def general(x):
    if isinstance(x, torch.Tensor):
        return x.as_subclass(Sub)
    return type(x)(general(t) for t in x) if isinstance(x, (list, tuple)) else x


def outcome(call, *args):
    try:
        r = call(*args)
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)
    return r


def test_calls_that_are_not_on_plain_tensors_are_left_alone():
    s = Slice(offset=0, sizes=[4], strides=[1])
    x = torch.zeros(4)
    for args in ((True, x, s, x), (True, None, s, x), (True, x, None, x), (True, 1, 2, 3)):
        assert host.slice_copy(*args) == host.NOT_TAKEN
    assert host.slice_copy_many(True, x, [s], [x]) == host.NOT_TAKEN and host.slice_copy_many(True, x, iter([s]), x) == host.NOT_TAKEN
    assert host.reduce(x, [x], 0) == host.NOT_TAKEN and host.stack(x, [x]) == host.NOT_TAKEN
    assert host.rdma_copy(True, 0, 4, x, 0) == host.NOT_TAKEN and host.rdma_copy(True, -1, 4, x, None) == host.NOT_TAKEN
    assert host.reduce_scatter([x], [s], [x], s, 0) == host.NOT_TAKEN
    assert host.transfer_many([1], [1], "x", 0) == host.NOT_TAKEN and host.transfer_many([], [], [], 0) == host.NOT_TAKEN
    assert host.flat_copy(True, x, x, x, 4, None, None) == host.NOT_TAKEN
    assert host.quantize_bucket(x, x, 4, None, x, x) == host.NOT_TAKEN
    assert host.dequant_accumulate_bucket(x, x, 4, None, [x], [x]) == host.NOT_TAKEN
    assert host.tensor_addresses([x], (4).to_bytes(8, "little"), x) is None
    with pytest.raises(TypeError):
        host.slice_copy(True)


@pytest.mark.parametrize("status", [1, 2, 719, 10201])
def test_transfers_that_fail_are_not_posted_again(monkeypatch, status):
    # minus a status (a C int) is none of a count, a status and the mark of a call that was left alone
    assert host.NOT_TAKEN < -(1 << 31)

    class Failing:
        NOT_TAKEN = host.NOT_TAKEN
        transfer_many = staticmethod(lambda *args: -status)

    monkeypatch.setattr(staging, "host", Failing)
    monkeypatch.setattr(staging, "lib", lambda: pytest.fail("posted a second time"))
    with pytest.raises(MhipError) as e:
        staging.transfer_many([16], [32], [8])
    assert e.value.status == status


def _filled(n, dtype=torch.float32, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-100, 100, (n,), device=DEV, generator=g).to(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.float64])
def test_slice_copies(dtype):
    base = _filled(600, dtype, 1)
    for s in (Slice(offset=3, sizes=[7, 20], strides=[40, 2]), Slice(offset=0, sizes=[600], strides=[1]), Slice(offset=5, sizes=[0, 3], strides=[3, 1]),
              Slice(offset=599, sizes=[], strides=[])):
        n = len(s)
        a, b = torch.zeros(n, dtype=dtype, device=DEV), torch.zeros(n, dtype=dtype, device=DEV)
        assert host.slice_copy(True, base, s, a) == 0 and host.slice_copy(True, general(base), s, a) == host.NOT_TAKEN
        assert staging.pack(base, s, a) is a
        staging.pack(general(base), s, b)
        back = [torch.zeros_like(base) for _ in range(2)]
        staging.unpack(back[0], s, a)
        staging.unpack(general(back[1]), s, b)
        sync()
        assert torch.equal(a, b) and torch.equal(*back)
        many = [[torch.zeros(n, dtype=dtype, device=DEV) for _ in range(3)] for _ in range(2)]
        assert staging.pack_many(base, [s] * 3, many[0]) is many[0]
        staging.pack_many(general(base), [s] * 3, many[1])
        sync()
        assert all(torch.equal(x, a) for x in many[0] + many[1])
    s = Slice(offset=0, sizes=[10], strides=[2])
    good = torch.zeros(10, dtype=dtype, device=DEV)
    bad = [(base, Slice(offset=590, sizes=[10], strides=[2]), good), (base, s, good[:9]), (base, s, torch.zeros(20, dtype=dtype, device=DEV)[::2]),
           (base.cpu(), s, good), (base, s, good.cpu()), (base, Slice(offset=0, sizes=[1 << 40, 4], strides=[1 << 30, 1], _validate=False), good)]
    for b, view, out in bad:
        for f in (staging.pack, staging.unpack):
            got = outcome(f, b, view, out)
            assert isinstance(got, tuple) and got == outcome(f, general(b), view, general(out)), (f, view)
        got = outcome(staging.pack_many, b, [view], [out])
        assert isinstance(got, tuple) and got == outcome(staging.pack_many, general(b), [view], [general(out)])


@pytest.mark.gpu
def test_buffer_transfers():
    x, y = _filled(1001, torch.uint8, 2), _filled(500, torch.uint8, 3)
    for offset in (0, 17, 501):
        a, b = torch.zeros(500, dtype=torch.uint8, device=DEV), torch.zeros(500, dtype=torch.uint8, device=DEV)
        assert host.rdma_copy(True, x.data_ptr(), 1001, a, offset) == 0
        assert RDMABuffer(x).read_into(a, offset) == RDMABuffer(x).read_into(general(b), offset) == 500
        z = [x.clone(), x.clone()]
        RDMABuffer(z[0]).write_from(y, offset)
        RDMABuffer(z[1]).write_from(general(y), offset)
        sync()
        assert torch.equal(a, x[offset: offset + 500]) and torch.equal(a, b) and torch.equal(*z) and torch.equal(z[0][offset: offset + 500], y)
    buf = RDMABuffer(x)
    for t, offset in ((y, 502), (y, -1), (y.view(torch.int8), 0), (y.view(5, 100), 0), (_filled(40, torch.uint8)[::2], 0), (y.cpu(), 0)):
        for f in (buf.read_into, buf.write_from):
            got = outcome(f, t, offset)
            assert isinstance(got, tuple) and got == outcome(f, general(t), offset)
    out = torch.zeros(300, dtype=torch.uint8, device=DEV)
    assert staging.transfer_many([out.data_ptr(), out.data_ptr() + 100], [x.data_ptr(), y.data_ptr()], [100, 200], 64) == 6
    sync()
    assert torch.equal(out, torch.cat([x[:100], y[:200]]))
    got = outcome(staging.transfer_many, [0], [x.data_ptr()], [5])
    assert isinstance(got, tuple) and got == outcome(staging.transfer_many, [0], [x.data_ptr()], [5], 0, torch.cuda.current_stream())
    with pytest.raises(ValueError):
        staging.transfer_many([1], [1, 2], [1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.float64])
def test_reductions(dtype):
    group = [_filled(333, dtype, r) for r in range(5)]
    ops = [R.ReduceOp.Sum, R.ReduceOp.Max] + ([R.ReduceOp.Avg] if dtype.is_floating_point else [])
    for op in ops:
        a, b = torch.zeros(333, dtype=dtype, device=DEV), torch.zeros(333, dtype=dtype, device=DEV)
        assert host.reduce(a, group, op) == 0
        R.all_reduce(a, tuple(group), op)
        R.all_reduce(general(b), general(group), op)
        c = R.stream_reduce(group, 2, R.Factory.of(a), R.Reduction(op), False, False, out=torch.zeros_like(a))
        d = R.stream_reduce([None] + group[1:], 2, R.Factory.of(a), R.Reduction(op), False, False, out=torch.zeros_like(a))
        e = torch.zeros_like(a)
        R.all_reduce(e, [torch.zeros_like(a)] + group[1:], op)
        sync()
        assert torch.equal(a, b) and torch.equal(a, c) and torch.equal(d, e)
    out = torch.zeros(5, 333, dtype=dtype, device=DEV)
    assert R.stream_reduce(group, 4, R.Factory.of(group[0]), R.Reduction(None), False, False, out=out) is out
    sync()
    assert torch.equal(out, torch.stack(group))
    views = [Slice(offset=k * 2, sizes=[30, 2], strides=[10, 1]) for k in range(5)]
    view = Slice(offset=3, sizes=[30, 10], strides=[11, 1])
    outs = [[torch.zeros(60, dtype=dtype, device=DEV) for _ in views] for _ in range(2)]
    R.reduce_scatter_views(outs[0], views, group, view, ops[0])
    R.reduce_scatter_views(general(outs[1]), views, group, view, ops[0])
    sync()
    assert all(torch.equal(x, y) for x, y in zip(*outs))
    a, f = torch.zeros(333, dtype=dtype, device=DEV), R.Factory.of(group[0])
    other = torch.int32
    for o, g, op in ((a, [group[0], group[1].to(other)], 0), (a, [group[0][:5]], 0), (a[:3], group, 0), (a, group, 99), (a.cpu(), group, 0), (a, [a.cpu()], 0),
                     (a.bool(), [a.bool()], 4), (torch.zeros(666, dtype=dtype, device=DEV)[::2], group, 0), (a, [], 0), (a, [group[0]] * 65, 0)):
        got = outcome(R.all_reduce, o, g, op)
        assert isinstance(got, tuple) and got == outcome(R.all_reduce, general(o), general(g), op)
    for o, rank in ((out[:4], 0), (out.to(other), 0), (out, 5)):
        args = (f, R.Reduction(None), False, False)
        got = outcome(R.stream_reduce, group, rank, *args, o)
        assert isinstance(got, tuple) and got == outcome(R.stream_reduce, general(group), rank, *args, general(o))
    got = outcome(R.reduce_scatter_views, [outs[0][0][:5]], views[:1], group, view, 0)
    assert isinstance(got, tuple) and got == outcome(R.reduce_scatter_views, general([outs[0][0][:5]]), views[:1], group, view, 0)


@pytest.mark.gpu
def test_buckets():
    sizes = [1500, 0, 1, 3000]
    total = sum(sizes)
    bucket = fp8.FlatBucket([_filled(n, torch.bfloat16, n) for n in sizes])
    acc = [fp8.FlatBucket([_filled(n, torch.float32, n) for n in sizes]) for _ in range(2)]
    for indexed in (False, True):
        if indexed:
            for b in (bucket, *acc):
                b.block_index()
        flat = [torch.zeros(total, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        assert bucket.pack(flat[0]) is flat[0]
        bucket.pack(general(flat[1]))
        outs = [[torch.zeros(n, dtype=torch.int16, device=DEV) for n in sizes] for _ in range(2)]
        bucket.unpack(flat[0], outs[0])
        bucket.unpack(general(flat[1]), outs[1])
        assert bucket.pointer_table(outs[0]).data_ptr() == bucket.pointer_table(general(outs[0])).data_ptr()
        qs = [[torch.zeros(total, dtype=torch.uint8, device=DEV), torch.zeros((total + 1023) // 1024, device=DEV)] for _ in range(2)]
        fp8.quantize_bucket(bucket, *qs[0])
        fp8.quantize_bucket(bucket, general(qs[1][0]), qs[1][1])
        for a, q in zip(acc, (qs[0][0], general(qs[0][0]))):
            fp8.dequant_accumulate_bucket_many(a, [q, q], [qs[0][1], qs[0][1]])
        sync()
        assert torch.equal(*flat) and torch.equal(flat[0], torch.cat(bucket.tensors))
        assert all(torch.equal(x, y) and torch.equal(x, t.view(torch.int16)) for x, y, t in zip(*outs, bucket.tensors))
        assert all(torch.equal(x, y) for x, y in zip(*qs)) and all(torch.equal(x, y) for x, y in zip(acc[0].tensors, acc[1].tensors))
    for f in (flat[0][:-1], flat[0].view(torch.float16), flat[0].float(), flat[0].cpu(), torch.zeros(2 * total, dtype=torch.bfloat16, device=DEV)[::2]):
        got = outcome(bucket.pack, f)
        assert isinstance(got, tuple) and got == outcome(bucket.pack, general(f))
    tables = len(bucket._tables)
    for f, o in ((flat[0][:-1], outs[0]), (flat[0].float(), outs[0]), (flat[0], outs[0][:-1]), (flat[0], outs[0][::-1]), (flat[0], [t.cpu() for t in outs[0]])):
        got = outcome(bucket.unpack, f, o)
        assert isinstance(got, tuple) and got == outcome(bucket.unpack, general(f), general(o))
    assert len(bucket._tables) == tables
    q, s = qs[0]
    for bad in ((q[:-1], s), (q, s[:-1]), (q, s.double()), (q.int(), s), (q.cpu(), s)):
        for call, b in ((lambda b, q, s: fp8.quantize_bucket(b, q, s), bucket), (lambda b, q, s: fp8.dequant_accumulate_bucket_many(b, [q], [s]), acc[0])):
            got = outcome(call, b, *bad)
            assert isinstance(got, tuple) and got == outcome(call, b, *general(bad))


@pytest.mark.gpu
def test_the_current_stream_is_the_one_that_is_used():
    # a call under torch.cuda.stream goes to that stream, from a second thread as well, and can be captured
    import threading
    x, s = _filled(4096, torch.float32, 5), Slice(offset=0, sizes=[2048], strides=[2])
    out, side = torch.zeros(2048, device=DEV), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    staging.pack(x, s, out)
    sync()
    out.zero_()
    with torch.cuda.graph(graph, stream=side):
        assert host.slice_copy(True, x, s, out) == 0
    for _ in range(3):
        out.zero_()
        graph.replay()
        sync()
        assert torch.equal(out, x[::2])
    outs = [torch.zeros(2048, device=DEV) for _ in range(4)]
    sync()

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                staging.pack(x, s, outs[k])
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(o, x[::2]) for o in outs)


@pytest.mark.gpu
def test_tensors_of_a_call_are_held_while_the_library_runs(tmp_path):
    here = os.path.dirname(os.path.abspath(__file__))
    shutil.copy(host.slice_copy.__self__.__file__, tmp_path)
    subprocess.check_call(["gcc", "-shared", "-fPIC", os.path.join(here, "c_abi", "held_library.c"), "-o", str(tmp_path / "libmonarch_hip.so")])
    p = subprocess.run([sys.executable, os.path.join(here, "host_calls_held.py"), str(tmp_path)], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.endswith("host_calls_held ok\n"), p.stdout + p.stderr[-2000:]
