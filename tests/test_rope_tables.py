"""The kept RoPE tables (decoder._kept_table): stream order, lifetime and captures.
The logic runs on the CPU with stand-ins for streams and events; on the GPU the
rope attention runs from threads on streams of their own and in a graph."""
import threading
import types

import pytest
import torch


class _Stream:
    def __init__(self, handle):
        self.cuda_stream, self.waited = handle, []

    def wait_event(self, event):
        self.waited.append(event)


class _Event:
    done = False

    def record(self, stream):
        self.stream = stream

    def query(self):
        return self.done


@pytest.fixture
def fake(ca, monkeypatch):
    """Streams, events and captures under the test's control; read notes in ``noted``."""
    st = types.SimpleNamespace(stream=_Stream(1), capturing=False, noted=[], event=_Event)
    monkeypatch.setattr(_Event, "done", False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: st.stream)
    monkeypatch.setattr(ca.native, "stream_handle", lambda device: st.stream.cuda_stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: st.capturing)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(torch.Tensor, "record_stream",
                        lambda t, s: st.noted.append((t.data_ptr(), s.cuda_stream)))
    st.cache, st.builds = {}, 0

    def get(key):
        def build():
            st.builds += 1
            return (torch.zeros(3),)
        return ca.decoder._kept_table(st.cache, key, torch.device("cuda", 0), build)[0]
    st.get = get
    return st


def test_another_stream_waits_until_the_table_is_written(fake):
    first, other = fake.stream, _Stream(2)
    t = fake.get("a")
    assert fake.get("a") is t and fake.builds == 1 and not first.waited  # its own stream: in order
    fake.stream = other
    assert fake.get("a") is t and len(other.waited) == 1
    assert other.waited[0].stream is first
    assert fake.noted == [(t.data_ptr(), 2)]  # the allocator knows the reader
    _Event.done = True
    assert fake.get("a") is t and len(other.waited) == 1  # written: no more waits
    third = fake.stream = _Stream(3)
    assert fake.get("a") is t and not third.waited and fake.noted[-1] == (t.data_ptr(), 3)


def test_captures_take_written_tables_only_and_keep_them(ca, fake):
    t = fake.get("a")
    fake.capturing = True
    inside = fake.get("a")  # not known to be written: built in the graph, not kept
    assert inside is not t and fake.get("b") is not None and list(fake.cache) == ["a"]
    fake.capturing = False
    _Event.done = True
    assert fake.get("a") is t
    fake.capturing = True
    assert fake.get("a") is t
    fake.capturing = False
    for n in range(2 * ca.decoder._TABLES_KEPT):  # the oldest go, a captured one stays
        fake.get(n)
    assert len(fake.cache) == ca.decoder._TABLES_KEPT and fake.get("a") is t


def test_table_built_in_inference_mode_serves_training(ca):
    q = torch.randn(1, 1, 19, 6, requires_grad=True)
    with torch.inference_mode():
        ca.decoder.apply_rope(q.detach(), q.detach(), 123.0)
    a, b = ca.decoder.apply_rope(q, q, 123.0)
    (a.sum() + b.sum()).backward()
    assert q.grad is not None


def _case(ca, T, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(2, T, 3 * 4 * 32, generator=g).to(torch.bfloat16).cuda().requires_grad_()
    r = (0.1 * torch.randn(4, generator=g)).cuda().requires_grad_()
    dy = torch.randn(2, T, 4 * 32, generator=g).to(torch.bfloat16).cuda()

    def run():
        y = ca.decoder.rope_continuum_attention(x, r, 1e4, 4)
        return [y.detach(), *torch.autograd.grad(y, [x, r], dy)]
    return run


@pytest.mark.gpu
def test_rope_from_threads_on_streams(gpu_ca):
    """Three threads on three streams, at a shape whose table none has built."""
    T = 333
    runs = [_case(gpu_ca, T, n) for n in range(3)]
    got = [None] * 3

    def work(n):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            for _ in range(3):
                got[n] = runs[n]()
        s.synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(n,)) for n in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for n in range(3):
        assert all(torch.equal(a, b) for a, b in zip(runs[n](), got[n]))


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [True, False])
def test_graph_replays_with_a_kept_table(gpu_ca, warm):
    """A captured rope attention after its table would have been dropped (warm)
    and with a table built inside the graph: every replay the eager result."""
    T = 211 if warm else 212
    qkv = torch.randn(1, T, 3 * 2 * 32, device="cuda")
    gain = torch.zeros(2, device="cuda")

    def call():
        with torch.no_grad():
            return gpu_ca.decoder.rope_continuum_attention(qkv, gain, 1e4, 2)

    if warm:
        call()
        torch.cuda.synchronize()
        gpu_ca.decoder._mark_written_tables()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for n in range(gpu_ca.decoder._TABLES_KEPT + 1):
        gpu_ca.decoder.rope_cos_sin(8, 32, 100.0 + n, qkv.device)
    for n in range(3):
        junk = [torch.full((T, 16, 2), 7.0, device="cuda") for _ in range(8)]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, call())
        del junk


def test_constant_gains_are_kept_the_same_way(ca, monkeypatch):
    """TinyLM's constant log-gain: one tensor per (device, value) through
    _kept_table, none on the module (which stays copyable)."""
    import copy
    A = ca.architecture
    seen = []
    monkeypatch.setattr(A, "_kept_table", lambda *a: seen.append(a[0]) or ca.decoder._kept_table(*a))
    attn = types.SimpleNamespace(variant="B", fixed_tau=0.5, heads=3)
    gain = A.CausalAttention._log_gain(attn, torch.device("cpu"))
    assert seen[0] is ca.decoder._GAIN_CACHE and gain.shape == (3,)
    assert A.CausalAttention._log_gain(attn, torch.device("cpu")) is gain
    assert set(vars(copy.deepcopy(attn))) == {"variant", "fixed_tau", "heads"}
