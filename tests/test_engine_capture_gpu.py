"""LoraUnorderedBatchInfer recorded into a HIP graph (an object that was built outside records its steps, the first one
included, and stays usable outside the graph), begun ahead of the device and on several streams."""
import numpy as np
import pytest
import torch

from test_engine_gpu import _Model

pytestmark = pytest.mark.gpu


def _engine(gpu, is_prefill, hidden=4096):
    """An engine that has run no step, its arguments of begin_step and one layer's tensors."""
    from slora_hip import LoraUnorderedBatchInfer
    m = _Model(gpu, "f16", hidden, hidden, 1, {"a": 8, "b": 16, "c": 8}, heads=hidden // 128)
    rng = np.random.default_rng(4)
    req = [m.names[i] for i in rng.integers(0, 3, size=7)]
    lens = np.asarray([40, 70, 3, 55, 64, 90, 21] if is_prefill else [9] * 7, np.int32)
    n_tok = int(lens.sum()) if is_prefill else len(req)
    step = dict(b_start_loc=torch.from_numpy(np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)).to(gpu),
                b_seq_len=torch.from_numpy(lens).to(gpu), is_prefill=is_prefill, max_b_seq_len=int(lens.max()),
                total_token_num=n_tok)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(8)
    t = [torch.empty((n_tok, hidden), dtype=m.tdt, device=gpu).normal_(generator=gen) for _ in range(6)]
    return m, (lambda: LoraUnorderedBatchInfer(m.ia, [m.adapters[n] for n in req])), step, t


def _layer(eng, step, t, y):
    for a, b in zip(y, t[2:]):
        a.copy_(b)
    eng.begin_step(**step)
    eng.lora_get_qkv(0, t[0], *y[:3])
    eng.lora_get_o(0, t[1], y[3])


@pytest.mark.parametrize("is_prefill", [False, True], ids=["decode", "prefill"])
def test_the_first_step_of_an_engine_is_recorded(gpu, is_prefill):
    """Built outside, first stepped inside a capture: every replay gives the eager bits, the object steps eagerly after the
    capture (before and between replays), and a step recorded a second time by the same object is right as well."""
    m, new, step, t = _engine(gpu, is_prefill)
    want = [torch.empty_like(v) for v in t[2:]]
    _layer(new(), step, t, want)              # (another object; also loads the kernels)
    torch.cuda.synchronize()
    eng = new()
    graphs = []
    for _ in range(2):
        y = [torch.zeros_like(v) for v in t[2:]]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            _layer(eng, step, t, y)
        graphs.append((g, y))
        late = [torch.zeros_like(v) for v in t[2:]]
        _layer(eng, step, t, late)            # nothing of the recorded step has run yet
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(late, want))
    for rep in range(3):
        for g, y in graphs:
            for v in y:
                v.zero_()
            g.replay()
            torch.cuda.synchronize()
            for a, b in zip(y, want):
                assert torch.equal(a, b), rep


@pytest.mark.parametrize("n", [0, 1, 447, 448, 449, 1000])
def test_stored_ids(gpu, n):
    """Indices of the host in a device tensor, around the number one launch carries, behind other work of the default stream;
    the list may change at once, other streams and the host can wait.  Not on a stream that may be recorded."""
    from slora_hip._kernels import store_ids
    like = torch.zeros(1, dtype=torch.float16, device=gpu)
    ids = np.random.default_rng(n).integers(-2**40, 2**40, size=n).tolist()
    want = list(ids)
    torch.cuda._sleep(2_000_000)
    stored = store_ids(ids, like)
    ids[:] = [0] * n
    with torch.cuda.stream(torch.cuda.Stream()):
        assert store_ids(ids, like) is None
        stored.order()
        copy = stored.ids.clone()
    stored.wait()
    assert stored.ids.dtype == torch.long and stored.ids.cpu().tolist() == want
    torch.cuda.synchronize()
    assert copy.tolist() == want


def test_a_pool_of_another_device_than_the_current_one(gpu, monkeypatch):
    """The indices' store is a launch on the current device's default stream; for a pool of another device they are copied."""
    from slora_hip import lora_unordered_batch_infer as module
    m, new, step, t = _engine(gpu, False, hidden=512)
    stored = []
    monkeypatch.setattr(module, "store_ids", lambda ids, like, store=module.store_ids: stored.append(ids) or store(ids, like))
    want = new().req_bins.tolist()
    assert len(stored) == 1
    other = torch.cuda.current_device() + 1
    with monkeypatch.context() as patch:
        patch.setattr(torch.cuda, "current_device", lambda: other)
        eng = new()
    assert len(stored) == 1 and eng.req_bins.tolist() == want and eng.req_bins.device == eng.key_buffer[0].device


def test_prefill_steps_begun_ahead_of_the_device(gpu):
    """Many prefill steps begun while the device is busy with the first: none takes a block of pinned memory (a block whose
    copy is still to come cannot be used again, so each of them would be a new allocation)."""
    m, new, step, t = _engine(gpu, True, hidden=512)
    y = [torch.zeros_like(v) for v in t[2:]]
    _layer(new(), step, t, y)
    torch.cuda.synchronize()
    before = torch.cuda.host_memory_stats()
    torch.cuda._sleep(20_000_000)
    engines = [new() for _ in range(8)]
    for eng in engines:
        eng.begin_step(**step)
    after = torch.cuda.host_memory_stats()
    torch.cuda.synchronize()
    for key in ("num_host_alloc", "active_bytes.allocated"):
        assert after.get(key, 0) == before.get(key, 0), key
    assert all(eng.req_bins.tolist() == engines[0].req_bins.tolist() for eng in engines)


def test_steps_of_one_engine_on_two_streams(gpu):
    """A decode step on a stream that knows nothing of the busy one on which the object's prefill step was begun."""
    m, new, step, t = _engine(gpu, True)
    rows = [v[:7].clone() for v in t]
    decode = dict(step, is_prefill=False)
    want = [torch.empty_like(v) for v in rows[2:]]
    _layer(new(), decode, rows, want)
    torch.cuda.synchronize()
    eng, y = new(), [torch.zeros_like(v) for v in rows[2:]]
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(20_000_000)
        eng.begin_step(**step)
    with torch.cuda.stream(other):
        _layer(eng, decode, rows, y)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(y, want))


@pytest.mark.parametrize("is_prefill", [False, True], ids=["decode", "prefill"])
def test_steps_under_inference_mode(gpu, is_prefill):
    """An object built outside torch.inference_mode(), stepped inside: the indices are an ordinary tensor, and a decode step
    builds its plan once."""
    import slora_hip
    m, new, step, t = _engine(gpu, is_prefill)
    want, y = [torch.empty_like(v) for v in t[2:]], [torch.empty_like(v) for v in t[2:]]
    _layer(new(), step, t, want)
    eng = new()
    slora_hip.clear_plan_cache()
    slora_hip.plan_cache_stats(reset=True)
    with torch.inference_mode():
        _layer(eng, step, t, y)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(y, want)) and not eng.req_bins.is_inference()
    stats = slora_hip.plan_cache_stats()
    assert is_prefill or (stats["builds"], stats["hits"]) == (1, 1)


@pytest.mark.parametrize("is_prefill", [False, True], ids=["decode", "prefill"])
@pytest.mark.parametrize("warm_up", [False, True])
def test_replays_follow_the_adapter_indices(gpu, is_prefill, warm_up):
    """A recorded step reads req_bins: other adapters written there in place are those of the next replay."""
    m, new, step, t = _engine(gpu, is_prefill)
    eng, y = new(), [torch.zeros_like(v) for v in t[2:]]
    if warm_up:
        _layer(eng, step, t, y)
        torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        _layer(eng, step, t, y)
    for shift in (0, 1, 2):
        other, want = new(), [torch.zeros_like(v) for v in t[2:]]
        other.req_bins.copy_((other.req_bins + shift) % 3)
        eng.req_bins.copy_(other.req_bins)
        _layer(other, step, t, want)
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(y, want)), shift


@pytest.mark.parametrize("is_prefill", [False, True], ids=["decode", "prefill"])
@pytest.mark.parametrize("same_stream", [False, True])
def test_a_capture_that_waits_for_nothing(gpu, is_prefill, same_stream):
    """Recorded with capture_begin alone, which waits for no stream, by an object whose indices are still behind other work;
    replayed at once on a stream that knows nothing of that work."""
    m, new, step, t = _engine(gpu, is_prefill)
    want, y = [torch.zeros_like(v) for v in t[2:]], [torch.zeros_like(v) for v in t[2:]]
    _layer(new(), step, t, want)
    records, replays = torch.cuda.Stream(), torch.cuda.Stream()
    busy = records if same_stream else torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(20_000_000)
        eng = new()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(records):
        g.capture_begin()
        _layer(eng, step, t, y)
        g.capture_end()
    with torch.cuda.stream(replays):
        g.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(y, want))


def test_indices_looked_at_while_their_stream_is_recorded(gpu):
    """The stream that an object was built on is being recorded; the host waits for the indices all the same, and the recording
    goes on."""
    m, new, step, t = _engine(gpu, False, hidden=512)
    want = new().req_bins.tolist()
    s, g, out = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.zeros(4, device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        torch.cuda._sleep(20_000_000)
        eng = new()
        g.capture_begin(capture_error_mode="thread_local")
    bins = eng.req_bins
    with torch.cuda.stream(s):
        out.add_(1)
        g.capture_end()
    g.replay()
    torch.cuda.synchronize()
    assert bins.tolist() == want and out.tolist() == [1, 1, 1, 1]
