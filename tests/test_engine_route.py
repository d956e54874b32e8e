"""Which kernels LoraUnorderedBatchInfer picks for a prefill batch, and what it keeps of its caller's
tensors, without a GPU: the engine's per-step part runs on CPU tensors, no kernel is called."""
import pytest
import torch


class _Adapter:
    def __init__(self, lora_dir, r):
        self.lora_dir, self.r = lora_dir, r


class _Table:
    """What the engine asks of an adapter table: two adapters of rank r over a pool of pages."""

    def __init__(self, r, width=4096, dtype=torch.float16):
        self.adapter_dirs = ["a", "b"]
        self.key_buffer = [torch.zeros((8, width // 64, 64), dtype=dtype)]
        self.value_buffer = [torch.zeros((8, width // 64, 64), dtype=dtype)]
        self.a_loc = torch.arange(8 * r, dtype=torch.long) % 8
        self.a_start = torch.tensor([0, 4 * r])
        self.a_len = torch.tensor([4 * r, 4 * r])
        self.a_scaling = torch.ones(2, dtype=torch.float16)


def engine(lens, r, width=4096, dtype=torch.float16, **kw):
    from slora_hip import LoraUnorderedBatchInfer
    eng = LoraUnorderedBatchInfer(_Table(r, width, dtype), [_Adapter("ab"[i % 2], r) for i in range(len(lens))])
    b_seq_len = torch.tensor(lens, dtype=torch.int32)
    eng.begin_step(torch.cumsum(b_seq_len, 0, dtype=torch.int32) - b_seq_len, b_seq_len, True, **kw)
    return eng, b_seq_len


@pytest.mark.parametrize("known", [False, True])
def test_a_step_keeps_its_own_lengths(known):
    """Lengths advanced in place between two layers (a server preparing its next step) do not reach the
    step that is running: its rows were laid out by begin_step."""
    lens = [300, 200, 500, 600]
    eng, b_seq_len = engine(lens, 32, **({"max_b_seq_len": 600, "total_token_num": 1600} if known else {}))
    starts, kept = eng._prompts
    b_seq_len += 1
    assert kept.tolist() == lens and starts.tolist() == [0, 300, 500, 1000]
    assert eng.batch_req_bins.tolist() == [0] * 300 + [1] * 200 + [0] * 500 + [1] * 600


@pytest.mark.parametrize("is_prefill", [False, True])
@pytest.mark.parametrize("built_inside", [False, True])
def test_adapter_indices_are_of_the_mode_the_object_was_built_in(is_prefill, built_inside):
    """A step begun under torch.inference_mode() by an object built outside reads ordinary tensors: those have the version
    that the library's plan reuse goes by, inference tensors have none."""
    from slora_hip import LoraUnorderedBatchInfer
    with torch.inference_mode(built_inside):
        eng = LoraUnorderedBatchInfer(_Table(32), [_Adapter("ab"[i % 2], 32) for i in range(4)])
    b_seq_len = torch.tensor([30, 20, 50, 60], dtype=torch.int32)
    with torch.inference_mode():
        eng.begin_step(torch.cumsum(b_seq_len, 0, dtype=torch.int32) - b_seq_len, b_seq_len, is_prefill)
    assert eng.req_bins.is_inference() == built_inside and eng.req_bins.tolist() == [0, 1, 0, 1]
    assert is_prefill or eng._bins is eng.req_bins


def test_two_threads_look_at_the_adapter_indices():
    """One thread has waited for the indices between another's look at what there is to wait for and its wait."""
    from slora_hip import LoraUnorderedBatchInfer

    class Stored:
        waits = 0

        def wait(self):
            Stored.waits += 1

    class Engine(LoraUnorderedBatchInfer):
        _looks = None

        @property
        def _stored(self):
            return self._looks.pop(0) if self._looks else None

        @_stored.setter
        def _stored(self, value):
            pass

    eng = Engine(_Table(32), [_Adapter("ab"[i % 2], 32) for i in range(4)])
    eng._looks = [Stored()]  # what the second look finds: nothing
    assert eng.req_bins.tolist() == [0, 1, 0, 1] and Stored.waits == 1
    eng._looks = [Stored()]
    b_seq_len = torch.tensor([1, 1, 1, 1], dtype=torch.int32)
    eng.begin_step(torch.cumsum(b_seq_len, 0, dtype=torch.int32) - b_seq_len, b_seq_len, False)
    assert eng._bins is eng.req_bins


def segments(eng, rows, layer=0):
    x, q, k, v = (torch.zeros((rows, eng.page_elems), dtype=eng.delta_dtype) for _ in range(4))
    return eng._segments(eng.key_buffer[layer], eng.value_buffer[layer], x, q, k, v)


def test_tables_and_pools_the_segmented_kernels_do_not_take_stay_with_the_per_token_operator():
    """What the per-token operator accepts (tables of any number of dimensions, a value pool of another page
    width) it still serves; what it refuses (a pool that is not contiguous) reaches it and is refused."""
    lens = [300, 200, 500, 600]
    eng, _ = engine(lens, 32)
    assert segments(eng, 1600) is not None
    for field in ("a_loc", "a_start", "a_len"):
        eng, _ = engine(lens, 32)
        setattr(eng.infer_adapter, field, getattr(eng.infer_adapter, field).view(2, -1))
        assert segments(eng, 1600) is None, field
    eng, _ = engine(lens, 32)
    eng.value_buffer[0] = torch.zeros((8, 16, 64), dtype=torch.float16)
    assert segments(eng, 1600) is None
    eng, _ = engine(lens, 32)
    eng.key_buffer[0] = eng.key_buffer[0].view(8, 64, 64, 1)
    eng.value_buffer[0] = eng.value_buffer[0].view(8, 64, 64, 1)
    assert segments(eng, 1600) is None
    for buffers in ("key_buffer", "value_buffer"):
        eng, _ = engine(lens, 32)
        getattr(eng, buffers)[0] = torch.zeros((8, 128, 64), dtype=torch.float16)[:, :64]
        assert segments(eng, 1600) is None, buffers


@pytest.mark.parametrize("tokens", [2311, 3073, 3500, 4096, 4097])
def test_prefill_of_rank_8_has_one_route(tokens):
    """The same kernels serve a handful of rank-8 prompts on both sides of 3072 and of 4096 tokens."""
    eng, _ = engine([tokens // 4, tokens // 4, tokens // 4, tokens - 3 * (tokens // 4)], 8)
    assert segments(eng, tokens) is not None


@pytest.mark.parametrize("width,r,prompts,rows,segmented", [
    (4096, 8, 1, 1, False), (4096, 64, 1, 1, False), (8192, 8, 1, 1, False), (8192, 64, 1, 1, False),  # one short prompt
    (4096, 8, 1, 15, False), (4096, 8, 1, 16, True), (4096, 64, 1, 16, True),
    (4096, 8, 4, 255, False), (4096, 8, 4, 256, True), (4096, 8, 16, 64, True), (4096, 8, 32, 63, False),
    (4096, 8, 100, 40, False), (4096, 8, 128, 40, True), (4096, 8, 200, 39, False), (4096, 8, 256, 33, True),
    (4096, 16, 4, 63, False), (4096, 16, 4, 64, True), (4096, 16, 64, 15, False), (4096, 16, 64, 16, True),
    (4096, 64, 4, 15, False), (4096, 64, 4, 16, True), (4096, 64, 200, 2, False), (4096, 64, 256, 1, False),
    (5120, 8, 8, 3, False), (5120, 8, 8, 4, True), (8192, 64, 9, 15, False), (8192, 64, 9, 16, True), (8192, 8, 256, 4, False),
])
def test_short_prompts_stay_token_by_token(width, r, prompts, rows, segmented):
    eng, _ = engine([rows] * prompts, r, width, max_b_seq_len=rows, total_token_num=prompts * rows)
    assert not eng.use_segmented and (segments(eng, prompts * rows) is not None) == segmented


def test_the_longest_prompt_is_the_one_begin_step_saw():
    """The segmented kernels are told the longest prompt where begin_step read it from the lengths; a caller's
    max_b_seq_len decides the reference's rule only, so that a wrong one loses no rows."""
    lens = [300, 200, 500, 600]
    eng, _ = engine(lens, 32)
    assert segments(eng, 1600)[1] == 600
    for claimed in (1, 600, 9999):
        eng, _ = engine(lens, 32, max_b_seq_len=claimed, total_token_num=1600)
        assert segments(eng, 1600)[1] == 1600
