"""The four operators through the raw C ABI on the GPU, with no PyTorch in the call path: device
memory comes from the HIP runtime (libamdhip64 through ctypes), the entry points of
include/slora_hip.h are called with plain device pointers through tests/cabi_ctypes.py, and the
results are compared with the oracle at rtol 1e-2 / atol 1e-3.  This is the surface a non-Python
caller binds (the reference's own: slora/csrc/lora_ops.cc:76-126)."""
import ctypes as C

import numpy as np
import pytest

from lora_cases import make_case, make_segments
from oracle import lora_oracle as O

pytestmark = pytest.mark.gpu
RTOL, ATOL = 1e-2, 1e-3
H2D, D2H = 1, 2  # hipMemcpyHostToDevice, hipMemcpyDeviceToHost


class Hip:
    """The handful of HIP runtime calls the test needs."""

    def __init__(self):
        self.rt = C.CDLL("libamdhip64.so")
        self.rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.rt.hipFree.argtypes = [C.c_void_p]
        self.rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.rt.hipMemset.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
        n = C.c_int(0)
        if self.rt.hipGetDeviceCount(C.byref(n)) != 0 or n.value < 1:
            pytest.skip("no GPU")
        assert self.rt.hipSetDevice(0) == 0
        self.owned = []

    def upload(self, a: np.ndarray) -> int:
        a = np.ascontiguousarray(a)
        p = C.c_void_p()
        assert self.rt.hipMalloc(C.byref(p), max(a.nbytes, 16)) == 0
        self.owned.append(p)
        assert self.rt.hipMemcpy(p, a.ctypes.data_as(C.c_void_p), a.nbytes, H2D) == 0
        return p.value

    def download(self, ptr: int, shape, dtype) -> np.ndarray:
        out = np.empty(shape, dtype=dtype)
        assert self.rt.hipDeviceSynchronize() == 0
        assert self.rt.hipMemcpy(out.ctypes.data_as(C.c_void_p), C.c_void_p(ptr), out.nbytes, D2H) == 0
        return out

    def close(self):
        self.rt.hipDeviceSynchronize()
        for p in self.owned:
            self.rt.hipFree(p)
        self.owned = []


@pytest.fixture(scope="module")
def hip():
    h = Hip()
    yield h
    h.close()


def to_bits(a, dtype):
    """float32 values representable in `dtype` -> the 16-bit patterns the kernels read"""
    a = np.ascontiguousarray(a, dtype=np.float32)
    if dtype == "f16":
        return a.astype(np.float16).view(np.uint16)
    return (a.view(np.uint32) >> 16).astype(np.uint16)


def from_bits(u, dtype):
    if dtype == "f16":
        return u.view(np.float16).astype(np.float32)
    return (u.astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_decode_operators_through_the_c_abi(hip, dtype):
    import cabi_ctypes as A
    lib = A.load_library()
    ranks = [64, 32, 16, 8, 8]
    H, batch, R = 1024, 37, 64
    c = make_case(21, H, ranks, batch, dtype=dtype, zipf_alpha=1.0)
    dt = A.DTYPE_F16 if dtype == "f16" else A.DTYPE_BF16
    key, val = hip.upload(to_bits(c.key, dtype)), hip.upload(to_bits(c.value, dtype))
    tables = A.SloraTables(hip.upload(c.a_start.astype(np.int64)), hip.upload(c.a_len.astype(np.int64)),
                           hip.upload(c.a_loc.astype(np.int64)), len(ranks), int(c.a_loc.size))
    bins = hip.upload(c.bins.astype(np.int64))
    scales = hip.upload(c.scales.astype(np.float16))           # the table is fp16 whatever the data type
    x = hip.upload(to_bits(c.x, dtype))
    for p in range(4):
        delta = hip.upload(np.zeros((batch, R), np.uint16))
        print(f"c-abi decode {dtype} projection {p}", flush=True)
        rc = lib.slora_bgmv_shrink(delta, x, key, C.byref(tables), bins, batch, H, R, c.page_elems, c.n_pages, p, dt,
                                   None)
        assert rc == A.OK, A.strerror(rc)
        d_gpu = from_bits(hip.download(delta, (batch, R), np.uint16), dtype)
        d_ref = O.ref_bgmv_shrink(np.zeros((batch, R), np.float32), c.x, c.key, c.a_start, c.a_len, c.a_loc, c.bins, p,
                                  dtype)
        np.testing.assert_allclose(d_gpu, d_ref, rtol=RTOL, atol=ATOL)
        y0 = O.round_to(np.random.default_rng(p).standard_normal((batch, H)).astype(np.float32) * 0.25, dtype)
        y = hip.upload(to_bits(y0, dtype))
        rc = lib.slora_bgmv_expand(y, delta, val, C.byref(tables), bins, scales, A.DTYPE_F16, batch, R, H,
                                   c.page_elems, c.n_pages, p, dt, None)
        assert rc == A.OK, A.strerror(rc)
        y_gpu = from_bits(hip.download(y, (batch, H), np.uint16), dtype)
        y_ref = O.ref_bgmv_expand(y0, d_gpu, c.value, c.a_start, c.a_len, c.a_loc, c.bins, p, c.scales, dtype)
        # y0 + update rounds once at the magnitude of the operands, here as in the reference
        step = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(y0), np.abs(y_ref - y0)) + 1e-30)) - (10 if dtype == "f16" else 7))
        assert np.all(np.abs(y_gpu - y_ref) <= ATOL + RTOL * np.abs(y_ref) + step)


@pytest.mark.parametrize("R", [12, 16])
def test_shrink_and_expand_in_one_call_without_outputs(hip, R):
    """slora_bgmv_lora_planned over outputs of no columns is the shrink alone, of any delta width; with outputs a width that is no
    multiple of 8 is refused and nothing is written."""
    import cabi_ctypes as A
    lib = A.load_library()
    H, batch = 512, 7
    c = make_case(24, H, [16, 8], batch, dtype="f16")
    key, val = hip.upload(to_bits(c.key, "f16")), hip.upload(to_bits(c.value, "f16"))
    tables = A.SloraTables(hip.upload(c.a_start.astype(np.int64)), hip.upload(c.a_len.astype(np.int64)),
                           hip.upload(c.a_loc.astype(np.int64)), 2, int(c.a_loc.size))
    bins, x = hip.upload(c.bins.astype(np.int64)), hip.upload(to_bits(c.x, "f16"))
    scales = hip.upload(c.scales.astype(np.float16))
    nbytes = lib.slora_bgmv_plan_bytes(batch, R)
    plan = hip.upload(np.zeros(nbytes, np.uint8))
    assert lib.slora_bgmv_plan_build(plan, nbytes, C.byref(tables), bins, batch, R, c.n_pages, None) == A.OK
    y0 = np.full((batch, H), 0x3c00, np.uint16)
    want = O.ref_bgmv_shrink(np.zeros((batch, R), np.float32), c.x, c.key, c.a_start, c.a_len, c.a_loc, c.bins, 1, "f16")
    for h_out in (0, H):
        delta, y = hip.upload(np.zeros((batch, R), np.uint16)), hip.upload(y0)
        print(f"c-abi lora R {R} h_out {h_out}", flush=True)
        rc = lib.slora_bgmv_lora_planned(plan, R, 0, 1, y, None, None, delta, None, None, x, key, val, C.byref(tables), bins,
                                         scales, A.DTYPE_F16, batch, H, R, h_out, 0, 0, c.page_elems, c.n_pages, 1, A.DTYPE_F16,
                                         None)
        refused = h_out > 0 and R % 8 != 0
        assert rc == (A.ERR_UNSUPPORTED if refused else A.OK), A.strerror(rc)
        d_gpu = from_bits(hip.download(delta, (batch, R), np.uint16), "f16")
        np.testing.assert_allclose(d_gpu, np.zeros_like(want) if refused else want, rtol=RTOL, atol=ATOL)
        assert np.array_equal(hip.download(y, (batch, H), np.uint16), y0) == (h_out == 0 or refused)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_prefill_operators_through_the_c_abi(hip, dtype):
    import cabi_ctypes as A
    lib = A.load_library()
    ranks = [64, 16, 8, 32]
    H, R = 512, 64
    start, lens, ids = make_segments(4, 9, 1, 90, len(ranks))
    T = int(lens.sum())
    c = make_case(22, H, ranks, T, dtype=dtype, bins=np.repeat(ids, lens))
    dt = A.DTYPE_F16 if dtype == "f16" else A.DTYPE_BF16
    key, val = hip.upload(to_bits(c.key, dtype)), hip.upload(to_bits(c.value, dtype))
    tables = A.SloraTables(hip.upload(c.a_start.astype(np.int64)), hip.upload(c.a_len.astype(np.int64)),
                           hip.upload(c.a_loc.astype(np.int64)), len(ranks), int(c.a_loc.size))
    st, ln, rq = hip.upload(start.astype(np.int32)), hip.upload(lens.astype(np.int32)), hip.upload(ids.astype(np.int64))
    scales = hip.upload(c.scales.astype(np.float16))
    x = hip.upload(to_bits(c.x, dtype))
    for p in range(4):
        o = hip.upload(np.full((T, R), 0x3c00, np.uint16))      # the operator writes every column up to max_rank
        print(f"c-abi prefill {dtype} projection {p}", flush=True)
        rc = lib.slora_sgmm_shrink(o, x, key, C.byref(tables), st, ln, rq, len(lens), int(lens.max()), T, H, R, H, H,
                                   R, c.n_pages, p, dt, None)
        assert rc == A.OK, A.strerror(rc)
        o_gpu = from_bits(hip.download(o, (T, R), np.uint16), dtype)
        o_ref = O.ref_prefill_shrink(np.ones((T, R), np.float32), c.x, c.key, c.a_loc, c.a_start, c.a_len, start, lens,
                                     ids, p, R, dtype)
        np.testing.assert_allclose(o_gpu, o_ref, rtol=RTOL, atol=ATOL)
        y = hip.upload(np.zeros((T, H), np.uint16))
        rc = lib.slora_sgmm_expand(y, o, val, C.byref(tables), scales, A.DTYPE_F16, st, ln, rq, len(lens),
                                   int(lens.max()), T, H, 0, R, R, H, H, c.n_pages, p, dt, None)
        assert rc == A.OK, A.strerror(rc)
        y_gpu = from_bits(hip.download(y, (T, H), np.uint16), dtype)
        y_ref = O.ref_prefill_expand(np.zeros((T, H), np.float32), o_gpu, c.value, c.scales, c.a_loc, c.a_start,
                                     c.a_len, start, lens, ids, p, R, dtype)
        np.testing.assert_allclose(y_gpu, y_ref, rtol=RTOL, atol=ATOL)


def test_a_plan_of_another_rank_cap_does_nothing_and_says_so(hip):
    """A planned launch that names another rank cap or batch than the plan was built for leaves its
    output alone and sets bit 0 of the plan's status word; the launch the plan was built for works
    and the word is 0 after a build.  The buffer is sized for the largest launch made with it: a
    launch reads its item records before it has seen the header."""
    import cabi_ctypes as A
    lib = A.load_library()
    ranks = [16, 8, 32]
    H, batch, R = 512, 9, 64
    c = make_case(23, H, ranks, batch, dtype="f16")
    key = hip.upload(to_bits(c.key, "f16"))
    tables = A.SloraTables(hip.upload(c.a_start.astype(np.int64)), hip.upload(c.a_len.astype(np.int64)),
                           hip.upload(c.a_loc.astype(np.int64)), len(ranks), int(c.a_loc.size))
    bins = hip.upload(c.bins.astype(np.int64))
    x = hip.upload(to_bits(c.x, "f16"))
    nbytes = lib.slora_bgmv_plan_bytes(batch, R)
    assert nbytes >= lib.slora_bgmv_plan_bytes(batch, 32) and nbytes >= lib.slora_bgmv_plan_bytes(batch - 1, R)
    plan = hip.upload(np.zeros(nbytes // 4, np.int32))
    status = C.c_int(-1)

    def shrink(n_tokens, rank_cap, delta):
        rc = lib.slora_bgmv_shrink_planned(plan, rank_cap, 0, 1, delta, None, None, x, key, C.byref(tables), bins,
                                           n_tokens, H, R, c.page_elems, c.n_pages, 0, A.DTYPE_F16, None)
        assert rc == A.OK, A.strerror(rc)

    for what, n_tokens, rank_cap in (("rank cap", batch, 32), ("batch", batch - 1, R)):
        assert lib.slora_bgmv_plan_build(plan, nbytes, C.byref(tables), bins, batch, R, c.n_pages, None) == A.OK
        assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 0
        delta = hip.upload(np.full((batch, R), 0x3c00, np.uint16))
        print(f"c-abi planned shrink that names another {what}", flush=True)
        shrink(n_tokens, rank_cap, delta)
        assert np.all(hip.download(delta, (batch, R), np.uint16) == 0x3c00)
        assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 1
    # the launch the plan was built for
    assert lib.slora_bgmv_plan_build(plan, nbytes, C.byref(tables), bins, batch, R, c.n_pages, None) == A.OK
    delta = hip.upload(np.zeros((batch, R), np.uint16))
    print("c-abi planned shrink with its own plan", flush=True)
    shrink(batch, R, delta)
    d_gpu = from_bits(hip.download(delta, (batch, R), np.uint16), "f16")
    d_ref = O.ref_bgmv_shrink(np.zeros((batch, R), np.float32), c.x, c.key, c.a_start, c.a_len, c.a_loc, c.bins, 0, "f16")
    np.testing.assert_allclose(d_gpu, d_ref, rtol=RTOL, atol=ATOL)
    assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 0


def test_a_prefill_plan_of_another_batch_does_nothing_and_says_so(hip):
    """slora_sgmm_shrink_planned with the plan of another batch shape leaves its output alone and sets
    the plan's status word; with its own plan it gives the oracle's result and the word is 0."""
    import cabi_ctypes as A
    lib = A.load_library()
    ranks = [64, 16, 8, 32]
    H, R, dtype = 512, 64, "f16"
    start, lens, ids = make_segments(5, 6, 20, 90, len(ranks))
    T = int(lens.sum())
    c = make_case(24, H, ranks, T, dtype=dtype, bins=np.repeat(ids, lens))
    key = hip.upload(to_bits(c.key, dtype))
    tables = A.SloraTables(hip.upload(c.a_start.astype(np.int64)), hip.upload(c.a_len.astype(np.int64)),
                           hip.upload(c.a_loc.astype(np.int64)), len(ranks), int(c.a_loc.size))
    st, ln, rq = hip.upload(start.astype(np.int32)), hip.upload(lens.astype(np.int32)), hip.upload(ids.astype(np.int64))
    x = hip.upload(to_bits(c.x, dtype))
    nbytes = lib.slora_sgmm_plan_bytes()
    plan = hip.upload(np.zeros(nbytes // 4, np.int32))
    usable, status = C.c_int(0), C.c_int(-1)

    def build(n_req, max_len, n_tokens):
        rc = lib.slora_sgmm_plan_build(plan, nbytes, C.byref(tables), st, ln, rq, n_req, max_len, n_tokens, R,
                                       C.byref(usable), None)
        assert rc == A.OK and usable.value == 1

    def shrink(o):
        return lib.slora_sgmm_shrink_planned(plan, o, x, key, C.byref(tables), st, ln, rq, len(lens), int(lens.max()), T, H,
                                             R, H, H, R, c.n_pages, 0, A.DTYPE_F16, None)

    # a plan for the first request alone: another number of row parts than the launch below has
    build(1, int(lens[0]), int(lens[0]))
    assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 0
    o = hip.upload(np.full((T, R), 0x3c00, np.uint16))
    print("c-abi planned prefill shrink with the plan of another batch", flush=True)
    assert shrink(o) == A.OK
    assert np.all(hip.download(o, (T, R), np.uint16) == 0x3c00)
    assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 1
    build(len(lens), int(lens.max()), T)
    assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 0
    print("c-abi planned prefill shrink with its own plan", flush=True)
    assert shrink(o) == A.OK
    o_gpu = from_bits(hip.download(o, (T, R), np.uint16), dtype)
    o_ref = O.ref_prefill_shrink(np.ones((T, R), np.float32), c.x, c.key, c.a_loc, c.a_start, c.a_len, start, lens, ids,
                                 0, R, dtype)
    np.testing.assert_allclose(o_gpu, o_ref, rtol=RTOL, atol=ATOL)
    assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 0


def _sgmm_case(hip, seed, H, ranks, lens, dtype="f16"):
    """Device copies of a prefill case: what the segmented entry points take."""
    import cabi_ctypes as A
    lens = np.asarray(lens, np.int32)
    ids = np.arange(len(lens)) % len(ranks)
    c = make_case(seed, H, ranks, int(lens.sum()), dtype=dtype, bins=np.repeat(ids, lens))
    c.start, c.lens, c.ids = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32), lens, ids.astype(np.int64)
    c.d_key, c.d_val = hip.upload(to_bits(c.key, dtype)), hip.upload(to_bits(c.value, dtype))
    c.tables = A.SloraTables(hip.upload(c.a_start.astype(np.int64)), hip.upload(c.a_len.astype(np.int64)),
                             hip.upload(c.a_loc.astype(np.int64)), len(ranks), int(c.a_loc.size))
    c.seg = (hip.upload(c.start), hip.upload(lens), hip.upload(c.ids))
    c.scal, c.d_x = hip.upload(c.scales.astype(np.float16)), hip.upload(to_bits(c.x, dtype))
    return c


def test_an_expand_does_not_take_what_an_older_plan_left_in_the_buffer(hip):
    """A plan buffer that is built for a small batch and then for a launch that describes no spans: an
    expand of the small batch's shape leaves its output alone and sets the status word, also where the
    two launches have as many row parts."""
    import cabi_ctypes as A
    lib = A.load_library()
    H, R = 512, 32
    c = _sgmm_case(hip, 25, H, [32, 16], [250] * 4)
    T, n = 1000, 4
    nbytes = lib.slora_sgmm_plan_bytes()
    plan = hip.upload(np.zeros(nbytes // 4, np.int32))
    usable, status = C.c_int(0), C.c_int(-1)
    delta = hip.upload(to_bits(O.round_to(np.random.default_rng(3).standard_normal((T, R)).astype(np.float32), "f16"), "f16"))
    y = hip.upload(np.full((T, H), 0x3c00, np.uint16))
    n_parts = []
    for max_rank in (R, 256):   # 1000 tokens of rank 32 are a small batch, of rank 256 they are not
        rc = lib.slora_sgmm_plan_build(plan, nbytes, C.byref(c.tables), *c.seg, n, 250, T, max_rank, C.byref(usable), None)
        assert rc == A.OK and usable.value == 1
        n_parts.append(int(hip.download(plan, (16,), np.int32)[1]))
    assert n_parts[0] == n_parts[1]   # the case this test is about
    print("c-abi expand with a buffer that held a plan of its shape before", flush=True)
    rc = lib.slora_sgmm_expand_planned(plan, 1, y, None, None, delta, None, None, c.d_val, C.byref(c.tables), c.scal, A.DTYPE_F16,
                                       *c.seg, n, 250, T, H, 0, H, R, R, H, H, 0, c.n_pages, 0, A.DTYPE_F16, None)
    assert rc == A.OK, A.strerror(rc)
    assert np.all(hip.download(y, (T, H), np.uint16) == 0x3c00)
    assert lib.slora_plan_status(plan, C.byref(status), None) == A.OK and status.value == 1


class _Segmented:
    """The segmented entry points on one case, with a plan and without."""

    def __init__(self, hip, c, R, dtype, max_len=None):
        import cabi_ctypes as A
        self.A, self.lib, self.hip, self.c, self.R, self.dtype = A, A.load_library(), hip, c, R, dtype
        self.dt = A.DTYPE_F16 if dtype == "f16" else A.DTYPE_BF16
        self.T, self.H, self.n = c.batch, c.hidden, len(c.lens)
        self.max_len = int(c.lens.max()) if max_len is None else max_len
        self.nbytes = self.lib.slora_sgmm_plan_bytes()
        self.plan = hip.upload(np.zeros(self.nbytes // 4, np.int32))

    def build(self):
        """Builds the plan and returns its header; word 1: row parts, word 2: -16 for a small batch, word 8: spans."""
        usable = C.c_int(0)
        rc = self.lib.slora_sgmm_plan_build(self.plan, self.nbytes, C.byref(self.c.tables), *self.c.seg, self.n, self.max_len,
                                            self.T, self.R, C.byref(usable), None)
        assert rc == self.A.OK and usable.value == 1
        return self.hip.download(self.plan, (16,), np.int32)

    def status(self):
        status = C.c_int(-1)
        assert self.lib.slora_plan_status(self.plan, C.byref(status), None) == self.A.OK
        return status.value

    def shrink(self, p, planned):
        o = self.hip.upload(np.full((self.T, self.R), 0x3c00, np.uint16))
        f = self.lib.slora_sgmm_shrink_planned if planned else self.lib.slora_sgmm_shrink
        rc = f(*((self.plan,) if planned else ()), o, self.c.d_x, self.c.d_key, C.byref(self.c.tables), *self.c.seg, self.n,
               self.max_len, self.T, self.H, self.R, self.H, self.H, self.R, self.c.n_pages, p, self.dt, None)
        assert rc == self.A.OK, self.A.strerror(rc)
        return self.hip.download(o, (self.T, self.R), np.uint16)

    def shrink_qkv(self, planned):
        o = [self.hip.upload(np.full((self.T, self.R), 0x3c00, np.uint16)) for _ in range(3)]
        rc = self.lib.slora_sgmm_shrink_qkv(self.plan if planned else None, *o, self.c.d_x, self.c.d_key, C.byref(self.c.tables),
                                            *self.c.seg, self.n, self.max_len, self.T, self.H, self.R, self.H, self.H, self.R,
                                            self.c.n_pages, self.dt, None)
        assert rc == self.A.OK, self.A.strerror(rc)
        return [self.hip.download(q, (self.T, self.R), np.uint16) for q in o]

    def expand(self, y0, d, planned, p=None):
        """Projection p, or q, k and v in one launch; y0 and d: bit patterns."""
        y = [self.hip.upload(y0) for _ in range(3 if p is None else 1)]
        x = [self.hip.upload(q) for q in d]
        lib, c, H, R = self.lib, self.c, self.H, self.R
        tail = (c.d_val, C.byref(c.tables), c.scal, self.A.DTYPE_F16, *c.seg, self.n, self.max_len, self.T)
        if planned:
            pad = (None,) * (3 - len(y))
            rc = lib.slora_sgmm_expand_planned(self.plan, len(y), *y, *pad, *x, *pad, *tail, H, H, H, R, R, H, H, H, c.n_pages,
                                               p or 0, self.dt, None)
        elif p is None:
            rc = lib.slora_sgmm_expand_qkv(*y, *x, *tail, H, H, H, R, R, H, H, H, c.n_pages, self.dt, None)
        else:
            rc = lib.slora_sgmm_expand(*y, *x, *tail, H, H, R, R, H, H, c.n_pages, p, self.dt, None)
        assert rc == self.A.OK, self.A.strerror(rc)
        return [self.hip.download(q, (self.T, H), np.uint16) for q in y]

    def ref_shrink(self, p):
        c = self.c
        return O.ref_prefill_shrink(np.ones((self.T, self.R), np.float32), c.x, c.key, c.a_loc, c.a_start, c.a_len, c.start, c.lens,
                                    c.ids, p, self.R, self.dtype)

    def ref_expand(self, y0, d, p):
        c = self.c
        return O.ref_prefill_expand(from_bits(y0, self.dtype), from_bits(d, self.dtype), c.value, c.scales, c.a_loc, c.a_start,
                                    c.a_len, c.start, c.lens, c.ids, p, self.R, self.dtype)


def _random_bits(seed, shape, dtype):
    return to_bits(O.round_to(np.random.default_rng(seed).standard_normal(shape).astype(np.float32), dtype), dtype)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("H,ranks,lens,one,three", [
    # `one`, `three`: tiles of 16 rank columns a workgroup of the single and of the q/k/v shrink takes
    (4096, [64, 8], [1, 15, 16, 17, 33], 1, 1),           # rows at the edges of a part
    (5120, [32, 16], [256] * 4, 1, 2),                    # chunks of 320 elements, two per wavefront; two tiles
    (5120, [64, 40], [256] * 5, 2, 4),                    # the same with four tiles; ranks that end inside one
    (2560, [48, 16, 8], [150, 17, 200, 33, 129, 1], 1, 2),   # one chunk of 320 per wavefront, the third tile alone in its group
    (4096, [64, 24], [250] * 5, 2, 4),                    # chunks of 512; rows that end inside a part
    (576, [64, 8], [256] * 5, 2, 4),                      # a last chunk of 64 elements; wavefronts with nothing to do
    (8192, [128, 32], [300, 300], 2, 4),                  # two chunks of 512 per wavefront; four groups of 32 columns
    (512, [64, 32, 16, 8], [65] * 30, 4, 4),              # more workgroups than compute units
    (512, [16, 8], [3] * 256, 1, 1),                      # as many requests as a plan describes
])
def test_small_prefill_batches_through_the_c_abi(hip, dtype, H, ranks, lens, one, three):
    """Every shape of the split-K shrink, planned and not, one projection and three, and the expand from the
    plan's spans: bit for bit each other, and the oracle's results."""
    R = max(ranks)
    c = _sgmm_case(hip, H + R, H, ranks, lens, dtype)
    g = _Segmented(hip, c, R, dtype)
    head = g.build()
    assert head[2] == -16                                    # a small batch
    tiles, parts = -(-R // 16), int(head[1])

    def columns(nproj):   # as few tiles per workgroup as keep the launch within 256 of them, or four
        return next((nt for nt in (1, 2) if nt >= tiles or parts * nproj * -(-tiles // nt) <= 256), 4)

    assert (columns(1), columns(3)) == (one, three)
    print(f"c-abi small prefill {dtype} hidden {H} ranks {ranks} {len(lens)} requests", flush=True)
    d = g.shrink_qkv(True)
    for p in range(3):
        np.testing.assert_allclose(from_bits(d[p], dtype), g.ref_shrink(p), rtol=RTOL, atol=ATOL)
        assert np.array_equal(g.shrink(p, True), d[p]), p
    assert np.array_equal(g.shrink(1, False), d[1])
    assert all(np.array_equal(a, b) for a, b in zip(g.shrink_qkv(False), d))
    y0 = _random_bits(7, (c.batch, H), dtype)
    y = g.expand(y0, d, True)
    assert all(np.array_equal(a, b) for a, b in zip(g.expand(y0, d, False), y))
    assert np.array_equal(g.expand(y0, d[1:2], True, 1)[0], y[1]) and np.array_equal(g.expand(y0, d[1:2], False, 1)[0], y[1])
    np.testing.assert_allclose(from_bits(y[2], dtype), g.ref_expand(y0, d[2], 2), rtol=RTOL, atol=ATOL)
    assert g.status() == 0


@pytest.mark.parametrize("lens,start,max_len", [
    ([40] * 8, [0] * 8, None),         # requests that overlap in the batch: parts of 32 rows
    ([40] * 16, [0] * 16, None),       # ... of 64
    ([60] * 8, None, 10),              # lengths beyond max_input_len, clipped at a whole tile: one part of 60 rows each
])
def test_split_shrink_parts_of_more_than_16_rows(hip, lens, start, max_len):
    H, R = 1024, 32
    ids_one = start is not None        # overlapping requests name one adapter: all write the same values
    c = _sgmm_case(hip, 26, H, [R] if ids_one else [R, 16], lens)
    if ids_one:                        # the batch is the rows they share
        c.batch, c.start = lens[0], np.asarray(start, np.int32)
        c.x = c.x[: c.batch]
        c.seg = (hip.upload(c.start), *c.seg[1:])
    g = _Segmented(hip, c, R, "f16", max_len)
    head = g.build()
    assert head[2] == -16 and int(head[1]) < sum(-(-n // 16) for n in lens)   # fewer parts than pieces of 16 rows
    print(f"c-abi split shrink {lens[:2]} x {len(lens)} max_len {max_len}", flush=True)
    d = g.shrink(2, True)
    np.testing.assert_allclose(from_bits(d, "f16"), g.ref_shrink(2), rtol=RTOL, atol=ATOL)
    assert np.array_equal(g.shrink(2, False), d) and np.array_equal(g.shrink_qkv(True)[2], d)
    assert g.status() == 0


def test_expand_spans_of_more_than_32_rows(hip):
    """Requests without an adapter's rank lie over the same rows: they take spans but touch nothing, and the one
    request that does gets a span of all its rows."""
    H, R, T, n = 1024, 16, 100, 8
    c = _sgmm_case(hip, 27, H, [R, 0], [T] * n)
    c.batch, c.start, c.ids = T, np.zeros(n, np.int32), np.array([1, 1, 0, 1, 1, 1, 1, 1], np.int64)
    c.seg = (hip.upload(c.start), c.seg[1], hip.upload(c.ids))
    g = _Segmented(hip, c, R, "f16")
    head = g.build()
    assert head[2] == -16 and int(head[8]) < n * 4           # fewer spans than pieces of 32 rows
    y0, d = _random_bits(8, (T, H), "f16"), _random_bits(9, (T, R), "f16")
    print("c-abi expand spans of more than 32 rows", flush=True)
    y = g.expand(y0, [d], True, 3)[0]
    np.testing.assert_allclose(from_bits(y, "f16"), g.ref_expand(y0, d, 3), rtol=RTOL, atol=ATOL)
    assert np.array_equal(g.expand(y0, [d], False, 3)[0], y) and g.status() == 0


def test_expand_with_the_plan_of_another_batch_does_nothing_and_says_so(hip):
    """slora_sgmm_expand_planned with the plan of another batch shape leaves its output alone and sets the
    status word; a batch too large for spans leaves the plan alone."""
    H, R = 512, 16
    other = _Segmented(hip, _sgmm_case(hip, 28, H, [R, 8], [30, 41]), R, "f16")
    g = _Segmented(hip, _sgmm_case(hip, 29, H, [R, 8], [30, 41, 50]), R, "f16")
    other.build()
    g.plan = other.plan
    y0, d = _random_bits(10, (g.T, H), "f16"), _random_bits(11, (g.T, R), "f16")
    print("c-abi expand with the plan of another batch", flush=True)
    assert g.status() == 0
    assert np.array_equal(g.expand(y0, [d], True, 0)[0], y0) and g.status() == 1
    assert all(np.array_equal(y, y0) for y in g.expand(y0, [d] * 3, True)) and g.status() == 1
    g.build()
    assert g.status() == 0
    assert np.array_equal(g.expand(y0, [d], True, 0)[0], g.expand(y0, [d], False, 0)[0]) and g.status() == 0
    big = _Segmented(hip, _sgmm_case(hip, 30, H, [R, 8], [1200, 1300]), R, "f16")   # 2500 tokens x 16 > 32768
    big.plan = other.plan
    y0, d = _random_bits(12, (big.T, H), "f16"), _random_bits(13, (big.T, R), "f16")
    assert np.array_equal(big.expand(y0, [d], True, 0)[0], big.expand(y0, [d], False, 0)[0]) and big.status() == 0


@pytest.mark.parametrize("R,lens,small", [
    (64, [84] * 32, False), (64, [2736], False), (64, [2688], True), (64, [210] * 10, True),   # two rounds of q/k/v workgroups
    (40, [341] * 8, False), (32, [84] * 32, True), (72, [62] * 33, True), (72, [2064], False),
])
def test_the_plan_says_which_batches_are_small(hip, R, lens, small):
    c = _sgmm_case(hip, 31, 64, [R], lens)
    assert (_Segmented(hip, c, R, "f16").build()[2] == -16) == small


@pytest.mark.parametrize("H,R,T,nproj,spans", [
    (512, 8, 2048, 1, True), (512, 8, 2064, 1, False), (1024, 8, 2064, 3, False),   # many tokens, few outputs
    (2048, 8, 2064, 3, True), (4096, 8, 2064, 1, True),
    (8192, 64, 320, 3, True), (8192, 64, 352, 3, False), (8192, 64, 512, 1, True),  # wide q, k and v
])
def test_which_expands_read_the_plans_spans(hip, H, R, T, nproj, spans):
    """An expand that reads spans leaves its output alone when the plan is another batch's; one that looks its
    rows up itself does not look at the plan."""
    g = _Segmented(hip, _sgmm_case(hip, 32, H, [R], [T // 2, T - T // 2]), R, "f16")
    other = _Segmented(hip, _sgmm_case(hip, 33, 64, [R], [30, 41]), R, "f16")
    assert other.build()[2] == -16
    g.plan = other.plan
    y0, d = _random_bits(14, (T, H), "f16"), _random_bits(15, (T, R), "f16")
    print(f"c-abi expand of {T} tokens of rank {R} at hidden {H}", flush=True)
    y = g.expand(y0, [d] * nproj, True, None if nproj == 3 else 0)
    assert all(np.array_equal(q, y0) == spans for q in y) and g.status() == int(spans)
