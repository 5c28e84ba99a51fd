"""Product ops around the prefill GEMM's plans: which one runs (the split over K, whole tiles, the small
GEMMs) by the workspace that is asked for or written, with the workspace of the reported size, less, and
none (the no-allocation entry point); the small shapes on which all of them meet, in the exact-integer
mode; Q2_K's rounded scales, group sums and mins beyond fp16. Each plan and tile width of the prefill GEMM:
test_gpu_prefill_plans.py. Needs an MI355X.
"""

import ctypes

import numpy as np
import pytest
import torch

import gguf_oracle as o
from _gpu import C, dev, exact_ref, exact_weights, exact_x, graph_replays_equal, w_rand, x_rand

pytestmark = pytest.mark.gpu

PACKED = (o.IQ3_S, o.IQ3_XXS)
TYPES = [o.IQ3_S, o.IQ3_XXS, o.Q4_K, o.Q6_K, o.IQ4_XS, o.Q2_K, o.IQ2_XXS, o.IQ2_XS, o.IQ2_S]
MUL_MAT_Q, PACKED_TILED = 1, 7


@pytest.fixture(scope="module")
def lib():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from vllm_gguf_plugin import _capi, ops  # noqa: F401

    return _capi.load()


def _weight(qt, raw):
    from vllm_gguf_plugin.quantization import iq3_pack

    return iq3_pack.pack(dev(raw), qt) if qt in PACKED else dev(raw)


def _torch_op(qt, w, x, rows):
    op = "lcpp_mul_mat_iq3_packed" if qt in PACKED else "lcpp_mul_mat_q"
    return getattr(C(), op)(w, x, qt, rows)


def _capi_op(lib, qt, w, x, rows, entry="workspace"):
    from vllm_gguf_plugin import _capi

    op, (n, k) = (PACKED_TILED if qt in PACKED else MUL_MAT_Q), x.shape
    y = torch.full((n, rows), float("nan"), dtype=x.dtype, device="cuda")
    nb = lib.gguf_op_workspace_bytes(op, qt, rows, k, n, 0)
    stream = torch.cuda.current_stream().cuda_stream
    args = (op, _capi.ref(_capi.view(w)), _capi.ref(_capi.view(x)), qt, rows, None, y.data_ptr(), y.numel() * y.element_size())
    if entry == "noalloc":
        rc = lib.gguf_mul_mat_noalloc(*args, stream)
    else:
        ws = torch.full((max(nb, 1),), 0xFF, dtype=torch.uint8, device="cuda")
        rc = lib.gguf_mul_mat(*args, ws.data_ptr(), nb, stream)
    assert rc == 0, _capi.error(lib)
    torch.cuda.synchronize()
    return y, nb


# rows (packed types: the next multiple of 16), K, activation rows: small weights, of which the small GEMMs
# run most
SHAPES = [(270, 4608, 257), (270, 4608, 300), (16, 1024, 513), (1030, 512, 259), (130, 2560, 1025)]


@pytest.mark.parametrize("rows,k,n", SHAPES)
@pytest.mark.parametrize("qt", TYPES, ids=lambda t: o.TYPE_NAMES[t])
def test_split_and_unsplit_exact(lib, qt, rows, k, n):
    rows = -(-rows // 16) * 16 if qt in PACKED else rows
    raw = exact_weights(qt, rows, k, seed=rows + n)
    x = exact_x(n, k, seed=n, dtype=torch.float32)
    ref = exact_ref(raw, qt, x, form="mmq")
    w, xg = _weight(qt, raw), x.cuda()
    assert np.array_equal(_torch_op(qt, w, xg, rows).cpu().numpy(), ref)
    y, nb = _capi_op(lib, qt, w, xg, rows)
    assert nb == -(-n // 16) * (k // 256) * (8192 + (2560 if qt == o.Q2_K else 1024))  # the prefill GEMM's layout
    assert np.array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("n", [1, 8, 16, 17, 63, 64, 65, 128, 129])
def test_q2k_every_row_count(n):
    """Q2_K's product op at every row count: the prefill GEMM from 17 rows at this K (64-column tiles, four
    row parts), the per-slice GEMM below; one row on the prefill GEMM: test_q2k_scales_rounded_as_the_model."""
    raw = exact_weights(o.Q2_K, 270, 2560, seed=n)
    x = exact_x(n, 2560, seed=n + 1, dtype=torch.float32)
    y = _torch_op(o.Q2_K, dev(raw), x.cuda(), 270).cpu().numpy()
    assert np.array_equal(y, exact_ref(raw, o.Q2_K, x, form="mmq"))


@pytest.mark.parametrize("qt", [o.Q4_K, o.IQ4_XS, o.Q6_K, o.IQ2_S], ids=lambda t: o.TYPE_NAMES[t])
@pytest.mark.parametrize("n", [33, 49, 64])
def test_rows_33_to_64(qt, n):
    """Weights of 24M values or more at 33..64 rows: the torch ops prefer the prefill GEMM there (K split;
    asserted in test_gpu_prefill_plans.py). fp32 X against the q81 model on sampled rows."""
    rows, k = 5120, 5120
    raw = w_rand(qt, rows, k, seed=n)
    x = x_rand(n, k, seed=n + 7)
    rs = np.unique(np.random.default_rng(n).choice(rows, 48, replace=False))
    y = _torch_op(qt, dev(raw), x.cuda(), rows).cpu().numpy()[:, rs]
    assert o.rel_l2(y, o.q81_model(raw[rs], qt, x, layout="mmq")) <= 1e-3


def test_split_graph_replays():
    """Replays of a captured product, with eager work between, equal the eager result bit for bit (the
    prefill GEMM's split plan: test_split_replays)."""
    raw = w_rand(o.Q4_K, 1030, 2560, seed=1)
    w, x = dev(raw), x_rand(300, 2560, seed=2, dtype=torch.bfloat16).cuda()
    eager = _torch_op(o.Q4_K, w, x, 1030)
    assert torch.equal(eager, _torch_op(o.Q4_K, w, x, 1030))
    graph_replays_equal(lambda: torch.ops._C_gguf.lcpp_mul_mat_q(w, x, o.Q4_K, 1030), eager)


def test_q6k_two_planes_largest_subscales():
    """Q6_K below the rounded plan's rows: every sub-scale +-127 or -128, products up to 4096 kept exact
    (the int8 GEMM; the prefill GEMM's two operand planes: test_q6k_two_planes_on_the_split_plan)."""
    rows, k, n = 270, 2560, 259
    raw = exact_weights(o.Q6_K, rows, k, seed=3)
    sc = np.random.default_rng(4).choice(np.array([127, -127, -128], np.int8), size=(rows * k // 256, 16))
    raw.reshape(-1, 210)[:, 192:208] = sc.view(np.uint8)
    x = exact_x(n, k, seed=5, dtype=torch.float32)
    y = _torch_op(o.Q6_K, dev(raw), x.cuda(), rows).cpu().numpy()
    ref = exact_ref(raw, o.Q6_K, x, form="mmq")
    # integers below 2^24 (exact_ref asserts it): any order of the fp32 sums is exact
    assert np.array_equal(y, ref)


@pytest.mark.parametrize("qt,n", [(o.IQ4_XS, 1100), (o.IQ2_S, 1100), (o.Q2_K, 900)], ids=["IQ4_XS", "IQ2_S", "Q2_K"])
def test_noalloc_in_parts(lib, qt, n):
    """Products whose fp16 activation copy exceeds the static scratch and whose int8 copy fits it: the
    no-allocation entry point runs them on the latter (in parts on larger weights, test_x_view_in_parts),
    with the same results."""
    rows, k = 400, 5120
    w = dev(w_rand(qt, rows, k, seed=n))
    x = x_rand(n, k, seed=n + 1, dtype=torch.float32).cuda()
    a, need = _capi_op(lib, qt, w, x, rows, "noalloc")
    assert need > lib.gguf_scratch_bytes()
    b, _ = _capi_op(lib, qt, w, x, rows)
    # the parts' plans may add in another order: 8 fp32 roundings of sums of 160 slice terms
    assert float((a - b).norm() / b.norm()) <= 8 * 2.0 ** -24 * np.sqrt(160)


@pytest.mark.parametrize("n", [16, 100])
def test_q2k_group_sum_beyond_fp16(n):
    """A 16-value group whose sum overflows fp16 (D2S6 keeps it as fp16): every weight row with a
    nonzero min there gives dmin m's infinity, not a NaN from 0 x inf in the second plane of mins."""
    rows, k = 400, 2560
    raw = w_rand(o.Q2_K, rows, k, seed=7)
    x = x_rand(n, k, seed=8, dtype=torch.float32)
    x[1, 64:80] = -60000.0
    y = _torch_op(o.Q2_K, dev(raw), x.cuda(), rows).cpu().numpy()
    blk = np.ascontiguousarray(raw).reshape(rows, k // 256, 84)[:, 0]
    dmin = np.ascontiguousarray(blk[:, 82:84]).view(np.float16)[:, 0].astype(np.float32)
    min4 = (dmin * (blk[:, 4] >> 4)).astype(np.float16)
    some = min4 != 0
    assert some.any() and np.array_equal(y[1, some], np.sign(min4[some]).astype(np.float32) * np.inf)
    assert np.isfinite(np.delete(y, 1, axis=0)).all()


# 64-column tiles; (4102, 2560, 600): 128; (16390, 2560, 1000): 256
@pytest.mark.parametrize("rows,k,n", [(270, 5120, 1), (270, 5120, 8), (270, 2560, 24), (270, 2560, 300),
                                      (4102, 2560, 600), (16390, 2560, 1000)])
@pytest.mark.parametrize("scales", ["ordinary", "subnormal", "wide"])
def test_q2k_scales_rounded_as_the_model(rows, k, n, scales):
    """Q2_K's products keep d times sub-scale as fp16, as the reference's tile loader does: fp32 X against
    the float64 model that rounds there. The rest is fp32 sums: 2^-24 of the partial sum at each of the
    K / 32 slices, adding up at random. (An unrounded d times sub-scale is 2.5e-4 off.) Scales of an
    ordinary file, of which many are fp16 subnormals, and from 2^-20 to 2^10 within a row with zeros
    among them, for which the rows' unit of account moves."""
    raw = o.random_blocks(np.random.default_rng(n), o.Q2_K, rows, k, scale_sigma=3e-6 if scales == "subnormal" else 2e-3)
    if scales == "wide":
        rng = np.random.default_rng(n + 1)
        b = raw.reshape(-1, 84)
        for at in o.SCALE_OFFSETS[o.Q2_K]:
            d = (2.0 ** rng.uniform(-20, 10, len(b)) * (rng.random(len(b)) > 0.1)).astype(np.float16)
            b[:, at:at + 2] = d.view(np.uint8).reshape(-1, 2)
    x = x_rand(n, k, seed=n + 2)
    y = _torch_op(o.Q2_K, dev(raw), x.cuda(), rows).cpu().numpy()
    rs = np.unique(np.random.default_rng(3).choice(rows, 64, replace=False))
    ref = o.q81_model(raw[rs], o.Q2_K, x, layout="mmq")
    assert o.rel_l2(y[:, rs], ref) <= 2 * np.sqrt(k / 32) * 2.0 ** -24


@pytest.mark.parametrize("n", [16, 100])
@pytest.mark.parametrize("group", [3, 6, 13, 15])
def test_q2k_min_beyond_fp16(n, group):
    """A min that overflows fp16 (dmin * m as the tile loader keeps it) of a group whose sum is stored
    (0..5 of each 128 values) or taken from q8 (6, 7): the weight row's outputs are minus the sum's
    infinity; the other rows stay finite."""
    rows, k = 144, 5120
    raw = w_rand(o.Q2_K, rows, k, seed=9)
    blk = raw.reshape(rows, k // 256, 84)
    bad = np.arange(0, rows, 7)
    blk[bad, 1, :16] = (blk[bad, 1, :16] & 0xF) | 0x10
    blk[bad, 1, group] |= 0xF0
    blk[bad, 1, 82:84] = np.array([30000], np.float16).view(np.uint8)  # m = 1: finite, 15: 450000
    x = x_rand(n, k, seed=10)
    y = _torch_op(o.Q2_K, dev(raw), x.cuda(), rows).cpu().numpy()
    q8 = o.quantize_q8_1_mmq(x, o.Q2_K)
    q, _ = o.dequant_q8_1_mmq(q8, n, k, o.Q2_K)
    sums = o.mmq_d2s6_sums(q8, n, k).reshape(n, k // 16)
    sums = np.where(np.isnan(sums), q.astype(np.int64).reshape(n, k // 16, 16).sum(-1), sums)[:, 16 + group]
    want = np.where(sums == 0, np.nan, np.where(sums < 0, np.inf, -np.inf)).astype(np.float32)
    assert (sums > 0).any() and (sums < 0).any()
    assert np.array_equal(y[:, bad], np.repeat(want[:, None], len(bad), 1), equal_nan=True)
    assert np.isfinite(np.delete(y, bad, axis=1)).all()


def _run_ws(lib, qt, w, x, rows, nbytes):
    """gguf_mul_mat with a workspace of nbytes bytes: (rc, output, bytes of the workspace that were written,
    counted to the last one; its fill is 0xFF)."""
    from vllm_gguf_plugin import _capi

    op, n = (PACKED_TILED if qt in PACKED else MUL_MAT_Q), x.shape[0]
    y = torch.full((n, rows), float("nan"), dtype=x.dtype, device="cuda")
    ws = torch.full((nbytes + 256,), 0xFF, dtype=torch.uint8, device="cuda")
    rc = lib.gguf_mul_mat(op, _capi.ref(_capi.view(w)), _capi.ref(_capi.view(x)), qt, rows, None, y.data_ptr(),
                          y.numel() * y.element_size(), ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    written = (ws != 0xFF).nonzero()
    return rc, y, int(written[-1]) + 1 if len(written) else 0


def _xh(qt, k, n):
    return -(-n // 16) * (k // 256) * (8192 + (2560 if qt == o.Q2_K else 1024))


def _int8(qt, k, n):
    return n * k // 128 * 144 if qt == o.Q2_K else -(-n // 16) * (k // 256) * 4608


# whole tiles of 128 rows on few CUs lose to the small GEMMs' 16-row tiles
@pytest.mark.parametrize("qt,rows,k,n,whole", [
    (o.IQ4_XS, 5120, 6144, 65, False), (o.IQ4_XS, 17408, 5120, 65, True), (o.IQ4_XS, 5120, 17408, 100, False),
    (o.Q6_K, 5120, 17408, 100, False), (o.Q6_K, 34816, 5120, 65, True), (o.IQ2_S, 1024, 5120, 300, False),
    (o.IQ2_XXS, 17408, 5120, 65, True), (o.IQ3_XXS, 1024, 5120, 257, False), (o.IQ3_S, 5120, 17408, 100, False),
    (o.Q2_K, 1024, 5120, 16, False), (o.Q2_K, 5120, 17408, 16, False), (o.Q2_K, 17408, 5120, 100, True)])
def test_whole_tiles_where_they_are_the_faster_plan(lib, qt, rows, k, n, whole):
    """Without room for the split's parts a product runs the prefill GEMM in whole tiles only where that is
    the faster plan, which shows in what it writes of a workspace of the reported size: the fp16 copy, or
    the int8 one of half the size (and what its own split needs)."""
    op = PACKED_TILED if qt in PACKED else MUL_MAT_Q
    need = lib.gguf_op_workspace_bytes(op, qt, rows, k, n, 0)
    assert need == _xh(qt, k, n)
    w = torch.zeros(rows, o.BLOCK_BYTES[qt] * (k // 256), dtype=torch.uint8, device="cuda")
    x = torch.randn(n, k, device="cuda")
    rc, y, used = _run_ws(lib, qt, w, x, rows, need)
    assert rc == 0 and (y == 0).all()
    assert used > 0.9 * need if whole else used <= _int8(qt, k, n)
    # a workspace with room for the int8 copy alone runs the small GEMM
    rc, y, used = _run_ws(lib, qt, w, x, rows, -(-_int8(qt, k, n) // 256) * 256)
    assert rc == 0 and (y == 0).all() and used <= _int8(qt, k, n)
    rc, _, used = _run_ws(lib, qt, w, x, rows, _int8(qt, k, n) // 2)
    assert rc != 0 and used == 0


@pytest.mark.parametrize("qt,rows,k,n,taken", [
    (o.IQ4_XS, 400, 5120, 1456, True), (o.IQ4_XS, 400, 5120, 1472, False), (o.IQ4_XS, 17408, 17408, 416, True),
    (o.IQ3_S, 1024, 5120, 720, True), (o.IQ3_S, 1024, 5120, 1100, False), (o.Q4_K, 400, 5120, 1100, False),
    (o.IQ3_S, 2048, 17408, 300, True), (o.IQ3_S, 8192, 17408, 300, False), (o.Q6_K, 400, 5120, 1400, True),
    (o.Q6_K, 8192, 5120, 1400, False), (o.IQ3_XXS, 400, 5120, 1400, True), (o.IQ3_XXS, 4096, 5120, 1400, False),
    (o.IQ2_XS, 17408, 5120, 1400, True), (o.Q2_K, 1024, 5120, 1456, True), (o.Q2_K, 1024, 5120, 1472, False)])
def test_noalloc_takes_what_the_small_gemms_copy_fits(lib, qt, rows, k, n, taken):
    """Beyond the scratch with its fp16 copy: taken where the small GEMM's workspace fits, refused on large
    grids of the types whose prefill GEMM has always read the fp16 copy, and where nothing fits."""
    from vllm_gguf_plugin import _capi

    w = torch.zeros(rows, o.BLOCK_BYTES[qt] * (k // 256), dtype=torch.uint8, device="cuda")
    x = torch.randn(n, k, device="cuda", dtype=torch.bfloat16)
    y = torch.full((n, rows), float("nan"), dtype=x.dtype, device="cuda")
    rc = lib.gguf_mul_mat_noalloc(PACKED_TILED if qt in PACKED else MUL_MAT_Q, _capi.ref(_capi.view(w)),
                                  _capi.ref(_capi.view(x)), qt, rows, None, y.data_ptr(), y.numel() * 2,
                                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (rc == 0) == taken, _capi.error(lib)
    assert (y == 0).all() if taken else "static scratch" in _capi.error(lib)


def _asked(lib, qt, w, x, rows):
    """gguf_mul_mat_alloc: (output, bytes of the workspace it asked for)."""
    from vllm_gguf_plugin import _capi

    n, got = x.shape[0], {}

    def alloc(_, what, nbytes):
        got[what] = torch.full((max(nbytes, 1),), 0xFF, dtype=torch.uint8, device="cuda")
        got[what, "bytes"] = nbytes
        return got[what].data_ptr()

    fn = _capi.ALLOC_FN(alloc)
    rc = lib.gguf_mul_mat_alloc(PACKED_TILED if qt in PACKED else MUL_MAT_Q, _capi.ref(_capi.view(w)),
                                _capi.ref(_capi.view(x)), qt, rows, None, fn, None,
                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _capi.error(lib)
    torch.cuda.synchronize()
    y = got[_capi.ALLOC_OUTPUT][:n * rows * x.element_size()].view(x.dtype).view(n, rows)
    return y, got[_capi.ALLOC_WORKSPACE, "bytes"]


# small products, few rows of a deep K, and few activation rows are faster on the small GEMMs
@pytest.mark.parametrize("qt,rows,k,n,split", [
    (o.IQ4_XS, 512, 512, 300, False), (o.IQ4_XS, 1024, 1024, 300, False), (o.IQ4_XS, 1024, 512, 1024, True),
    (o.IQ2_S, 512, 512, 300, False), (o.IQ2_S, 1024, 2048, 257, True), (o.Q6_K, 1024, 1024, 512, False),
    (o.IQ4_XS, 1024, 17408, 100, False), (o.IQ4_XS, 1024, 17408, 129, True), (o.Q6_K, 512, 17408, 512, False),
    (o.Q4_K, 2048, 17408, 65, False), (o.Q4_K, 3072, 17408, 65, True), (o.IQ2_XS, 1024, 17408, 65, True),
    (o.IQ3_XXS, 8192, 5120, 33, False), (o.IQ3_XXS, 17408, 5120, 33, True), (o.IQ3_XXS, 4096, 4096, 64, True),
    (o.IQ4_XS, 2048, 17408, 49, False), (o.IQ4_XS, 3072, 17408, 33, False), (o.IQ4_XS, 3072, 17408, 49, True),
    (o.Q2_K, 1024, 1024, 16, False), (o.Q2_K, 1024, 2048, 32, False), (o.Q2_K, 1024, 2048, 48, True),
    (o.Q2_K, 12288, 5120, 1, True)])
def test_split_where_it_is_the_faster_plan(lib, qt, rows, k, n, split):
    """The workspace the library sizes itself: with the split's parts (a slot of 2 x 4096 bytes for each row
    tile and column pair of a workgroup's tile, a counter a tile) only where that plan is the faster one; the
    small GEMM's otherwise, of at most the int8 copy and its own split."""
    w = torch.zeros(rows, o.BLOCK_BYTES[qt] * (k // 256), dtype=torch.uint8, device="cuda")
    y, asked = _asked(lib, qt, w, torch.randn(n, k, device="cuda"), rows)
    assert (y == 0).all()
    small = -(-_int8(qt, k, n) // 256) * 256
    if split:  # at least the copy: runs of whole tiles need no parts
        assert asked >= -(-_xh(qt, k, n) // 256) * 256
    else:  # the int8 GEMM on few row tiles splits K too (at most four ways)
        slots = 4 * 1024 * -(-n // 16) * -(-rows // 16) + 1024 if qt in (o.Q4_K, o.Q6_K, o.IQ4_XS) else 0
        assert small <= asked <= small + slots and asked != -(-_xh(qt, k, n) // 256) * 256


@pytest.mark.parametrize("qt,rows,k,n,split", [(o.IQ3_S, 512, 512, 300, False), (o.IQ3_S, 4096, 4096, 64, False),
                                               (o.IQ3_S, 6144, 4096, 64, True), (o.Q4_K, 1024, 1024, 512, False)])
def test_split_plan_of_the_fp16_small_gemms_types(lib, qt, rows, k, n, split):
    """The same where the small GEMM reads the fp16 copy too: its workspace is the copy alone."""
    w = torch.zeros(rows, o.BLOCK_BYTES[qt] * (k // 256), dtype=torch.uint8, device="cuda")
    y, asked = _asked(lib, qt, w, torch.randn(n, k, device="cuda"), rows)
    assert (y == 0).all() and (asked > _xh(qt, k, n) if split else asked == -(-_xh(qt, k, n) // 256) * 256)
