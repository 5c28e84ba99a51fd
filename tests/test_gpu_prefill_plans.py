"""The prefill GEMM's three tile widths (64, 128 and 256 activation rows a workgroup) in both plans, K
split over the CUs and whole tiles, for every decoder of it (Q6_K's exact and its rounded operands
apart), in the exact-integer mode: with every scale 1 any order of the sums gives the oracle's int64 sum.
The width is asserted: from the bytes of workspace that the split plan asks for, and for whole tiles from
the cost model restated here, with the written part of the workspace. Then activations that are not
16-byte aligned or have rows further apart than K, the products of 33..64 rows, and Q6_K's rounded
operands at the largest sub-scales. Needs an MI355X.
"""

import numpy as np
import pytest
import torch

import gguf_oracle as o
from _gpu import dev, exact_ref, exact_weights, exact_x, graph_replays_equal, w_rand, x_rand
from test_gpu_prefill_split import PACKED, TYPES, _asked, _capi_op, _int8, _run_ws, _torch_op, _weight, _xh, lib  # noqa: F401

pytestmark = pytest.mark.gpu

CUS = 256


def _tiles(rows, n, rs):
    return -(-rows // 128) * -(-(-(-n // 16)) // (16 // rs))


def _split_plan(rows, k, n):
    """pf_shape's choice: (row parts, workspace bytes of the parts and the tiles' counters)."""
    best = None
    for rs, fixed, few, full in ((1, 20, 3.5, 5.6), (2, 16, 2.3, 3.0), (4, 14, 1.7, 2.3)):
        tiles = _tiles(rows, n, rs)
        units = tiles * (k // 256)
        wgs = max(1, min(CUS, units // 4))
        t = fixed + -(-units // wgs) * (few + (full - few) * wgs / CUS)
        if best is None or t < best[0]:
            best = (t, rs, tiles, units, wgs)
    _, rs, tiles, units, wgs = best
    if units % wgs == 0 and units // wgs % (k // 256) == 0:
        return rs, 0
    return rs, (wgs + min(wgs, tiles)) * (16 // rs) * 2 * 4096 + -(-tiles * 4 // 256) * 256


def _whole_rs(qt, exact, rows, k, n):
    """pf_whole_shape's choice of row parts."""
    block = {o.IQ4_XS: (5.5, 3.3, 2.2), o.Q2_K: (6.2, 4.2, 3.2)}.get(qt, (4.1, 2.75, 2.0))
    if qt == o.Q6_K and exact:
        block = (6.2, 4.2, 3.2)
    us = [-(-_tiles(rows, n, rs) // CUS) * (a + k // 256 * b) for rs, a, b in zip((1, 2, 4), (14, 11, 8.5), block)]
    return (1, 2, 4)[us.index(min(us))]


def _q6k_exact(rows, n):
    return not (n >= 256 and -(-rows // 128) * -(-n // 256) >= 64)


def _case(qt, rows, k, n):
    """(weight rows, raw rows, X, the weight rows checked, their exact outputs): the first and last rows and
    some between."""
    rows = -(-rows // 16) * 16 if qt in PACKED else rows
    raw = exact_weights(qt, rows, k, seed=rows + n)
    x = exact_x(n, k, seed=n, dtype=torch.float32)
    rs = np.unique(np.r_[0:20, rows - 40:rows, np.random.default_rng(n).choice(rows, 20)])
    return rows, raw, x, rs, exact_ref(raw[rs], qt, x, form="mmq")


# rows and activation rows that are multiples of no tile
SPLIT = [(4, 1030, 4608, 257), (2, 4102, 2560, 513), (1, 16390, 2560, 993)]
Q6K_SPLIT = [(4, 4102, 512, 257, False), (2, 16390, 2560, 100, True), (1, 34822, 2560, 200, True)]


@pytest.mark.parametrize("width,qt,rows,k,n", [(s[0], qt, *s[1:]) for s in SPLIT for qt in TYPES]
                         + [(s[0], o.Q6_K, *s[1:4]) for s in Q6K_SPLIT])
def test_split_widths_exact(lib, width, qt, rows, k, n):  # noqa: F811
    rows, raw, x, rs, ref = _case(qt, rows, k, n)
    parts, extra = _split_plan(rows, k, n)
    assert parts == width and extra > 0
    w, xg = _weight(qt, raw), x.cuda()
    y, asked = _asked(lib, qt, w, xg, rows)
    assert asked == -(-_xh(qt, k, n) // 256) * 256 + extra
    assert np.array_equal(y.cpu().numpy()[:, rs], ref)


def test_q6k_split_widths_cover_both_operand_forms():
    """SPLIT and Q6K_SPLIT run Q6_K with exact and with rounded operands at every width."""
    seen = {(w, _q6k_exact(r, n)) for w, r, _, n in SPLIT} | {(s[0], _q6k_exact(s[1], s[3])) for s in Q6K_SPLIT}
    assert seen == {(w, e) for w in (1, 2, 4) for e in (True, False)}
    assert all(_q6k_exact(s[1], s[3]) == s[4] for s in Q6K_SPLIT)


WHOLE = [(4, 8198, 2048, 65), (2, 17414, 1024, 100), (1, 17414, 1024, 200)]
Q6K_WHOLE = [(4, 4102, 2048, 257), (2, 17414, 1024, 300), (1, 17414, 1024, 500)]  # rounded operands


@pytest.mark.parametrize("width,qt,rows,k,n", [(s[0], qt, *s[1:]) for s in WHOLE for qt in TYPES]
                         + [(s[0], o.Q6_K, *s[1:]) for s in Q6K_WHOLE])
def test_whole_tile_widths_exact(lib, width, qt, rows, k, n):  # noqa: F811
    rows, raw, x, rs, ref = _case(qt, rows, k, n)
    exact = _q6k_exact(rows, n)
    assert exact == ((width, rows, k, n) not in Q6K_WHOLE) and _whole_rs(qt, exact, rows, k, n) == width
    need = lib.gguf_op_workspace_bytes(7 if qt in PACKED else 1, qt, rows, k, n, 0)
    assert need == -(-_xh(qt, k, n) // 256) * 256
    rc, y, used = _run_ws(lib, qt, _weight(qt, raw), x.cuda(), rows, need)
    assert rc == 0 and used > _int8(qt, k, n)  # the fp16 copy
    assert np.array_equal(y.cpu().numpy()[:, rs], ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("qt", [o.IQ3_S, o.Q4_K, o.Q2_K, o.IQ4_XS], ids=lambda t: o.TYPE_NAMES[t])
@pytest.mark.parametrize("off,pad", [(0, 8), (1, 0), (3, 5)], ids=["rows_apart", "offset", "offset_and_odd_stride"])
def test_x_views(lib, qt, off, pad, dtype):  # noqa: F811
    """X as a view whose rows lie further apart than K, start off a 16-byte boundary, or both: the bits of a
    contiguous copy, in both plans of the prefill GEMM and without it (the fp16 small GEMM for IQ3_S and Q4_K,
    the int8 or per-slice one else)."""
    for rows, k, n in ((1040, 4608, 257), (96, 1024, 200)):
        w = _weight(qt, w_rand(qt, rows, k, seed=n))
        buf = torch.zeros(n * (k + pad) + off + 8, dtype=dtype, device="cuda")
        x = buf[off:off + n * (k + pad)].view(n, k + pad)[:, :k]
        x.copy_(x_rand(n, k, seed=n, dtype=dtype))
        copy = x.clone()
        assert copy.is_contiguous() and (x.stride(0), x.data_ptr() % 16) == (k + pad, off * x.element_size() % 16)
        assert torch.equal(_torch_op(qt, w, x, rows), _torch_op(qt, w, copy, rows))
        a, b = (_capi_op(lib, qt, w, v, rows)[0] for v in (x, copy))
        assert torch.equal(a, b)


def test_x_view_in_parts(lib):  # noqa: F811
    """The no-allocation entry point's parts of the activation rows (512 and 228 of them: the fp16 copy of all
    exceeds the scratch, and two products in whole tiles are faster than the int8 GEMM) on rows further apart
    than K: what a contiguous X gives, and what a workspace with room for all rows does."""
    rows, k, n = 8200, 5120, 740
    w = dev(w_rand(o.IQ4_XS, rows, k, seed=1))
    x = torch.zeros(n, k + 24, dtype=torch.bfloat16, device="cuda")[:, 8:8 + k]
    x.copy_(x_rand(n, k, seed=2, dtype=torch.bfloat16))
    a, need = _capi_op(lib, o.IQ4_XS, w, x, rows, "noalloc")
    assert need > lib.gguf_scratch_bytes()
    b, _ = _capi_op(lib, o.IQ4_XS, w, x.contiguous(), rows, "noalloc")
    assert torch.equal(a, b)
    # whole tiles add K in one order at any width, and the fp16 copy is used: the same bits
    assert torch.equal(a, _capi_op(lib, o.IQ4_XS, w, x, rows)[0])
    assert o.rel_l2(a[:, :48].float().cpu().numpy(),
                    o.q81_model(w[:48].cpu().numpy(), o.IQ4_XS, x.cpu(), layout="mmq")) <= 5e-3  # bf16 output


@pytest.mark.parametrize("qt", [o.IQ3_S, o.IQ3_XXS, o.Q4_K, o.Q6_K, o.IQ2_XXS], ids=lambda t: o.TYPE_NAMES[t])
@pytest.mark.parametrize("n", [49, 63])
def test_rows_49_to_63_split(lib, qt, n):  # noqa: F811
    """Below the rows of the reported workspace the torch ops' products on 24M values or more take the split
    plan (its workspace asked for), packed types too."""
    rows, k = (4112 if qt in PACKED else 4102), 6144
    raw = exact_weights(qt, rows, k, seed=n)
    x = exact_x(n, k, seed=n + 1, dtype=torch.float32)
    y, asked = _asked(lib, qt, _weight(qt, raw), x.cuda(), rows)
    assert asked == -(-_xh(qt, k, n) // 256) * 256 + _split_plan(rows, k, n)[1]
    rs = np.r_[0:20, rows - 20:rows]
    assert np.array_equal(y.cpu().numpy()[:, rs], exact_ref(raw[rs], qt, x, form="mmq"))


@pytest.mark.parametrize("qt", [o.Q4_K, o.Q2_K, o.IQ3_S], ids=lambda t: o.TYPE_NAMES[t])
def test_split_replays(lib, qt):  # noqa: F811
    """Replays of a captured product on the split plan, whose tile counters the captured quantise launch
    clears, with eager work on the same operands between them, equal the eager result bit for bit."""
    rows, k, n = 1040, 4608, 257
    w, x = _weight(qt, w_rand(qt, rows, k, seed=1)), x_rand(n, k, seed=2, dtype=torch.bfloat16).cuda()
    eager, asked = _asked(lib, qt, w, x, rows)
    assert asked == -(-_xh(qt, k, n) // 256) * 256 + _split_plan(rows, k, n)[1]
    op = getattr(torch.ops._C_gguf, "lcpp_mul_mat_iq3_packed" if qt in PACKED else "lcpp_mul_mat_q")
    assert torch.equal(op(w, x, qt, rows), eager)
    graph_replays_equal(lambda: op(w, x, qt, rows), eager)


def test_q6k_two_planes_on_the_split_plan(lib):  # noqa: F811
    """Q6_K below the rounded operands' sizes: every sub-scale +-127 or -128, products up to 4096 exact in the
    prefill GEMM's two planes of operands."""
    rows, k, n = 2054, 2560, 257
    assert _q6k_exact(rows, n)
    raw = exact_weights(o.Q6_K, rows, k, seed=3)
    sc = np.random.default_rng(4).choice(np.array([127, -127, -128], np.int8), size=(rows * k // 256, 16))
    raw.reshape(-1, 210)[:, 192:208] = sc.view(np.uint8)
    x = exact_x(n, k, seed=5, dtype=torch.float32)
    y, asked = _asked(lib, o.Q6_K, dev(raw), x.cuda(), rows)
    assert asked == -(-_xh(o.Q6_K, k, n) // 256) * 256 + _split_plan(rows, k, n)[1]
    rs = np.r_[0:40, rows - 40:rows]
    # integers below 2^24 (exact_ref asserts it): any order of the fp32 sums is exact
    assert np.array_equal(y.cpu().numpy()[:, rs], exact_ref(raw[rs], o.Q6_K, x, form="mmq"))


def test_q6k_rounded_operands_largest_subscales():
    """Q6_K from 256 rows on 64 tiles of 128 x 256 or more: (q - 32) x sub-scale is rounded to fp16 where it
    passes 2048, by at most 2^-12 of it, and everything else is exact but for the fp32 sums. Every sub-scale
    +-127 or -128."""
    rows, k, n = 4102, 2560, 513
    assert not _q6k_exact(rows, n)
    raw = w_rand(o.Q6_K, rows, k, seed=3)
    sc = np.random.default_rng(4).choice(np.array([127, -127, -128], np.int8), size=(rows * k // 256, 16))
    raw.reshape(-1, 210)[:, 192:208] = sc.view(np.uint8)
    x = x_rand(n, k, seed=5)
    y = _torch_op(o.Q6_K, dev(raw), x.cuda(), rows).cpu().numpy()
    rs = np.unique(np.random.default_rng(6).choice(rows, 48))
    w = o.dequantize(raw[rs].reshape(-1), o.Q6_K).astype(np.float64).reshape(len(rs), k)
    q, d = o.dequant_q8_1_mmq(o.quantize_q8_1_mmq(x, o.Q6_K), n, k, o.Q6_K)
    xq = (q.astype(np.float64).reshape(n, k // 32, 32) * d.astype(np.float64)[..., None]).reshape(n, k)
    err = np.abs(y[:, rs] - xq @ w.T)
    assert (err <= (2.0 ** -12 + k / 32 * 2.0 ** -24) * (np.abs(xq) @ np.abs(w).T)).all()
    assert err.max() > 0  # the rounded form is the one that runs
