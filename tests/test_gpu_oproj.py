"""o_proj on the GPU vs the oracle (engine.c:969-973, matvec.c:98-122).

x[b] += W_o . att[b].  Up to 8 tokens every product and sum is in f32 (the
reference's arithmetic in another order), in the one-pass kernel or the rows
kernel; more tokens go through the rows kernel or the MFMA GEMM with f16
weights times the f16 hi + lo parts of f32 att (about 22 bits of each
activation), f16 weights times f16 att (the attention kernel's f16 output) or,
for f32 weights, the hi + lo parts of both.  Either way the result must be
within relative L2 1e-5 of the f32 oracle (the stated bar is 1e-3), on the
updated x and on the product alone.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle_lib import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5


def gen(seed, shape, sigma=1.0):
    from yllm_amd.attention import synth_normal

    return synth_normal(seed, int(np.prod(shape)), sigma).reshape(shape)


def weights(oracle, seed, hidden, qdim, f16):
    w = gen(seed, (hidden, qdim), 1.0 / np.sqrt(qdim))
    return oracle.f32_to_f16(w) if f16 else w


def to_dev(cuda, w):
    t = torch.from_numpy(np.ascontiguousarray(w)).to(cuda)
    return t.view(torch.float16) if w.dtype == np.uint16 else t


@pytest.mark.parametrize("B,hidden,qdim,f16", [
    (1, 896, 896, True),      # decode, the 0.5B shape (14 heads x 64)
    (3, 4096, 4096, True),
    (8, 2048, 4096, True),    # the largest batch with f32 products
    (1, 1000, 512, False),    # f32 weights, a hidden size that is no multiple of the rows per wave
    (9, 896, 896, True),      # the smallest batch with split products
    (64, 4096, 4096, True),
    (300, 2048, 4096, True),
    (77, 1024, 2048, False),  # f32 GEMM
    (200, 4096, 4096, True),  # 64 x 64 tiles, a partial token tile
    (200, 1000, 904, False),  # f32 weights; hidden and qdim no multiples of the tiles or of 64
    (130, 520, 1032, True),   # ragged edges
    (64, 333, 904, True),     # the engine's 64-token chunk, ragged edges
])
def test_o_proj_matches_oracle(cuda, oracle, B, hidden, qdim, f16):
    from yllm_amd.attention import o_proj

    x0 = gen(2001 + B, (B, hidden))
    att = gen(2002 + B, (B, qdim), 0.5)
    w = weights(oracle, 2003 + B, hidden, qdim, f16)
    want = oracle.o_proj(x0, att, w)
    xt = torch.from_numpy(x0).to(cuda)
    o_proj(xt, torch.from_numpy(att).to(cuda), to_dev(cuda, w))
    got = xt.cpu().numpy()
    err = rel_l2(got, want)
    err_p = rel_l2(got.astype(np.float64) - x0, want.astype(np.float64) - x0)
    print(f"o_proj B={B} {hidden}x{qdim} {'f16' if f16 else 'f32'}: rel_l2 {err:.2e}, product only {err_p:.2e}")
    assert err <= TOL and err_p <= TOL
    assert max(rel_l2(got[b], want[b]) for b in range(B)) <= 3 * TOL


@pytest.mark.parametrize("B", [1, 6, 200])
def test_o_proj_f16_attention_output(cuda, oracle, B):
    """att written as f16 by the attention kernel: the one-pass kernel widens
    it, the MFMA kernels take it as it is; the oracle sees the same f16 values."""
    from yllm_amd.attention import o_proj

    hidden, qdim = 2048, 4096
    x0 = gen(2401 + B, (B, hidden))
    att16 = oracle.f32_to_f16(gen(2402 + B, (B, qdim), 0.5))
    w = weights(oracle, 2403 + B, hidden, qdim, True)
    want = oracle.o_proj(x0, att16.view(np.float16).astype(np.float32), w)
    xt = torch.from_numpy(x0).to(cuda)
    o_proj(xt, to_dev(cuda, att16), to_dev(cuda, w))
    err = rel_l2(xt.cpu().numpy(), want)
    print(f"o_proj f16 att B={B}: rel_l2 {err:.2e}")
    assert err <= TOL


def gemm_tile(B, hidden, kind):
    """The tile launch_gemm takes for B tokens: the largest of its list of which
    there are three quarters of the CUs, else the last."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = {"f16": [(256, 256), (128, 256), (128, 128), (64, 128), (64, 64)],
             "f32": [(128, 256), (64, 128), (64, 64)],
             "w32": [(128, 128), (64, 64)]}[kind]
    for bt, bo in tiles[:-1]:
        if -(-B // bt) * -(-hidden // bo) >= cus * 3 // 4:
            return bt, bo
    return tiles[-1]


# B, hidden, qdim and, past the rows kernel, the tile of f32 / f16 att (f16 weights)
EDGES = [
    (3, 40, 72), (5, 1000, 904), (8, 56, 4200),  # one-pass or rows kernel, f32 products up to 8 f32 tokens
    (3, 300, 3072), (4, 300, 904), (5, 4096, 72), (6, 333, 72), (7, 5000, 136),  # where the rows kernel starts
    (16, 896, 896), (17, 40, 264), (33, 1000, 4104), (63, 48, 4200),  # rows kernel: 16-token blocks, ragged K, two rounds
    (65, 300, 72, (64, 64), (64, 64)), (250, 1100, 40, (64, 64), (64, 64)),  # fewer K steps than LDS stages
    (520, 1540, 360, (64, 64), (64, 64)),      # partial in both directions, as all below
    (520, 2900, 72, (64, 128), (64, 128)),
    (1030, 3100, 136, (64, 128), (128, 128)),
    (2050, 3330, 200, (128, 256), (128, 256)),
    (3600, 4000, 104, (128, 256), (256, 256)),
]


@pytest.mark.parametrize("att16", [False, True], ids=["f32att", "f16att"])
@pytest.mark.parametrize("B,hidden,qdim,tile", [(*e[:3], e[3:]) for e in EDGES],
                         ids=["-".join(map(str, e[:3])) for e in EDGES])
def test_o_proj_tile_edges(cuda, B, hidden, qdim, tile, att16):
    """Every kernel and tile of the dispatch of f16 weights at sizes that leave
    partial tiles, partial K steps and a K shorter than the pipeline, against
    float64.  Bound:
    qdim products of |w att| accumulate in fp32 (each addition within 2^-24 of
    the running sum) and the split of f32 att leaves 2^-22 of each product, so
    the error stays under (qdim 2^-24 + 2^-22) sum |w att| + 2^-23 |x|."""
    from yllm_amd.attention import o_proj

    if B > 64:
        assert gemm_tile(B, hidden, "f16" if att16 else "f32") == tile[att16]
    g = torch.Generator(device="cuda").manual_seed(B)
    att = torch.randn(B, qdim, generator=g, device=cuda) * 0.5
    att = att.half() if att16 else att
    w = (torch.randn(hidden, qdim, generator=g, device=cuda) * qdim ** -0.5).half()
    x0 = torch.randn(B, hidden + 8, generator=g, device=cuda)
    x = x0.clone()
    o_proj(x[:, :hidden], att, w)
    want = x0[:, :hidden].double() + att.double() @ w.double().t()
    bound = (qdim * 2.0 ** -24 + 2.0 ** -22) * (att.double().abs() @ w.double().abs().t()) \
        + 2.0 ** -23 * want.abs() + 2.0 ** -23 * x0[:, :hidden].double().abs()
    assert ((x[:, :hidden].double() - want).abs() <= bound).all()
    assert torch.equal(x[:, hidden:], x0[:, hidden:])


@pytest.mark.parametrize("B,hidden,qdim,tile", [
    (9, 40, 72, (64, 64)), (64, 300, 1032, (64, 64)), (300, 1100, 40, (64, 64)),
    (1800, 1700, 40, (128, 128)), (1800, 1700, 328, (128, 128)),  # fewer K steps than stages, a ragged last one
    (2048, 2048, 256, (128, 128)),                                # whole tiles only
])
def test_o_proj_f32_weight_tiles(cuda, B, hidden, qdim, tile):
    """Both tiles of f32 weights against float64.  Three products per pair (hi
    hi, lo hi, hi lo), so 3 qdim additions in fp32, and 2^-22 each of att's
    split, w's and the dropped lo lo: under (3 qdim 2^-24 + 3 2^-22) sum
    |w att| + 2^-23 |x|."""
    from yllm_amd.attention import o_proj

    assert gemm_tile(B, hidden, "w32") == tile
    g = torch.Generator(device="cuda").manual_seed(B + qdim)
    att = torch.randn(B, qdim, generator=g, device=cuda) * 0.5
    w = torch.randn(hidden, qdim, generator=g, device=cuda) * qdim ** -0.5
    x0 = torch.randn(B, hidden + 8, generator=g, device=cuda)
    x = x0.clone()
    o_proj(x[:, :hidden], att, w)
    want = x0[:, :hidden].double() + att.double() @ w.double().t()
    bound = (3 * qdim * 2.0 ** -24 + 3 * 2.0 ** -22) * (att.double().abs() @ w.double().abs().t()) \
        + 2.0 ** -23 * want.abs() + 2.0 ** -23 * x0[:, :hidden].double().abs()
    assert ((x[:, :hidden].double() - want).abs() <= bound).all()
    assert torch.equal(x[:, hidden:], x0[:, hidden:])


@pytest.mark.parametrize("att16", [False, True], ids=["f32att", "f16att"])
def test_o_proj_few_large_tokens(cuda, att16):
    """Up to 8 f32 tokens keep f32 products: values past f16's range stay finite."""
    from yllm_amd.attention import o_proj

    g = torch.Generator(device="cuda").manual_seed(6)
    att = torch.randn(8, 128, generator=g, device=cuda) * (1000.0 if att16 else 1e6)
    att = att.half() if att16 else att
    w = torch.randn(80, 128, generator=g, device=cuda).half()
    x = torch.zeros(8, 80, device=cuda)
    want = att.double() @ w.double().t()
    o_proj(x, att, w)
    assert float((x.double() - want).norm() / want.norm()) <= 1e-6


@pytest.mark.parametrize("att16", [False, True], ids=["f32att", "f16att"])
def test_o_proj_rows_too_far_apart_for_a_tile(cuda, att16):
    """att rows 2^22 elements apart: a tile's 32-bit offsets do not reach.  f32
    rows are made contiguous in the workspace, f16 rows (which bring none) go
    through the one-pass kernel eight tokens at a time."""
    from yllm_amd.attention import o_proj

    B, hidden, qdim, stride = 11, 72, 64, 1 << 22
    g = torch.Generator(device="cuda").manual_seed(5)
    att = torch.zeros(B, stride, dtype=torch.float16 if att16 else torch.float32, device=cuda)[:, :qdim]
    att.copy_(torch.randn(B, qdim, generator=g, device=cuda) * 0.5)
    w = (torch.randn(hidden, qdim, generator=g, device=cuda) * qdim ** -0.5).half()
    x = torch.randn(B, hidden, generator=g, device=cuda)
    want = x.double() + att.double() @ w.double().t()
    o_proj(x, att, w)
    assert float((x.double() - want).norm() / want.norm()) <= 1e-6


def test_o_proj_strided_rows_and_repeat(cuda, oracle):
    """att and x as slices of wider rows; a second call adds again (x is the
    residual stream, updated in place); a smaller batch after a larger one."""
    from yllm_amd.attention import o_proj, o_proj_workspace_bytes

    hidden, qdim = 1024, 2048
    w = weights(oracle, 2101, hidden, qdim, True)
    wt = to_dev(cuda, w)
    ws = torch.empty(o_proj_workspace_bytes(40, hidden, qdim, torch.float16), dtype=torch.uint8, device=cuda)
    for B in (40, 12, 5):
        x0 = gen(2102 + B, (B, hidden + 64))
        att = gen(2103 + B, (B, qdim + 32), 0.5)
        xt = torch.from_numpy(x0).to(cuda)
        at = torch.from_numpy(att).to(cuda)
        o_proj(xt[:, 16:16 + hidden], at[:, 8:8 + qdim], wt, workspace=ws)
        o_proj(xt[:, 16:16 + hidden], at[:, 8:8 + qdim], wt, workspace=ws)
        got = xt.cpu().numpy()
        once = oracle.o_proj(x0[:, 16:16 + hidden], att[:, 8:8 + qdim], w)
        want = oracle.o_proj(once, att[:, 8:8 + qdim], w)
        assert rel_l2(got[:, 16:16 + hidden], want) <= TOL
        # the columns around the slice are untouched
        assert np.array_equal(got[:, :16], x0[:, :16]) and np.array_equal(got[:, 16 + hidden:], x0[:, 16 + hidden:])


def test_o_proj_full_size_sampled_rows(cuda, oracle):
    """8192 tokens of a 4096 x 4096 f16 o_proj in one call (the GEMM path);
    rows sampled across the batch are checked against the oracle."""
    from yllm_amd.attention import o_proj

    B, hidden, qdim = 8192, 4096, 4096
    w = weights(oracle, 2201, hidden, qdim, True)
    x0 = gen(2202, (B, hidden))
    att = gen(2203, (B, qdim), 0.5)
    xt = torch.from_numpy(x0).to(cuda)
    o_proj(xt, torch.from_numpy(att).to(cuda), to_dev(cuda, w))
    got = xt.cpu().numpy()
    rows = np.array([0, 1, 1000, 4095, 4096, 8191])
    want = oracle.o_proj(x0[rows], att[rows], w)
    assert rel_l2(got[rows], want) <= TOL


def test_o_proj_after_gated_decode(cuda, oracle):
    """The qwen35 step after attention (engine.c:958-973): split-K decode with
    the sigmoid gate in its epilogue, then o_proj into the residual stream."""
    from yllm_amd.attention import LayerKV, attn_decode, kv_store, o_proj

    nh, nkv, d, L, hidden = 16, 2, 256, 300, 1024
    kvd, qd = nkv * d, nh * d
    K = oracle.f32_to_f16(gen(2301, (L, kvd), 0.5)).view(np.float16).astype(np.float32)
    V = oracle.f32_to_f16(gen(2302, (L, kvd), 0.5)).view(np.float16).astype(np.float32)
    q = gen(2303, (qd,), 0.5)
    gate = gen(2304, (qd,))
    w = weights(oracle, 2305, hidden, qd, True)
    x0 = gen(2306, (1, hidden))
    cache = LayerKV.empty(nkv, d, L, device=cuda)
    kv_store(cache, torch.from_numpy(K).to(cuda), torch.from_numpy(V).to(cuda), 0)
    att = attn_decode(torch.from_numpy(q).to(cuda), cache, L - 1, nh, gate=torch.from_numpy(gate).to(cuda))
    xt = torch.from_numpy(x0).to(cuda)
    o_proj(xt, att.view(1, -1), to_dev(cuda, w))
    kc, vc = oracle.f32_to_f16(K), oracle.f32_to_f16(V)
    att_want = oracle.gate_sigmoid(oracle.decode(q, kc, vc, L - 1, nh, nkv, d), gate)
    want = oracle.o_proj(x0, att_want[None, :], w)
    err = rel_l2(xt.cpu().numpy(), want)
    print(f"gated decode + o_proj: rel_l2 {err:.2e}")
    assert err <= 1e-3


@pytest.mark.parametrize("B", [9, 64, 300])
@pytest.mark.parametrize("wdt", ["f16", "f32"])
@pytest.mark.parametrize("how", ["same", "rows", "columns", "beside"])
def test_o_proj_reads_att_that_overlaps_x(cuda, B, wdt, how):
    """f32 att that shares memory with x, more than 8 tokens (fewer never
    allowed it): all of att is read before x changes, so x += W x is what it
    says.  Same rows, x one row further on, overlapping columns, and columns
    side by side in one matrix, which share no element.  Bound as in the tile
    tests: att is split (and f32 w), sums in fp32."""
    from yllm_amd.attention import o_proj

    n = 520
    g = torch.Generator(device="cuda").manual_seed(B)
    w = torch.randn(n, n, generator=g, device=cuda) * n ** -0.5
    w = w.half() if wdt == "f16" else w
    m = torch.randn(B + 1, 2 * n, generator=g, device=cuda)
    att, x = {"same": (m[:B, :n], m[:B, :n]), "rows": (m[:B, :n], m[1:, :n]), "columns": (m[:B, :n], m[:B, 13:n + 13]),
              "beside": (m[:B, :n], m[:B, n:])}[how]
    m0, a64, x64 = m.clone(), att.double(), x.double()
    o_proj(x, att, w)
    want = x64 + a64 @ w.double().t()
    bound = (3 * n * 2.0 ** -24 + 3 * 2.0 ** -22) * (a64.abs() @ w.double().abs().t()) + 2.0 ** -23 * (want.abs() + x64.abs())
    assert ((x.double() - want).abs() <= bound).all()
    x.copy_(x64)  # nothing else changed
    assert torch.equal(m, m0)


def test_o_proj_reads_weights_that_overlap_x(cuda):
    """f32 weights that share memory with x: all of them are read before x changes."""
    from yllm_amd.attention import o_proj

    B, hidden, qdim = 40, 72, 80
    g = torch.Generator(device="cuda").manual_seed(1)
    m = torch.randn(64 * 128, generator=g, device=cuda)
    w, x = m[:hidden * qdim].view(hidden, qdim), m[2048:2048 + B * hidden].view(B, hidden)
    att = torch.randn(B, qdim, generator=g, device=cuda)
    w64, x64 = w.double(), x.double()
    o_proj(x, att, w)
    want = x64 + att.double() @ w64.t()
    bound = (3 * qdim * 2.0 ** -24 + 3 * 2.0 ** -22) * (att.double().abs() @ w64.abs().t()) + 2.0 ** -23 * (want.abs() + x64.abs())
    assert ((x.double() - want).abs() <= bound).all()
