"""GPU parity of the expert GEMMs' work schedule on 256-row tiles.

The up GEMM on 256-row tiles with an even n-tile count pairs an expert's last
M tile of at most 128 rows with two n-tiles (one work item), and the items of
the last, partial round of workgroups (one per CU) are split into K ranges
whose fp32 partials fold_up_kernel sums before the epilogue.  These cases are
built so that both happen, checked against the oracle (layer) or an fp64
product (one expert), within the tolerances of the layer (2e-2 bf16, 5e-2 fp8
weights).  256-row tiles are taken by bf16 calls of 192 rows per expert or more
and four rounds of work items or more, (rows / 256 + experts) n-tiles >= 4 CUs;
each case asserts the tile height of the kernels that ran.
"""
import numpy as np
import pytest

from test_gpu_layer import TOL, Case, check_case, rel_err, tile_heights
from test_gpu_stages import _bf16_round

pytestmark = pytest.mark.gpu


def _up_items(counts, n_tiles, bm=256):
    """Work items of the up GEMM: per expert n_tiles times its M tiles, with a
    last M tile of at most bm / 2 rows serving two n-tiles in one item."""
    w, paired = 0, 0
    for c in counts:
        f, r = divmod(int(c), bm)
        if 0 < r <= bm // 2:
            w += n_tiles * f + n_tiles // 2
            paired += 1
        else:
            w += n_tiles * (f + (1 if r else 0))
    return w, paired


@pytest.mark.parametrize("etype,act,wdtype,H,bm", [
    ("gated", "silu", "bf16", 2816, 256),
    ("gated", "silu", "fp8", 2816, 128),  # fp8 weights stay on 128 rows
    ("standard", "gelu", "bf16", 5632, 256),
])
def test_paired_items_and_up_tail_split(moe, oracle, etype, act, wdtype, H, bm):
    import torch

    # 16 experts averaging 512 rows, 22 n-tiles: 256-row tiles; a skewed router
    # bias spreads the counts so that several experts end in a tile of <= 128
    # rows and some have no other (a lone paired item per n-tile pair); D = 256
    # gives 8 K stages, which the items of the last round are split over
    rng = np.random.default_rng(60)
    bias = (rng.standard_normal(16) * 0.6).astype(np.float32)
    c = Case(moe, oracle, T=4096, D=256, H=H, E=16, k=2, gate="topk", expert_type=etype, act=act,
             wdtype=wdtype, xdtype="bf16", seed=60, router_bias=bias)
    try:
        _, loss, res = c.run(training=True)
        n_tiles = H // (128 if etype == "gated" else 256)
        w, paired = _up_items(res["counts"], n_tiles)
        ncu = torch.cuda.get_device_properties(0).multi_processor_count
        print(f"up items {w} (paired {paired} experts) on {ncu} CUs", flush=True)
        assert paired > 0, "the case must hold paired items"
        assert ((res["counts"] > 0) & (res["counts"] <= 128)).any(), "... and an expert of a lone one"
        assert w > ncu and w % ncu != 0 and 2 * (w % ncu) <= ncu, "the case must split a partial last round"
        assert tile_heights(lambda: c.run(training=True)) == {bm}
        check_case(c, TOL[wdtype])
    finally:
        c.dev.close()


@pytest.mark.parametrize("n,bm", [(100, 128), (300, 256), (700, 256)])
def test_expert_forward_paired_and_split(moe, oracle, n, bm):
    # one expert's rows: n = 300 is one full 256-row tile and a paired item per
    # n-tile pair, 700 = two full tiles + a 188-row tile (no pairing); every
    # item of such a small list is split into K ranges and folded.  n = 100 is
    # below 192 rows and takes a 128-row tile
    c = Case(moe, oracle, T=4096, D=256, H=4096, E=16, k=2, wdtype="bf16", xdtype="bf16", seed=82)
    try:
        x = np.ascontiguousarray(c.x[:n])
        print(f"expert_forward {bm}-row tiles n={n}", flush=True)
        y = c.dev.expert_forward(5, x)
        assert tile_heights(lambda: c.dev.expert_forward(5, x)) == {bm}
        ex = c.ex[5]
        xd = x.astype(np.float64)
        g = xd @ ex["w1"].T.astype(np.float64)
        u = xd @ ex["w3"].T.astype(np.float64)
        h = _bf16_round(oracle, (g / (1.0 + np.exp(-g))) * u).astype(np.float64)
        ref = h @ ex["w2"].T.astype(np.float64)
        err = rel_err(y, ref)
        assert err <= TOL["bf16"], f"relative error {err:.3e}"
        y2 = c.dev.expert_forward(5, x)
        assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))
    finally:
        c.dev.close()


@pytest.mark.parametrize("etype,act,H", [("gated", "silu", 2816), ("standard", "gelu", 5632)])
def test_256_row_tiles_and_their_change_between_calls(moe, oracle, etype, act, H):
    # 16 experts averaging 512 rows with 22 n-tiles: at least four rounds of
    # up items, so 256-row tiles, several experts ending in a tile of at most
    # 128 rows (paired items); calls of fewer tokens on the same handle take
    # 128-row tiles.  D = 100 ends inside a K stage: the pads of either
    # layout must not show what the other left there, an infinity or a NaN
    # included
    import torch

    rng = np.random.default_rng(60)
    bias = (rng.standard_normal(16) * 0.6).astype(np.float32)
    c = Case(moe, oracle, T=4096, D=100, H=H, Dout=72, E=16, k=2, expert_type=etype, act=act, wdtype="bf16",
             xdtype="bf16", seed=60, router_bias=bias)
    try:
        print(f"256-row tiles {etype} H={H}", flush=True)
        big, loss, res = c.run(training=True)
        w, paired = _up_items(res["counts"], 22)
        ncu = torch.cuda.get_device_properties(0).multi_processor_count
        assert paired > 0 and w > ncu and 0 < 2 * (w % ncu) <= ncu  # the items of the last round are split
        assert tile_heights(lambda: c.run(training=True)) == {256}
        assert tile_heights(lambda: c.run(training=True, T=300)) == {128}
        check_case(c, TOL["bf16"])
        check_case(c, TOL["bf16"], T=300)
        small = c.run(training=True, T=300)[0]
        x = c.x_dev.copy()
        x[::7, 99], x[::5, 3] = 0x7f80, 0x7fc0  # +Inf and NaN bit patterns
        c.dev.forward(np.ascontiguousarray(x), c.xcode, True)
        again = c.run(training=True, T=300)[0]
        assert np.array_equal(again.view(np.uint32), small.view(np.uint32))
        c.dev.forward(np.ascontiguousarray(x[:300]), c.xcode, True)
        again = c.run(training=True)[0]
        assert np.array_equal(again.view(np.uint32), big.view(np.uint32))
    finally:
        c.dev.close()


@pytest.mark.parametrize("n", [600, 700])
def test_expert_forward_256_row_tiles(moe, oracle, n):
    # one expert's rows on such a handle: two full tiles and a paired one of 88
    # rows, or an unpaired one of 188
    c = Case(moe, oracle, T=4096, D=100, H=2816, E=16, k=2, wdtype="bf16", xdtype="bf16", seed=84)
    try:
        print(f"expert_forward 256-row tiles, 22 n-tiles, n={n}", flush=True)
        x = np.ascontiguousarray(c.x[:n])
        y = c.dev.expert_forward(5, x)
        ex = c.ex[5]
        xd = x.astype(np.float64)
        g, u = xd @ ex["w1"].T.astype(np.float64), xd @ ex["w3"].T.astype(np.float64)
        h = _bf16_round(oracle, (g / (1.0 + np.exp(-g))) * u).astype(np.float64)
        err = rel_err(y, h @ ex["w2"].T.astype(np.float64))
        assert err <= TOL["bf16"], err
    finally:
        c.dev.close()


@pytest.mark.parametrize("D,xdtype", [(5, "bf16"), (9, "bf16"), (63, "f32"), (100, "f32"), (513, "bf16"), (1031, "bf16"),
                                      (2052, "f32"), (2055, "bf16")])
def test_permute_rows_of_any_width(moe, oracle, D, xdtype):
    # the tile image's rows: widths below one 16-byte chunk, cut inside a
    # chunk, past one batch of chunks, of rows at 2- and 4-byte alignment
    c = Case(moe, oracle, T=70, D=D, H=64, Dout=64, E=4, k=2, wdtype="bf16", xdtype=xdtype, seed=90 + D)
    try:
        check_case(c, TOL["bf16"])
    finally:
        c.dev.close()
