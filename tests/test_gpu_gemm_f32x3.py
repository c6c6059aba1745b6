"""The fp32 layer on expert segments long enough for the bf16 matrix unit
(three exact bf16 parts per value, six products): against the oracle and, more
tightly, against 64-bit sums, with infinities and NaN as fp32 gives them.

Bound of the error against 64 bits: each of the two GEMMs sums K products with
fp32 rounding, a relative error of about sqrt(K) 2^-25 per output (rounding
errors of random sign on partial sums that grow like sqrt(k)); the layer
combines both: 8 sqrt(K) 2^-25 <= 1.3e-5 at K = 2816, 4.6e-6 at K = 330."""
import numpy as np
import pytest

from kernel_names import kernels_of
from test_gpu_layer import Case, check_case

pytestmark = pytest.mark.gpu


def exact_forward(c, idx, gates):
    x = c.x.astype(np.float64)
    out = np.zeros((c.T, c.Dout))
    act = {"silu": lambda a: a / (1 + np.exp(-a)), "relu": lambda a: np.maximum(a, 0), "identity": lambda a: a,
           "gelu": lambda a: 0.5 * a * (1 + np.tanh(np.sqrt(2 / np.pi) * (a + 0.044715 * a ** 3)))}[c.act]
    for e, w in enumerate(c.ex):
        t, s = np.nonzero(idx == e + 1)
        a = x[t] @ w["w1"].T.astype(np.float64)
        if c.expert_type == "gated":
            y = (act(a) * (x[t] @ w["w3"].T.astype(np.float64))) @ w["w2"].T.astype(np.float64)
        else:
            y = act(a + w["b1"]) @ w["w2"].T.astype(np.float64) + w["b2"]
        np.add.at(out, t, gates[t, s][:, None].astype(np.float64) * y)
    return out


# each layer has 96 tiles of 128 x 128 or more in one of its GEMMs, from where
# on the kernel is chosen
@pytest.mark.parametrize("T,D,H,Dout,E,k,etype,act", [
    (2048, 100, 330, 90, 32, 2, "gated", "silu"),     # partial tiles, pads in every dimension
    (3072, 64, 128, 260, 96, 1, "gated", "gelu"),     # about 32 rows per expert: one row block, two K stages
    (4000, 330, 260, 512, 12, 2, "standard", "gelu"),  # both row blocks, std tiles of 256 columns, biases
    (300, 2816, 64, 64, 2, 2, "standard", "relu"),    # a K split of a small tile grid (88 stages)
    (700, 64, 2816, 40, 2, 1, "gated", "identity"),   # ... of the down GEMM
])
def test_f32x3_layer(moe, oracle, T, D, H, Dout, E, k, etype, act):
    c = Case(moe, oracle, T=T, D=D, H=H, Dout=Dout, E=E, k=k, gate="switch" if k == 1 else "topk", expert_type=etype,
             act=act, wdtype="f32", seed=500 + T)
    try:
        out, _ = check_case(c, 1e-5)
        again, _, res = c.run(training=True)
        assert np.array_equal(out.view(np.uint32), again.view(np.uint32))
        ref = exact_forward(c, res["indices"], res["gates"])
        err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
        assert err <= 8 * np.sqrt(max(D, H)) * 2.0 ** -25, err
    finally:
        c.dev.close()


def test_fp32_kernel_follows_the_calls_rows(moe, oracle):
    # ExpertChoice: the slots a token may hold grow with the handle's
    # max_tokens, the rows of a call do not.  64 tokens choose 4 rows per expert,
    # far below the 32 from which on the bf16 matrix unit takes an fp32 layer;
    # on a handle for 2048 tokens the call has the bits it has on one for 64
    outs = []
    for cap in (64, 2048):
        c = Case(moe, oracle, T=64, D=256, H=512, E=32, k=2, gate="expert_choice", gate_param=2.0, wdtype="f32", seed=71,
                 max_tokens=cap)
        try:
            out, _, res = c.run(training=True)
            assert res["counts"].max() <= 4
            outs.append(out)
        finally:
            c.dev.close()
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


def test_expert_forward_takes_the_layers_kernel(moe, oracle):
    # one expert's rows are as long a segment for moe_expert_forward as in a
    # layer call that gives them all to that expert: the same bits (at sizes
    # where the layer grid's further M tiles change no K split)
    T, D = 1000, 260
    c = Case(moe, oracle, T=T, D=D, H=4096, Dout=40, E=12, k=1, gate="switch", wdtype="f32", seed=72)
    try:
        print("expert_forward against the layer", flush=True)
        x = np.ascontiguousarray(c.x)
        out = c.dev.forward_routed(x, 0, False, np.full((T, 1), 2, np.int32), np.ones((T, 1), np.float32))[0]
        y = c.dev.expert_forward(1, x)
        assert np.array_equal(y.view(np.uint32), out.view(np.uint32))
    finally:
        c.dev.close()


@pytest.mark.parametrize("T,D,H,E,k,etype,act", [
    (4608, 64, 64, 96, 1, "gated", "silu"),     # two stages per sum
    (2048, 128, 256, 64, 2, "standard", "gelu"),
    (1024, 300, 300, 32, 2, "gated", "silu"),   # a partial last stage
    (2400, 480, 448, 12, 2, "gated", "silu"),   # the largest K below the running sums', both row blocks
])
def test_f32x3_small_k(moe, oracle, T, D, H, E, k, etype, act):
    # Small K: as accurate as the fp32 matrix unit (2.0e-7, 1.8e-7 and 2.5e-7 on the
    # first three).  Per GEMM sqrt(K / 32) 2^-25 for the rounded additions of the
    # stages (1.2e-7 at 480) and for each stage's own sum, rounded in several
    # steps, at most 2^-23 of it, random over the stages: about 0.6 x 2^-23; h
    # rounds once more.  Two GEMMs in
    # turn and the gates: below 10 x 2^-25.
    c = Case(moe, oracle, T=T, D=D, H=H, E=E, k=k, gate="switch" if k == 1 else "topk", expert_type=etype, act=act,
             wdtype="f32", seed=700 + D)
    try:
        out, _, res = c.run(training=True)
        ref = exact_forward(c, res["indices"], res["gates"])
        err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
        assert err <= 10 * 2.0 ** -25, err
    finally:
        c.dev.close()


@pytest.mark.parametrize("T,D,H,E,k,etype,act,ran,fp32_unit", [
    (1037, 520, 2731, 6, 2, "gated", "silu", "<0, false>", 8.2e-7),
    (1037, 520, 2731, 6, 2, "standard", "gelu", "<1, false>", 7.0e-7),
])
def test_f32x3_running_sums(moe, oracle, T, D, H, E, k, etype, act, ran, fp32_unit):
    # the up GEMMs of large layers: K of 512 or more, tiles for every CU and none
    # cut into K ranges (22 M tiles of 22 or 11 n-tiles), ragged in every
    # dimension.  Running sums are used where they are no less accurate than the
    # fp32 matrix unit, whose error on the same layers is the bound (5.3e-7 and
    # 3.9e-7 measured)
    c = Case(moe, oracle, T=T, D=D, H=H, E=E, k=k, expert_type=etype, act=act, wdtype="f32", seed=800)
    try:
        out, _ = check_case(c, 1e-5)
        res = c.run(training=True)[2]
        assert "grouped_gemm_f32x3_kernel" + ran in kernels_of(lambda: c.run(training=True))
        ref = exact_forward(c, res["indices"], res["gates"])
        err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
        print(f"error against 64 bits {err:.2e}", flush=True)
        assert err <= fp32_unit, err
        # an infinity, a NaN and a value above bf16's largest in x: their tokens'
        # outputs as fp32 sums give them, the others' bits as they were
        bad = np.ascontiguousarray(c.x)
        o0 = c.dev.forward_routed(bad, 0, False, res["indices"], res["gates"])[0]
        bad = bad.copy()
        bad[5, 519], bad[700, 0], bad[1036, 77] = np.inf, np.nan, 3.4e38
        o = c.dev.forward_routed(bad, 0, False, res["indices"], res["gates"])[0]
        keep = np.ones(T, bool)
        keep[[5, 700, 1036]] = False
        assert np.array_equal(o[keep].view(np.uint32), o0[keep].view(np.uint32))
        assert np.isnan(o[700]).all() and not np.isfinite(o[5]).any()
        if etype == "standard":  # 3.4e38 times the weights is finite, the value's first part is not
            c.x[1036] = bad[1036]
            big = exact_forward(c, res["indices"], res["gates"])[1036]
            assert np.max(np.abs(o[1036] - big)) <= 1e-5 * np.max(np.abs(big))
    finally:
        c.dev.close()


@pytest.mark.parametrize("T,H", [(12800, 96), (200, 6400)])
def test_f32x3_infinities_and_nan(moe, oracle, T, H):
    # values whose parts overflow or are not finite: the outputs they enter
    # are the ones a sequence of fp32 operations gives, the others keep their
    # bits.  Identity experts whose first output columns copy x (w1 = 1 on one
    # input, w2 = 1 on one unit), the rest random.  H = 6400: K ranges.
    D = 64
    c = Case(moe, oracle, T=T, D=D, H=H, E=2, k=1, gate="switch", expert_type="standard", act="identity", wdtype="f32",
             seed=61, max_tokens=T)
    try:
        print(f"f32x3 infinities H={H}", flush=True)
        w1 = np.zeros((H, D), np.float32)
        w1[np.arange(D), np.arange(D)] = 1.0
        w2 = np.zeros((D, H), np.float32)
        w2[np.arange(D), np.arange(D)] = 1.0
        for e in range(2):
            c.dev.set_expert(e, w1, w2, None, np.zeros(H, np.float32), np.zeros(D, np.float32))
        # the caller's routing, every token to expert 1 with gate 1: the gates
        # do not depend on x then
        def forward(x):
            return c.dev.forward_routed(x, 0, False, np.ones((T, 1), np.int32), np.ones((T, 1), np.float32))[0]

        x = np.ascontiguousarray(c.x)
        out = forward(x)
        assert np.array_equal(out, x)
        big = x.copy()
        big[3, :] = 3.4e38     # finite in fp32, above bf16's largest value
        big[4, :] = -3.4028235e38
        o = forward(big)
        assert np.array_equal(o, big)
        bad = x.copy()
        bad[5, 7], bad[6, 9], bad[130, 0] = np.inf, np.nan, -np.inf
        o = forward(bad)
        # an infinity or NaN times the zero weights of a row is NaN, as in fp32
        assert np.isnan(o[6]).all() and o[5, 7] != x[5, 7] and not np.isfinite(o[5, 7])
        keep = np.ones(T, bool)
        keep[[5, 6, 130]] = False
        assert np.array_equal(o[keep], x[keep])
    finally:
        c.dev.close()


@pytest.mark.parametrize("etype,H", [("standard", 4096), ("gated", 2048)])
def test_f32x3_calls_with_infinities_take_their_time(moe, oracle, etype, H):
    # positive weights, so that an infinity in x is one in every output of
    # its row; in one row and in all of them.  Redone sums take about four
    # times a tile's own MFMAs, a part of this host call: 1.4 x its time; one
    # lane per output and one K value after the other took 5 x with one such
    # row, 28 and 38 x with all
    import time

    T, D = 512, 512
    c = Case(moe, oracle, T=T, D=D, H=H, E=2, k=1, gate="switch", expert_type=etype, act="identity", wdtype="f32", seed=63)
    try:
        print(f"f32x3 calls with infinities {etype} H={H}", flush=True)
        for e in range(2):
            w = c.ex[e]
            c.dev.set_expert(e, np.abs(w["w1"]), np.abs(w["w2"]), None if w["w3"] is None else np.abs(w["w3"]), w["b1"], w["b2"])

        def forward(x):
            return c.dev.forward_routed(x, 0, False, 1 + np.arange(T, dtype=np.int32)[:, None] % 2, np.ones((T, 1), np.float32))[0]

        def fastest(x):
            best = 1e9
            for _ in range(6):
                t0 = time.perf_counter()
                forward(x)
                best = min(best, time.perf_counter() - t0)
            return best

        x = np.ascontiguousarray(c.x)
        out, clean = forward(x), fastest(x)
        one, every = x.copy(), x.copy()
        one[5, 300], every[:, 300] = np.inf, np.inf
        for bad in (one, every):
            o, held = forward(bad), fastest(bad)
            rows = np.isinf(bad).any(axis=1)
            assert np.array_equal(o[~rows].view(np.uint32), out[~rows].view(np.uint32))
            assert np.all(o[rows] == np.inf)
            print(f"{rows.sum()} rows: {clean * 1e6:.0f} us, {held * 1e6:.0f} us", flush=True)
            assert held <= 5 * clean, (clean, held)
    finally:
        c.dev.close()


@pytest.mark.parametrize("exp", [-126, -120, -112, -100])
@pytest.mark.parametrize("T,H", [(12800, 96), (200, 6400)])
def test_f32x3_tiny_values(moe, oracle, T, H, exp):
    # values whose low parts are below bf16's smallest: identity experts give
    # them back bit for bit, as fp32 products and sums with zeros do (H = 6400:
    # K ranges)
    D = 64
    c = Case(moe, oracle, T=T, D=D, H=H, E=2, k=1, gate="switch", expert_type="standard", act="identity", wdtype="f32",
             seed=64, max_tokens=T)
    try:
        print(f"f32x3 values of 2^{exp} H={H}", flush=True)
        w1, w2 = np.zeros((H, D), np.float32), np.zeros((D, H), np.float32)
        w1[np.arange(D), np.arange(D)] = 1.0
        w2[np.arange(D), np.arange(D)] = 1.0
        for e in range(2):
            c.dev.set_expert(e, w1, w2, None, np.zeros(H, np.float32), np.zeros(D, np.float32))
        x = np.ascontiguousarray((1 + np.random.default_rng(65).random((T, D))) * 2.0 ** exp).astype(np.float32)
        x[3] = 0.0

        def forward():
            return c.dev.forward_routed(x, 0, False, np.ones((T, 1), np.int32), np.ones((T, 1), np.float32))[0]

        assert any(n.startswith("grouped_gemm_f32x3_kernel") for n in kernels_of(forward))
        assert np.array_equal(forward().view(np.uint32), x.view(np.uint32))
    finally:
        c.dev.close()
