"""Host-buffer calls whose x, out and routing rows pass through the handle's
pinned memory (256 KB each) and calls that are too large for it: both sides of
the limit against the oracle, mixed on one handle."""
import numpy as np
import pytest

from test_gpu_layer import Case, check_case, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,Dout,Ts", [
    (1024, 1024, (64, 65, 1, 64)),  # 262144 bytes of x and of out, one row more, one row
    (2048, 40, (32, 33, 32)),       # x at and past the limit, out far below
    (40, 2048, (33, 32, 33)),       # out past and at the limit, x far below
])
def test_forward_around_the_pinned_size(moe, oracle, D, Dout, Ts):
    c = Case(moe, oracle, T=max(Ts), D=D, H=96, Dout=Dout, E=6, k=2, wdtype="f32", seed=700 + D)
    try:
        for T in Ts:
            print(f"host forward T={T} D={D} Dout={Dout}", flush=True)
            check_case(c, 1e-5, T=T)
    finally:
        c.dev.close()


def test_decode_around_the_pinned_size(moe, oracle):
    c = Case(moe, oracle, T=130, D=512, H=128, E=6, k=2, wdtype="f32", seed=710, max_tokens=130)
    try:
        for n in (128, 129, 1, 130):  # 262144 bytes of x and of out at 128 tokens
            print(f"host decode n={n}", flush=True)
            x = np.ascontiguousarray(c.x[:n])
            out, logits, idx, gates = c.dev.decode(x)
            ref, ridx, rgates, _ = oracle.decode_ffn(x, c.wr, c.ex, k=2, logits=logits)
            assert np.array_equal(idx, ridx) and np.array_equal(gates.view(np.uint32), rgates.view(np.uint32))
            assert rel_err(out, ref) <= 1e-5
    finally:
        c.dev.close()
