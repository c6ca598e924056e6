"""GPU parity of MTGP32 over call lengths: the kernel runs whole turns of its ring (four
block-steps), then single steps, and leaves the ring at any of the four phases for the next
call.  Whole numbers equal the oracle's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from rocrand_amd import rocrand as R  # noqa: E402

USE = 512 * 256  # words of one block-step of all generators


def _call(g, kind, n):
    dtype = {"u32": torch.uint32, "u8": torch.uint8}.get(kind, torch.float64)
    buf = torch.zeros(n, dtype=dtype, device="cuda")
    if kind == "uniform_f64":
        g.uniform(buf)
    elif kind == "normal_f64":
        g.normal(buf, 0.0, 1.0)
    else:
        g.generate(buf)
    torch.cuda.synchronize()
    return buf


@pytest.mark.parametrize("calls", [
    [("u32", k * USE) for k in (1, 2, 3, 4, 5)],  # from every phase to every other
    [("u32", n) for n in (1, USE - 1, 7 * USE + 255, 256, 9 * USE + 257)],  # partial blocks, an extra use
    # one, two and four steps a vec, each begun at an odd phase
    [("u32", 3 * USE), ("uniform_f64", 3 * USE), ("u32", 1), ("normal_f64", 6 * USE), ("u8", 11 * USE + 1), ("u32", 257)],
], ids=["steps", "ragged", "kinds"])
def test_mtgp32_over_calls(calls):
    g, want = R.PRNG(R.MTGP32), O.OracleGen(O.MTGP32, seed=99)
    g.seed = 99
    for kind, n in calls:
        print(f"case mtgp32 {kind} n={n}", flush=True)
        buf = _call(g, kind, n)
        st, w = want.generate(kind, n, addr=buf.data_ptr())
        assert st == 0
        if kind != "normal_f64":  # its words are checked by the calls after it
            assert np.array_equal(buf.cpu().numpy(), w)
