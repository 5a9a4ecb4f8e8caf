"""GPU parity of the Gabor impulse scan's two forms (per wave over a small
box of cells, per lane otherwise) and of the drain of its queues, against
the oracle's interpreter, bit for bit: boxes at and beyond the per-wave
limits, lattice planes, partly filled waves, a noise under a branch, few and
many impulses (the most fill a queue several times), every direction mode,
1D to 3D, lanes with NaN or infinite coordinates, in a split launch and in
one too large to be split. Also exp() at the ends of
its range, where the result is formed by one scaling."""
import numpy as np
import pytest

import _gsprogs as GS
import _oracle as O
from openshadinglanguage_amd import shadingsys as S

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N = 64 * 21 + 37  # the last wave is partly filled
# copies of the points: in a launch that shares 64 points' cells among four
# waves, and in one too large for that
COPIES = {"split": 1, "whole": 36}


@pytest.fixture(scope="module")
def dev():
    from openshadinglanguage_amd import check, lib
    check(lib().oslmi_init())
    return torch.device("cuda:0")


def _inputs(kind):
    rng = np.random.default_rng(5)
    t = np.arange(N) / 64.0
    if kind == "row":        # about four cells along x a wave
        P = np.stack([t * 3.0, 0.3 + 0.01 * t, rng.uniform(-0.4, 0.4, N)])
    elif kind == "sparse":   # the same, one or two lanes of a wave in the branch
        P = np.stack([t * 3.0, 0.3 + 0.01 * t, np.where(np.arange(N) % 37 == 0, 0.2, -0.2)])
    elif kind == "wide":     # about eight cells a wave: on both sides of the limit
        P = np.stack([t * 4.9, 1.7 * t, 0.2 * np.sin(t)])
    elif kind == "lattice":  # exactly on cell corners, and one step beside them
        cell = np.float32(0.7862812876701355)
        P = np.stack([np.round(t * 4) * cell, np.round(t) * cell, np.zeros(N)])
        P = np.where(np.arange(N) % 3 == 1, np.nextafter(P, 9, dtype=np.float64), P)
    else:                    # unrelated points, a few of them not finite
        P = rng.uniform(-40, 40, (3, N))
        P[0, 5::97] = np.nan
        P[1, 17::89] = np.inf
    return np.ascontiguousarray(P.astype(np.float32))


@pytest.mark.parametrize("copies", COPIES.values(), ids=COPIES.keys())
@pytest.mark.parametrize("kind", ["row", "sparse", "wide", "lattice", "far"])
@pytest.mark.parametrize("aniso,impulses", GS.SPECS)
def test_scan_matches_interpreter(dev, kind, aniso, impulses, copies):
    text = GS.program(aniso, impulses)
    name = "gs_%d_%d" % (aniso, impulses)
    P = _inputs(kind)
    outs = GS.OUTPUTS
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([(name, "surface", text)], []), name, outputs=outs)
    ss.jit_group(g)
    n = N * copies
    out = torch.full((4, n), -7.0, device=dev)
    print("gabor scan %s %s: %d points" % (kind, name, n), flush=True)
    ss.execute(g, n, {"P": torch.from_numpy(np.tile(P, (1, copies))).to(dev), "dPdx": (0.0,) * 3,
                      "dPdy": (0.0,) * 3}, outputs=out)
    torch.cuda.synchronize()
    gr = O.Group([(name, "surface", text)], [])
    zero = np.zeros((3, N), np.float32)
    got = out.cpu().numpy().reshape(4, copies, N)
    for j, out_name in enumerate(outs):
        gr.outputs(out_name, "C")
        ref, _, _ = O.group_run_ex(gr, P, zero, zero, nthreads=8)
        for c in range(copies):
            np.testing.assert_array_equal(got[j, c], ref[0], err_msg="%s copy %d" % (out_name, c))


def test_exp_range_ends(dev):
    """exp() where it overflows, underflows to subnormals and to zero."""
    ends = np.array([88.72283935546875, 88.722846984863281, 89, 129, 200, 201, 1e30, np.inf,
                     -87.3365478515625, -103.97208404541016, -103.97209167480469, -104, -1e30,
                     -np.inf, np.nan, 0.0, -0.0], np.float32)
    xs = np.concatenate([ends, np.linspace(-104.5, -86, 4000), np.linspace(-3, 3, 1000),
                         np.linspace(88, 89, 500)]).astype(np.float32)
    P = np.ascontiguousarray(np.stack([xs, xs, xs]))
    n = len(xs)
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([("exp_ends", "surface", GS.exp_program())], []), "exp_ends",
                                outputs=["E"])
    ss.jit_group(g)
    out = torch.full((1, n), -7.0, device=dev)
    ss.execute(g, n, {"P": torch.from_numpy(P).to(dev)}, outputs=out)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy()[0], O.omath("exp", xs))
