"""Split launches of groups with Gabor noise (few points: four waves share the
cells of 64 points) against launches that give each point its own work-item,
bit for bit: the same points shaded in a call too large to split, and in a
call whose outputs overlap its inputs, which is not split either. Sizes are
the edges of a wave and of the rule; the programs cover every direction mode,
a noise under a branch, and filtered noise with derivatives and a closure."""
import numpy as np
import pytest

import _gsprogs as GS
from openshadinglanguage_amd import shadingsys as S

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MOST = 3 * 64 * 256  # points of the largest split launch
LIMIT = "split launches: up to %d points" % MOST
SIZES = [1, 63, 64, 65, 64 * 21 + 37, MOST]


@pytest.fixture(scope="module")
def dev():
    from openshadinglanguage_amd import check, lib
    check(lib().oslmi_init())
    return torch.device("cuda:0")


def _points(dev):
    """Rows of neighbours and unrelated points, in turn; a few not finite."""
    rng = np.random.default_rng(11)
    n = MOST + 1
    t = np.arange(n) / 64.0
    P = np.stack([t * 3.0, 0.3 + 0.01 * t, rng.uniform(-0.4, 0.4, n)])
    far = (np.arange(n) // 64) % 3 == 1
    P[:, far] = rng.uniform(-40, 40, (3, n))[:, far]
    P[0, 5::997] = np.nan
    return torch.from_numpy(P.astype(np.float32)).to(dev)


def _same(a, b, what):
    assert torch.equal(a.view(torch.int32), b.view(torch.int32)), what


@pytest.mark.parametrize("aniso,impulses", GS.SPECS)
def test_split_matches_whole(dev, aniso, impulses):
    name = "gs_%d_%d" % (aniso, impulses)
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([(name, "surface", GS.program(aniso, impulses))], []), name,
                                outputs=GS.OUTPUTS)
    assert LIMIT in ss.emit(g)
    ss.jit_group(g)
    P = _points(dev)
    zero = {"dPdx": (0.0,) * 3, "dPdy": (0.0,) * 3}

    def shade(p, out):
        ss.execute(g, p.shape[1], dict(zero, P=p), outputs=out)
        torch.cuda.synchronize()
        return out

    ref = shade(P, torch.empty((4, MOST + 1), device=dev))
    for n in SIZES:
        print("gabor split %s: %d points" % (name, n), flush=True)
        p = P[:, -n:].contiguous()
        _same(shade(p, torch.empty((4, n), device=dev)), ref[:, -n:], n)
    # outputs over the inputs: P is planes 1 to 3 of the buffer, and every
    # output of a point is stored after its P has been read
    n = 1381
    buf = torch.empty((4, n), device=dev)
    buf[1:] = P[:, -n:]
    _same(shade(buf[1:], buf), ref[:, -n:], "overlapping")


@pytest.mark.parametrize("n", SIZES)
def test_split_layered3(dev, n):
    """Filtered Gabor noise with derivatives, closure evaluated."""
    ss, g = S.build_layered3()
    assert LIMIT in ss.emit(g)
    ss.jit_group(g)
    d = torch.nn.functional.normalize(torch.randn((3, MOST + 1), device=dev,
                                                  generator=torch.Generator(dev).manual_seed(7)), dim=0)
    P = _points(dev).nan_to_num(0.5)

    def shade(m):
        ev = torch.empty((4, m), device=dev)
        pick = lambda t: t[:, -m:].contiguous()  # noqa: E731
        ss.execute(g, m, {"P": pick(P), "N": pick(d), "dPdx": (1 / 128, 0.0, 0.0),
                          "dPdy": (0.0, 1 / 128, 0.0)}, wo=pick(d), wi=pick(d), eval_out=ev)
        torch.cuda.synchronize()
        return ev

    _same(shade(n), shade(MOST + 1)[:, -n:], n)
