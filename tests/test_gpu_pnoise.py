"""GPU parity of periodic and vector noise in emitted kernels: pnoise /
psnoise with and without a name (periodic perlin, cell, hash), the periodic
gabor (pgabor / pgabor3) and the vector gabor (gabor3), in 1-4 dimensions
with float and color results, against the oracle's interpreter, over
unrelated points with periods of their own. The gabor programs also over
neighbouring points, whose waves scan their cells together (periods alike in
the launch, in a wave, or in neither), in a launch that shares points' cells
among waves and in one too large for that. Bar: bit for bit (the emitted code
evaluates the interpreter's IEEE operations in the same order)."""
import numpy as np
import pytest

import _oracle as O
import _pnprogs as PN
from openshadinglanguage_amd import shadingsys as S

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from openshadinglanguage_amd import check, lib
    check(lib().oslmi_init())
    return torch.device("cuda:0")


@pytest.mark.parametrize("k", range(len(PN.SPECS)), ids=[p[0] for p in PN.SPECS])
def test_periodic_noise_programs_match_interpreter(dev, k):
    name, text = PN.programs()[k]
    n = 2000 if "gabor" in name else 20000
    inp = PN.inputs(n, 90 + k)
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([(name, "surface", text)], []), name, outputs=PN.OUTPUTS)
    ss.jit_group(g)
    assert ss.output_planes(g) == 16
    glob = {key: torch.from_numpy(np.ascontiguousarray(inp[key])).to(dev)
            for key in ("P", "N", "dPdu", "dPdv")}
    glob.update({"dPdx": (0.0, 0.0, 0.0), "dPdy": (0.0, 0.0, 0.0)})
    out = torch.full((16, n), -7.0, device=dev)
    print("periodic noise %s: %d points" % (name, n), flush=True)
    ss.execute(g, n, glob, outputs=out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    gr = O.Group([(name, "surface", text)], [])
    for d in range(1, 5):
        gr.outputs("F%d" % d, "C%d" % d)
        ref, _, _ = O.group_run_ex(gr, inp["P"], inp["N"], np.zeros((3, n), np.float32),
                                   dPdu=inp["dPdu"], dPdv=inp["dPdv"], nthreads=8)
        np.testing.assert_array_equal(got[d - 1], ref[0], err_msg="%s F%d" % (name, d))
        c0 = 4 + 3 * (d - 1)
        np.testing.assert_array_equal(got[c0:c0 + 3], ref[1:4], err_msg="%s C%d" % (name, d))


N = 64 * 21 + 37  # the last wave is partly filled


def _neighbours(periods):
    """A row of points, about four cells along x a wave."""
    rng = np.random.default_rng(17)
    t = np.arange(N) / 64.0
    choices = np.array([0.5, 1.0, 2.0, 3.0, 3.5, 4.0, 7.25], np.float32)
    inp = {"P": np.stack([t * 3.0 - 20.0, 0.3 + 0.01 * t, rng.uniform(-0.4, 0.4, N)]),
           "dPdu": np.zeros((3, N))}
    for key in ("N", "dPdv"):
        if periods == "same":
            inp[key] = np.tile(rng.choice(choices, (3, 1)), (1, N))
        elif periods == "wave":
            inp[key] = np.repeat(rng.choice(choices, (3, N // 64 + 1)), 64, axis=1)[:, :N]
        else:
            inp[key] = rng.choice(choices, (3, N))
    return {k: np.ascontiguousarray(v, np.float32) for k, v in inp.items()}


@pytest.mark.parametrize("copies", [1, 36], ids=["split", "whole"])
@pytest.mark.parametrize("prog,periods", [("pn_gabor", "same"), ("pn_gabor", "wave"),
                                          ("pn_gabor", "varying"), ("n_gabor3", "same")])
def test_gabor_of_neighbouring_points_matches_interpreter(dev, prog, periods, copies):
    """36 copies of the points are more than a split launch takes."""
    text = dict(PN.programs())[prog]
    inp = _neighbours(periods)
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([(prog, "surface", text)], []), prog, outputs=PN.OUTPUTS)
    ss.jit_group(g)
    n = N * copies
    glob = {key: torch.from_numpy(np.tile(v, (1, copies))).to(dev) for key, v in inp.items()}
    glob.update({"dPdx": (0.0, 0.0, 0.0), "dPdy": (0.0, 0.0, 0.0)})
    out = torch.full((16, n), -7.0, device=dev)
    print("gabor of neighbours %s, periods %s: %d points" % (prog, periods, n), flush=True)
    ss.execute(g, n, glob, outputs=out)
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(16, copies, N)
    gr = O.Group([(prog, "surface", text)], [])
    for d in range(1, 5):
        gr.outputs("F%d" % d, "C%d" % d)
        ref, _, _ = O.group_run_ex(gr, inp["P"], inp["N"], np.zeros((3, N), np.float32),
                                   dPdu=inp["dPdu"], dPdv=inp["dPdv"], nthreads=8)
        c0 = 4 + 3 * (d - 1)
        for c in range(copies):
            np.testing.assert_array_equal(got[d - 1, c], ref[0], err_msg="F%d copy %d" % (d, c))
            np.testing.assert_array_equal(got[c0:c0 + 3, c], ref[1:4], err_msg="C%d copy %d" % (d, c))
