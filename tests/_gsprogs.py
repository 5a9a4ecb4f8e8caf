"""Programs of the Gabor scan's parity test."""
from openshadinglanguage_amd import groupgen as G

SPECS = [(0, 16), (1, 1), (1, 32), (2, 8)]  # direction mode, impulses
OUTPUTS = ["F1", "F2", "F3", "F4"]


def program(aniso, impulses):
    """F1..F3: the noise in 1-3 dimensions; F4: in 2 dimensions, only where
    P[2] > 0."""
    o = G.Oso("surface", "gs_%d_%d" % (aniso, impulses))
    o.sym("global", "point", "P")
    for k in range(1, 5):
        o.sym("oparam", "float", "F%d" % k, "0")
    px, py, pz = o.tmp("float"), o.tmp("float"), o.tmp("float")
    o.sym("oparam", "color", "C", "0 0 0")
    for k, t in enumerate((px, py, pz)):
        o.op("compref", t, "P", o.const("int", k))
    opts = [o.const("string", "do_filter"), o.const("int", 0), o.const("string", "anisotropic"),
            o.const("int", aniso), o.const("string", "direction"), o.const("vector", 1.0, 0.5, 0.25),
            o.const("string", "impulses"), o.const("float", float(impulses))]
    name = o.const("string", "gabor")
    o.op("noise", "F1", name, px, *opts)
    o.op("noise", "F2", name, px, py, *opts)
    o.op("noise", "F3", name, "P", *opts)
    cond = o.tmp("int")
    o.op("gt", cond, pz, o.const("float", 0.0))
    i_if = o.op("if", cond)
    o.op("noise", "F4", name, px, py, *opts)
    o.code[i_if][2] = [len(o.code), len(o.code)]
    return o.text()


def exp_program():
    """E = exp(P[0])."""
    o = G.Oso("surface", "exp_ends")
    o.sym("global", "point", "P")
    o.sym("oparam", "float", "E", "0")
    x = o.tmp("float")
    o.op("compref", x, "P", o.const("int", 0))
    o.op("exp", "E", x)
    return o.text()


def programs():
    return [("gs_%d_%d" % s, program(*s), OUTPUTS) for s in SPECS] + [
        ("exp_ends", exp_program(), ["E"])]
