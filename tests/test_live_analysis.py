"""Emitter rules that choose what a kernel holds and its occupancy target (no
GPU needed)."""
import os
import re

import pytest

from openshadinglanguage_amd import groupgen as G
from openshadinglanguage_amd import shadingsys as S


def test_unread_gabor_is_left_out():
    """A Gabor noise whose result reaches no output, closure or branch is
    not emitted (its LDS queues keep the compiler from dropping it); the same
    noise read through a connection, or by a loop condition, is."""
    def source(outputs):
        ss, g = S.build_layered3()
        ss.set_outputs(g, outputs)
        return ss.emit(g)
    assert "gabor(gu_" in source([])  # the closure's color reads it
    ss = S.ShadingSystem()
    ss.load_shader_file("c2_pattern", os.path.join(S.SHADER_DIR, "layered3_pattern.oso"))
    g = ss.ShaderGroupBegin("pattern_only")
    ss.Shader(g, "surface", "c2_pattern", "pattern")
    ss.ShaderGroupEnd(g)
    ss.set_outputs(g, ["pattern.fbm"])
    assert "gabor(gu_" not in ss.emit(g)
    ss.set_outputs(g, ["fbm", "gab"])
    assert "gabor(gu_" in ss.emit(g)
    for op in ("while", "if"):
        o = G.Oso("surface", "cond_" + op)
        o.sym("global", "point", "P")
        o.sym("oparam", "float", "F", "0")
        x, v, c = o.tmp("float"), o.tmp("float"), o.tmp("int")
        o.op("compref", x, "P", o.const("int", 0))
        o.op("noise", v, o.const("string", "gabor"), x)
        if op == "while":
            w = o.op("while", c)
            o.op("gt", c, v, o.const("float", 10.0))
            j = len(o.code)
            o.op("add", "F", "F", x)
            o.code[w][2] = [w + 1, j, len(o.code), len(o.code)]
        else:
            o.op("gt", c, v, o.const("float", 0.0))
            w = o.op("if", c)
            o.op("assign", "F", x)
            o.code[w][2] = [len(o.code), len(o.code)]
        gg = S.build_generated_group(ss, ([("cond_" + op, "surface", o.text())], []),
                                     "cond_" + op, outputs=["F"])
        assert "gabor(gu_" in ss.emit(gg)


def test_gabor_of_a_structure_member_output_is_emitted():
    """An output may be a structure's member, whose name holds a dot."""
    o = G.Oso("surface", "member")
    o.sym("global", "point", "P")
    o.sym("oparam", "float", "out.val", "0")
    o.op("noise", "out.val", o.const("string", "gabor"), "P")
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([("member", "surface", o.text())], []), "member",
                                outputs=["surface.out.val"])
    assert "gabor(gu_" in ss.emit(g)


def _gabor_program(kind):
    """A Gabor noise of 8 impulses per point beside other work."""
    o = G.Oso("surface", "work")
    o.sym("global", "point", "P")
    o.sym("oparam", "float", "F", "0")
    o.sym("oparam", "float", "H", "0")
    gabor = [o.const("string", "gabor"), "P", o.const("string", "impulses"), o.const("float", 8.0)]
    x, c = o.tmp("float"), o.tmp("int")
    o.op("compref", x, "P", o.const("int", 2))
    if "after return" in kind:
        o.op("gt", c, x, o.const("float", 0.5))
        w = o.op("if", c)
        o.op("return")
        o.code[w][2] = [len(o.code), len(o.code)]
    if "branch" in kind:
        o.op("gt", c, x, o.const("float", 0.5))
        w = o.op("if", c)
        o.op("noise", "F", *gabor)
        o.code[w][2] = [len(o.code), len(o.code)]
    else:
        o.op("noise", "F", *gabor)
    noises = {"none": 0, "18": 18, "30": 30, "40": 40, "dead 40": 40, "loop 19": 19, "loop 40": 40,
              "unknown loop": 1, "branch 2": 2, "after return 2": 2}.get(kind, 0)
    if "loop" in kind:
        i = o.sym("local", "int", "i")
        w = o.op("for", c)
        o.op("assign", i, o.const("int", 0))
        j0 = len(o.code)
        n = o.const("int", noises)
        if kind == "unknown loop":
            n = o.tmp("int")
            o.op("assign", n, x)
            j0 = len(o.code)
        o.op("lt", c, i, n)
        j1 = len(o.code)
        o.op("noise", x, o.const("string", "perlin"), "P")
        o.op("add", "H", "H", x)
        j2 = len(o.code)
        o.op("add", i, i, o.const("int", 1))
        o.code[w][2] = [j0, j1, j2, len(o.code)]
    else:
        for _ in range(noises):
            v = o.tmp("float")
            o.op("noise", v, o.const("string", "perlin"), "P")
            if kind != "dead 40":
                o.op("add", "H", "H", v)
    return o.text()


@pytest.mark.parametrize("kind,most", [
    ("none", 49152), ("18", 49152), ("30", 32768), ("40", 8192), ("dead 40", 49152),
    ("loop 19", 32768), ("loop 40", 8192), ("unknown loop", 8192), ("branch", 49152),
    ("branch 2", 8192), ("after return", 49152), ("after return 2", 8192)])
def test_points_of_a_split_launch_by_the_other_work(kind, most):
    """Split launches repeat what the group does besides its Gabor noise, so
    they end earlier the more that is; a Gabor noise that not every point
    evaluates counts 1/32."""
    ss = S.ShadingSystem()
    g = S.build_generated_group(ss, ([("work", "surface", _gabor_program(kind))], []), "work",
                                outputs=["F", "H"])
    assert re.findall(r"split launches: up to (\d+) points", ss.emit(g)) == [str(most)]


def test_occupancy_target_by_kernel():
    """Unset, the target follows the kernel's closures; a set one holds."""
    for mode, want in ((None, 3), ("closure_sample", 3), ("closure_export", 2)):
        ss = S.ShadingSystem()
        if mode:
            ss.attribute(mode, 1)
        ss, g = S.build_mx_layered(ss)
        assert "amdgpu_waves_per_eu(%d)" % want in ss.emit(g), mode
        ss.attribute("gpu_waves_per_eu", 5)
        assert "amdgpu_waves_per_eu(5)" in ss.emit(g)
    ss, g = S.build_layered3()
    assert "amdgpu_waves_per_eu(6)" in ss.emit(g)
