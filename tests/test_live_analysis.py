"""Emitter rules that choose what a kernel holds and its occupancy target (no
GPU needed)."""
import os

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
