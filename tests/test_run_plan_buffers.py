"""Which buffer a scatter_add of a planned function adds into: a splat
constant that nothing else uses or names is filled there and added into where
it is; any other input (an argument, a constant read again, one that a reshape
also names) is copied first, so that it keeps its value.  And that a program's
plan follows the f32 GEMM mode that is set at the time of the call.
"""
import pytest

import nova_run

_FILL = "%b = nova.constant {value = dense<0.0> : tensor<8x4xf32>} : tensor<8x4xf32>\n"
_ADD = ("%r = nova.scatter_add {src}, %i, %s : tensor<8x4xf32>, tensor<3xi32>, tensor<3x4xf32>"
        " -> tensor<8x4xf32>\n")
_RESHAPE = "%{to} = nova.reshape %{frm} : tensor<{a}xf32> -> tensor<{b}xf32>\n"


def _program(body, ret, rets):
    return ("func.func @f(%a: tensor<8x4xf32>, %i: tensor<3xi32>, %s: tensor<3x4xf32>) -> "
            f"({rets}) {{\n{body}return {ret} : {rets}\n}}\n")


@pytest.mark.parametrize("body,ret,rets,copies", [
    (_FILL + _ADD.format(src="%b"), "%r", "tensor<8x4xf32>", 0),
    (_ADD.format(src="%a"), "%r", "tensor<8x4xf32>", 1),
    (_FILL + _ADD.format(src="%b"), "%r, %b", "tensor<8x4xf32>, tensor<8x4xf32>", 1),
    (_FILL + _RESHAPE.format(to="c", frm="b", a="8x4", b="32") + _ADD.format(src="%b"),
     "%r, %c", "tensor<8x4xf32>, tensor<32xf32>", 1),
    (_FILL + _RESHAPE.format(to="c", frm="b", a="8x4", b="8x4") + _ADD.format(src="%c"),
     "%r, %b", "tensor<8x4xf32>, tensor<8x4xf32>", 1),
], ids=["sole_use", "argument", "returned_too", "reshaped_before", "reshape_is_the_input"])
def test_scatter_add_copies_an_input_that_is_read_again(body, ret, rets, copies):
    plan = nova_run.Program(_program(body, ret, rets)).plan("f")
    assert plan.count("nova.scatter_add input -> hipMemcpyAsync") == copies, plan
    assert plan.count("_mlir_ciface_nova_hip_scatter_add_f32") == 1


def test_plan_follows_the_f32_gemm_mode():
    p = nova_run.Program(
        "func.func @f(%a: tensor<8x4xf32>, %b: tensor<4x8xf32>) -> tensor<8x8xf32> {\n"
        "%r = nova.matmul %a, %b : tensor<8x4xf32>, tensor<4x8xf32> -> tensor<8x8xf32>\n"
        "return %r : tensor<8x8xf32>\n}\n")
    exact = p.plan("f")
    p.set_f32_gemm(nova_run.F32_GEMM_MFMA)
    mfma = p.plan("f")
    assert mfma != exact
    p.set_f32_gemm(nova_run.F32_GEMM_EXACT)
    assert p.plan("f") == exact
    assert p.args("f") == p.args("f") and p.results("f")[0][1] == (8, 8)
    p.args("f").clear()   # what a caller does to a list it was given stays with it
    assert len(p.args("f")) == 2
