"""What the entry points launch, checked on the CPU against a stand-in for the HIP runtime (hip_recorder.py)."""
from hip_recorder import recorded


def test_sum_and_gate_of_a_data_gradient_whose_kernel_is_refused():
    """sgh_conv_dgrad_add_relu_*: where the kernel that would add and gate cannot be launched, another one forms the data gradient, and
    the sum and the gate are a launch of their own; where it can, it is the last launch."""
    fused, refused = recorded("""
g = conv(2, 64, 8, 8, 64, 1, 1, 1, 1, 0, 0)
need = lib.sgh_conv_workspace_bytes_h(C.byref(g), _lib.SGH_CONV_DGRAD)
def run():
    assert lib.sgh_conv_dgrad_add_relu_f16(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, 5 * SPACE, 6 * SPACE, need, None) == 0
    return kernels()
recorder.recorder_refuse(b"k_pw16")
refused = run()
recorder.recorder_refuse(b"")
answer([run(), refused])
""")
    assert fused[-1] == "k_pw16", fused
    assert "k_pw16" not in refused and "relu_bwd_add" in refused[-1], refused


def test_data_gradient_of_too_many_tiny_planes_is_unsupported():
    """A workgroup per 8 x 32 pixels of an image: 2^24 planes of one pixel are more than a launch can hold (2^32 threads).  They are left
    to the column GEMM, which says that its grid does not hold them either; one plane less is launched."""
    most, beyond = recorded("""
def run(n):
    g = conv(n, 1, 1, 1, 1, 3, 3, 1, 1, 1, 1)
    need = max(lib.sgh_conv_workspace_bytes(C.byref(g), _lib.SGH_CONV_DGRAD), 9 << 26)
    return lib.sgh_conv_dgrad_f32(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, need, None) == _lib.SGH_EUNSUPPORTED, kernels()
answer([run((1 << 24) - 1), run(1 << 24)])
""")
    assert most == [False, ["k_dgrad_few"]] and beyond == [True, []], (most, beyond)
