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
