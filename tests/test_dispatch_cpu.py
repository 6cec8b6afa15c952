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


def test_data_gradient_with_few_input_channels_takes_no_workspace():
    """Layers of k_dgrad_few write no columns: no workspace is asked for, in fp32 none is needed, and the 16-bit passes, which widen
    into theirs, need no more than that; one filter more than it takes, and the columns are there."""
    few, few16, columns = recorded("""
which = _lib.SGH_CONV_DGRAD
g, wider = conv(128, 3, 32, 32, 64, 5, 5, 1, 1, 2, 2), conv(128, 3, 32, 32, 65, 5, 5, 1, 1, 2, 2)
least = lib.sgh_conv_workspace_least_bytes(C.byref(g), which, 0)
rc = lib.sgh_conv_dgrad_f32(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, None, 0, None)
few = [lib.sgh_conv_workspace_bytes(C.byref(g), which), least, rc, kernels()]
need = lib.sgh_conv_workspace_bytes_h(C.byref(g), which)
rc = lib.sgh_conv_dgrad_bf16(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, need, None)
few16 = [need, rc, kernels()]
need = lib.sgh_conv_workspace_bytes(C.byref(wider), which)
rc = lib.sgh_conv_dgrad_f32(C.byref(wider), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, need, None)
columns = [need, rc, kernels(), lib.sgh_conv_dgrad_f32(C.byref(wider), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, need - 4, None) == -2]
answer([few, few16, columns])
""")
    assert few == [0, 0, 0, ["k_dgrad_few"]], few
    tensors = 4 * (128 * 64 * 32 * 32 + 64 * 3 * 25 + 128 * 3 * 32 * 32)   # dy, W and dx in fp32
    assert few16[1] == 0 and few16[2].count("k_dgrad_few") == 1 and few16[0] <= tensors + 4096, few16
    assert columns == [4 * 25 * 3 * 128 * 32 * 32, 0, ["k_igemm", "k_col2im_gather"], True], columns


def test_gates_and_sums_that_overlap_the_result_are_refused():
    """The other branch's gradient, the gate and the result of sgh_conv_dgrad_add_relu_*, the gate and the result of
    sgh_linear_bwd_x_f32: read after parts of the result have been written.  Shared or overlapping they are refused and nothing is launched;
    side by side they are taken."""
    refused, taken = recorded("""
bytes_ = 2 * 64 * 9 * 9 * 2
g = conv(2, 64, 9, 9, 64, 1, 1, 1, 1, 0, 0)
need = lib.sgh_conv_workspace_bytes_h(C.byref(g), _lib.SGH_CONV_DGRAD)
def block(fn, add, x, dx):
    return fn(C.byref(g), SPACE, 2 * SPACE, add, x, dx, 6 * SPACE, need, None), len(kernels())
A, X, D = 3 * SPACE, 4 * SPACE, 5 * SPACE
refused, taken = [], []
for fn in (lib.sgh_conv_dgrad_add_relu_f16, lib.sgh_conv_dgrad_add_relu_bf16):
    refused += [block(fn, D, X, D), block(fn, A, D, D), block(fn, D + bytes_ - 2, X, D), block(fn, A, D - bytes_ + 2, D)]
    taken += [block(fn, D + bytes_, X, D), block(fn, A, D - bytes_, D), block(fn, A, A, D)]
for rows, inner, out in ((33, 70, 50), (3000, 700, 800)):
    linear = lambda gate, dx: (lib.sgh_linear_bwd_x_f32(SPACE, 2 * SPACE, gate, dx, rows, inner, out, None), len(kernels()))
    bytes_ = rows * inner * 4
    refused += [linear(D, D), linear(D + bytes_ - 4, D), linear(D - bytes_ + 4, D)]
    taken += [linear(D + bytes_, D), linear(None, D)]
answer([refused, taken])
""")
    assert all(r == [-1, 0] for r in refused), refused
    assert all(rc == 0 and n > 0 for rc, n in taken), taken


def test_which_16bit_gemm_takes_a_product():
    """Few tiles and a long reduction stay with the split kernel (64-wide tiles would leave most CUs idle), as do many tiles with hardly
    any reduction; many tiles with some, and odd rows, go to the tiled one.  (M, N, K, layouts): measured on both."""
    split = [(256, 1000, 2048, "NN"), (256, 1000, 2048, "NT"), (472, 54, 5911, "NN"), (208, 744, 4304, "NT"), (840, 88, 6296, "NT"),
             (974, 36, 6700, "NN"), (44, 5002, 49, "NT"), (1357, 337, 9, "NT"), (1643, 69, 7633, "TN"), (231, 791, 695, "TN"),
             (857, 62, 3323, "NN")]
    tiled = [(512, 1024, 2048, "NN"), (1024, 1024, 1024, "NN"), (48, 6256, 2536, "NT"), (780, 213, 4336, "NN"), (807, 211, 6728, "NN"),
             (161, 621, 2303, "TT"), (129, 1648, 587, "TT"), (700, 6000, 700, "NT")]
    got = recorded("""
def kernel(M, N, K, layout, pad=0):
    tA, tB = layout[0] == "T", layout[1] == "T"
    lda, ldb = (M if tA else K) + pad, (K if tB else N) + pad
    assert lib.sgh_gemm_bf16(tA, tB, M, N, K, 1.0, SPACE, lda, 2 * SPACE, ldb, 0.0, 3 * SPACE, N, None) == 0
    return kernels()
from test_gpu_half import TILE_EDGES
answer([[kernel(*p) for p in %r], [kernel(*p) for p in %r],
        [kernel(*p, a + b, pad) for p in TILE_EDGES for a in "NT" for b in "NT" for pad in range(4)]])
""" % (split, tiled))
    for products, kernels, name in zip((split, tiled, None), got, ("k_gemm16_split", "k_gemm16_tile", "k_gemm16_tile")):
        wrong = [(p, k) for p, k in zip(products or kernels, kernels) if k != [name]]
        assert not wrong, (name, wrong)


def test_16bit_gemm_of_more_tiles_than_a_launch_holds():
    """The tiled kernel's workgroups are counted in one dimension, 2^24 of 256 threads at most: a short product of 2^18 x 2^18 goes to the
    kernel with two, as do extents below eight; a row of tiles less is tiled."""
    got = recorded("""
def kernel(M, N, K):
    assert lib.sgh_gemm_f16(0, 0, M, N, K, 1.0, SPACE, K, 2 * SPACE, N, 0.0, 3 * SPACE, N, None) == 0
    return kernels()
answer([kernel(1 << 18, 1 << 18, 8), kernel((1 << 18) - 64, 1 << 18, 8), kernel(1 << 18, 4, 8)])
""")
    assert got == [["k_gemm16"], ["k_gemm16_tile"], ["k_gemm16"]], got


def test_strided_forward_passes_are_planned_once():
    """A forward pass of stride 2 looks at the places in an image where its tiles begin, up to 256: host work of a microsecond when it
    is done once per call.  Against the same layer of stride 1, which has none of it, a call took 3.5 times as long with six plans, 1.8
    with one."""
    ratios = recorded("""
import time
def call(s):
    g = conv(13, 64, 15 * s, 15 * s, 128, 3, 3, s, s, 1, 1)
    need = lib.sgh_conv_workspace_bytes(C.byref(g), _lib.SGH_CONV_FWD)
    return lambda p=C.byref(g): lib.sgh_conv_fwd_f32(p, SPACE, 2 * SPACE, None, 3 * SPACE, 4 * SPACE, need, None)
def time_of(f):
    t = time.perf_counter()
    for _ in range(100):
        f()
    t = time.perf_counter() - t
    assert set(kernels()) <= {"k_conv_split", "k_conv_split_weights", "k_conv_split_fixup"}
    return t
plain, strided = call(1), call(2)
answer([min(time_of(strided) for _ in range(15)) / min(time_of(plain) for _ in range(15)) for _ in range(5)])
""")
    assert min(ratios) < 2.5, ratios


def test_strided_weight_gradients_fill_the_chip_where_their_workspace_allows():
    """132 tiles and strips of a layer of stride 2 are 132 workgroups on 256 CUs, or, with room for their partial images, more and shorter
    ones; a workspace for the 132 still runs them, less is refused (the fp32 kernel wants more).  Layers of few tiles have the workgroups
    that they had."""
    full, least, less, few = recorded("""
which = _lib.SGH_CONV_WGRAD
def run(g, size):
    if lib.sgh_conv_wgrad_f32(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, size, None) == -2:   # SGH_EWORKSPACE
        return None
    (name, grid, _), *_rest = launched()
    return "k_wgrad_oct" in name, grid[0]
g = conv(35, 654, 31, 36, 344, 3, 3, 2, 2, 1, 1)
image = 9 * 64 * 64 * 4
few = conv(64, 64, 56, 56, 128, 3, 3, 2, 2, 1, 1)
answer([run(g, lib.sgh_conv_workspace_bytes(C.byref(g), which)) + (lib.sgh_conv_workspace_bytes(C.byref(g), which) // image,),
        run(g, 132 * image), run(g, 132 * image - 4), run(few, lib.sgh_conv_workspace_bytes(C.byref(few), which))])
""")
    assert full[0] and full[1] == full[2] and 400 < full[1] <= 768, full
    assert least == [True, 132], least
    assert less is None and few == [True, 256], (less, few)


def test_which_kernels_take_strided_layers():
    """3x3 weight gradients of stride 2 that the fp32 kernels do in less time stay there: octets or tiles half empty.  Data gradients are the
    split kernel's, whose taps outside dy do not exist whatever the weights are, but for two or three chunks of filters on few tiles.
    (n, c, h, w, k): measured on both."""
    fp32_dgrad = [(5, 131, 9, 11, 31), (2, 64, 20, 22, 40)]
    split_dgrad = [(2, 360, 14, 17, 14), (30, 252, 17, 13, 56), (2, 717, 46, 43, 9), (2, 593, 8, 7, 51), (64, 64, 56, 56, 128)]
    fp32_wgrad = [(98, 84, 16, 17, 380), (90, 731, 8, 7, 904), (69, 42, 89, 67, 116)]
    split_wgrad = [(35, 654, 31, 36, 344), (7, 811, 73, 70, 488), (122, 319, 20, 15, 356), (64, 256, 14, 14, 512)]
    got = recorded("""
def names(which, layers):
    out = []
    for n, c, h, w, k in layers:
        g = conv(n, c, h, w, k, 3, 3, 2, 2, 1, 1)
        need = lib.sgh_conv_workspace_bytes(C.byref(g), which)
        fn = (None, lib.sgh_conv_dgrad_f32, lib.sgh_conv_wgrad_f32)[which]
        assert fn(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, 4 * SPACE, need, None) == 0
        out.append(kernels())
    return out
answer([names(1, %r), names(1, %r), names(2, %r), names(2, %r)])
""" % (fp32_dgrad, split_dgrad, fp32_wgrad, split_wgrad))
    assert not any("k_dgrad_split2" in k for k in got[0]) and all("k_dgrad_split2" in k for k in got[1]), got[:2]
    assert not any("k_wgrad_oct" in k for k in got[2]) and all("k_wgrad_oct" in k for k in got[3]), got[2:]


def test_wavefronts_of_data_gradients_onto_few_channels():
    """Eight where a workgroup has its CU to itself, or nearly, and filters for them; four where the chip is full."""
    got = recorded("""
def threads(n, c, h, w, k, r):
    g = conv(n, c, h, w, k, r, r, 1, 1, r // 2, r // 2)
    assert lib.sgh_conv_dgrad_f32(C.byref(g), SPACE, 2 * SPACE, 3 * SPACE, None, 0, None) == 0
    (_, _, t), = launched()
    return t
answer([threads(2, 4, 16, 13, 64, 5), threads(16, 4, 17, 17, 63, 5), threads(128, 3, 32, 32, 33, 5), threads(128, 3, 32, 32, 32, 5), threads(1, 3, 8, 8, 8, 3),
        threads(15, 4, 57, 78, 10, 3), threads(13, 3, 96, 112, 44, 3), threads(128, 4, 112, 112, 64, 5)])
""")
    assert got == [512, 512, 512, 256, 256, 256, 256, 256], got
