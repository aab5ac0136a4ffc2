"""The streamed-weight fp16 convolutions at the edges of their tiles: every
tile pinned in turn, and the built-in choice, against the 128-row tile kernel,
which stages its operands quite differently and sums in the same order, so the
outputs are the same bits. Row counts are below, at and one past 32, 64, 128
and 192; boards are one column wide, one row high, rectangular, or wider than
19; channel counts give one to twelve 32-channel chunks and one or several
column tiles."""
import dataclasses

import numpy as np
import pytest

from katago_amd import modelgen, nn

pytestmark = pytest.mark.gpu

TILE_64 = 11  # ConvVariant in kgh_common.h
STREAM = [25, 26, 27, 28, 29, 30]
BOARDS = [(1, 31, 1), (32, 1, 1), (3, 1, 11), (7, 3, 3), (1, 8, 8), (13, 5, 1), (127, 1, 1), (1, 16, 8), (3, 43, 1), (1, 19, 10),
          (3, 8, 8), (1, 3, 64), (1, 64, 4), (2, 19, 19), (5, 9, 13), (40, 9, 9)]  # batch, x, y


def _regular(c):
    return modelgen.Arch("stream%d" % c, 15, c, c, 32, ["regular", "regulargpool"], 16, 16, 32, 48, "ACTIVATION_RELU",
                         residual_gain=0.5)


def _nbt(t, m):
    return modelgen.Arch("stream%d-%d" % (t, m), 15, t, m, 32, ["bottlenest2", "bottlenest2gpool"], 16, 16, 32, 48,
                         "ACTIVATION_MISH", residual_gain=0.5)


def _block(c):
    return modelgen.Arch("block%d" % c, 15, c, c, 32, ["regular"], 16, 16, 32, 48, "ACTIVATION_RELU", residual_gain=0.5)


TRANSFORMER = modelgen.Arch("streamtflrs", 17, 128, 128, 32, ["attention", "ffn"], 16, 16, 32, 48, "ACTIVATION_SILU", heads=2,
                            kv_heads=2, q_head_dim=64, v_head_dim=64, ffn_c=192, learnable_rope=True, trunk_rmsnorm=True)


@pytest.mark.parametrize("arch", [_regular(64), _regular(320), _nbt(128, 64), _nbt(384, 192), TRANSFORMER], ids=lambda a: a.name)
def test_every_tile_gives_the_tile_kernels_bits(model_dir, arch):
    lm = nn.LoadedModel(modelgen.write_model(arch, 57, f"{model_dir}/{arch.name}.bin"))
    model = nn.DeviceModel(lm, use_fp16=True)
    for n, x, y in BOARDS:
        h = nn.DeviceHandle(model, n, x, y)
        sp, gl = modelgen.synthetic_inputs(9, n, x, y, board_sizes=((x, y), (max(x - 1, 1), y)))
        rows = (sp, gl, np.zeros(n, np.int32), np.zeros(n, np.float32))
        dev = [nn.DeviceBuffer.from_array(r) for r in rows]
        out = nn.DeviceBuffer(n * h.row_floats * 4)
        shapes = [l.split()[:8] for l in h.autotune(1).splitlines() if l.strip()]

        def forward(variant):
            h.set_tuning("".join(" ".join(s) + f" {variant}\n" for s in shapes))
            h.forward_device(n, *[b.ptr for b in dev], out.ptr)
            h.synchronize()
            return out.to_array(np.float32, (n, h.row_floats))

        want = forward(TILE_64)
        assert np.isfinite(want).all()
        for v in [0] + STREAM:
            assert np.array_equal(forward(v), want), (n, x, y, v)
        h.close()


# Channels, then (boards, side, what the kernel's name holds) on both sides of
# the lines that the built-in choice draws for 3x3 convs.
CHOICES = [
    (64, [(160, 19, "128x64 tiles"), (192, 19, "192x64 tiles")]),
    (192, [(256, 18, "128x64 tiles"), (284, 18, "convTapWindowKernel<3x3 fp16, BN=192")]),
    (256, [(64, 19, "192x64 tiles"), (80, 19, "BN=128, one board"), (200, 13, "192x64 tiles"), (256, 13, "convTapWindowKernel<3x3 fp16, BN=128")]),
    (320, [(80, 19, "192x64 tiles"), (96, 19, "BN=64, one board")]),
    (384, [(14, 19, "128x64 tiles"), (16, 19, "half a board per workgroup, 32-row"), (24, 19, "128x64 tiles"), (32, 19, "BN=64, one board"),
           (48, 19, "BN=128, one board"), (150, 13, "128x64 tiles"), (200, 13, "convTapWindowKernel<3x3 fp16, BN=192")]),
    (448, [(36, 19, "BN=64, one board"), (40, 19, "128x64 tiles"), (56, 19, "BN=64, one board")]),
    (512, [(8, 19, "64x64 tiles"), (16, 19, "half a board per workgroup, 32-row"), (60, 13, "64x64 tiles"),
           (80, 13, "convTapWindowKernel<3x3 fp16, BN=128")]),
    (768, [(2, 19, "32x64 tiles"), (8, 19, "half a board per workgroup, 32-row"), (22, 19, "BN=128, one board"),
           (32, 18, "convTapWindowKernel<3x3 fp16, BN=128"), (44, 19, "BN=192, one board")]),
    (832, [(20, 19, "half a board per workgroup, 96-row")]),
    (1024, [(16, 13, "32x64 tiles"), (20, 13, "convTapWindowKernel<3x3 fp16, BN=128"), (3, 25, "convMfmaKernel")]),
]


def _run(model, n, x, kind):
    """A forward by the built-in choice: handle, outputs, a function that runs
    it again, and the kernels of the kind's launches by name."""
    h = nn.DeviceHandle(model, n, x, x)
    sp, gl = modelgen.synthetic_inputs(9, n, x, x, board_sizes=(x, x - 1))
    dev = [nn.DeviceBuffer.from_array(r) for r in (sp, gl, np.zeros(n, np.int32), np.zeros(n, np.float32))]
    out = nn.DeviceBuffer(n * h.row_floats * 4)

    def forward():
        h.forward_device(n, *[b.ptr for b in dev], out.ptr)
        h.synchronize()
        return out.to_array(np.float32, (n, h.row_floats))

    h.set_profiling(True)
    got = forward()
    launches = {r[4]: r[1] for r in h.profile_kernels() if r[0] == kind}
    h.set_profiling(False)
    return h, got, forward, launches


@pytest.mark.parametrize("c,choices", CHOICES, ids=lambda v: str(v) if isinstance(v, int) else "")
def test_built_in_choice_for_3x3_convs(model_dir, c, choices):
    """The kernel that measured fastest runs, and gives the tile kernel's bits."""
    lm = nn.LoadedModel(modelgen.write_model(_block(c), 57, f"{model_dir}/block{c}.bin"))
    model = nn.DeviceModel(lm, use_fp16=True)
    for n, x, kernel in choices:
        h, got, forward, launches = _run(model, n, x, 0)
        assert any(kernel in k for k in launches), (n, x, kernel, launches)
        h.set_tuning("".join(f"3 3 {k} {c} {n * x * x} 0 {r} 0 {TILE_64}\n" for k in (32, c) for r in (0, 1)))
        assert np.array_equal(forward(), got), (n, x, kernel)
        h.close()


T768 = dataclasses.replace(modelgen.transformer_d384(), name="t2d768", trunk_c=768, mid_c=768, heads=12, kv_heads=12, ffn_c=2048,
                           blocks=["attention", "ffn"])
T384 = dataclasses.replace(modelgen.transformer_d384(), name="t2d384", blocks=["attention", "ffn"])


@pytest.mark.parametrize("arch,cases", [
    # (boards, side, launches of the streamed kernel, of those on 64-row tiles):
    # post convs of 192 input channels always, pre convs of 384 up to 4400
    # tiles, the heads' conv.
    (_nbt(384, 192), [(16, 19, 5, 2), (128, 19, 5, 2), (160, 19, 3, 2)]),
    # every GEMM up to a million of tiles times K, which leaves out the gated one;
    # from 24 tiles of 192 rows no gated one nor K = 1024, [Q|K|V] up
    # to 4400 tiles, the masked residual up to 2200; the heads' conv.
    (T384, [(4, 19, 5, 0), (12, 19, 4, 0), (16, 19, 3, 0), (32, 19, 2, 0), (40, 19, 1, 0)]),
    # wide GEMMs: the gated one from two boards, [Q|K|V] and linear2 from eight
    # and the output projection from twelve are past a million.
    (T768, [(2, 19, 4, 0), (8, 19, 2, 0), (12, 19, 1, 0)]),
], ids=["nbt", "transformer", "wide-transformer"])
def test_built_in_choice_for_1x1_convs(model_dir, arch, cases):
    lm = nn.LoadedModel(modelgen.write_model(arch, 57, f"{model_dir}/{arch.name}-1x1.bin"))
    model = nn.DeviceModel(lm, use_fp16=True)
    for n, x, streamed, rows64 in cases:
        h, got, forward, launches = _run(model, n, x, 1)
        count = lambda name: sum(v for k, v in launches.items() if k.startswith("convStreamKernel") and name in k)
        assert (count(""), count("64x64")) == (streamed, rows64), (n, x, launches)
        h.set_tuning("")
        shapes = [l.split()[:8] for l in h.autotune(1).splitlines() if l.startswith("1 1 ")]
        h.set_tuning("".join(" ".join(s) + f" {TILE_64}\n" for s in shapes))
        assert np.array_equal(forward(), got), (n, x)
        h.close()
