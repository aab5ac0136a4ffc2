"""The streamed-weight fp16 convolutions at the edges of their tiles: every
tile pinned in turn, and the built-in choice, against the 128-row tile kernel,
which stages its operands quite differently and sums in the same order, so the
outputs are the same bits. Row counts are below, at and one past 32, 64, 128
and 192; boards are one column wide, one row high, rectangular, or wider than
19; channel counts give one to twelve 32-channel chunks and one or several
column tiles."""
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
