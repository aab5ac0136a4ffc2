"""fp32 convolutions on bf16 matrix cores at the edges of their tiles: row
counts below, at and past 32, 64 and 96, on narrow, flat and square boards,
channel counts that give uneven and empty K groups (two to 24 16-channel
chunks) and column tiles of 32 and 64, through whole nets against the
oracle; and the same bits for a row on every tile."""
import numpy as np
import pytest

from katago_amd import modelgen, nn
from test_gpu_conv_stream import TRANSFORMER, _nbt, _regular
from test_gpu_parity import _run_parity

pytestmark = pytest.mark.gpu

NARROW = modelgen.Arch("narrowtflrs", 17, 48, 48, 16, ["attention", "ffn"], 16, 16, 32, 48, "ACTIVATION_SILU", heads=2, kv_heads=2,
                       q_head_dim=32, v_head_dim=32, ffn_c=96, learnable_rope=True, trunk_rmsnorm=True)
NETS = [NARROW, _regular(80), _regular(96), _nbt(384, 192), TRANSFORMER]


def _file(model_dir, arch):
    return modelgen.write_model(arch, 91, f"{model_dir}/{arch.name}-fp32.bin.gz")


@pytest.mark.parametrize("nn_x,nn_y", [(2, 2), (15, 2), (2, 16), (11, 3), (9, 7), (8, 8), (13, 5), (19, 5), (6, 16), (7, 14), (19, 19)], ids=str)
@pytest.mark.parametrize("arch", NETS, ids=lambda a: a.name)
def test_edges_match_oracle(model_dir, arch, nn_x, nn_y):
    """Tolerances are _compare's fp32 bounds (1e-3 absolute on the raw
    outputs; products are exact to 2^-24 of their terms, as in fp32)."""
    _run_parity(_file(model_dir, arch), False, 1, board_sizes=((nn_x, nn_y),), label=f"fp32 {nn_x}x{nn_y}", nn_x=nn_x, nn_y=nn_y)


@pytest.mark.parametrize("arch", [_regular(64), _nbt(384, 192), TRANSFORMER, NARROW], ids=lambda a: a.name)
def test_rows_do_not_depend_on_batch(model_dir, arch):
    """Batches whose convolutions run on 32-, 64- and 96-row tiles and with K
    or columns over the waves."""
    h = nn.ComputeHandle(nn.ComputeContext(nn.LoadedModel(_file(model_dir, arch)), use_fp16=False), max_batch=60)
    sp, gl = modelgen.synthetic_inputs(5, 60, board_sizes=(19, 9))
    want = h.get_output(sp, gl)
    for n in (1, 7, 13, 30, 46):
        got = h.get_output(sp[:n], gl[:n])
        for k in want:
            assert np.array_equal(got[k], want[k][:n]), (n, k)
