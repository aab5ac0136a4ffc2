"""fp32 attention on the matrix cores at the edges of its tiles: key counts
below, at and one past a 32-key tile, a 64-key chunk and a 128-query
workgroup, masked boards, grouped and shared kv heads, every head shape the
kernel is built for, through whole nets against the oracle."""
import dataclasses

import numpy as np
import pytest

import torch_reference
from katago_amd import modelgen, nn
from test_gpu_parity import _run_parity, _tiny_transformer

pytestmark = pytest.mark.gpu

HEADS = [(2, 2, 32, 32, 64), (4, 2, 32, 16, 64), (2, 1, 64, 64, 128)]


def _model(model_dir, heads, kv, dq, dv, c):
    arch = _tiny_transformer(heads, kv, dq, dv, c, True, True)
    return modelgen.write_model(arch, 31 + heads + dq, f"{model_dir}/{arch.name}-edges.bin.gz")


@pytest.mark.parametrize("nn_x,nn_y,boards", [(5, 5, (5, 4)), (8, 4, ((8, 4), 3)), (8, 8, (8, 5)), (13, 5, ((13, 5), 5)), (16, 8, ((16, 8), 7)),
                                              (19, 7, ((19, 7), 6)), (19, 19, (19, 9))], ids=lambda v: str(v))
@pytest.mark.parametrize("heads", HEADS, ids=["mha-q32v32", "gqa-q32v16", "mqa-q64v64"])
def test_key_counts_match_oracle(model_dir, heads, nn_x, nn_y, boards):
    """Tolerances are _compare's fp32 bounds (1e-3 absolute on the raw
    outputs): edges and masks; test_one_layer_matches_float64 holds the sums."""
    _run_parity(_model(model_dir, *heads), False, 3, board_sizes=boards, label=f"attention {nn_x}x{nn_y}", nn_x=nn_x, nn_y=nn_y)


def test_rows_do_not_depend_on_batch(model_dir):
    lm = nn.LoadedModel(_model(model_dir, *HEADS[2]))
    h = nn.ComputeHandle(nn.ComputeContext(lm, 13, 13, use_fp16=False), max_batch=21)
    sp, gl = modelgen.synthetic_inputs(77, 21, 13, 13, board_sizes=(13, 9))
    full = h.get_output(sp, gl)
    one = h.get_output(sp[20:], gl[20:])
    for k in full:
        assert np.array_equal(full[k][20], one[k][0]), k


@pytest.mark.parametrize("nn_x,nn_y", [(5, 5), (13, 5), (16, 8), (19, 19)], ids=str)
@pytest.mark.parametrize("heads", HEADS, ids=["mha-q32v32", "gqa-q32v16", "mqa-q64v64"])
def test_one_layer_matches_float64(model_dir, heads, nn_x, nn_y):
    """A net of one attention layer against float64, each output in the 2-norm:
    sums and the softmax in fp32 measured up to 5.1e-7 here; a term in 16 bits
    would be 1e-3."""
    arch = dataclasses.replace(_tiny_transformer(*heads, True, True), blocks=["attention"])
    lm = nn.LoadedModel(modelgen.write_model(arch, 5, f"{model_dir}/{arch.name}-one.bin"))
    sp, gl = modelgen.synthetic_inputs(3, 3, nn_x, nn_y, board_sizes=((nn_x, nn_y), min(nn_x, nn_y) - 1))
    got = nn.ComputeHandle(nn.ComputeContext(lm, nn_x, nn_y, use_fp16=False), max_batch=3).get_output(sp, gl)
    want = torch_reference.forward(*nn.flatten_model(lm), sp, gl, nn_x, nn_y)
    for k in got:
        raw = got[k] * lm.info.output_scale_multiplier
        assert np.linalg.norm(raw - np.asarray(want[k]).reshape(raw.shape)) <= 2e-6 * np.linalg.norm(raw), k
