"""Records low_latency.npz: outputs of the low-latency mode on an MI355X, with
every 3x3 convolution as split-K workgroups whose fp32 sums a second kernel
added in split order (the kernels the mode ran on every width at first).
Run from the repository's root: python3 tests/golden/make_low_latency_golden.py OUT.npz"""
import os
import sys
import tempfile

import numpy as np

sys.path.insert(0, os.getcwd())
from katago_amd import modelgen, nn

ROWS = 2


def _net(name, c, mid, blocks):
    return modelgen.Arch(name, 15, c, mid, 32, blocks, 16, 16, 32, 48, "ACTIVATION_RELU", residual_gain=0.5)


# 2 to 24 32-channel chunks per convolution: one to three chunks per split, the
# last split shorter than the others or not.
NETS = [_net("ll64", 64, 64, ["regular", "regulargpool"]), _net("ll128", 128, 128, ["regular", "regulargpool"]),
        _net("ll384-192", 384, 192, ["bottlenest2", "bottlenest2gpool"]), _net("ll320", 320, 320, ["regular", "regulargpool"]),
        _net("ll448", 448, 448, ["regular", "regulargpool"]), _net("ll704", 704, 704, ["regular"]), _net("ll768", 768, 768, ["regular"])]


def inputs(rows=ROWS):
    sp, gl = modelgen.synthetic_inputs(23, rows, board_sizes=(19, 13))
    return sp, gl, np.arange(rows, dtype=np.int32) % 8, np.full(rows, 0.25, np.float32)


def model_file(folder, arch):
    return modelgen.write_model(arch, 61, os.path.join(str(folder), arch.name + ".bin"))


if __name__ == "__main__":
    out = {}
    with tempfile.TemporaryDirectory() as d:
        for arch in NETS:
            lm = nn.LoadedModel(model_file(d, arch))
            h = nn.ComputeHandle(nn.ComputeContext(lm, 19, 19, use_fp16=True, low_latency=True), max_batch=ROWS)
            for k, v in h.get_output(*inputs()).items():
                out[arch.name + "/" + k] = v
    np.savez_compressed(sys.argv[1], **out)
