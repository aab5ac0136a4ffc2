"""The workloads that the performance of this backend is judged on.

Each case is one batched evaluation through a public entry point, as a program
that plays or analyses games makes it: ``ComputeHandle.get_output`` (rows in
host memory, the call KataGo's search makes) for small batches and
``DeviceHandle.forward_device`` (rows already on the GPU, outputs left there)
for large ones. Nets are the architectures of ``katago_amd.modelgen`` with
weights from a fixed seed; rows come from the case's seed.

A case:
  net          name of a modelgen architecture
  dtype        "fp16" (the default of every GPU backend) or "fp32" (useFP16 = false)
  batch        boards per call
  x, y         size of the net's input tensor (nnXLen, nnYLen)
  boards       side lengths of the boards in it, cycled over the rows ("9,13,19")
  path         "host" or "device"
  low_latency  the hipLowLatency option
  vary         rows use all symmetries and any policy optimism (else 0)
"""
import math
import os
import tempfile

import numpy as np
import torch

from katago_amd import modelgen, nn

NETS = {"b6c96": modelgen.b6c96, "b10c128": modelgen.b10c128, "b18c384nbt": modelgen.b18c384nbt,
        "t12d384h6": modelgen.transformer_d384}
WEIGHT_SEED = 1000
NUM_SPATIAL, NUM_GLOBAL, SCORE_C = 22, 19, 6


def _case(name, net, batch, dtype="fp16", x=19, y=19, boards="19", path="host", low_latency=False, vary=False):
    return {"name": name, "net": net, "dtype": dtype, "batch": batch, "x": x, "y": y, "boards": boards, "path": path,
            "low_latency": low_latency, "vary": vary}


def listed():
    return [
        # A search with one thread: one leaf per call, latency is all that counts.
        _case("b18 fp16 1 board", "b18c384nbt", 1),
        # The same for a user who set hipLowLatency.
        _case("b18 fp16 1 board low latency", "b18c384nbt", 1, low_latency=True),
        # An ordinary search (16 threads) with the net loaded at 19x19 and games on 9x9 to 19x19.
        _case("b18 fp16 16 mixed boards", "b18c384nbt", 16, boards="9,13,19", vary=True),
        # Small-board play: the net's tensor sized to the board.
        _case("b18 fp16 24 boards 9x9", "b18c384nbt", 24, x=9, y=9, boards="9", vary=True),
        # Analysis of 13x13 games in batches, rows on the GPU.
        _case("b18 fp16 96 boards 13x13", "b18c384nbt", 96, x=13, y=13, boards="13", path="device"),
        # Self-play or batched analysis at full batch: the headline throughput.
        _case("b18 fp16 256 boards", "b18c384nbt", 256, path="device"),
        # A mid-size net at a common server batch.
        _case("b10 fp16 64 boards", "b10c128", 64, path="device"),
        # The parity configuration: a small net in fp32.
        _case("b6 fp32 8 boards", "b6c96", 8, dtype="fp32"),
        # The main net with useFP16 = false.
        _case("b18 fp32 16 boards", "b18c384nbt", 16, dtype="fp32", vary=True),
        # The transformer net at full batch, for a search of a few threads, and in fp32.
        _case("t12 fp16 128 boards", "t12d384h6", 128, path="device"),
        _case("t12 fp16 4 boards", "t12d384h6", 4, vary=True),
        _case("t12 fp32 8 boards", "t12d384h6", 8, dtype="fp32"),
    ]


def draw(rng):
    """One more case of the same ranges: batches over their logarithm, any
    board size a game may have (square or not), mixed sizes, both dtypes."""
    net, dtype, lo, hi = rng.choices(
        [("b18c384nbt", "fp16", 361, 256 * 361), ("b10c128", "fp16", 361, 192 * 361), ("t12d384h6", "fp16", 361, 128 * 361),
         ("b6c96", "fp32", 361, 48 * 361), ("b18c384nbt", "fp32", 361, 16 * 361), ("t12d384h6", "fp32", 361, 8 * 361)],
        weights=[8, 3, 4, 2, 1, 1])[0]
    x = y = 19
    shape = rng.random()
    if shape > 0.75:
        x, y = rng.randint(7, 19), rng.randint(7, 19)
    elif shape > 0.4:
        x = y = rng.randint(7, 18)
    most = hi // (x * y)
    batch = max(1, min(most, int(round(math.exp(rng.uniform(0.0, math.log(most + 0.49)))))))
    side = min(x, y)
    boards = str(side) if rng.random() < 0.7 else ",".join(str(max(5, side - k)) for k in (rng.randint(1, 9), rng.randint(1, 4), 0))
    low = dtype == "fp16" and batch <= 8 and net != "t12d384h6" and rng.random() < 0.3
    case = _case("", net, batch, dtype, x, y, boards, "host" if batch <= 32 else "device", low, rng.random() < 0.5)
    del case["name"]
    return case


# -- inputs -------------------------------------------------------------------

def _sizes(case):
    sides = [int(s) for s in case["boards"].split(",")]
    full = max(sides) == min(case["x"], case["y"])
    # The largest entry stands for a board that fills the tensor, square or not.
    return [(case["x"], case["y"]) if full and s == max(sides) else (s, s) for s in (sides[i % len(sides)] for i in range(case["batch"]))]


def _inputs(case, seed):
    """Feature rows with the densities of game positions: the on-board mask,
    stones of both colours on disjoint points, sparse other planes."""
    rng = np.random.default_rng(seed)
    n, h, w = case["batch"], case["y"], case["x"]
    on = np.zeros((n, h, w), bool)
    for i, (bx, by) in enumerate(_sizes(case)):
        on[i, :by, :bx] = True
    u = rng.random((n, h, w, NUM_SPATIAL), dtype=np.float32)
    sp = (u < 0.1).astype(np.float32)
    sp[..., 1] = u[..., 1] < 0.35
    sp[..., 2] = (u[..., 2] < 0.35) & (u[..., 1] >= 0.35)
    sp[..., 0] = 1.0
    sp *= on[..., None]
    gl = rng.uniform(-1.0, 1.0, (n, NUM_GLOBAL)).astype(np.float32)
    sym = np.zeros(n, np.int32)
    opt = np.zeros(n, np.float32)
    if case["vary"]:
        sym = rng.integers(0, 8 if h == w else 4, n).astype(np.int32)
        opt = rng.random(n).astype(np.float32)
    return sp.reshape(n, -1), gl, sym, opt


# -- what a program keeps: loaded nets, contexts and handles ----------------------

_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _model_file(net):
    folder = os.path.join(tempfile.gettempdir(), "katago_amd_models")
    os.makedirs(folder, exist_ok=True)
    path = os.path.join(folder, "%s-perf-s%d.bin" % (net, WEIGHT_SEED))
    if not os.path.exists(path):
        part = path + ".%d.bin" % os.getpid()
        modelgen.write_model(NETS[net](), WEIGHT_SEED, part)
        os.replace(part, path)
    return path


def _loaded(net):
    return _keep(("net", net), lambda: nn.LoadedModel(_model_file(net)))


def _host_handle(case):
    net, fp16, x, y, low = case["net"], case["dtype"] == "fp16", case["x"], case["y"], case["low_latency"]
    # The built-in kernel choices: a tuning run per handle would time the boxes, not the code.
    ctx = _keep(("context", net, fp16, x, y, low),
                lambda: nn.ComputeContext(_loaded(net), x, y, use_fp16=fp16, auto_tune=False, low_latency=low))
    return _keep(("handle", net, fp16, x, y, low, case["batch"]), lambda: nn.ComputeHandle(ctx, case["batch"]))


def _device_handle(case):
    net, fp16 = case["net"], case["dtype"] == "fp16"
    dm = _keep(("device net", net, fp16), lambda: nn.DeviceModel(_loaded(net), use_fp16=fp16))
    return _keep(("device handle", net, fp16, case["x"], case["y"], case["batch"]),
                 lambda: nn.DeviceHandle(dm, case["batch"], case["x"], case["y"]))


def prepare(case, seed):
    rows = _inputs(case, seed)
    if case["path"] == "host":
        return {"handle": _host_handle(case), "rows": rows}
    h = _device_handle(case)
    n, hw = case["batch"], case["x"] * case["y"]
    rows = [torch.from_numpy(r).cuda() for r in rows]
    out = torch.zeros((n, h.row_floats), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()  # the handle runs on a stream of its own
    parts = {"policy": out[:, :hw + 1], "value": out[:, hw + 1:hw + 4], "score": out[:, hw + 4:hw + 4 + SCORE_C],
             "ownership": out[:, hw + 4 + SCORE_C:]}
    return {"handle": h, "rows": rows, "n": n, "out": out, "ptrs": [t.data_ptr() for t in (*rows, out)], "parts": parts}


def run(state):
    if "out" in state:
        state["handle"].forward_device(state["n"], *state["ptrs"])
        return state["parts"]
    return state["handle"].get_output(*state["rows"])


# -- the work a pass cannot do without --------------------------------------------

def _net_work(arch, hw):
    """(weights, FLOPs per board) of an architecture: every weight once, 2 FLOPs
    per multiply-add of the direct convolutions, products and attention."""
    weights = flops = 0.0

    def mul(cin, cout, times):
        nonlocal weights, flops
        weights += cin * cout
        flops += 2.0 * cin * cout * times

    def ordinary(c, mid):
        mul(9 * c, mid, hw)
        mul(9 * mid, c, hw)

    def gpool(c, mid, gp):
        mul(9 * c, mid, hw)
        mul(3 * gp, mid - gp, 1)
        mul(9 * (mid - gp), c, hw)

    c, mid, gp = arch.trunk_c, arch.mid_c, arch.gpool_c
    mul(9 * arch.num_input, c, hw)
    mul(arch.num_global, c, 1)
    for kind in arch.blocks:
        if kind == "regular":
            ordinary(c, mid)
        elif kind == "regulargpool":
            gpool(c, mid, gp)
        elif kind == "attention":
            q, k, v = arch.heads * arch.q_head_dim, arch.kv_heads * arch.q_head_dim, arch.kv_heads * arch.v_head_dim
            mul(c, q + k + v, hw)
            flops += 2.0 * hw * hw * arch.heads * (arch.q_head_dim + arch.v_head_dim)
            mul(arch.heads * arch.v_head_dim, c, hw)
        elif kind == "ffn":
            mul(c, 2 * arch.ffn_c, hw)
            mul(arch.ffn_c, c, hw)
        else:
            mul(c, mid, hw)
            gpool(mid, mid, gp) if kind.endswith("gpool") else ordinary(mid, mid)
            ordinary(mid, mid)
            mul(mid, c, hw)
    mul(c, arch.p1_c + arch.g1_c + arch.v1_c, hw)
    mul(arch.p1_c, 2, hw)
    mul(arch.v1_c, 1, hw)
    mul(3 * arch.g1_c, 2 * arch.p1_c, 1)
    mul(arch.p1_c, 2, 1)
    mul(3 * arch.v1_c, arch.v2_c, 1)
    mul(arch.v2_c, 3 + SCORE_C, 1)
    return weights, flops


def work(case):
    hw, n = case["x"] * case["y"], case["batch"]
    weights, flops = _net_work(NETS[case["net"]](), hw)
    row = 4 * (hw * NUM_SPATIAL + NUM_GLOBAL + 2 + 2 * hw + 4 + SCORE_C)  # fp32 rows in and out
    return {"bytes": weights * (2 if case["dtype"] == "fp16" else 4) + n * row, "flops": n * flops}


def tolerance(case):
    """About four times what whole nets measured against exact() on MI355X, the
    worst of the four outputs: up to 1.8e-3 in fp16 (activations and weights
    rounded to 11 bits, fp32 sums) and 2.3e-6 in fp32."""
    return {"rel": 7e-3, "max": 0.1} if case["dtype"] == "fp16" else {"rel": 1e-5, "max": 3e-4}


# -- the same in 64 bits -----------------------------------------------------------

class _File:
    """Reads a binary model file token by token."""

    def __init__(self, path, device):
        with open(path, "rb") as f:
            self.data = f.read()
        self.pos, self.device = 0, device

    def token(self):
        while self.data[self.pos:self.pos + 1].isspace():
            self.pos += 1
        end = self.pos
        while not self.data[end:end + 1].isspace():
            end += 1
        self.pos, t = end, self.data[self.pos:end]
        return t.decode()

    def skip(self, count):
        for _ in range(count):
            self.token()

    def floats(self, *shape):
        at = self.data.index(b"@BIN@", self.pos) + 5
        n = int(np.prod(shape))
        self.pos = at + 4 * n
        return torch.from_numpy(np.frombuffer(self.data, "<f4", n, at).astype(np.float64).reshape(shape)).to(self.device)

    def conv(self):
        self.token()
        ky, kx, cin, cout, _, _ = (int(self.token()) for _ in range(6))
        return self.floats(ky, kx, cin, cout)

    def matmul(self):
        self.token()
        cin, cout = int(self.token()), int(self.token())
        return self.floats(cin, cout)

    def vector(self):
        self.token()
        return self.floats(int(self.token()))

    def bn_act(self):
        self.token()
        c, eps = int(self.token()), float(self.token())
        self.skip(2)
        mean, var, scale, bias = (self.floats(c) for _ in range(4))
        scale = scale / torch.sqrt(var + eps)
        return scale, bias - mean * scale, self.act()

    def act(self):
        self.token()
        return self.token()

    def norm(self):
        self.token()
        c, eps = int(self.token()), float(self.token())
        return self.floats(c), eps


def _act(x, kind):
    if kind == "ACTIVATION_RELU":
        return torch.relu(x)
    if kind == "ACTIVATION_MISH":
        return x * torch.tanh(torch.nn.functional.softplus(x, threshold=60.0))
    if kind == "ACTIVATION_SILU":
        return x * torch.sigmoid(x)
    return x


class _Net:
    """KataGo's forward pass over [n, h, w, channels] tensors in float64,
    evaluated while the model file is read."""

    def __init__(self, arch, path, device):
        self.arch, self.file = arch, _File(path, device)

    @staticmethod
    def conv(x, wt):
        if wt.shape[0] == 1:
            return x @ wt[0, 0]
        h, w = x.shape[1:3]
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        return sum(xp[:, dy:dy + h, dx:dx + w].contiguous() @ wt[dy, dx] for dy in range(3) for dx in range(3))

    def bn(self, x, p):
        return _act(x * p[0] + p[1], p[2]) * self.mask

    def pool(self, x, value):
        mean = x.sum(dim=(1, 2)) / self.area[:, None]
        root = torch.sqrt(self.area)[:, None] - 14.0
        last = mean * (root * root * 0.01 - 0.1) if value else (x + self.mask - 1.0).amax(dim=(1, 2)).clamp(min=-1.0)
        return torch.cat([mean, mean * root * 0.1, last], dim=1)

    def ordinary(self, x):
        f = self.file
        f.skip(1)
        y = self.conv(self.bn(x, f.bn_act()), f.conv())
        return x + self.conv(self.bn(y, f.bn_act()), f.conv())

    def gpool(self, x):
        f = self.file
        f.skip(1)
        a = self.bn(x, f.bn_act())
        reg, gp = self.conv(a, f.conv()), self.conv(a, f.conv())
        reg = reg + (self.pool(self.bn(gp, f.bn_act()), False) @ f.matmul())[:, None, None, :]
        return x + self.conv(self.bn(reg, f.bn_act()), f.conv())

    def rms(self, x, p):
        return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + p[1]) * p[0]

    def rotate(self, t, angle):
        c, s = torch.cos(angle), torch.sin(angle)
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], dim=-1).flatten(-2)

    def attention(self, x):
        f = self.file
        f.skip(1)
        heads, kv, dq, dv, _, _ = (int(f.token()) for _ in range(6))
        xn = self.rms(x, f.norm()) * self.mask
        n, h, w, _ = x.shape
        q, k, v = (((xn @ f.matmul()).reshape(n, h * w, nh, d).permute(0, 2, 1, 3)) for nh, d in ((heads, dq), (kv, dq), (kv, dv)))
        out = f.matmul()
        f.skip(4)
        freqs = f.floats(kv, dq // 2, 2)
        ys, xs = torch.meshgrid(torch.arange(h, device=x.device), torch.arange(w, device=x.device), indexing="ij")
        # Position angles as the model's fp32 tables hold them are within an ulp of these.
        angle = (xs.reshape(-1)[None, :, None] * freqs[:, None, :, 0] + ys.reshape(-1)[None, :, None] * freqs[:, None, :, 1])
        rep = heads // kv
        q = self.rotate(q, angle.repeat_interleave(rep, 0))
        k = self.rotate(k, angle).repeat_interleave(rep, 1)
        v = v.repeat_interleave(rep, 1)
        s = torch.matmul(q.contiguous(), k.transpose(2, 3).contiguous()) / math.sqrt(dq)
        s = s.masked_fill(self.mask.reshape(n, 1, 1, h * w) == 0, -math.inf).softmax(dim=-1)
        o = torch.matmul(s, v.contiguous()).permute(0, 2, 1, 3).reshape(n, h, w, heads * dv)
        return x + (o * self.mask @ out) * self.mask

    def ffn(self, x):
        f = self.file
        f.skip(4)
        xn = self.rms(x, f.norm()) * self.mask
        a = _act(xn @ f.matmul(), "ACTIVATION_SILU") * (xn @ f.matmul())
        return x + (a @ f.matmul()) * self.mask

    def block(self, x):
        f = self.file
        kind = f.token()
        if kind == "ordinary_block":
            return self.ordinary(x)
        if kind == "gpool_block":
            return self.gpool(x)
        if kind == "transformer_attention_block":
            return self.attention(x)
        if kind == "transformer_ffn_block":
            return self.ffn(x)
        f.skip(1)
        inner = int(f.token())
        m = self.conv(self.bn(x, f.bn_act()), f.conv())
        for _ in range(inner):
            m = self.block(m)
        return x + self.conv(self.bn(m, f.bn_act()), f.conv())

    def forward(self, x, g):
        f, a = self.file, self.arch
        self.mask, self.area = x[..., :1], x[..., 0].sum(dim=(1, 2))
        f.skip(4 + 7 + 8)
        f.skip(7 + 6)
        t = self.conv(x, f.conv()) + (g @ f.matmul())[:, None, None, :]
        for _ in a.blocks:
            t = self.block(t)
        if a.trunk_rmsnorm:
            f.token()
            c, eps = int(f.token()), float(f.token())
            gamma, beta = f.floats(c), f.floats(c)
            t = _act(self.rms(t, (gamma, eps)) + beta, f.act()) * self.mask
        else:
            t = self.bn(t, f.bn_act())
        f.skip(5 if a.version >= 17 else 1)
        p1, g1 = self.conv(t, f.conv()), self.conv(t, f.conv())
        gp = self.pool(self.bn(g1, f.bn_act()), False)
        p1 = p1 + (gp @ f.matmul())[:, None, None, :]
        policy = self.conv(self.bn(p1, f.bn_act()), f.conv())
        passes = _act(gp @ f.matmul() + f.vector(), f.act()) @ f.matmul()
        f.skip(4 if a.version >= 17 else 1)
        v1 = self.conv(t, f.conv())
        v1 = self.bn(v1, f.bn_act())
        hidden = _act(self.pool(v1, True) @ f.matmul() + f.vector(), f.act())
        value = hidden @ f.matmul() + f.vector()
        score = hidden @ f.matmul() + f.vector()
        return policy, passes, value, score, self.conv(v1, f.conv())[..., 0]


def _turn(a, sym, back):
    """A [h, w, ...] array under symmetry sym (bit 0 flips y, bit 1 flips x,
    then bit 2 transposes), or back."""
    if back and sym & 4:
        a = np.swapaxes(a, 0, 1)
    if sym & 1:
        a = a[::-1]
    if sym & 2:
        a = a[:, ::-1]
    if not back and sym & 4:
        a = np.swapaxes(a, 0, 1)
    return a


def exact(case, seed):
    n, h, w = case["batch"], case["y"], case["x"]
    sp, gl, sym, opt = _inputs(case, seed)
    sp = sp.reshape(n, h, w, NUM_SPATIAL).astype(np.float64)
    x = np.stack([_turn(sp[i], sym[i], False) for i in range(n)])
    device = "cuda" if torch.cuda.is_available() else "cpu"
    net = _Net(NETS[case["net"]](), _model_file(case["net"]), device)
    out = net.forward(torch.from_numpy(x).to(device), torch.from_numpy(gl.astype(np.float64)).to(device))
    policy, passes, value, score, own = (t.cpu().numpy() for t in out)
    mix = opt.astype(np.float64)
    policy = policy[..., 0] + (policy[..., 1] - policy[..., 0]) * mix[:, None, None]
    passes = passes[:, 0] + (passes[:, 1] - passes[:, 0]) * mix
    policy, own = (np.stack([_turn(a[i], sym[i], True) for i in range(n)]).reshape(n, h * w) for a in (policy, own))
    # Raw outputs are the net's divided by this constant of the loaded model.
    scale = _loaded(case["net"]).info.output_scale_multiplier
    return {"policy": np.concatenate([policy, passes[:, None]], axis=1) / scale, "value": value / scale, "score": score / scale,
            "ownership": own / scale}
