"""Write tests/golden/gradient_hashes.json: SHA-256 digests of the network's
weight and bias gradients, of single layers and of the first steps of a training
run.

The order in which a gradient's products are summed is part of a training run's
results: Adam divides a gradient by its own size, so a difference of 1e-7 in a
sum becomes another BF16 weight a few steps later, and a percent in the outputs
after that.  The digests were made with the kernels that staged the tiles of the
weight gradient transposed and summed the bias gradients in launches of their
own; any later kernel gives the same bits.  Run from the repository root on an
MI355X:
    python tests/golden/make_gradient_hashes.py
"""
import hashlib
import json
import os
import sys

import numpy as np
import torch

OUT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gradient_hashes.json")

# N, H, W, Cin, Cout: ragged tiles, one to many ranges of tiles per layer, and a
# pixel count beyond one partial of the bias sums
LAYERS = [(1, 1, 1, 32, 32), (1, 7, 5, 96, 128), (3, 21, 35, 32, 64), (5, 16, 16, 128, 128),
          (2, 66, 130, 64, 32), (1, 200, 40, 224, 96), (6, 104, 152, 96, 32)]
# N, H, W, steps of a training run
RUNS = [(3, 104, 152, 6), (4, 32, 48, 5)]


def digest(*tensors) -> str:
    h = hashlib.sha256()
    for t in tensors:
        t = t.detach()
        h.update((t.view(torch.int16) if t.dtype == torch.bfloat16 else t).cpu().numpy().tobytes())
    return h.hexdigest()


def layer(sg, n, h, w, cin, cout):
    """Digests of a layer's dw and db."""
    gen = torch.Generator().manual_seed(h * w + cin + cout)
    conv = sg.Conv(cin, cout, 9, np.random.default_rng(0), "cuda:0")
    x, g = (torch.randn(n, h, w, c, generator=gen).to(torch.bfloat16).cuda() for c in (cin, cout))
    conv.backward(x, g, (n, h, w), sg.Scratch("cuda:0"), need_dx=False)
    return {"dw": digest(conv.dw), "db": digest(conv.db)}


def run(sg, n, h, w, steps):
    """Digests of each step's output, gradients and updated weights."""
    gen = torch.Generator().manual_seed(h + w)
    net = sg.UNet(seed=n, device="cuda:0")
    x = torch.randn(n, h, w, 8, generator=gen).to(torch.bfloat16).cuda()
    t = torch.randn(n, h, w, 3, generator=gen).cuda()
    out = []
    for _ in range(steps):
        y = net.forward(x)
        _, gy = sg.mse_loss_and_grad(y, t)
        net.backward(gy)
        net.step(2e-4)
        cs = net.convs()
        out.append({"out": digest(y), "dw": digest(*(c.dw for c in cs)),
                    "db": digest(*(c.db for c in cs)), "w": digest(*(c.w for c in cs))})
    return out


def key(*dims) -> str:
    return "x".join(map(str, dims))


def main():
    sys.path.insert(0, os.getcwd())
    from simplehydrology_amd import surrogate as sg
    res = {"layers": {key(*a): layer(sg, *a) for a in LAYERS},
           "runs": {key(*a): run(sg, *a) for a in RUNS}}
    with open(sys.argv[1] if len(sys.argv) > 1 else OUT, "w") as f:
        json.dump(res, f, indent=1)


if __name__ == "__main__":
    main()
