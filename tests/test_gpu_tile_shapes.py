"""The tile shapes that the expert products are launched in, alone and with the shared experts beside: every row has the
bits that it has in a call of many more rows, which takes other shapes.

Rows and widths stand on either side of a tile's edges; reductions end whole and ragged, and are long enough for a
kernel's stages or a step too short.  tests/test_kernel_choice.py holds the lists to all the tiles that there are.
"""

from __future__ import annotations

import pytest
import torch

from research_amd import grad

pytestmark = pytest.mark.gpu


def drawer(gpu, seed):
    generator = torch.Generator(device=gpu).manual_seed(seed)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    return normal


DENSE = [
    # hidden, inter, rows
    (512, 512, (97, 128, 129, 191, 193, 256, 257, 449, 700)),  # 64 x 64 to 128 x 128; just eight 64-deep steps
    (456, 520, (97, 129, 193, 257, 449, 700)),                 # ... the last of one chunk
    (448, 576, (97, 129, 193, 257, 449, 700)),                 # seven steps
    (320, 328, (97, 257, 700, 1500)),                          # five
    (2048, 1416, (97, 193, 449, 700, 1281, 2048)),
    (576, 4104, (97, 193, 449, 1281, 2049, 3000)),             # up to 256 x 128 and 128 x 256
    (384, 8200, (1023, 2048, 2177)),                           # ... six steps
]
LAYERS = [
    # hidden, inter, shared, experts, top-k, tokens
    (512, 512, 1024, 5, 2, (97, 161, 320, 333, 640)),
    (1024, 456, 0, 5, 2, (97, 161, 320, 333, 640)),
    (520, 1352, 520, 5, 2, (97, 161, 320, 333, 640)),
    (2048, 1408, 2816, 5, 2, (97, 320, 640)),
    (1472, 1416, 0, 40, 4, (640, 1024, 1080, 1400, 2400)),  # few rows a group, some 128, and more
    (320, 1032, 0, 40, 4, (640, 1000, 1500)),               # ... reductions too short for them
    (1024, 2056, 2048, 8, 2, (900, 1500, 3000)),            # joint launches
    (240, 256, 256, 24, 4, (500, 4200)),                    # ... of the shortest reductions
    (504, 1024, 1024, 4, 4, (161, 260, 2000, 4200)),
    (1728, 320, 216, 12, 3, (500, 2000, 3300, 4200)),
    (256, 640, 112, 12, 3, (260, 2000, 4200)),
    (576, 584, 576, 40, 2, (2600,)),
    (208, 1408, 576, 40, 2, (2000,)),
    (168, 128, 128, 4, 4, (4200,)),
    (448, 4312, 2176, 8, 1, (3300,)),
    (256, 7680, 1024, 8, 2, (1100, 4200)),                  # many rounds: rows beyond 256 in joint gate/up and dZ
    (7680, 256, 1024, 8, 2, (1100, 4200)),                  # ... down and dX
]


@pytest.mark.parametrize("hidden,inter,rows", DENSE)
def test_dense_rows(gpu, hidden, inter, rows):
    normal = drawer(gpu, hidden)
    x, dy = normal(9000, hidden, std=1.0), normal(9000, hidden, std=1.0)
    matrices = normal(hidden, inter), normal(hidden, inter), normal(inter, hidden)
    whole, kept = grad.shared_swiglu_train(x, *matrices)
    dx = grad.shared_backward(x, dy, *matrices, kept)[0]
    for n in rows:
        part, kept = grad.shared_swiglu_train(x[:n].contiguous(), *matrices)
        assert torch.equal(part, whole[:n]), f"{n} rows"
        part = grad.shared_backward(x[:n].contiguous(), dy[:n].contiguous(), *matrices, kept)[0]
        assert torch.equal(part, dx[:n]), f"dx of {n} rows"


@pytest.mark.parametrize("hidden,inter,shared,experts,top_k,tokens", LAYERS)
def test_layer_rows(gpu, hidden, inter, shared, experts, top_k, tokens):
    normal = drawer(gpu, inter)
    x, dy = normal(4500, hidden, std=1.0), normal(4500, hidden, std=1.0)
    bias = torch.zeros(experts, device=gpu)
    weights = normal(experts, hidden, inter), normal(experts, hidden, inter), normal(experts, inter, hidden)
    router = normal(hidden, experts)
    extra = (normal(hidden, shared), normal(hidden, shared), normal(shared, hidden)) if shared else None

    def run(n):
        rows = x[:n].contiguous()
        out, kept = grad.moe_forward_train(rows, router, bias, *weights, top_k, 1.0, shared=extra)
        back = grad.moe_backward(rows, dy[:n].contiguous(), None, router, *weights, extra, out, kept)
        return out.y, back.dx

    y, dx = run(4500)
    for n in tokens:
        part_y, part_dx = run(n)
        assert torch.equal(part_y, y[:n]), f"{n} tokens"
        assert torch.equal(part_dx, dx[:n]), f"dx of {n} tokens"
